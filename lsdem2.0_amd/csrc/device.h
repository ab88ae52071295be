// Device data layout of one LS-DEM context.  All arrays live in HBM; the struct is passed by
// value to every kernel.
#pragma once
#include <cstddef>

#include "dmath.h"
#include "surrogate.h"

namespace lsd {

enum PairType : uint32_t { PT_PP = 0, PT_PW = 1, PT_GX = 2, PT_GY = 3, PT_GXY = 4 };
constexpr uint32_t kPartnerMask = 0x0FFFFFFFu;
constexpr uint64_t kHashEmpty = ~0ull;

// Shape: FP32 SDF grid (x fastest) + boundary nodes grouped into clusters of <= 64 nodes.
struct ShapeDev {
  int nx, ny, nz, nNodes;
  int nodeOff, nClusters, clusterOff, pad0;
  long long sdfOff;
  double ox, oy, oz, h;  // unscaled grid origin and spacing
  double boxR;           // max |corner| of the grid box (unscaled), used for fixed-partner culls
  double lip;            // Lipschitz bound of the trilinear interpolant over cells with a positive
                         // corner (scale invariant)
  double nodeR;          // max |node| (unscaled): how far a node lies from the body origin
};
struct ClusterDev {
  double cx, cy, cz, rho;  // bounding sphere of the cluster's nodes (unscaled)
  int first, count;        // node range in the shape's cluster-ordered nodes
  int subFirst, nSub;      // sub-clusters (<= 16 nodes each)
};
struct ClusterF32 {
  float cx, cy, cz, rho;  // FP32 copy of the bounding sphere, rho rounded up
  int first, count;
  int subFirst, nSub;     // clusters: global index of the first sub-cluster and their number
};
struct NodeDev {
  double x, y, z;  // unscaled local position
  int orig;        // index of the node in the shape's node list as given by the caller
  int pad;
};

struct GridGeom {  // geometry of the reference spatial grid (spatialGrid::set)
  d3 mn, mx, inv;
  i3 size;
  int pad;
};
struct SearchGrid {  // this library's own broad-phase grid
  d3 mn;
  double cell, invCell;
  i3 size;
  int ncell;
};

// A particle's per-step record for the pair check:
//   motion: displacement of posDet since the build (x, y, z) and the chord 2 sin(angle / 2) of the
//           rotation since the build (w);
//   key:    reference-grid key (x; -1 outside the domain) and the keys of ghost images 0..2 (y, z, w;
//           -1: no image), each with bit kFlipBit set when the image's shift state differs from the
//           build's.
// (32 bytes: one read per partner.)  The rotation since the build as a quaternion is kept apart
// (qrel), read only when a certificate is checked against the motion since an evaluation.
struct alignas(16) BodyStep {
  float4 motion;
  int4 key;
};
constexpr int kFlipBit = 30;

// The state vectors' places in their block (Params::pos).
enum { kSvPos = 0, kSvDet = 1, kSvVel = 2, kSvAng = 3, kSvImg = 4, kSvImgVel = 7 };

// What does not change of a particle or wall, in one 128-byte line: the narrow phase reads it for pairs
// picked from anywhere in the list, where an array per property cost a line each.
struct alignas(128) BodyProp {
  double origin[3];           // scale * grid origin
  double scale, radius;       // a wall: 1, 0
  double invSp;               // 1 / (scale * spacing)
  double kn, ks;              // a wall: 0
  double mu, res, diss;       // diss = dissipation(res), computed on the device at initialisation
  double invM;                // a wall: 0
  double rNode;               // scale * largest node distance from the body's origin
  int nodeStart, shape;       // first of its boundary nodes in the numbering over all particles
  int nNodes, pad[3];
};
static_assert(sizeof(BodyProp) == 128, "a line each");
// its values by number, as doubles (kPropInts: nodeStart and shape)
enum { kPropOrigin = 0, kPropScale = 3, kPropRadius = 4, kPropInvSp = 5, kPropKn = 6, kPropKs = 7, kPropMu = 8, kPropRes = 9,
       kPropDiss = 10, kPropInvM = 11, kPropInts = 13 };
static_assert(offsetof(BodyProp, nodeStart) == 8 * kPropInts && offsetof(BodyProp, invM) == 8 * kPropInvM &&
                  offsetof(BodyProp, radius) == 8 * kPropRadius, "kProp* name BodyProp's doubles");
static_assert(sizeof(BodyStep) == 32 && alignof(BodyStep) == 16, "step record: motion then key, 16 B each");

constexpr int kBarrierLine = 32;                  // ints per barrier word (one 128-byte line each)

struct Params {
  // ---- sizes and scalars ----
  int nP, nW, nBonds;
  d3 g;
  double dt;
  int quirks, periodicX, periodicY, sdfCull;
  int narrowBatch;    // pairs per wavefront batch of k_candidates (0: chosen on the device)
  int prime;          // 1: the pre-loop build of a solve phase (detection at the current poses: no
                      // kick, no drift, no contact law; springs carried over as found)
  int callStep;       // index of this step within the lsdem_step call (recorded with an error flag)
  int barrierSpin;    // poll limit of a broad-phase grid barrier before it gives up (time-out error)
  int periodicSector; // quarter-sector rotational periodicity about the z axis through gridP.mn
  GridGeom gridP, gridW;
  SearchGrid sg;
  double rMax;        // max particle bounding radius
  double halfSkin;    // candidate pairs are reused until a body has moved this far since they were built
  double boxRMax;     // max scaled grid-box radius over particles (ghost search reach)
  long long pairCap, contactCap;
  unsigned long long hashMask;

  // ---- shapes ----
  const ShapeDev* shapes;
  const NodeDev* nodes;
  const ClusterF32* clusters32;
  const ClusterF32* subs32;  // sub-clusters of <= 16 nodes
  float4* pairMap;        // per evaluated pair (list position): 160-byte FP32 map record
  const float4* nodes32;  // same nodes in FP32 (x, y, z, 0) for the conservative prefilter
  const float* sdf;
  int maxClusters;        // largest cluster count of any shape
  int residentWaves;      // wavefronts of the candidate kernel that are on the GPU together

  // ---- particles ----
  // State vectors lie in one block of nBodies = nP + nW entries each, walls after the particles, in the
  // order of kSv* (pos, posDet, vel, angvel, then the image positions and, with sector periodicity, their
  // velocities); orientations likewise (quat, then quatDet and the three image sets with sector
  // periodicity).  Vector s of body i is pos[s * nBodies + i].
  int nBodies;
  d3* pos;      // state position (after any periodic wrap)
  d3* posDet;   // position used by the particle-particle and wall detection of this step (particles only: a
                // wall is detected where it is)
  q4* quat;
  d3* vel;
  d3* angvel;
  d3* force;
  d3* torque;
  const s6* invI;
  const double* invM;
  const double* radius;
  const double* scale;
  const int* shape;
  const BodyProp* prop;  // per particle, then per wall
  int* scell;            // search-grid cell of pos (post-wrap), rebuild steps only
  d3* xBuild;            // posDet when the candidate pairs were built
  d3* xBuildW;           // pos when the candidate pairs were built
  q4* qBuild;            // quat when the candidate pairs were built
  int* imgBuild;         // image shift states at the build (bit g: image g lies a period away)
  BodyStep* step;        // per particle, written every step: motion since the build and keys
  float4* qrel;          // per particle: conj(q_build) q in FP32 (rotation since the build)

  // ---- walls (state vectors: nP entries into the particles') ----
  d3* wpos;
  q4* wquat;
  d3* wvel;
  d3* wangvel;
  const int* wshape;
  int* wkey;
  d3* wBuildPos;         // wall pose when the candidate pairs were built
  q4* wBuildQ;
  float4* wMotion;       // as motion, for walls
  float4* wSph;          // FP32 bounding sphere of each wall's grid box at its current pose (centre,
                         // boxR), written at every drift: the pair search's first wall test
  float4* wQrel;         // as qrel, for walls

  // ---- periodic ghost images (3 sets: +x, +y, +x+y; with sector periodicity, turned by +90, 180
  // and -90 degrees about the z axis through gridP.mn) ----
  d3* gpos[3];       // image positions, written only for images that exist (key >= 0 in the step
                     // record); the keys live in the step record
  q4* gquat[3];      // sector images only: orientation and velocity of each existing image
  d3* gvel[3];
  q4* quatDet;       // sector periodicity: orientation used for particle-particle detection (before
                     // this step's turn of a body that left the sector)
  d3 secW[3];        // rotation vectors (0, 0, angle) of the three sector image sets
  double secA[3], secB[3];  // their Rodrigues coefficients, computed on the host
  q4 secR[3];        // their unit quaternions, computed on the host

  // ---- search grid of particles ----
  int* cellCount;   // ncell (scratch)
  int* cellStart;   // ncell + 1
  int* sorted;      // nP: particle ids in (cell, id) order
  int* rank;        // nP (scratch)
  // particle data gathered into sorted order (contiguous runs per search-grid row)
  float4* sPR;      // FP32 (posDet, bounding radius; radius -1 when the particle has no reference key)
  float4* sPRw;     // FP32 (pos after the periodic wrap, bounding radius)
  float* sBoxR;     // scaled grid-box radius (ghost-image reach)
  int* rcTmp;       // reaction pairs before the per-partner sort
  int* sortTmp;     // counting-sort scratch (items before the per-bucket sort)
  int* sortBig;     // counting-sort scratch (list of buckets of more than 16 items)
  int* scanTiles;   // scan scratch (tile sums)
  uint32_t* pairSlab;  // nP x kPairSlab: first candidate pairs of each master (32 of each master in a row)
  unsigned long long* wallMask;  // per sorted position, with up to 64 walls: those the particle can reach

  // ---- candidate pairs (current step) ----
  int* pairCount;   // nP (+1) counts then exclusive prefix pairStart
  int* pairStart;   // nP + 1
  int* pairA;       // pairCap
  uint32_t* pairInfo;  // (type << 28) | partner
  int* pairCcnt;    // contacts of the pair
  int2* pairSpan;   // of a pair with contacts: the first of its terms in cTerm and their number
  // separation certificates: a pair whose nodes were all culled with slack s (world units, less
  // the motion bound at that step) is skipped while the motion bound since the build stays below s
  int* oldStart;           // the previous pair list kept through a rebuild: per-master starts (nP + 1),
  uint32_t* oldInfo;       // pair entries and certificates, for the certificates the new list inherits
  float4* oldCert;
  float4* cert;     // pairCap: (s_build or -1, cB, cA, s or -1): s_build against the motion since the
                    // build, s against the motion since the pair's last evaluation (below)
  float4* certE;    // pairCap: at the last evaluation, dA - dB (x, y, z) and the image's flip state (w)
  float4* certQA;   // pairCap: at the last evaluation, the master's qrel
  float4* certQB;   // pairCap: at the last evaluation, the partner's qrel
  int* pairRec;     // pair -> position of its map record in pairMap this step
  int useCert;
  // reaction CSR (pairs whose partner is a particle that receives the reaction)
  int* rcCount;     // nP
  int* rcStart;     // nP + 1
  int* rcPair;      // pairCap
  int* rcSlot;      // pairCap: place of a reaction pair in rcPair
  int2* rcSpan;     // pairSpan of the pairs in rcPair's order
  int* rcRank;      // pairCap (scratch)

  // ---- contacts (current step) ----
  int* cNode;
  uint32_t* cInfo;      // (type << 28) | partner, kInvalidInfo for an unused slot
  int* cPair;           // candidate pair of the contact
  double* cTerm;        // 9 per contact (force, torque on the master, torque on the partner), a pair's
                        // contacts side by side from its first candidate slot on
  d3* cSpring;
  d3* cPoint;
  d3* cNormal;
  double* cOverlap;
  double* cEn;
  double* cEs;
  // history: two hash tables keyed by (list, node, partner), used in alternate steps; this step
  // inserts its contacts into one and looks up the previous step's springs in the other
  const d3* prevSpring;
  unsigned long long* hashKey;        // this step's table
  int* hashVal;
  int* hashSlot;                      // slot taken by each contact slot (-1: none), per table
  const unsigned long long* prevHashKey;  // the previous step's table
  const int* prevHashVal;
  int curBuf;                         // which of the two tables and contact buffers is this step's

  // ---- bonds ----
  const int* bI;
  const int* bJ;
  int* bActive;
  const double* bConst;  // 9 per bond: B1 B2 B3 B4 radius L0 sigmaT cohesion mu
  const d3* bLocal;      // 8 per bond: n1i n2i n3i pi n1j n2j n3j pj
  d3* bPoint;
  double* bOut;          // 6 per bond: Un Us Ub Ut sigmaMax tauMax
  double* bEnd;          // 6 per bond end, in the CSR's order: force and torque (moment + arm x F) there
  const int* bEndAt;     // 2*nBonds: place of bond k's i end (2k) and j end (2k + 1) in bEnd
  const int* bcStart;    // nP + 1 CSR of bond ends per particle, in bond order

  // ---- device counters ----
  // devInt: [1] contact slots allocated this step, [3] error flags (kErr*: any flag halts every later
  //         kernel of the call),
  //         [4] peak pairs, [5] peak candidate slots, [6] slots scanned by the history insert,
  //         [7] images at their source's own position, [8] rebuild flag of the step,
  //         [9] (unused), [10 + b] contact slots of the
  //         last step that filled history table b, [12] grid-barrier arrivals of the broad phase,
  //         [20] callStep of the step that raised the first error flag (-1: none), [21], [22] a rebuild's
  //         large buckets (kBigCellsIdx, kBigRcIdx), [23] error flags that a launch found up when it
  //         began (kHaltedIdx)
  int* devInt;
  int* barrier;          // grid barrier of the single-launch broad phase: kBarrierLine-int lines, one per
                         // block group (blockIdx mod 8), then the groups' counter, then the release word;
                         // then 8 lines of evalCount(P)
  // devStat: [0] node tests, [1] sdf queries, [2] contacts (this step);
  //          [3] pairs, [4] node tests, [5] sdf queries, [6] contacts, [8] cluster entries
  //          (summed while profiling); [9] audits, [10] audited contacts, [11] missed contacts
  //          (cumulative); [12] master nodes of the candidate pairs, [13] evaluated pairs,
  //          [14] rebuild steps (summed while profiling)
  unsigned long long* devStat;
  unsigned long long* statSlots;  // 5 families x kStatSlots spread accumulators of the narrow phase,
                                  // kStatStride words apart

  // ---- learned culling surrogate ----
  SurNet sur;              // network (valid when surSlot != nullptr)
  const int* surSlot;      // family slot of each shape id, -1 outside the family; nullptr: untrained
  float surBand;           // cull band, unscaled SDF units (2 x measured max error)
  const int* nodeCluster;  // per shape node (caller order, at the shape's node offset): its cluster
  unsigned long long* surMask;  // per evaluated pair (list position): bit c = 0 when the network
                                // culls cluster c
  float* surSlack;              // per evaluated pair: smallest slack of the clusters it culled
  uint2* hitMask;               // per particle: which of its pairs as master (x) and of its reactions (y)
                                // hold contacts this step (hitBit), set by the narrow phase, cleared by
                                // the sums that read it
  unsigned char* forceSet;      // per particle: 0 when its stored force and torque are exactly zero
};

// Word g * kBarrierLine: map records the pair check's block group g (blockIdx mod 8) wrote this step, in its own
// region of pairMap.
__device__ inline int* evalCount(const Params& P) { return P.barrier + 10 * kBarrierLine; }

// What opens a step besides the bodies: the table of tangential history this step fills, its slot
// list from two steps ago, the step's buffer (flag set, clear count) and the host's rebuild request.
struct StepHead {
  unsigned long long* hashKey;
  const int* hashSlot;
  int buf;
  int forceRebuild;
};

// Error flags in devInt[3].  Any of them halts the call: every kernel launched after the flag is up
// returns at once (the gated broad-phase launches find their gate cleared), so the host can restore
// the state of the call's start, grow the buffers and run the call again.
constexpr int kErrPairs = 1;      // candidate pairs beyond pairCap
constexpr int kErrContacts = 2;   // candidate slots beyond contactCap
constexpr int kErrBarrier = 4;    // a grid barrier of the single-launch broad phase gave up waiting
constexpr int kErrHash = 8;       // a history table probe found no free slot
constexpr int kErrStepIdx = 20;   // devInt index of the failing step

// Copy of the state at the start of an lsdem_step call, so that a call that halted on an error can
// be run again from there (after the buffers grew): the bodies' state, the walls' poses, the bonds'
// flags and the contact slots of the step before the call (their springs are the next step's
// history; the table that finds them is rebuilt from the slots).
struct SnapDev {
  d3 *pos, *vel, *ang, *force, *torque, *wpos;
  q4 *quat, *wquat;
  int* bActive;
  unsigned char* forceSet;
  unsigned long long* devStat;  // kDevStats counters
  int* meta;                    // [0] history slots kept
  int* hNode;                   // history slots: node, info, spring
  uint32_t* hInfo;
  d3* hSpring;
  long long hCap;
  // the live contact buffer of the step before the call (1 - cur at the call's start)
  int* prevNode;
  uint32_t* prevInfo;
  d3* prevSpring;
  int prevBuf;
};

constexpr int kStatSlots = 32;
// bodies up to which the drift after a step closes the step's counters with a wavefront (k_reduce_drift_small)
constexpr int kWaveEndBodies = 65536;
// u64 words per stat slot: each slot has a 128-byte line of its own, since atomics on one line are
// served one after another (~10 ns each), whatever words of the line they touch
constexpr int kStatStride = 16;
constexpr int kStatWords = 5 * kStatSlots * kStatStride;
constexpr int kDevInts = 32;   // devInt entries
constexpr int kBarrierInts = 18 * kBarrierLine;   // 8 groups, the groups' counter, the release word, evalCount
// The step's rebuild flag and its count of ghost images left at their source's position, two sets
// used in alternate steps (buffer = Params::curBuf): the kernel that closes one step may already
// raise the next step's.
__host__ __device__ inline int rebuildFlagIdx(int buf) { return 16 + buf; }
__host__ __device__ inline int ghostCountIdx(int buf) { return 18 + buf; }
constexpr int kDevStats = 16;  // devStat entries
constexpr int kPairSlabHost = 32;        // candidate pairs of a master kept by the search (kPairSlab in the kernels)
constexpr int kBroadThreadsHost = 1024;  // block of the single-launch broad phase (kBroadThreads)
constexpr int kHaltedIdx = 23;           // devInt: error flags that a launch found up, for the launch after it
constexpr int kBigCellsIdx = 21, kBigRcIdx = 22;  // devInt: a rebuild has cells (reaction lists) of many items
constexpr uint32_t kInvalidInfo = 0xFFFFFFFFu;  // unused contact slot

}  // namespace lsd
