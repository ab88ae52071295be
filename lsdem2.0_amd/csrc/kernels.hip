// HIP kernels of the LS-DEM timestep for gfx950 (CDNA4, wave64).
//
// Per step (launch order, one stream):
//   k_kick_drift      half-kick, drift, reference-grid key, search cell, periodic wrap + ghost images,
//                     per-body motion record for the rebuild test and the separation certificates
//   k_broad_phase     on rebuild steps only (else it returns at once): counting sort of particles and
//                     ghost images by search-grid cell, FP32 bounding-sphere / grid-box candidate pairs,
//                     pair list in master order and the reaction CSR, phases joined by grid barriers
//                     (the same phases also run as separate gated launches)
//   k_pair_check      per candidate pair: partner this step, separation certificate against the motion
//                     since it was issued; the pairs to evaluate are compacted
//   k_candidates      one wavefront per batch of evaluated pairs: FP32 cluster cull and node prefilter
//                     (conservative), survivors written to a contiguous range per pair, then the exact
//                     FP64 node-vs-SDF test, tangential history and linear spring-dashpot per survivor
//   k_bonds           parallel bonds
//   k_reduce_kick     per-body segmented sum of contact and bond contributions + second half-kick
#include "device.h"
#include "launch_rules.h"
#include "surrogate.h"

namespace lsd {

// ------------------------------------------------------------------------------------------
// Reference grid (spatialGrid) and search grid helpers
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ i3 refCell(const GridGeom& G, d3 p) {
  return i3{int((p.x - G.mn.x) * G.inv.x), int((p.y - G.mn.y) * G.inv.y), int((p.z - G.mn.z) * G.inv.z)};
}
__device__ __forceinline__ int refKey(const GridGeom& G, d3 p) {
  if (p.x < G.mn.x) return -1; else if (p.x >= G.mx.x) return -1;
  if (p.y < G.mn.y) return -1; else if (p.y >= G.mx.y) return -1;
  if (p.z < G.mn.z) return -1; else if (p.z >= G.mx.z) return -1;
  return lin3(refCell(G, p), G.size);
}
// Squared distance from p to the reference domain box (0 inside).
__device__ __forceinline__ double domainDist2(const GridGeom& G, d3 p) {
  const double dx = fmax(0.0, fmax(G.mn.x - p.x, p.x - G.mx.x));
  const double dy = fmax(0.0, fmax(G.mn.y - p.y, p.y - G.mx.y));
  const double dz = fmax(0.0, fmax(G.mn.z - p.z, p.z - G.mx.z));
  return dx * dx + dy * dy + dz * dz;
}
// Ghost-image eligibility of a source at post-wrap position p, widened by hs (half the skin) so
// that it holds for every position within hs of p.  Set s: 0 = +x, 1 = +y, 2 = +x+y.
__device__ __forceinline__ bool potInColumn(const GridGeom& G, d3 p, int s, double hs) {
  const bool cx = (p.x - G.mn.x) * G.inv.x < 1.0 + hs * G.inv.x + 1e-9;
  const bool cy = (p.y - G.mn.y) * G.inv.y < 1.0 + hs * G.inv.y + 1e-9;
  return s == 0 ? cx : (s == 1 ? cy : (cx && cy));
}
__device__ __forceinline__ bool potOutColumn(const GridGeom& G, d3 p, int s, double hs) {
  const bool nx = (p.x - G.mn.x) * G.inv.x >= 1.0 - hs * G.inv.x - 1e-9;
  const bool ny = (p.y - G.mn.y) * G.inv.y >= 1.0 - hs * G.inv.y - 1e-9;
  return s == 0 ? nx : (s == 1 ? ny : (nx || ny));
}
// Can the image key of an unshifted image be valid (the source outside the ghost domain)?
__device__ __forceinline__ bool potOutOfDomain(const Params& P, d3 p, double hs) {
  const GridGeom& G = P.gridP;
  const double zmax = (P.quirks & 2) ? G.mx.y : G.mx.z;
  bool out = p.z < G.mn.z + hs || p.z >= zmax - hs;
  if (!P.periodicX) out = out || p.x < G.mn.x + hs || p.x >= G.mx.x - hs;
  if (!P.periodicY) out = out || p.y < G.mn.y + hs || p.y >= G.mx.y - hs;
  return out;
}

// Clamped cell and +-1 window of a node (the reference's 27-cell traversal bounds).
__device__ __forceinline__ void refWindow(const GridGeom& G, d3 p, i3& c, i3& lo, i3& hi) {
  c = refCell(G, p);
  lo = i3{-1, -1, -1};
  hi = i3{1, 1, 1};
  if (c.x <= 0) { c.x = 0; lo.x = 0; }
  if (c.x >= G.size.x - 1) { c.x = G.size.x - 1; hi.x = 0; }
  if (c.y <= 0) { c.y = 0; lo.y = 0; }
  if (c.y >= G.size.y - 1) { c.y = G.size.y - 1; hi.y = 0; }
  if (c.z <= 0) { c.z = 0; lo.z = 0; }
  if (c.z >= G.size.z - 1) { c.z = G.size.z - 1; hi.z = 0; }
}
__device__ __forceinline__ bool keyInWindow(const GridGeom& G, int key, d3 p) {
  i3 c, lo, hi;
  refWindow(G, p, c, lo, hi);
  const int kx = key % G.size.x, ky = (key / G.size.x) % G.size.y, kz = key / (G.size.x * G.size.y);
  return kx >= c.x + lo.x && kx <= c.x + hi.x && ky >= c.y + lo.y && ky <= c.y + hi.y &&
         kz >= c.z + lo.z && kz <= c.z + hi.z;
}
__device__ __forceinline__ int clampCell(double v, int n) {
  v = fmin(fmax(v, 0.0), double(n - 1));
  return int(v);
}
__device__ __forceinline__ i3 searchCell(const SearchGrid& S, d3 p) {
  return i3{clampCell(floor((p.x - S.mn.x) * S.invCell), S.size.x),
            clampCell(floor((p.y - S.mn.y) * S.invCell), S.size.y),
            clampCell(floor((p.z - S.mn.z) * S.invCell), S.size.z)};
}
__device__ __forceinline__ int ghostKey(const Params& P, d3 p) {
  const GridGeom& G = P.gridP;
  i3 c = refCell(G, p);
  bool out = false;
  if (p.x < G.mn.x) { c.x = 0; out = true; }
  else if (p.x >= G.mx.x) { c.x = G.size.x - 1; out = true; }
  if (p.y < G.mn.y) { c.y = 0; out = true; }
  else if (p.y >= G.mx.y) { c.y = G.size.y - 1; out = true; }
  const double zmax = (P.quirks & 2) ? G.mx.y : G.mx.z;
  if (p.z < G.mn.z) { c.z = 0; out = true; }
  else if (p.z >= zmax) { c.z = G.size.z - 1; out = true; }
  return out ? lin3(c, G.size) : -1;
}

// ------------------------------------------------------------------------------------------
// Small utilities
// ------------------------------------------------------------------------------------------
// Broad-phase kernels run only on steps that rebuild the candidate pairs: `gate` points at the
// step's rebuild flag (nullptr = always run).
#define LSD_GATE(g) \
  if ((g) != nullptr && *(g) == 0) return

// Raise error flag `bit` (kErr*): the call halts (every later kernel returns at entry); the index of the
// failing step is kept for the host.
__device__ __forceinline__ void raiseFlag(const Params& P, int bit) {
  atomicOr(&P.devInt[3], bit);
  atomicMax(&P.devInt[kErrStepIdx], P.callStep);
}
// The rebuild gates of both step buffers are cleared with it so that gated broad-phase launches skip as well.
// (Not by the single-launch broad phase, whose blocks read their gate while others may raise.)
__device__ __forceinline__ void dropGates(const Params& P) {
  atomicExch(&P.devInt[rebuildFlagIdx(0)], 0);
  atomicExch(&P.devInt[rebuildFlagIdx(1)], 0);
}
__device__ __forceinline__ void raiseError(const Params& P, int bit) {
  raiseFlag(P, bit);
  dropGates(P);
}
// Touches every 64-byte line of the kernel's Params (its first argument) at once.  The block is 1.6 KB and
// more than the scalar registers hold, so the compiler reads members where it needs them; each first touch
// of a line was a cold miss of the scalar cache in the middle of a dependent chain, several in a row.  One
// round of misses here and the later reads hit: 1 to 1.5 us less per kernel (a falling column of 20,000:
// 63.1 -> 60.6 us per step, 1,000 bodies in a box 73.5 -> 70.6).  All loads are waited for inside the block;
// their target is not used.
constexpr int kArgLines = (int(sizeof(Params)) + 63) / 64;
// Returns `v`, which ties the block to a use: it is no volatile asm, which the compiler would take for a
// write to memory, and read uniform values with vector loads from there on.
__device__ __forceinline__ int prefetchArgs(int v) {
  auto* a = __builtin_amdgcn_kernarg_segment_ptr();
  int unused;
#define LSD_LINE(n) "s_load_dword %1, %2, " #n "*64\n\t"
  static_assert(kArgLines == 25, "prefetchArgs touches the lines of the argument block and no others");
  asm(LSD_LINE(0) LSD_LINE(1) LSD_LINE(2) LSD_LINE(3) LSD_LINE(4) LSD_LINE(5) LSD_LINE(6) LSD_LINE(7)
      LSD_LINE(8) LSD_LINE(9) LSD_LINE(10) LSD_LINE(11) LSD_LINE(12) LSD_LINE(13) LSD_LINE(14)
      LSD_LINE(15) LSD_LINE(16) LSD_LINE(17) LSD_LINE(18) LSD_LINE(19) LSD_LINE(20) LSD_LINE(21)
      LSD_LINE(22) LSD_LINE(23) LSD_LINE(24) "s_waitcnt lgkmcnt(0)"
      : "+s"(v), "=&s"(unused) : "s"(a));
#undef LSD_LINE
  return v;
}
// v, as a value of turn `turn` of a loop (of item `item`): what is computed from it is worked out there, and not kept
// in registers from before.  (No volatile asm, as for prefetchArgs.)
__device__ __forceinline__ int inLoop(int v, int turn) {
  asm("" : "+v"(v) : "s"(turn));
  return v;
}
__device__ __forceinline__ int uniformInItem(int v, int item) {
  asm("" : "+s"(v) : "v"(item));
  return v;
}
__device__ __forceinline__ double inItem(double v, int item) {
  asm("" : "+v"(v) : "v"(item));
  return v;
}
// An error flag is up: this kernel has nothing to do.  Each wavefront reads the flag for itself, which is
// enough for a kernel that raises none: the flag then stays as it was when the launch began.
#define LSD_HALT(P) \
  if ((P).devInt[prefetchArgs(3)] != 0) return
// The same in a kernel that is followed by one which raises flags while its blocks meet at barriers: that a flag was
// up when this launch began is kept for that one ...
#define LSD_HALT_LATCH(P)                                                              \
  if (const int halted = (P).devInt[prefetchArgs(3)]) {                                \
    if (blockIdx.x == 0 && threadIdx.x == 0) (P).devInt[kHaltedIdx] = halted;          \
    return;                                                                            \
  }
// ... which reads it in the flag's place.  A flag that another block raises while this one starts must not send
// some of its wavefronts home and the rest on to the barriers: what the missing ones were to leave in LDS, a
// reservation's first slot among it, would be garbage.  (One wavefront's read of the flag for its block, behind a
// barrier, costs 2.5 to 3 us a step: 1,000 bodies in a box 9.94 -> 10.50 ms for 200.)
#define LSD_HALT_LATCHED(P) \
  if ((P).devInt[prefetchArgs(kHaltedIdx)] != 0) return

__global__ void k_fill_int(int* a, long long n, int v, const int* gate) {
  LSD_GATE(gate);
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    a[i] = v;
}
__global__ void k_fill_u64(unsigned long long* a, long long n, unsigned long long v) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    a[i] = v;
}

// Exclusive scan of n ints (n + 1 outputs, out[n] = total) in two phases over tiles.
constexpr int kScanThreads = 256;   // block of the separate scan launches
constexpr int kScanLds = 1024 / 64 + 1;  // LDS ints of blockExclusiveScan (blocks of up to 1024)
constexpr int kScanItems = 8;

__device__ __forceinline__ int blockExclusiveScan(int v, int* lds, int& total) {
  // any block size that is a multiple of 64 up to 1024; lds needs kScanLds ints
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    int t = __shfl_up(incl, o, 64);
    if (lane >= o) incl += t;
  }
  if (lane == 63) lds[wid] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int w = 0; w < int(blockDim.x >> 6); ++w) {
      int t = lds[w];
      lds[w] = acc;
      acc += t;
    }
    lds[blockDim.x >> 6] = acc;
  }
  __syncthreads();
  total = lds[blockDim.x >> 6];
  int r = lds[wid] + incl - v;
  __syncthreads();
  return r;
}

// Grid-stride loop bounds of one phase: this thread's index and the number of threads.
struct Span {
  int tid, nth;
};
__device__ __forceinline__ Span gridSpan() {
  return Span{int(blockIdx.x * blockDim.x + threadIdx.x), int(gridDim.x * blockDim.x)};
}
// Phase 1 of the scan: the sum of each tile of blockDim.x x kScanItems inputs (blocks loop over
// tiles).
__device__ void scanReduceTiles(const int* in, long long n, int* tileSum, int* lds) {
  const long long tile = (long long)blockDim.x * kScanItems;
  const long long nTiles = (n + tile - 1) / tile;
  for (long long t = blockIdx.x; t < nTiles; t += gridDim.x) {
    const long long base = t * tile + (long long)threadIdx.x * kScanItems;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
      if (base + k < n) s += in[base + k];
    int total;
    blockExclusiveScan(s, lds, total);
    if (threadIdx.x == 0) tileSum[t] = total;
  }
}
// Phase 2: each tile adds the sums of the tiles before it and writes its exclusive prefix; the
// last tile writes the total to out[n].  n == 0 writes out[0] = 0.
// bigFlag (may be null): set to 1 when an input is above kSmallBucket.
constexpr int kSmallBucket = 16;  // items of a bucket that bucketSortSmall sorts
__device__ void scanApplyTiles(const int* in, long long n, const int* tileSum, int* out, int* lds,
                               int* bigFlag = nullptr) {
  const long long tile = (long long)blockDim.x * kScanItems;
  const long long nTiles = (n + tile - 1) / tile;
  if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
  for (long long t = blockIdx.x; t < nTiles; t += gridDim.x) {
    int pre = 0;
    for (long long u = threadIdx.x; u < t; u += blockDim.x) pre += tileSum[u];
    int preTotal;
    blockExclusiveScan(pre, lds, preTotal);
    const long long base = t * tile + (long long)threadIdx.x * kScanItems;
    int v[kScanItems];
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      v[k] = (base + k < n) ? in[base + k] : 0;
      s += v[k];
      if (bigFlag && v[k] > kSmallBucket) *bigFlag = 1;
    }
    int total;
    int ex = blockExclusiveScan(s, lds, total) + preTotal;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      if (base + k < n) out[base + k] = ex;
      ex += v[k];
    }
    if (t == nTiles - 1 && threadIdx.x == 0) out[n] = preTotal + total;
  }
}
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const int* in, long long n, int* tileSum,
                                                               const int* gate) {
  LSD_GATE(gate);
  __shared__ int lds[kScanLds];
  scanReduceTiles(in, n, tileSum, lds);
}
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(const int* in, long long n, const int* tileSum, int* out,
                                                              const int* gate) {
  LSD_GATE(gate);
  __shared__ int lds[kScanLds];
  scanApplyTiles(in, n, tileSum, out, lds);
}

// ------------------------------------------------------------------------------------------
// Integration: first half-kick + drift (+ keys, wrap, ghost images)
// ------------------------------------------------------------------------------------------
// Chord 2 sin(angle / 2) of the rotation from unit quaternion b to unit quaternion q: the largest
// displacement of a unit vector between the two orientations (|R(q) - R(b)| in the 2-norm).
__device__ __forceinline__ double relChord(q4 b, q4 q) {
  const double vx = b.q0 * q.q1 - q.q0 * b.q1 - (b.q2 * q.q3 - b.q3 * q.q2);
  const double vy = b.q0 * q.q2 - q.q0 * b.q2 - (b.q3 * q.q1 - b.q1 * q.q3);
  const double vz = b.q0 * q.q3 - q.q0 * b.q3 - (b.q1 * q.q2 - b.q2 * q.q1);
  return 2.0 * sqrt(vx * vx + vy * vy + vz * vz);
}

// conj(b) q in FP32: the rotation from b to q as a quaternion.
__device__ __forceinline__ float4 relQuat(q4 b, q4 q) {
  const double w = b.q0 * q.q0 + b.q1 * q.q1 + b.q2 * q.q2 + b.q3 * q.q3;
  const double vx = b.q0 * q.q1 - q.q0 * b.q1 - (b.q2 * q.q3 - b.q3 * q.q2);
  const double vy = b.q0 * q.q2 - q.q0 * b.q2 - (b.q3 * q.q1 - b.q1 * q.q3);
  const double vz = b.q0 * q.q3 - q.q0 * b.q3 - (b.q1 * q.q2 - b.q2 * q.q1);
  return make_float4(float(w), float(vx), float(vy), float(vz));
}
// Chord between the rotations of two FP32 quaternions (as relChord), plus an allowance for their
// FP32 rounding.
__device__ __forceinline__ float relChordF(float4 b, float4 q) {
  const float vx = b.x * q.y - q.x * b.y - (b.z * q.w - b.w * q.z);
  const float vy = b.x * q.z - q.x * b.z - (b.w * q.y - b.y * q.w);
  const float vz = b.x * q.w - q.x * b.w - (b.y * q.z - b.z * q.y);
  return 2.f * sqrtf(vx * vx + vy * vy + vz * vz) * (1.f + 1e-5f) + 1e-6f;
}

// Which ghost images of a particle at (wrapped) position p lie a period away from it: bit 0 the
// +x image (first reference-grid column), bit 1 the +y image, bit 2 the corner image.
// (SEC: quarter-sector periodicity, known at compile time in the per-step kernels)
template <bool SEC>
__device__ __forceinline__ int imgShiftMask(const Params& P, d3 p) {
  const i3 c = refCell(P.gridP, p);
  if (SEC)  // turned images: +90 (first y cell), 180 (first x and y cells), -90 (first x cell)
    return (c.y == 0 ? 1 : 0) | (c.x == 0 && c.y == 0 ? 2 : 0) | (c.x == 0 ? 4 : 0);
  return (c.x == 0 ? 1 : 0) | (c.y == 0 ? 2 : 0) | (c.x == 0 && c.y == 0 ? 4 : 0);
}
// Lanes of the wavefront below this one.
__device__ __forceinline__ unsigned long long laneLtMask() {
  const int lane = int(__lane_id());
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Members of Params chosen by an image set known only at run time, read through selects: indexing
// a by-value kernel argument with a run-time index makes the compiler copy the whole argument block
// into per-lane scratch memory.
template <class T>
__device__ __forceinline__ T pick3(int s, T a, T b, T c) { return s == 0 ? a : (s == 1 ? b : c); }

// (an image position array indexed directly compiles to one load of the pointer when no other
// member is indexed at run time: the per-step kernels without sector periodicity keep that form)
template <bool SEC>
__device__ __forceinline__ d3* imgPos(const Params& P, int s) {
  return SEC ? pick3(s, P.gpos[0], P.gpos[1], P.gpos[2]) : P.gpos[s];
}
__device__ __forceinline__ q4* imgQuat(const Params& P, int s) { return pick3(s, P.gquat[0], P.gquat[1], P.gquat[2]); }
__device__ __forceinline__ d3* imgVel(const Params& P, int s) { return pick3(s, P.gvel[0], P.gvel[1], P.gvel[2]); }
// v turned by the rotation of sector image set s (about the z axis through the origin)
__device__ __forceinline__ d3 secTurn(const Params& P, int s, d3 v) {
  return rodrigues(v, pick3(s, P.secW[0], P.secW[1], P.secW[2]), pick3(s, P.secA[0], P.secA[1], P.secA[2]),
                   pick3(s, P.secB[0], P.secB[1], P.secB[2]));
}
// The same, with the set's constants read by their index from the argument block (Params is its first member): picked
// from all three sets they take the registers of all three.  For kernels, not for functions that are called.
__device__ __forceinline__ d3 secTurnByIndex(int s, d3 v) {
  const auto* a = (const __attribute__((address_space(4))) Params*)__builtin_amdgcn_kernarg_segment_ptr();
  return rodrigues(v, mk3(a->secW[s].x, a->secW[s].y, a->secW[s].z), a->secA[s], a->secB[s]);
}
__device__ __forceinline__ q4 secQuat(const Params& P, int s) { return pick3(s, P.secR[0], P.secR[1], P.secR[2]); }

// Column predicate (potInColumn / potOutColumn set) of image set s: with sector periodicity the sets
// turned by +90, 180 and -90 degrees take the sources of the first y cell, of the corner and of the
// first x cell.
template <bool SEC>
__device__ __forceinline__ int imageColumn(int s) { return SEC ? (s == 0 ? 1 : (s == 1 ? 2 : 0)) : s; }
// A body that left the quarter sector across x = min (y = min) turns by -90 (+90) degrees about the
// z axis through the corner: position, velocity and orientation (updateVelocityPositionOrientation-
// OutOfSectorKernel, mySpatialGrid.cu:58-85).  Returns whether it turned.
__device__ __forceinline__ bool sectorWrap(const Params& P, d3& p, d3& v, q4& q) {
  const d3 mn = P.gridP.mn;
  bool turned = false;
  if (p.x < mn.x && p.y >= mn.y) {
    v = rodrigues(v, P.secW[2], P.secA[2], P.secB[2]);
    p = mn + rodrigues(p - mn, P.secW[2], P.secA[2], P.secB[2]);
    q = qrotate(P.secR[2], q);
    turned = true;
  }
  if (p.y < mn.y && p.x >= mn.x) {
    v = rodrigues(v, P.secW[0], P.secA[0], P.secB[0]);
    p = mn + rodrigues(p - mn, P.secW[0], P.secA[0], P.secB[0]);
    q = qrotate(P.secR[0], q);
    turned = true;
  }
  return turned;
}

__device__ __forceinline__ void halfKick(const Params& P, int i, d3 F, d3 T) {
  const double invM = P.invM[i];
  if (isZero(invM)) return;
  const double h = 0.5 * P.dt;
  P.vel[i] += (F * invM + P.g) * h;
  P.angvel[i] += (mul(rotInvInertia(P.quat[i], P.invI[i]), T)) * h;
}

__device__ void wallDrift(const Params& P, int w, int buf);

// Thread 0 clears the step's counters and raises the host's rebuild request; all threads empty the
// entries of the history table this step fills (left there two steps ago; their slots were
// recorded at insertion).
__device__ __forceinline__ void stepHead(const Params& P, const StepHead& H, int i, int nth) {
  if (i == 0) {
    if (H.forceRebuild) atomicOr(&P.devInt[rebuildFlagIdx(H.buf)], 1);
    P.devInt[1] = 0;   // contact slots allocated
  }
  if (i < 8) evalCount(P)[i * kBarrierLine] = 0;  // map records of the pair check's block groups
  const int nClear = P.devInt[10 + H.buf];
  for (int c = i; c < nClear; c += nth) {
    const int slot = H.hashSlot[c];
    if (slot >= 0) H.hashKey[slot] = kHashEmpty;
  }
}

// Half-kick(s) with (F, T), drift, reference-grid key, search cell, periodic wrap and ghost images,
// the rebuild test and the motion record of particle i.  kicks = 2 applies the previous step's
// second half-kick and this step's first, the same increment twice (the force of a step is used by
// both), exactly as two separate half-kicks round.
// Everything the kick and drift of particle i read, loaded before any of its stores (the stores
// could alias later loads as far as the compiler knows, which would serialise the round trips).
// (the inverse inertia is read by kickDrift only for a body with a torque)
struct BodyIn {
  d3 vel, w, pos, xBuild, xBuildW;
  q4 quat, qBuild;
  double invM;
  int imgBuild;
};
template <bool SEC>
__device__ __forceinline__ BodyIn loadBody(const Params& P, int i) {
  BodyIn b;
  b.vel = P.vel[i];
  b.w = P.angvel[i];
  b.quat = P.quat[i];
  b.invM = P.invM[i];
  b.pos = P.pos[i];
  b.xBuild = P.xBuild[i];
  b.xBuildW = P.xBuildW[i];
  b.qBuild = P.qBuild[i];
  b.imgBuild = (P.periodicX || P.periodicY || SEC) ? P.imgBuild[i] : 0;
  return b;
}
// SEC: quarter-sector periodicity (a compile-time switch, so that simulations without it run the code
// they ran before it existed)
template <bool SEC>
__device__ __forceinline__ void kickDrift(const Params& P, int i, const BodyIn& in, d3 F, d3 T, int kicks, int buf) {
  d3 vel = in.vel, w = in.w;
  const q4 q0 = in.quat;
  const double invM = in.invM;
  // a body without a torque keeps its angular velocity: R I^-1 R^T 0 adds only zeros, so neither its
  // inverse inertia (48 bytes) is read nor its angular velocity written back
  const bool torqued = T.x != 0.0 || T.y != 0.0 || T.z != 0.0;
  const s6 invI = torqued ? P.invI[i] : s6{};
  if (!isZero(invM) && !P.prime) {
    const double h = 0.5 * P.dt;
    const d3 dv = (F * invM + P.g) * h;
    vel += dv;
    if (kicks == 2) vel += dv;
    P.vel[i] = vel;
    if (torqued) {
      const d3 dw = (mul(rotInvInertia(q0, invI), T)) * h;
      w += dw;
      if (kicks == 2) w += dw;
      P.angvel[i] = w;
    }
  }
  d3 p = in.pos;
  q4 qn = q0;
  if (!P.prime) {  // (the pre-loop build detects at the current poses)
    p += P.dt * vel;
    qn = qintegrate(q0, w, P.dt);
    P.quat[i] = qn;
  }
  constexpr bool sector = SEC;
  const bool periodic = P.periodicX || P.periodicY || sector;
  const bool wrapAfter = (P.quirks & 4) != 0;
  const GridGeom& G = P.gridP;
  const d3 ox = mk3(G.mx.x - G.mn.x, 0., 0.), oy = mk3(0., G.mx.y - G.mn.y, 0.);
  bool turned = false;  // (sector periodicity: the body left the sector and turned this step)
  if (periodic && !wrapAfter) {
    if (P.periodicX) { if (p.x < G.mn.x) p += ox; else if (p.x >= G.mx.x) p -= ox; }
    if (P.periodicY) { if (p.y < G.mn.y) p += oy; else if (p.y >= G.mx.y) p -= oy; }
    if (sector) turned = sectorWrap(P, p, vel, qn);
  }
  P.posDet[i] = p;
  const d3 pDet = p;
  const q4 qDet = qn;  // orientation of particle-particle detection (before a turn after the build)
  if (sector) P.quatDet[i] = qn;
  const int keyRef = refKey(G, p);
  int gk[3] = {-1, -1, -1};  // image keys; an image's position is stored only when it exists
  int unshifted = 0;  // valid images at the particle's own position (particle outside the domain)
  if (periodic) {
    d3 img;
    if (P.periodicX) {
      if (wrapAfter) { if (p.x < G.mn.x) p += ox; else if (p.x >= G.mx.x) p -= ox; }
      img = p;
      if (refCell(G, p).x == 0) img += ox;
      const int k = ghostKey(P, img);
      if (k >= 0) P.gpos[0][i] = img;
      gk[0] = k;
      unshifted += (k >= 0 && refCell(G, p).x != 0);
    }
    if (P.periodicY) {
      if (wrapAfter) { if (p.y < G.mn.y) p += oy; else if (p.y >= G.mx.y) p -= oy; }
      img = p;
      if (refCell(G, p).y == 0) img += oy;
      const int k = ghostKey(P, img);
      if (k >= 0) P.gpos[1][i] = img;
      gk[1] = k;
      unshifted += (k >= 0 && refCell(G, p).y != 0);
    }
    if (P.periodicX && P.periodicY) {
      img = p;
      const i3 c = refCell(G, p);
      if (c.x == 0 && c.y == 0) img += ox + oy;
      const int k = ghostKey(P, img);
      if (k >= 0) P.gpos[2][i] = img;
      gk[2] = k;
      unshifted += (k >= 0 && !(c.x == 0 && c.y == 0));
    }
    if (sector) {
      // (mySpatialGrid.cu:154-212) images turned by +90 degrees for bodies in the first y cell, 180 for
      // those in the first x and y cells, -90 for those in the first x cell; other copies keep the pose
      if (wrapAfter) turned = sectorWrap(P, p, vel, qn) || turned;
      const i3 c = refCell(G, p);
      for (int s = 0; s < 3; ++s) {
        const bool on = s == 0 ? c.y == 0 : (s == 1 ? (c.x == 0 && c.y == 0) : c.x == 0);
        const d3 im = on ? G.mn + secTurn(P, s, p - G.mn) : p;
        const int k = ghostKey(P, im);
        if (k >= 0) {
          imgPos<SEC>(P, s)[i] = im;
          imgQuat(P, s)[i] = on ? qrotate(secQuat(P, s), qn) : qn;
          imgVel(P, s)[i] = on ? secTurn(P, s, vel) : vel;
        }
        gk[s] = k;
        unshifted += (k >= 0 && !on);
      }
    }
  }
  if (turned) {
    P.vel[i] = vel;
    P.quat[i] = qn;
  }
  P.pos[i] = p;
  // sources that may hold an unshifted image before the next rebuild
  if (periodic && P.halfSkin > 0.0) {
    unshifted = 0;
    if (potOutOfDomain(P, p, P.halfSkin))
      for (int s = 0; s < 3; ++s) unshifted += potOutColumn(G, p, imageColumn<SEC>(s), P.halfSkin);
  }
  if (unshifted) atomicAdd(&P.devInt[ghostCountIdx(buf)], unshifted);
  // rebuild the candidate pairs when a body has moved half the skin since the last build (a
  // periodic wrap always does, and a turn across a sector's face is one wherever it ends).  Sector images
  // are turned about the corner's axis, so they move as far as their sources and the skin covers them as it
  // covers shifted ones.  (Rebuilt every step, as sector periodicity once did: 4,000 bodies 0.22 ms a step
  // with the 32-lane search, 0.05 now.)
  const double hs2 = P.halfSkin * P.halfSkin;
  const d3 dd = pDet - in.xBuild, dw = p - in.xBuildW;
  const bool moved = turned || len2(dd) > hs2 || len2(dw) > hs2;
  if (__ballot(moved) && (threadIdx.x & 63) == __builtin_ctzll(__ballot(moved))) atomicOr(&P.devInt[rebuildFlagIdx(buf)], 1);
  // motion since the build for the separation certificates (a step that wraps rebuilds, so posDet
  // and pos move alike on every step that reads this)
  BodyStep st;
  const q4 qb = in.qBuild;
  st.motion = make_float4(float(dd.x), float(dd.y), float(dd.z), float(relChord(qb, qDet)));
  P.qrel[i] = relQuat(qb, qDet);
  st.key = make_int4(keyRef, -1, -1, -1);
  if (periodic) {
    const int flip = imgShiftMask<SEC>(P, p) ^ in.imgBuild;
    int* sk = &st.key.y;
    for (int g = 0; g < 3; ++g) sk[g] = gk[g] >= 0 ? (gk[g] | (((flip >> g) & 1) << kFlipBit)) : -1;
  }
  P.step[i] = st;
}

// One thread per particle, then one per wall.
template <bool SEC>
__global__ void k_kick_drift(Params P, int forceRebuild) {
  LSD_HALT_LATCH(P)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  BodyIn in;
  d3 F, T;
  if (i < P.nP) {
    in = loadBody<SEC>(P, i);
    F = P.force[i];
    T = P.torque[i];
  }
  stepHead(P, StepHead{P.hashKey, P.hashSlot, P.curBuf, forceRebuild}, i, int(gridDim.x * blockDim.x));
  if (i >= P.nP) {
    if (i - P.nP < P.nW) wallDrift(P, i - P.nP, P.curBuf);
    return;
  }
  kickDrift<SEC>(P, i, in, F, T, 1, P.curBuf);
}

__device__ void wallDrift(const Params& P, int w, int buf) {
  d3 p = P.wpos[w];
  q4 q = P.wquat[w];
  if (!P.prime) {
    p += P.dt * P.wvel[w];
    P.wpos[w] = p;
    q = qintegrate(q, P.wangvel[w], P.dt);
    P.wquat[w] = q;
  }
  P.wkey[w] = refKey(P.gridW, p);
  // displacement bound of any point of the wall's grid box since the last build: translation plus
  // 2 R sin(angle / 2) for the rotation
  const double chord = relChord(P.wBuildQ[w], q);
  const double R = P.shapes[P.wshape[w]].boxR;
  const d3 dp = p - P.wBuildPos[w];
  const double disp = len(dp) + R * chord;
  if (disp > P.halfSkin) atomicOr(&P.devInt[rebuildFlagIdx(buf)], 1);
  P.wMotion[w] = make_float4(float(dp.x), float(dp.y), float(dp.z), float(chord));
  P.wQrel[w] = relQuat(P.wBuildQ[w], q);
  P.wSph[w] = make_float4(float(p.x), float(p.y), float(p.z), float(R));
}

// Record the poses the candidate pairs were built from (rebuild steps only).
__device__ void markBuildOne(const Params& P, int i);
__device__ void markBuild(const Params& P, Span g) {
  for (int i = g.tid; i < max(P.nP, P.nW); i += g.nth) markBuildOne(P, i);
}
__device__ void markBuildOne(const Params& P, int i) {
  if (i < P.nP) {
    P.xBuild[i] = P.posDet[i];
    P.xBuildW[i] = P.pos[i];
    P.qBuild[i] = P.periodicSector ? P.quatDet[i] : P.quat[i];
    // (zero already, unless the last call halted on an error between the narrow phase and the sums: the bits
    // would then name pairs of another list)
    P.hitMask[i] = make_uint2(0u, 0u);
    BodyStep st = P.step[i];
    st.motion = make_float4(0.f, 0.f, 0.f, 0.f);
    P.qrel[i] = make_float4(1.f, 0.f, 0.f, 0.f);
    st.key.y = st.key.y >= 0 ? (st.key.y & ~(1 << kFlipBit)) : -1;
    st.key.z = st.key.z >= 0 ? (st.key.z & ~(1 << kFlipBit)) : -1;
    st.key.w = st.key.w >= 0 ? (st.key.w & ~(1 << kFlipBit)) : -1;
    P.step[i] = st;
    if (P.periodicX || P.periodicY || P.periodicSector)
      P.imgBuild[i] = P.periodicSector ? imgShiftMask<true>(P, P.pos[i]) : imgShiftMask<false>(P, P.pos[i]);
  }
  if (i < P.nW) {
    P.wBuildPos[i] = P.wpos[i];
    P.wBuildQ[i] = P.wquat[i];
    P.wMotion[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    P.wQrel[i] = make_float4(1.f, 0.f, 0.f, 0.f);
  }
}

// ------------------------------------------------------------------------------------------
// Deterministic counting sort by bucket: count (atomic rank) -> scan -> scatter -> per-bucket
// insertion sort by item index.
// ------------------------------------------------------------------------------------------
__device__ void bucketCount(const int* bucket, int n, int* count, int* rank, Span g) {
  for (int i = g.tid; i < n; i += g.nth) {
    const int b = bucket[i];
    rank[i] = b >= 0 ? atomicAdd(&count[b], 1) : -1;
  }
}
__device__ void bucketScatter(const int* bucket, int n, const int* start, const int* rank, int* out, Span g) {
  for (int i = g.tid; i < n; i += g.nth) {
    const int b = bucket[i];
    const int d = b >= 0 ? start[b] + rank[i] : -1;
    if (d >= 0 && d < n) out[d] = i;  // (always in range when the counts and the scan are complete)
  }
}
// Buckets of up to 16 items are sorted in registers (odd-even transposition network) from
// `tmp` into `items`; larger ones are listed for bucketSortBig (*bigCount starts at 0).
// inv (may be null): also records each item's place, inv[item] = position in items.
__device__ void bucketSortSmall(const int* start, int nb, const int* tmp, int* items, int* inv, int* bigList,
                                int* bigCount, Span g, int nItems) {
  for (int b = g.tid; b < nb; b += g.nth) {
    const int s = start[b], e = start[b + 1];
    const int n = e - s;
    if (n <= 0 || s < 0 || e > nItems) continue;  // (never with a complete scan of the counts)
    if (n == 1) {
      const int v0 = tmp[s];
      items[s] = v0;
      if (inv) inv[v0] = s;
      continue;
    }
    if (n > kSmallBucket) {
      const int q = atomicAdd(bigCount, 1);
      if (q < nb) bigList[q] = b;
      continue;
    }
    int v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = k < n ? tmp[s + k] : 0x7fffffff;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
#pragma unroll
      for (int k = (r & 1); k + 1 < 16; k += 2) {
        const int a = v[k], c = v[k + 1];
        v[k] = min(a, c);
        v[k + 1] = max(a, c);
      }
    }
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k < n) {
        items[s + k] = v[k];
        if (inv) inv[v[k]] = s + k;
      }
  }
}
// One wavefront per listed bucket: each item's place is the number of smaller items (items are
// distinct indices).
__device__ void bucketSortBig(const int* start, const int* tmp, int* items, int* inv, const int* bigList,
                              const int* bigCount, Span g, int nb, int nItems) {
  const int lane = threadIdx.x & 63, wave = g.tid >> 6, nWaves = g.nth >> 6;
  const int nBig = min(*bigCount, nb);
  for (int q = wave; q < nBig; q += nWaves) {
    const int b = bigList[q];
    const int s = start[b], e = start[b + 1];
    if (s < 0 || e > nItems || s >= e) continue;  // (never with a complete scan of the counts)
    for (int c0 = s; c0 < e; c0 += 64) {
      const int v = c0 + lane < e ? tmp[c0 + lane] : 0x7fffffff;
      int rank = 0;
      for (int c1 = s; c1 < e; c1 += 64) {
        const int u = c1 + lane < e ? tmp[c1 + lane] : 0x7fffffff;
        for (int k = 0; k < 64; ++k) rank += __shfl(u, k, 64) < v ? 1 : 0;
      }
      if (c0 + lane < e) {
        items[s + rank] = v;
        if (inv) inv[v] = s + rank;
      }
    }
  }
}
__global__ void k_bucket_count(const int* bucket, int n, int* count, int* rank, const int* gate) {
  LSD_GATE(gate);
  bucketCount(bucket, n, count, rank, gridSpan());
}
__global__ void k_bucket_scatter(const int* bucket, int n, const int* start, const int* rank, int* out,
                                 int* bigCount, const int* gate) {
  LSD_GATE(gate);
  if (blockIdx.x == 0 && threadIdx.x == 0) *bigCount = 0;  // list of large buckets of k_bucket_sort
  bucketScatter(bucket, n, start, rank, out, gridSpan());
}
__global__ void k_bucket_sort(const int* start, int nb, const int* tmp, int* items, int* inv, int* bigList,
                              int* bigCount, const int* gate, int nItems) {
  LSD_GATE(gate);
  bucketSortSmall(start, nb, tmp, items, inv, bigList, bigCount, gridSpan(), nItems);
}
__global__ void k_bucket_sort_big(const int* start, int nb, const int* tmp, int* items, int* inv, const int* bigList,
                                  const int* bigCount, const int* gate, int nItems) {
  LSD_GATE(gate);
  bucketSortBig(start, tmp, items, inv, bigList, bigCount, gridSpan(), nb, nItems);
}

__device__ __forceinline__ double triAt(const Params& P, const ShapeDev& S, double sc, d3 loc, d3 go, double invSp,
                                        bool& inside, double& cmax) {
  // trilinear SDF value at a local point (for pair-level culls), inside = within the grid box,
  // cmax = largest |corner| (bounds the rounding of the value)
  const double gx = (loc.x - go.x) * invSp, gy = (loc.y - go.y) * invSp, gz = (loc.z - go.z) * invSp;
  const int i0 = (int)floor(gx), j0 = (int)floor(gy), k0 = (int)floor(gz);
  inside = !(i0 < 0 || j0 < 0 || k0 < 0 || i0 >= S.nx - 1 || j0 >= S.ny - 1 || k0 >= S.nz - 1);
  if (!inside) return 0.0;
  const i3 n{S.nx, S.ny, S.nz};
  const float* g = P.sdf + S.sdfOff;
  double p[8];
  p[0] = double(g[lin3(i3{i0, j0, k0}, n)]) * sc;
  p[1] = double(g[lin3(i3{i0 + 1, j0, k0}, n)]) * sc;
  p[2] = double(g[lin3(i3{i0, j0 + 1, k0}, n)]) * sc;
  p[3] = double(g[lin3(i3{i0 + 1, j0 + 1, k0}, n)]) * sc;
  p[4] = double(g[lin3(i3{i0, j0, k0 + 1}, n)]) * sc;
  p[5] = double(g[lin3(i3{i0 + 1, j0, k0 + 1}, n)]) * sc;
  p[6] = double(g[lin3(i3{i0, j0 + 1, k0 + 1}, n)]) * sc;
  p[7] = double(g[lin3(i3{i0 + 1, j0 + 1, k0 + 1}, n)]) * sc;
  cmax = 0.0;
  for (int c = 0; c < 8; ++c) cmax = fmax(cmax, fabs(p[c]));
  return triValue(gx - double(i0), gy - double(j0), gz - double(k0), p);
}

// Distance from a point to the grid box [o, o + (n-1) h] (all in the same local frame).
__device__ __forceinline__ double boxDist2(d3 loc, d3 o, double h, const ShapeDev& S) {
  const double ex = (S.nx - 1) * h, ey = (S.ny - 1) * h, ez = (S.nz - 1) * h;
  const double dx = fmax(0.0, fmax(o.x - loc.x, loc.x - (o.x + ex)));
  const double dy = fmax(0.0, fmax(o.y - loc.y, loc.y - (o.y + ey)));
  const double dz = fmax(0.0, fmax(o.z - loc.z, loc.z - (o.z + ez)));
  return dx * dx + dy * dy + dz * dz;
}

// Which walls particle A can reach before the next rebuild: sphere vs grid box, then a Lipschitz bound on
// the wall SDF at the centre.  Every point of a wall's grid box lies within boxR of the wall's origin: walls
// far away (the other drums of an ensemble) are dropped on an FP32 sphere test (its margin covers the FP32
// roundings of the centres, of boxR and of the test) before the shape record is read and the centre turned
// into the wall's frame.
// Up to kMaskWalls walls, one thread per particle tests them all (64 particles in a wavefront: six walls of a
// box have few lanes' work); beyond that the lanes of a particle's search take a wall each.
constexpr int kMaskWalls = 64;
struct WallReach {
  d3 xA;
  double rs, rr;
  float fx, fy, fz, fr, mA;
  __device__ __forceinline__ WallReach(const Params& P, int A) {
    xA = P.posDet[A];
    rs = P.radius[A] + 2.0 * inItem(P.halfSkin, A);  // the wall and the particle each move < half the skin
    rr = rs * (1.0 + 1e-9) + 1e-12;
    fx = float(xA.x); fy = float(xA.y); fz = float(xA.z);
    fr = float(rr);
    mA = fmaxf(fmaxf(fabsf(fx), fabsf(fy)), fabsf(fz));
  }
  __device__ __forceinline__ bool reaches(const Params& P, int w) const {
    const float4 sw = P.wSph[w];
    const float dx = fx - sw.x, dy = fy - sw.y, dz = fz - sw.z;
    const float ms = fmaxf(fmaxf(fabsf(sw.x), fabsf(sw.y)), fabsf(sw.z));
    const float reach = (sw.w + fr) * (1.f + 1e-5f) + 1e-6f * (mA + ms) + 1e-30f;
    if (dx * dx + dy * dy + dz * dz > reach * reach * (1.f + 1e-5f)) return false;
    const d3 dw = xA - P.wpos[w];
    const ShapeDev S = P.shapes[P.wshape[w]];
    const d3 loc = rotInv(dw, P.wquat[w]);
    const d3 o = mk3(S.ox, S.oy, S.oz);
    if (boxDist2(loc, o, S.h, S) > rr * rr) return false;
    bool inside;
    double cmax;
    const double phi = triAt(P, S, 1.0, loc, o, 1. / S.h, inside, cmax);
    return !(inside && phi > S.lip * rs * (1.0 + 1e-6) + 1e-9 * S.h + 1e-12 * cmax);
  }
};

// Search-grid cell of a particle's post-wrap centre: ghost images are searched through their
// sources, and a particle that wrapped this step is outside the domain before the wrap (never a pp
// partner).
__device__ __forceinline__ int searchCellOf(const Params& P, int i) {
  return lin3(searchCell(P.sg, P.pos[i]), P.sg.size);
}

// Gather particle (or ghost-image) data into the sorted order of the search-grid table so
// that the candidate loops stream contiguous memory, and, where there are few walls, the walls each
// particle can reach.
__device__ void gatherParticle(const Params& P, int k) {
  const int i = P.sorted[k];
  const d3 x = P.posDet[i], w = P.pos[i];
  const float r = float(P.radius[i]);
  // a pp partner must be inside the domain when the pair is used; one that can get there before
  // the next rebuild (within half the skin) stays a candidate
  const bool eligible = P.step[i].key.x >= 0 || domainDist2(P.gridP, x) <= P.halfSkin * P.halfSkin;
  P.sPR[k] = make_float4(float(x.x), float(x.y), float(x.z), eligible ? r : -1.f);
  P.sPRw[k] = make_float4(float(w.x), float(w.y), float(w.z), r);
  P.sBoxR[k] = float(P.scale[i] * P.shapes[P.shape[i]].boxR);
  if (P.nW > 0 && P.nW <= kMaskWalls) {
    const WallReach R(P, i);
    unsigned long long m = 0;
    for (int wl = 0; wl < P.nW; ++wl) m |= (unsigned long long)(R.reaches(P, wl) ? 1 : 0) << wl;
    P.wallMask[k] = m;
  }
}
__global__ void k_search_cells(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  const Span g = gridSpan();
  for (int i = g.tid; i < P.nP; i += g.nth) P.scell[i] = searchCellOf(P, i);
}
__global__ void k_gather_particles(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  const Span g = gridSpan();
  for (int k = g.tid; k < P.nP; k += g.nth) gatherParticle(P, k);
}

// ------------------------------------------------------------------------------------------
// Candidate pairs
// ------------------------------------------------------------------------------------------
// Squared distance from x to the search grid's box (0 inside).
__device__ __forceinline__ double searchBoxDist2(const SearchGrid& S, d3 x) {
  const double ex = S.size.x * S.cell, ey = S.size.y * S.cell, ez = S.size.z * S.cell;
  const double dx = fmax(0.0, fmax(S.mn.x - x.x, x.x - (S.mn.x + ex)));
  const double dy = fmax(0.0, fmax(S.mn.y - x.y, x.y - (S.mn.y + ey)));
  const double dz = fmax(0.0, fmax(S.mn.z - x.z, x.z - (S.mn.z + ez)));
  return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ int clampCellF(float v, int n) { return int(fminf(fmaxf(v, 0.f), float(n - 1))); }

// 32 lanes that search one master's neighbourhood together: its lane l of the group, the group's first lane
// in the wavefront, and kFindQueue ints of LDS of its own.
constexpr int kFindQueue = 256;
struct FindGroup {
  int l, first;
  int* q;
  __device__ __forceinline__ unsigned int ballot(bool v) const { return (unsigned int)(__ballot(v) >> first); }
  __device__ __forceinline__ unsigned int below() const { return (1u << l) - 1u; }  // the group's lanes before this one
};
__device__ __forceinline__ FindGroup findGroup(int* queues) {  // queues: kFindQueue ints per group of the block
  const int lane = threadIdx.x & 63;
  return FindGroup{lane & (kFindLanes - 1), lane & ~(kFindLanes - 1), queues + (threadIdx.x / kFindLanes) * kFindQueue};
}

// Visit every item of a search-grid table lying in cells that can hold a point within `reach` of x, 32 at a
// time, by the whole group (`in` tells which lanes hold an item, sorted position k).  Rows
// (y, z) are pruned by their distance to x; the x-run of cells of a row is contiguous in the sorted order,
// so each row costs one range lookup.  Lanes = rows for the lookups (one round trip for 32 rows), then lanes =
// items, listed in LDS; items come row by row, each row in sorted order.
// K rounds of items are read together (load(k)), then taken in order (use(item, k, in)).
template <int K, class Load, class Use>
__device__ __forceinline__ void visitNear(const SearchGrid& S, const int* cellStart, d3 x, double reach,
                                          const FindGroup& G, Load&& load, Use&& use) {
  // (FP32 relative to the grid's corner: the reach is widened by far more than its rounding, and an item
  // visited in vain fails its own test)
  const float cell = float(S.cell), inv = float(S.invCell);
  const float rx = float(x.x - S.mn.x), ry = float(x.y - S.mn.y), rz = float(x.z - S.mn.z);
  const float far = fmaxf(fmaxf(fabsf(rx), fabsf(ry)), fabsf(rz));
  const float rr = float(reach) * (1.f + 1e-6f) + 1e-5f * cell + 1e-6f * far, r2 = rr * rr;
  const int cyLo = clampCellF(floorf((ry - rr) * inv), S.size.y), cyHi = clampCellF(floorf((ry + rr) * inv), S.size.y);
  const int czLo = clampCellF(floorf((rz - rr) * inv), S.size.z), czHi = clampCellF(floorf((rz + rr) * inv), S.size.z);
  const int ny = cyHi - cyLo + 1, nRows = ny * (czHi - czLo + 1);
  for (int r0 = 0; r0 < nRows; r0 += kFindLanes) {
    const int r = r0 + G.l;
    int2 run = make_int2(0, 0);
    if (r < nRows) {
      const int zi = r / ny, cz = czLo + zi, cy = cyLo + (r - zi * ny);
      // (a body beyond the grid lies in a cell of its boundary, which has no end there)
      const float y0 = cy == 0 ? -3e38f : float(cy) * cell, y1 = cy == S.size.y - 1 ? 3e38f : float(cy + 1) * cell;
      const float z0 = cz == 0 ? -3e38f : float(cz) * cell, z1 = cz == S.size.z - 1 ? 3e38f : float(cz + 1) * cell;
      const float dy = fmaxf(0.f, fmaxf(y0 - ry, ry - y1)), dz = fmaxf(0.f, fmaxf(z0 - rz, rz - z1));
      const float rem = r2 - dy * dy - dz * dz;
      if (rem >= 0.f) {
        const float hw = sqrtf(rem);
        const int row = (cz * S.size.y + cy) * S.size.x;
        run = make_int2(cellStart[row + clampCellF(floorf((rx - hw) * inv), S.size.x)],
                        cellStart[row + clampCellF(floorf((rx + hw) * inv), S.size.x) + 1]);
      }
    }
    const int len = max(0, run.y - run.x);
    int incl = len;
#pragma unroll
    for (int o = 1; o < kFindLanes; o <<= 1) {
      const int t = __shfl_up(incl, o, kFindLanes);
      if (G.l >= o) incl += t;
    }
    const int total = __shfl(incl, kFindLanes - 1, kFindLanes), before = incl - len;
    for (int w0 = 0; w0 < total; w0 += kFindQueue) {
      for (int u = max(0, w0 - before); u < min(len, w0 + kFindQueue - before); ++u) G.q[before + u - w0] = run.x + u;
      __builtin_amdgcn_wave_barrier();
      const int n = min(kFindQueue, total - w0);
      for (int i0 = G.l; i0 - G.l < n; i0 += K * kFindLanes) {
        int k[K];
        decltype(load(0)) item[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
          k[u] = 0;
          if (i0 + u * kFindLanes < n) {
            k[u] = G.q[i0 + u * kFindLanes];
            item[u] = load(k[u]);
          }
        }
#pragma unroll
        for (int u = 0; u < K; ++u)
          if (i0 - G.l + u * kFindLanes < n) use(item[u], k[u], i0 + u * kFindLanes < n);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// FP32 sphere-overlap test with a margin covering the FP32 rounding of both centres and radii:
// accepts every pair whose FP64 bounding spheres overlap (a superset is harmless, every pair is
// settled by the exact node tests).
__device__ __forceinline__ bool spheresMayOverlap(float4 a, float4 b, float rb) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  const float ma = fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fabsf(a.z));
  const float mb = fmaxf(fmaxf(fabsf(b.x), fabsf(b.y)), fabsf(b.z));
  const float rr = (a.w + rb) * (1.f + 1e-6f) + 3e-7f * (ma + mb) + 1e-30f;
  return dx * dx + dy * dy + dz * dz <= rr * rr * (1.f + 1e-6f);
}

// Rank of a candidate pair among its partner's reactions as counted so far (sorted later), where the partner
// takes the reaction (particle-particle, ghosts with j != A); else -1.
__device__ __forceinline__ int reactionRank(const Params& P, int A, uint32_t info) {
  const uint32_t type = info >> 28;
  const int partner = int(info & kPartnerMask);
  return type == PT_PP || (type >= PT_GX && partner != A) ? atomicAdd(&P.rcCount[partner], 1) : -1;
}

// Candidate pairs of the master in sorted position t (A = sorted[t]) come in a fixed order, particle
// partners, walls, then ghost images set by set, found by a group of 32 lanes.  The first `room` of them go to
// `list` (the master's part of the slab, or its entries of the pair list) and all are counted.
constexpr int kPairSlab = kPairSlabHost;
struct PairSink {
  int t, A;
  uint32_t* list;
  int room, cnt;
  // (by the whole group: the lanes with a hit are numbered in lane order)
  __device__ __forceinline__ void put(const FindGroup& G, bool hit, uint32_t type, int partner) {
    const unsigned int m = G.ballot(hit);
    const int k = cnt + __popc(m & G.below());
    if (hit && k < room) list[k] = (type << 28) | uint32_t(partner);
    cnt += __popc(m);
  }
};

// Particle partners (B > A, B inside the domain, bounding spheres within the skin), then walls (each wall's
// key is checked each step when the pair is used).
__device__ __forceinline__ void nearPairs(const Params& P, PairSink& sink, const FindGroup& G) {
  const int A = sink.A;
  const float4 a = P.sPR[sink.t];
  const unsigned long long walls = P.nW > 0 && P.nW <= kMaskWalls ? P.wallMask[sink.t] : 0ull;
  const float skin = float(2.0 * P.halfSkin);
  const float ma = fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fabsf(a.z));
  const double reach = (double(a.w) + P.rMax + 2.0 * P.halfSkin) * (1.0 + 2e-6) + 1e-6 * double(ma) + 1e-12;
  struct Item {
    float4 b;
    int id;
  };
  visitNear<4>(P.sg, P.cellStart, mk3(a.x, a.y, a.z), reach, G, [&](int k) { return Item{P.sPR[k], P.sorted[k]}; },
               [&](const Item& it, int, bool in) {
                 sink.put(G, in && it.b.w >= 0.f && it.id > A && spheresMayOverlap(a, it.b, it.b.w + skin), PT_PP,
                          it.id);
               });
  if (P.nW > kMaskWalls) {
    const WallReach R(P, A);
    for (int w0 = 0; w0 < P.nW; w0 += kFindLanes) {
      const int w = w0 + G.l;
      sink.put(G, w < P.nW && R.reaches(P, w), PT_PW, w);
    }
  } else if (P.nW > 0) {
    for (int w0 = 0; w0 < P.nW; w0 += kFindLanes) sink.put(G, (walls >> (w0 + G.l)) & 1ull, PT_PW, w0 + G.l);
  }
}

// Periodic ghost images of a master: any node inside the image's grid box is tested, so the reach is
// the image's grid-box radius.  Images are found through their sources in the particle grid:
// an image shifted by the set's offset lies near x_A - offset; images left at the source's own
// position (a source outside the domain) are searched around x_A only when such images exist.
struct ImageSearch {
  const Params& P;
  float4 g;      // post-wrap centre (images are built from it)
  double reach;
  float lx, ly;
  bool sector, anyUnshifted;
  __device__ __forceinline__ ImageSearch(const Params& P_, int t) : P(P_) {
    g = P.sPRw[t];
    const float mg = fmaxf(fmaxf(fabsf(g.x), fabsf(g.y)), fabsf(g.z));
    reach = (double(g.w) + P.boxRMax + 2.0 * P.halfSkin) * (1.0 + 2e-6) + 1e-6 * double(mg) + 1e-12;
    lx = float(P.gridP.mx.x - P.gridP.mn.x);
    ly = float(P.gridP.mx.y - P.gridP.mn.y);
    sector = P.periodicSector != 0;
    anyUnshifted = P.devInt[ghostCountIdx(P.curBuf)] > 0;
  }
  __device__ __forceinline__ bool on(int s) const {
    return sector || (s == 0 && P.periodicX) || (s == 1 && P.periodicY) || (s == 2 && P.periodicX && P.periodicY);
  }
  // where the sources of set s's images near the master lie (a turn the other way for sector images);
  // shifted = false: of its images at their source's own position
  __device__ __forceinline__ d3 centre(int s, bool shifted) const {
    const d3 x = mk3(g.x, g.y, g.z);
    if (!shifted) return x;
    if (sector) return P.gridP.mn + secTurnByIndex(2 - s, x - P.gridP.mn);
    return mk3(x.x - double(s != 1 ? lx : 0.f), x.y - double(s != 0 ? ly : 0.f), x.z);
  }
  // the image of a source at b (shifted by the period, or turned about the corner's z axis)
  __device__ __forceinline__ float4 image(int s, float4 b) const {
    if (!sector) return make_float4(b.x + (s != 1 ? lx : 0.f), b.y + (s != 0 ? ly : 0.f), b.z, 0.f);
    const d3 r = P.gridP.mn + secTurnByIndex(s, mk3(b.x, b.y, b.z) - P.gridP.mn);
    return make_float4(float(r.x), float(r.y), float(r.z), 0.f);
  }
  __device__ __forceinline__ bool reaches(int s, bool shifted) const {
    return on(s) && !(searchBoxDist2(P.sg, centre(s, shifted)) > reach * reach);
  }
};
// Whether a master has any images to search for (most lie too far from the periodic faces).
__device__ __forceinline__ bool mayMeetImages(const Params& P, int t) {
  const ImageSearch I(P, t);
  bool any = false;
#pragma unroll 1
  for (int s = 0; s < 3; ++s) any = any || I.reaches(s, true) || (I.anyUnshifted && I.reaches(s, false));
  return any;
}
__device__ __forceinline__ void imagePairs(const Params& P, PairSink& sink, const FindGroup& G) {
  const ImageSearch I(P, sink.t);
  const GridGeom& grid = P.gridP;
  const float skin = float(2.0 * P.halfSkin);
  for (int s = 0; s < 3; ++s) {
    const int col = I.sector ? imageColumn<true>(s) : imageColumn<false>(s);
    for (int pass = 0; pass < 2; ++pass) {
      const bool shifted = pass == 0;
      if (!shifted && !I.anyUnshifted) break;
      if (!I.reaches(s, shifted)) continue;
      struct Item {
        float4 b;
        float box;
      };
      visitNear<1>(P.sg, P.cellStart, I.centre(s, shifted), I.reach, G,
                   [&](int k) { return Item{P.sPRw[k], P.sBoxR[k]}; },
                   [&](const Item& it, int k, bool in) {
                     bool hit = false;
                     int j = -1;
                     // (the set and half the skin as values of this item: what follows from them in FP64, a turn's
                     // terms and the bounds of the tests below, would be kept in registers through the search)
                     const int si = uniformInItem(s, k);
                     const float rb = it.box + skin;
                     if (in && spheresMayOverlap(I.g, shifted ? I.image(si, it.b) : it.b, rb)) {
                       j = P.sorted[k];
                       const double hs = inItem(P.halfSkin, j);
                       const d3 pj = P.pos[j];
                       if (shifted) {
                         hit = potInColumn(grid, pj, col, hs);
                       } else {
                         // (one pair per master and image: the shifted pass already took it)
                         hit = potOutOfDomain(P, pj, hs) && potOutColumn(grid, pj, col, hs) &&
                               !(potInColumn(grid, pj, col, hs) && spheresMayOverlap(I.g, I.image(si, it.b), rb));
                       }
                     }
                     sink.put(G, hit, PT_GX + s, j);
                   });
    }
  }
}

// Lists the masters of the share of a block of THREADS threads that want(t), THREADS at a time (many: an int per
// thread, and one), and takes them one per group of 32 lanes: use(t).
template <int THREADS, class Want, class Use>
__device__ __forceinline__ void listedMasters(const Params& P, const MasterShare<THREADS / kFindLanes>& share, int* many,
                                              Want&& want, Use&& use) {
  int* const nMany = many + THREADS;
  const int group = int(threadIdx.x) / kFindLanes, groups = THREADS / kFindLanes;
  for (int i0 = 0; i0 < share.chunk; i0 += THREADS) {
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x == 0) *nMany = 0;
    __syncthreads();
    const int i = i0 + int(threadIdx.x), t = share.at(i);
    if (i < share.chunk && t < P.nP && want(t)) many[atomicAdd(nMany, 1)] = t;
    __syncthreads();
    for (int m = group; m < *nMany; m += groups) use(many[m]);
  }
}

// Broad phase, 32 lanes per master: count its candidates and keep the first.  Bound by each master's chain of
// round trips (its own data, the row lookups, four rounds of 32 items at a time) and by how unevenly masters
// meet neighbours.  Images are searched in a turn of their own for the masters that may have any.  (One
// thread per master, an item a round trip: 398 us of a rebuild's 522 for 4,000 bodies in a quarter sector, 340
// of 507 for 20,000 of scattered sizes, 597 of 1,028 for 200,000; whole rebuilds on the same grids now: 301, 319, 683.
// Tried and left out: a largest radius per search cell to shorten the runs, with cells of 1, 0.5 and 0.35
// of this edge: 348 us of search at 200,000 for 440 then, 139 for 148 at 20,000, slower below; finer
// cells slower everywhere.)
// queues: kFindQueue ints of LDS per group of the block; many: an int per thread, and one.
template <int THREADS>
__device__ __forceinline__ void pairsFind(const Params& P, int* queues, int* many) {
  const FindGroup G = findGroup(queues);
  constexpr int groups = THREADS / kFindLanes;
  const MasterShare<groups> share(P.nP, int(gridDim.x), int(blockIdx.x));
  const int group = int(threadIdx.x) / kFindLanes;
  for (int i = group; i < share.chunk; i += groups) {
    const int t = share.at(i);
    if (t >= P.nP) continue;
    PairSink sink{t, P.sorted[t], P.pairSlab + (long long)t * kPairSlab, kPairSlab, 0};
    nearPairs(P, sink, G);
    if (G.l == 0) P.pairCount[sink.A] = sink.cnt;
  }
  if (!(P.periodicX || P.periodicY || P.periodicSector)) return;
  listedMasters<THREADS>(P, share, many, [&](int t) { return mayMeetImages(P, t); }, [&](int t) {
    const int A = P.sorted[t];
    PairSink sink{t, A, P.pairSlab + (long long)t * kPairSlab, kPairSlab, P.pairCount[A]};
    imagePairs(P, sink, G);
    if (G.l == 0) P.pairCount[inLoop(A, 1)] = sink.cnt;
  });
}
__global__ __launch_bounds__(kFindThreads) void k_pairs_find(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  __shared__ int queues[kFindThreads / kFindLanes * kFindQueue], many[kFindThreads + 1];
  pairsFind<kFindThreads>(P, queues, many);
}
// Entry k of master A's part of the pair list (from `out` on), its rank among the partner's reactions with it.
__device__ __forceinline__ void emitPair(const Params& P, int A, long long out, int k, uint32_t info) {
  const int rank = reactionRank(P, A, info);
  if (out + k < P.pairCap) {
    P.pairA[out + k] = A;
    P.pairInfo[out + k] = info;
    P.rcRank[out + k] = rank;
  }
}
// Pair list in master order: eight lanes per master copy its part of the slab, eight candidates a turn (a thread
// per master took as many turns as a master has candidates: 24 us of a rebuild for 4,000 bodies in a quarter
// sector, now 7); masters with more candidates than the slab holds are searched again, into their part of the list.
// queues, many: as pairsFind.
template <int THREADS>
__device__ __forceinline__ void pairsEmit(const Params& P, int* queues, int* many) {
  constexpr int kLanes = 8;
  const FindGroup G = findGroup(queues);
  const MasterShare<THREADS / kFindLanes> share(P.nP, int(gridDim.x), int(blockIdx.x));
  const int l = int(threadIdx.x) & (kLanes - 1);
  int* const anyLarge = many + THREADS;
  if (threadIdx.x == 0) *anyLarge = 0;
  __syncthreads();
  for (int i = int(threadIdx.x) / kLanes; i < share.chunk; i += THREADS / kLanes) {
    const int t = share.at(i);
    if (t >= P.nP) continue;
    const int A = P.sorted[t];
    const int n = P.pairCount[A];
    const long long out = P.pairStart[A];
    if (n > kPairSlab) *anyLarge = 1;
    else
      for (int k = l; k < n; k += kLanes) emitPair(P, A, out, k, P.pairSlab[(long long)t * kPairSlab + k]);
  }
  __syncthreads();
  if (!*anyLarge) return;
  // (three passes over the block's large masters: with both searches in one loop, registers spill.  rank, free
  // since the sort, keeps how many partners and walls the first found.)
  const auto isLarge = [&](int t) { return P.pairCount[P.sorted[t]] > kPairSlab; };
  listedMasters<THREADS>(P, share, many, isLarge, [&](int t) {
    const int A = P.sorted[t];
    PairSink sink{t, A, P.pairInfo + P.pairStart[A], P.pairCount[A], 0};
    nearPairs(P, sink, G);
    if (G.l == 0) P.rank[t] = sink.cnt;
  });
  if (P.periodicX || P.periodicY || P.periodicSector)
    listedMasters<THREADS>(P, share, many, isLarge, [&](int t) {
      const int A = P.sorted[t];
      PairSink sink{t, A, P.pairInfo + P.pairStart[A], P.pairCount[A], P.rank[t]};
      imagePairs(P, sink, G);
    });
  listedMasters<THREADS>(P, share, many, isLarge, [&](int t) {
    const int A = P.sorted[t], n = P.pairCount[A];
    const long long out = P.pairStart[A];
    for (int k = G.l; k < n; k += kFindLanes) emitPair(P, A, out, k, P.pairInfo[out + k]);
  });
}
// Keep the pair list being replaced (per-master starts, entries, certificates) for the
// certificates the new list inherits; runs before the new starts and entries are written.
__device__ void backupPairs(const Params& P, Span g) {
  const int n = min(P.pairStart[P.nP], (int)P.pairCap);
  for (int i = g.tid; i <= P.nP; i += g.nth) P.oldStart[i] = P.pairStart[i];
  for (int p = g.tid; p < n; p += g.nth) {
    P.oldInfo[p] = P.pairInfo[p];
    P.oldCert[p] = P.cert[p];
  }
}
__global__ void k_backup_pairs(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  backupPairs(P, gridSpan());
}
// A particle-particle pair of the new list that was in the previous one keeps its certificate,
// rebased to this build: the room its fast check leaves now (bound from the old motion records,
// read before they restart), with the rotation coefficients of this build's poses (|d| + r_A and
// r_A).  A node's motion since the old evaluation is at most the old bound now plus the new bound
// later, so the new bound staying below that room keeps the pair separated.  Other pairs start
// without a certificate.
__device__ void inheritCerts(const Params& P, Span g) {
  const int n = min(P.pairStart[P.nP], (int)P.pairCap);
  for (int p = g.tid; p < n; p += g.nth) {
    float4 nc = make_float4(-1.f, 0.f, 0.f, -1.f);
    const uint32_t info = P.pairInfo[p];
    if (P.useCert && (info >> 28) == PT_PP) {
      const int A = P.pairA[p], j = int(info & kPartnerMask);
      const int q1 = min(P.oldStart[A + 1], (int)P.pairCap);
      for (int q = P.oldStart[A]; q < q1; ++q) {
        if (P.oldInfo[q] != info) continue;
        const float4 c = P.oldCert[q];
        if (c.x > 0.f) {
          const float4 mA = P.step[A].motion, mB = P.step[j].motion;
          const float ex = mA.x - mB.x, ey = mA.y - mB.y, ez = mA.z - mB.z;
          const float bound = (sqrtf(ex * ex + ey * ey + ez * ez) + mB.w * c.y + mA.w * fabsf(c.z)) * (1.f + 1e-5f);
          const float rem = (c.x - bound) * (1.f - 1e-5f) - 1e-6f * c.x;  // the roundings of both checks
          if (rem > 0.f) {
            const double cA = P.scale[A] * P.shapes[P.shape[A]].nodeR * (1.0 + 1e-6);
            const double cB = (len(P.posDet[A] - P.posDet[j]) + cA) * (1.0 + 1e-6);
            nc = make_float4(rem, float(cB * (1.0 + 1e-6)), copysignf(float(cA * (1.0 + 1e-6)), c.z), -1.f);
          }
        }
        break;
      }
    }
    P.cert[p] = nc;
  }
}
__global__ void k_inherit_certs(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  inheritCerts(P, gridSpan());
}
// The new list does not fit: raise the error (the rest of the call halts) instead of writing it.
__device__ __forceinline__ bool pairOverflow(const Params& P) {
  const int np = P.pairStart[P.nP];
  if ((long long)np <= P.pairCap) return false;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    atomicMax(&P.devInt[4], np);
    raiseFlag(P, kErrPairs);
  }
  return true;
}
__global__ __launch_bounds__(kFindThreads) void k_pairs_emit(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  if (pairOverflow(P)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) dropGates(P);
    return;
  }
  __shared__ int queues[kFindThreads / kFindLanes * kFindQueue], many[kFindThreads + 1];
  pairsEmit<kFindThreads>(P, queues, many);
}
__global__ void k_mark_build(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  markBuild(P, gridSpan());
}

__device__ void rcScatterPairs(const Params& P, Span g) {
  const int n = min(P.pairStart[P.nP], (int)P.pairCap);
  for (int p = g.tid; p < n; p += g.nth) {
    const int r = P.rcRank[p];
    if (r < 0) continue;
    const int partner = int(P.pairInfo[p] & kPartnerMask);
    const int d = P.rcStart[partner] + r;
    if (d < P.pairCap) P.rcTmp[d] = p;
  }
}
__global__ void k_rc_scatter(Params P) {
  LSD_GATE(P.devInt + rebuildFlagIdx(P.curBuf));
  if (blockIdx.x == 0 && threadIdx.x == 0) P.devInt[2] = 0;  // large-bucket list of the following sort
  rcScatterPairs(P, gridSpan());
}

// ------------------------------------------------------------------------------------------
// History table
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long histKey(uint32_t type, int gnode, int partner) {
  return ((unsigned long long)type << 59) | ((unsigned long long)(unsigned)gnode << 28) | (unsigned long long)partner;
}
__device__ __forceinline__ unsigned long long mix64(unsigned long long x) {
  x ^= x >> 30;
  x *= 0xbf58476d1ce4e5b9ull;
  x ^= x >> 27;
  x *= 0x94d049bb133111ebull;
  x ^= x >> 31;
  return x;
}
// Insert a contact of this step into this step's table (open addressing, linear probing); returns
// the slot, recorded so that the entry can be removed when the table is reused two steps later.
// The table holds at least twice the contact capacity, so a probe finds a free slot long before it
// has seen every slot; a probe that does see every slot raises kErrHash and gives up.
__device__ __forceinline__ int histInsert(const Params& P, unsigned long long key, int c) {
  unsigned long long slot = mix64(key) & P.hashMask;
  for (unsigned long long probe = 0; probe <= P.hashMask; ++probe) {
    const unsigned long long old = atomicCAS(&P.hashKey[slot], kHashEmpty, key);
    if (old == kHashEmpty || old == key) {
      P.hashVal[slot] = c;
      return int(slot);
    }
    slot = (slot + 1) & P.hashMask;
  }
  raiseError(P, kErrHash);
  return -1;
}

// The previous step's spring of a contact key (zero when it had none), from the previous table,
// given the key k0 and value v0 already read at the key's first slot slot0.
__device__ __forceinline__ d3 histLookup(const Params& P, unsigned long long key, unsigned long long slot0,
                                         unsigned long long k0, int v0) {
  if (k0 == key) return P.prevSpring[v0];
  unsigned long long slot = slot0, k = k0;
  for (unsigned long long probe = 0; probe <= P.hashMask; ++probe) {
    if (k == key) return P.prevSpring[P.prevHashVal[slot]];
    if (k == kHashEmpty) return mk3(0., 0., 0.);
    slot = (slot + 1) & P.hashMask;
    k = P.prevHashKey[slot];
  }
  return mk3(0., 0., 0.);  // (a full table: the insert that filled it raised kErrHash)
}

// ------------------------------------------------------------------------------------------
// Narrow phase: node-vs-SDF detection, one wavefront per batch of evaluated pairs
// ------------------------------------------------------------------------------------------
constexpr int kNarrowBlock = 256;

// Contact terms and masks.  Bit of the k-th pair of a body's list in its contact mask: the first kHitBits pairs have a bit each, the
// rest share the last one (and are then told apart by their contact counts).
constexpr int kTermDoubles = 9;  // of a contact in cTerm: force, torque on the master, torque on the partner
constexpr int kHitBits = 31;
constexpr unsigned int kHitRest = 1u << kHitBits;
__device__ __forceinline__ unsigned int hitBit(int k) { return k < kHitBits ? 1u << k : kHitRest; }

// Stat slot `slot` of accumulator family f (one 128-byte line per slot).
__device__ __forceinline__ unsigned long long* statSlot(const Params& P, int f, int slot) {
  return P.statSlots + (f * kStatSlots + slot) * kStatStride;
}

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Detection-side view of a pair (everything the node tests need).
struct PairView {
  int pair, A, partner, nodeBase, nNodes, valid;
  uint32_t type, info;
  d3 xA;        // master position used for detection
  q4 qA;
  double sA;
  double rA;    // largest distance of a node of A from A's origin (scaled)
  int clusterOff, nClusters, nodeOff, shapeB;
  d3 xB;        // partner pose used for detection
  q4 qB;
  double rB;    // particle-particle radius cull (0 for fixed partners)
  double invSpB;
  d3 goB;
};

// (info and A as in pairInfo[p], pairA[p], when the caller already holds them)
template <bool SEC>
__device__ __forceinline__ PairView loadPair(const Params& P, int p, uint32_t info, int A) {
  PairView v;
  v.pair = p;
  v.info = info;
  v.type = v.info >> 28;
  v.partner = int(v.info & kPartnerMask);
  v.A = A;
  const bool ghost = v.type >= PT_GX;
  v.xA = ghost ? P.pos[v.A] : P.posDet[v.A];
  v.qA = (SEC && !ghost) ? P.quatDet[v.A] : P.quat[v.A];
  const BodyProp& pA = P.prop[v.A];
  v.sA = pA.scale;
  v.rA = pA.rNode;
  v.nodeBase = pA.nodeStart;
  v.nNodes = pA.nNodes;
  const ShapeDev& SA = P.shapes[pA.shape];
  v.clusterOff = SA.clusterOff;
  v.nClusters = SA.nClusters;
  v.nodeOff = SA.nodeOff;
  const int j = v.type == PT_PW ? P.nP + v.partner : v.partner;  // (walls follow the particles)
  if (ghost) {
    v.xB = imgPos<SEC>(P, int(v.type - PT_GX))[j];
    v.qB = SEC ? imgQuat(P, int(v.type - PT_GX))[j] : P.quat[j];
  } else {
    // (a wall's one position, which a caller may set between two phases of a step, is its detection position too)
    v.xB = P.pos[(long long)(v.type == PT_PW ? kSvPos : kSvDet) * P.nBodies + j];
    v.qB = SEC && v.type == PT_PP ? P.quatDet[j] : P.quat[j];
  }
  const BodyProp& pB = P.prop[j];
  v.rB = pB.radius;
  v.shapeB = pB.shape;
  v.invSpB = pB.invSp;
  v.goB = mk3(pB.origin[0], pB.origin[1], pB.origin[2]);
  v.valid = 1;
  return v;
}

// The step record's key of a pair's partner of type t (the body's own key, or its image's): a
// select, since a runtime index into the record's fields would go through scratch memory.
__device__ __forceinline__ int partnerKey(int4 key, uint32_t t) {
  return t == PT_PP ? key.x : (t == PT_GX ? key.y : (t == PT_GY ? key.z : key.w));
}

struct NodeHit {
  d3 point, normal;
  double ov;
};

// What the exact test and the contact law of a pair need, in LDS (k_candidates fills it for the pairs of
// its batch that hold candidate nodes): the state vectors, orientation and properties of both bodies
// ([0] the master), the law's constants and the partner's cell key.
struct BodySide {
  double v[4][3];    // kSvPos, kSvDet, kSvVel, kSvAng (an image's own in place of its body's)
  double q[4];       // orientation used by the detection
  double prop[16];   // BodyProp
};
struct alignas(16) PairExact {
  BodySide side[2];
  double law[5];     // kn, ks, mu, dissipation, effective mass
  int keyB, pad;
};
static_assert(sizeof(PairExact) % 16 == 0, "PairExact records follow one another in LDS");
__device__ __forceinline__ d3 lds3(const double* v) { return mk3(v[0], v[1], v[2]); }
__device__ __forceinline__ q4 lds4(const double* v) { return q4{v[0], v[1], v[2], v[3]}; }

// Exact node-vs-SDF test of a node of the pair's master in the reference's arithmetic: node transform,
// radius cull or cell window, grid bounds, trilinear overlap >= 0.
// (nB and sdfOff: the partner's grid size and its offset in the SDF pool)
__device__ __forceinline__ bool exactTest(const Params& P, const PairExact& X, uint32_t type, d3 nd, i3 nB, int sdfOff,
                                          NodeHit& h, unsigned int& queries) {
  const BodySide &A = X.side[0], &B = X.side[1];
  const double sA = A.prop[kPropScale];
  // (the images are built after the periodic wrap, from the position the master then has)
  const d3 xA = lds3(type >= PT_GX ? A.v[kSvPos] : A.v[kSvDet]);
  const d3 xw = rot(lds4(A.q), mk3(nd.x * sA, nd.y * sA, nd.z * sA)) + xA;
  const d3 dB = xw - lds3(B.v[kSvDet]);
  if (type == PT_PP) {
    const double rB = B.prop[kPropRadius];
    if (len2(dB) > rB * rB) return false;
  } else {
    if (!keyInWindow(type == PT_PW ? P.gridW : P.gridP, X.keyB, xw)) return false;
  }
  const q4 qB = lds4(B.q);
  const d3 loc = rotInv(dB, qB), goB = lds3(B.prop + kPropOrigin);
  const double invSp = B.prop[kPropInvSp];
  const double gx = (loc.x - goB.x) * invSp, gy = (loc.y - goB.y) * invSp, gz = (loc.z - goB.z) * invSp;
  const int i0 = (int)floor(gx), j0 = (int)floor(gy), k0 = (int)floor(gz);
  if (i0 < 0 || j0 < 0 || k0 < 0 || i0 >= nB.x - 1 || j0 >= nB.y - 1 || k0 >= nB.z - 1) return false;
  const double x = gx - double(i0), y = gy - double(j0), z = gz - double(k0);
  const float* g = P.sdf + sdfOff + lin3(i3{i0, j0, k0}, nB);
  const int sy = nB.x, sz = nB.x * nB.y;
  const float f000 = g[0], f100 = g[1], f010 = g[sy], f110 = g[sy + 1];
  const float f001 = g[sz], f101 = g[sz + 1], f011 = g[sz + sy], f111 = g[sz + sy + 1];
  const double sc = B.prop[kPropScale];
  const double cc[8] = {double(f000) * sc, double(f100) * sc, double(f010) * sc, double(f110) * sc,
                        double(f001) * sc, double(f101) * sc, double(f011) * sc, double(f111) * sc};
  queries++;
  h.ov = -triValue(x, y, z, cc);
  if (!(h.ov >= 0.)) return false;
  d3 n = triGradient((P.quirks & 1) ? double(int(x)) : x, y, z, cc);
  n = rot(qB, n);
  n = normalize(n);
  h.normal = n;
  h.point = xw + 0.5 * h.ov * n;
  return true;
}

// FP32 map of A's unscaled node coordinates n into the partner's grid index space,
// g = M n + t (g = (R_B^T (x_world - x_B) - origin_B) / spacing_B), with conservative acceptance
// regions: every margin is far above the FP32 rounding of the map and of the interpolation.
struct alignas(16) PairF32 {
  float m[9], t[3];
  float c[3], r2;     // pp: partner centre in g and squared bounding radius (g units); r2 < 0: no sphere test
  float lo;           // grid box in g: [lo, n - 1 - lo] per axis
  float phiMargin;    // SDF prefilter margin for FP32 map rounding (unscaled SDF units)
  float rhoScale;     // A's unscaled cluster radius -> g units
  float lipH;         // Lipschitz bound of the partner's SDF per g unit
  int nx, ny, nz, sdfOff;
  int nodeOff, clusterOff, nClusters;  // A's shape
  int pair, A;        // candidate pair index, its master
  uint32_t info;      // its list entry
  float gToWorld;     // world length of one g unit (the partner's scaled spacing)
  float o[3], h;      // partner's unscaled grid origin and spacing (g -> local point)
  int slot;           // partner's surrogate family slot, -1 if none (walls)
  float certD0;       // motion bound of the pair since the build, at this step (inf: none)
  float certCB, certCA;  // certificate coefficients of the partner's and the master's rotation
};
static_assert(sizeof(PairF32) == 160, "pair map record is 160 bytes");
// Upper bound of the grid box on an axis of n nodes (rounded to FP32 once more: 4e-6 for 50 nodes, within
// the 13 margins to spare in -lo).
__device__ __forceinline__ float boxHi(const PairF32& f, int n) { return float(n - 1) - f.lo; }

__device__ __forceinline__ void makeF32(const Params& P, const PairView& v, PairF32& f) {
  const ShapeDev SB = P.shapes[v.shapeB];
  const double is = v.invSpB;  // 1 / (scaled spacing)
  const d3 c0 = rotInv(rot(v.qA, mk3(v.sA, 0., 0.)), v.qB) * is;
  const d3 c1 = rotInv(rot(v.qA, mk3(0., v.sA, 0.)), v.qB) * is;
  const d3 c2 = rotInv(rot(v.qA, mk3(0., 0., v.sA)), v.qB) * is;
  const d3 t = (rotInv(v.xA - v.xB, v.qB) - v.goB) * is;
  f.m[0] = float(c0.x); f.m[1] = float(c1.x); f.m[2] = float(c2.x);
  f.m[3] = float(c0.y); f.m[4] = float(c1.y); f.m[5] = float(c2.y);
  f.m[6] = float(c0.z); f.m[7] = float(c1.z); f.m[8] = float(c2.z);
  f.t[0] = float(t.x); f.t[1] = float(t.y); f.t[2] = float(t.z);
  // Every term of g = M n + t lies below reach: |M n| <= rA / spacing for a node (and sqrt(3) times
  // that for a cluster's box centre).  The FP32 rounding of M, n, t, the products and the sums is below
  // 12 x 2^-24 reach = 7e-7 reach, so the margins below are 14 times what they have to cover.  (A bound
  // of 8 scale / spacing in rA's place is right for shapes of unit size only: shapes given in metres at
  // scale 1 had margins of 0.16 grid cells, and 4.06M candidate nodes for 0.21M contacts in an ordered
  // bed of 27,000 of them; with rA 0.21M, and its candidate kernel takes 184 us instead of 497.)
  const double cg = len(v.goB) * is;
  const double reach = len(t) + v.rA * is + cg + double(SB.nx + SB.ny + SB.nz);
  const double abs = 1e-5 * reach + 1e-6;
  f.c[0] = float(-v.goB.x * is); f.c[1] = float(-v.goB.y * is); f.c[2] = float(-v.goB.z * is);
  if (v.type == PT_PP) {
    const double r = v.rB * is * (1.0 + 1e-5) + abs;
    f.r2 = float(r * r);
  } else {
    f.r2 = -1.f;
  }
  f.lo = float(-abs);
  f.lipH = float(SB.lip * SB.h * (1.0 + 1e-5));
  f.phiMargin = float(SB.lip * SB.h * abs * 2.0 + 1e-30);
  f.rhoScale = float(v.sA * is * (1.0 + 1e-5));
  f.nx = SB.nx; f.ny = SB.ny; f.nz = SB.nz;
  f.sdfOff = int(SB.sdfOff);
  f.nodeOff = v.nodeOff;
  f.clusterOff = v.clusterOff;
  f.nClusters = v.nClusters;
  f.pair = v.pair;
  f.A = v.A;
  f.info = v.info;
  f.gToWorld = float(1.0 / is);
  f.o[0] = float(SB.ox); f.o[1] = float(SB.oy); f.o[2] = float(SB.oz);
  f.h = float(SB.h);
  f.slot = (P.surSlot && v.type != PT_PW) ? P.surSlot[v.shapeB] : -1;
  // Separation-certificate coefficients.  A node u of A (|u| <= rA) sits at
  // g = R_B^T (d + R_A u) / spacing, d = x_A - x_B.  Between the build and now it moved at most
  //   |dA - dB| + chord_B |d_build| + (chord_A + chord_B) rA,   |d_build| <= |d| + |dA - dB|,
  // with dA, dB the displacements and chord the rotation chords since the build.
  const float4 mA = P.step[v.A].motion;
  float4 mB;
  bool flip = false;  // an image that changed its shift state has no motion bound
  if (v.type == PT_PW) mB = P.wMotion[v.partner];
  else {
    const BodyStep sb = P.step[v.partner];
    mB = sb.motion;
    if (v.type >= PT_GX) flip = ((partnerKey(sb.key, v.type) >> kFlipBit) & 1) != 0;
  }
  const double ex = double(mA.x) - double(mB.x), ey = double(mA.y) - double(mB.y), ez = double(mA.z) - double(mB.z);
  const double del = sqrt(ex * ex + ey * ey + ez * ez);
  const double cA = v.rA * (1.0 + 1e-6);
  const double cB = (len(v.xA - v.xB) + del + cA) * (1.0 + 1e-6);
  const double d0 = del + double(mB.w) * cB + double(mA.w) * cA;
  f.certD0 = flip ? __builtin_huge_valf() : float(d0 * (1.0 + 1e-5));
  f.certCB = float(cB * (1.0 + 1e-6));
  f.certCA = float(cA * (1.0 + 1e-6));
}

// Which pairs the narrow phase evaluates this step, one thread per candidate pair.  A pair is
// skipped when its partner does not exist now (pp: outside the domain; wall: its key; ghost: the
// image) or when its separation certificate still holds: the motion bound of its nodes since the
// build stays below the slack recorded at its last evaluation (all its nodes were culled then
// with that much room).  Skipped pairs have no contacts.  full != 0 (an audit step of the
// surrogate) also evaluates every live pair whose certificate rests on the surrogate's slack.
// A block compacts a tile of pairs in LDS, appends it with one atomic, then writes the FP32
// map records of its evaluated pairs (FP64 poses in, one 160-byte record out, in evaluation
// order).  A tile has 256 pairs, one per thread, as long as those tiles are resident together (two
// blocks per CU), else 1024: a short list is bound by each thread's chain of reads, which a thread's four
// pairs lengthen (those near contact read the state of their last evaluation one after another, and their
// records take several rounds), a long one by the number of tiles.  (Four pairs per thread on every list, before
// -> now: 15.7 -> 7.1 us for 1,000 bodies in a box, 15.2 -> 8.6 for 20,000 falling, 13.1 -> 7.3 for 8,000 bonded.)  A block group g (blockIdx mod 8) checks one contiguous eighth of the tiles and writes the
// records of its evaluated pairs from the first pair of its first tile on, with its own counter
// (evalCount[g]): 8 counters on 8 lines instead of one, since returning atomics on one address are
// served one after another (~11 ns each) and every tile takes one.
constexpr int kCheckTile = 1024, kCheckTileShort = 256, kShortPairs = 512 * kCheckTileShort;
__device__ __forceinline__ int checkTileSize(int nPairs) { return nPairs <= kShortPairs ? kCheckTileShort : kCheckTile; }

// The evaluated pairs' map records, numbered densely group after group (record a of the narrow
// phase) and found at their place in the groups' regions of pairMap.
struct EvalRecords {
  int n;  // records this step
  int pre[8], base[8];
  // position in pairMap of record a (0 <= a < n): the last group whose first record is at or below a
  // (a group without records has the same first record as the next one)
  __device__ __forceinline__ int at(int a) const {
    int pos = a;
#pragma unroll
    for (int g = 0; g < 8; ++g)
      if (a >= pre[g]) pos = base[g] + (a - pre[g]);
    return pos;
  }
};
__device__ __forceinline__ int groupFirstTile(int nTiles, int g) { return int((long long)nTiles * g / 8); }
__device__ __forceinline__ EvalRecords evalRecords(const Params& P) {
  EvalRecords e;
  const int nPairs = min(P.pairStart[P.nP], (int)P.pairCap), tile = checkTileSize(nPairs);
  const int nTiles = (nPairs + tile - 1) / tile;
  int sum = 0;
#pragma unroll
  for (int g = 0; g < 8; ++g) {
    e.pre[g] = sum;
    e.base[g] = groupFirstTile(nTiles, g) * tile;
    sum += evalCount(P)[g * kBarrierLine];
  }
  e.n = sum;
  return e;
}
struct CheckLds {
  int list[kCheckTile], A[kCheckTile];
  uint32_t info[kCheckTile];
  int count, base;
};
// R: pairs of a tile per thread (tiles of 256 R)
template <bool SEC, int R>
__device__ void checkPairs(const Params& P, int full, int nPairs, CheckLds& L) {
  constexpr int kTile = 256 * R;
  int *const sList = L.list, *const sA = L.A;
  uint32_t* const sInfo = L.info;
  int &sCount = L.count, &sBase = L.base;
  PairF32* out = reinterpret_cast<PairF32*>(P.pairMap);
  const bool rebuilt = P.devInt[rebuildFlagIdx(P.curBuf)] != 0;  // a new pair list this step
  const bool fresh = !P.useCert;  // (a new list holds the certificates it inherited)
  const int lane = threadIdx.x & 63;
  const unsigned long long ltMask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  // XCD-aware tiles: workgroups go to the 8 XCDs in turn (blockIdx mod 8), so each XCD takes one
  // contiguous eighth of the pair list and its partners' data stays in that XCD's L2
  const int nTiles = (nPairs + kTile - 1) / kTile;
  const int xcd = int(blockIdx.x) & 7, perX = (int(gridDim.x) - xcd + 7) >> 3;  // blocks on this XCD
  const int tLo = groupFirstTile(nTiles, xcd), tHi = groupFirstTile(nTiles, xcd + 1);
  const int region = tLo * kTile;  // this group's records: at most its pairs, from its first pair on
  unsigned int evNodes = 0;  // boundary nodes of the masters of this thread's evaluated pairs
  for (int t = tLo + (int(blockIdx.x) >> 3); t < tHi; t += perX) {
    const int t0 = t * kTile;
    if (threadIdx.x == 0) sCount = 0;
    __syncthreads();
    // the tile's pairs of this thread, with the loads of one kind issued together
    // (vector types: an element picked by a runtime index stays in registers, where an array's
    // would be read from scratch)
    typedef int IntR __attribute__((ext_vector_type(R)));
    typedef uint32_t UintR __attribute__((ext_vector_type(R)));
    IntR pv, Av, jv;
    UintR tv;
    int key[R];
    float4 cv[R], mB[R], mA[R];
#pragma clang loop unroll(full)
    for (int r = 0; r < R; ++r) {
      pv[r] = t0 + r * 256 + int(threadIdx.x);
      const bool in = pv[r] < nPairs;
      const uint32_t info = in ? P.pairInfo[pv[r]] : (uint32_t(PT_PW) << 28);
      tv[r] = info >> 28;
      jv[r] = int(info & kPartnerMask);
      Av[r] = in ? P.pairA[pv[r]] : 0;
      cv[r] = (in && !fresh) ? P.cert[pv[r]] : make_float4(-1.f, 0.f, 0.f, -1.f);
    }
#pragma clang loop unroll(full)
    for (int r = 0; r < R; ++r) {
      // the partner's step record (liveness key with the image's flip, motion): one 32-byte read
      if (pv[r] >= nPairs) {
        key[r] = -1;
        mB[r] = make_float4(0.f, 0.f, 0.f, 0.f);
      } else if (tv[r] == PT_PW) {
        key[r] = P.wkey[jv[r]];
        mB[r] = P.wMotion[jv[r]];
      } else {
        const BodyStep sb = P.step[jv[r]];
        key[r] = partnerKey(sb.key, tv[r]);
        mB[r] = sb.motion;
      }
      mA[r] = (cv[r].x > 0.f || cv[r].w > 0.f) ? P.step[Av[r]].motion : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // A pair whose bound against the motion since the build is spent (c.x <= 0) is checked against
    // the motion since its evaluation whatever the partner's motion: the inputs of that bound are
    // read now, with the partner's record, for the first such pair of the thread (about 1 % of the
    // pairs are; a thread's others read them one round trip later).
    int early = -1;
#pragma clang loop unroll(full)
    for (int r = R - 1; r >= 0; --r)
      if (pv[r] < nPairs && cv[r].x <= 0.f && cv[r].w > 0.f) early = r;
    float4 e0e, qa0e, qb0e, qae, qbe;
    if (early >= 0) {
      const int p = pv[early], A = Av[early], j = jv[early];
      e0e = P.certE[p];
      qa0e = P.certQA[p];
      qb0e = P.certQB[p];
      qae = P.qrel[A];
      qbe = tv[early] == PT_PW ? P.wQrel[j] : P.qrel[j];
    }
    bool actv[R];
#pragma clang loop unroll(full)
    for (int r = 0; r < R; ++r) {
      const int p = pv[r];
      const bool live = key[r] >= 0;
      bool act = live;
      // an audit step of the surrogate (full) trusts only certificates of the exact culls; the
      // turned images of sector periodicity are evaluated every step (their motion bound would need
      // the turn)
      if (live && !fresh && (cv[r].x > 0.f || cv[r].w > 0.f) && !(full && signbit(cv[r].z)) &&
          !(SEC && tv[r] >= PT_GX)) {
        float4 c = cv[r];
        c.z = fabsf(c.z);
        const bool flip = tv[r] >= PT_GX && ((key[r] >> kFlipBit) & 1);
        const float ex = mA[r].x - mB[r].x, ey = mA[r].y - mB[r].y, ez = mA[r].z - mB[r].z;
        if (!flip && c.x > 0.f) {
          // against the motion since the build (the slack net of the motion at the evaluation); a
          // pair that fails it is evaluated, which issues it a new certificate (checking it against
          // the motion since the evaluation instead would cost one more round trip)
          const float bound = (sqrtf(ex * ex + ey * ey + ez * ez) + mB[r].w * c.y + mA[r].w * c.z) * (1.f + 1e-5f);
          act = !(bound < c.x);
        } else if (c.x <= 0.f && c.w > 0.f) {
          // against the motion since the evaluation: the same bound with the displacement and the
          // rotations taken from that step
          float4 e0, qa0, qb0, qa, qb;
          if (r == early) {
            e0 = e0e; qa0 = qa0e; qb0 = qb0e; qa = qae; qb = qbe;
          } else {
            e0 = P.certE[p];
            qa0 = P.certQA[p];
            qb0 = P.certQB[p];
            qa = P.qrel[Av[r]];
            qb = tv[r] == PT_PW ? P.wQrel[jv[r]] : P.qrel[jv[r]];
          }
          if ((e0.w != 0.f) == flip) {
            const float fx = ex - e0.x, fy = ey - e0.y, fz = ez - e0.z;
            const float chA = relChordF(qa0, qa), chB = relChordF(qb0, qb);
            const float bound = (sqrtf(fx * fx + fy * fy + fz * fz) + chB * c.y + chA * c.z) * (1.f + 1e-5f);
            act = !(bound < c.w);
          }
        }
      }
      if (p < nPairs) {
        if (!live && rebuilt) P.cert[p] = make_float4(-1.f, 0.f, 0.f, -1.f);
        // a pair skipped under a certificate has had no contacts since the evaluation that issued
        // it (a pair with candidate nodes gets no certificate); others drop last step's count
        // (on a new list every count is the old list's)
        if (!act && (rebuilt || !(cv[r].x > 0.f || cv[r].w > 0.f))) P.pairCcnt[p] = 0;
      }
      actv[r] = act && p < nPairs;
    }
#pragma clang loop unroll(full)
    for (int r = 0; r < R; ++r) {
      const unsigned long long m = __ballot(actv[r]);
      int first = 0;
      if (lane == 0 && m) first = atomicAdd(&sCount, __popcll(m));
      first = __shfl(first, 0, 64);
      if (actv[r]) {
        const int slot = first + __popcll(m & ltMask);
        sList[slot] = pv[r];
        sInfo[slot] = (tv[r] << 28) | uint32_t(jv[r]);
        sA[slot] = Av[r];
      }
    }
    __syncthreads();
    // (a short list's reservation returns while the pairs' states are read: it is the last wavefront's, which
    // has a pair to read only when three quarters of the round are full; on a long one the others' reads hide it
    // and the records, kept over the barrier, cost 1 us of 37)
    const int count = sCount;
    if (threadIdx.x == (R == 1 ? 255 : 0) && count) sBase = region + atomicAdd(&evalCount(P)[xcd * kBarrierLine], count);
    if (R > 1) __syncthreads();
    for (int k0 = 0; k0 < count; k0 += 256) {
      const int k = k0 + int(threadIdx.x);
      const bool on = k < count;
      PairF32 f;
      float4 e0 = make_float4(0.f, 0.f, 0.f, 0.f), qA = e0, qB = e0;
      int p = 0;
      if (on) {
        p = sList[k];
        const PairView v = loadPair<SEC>(P, p, sInfo[k], sA[k]);
        // the motion state of this evaluation, for the pair's certificate against later motion
        // (loaded before the stores below)
        const BodyStep sa = P.step[v.A];
        qA = P.qrel[v.A];
        float4 mB;
        float flip = 0.f;
        if (v.type == PT_PW) {
          mB = P.wMotion[v.partner];
          qB = P.wQrel[v.partner];
        } else {
          const BodyStep sb = P.step[v.partner];
          mB = sb.motion;
          qB = P.qrel[v.partner];
          if (v.type >= PT_GX) flip = float((partnerKey(sb.key, v.type) >> kFlipBit) & 1);
        }
        makeF32(P, v, f);
        e0 = make_float4(sa.motion.x - mB.x, sa.motion.y - mB.y, sa.motion.z - mB.z, flip);
        evNodes += unsigned(v.nNodes);
      }
      if (R == 1) __syncthreads();  // sBase (one round)
      if (on) {
        const int a = sBase + k;
        out[a] = f;
        P.pairRec[p] = a;
        P.certE[p] = e0;
        P.certQA[p] = qA;
        P.certQB[p] = qB;
      }
    }
    __syncthreads();
  }
  // (only threads that wrote map records count: a few thousand atomics per step at 200k particles)
  if (__ballot(evNodes != 0)) {  // (one atomic per wavefront)
    const unsigned long long sum = (unsigned long long)wsum(double(evNodes));
    if (lane == 0) atomicAdd(statSlot(P, 4, blockIdx.x & (kStatSlots - 1)), sum);
  }
}
template <bool SEC>
__global__ __launch_bounds__(256) void k_pair_check(Params P, int full) {
  __shared__ CheckLds L;
  LSD_HALT_LATCH(P)  // (a failed broad phase leaves no pair list to read)
  // the broad phase of this step is over: its grid barrier's words start the next one at zero
  if (blockIdx.x == 0 && threadIdx.x < 10) P.barrier[threadIdx.x * kBarrierLine] = 0;
  const int nPairs = min(P.pairStart[P.nP], (int)P.pairCap);
  if (checkTileSize(nPairs) == kCheckTileShort) checkPairs<SEC, 1>(P, full, nPairs, L);
  else checkPairs<SEC, 4>(P, full, nPairs, L);
}

// The FP32 prefilters may contract a * b + c into one rounding: their margins bound the rounding
// of separate operations, and a fused operation rounds less.  (The FP64 membership tests keep the
// file-wide -ffp-contract=off.)
#define FP32_CONTRACT _Pragma("clang fp contract(fast)")

__device__ __forceinline__ void mapF32(const PairF32& f, float nx, float ny, float nz, float& gx, float& gy, float& gz) {
  FP32_CONTRACT
  gx = f.m[0] * nx + f.m[1] * ny + f.m[2] * nz + f.t[0];
  gy = f.m[3] * nx + f.m[4] * ny + f.m[5] * nz + f.t[1];
  gz = f.m[6] * nx + f.m[7] * ny + f.m[8] * nz + f.t[2];
}

// FP32 trilinear SDF value (unscaled) at grid coordinates g, clamped into the grid; a prefilter
// only.  Its rounding error is below 1e-6 of the largest |corner|, which the caller adds (kRelPhi).
constexpr float kRelPhi = 4e-6f;
__device__ __forceinline__ float phiF32(const float* __restrict__ sdf, const PairF32& f, float gx, float gy, float gz,
                                        float& cmax) {
  FP32_CONTRACT
  const int i0 = min(max(int(floorf(gx)), 0), f.nx - 2), j0 = min(max(int(floorf(gy)), 0), f.ny - 2),
            k0 = min(max(int(floorf(gz)), 0), f.nz - 2);
  const float x = fminf(fmaxf(gx - float(i0), 0.f), 1.f), y = fminf(fmaxf(gy - float(j0), 0.f), 1.f),
              z = fminf(fmaxf(gz - float(k0), 0.f), 1.f);
  const int sx = 1, sy = f.nx, sz = f.nx * f.ny;
  const float* g = sdf + f.sdfOff + i0 + j0 * sy + k0 * sz;
  const float c000 = g[0], c100 = g[sx], c010 = g[sy], c110 = g[sx + sy];
  const float c001 = g[sz], c101 = g[sx + sz], c011 = g[sy + sz], c111 = g[sx + sy + sz];
  cmax = fmaxf(fmaxf(fmaxf(fabsf(c000), fabsf(c100)), fmaxf(fabsf(c010), fabsf(c110))),
               fmaxf(fmaxf(fabsf(c001), fabsf(c101)), fmaxf(fabsf(c011), fabsf(c111))));
  const float a = (c000 * (1.f - x) + c100 * x) * (1.f - y) + (c010 * (1.f - x) + c110 * x) * y;
  const float b = (c001 * (1.f - x) + c101 * x) * (1.f - y) + (c011 * (1.f - x) + c111 * x) * y;
  return a * (1.f - z) + b * z;
}

// Cluster acceptance (conservative): the cluster's bounding sphere must reach the partner's
// bounding sphere (particle partners) and grid box, and, when its centre lies in the box, the
// partner's SDF at the centre must be within Lipschitz reach of zero.
//
// Every test below is a function of the g coordinates of A's nodes alone (the partner's sphere,
// box and SDF are fixed in its frame).  When a test culls, `slack` (g units) is how far the
// cluster's radius could grow with the same test still culling it: while no node has moved
// further than that in the partner's frame, the test still rules out every node of the cluster.
// Slacks are rounded down; a cull that holds by less than the rounding gives a slack <= 0.

// A slack is rounded down by kSlackRound, which covers the FP32 rounding of computing it (a few
// ulps of the distances involved).  The rounding of the map itself needs no allowance: every
// threshold already contains it (the margins abs, phiMargin), so a test that fails with a radius
// grown by the slack fails for every exact point of the grown ball.
constexpr float kSlackRound = 1.f - 2e-6f;

// Geometric part: bounding spheres and grid box.  `inside` reports whether the centre lies in the
// grid box (then an SDF bound at the centre can cull the cluster).
__device__ __forceinline__ bool clusterGeomF32(const PairF32& f, const ClusterF32& cl, float& gx, float& gy, float& gz,
                                               float& rho, bool& inside, float& slack) {
  FP32_CONTRACT
  mapF32(f, cl.cx, cl.cy, cl.cz, gx, gy, gz);
  rho = cl.rho * f.rhoScale;
  inside = false;
  slack = 0.f;
  if (f.r2 >= 0.f) {
    const float dx = gx - f.c[0], dy = gy - f.c[1], dz = gz - f.c[2];
    const float d2 = dx * dx + dy * dy + dz * dz;
    const float r = sqrtf(f.r2) + rho;
    if (d2 > r * r * 1.0001f) {
      slack = sqrtf(d2) * kSlackRound - r * 1.00005f;
      return false;
    }
  }
  const float dx = fmaxf(0.f, fmaxf(f.lo - gx, gx - boxHi(f, f.nx)));
  const float dy = fmaxf(0.f, fmaxf(f.lo - gy, gy - boxHi(f, f.ny)));
  const float dz = fmaxf(0.f, fmaxf(f.lo - gz, gz - boxHi(f, f.nz)));
  const float d2 = dx * dx + dy * dy + dz * dz;
  if (d2 > rho * rho * 1.0001f) {
    slack = sqrtf(d2) * kSlackRound - rho * 1.00005f;
    return false;
  }
  inside = dx == 0.f && dy == 0.f && dz == 0.f;
  return true;
}
// Radius growth that a Lipschitz bound phi > lipH * 1.001 * radius + lim still allows.
__device__ __forceinline__ float lipSlack(const PairF32& f, float phi, float lim, float rho) {
  FP32_CONTRACT
  // hardware reciprocal (1 ulp), covered by kSlackRound
  return f.lipH > 0.f ? (phi - lim) * __builtin_amdgcn_rcpf(f.lipH * 1.001f) * kSlackRound - rho : 0.f;
}
// SDF part with the exact grid: phi(centre) beyond Lipschitz reach of zero culls the cluster.
__device__ __forceinline__ bool clusterSdfF32(const float* __restrict__ sdf, const PairF32& f, float gx, float gy,
                                              float gz, float rho, float& slack) {
  FP32_CONTRACT
  float cmax;
  const float phi = phiF32(sdf, f, gx, gy, gz, cmax);
  const float lim = f.phiMargin + kRelPhi * cmax;
  if (phi > f.lipH * rho * 1.001f + lim) {
    slack = lipSlack(f, phi, lim, rho);
    return false;
  }
  return true;
}
__device__ __forceinline__ bool clusterF32(const float* __restrict__ sdf, const PairF32& f, const ClusterF32& cl,
                                           bool sdfCull) {
  float gx, gy, gz, rho, slack;
  bool inside;
  if (!clusterGeomF32(f, cl, gx, gy, gz, rho, inside, slack)) return false;
  return !inside || !sdfCull || clusterSdfF32(sdf, f, gx, gy, gz, rho, slack);
}
// Surrogate part: the same bound with the learned distance, widened by the band (twice the
// surrogate's measured maximum error).  `d` is the network output in normalised units.
__device__ __forceinline__ bool clusterSurKeep(const Params& P, const PairF32& f, float d, float rho) {
  const float phi = d * (1.0f / P.sur.invLen);
  return !(phi - P.surBand > f.lipH * rho * 1.001f + f.phiMargin);
}
__device__ __forceinline__ float clusterSurSlack(const Params& P, const PairF32& f, float d, float rho) {
  return lipSlack(f, d * (1.0f / P.sur.invLen), P.surBand + f.phiMargin, rho);
}
// Lane's surrogate query for a cluster centre at grid coordinates g (normalised local point).
__device__ __forceinline__ void surQueryPoint(const Params& P, const PairF32& f, float gx, float gy, float gz,
                                              float& ux, float& uy, float& uz) {
  ux = (f.o[0] + gx * f.h) * P.sur.invLen;
  uy = (f.o[1] + gy * f.h) * P.sur.invLen;
  uz = (f.o[2] + gz * f.h) * P.sur.invLen;
}
// Node acceptance (conservative superset of the exact FP64 test); slack as for clusters, with
// the node as a cluster of radius 0.
__device__ __forceinline__ bool nodeF32(const float* __restrict__ sdf, const PairF32& f, float4 n, float& slack) {
  FP32_CONTRACT
  float gx, gy, gz;
  mapF32(f, n.x, n.y, n.z, gx, gy, gz);
  slack = 0.f;
  if (f.r2 >= 0.f) {
    const float dx = gx - f.c[0], dy = gy - f.c[1], dz = gz - f.c[2];
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > f.r2) {
      slack = sqrtf(d2) * kSlackRound - sqrtf(f.r2);
      return false;
    }
  }
  const float out = fmaxf(fmaxf(fmaxf(f.lo - gx, gx - boxHi(f, f.nx)), fmaxf(f.lo - gy, gy - boxHi(f, f.ny))),
                          fmaxf(f.lo - gz, gz - boxHi(f, f.nz)));
  if (out > 0.f) {  // outside the grid box on some axis, by `out`
    slack = out * kSlackRound;
    return false;
  }
  float cmax;
  const float phi = phiF32(sdf, f, gx, gy, gz, cmax);
  const float lim = f.phiMargin + kRelPhi * cmax;
  if (phi <= lim) return true;
  slack = lipSlack(f, phi, lim, 0.f);
  return false;
}

// nodeF32 in three stages, so that the grid reads of several nodes can be in flight together:
// the sphere and box tests (slack when they cull), the eight corner reads, the SDF test.
__device__ __forceinline__ bool nodeGeomF32(const PairF32& f, float4 n, float& gx, float& gy, float& gz, float& slack) {
  FP32_CONTRACT
  mapF32(f, n.x, n.y, n.z, gx, gy, gz);
  slack = 0.f;
  if (f.r2 >= 0.f) {
    const float dx = gx - f.c[0], dy = gy - f.c[1], dz = gz - f.c[2];
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (d2 > f.r2) {
      slack = sqrtf(d2) * kSlackRound - sqrtf(f.r2);
      return false;
    }
  }
  const float out = fmaxf(fmaxf(fmaxf(f.lo - gx, gx - boxHi(f, f.nx)), fmaxf(f.lo - gy, gy - boxHi(f, f.ny))),
                          fmaxf(f.lo - gz, gz - boxHi(f, f.nz)));
  if (out > 0.f) {
    slack = out * kSlackRound;
    return false;
  }
  return true;
}
__device__ __forceinline__ void sdfCorners(const float* __restrict__ sdf, const PairF32& f, float gx, float gy, float gz,
                                           float (&c)[8], float& x, float& y, float& z) {
  FP32_CONTRACT
  const int i0 = min(max(int(floorf(gx)), 0), f.nx - 2), j0 = min(max(int(floorf(gy)), 0), f.ny - 2),
            k0 = min(max(int(floorf(gz)), 0), f.nz - 2);
  x = fminf(fmaxf(gx - float(i0), 0.f), 1.f);
  y = fminf(fmaxf(gy - float(j0), 0.f), 1.f);
  z = fminf(fmaxf(gz - float(k0), 0.f), 1.f);
  const int sx = 1, sy = f.nx, sz = f.nx * f.ny;
  const float* g = sdf + f.sdfOff + i0 + j0 * sy + k0 * sz;
  c[0] = g[0]; c[1] = g[sx]; c[2] = g[sy]; c[3] = g[sx + sy];
  c[4] = g[sz]; c[5] = g[sx + sz]; c[6] = g[sy + sz]; c[7] = g[sx + sy + sz];
}
// Same arithmetic as phiF32 and the SDF part of nodeF32.
__device__ __forceinline__ bool nodeSdfF32(const PairF32& f, const float (&c)[8], float x, float y, float z,
                                           float& slack) {
  FP32_CONTRACT
  const float cmax = fmaxf(fmaxf(fmaxf(fabsf(c[0]), fabsf(c[1])), fmaxf(fabsf(c[2]), fabsf(c[3]))),
                           fmaxf(fmaxf(fabsf(c[4]), fabsf(c[5])), fmaxf(fabsf(c[6]), fabsf(c[7]))));
  const float a = (c[0] * (1.f - x) + c[1] * x) * (1.f - y) + (c[2] * (1.f - x) + c[3] * x) * y;
  const float b = (c[4] * (1.f - x) + c[5] * x) * (1.f - y) + (c[6] * (1.f - x) + c[7] * x) * y;
  const float phi = a * (1.f - z) + b * z;
  const float lim = f.phiMargin + kRelPhi * cmax;
  if (phi <= lim) return true;
  slack = lipSlack(f, phi, lim, 0.f);
  return false;
}

// Exact test and contact law of one candidate slot: the reference's node-vs-SDF membership in
// FP64, then (for contacts) tangential history and the linear spring-dashpot.  f, X: the pair's records in
// LDS; info: its list entry; node: the candidate in cluster order.  Returns whether the slot is a contact;
// out: its force and torque on the master, torque on the partner.
struct SlotTerms {
  d3 F, TA, TB;
};
__device__ __forceinline__ bool exactSlot(const Params& P, int c, const PairF32& f, const PairExact& X, uint32_t info,
                                          int node, SlotTerms& out, unsigned int& statQueries,
                                          unsigned int& statContacts) {
  const NodeDev nd = P.nodes[node];
  const uint32_t type = info >> 28;
  // tangential history of the same (list, node, partner) from the previous step (its first slot is read
  // with the SDF's corners); this step's contact goes into this step's table for the next one
  const int gnode = reinterpret_cast<const int*>(X.side[0].prop + kPropInts)[0] + nd.orig;
  const unsigned long long key = histKey(type, gnode, int(info & kPartnerMask));
  const unsigned long long slot0 = mix64(key) & P.hashMask;
  const unsigned long long k0 = P.prevHashKey[slot0];
  const int v0 = P.prevHashVal[slot0];
  NodeHit h;
  if (!exactTest(P, X, type, mk3(nd.x, nd.y, nd.z), i3{f.nx, f.ny, f.nz}, f.sdfOff, h, statQueries)) {
    P.cInfo[c] = kInvalidInfo;
    P.hashSlot[c] = -1;
    return false;
  }
  statContacts++;
  d3 spring = histLookup(P, key, slot0, k0, v0);
  // (the slot's stores after every load above)
  P.cInfo[c] = info;
  P.cNode[c] = gnode;
  P.cPoint[c] = h.point;
  P.cNormal[c] = h.normal;
  P.cOverlap[c] = h.ov;
  P.hashSlot[c] = histInsert(P, key, c);
  d3 F = mk3(0., 0., 0.);
  if (P.prime) {
    // the pre-loop build only lists the contact with the spring it found
    // (LSParticleContactDetectionKernel.cu:280-289); the force kernels do not run
    P.cSpring[c] = spring;
    P.cEn[c] = 0.;
    P.cEs[c] = 0.;
    out = SlotTerms{F, F, F};
    return true;
  }
  // (the real body's angular velocity for an image, contactKernel.cu:236-238)
  const BodySide &A = X.side[0], &B = X.side[1];
  const d3 armA = h.point - lds3(A.v[kSvPos]), armB = h.point - lds3(B.v[kSvPos]);
  const d3 vc = lds3(A.v[kSvVel]) + cross(lds3(A.v[kSvAng]), armA) - (lds3(B.v[kSvVel]) + cross(lds3(B.v[kSvAng]), armB));
  const double kn = X.law[0], ks = X.law[1];
  const ContactLaw law = linearContact(spring, vc, h.normal, h.ov, P.dt, kn, ks, X.law[2], X.law[3], X.law[4]);
  F = law.F;
  spring = law.spring;
  P.cSpring[c] = spring;
  P.cEn[c] = 0.5 * h.ov * h.ov * kn;
  P.cEs[c] = 0.5 * len2(spring) * ks;
  out = SlotTerms{F, cross(armA, F), cross(armB, -F)};
  return true;
}

// One lane's share of a pair's PairExact record: 8 lanes fill a record, 4 per body.  Lane t of a body reads
// its t-th state vector, the t-th component of its orientation and the t-th quarter of its properties; the
// state vectors of particles, walls and images lie in one block, so a lane's address needs no choice
// between arrays.  All reads of a record are in flight together (one round trip).
struct PairShare {
  double v[3], q, prop[4];
  int key;
};
template <bool SEC>
__device__ __forceinline__ PairShare readShare(const Params& P, uint32_t info, int A, int k) {
  const uint32_t type = info >> 28;
  const int j = int(info & kPartnerMask), t = k & 3;
  const bool B = k >= 4, wall = type == PT_PW, ghost = type >= PT_GX;
  const int g = int(type) - int(PT_GX);
  const int idx = !B ? A : wall ? P.nP + j : j;
  int vSlot = t, qSlot = 0;
  if (B && wall && t == kSvDet) vSlot = kSvPos;  // (as loadPair)
  if (B && ghost && t < 2) vSlot = kSvImg + g;
  if (SEC) {
    if (B && ghost && t == kSvVel) vSlot = kSvImgVel + g;
    qSlot = ghost ? (B ? 2 + g : 0) : (B && wall ? 0 : 1);
  }
  const double* v = reinterpret_cast<const double*>(P.pos + ((long long)vSlot * P.nBodies + idx));
  const double* q = reinterpret_cast<const double*>(P.quat + ((long long)qSlot * P.nBodies + idx));
  const double* prop = reinterpret_cast<const double*>(P.prop + idx) + 4 * t;
  PairShare r;
  r.v[0] = v[0]; r.v[1] = v[1]; r.v[2] = v[2];
  r.q = q[t];
  r.prop[0] = prop[0]; r.prop[1] = prop[1]; r.prop[2] = prop[2]; r.prop[3] = prop[3];
  r.key = 0;
  if (k == 4 && type != PT_PP)
    r.key = *(wall ? P.wkey + j : reinterpret_cast<const int*>(P.step + j) + 5 + g);  // (BodyStep::key from its y on)
  return r;
}
__device__ __forceinline__ void writeShare(const PairShare& r, uint32_t info, int k, PairExact& X) {
  const int t = k & 3;
  BodySide& S = X.side[k >> 2];
  S.v[t][0] = r.v[0]; S.v[t][1] = r.v[1]; S.v[t][2] = r.v[2];
  S.q[t] = r.q;
  S.prop[4 * t] = r.prop[0]; S.prop[4 * t + 1] = r.prop[1]; S.prop[4 * t + 2] = r.prop[2]; S.prop[4 * t + 3] = r.prop[3];
  // (an image's key carries its shift-flip bit)
  if (k == 4) X.keyB = ((info >> 28) == PT_PW || r.key < 0) ? r.key : (r.key & ~(1 << kFlipBit));
}
// The contact law's constants, once per pair (the master's own stiffnesses and mass against a wall, whose
// properties hold zeros there): lane k of the pair's 8 takes constant k.
__device__ __forceinline__ void pairLaw(uint32_t info, int k, PairExact& X) {
  if (k >= 5) return;
  const bool wall = (info >> 28) == PT_PW;
  const int at = k == 0 ? kPropKn : k == 1 ? kPropKs : k == 2 ? kPropMu : k == 3 ? kPropDiss : kPropInvM;
  const double a = X.side[0].prop[at], b = X.side[1].prop[at];
  const double resA = X.side[0].prop[kPropRes], resB = X.side[1].prop[kPropRes];
  const double quot = (k < 2 ? a * b : 1.) / (a + b);
  double c;
  if (k < 2) c = wall ? a : (a > 0. && b > 0. ? quot : 0.);              // stiffnesses in series
  else if (k == 2) c = fmin(a, b);
  else if (k == 3) c = (resA <= resB || resB != resB) ? a : b;           // of the smaller restitution
  else c = (a > 0. || b > 0.) ? quot : 0.;                               // 1 / (1 / m_A + 1 / m_B)
  X.law[k] = c;
}

// Dissipation of each particle's and wall's restitution for the contact law (once, at initialisation).
__global__ void k_dissipation(BodyProp* prop, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) prop[i].diss = dissipation(prop[i].res);
}

constexpr int kBatch = 8;  // candidate pairs per wave batch
constexpr int kMaxSub = 4;  // sub-clusters per cluster (64 / 16)
constexpr int kSlotStage = 128;  // candidate slots of a batch handed to the exact test through LDS

// Per-wave LDS of k_candidates: pair maps, surviving (pair, cluster) entries, surviving
// (pair, sub-cluster) entries with their 16-bit node masks, per-pair counts, offsets and slacks.
__host__ __device__ inline int candWaveBytes(int maxClusters) {
  const int nEnt = kBatch * maxClusters, nSub = kMaxSub * nEnt;
  const int b = int(sizeof(PairF32)) * kBatch + int(sizeof(PairExact)) * kBatch + 8 * kSlotStage + 16 * kBatch +
                8 * nEnt + 8 * nSub + 4 * nSub;
  return (b + 15) & ~15;
}
size_t candidatesLdsBytes(int maxClusters) { return size_t(candWaveBytes(maxClusters)) * (kNarrowBlock / 64); }

// Value of another lane of the same 16-lane row (every lane active).
template <int CTRL>
__device__ __forceinline__ float dppMove(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
// Minimum over aligned groups of W lanes (4, 8 or 16).
template <int W>
__device__ __forceinline__ float groupMin(float v) {
  // lane exchanges within 16-lane rows (DPP): quad permutations, half-row mirror, row rotations
  static_assert(W == 4 || W == 8 || W == 16, "group of 4, 8 or 16 lanes");
  v = fminf(v, dppMove<0xB1>(v));  // quad_perm [1,0,3,2]
  v = fminf(v, dppMove<0x4E>(v));  // quad_perm [2,3,0,1]: min of the quad
  if (W == 8) v = fminf(v, dppMove<0x141>(v));  // row_half_mirror: the other quad of the 8
  if (W == 16) {
    v = fminf(v, dppMove<0x124>(v));  // row_ror 4
    v = fminf(v, dppMove<0x128>(v));  // row_ror 8
  }
  return v;
}

// Candidate nodes: one wavefront per batch of up to 8 evaluated pairs, three levels of conservative
// FP32 culls, then the exact test of what is left.  Bound by each wavefront's chain of round trips (about 9
// with the exact test) and by how many wavefronts share a SIMD: 150 registers, 3 wavefronts (256 and 2 when
// every lane of the exact test loaded its pair's state itself; 101 us then and 74 now for 200,000 falling bodies that
// evaluate some 15,000 pairs a step, 184 and 146 us for an ordered bed that evaluates 80,000, the block-wide
// reservations below included, 20 and 19 us for a falling column of 20,000).  A limit of 128 registers spills 24 and LDS has no room for a
// fourth wavefront.
//   1. lanes = (pair, cluster of <= 64 nodes): bounding spheres, grid box, SDF Lipschitz bound at
//      the cluster centre (or the surrogate's decision); survivors become entries;
//   2. lanes = (entry, sub-cluster of <= 16 nodes), 16 entries per pass: the same tests with the
//      sub-cluster's smaller sphere; survivors become sub-entries;
//   3. lanes = (sub-entry, node), 4 sub-entries per pass: the node prefilter.
// The batch reserves its exact candidate count with one atomic and numbers each pair's candidates
// consecutively, in (cluster, sub-cluster, node) order.  Every node of a pair is ruled
// out by exactly one cull (cluster, sub-cluster or node) or becomes a candidate; the smallest
// slack of those culls, less the rounding of the map, is the pair's separation certificate
// (none when a node is a candidate).
template <bool SUR, bool SEC>
__global__ __launch_bounds__(kNarrowBlock, 3) void k_candidates(Params P) {
  extern __shared__ __align__(16) unsigned char candLds[];
  const int lane0 = threadIdx.x & 63, wl = threadIdx.x >> 6;
  const int maxC = P.maxClusters;
  const int entCap = kBatch * maxC, subCap = kMaxSub * entCap;
  unsigned char* wb = candLds + wl * candWaveBytes(maxC);
  PairF32* sF = reinterpret_cast<PairF32*>(wb);
  PairExact* sX = reinterpret_cast<PairExact*>(sF + kBatch);
  int2* sStage = reinterpret_cast<int2*>(sX + kBatch);           // (batch pair, node) of the first slots
  int* sCnt = reinterpret_cast<int*>(sStage + kSlotStage);       // candidates of each pair
  int* sOff = sCnt + kBatch;                                     // next free slot of each pair
  int* sHits = sOff + kBatch;                                    // contacts of each pair
  unsigned int* sSlack = reinterpret_cast<unsigned int*>(sHits + kBatch);  // bits of a float >= 0
  int2* sEnt = reinterpret_cast<int2*>(sSlack + kBatch);         // (first sub-cluster, count | pair j << 4)
  int2* sSub = sEnt + entCap;                                    // (first node, count | j << 16)
  unsigned int* sMask = reinterpret_cast<unsigned int*>(sSub + subCap);  // 16-bit node masks, then also first slot << 16
  static_assert(kBatch * 4096 <= 65536, "a batch's slot offsets fit 16 bits (shapes have at most 4096 nodes)");
  const float kInf = __builtin_huge_valf();
  __shared__ int sTotal[kNarrowBlock / 64], sFirst;
  LSD_HALT_LATCHED(P);
  unsigned int statCand = 0, statEnt = 0, statQueries = 0, statContacts = 0;
  const EvalRecords rec = evalRecords(P);
  const int nAct = rec.n;
  const int wave = __builtin_amdgcn_readfirstlane(int(blockIdx.x * (kNarrowBlock / 64) + wl));
  const int nWaves = int(gridDim.x * (kNarrowBlock / 64));
  if (wave == 0 && lane0 == 0) P.devStat[13] += (unsigned long long)nAct;  // evaluated pairs, summed over steps
  const int iters = (maxC + 7) >> 3;
  // batch bi takes the evaluated pairs bi, bi + NB, bi + 2 NB, ...: pairs near contact come in
  // spatial runs, and spreading them over the batches keeps the slowest wavefront short
  // pairs per batch: the smallest number whose batches are all on the GPU together, which spreads the slowest
  // pairs (those near contact, with many surviving clusters) over the most wavefronts; eight beyond that, since
  // the lanes of a batch of eight are all used.  (One only from eight wavefronts per pair on, two from two: 11.2
  // ms for 200 steps of 1,000 bodies in a box, now 10.3; 4.14 and 3.98 for 50 of 27; others within 2 %.)
  const int fit = min(nWaves, P.residentWaves);
  const int nb = P.narrowBatch > 0 ? P.narrowBatch
                                   : (nAct <= fit ? 1 : (nAct <= 2 * fit ? 2 : (nAct <= 4 * fit ? 4 : kBatch)));
  const int NB = (nAct + nb - 1) / nb;
  // (the block's wavefronts turn together: each turn reserves for all four; one past the last batch has no pairs)
  for (int b0 = int(blockIdx.x * (kNarrowBlock / 64)); b0 < NB; b0 += nWaves) {
    const int bi = b0 + wave % (kNarrowBlock / 64);
    const int nAct = bi < NB ? rec.n : 0;
    // (what follows from the lane is worked out in each batch: kept in registers through the loop, the
    // addresses of every stage together take half of a wavefront's registers)
    const int lane = inLoop(lane0, bi);
    const int j = lane >> 3, k = lane & 7, q = lane >> 4, b16 = lane & 15;
    const unsigned int lt16 = (1u << b16) - 1u;
    const unsigned long long ltMask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    // ---- level 1: clusters ----
    const int a = bi + j * NB;  // map record
    const bool own = j < nb && a < nAct;
    // the 8 lanes of a pair copy its 160-byte map record into LDS, 20 bytes each
    if (own) {
      const unsigned int* src = reinterpret_cast<const unsigned int*>(P.pairMap) + (long long)rec.at(a) * 40 + 5 * k;
      unsigned int* dst = reinterpret_cast<unsigned int*>(&sF[j]) + 5 * k;
#pragma unroll
      for (int w = 0; w < 5; ++w) dst[w] = src[w];
    }
    if (lane < kBatch) sCnt[lane] = 0;
    __builtin_amdgcn_wave_barrier();
    const PairF32& f = sF[j];
    const int clusterOff = own ? f.clusterOff : 0, nCl = own ? f.nClusters : 0;
    int E = 0;
    float lmin = kInf;  // smallest slack of this lane's culled clusters
    for (int it = 0; it < iters; ++it) {
      const int c = it * 8 + k;
      bool keep = false;
      int subFirst = 0, nSub = 0;
      if (own && c < nCl) {
        const ClusterF32 cl = P.clusters32[clusterOff + c];
        subFirst = cl.subFirst;
        nSub = cl.nSub;
        float gx, gy, gz, rho, slack;
        bool inside;
        keep = clusterGeomF32(f, cl, gx, gy, gz, rho, inside, slack);
        if (keep && inside) {
          if (SUR && f.slot >= 0) keep = (P.surMask[a] >> c) & 1ull;  // slack: surSlack
          else if (P.sdfCull) keep = clusterSdfF32(P.sdf, f, gx, gy, gz, rho, slack);
          if (!keep && SUR && f.slot >= 0) slack = kInf;
        }
        if (!keep) lmin = fminf(lmin, fmaxf(slack, 0.f));
      }
      const unsigned long long m = __ballot(keep);
      // (the entry carries the cluster's sub-cluster range: level 2 reads no cluster record)
      if (keep) sEnt[E + __popcll(m & ltMask)] = make_int2(subFirst, nSub | (j << 4));
      E += __popcll(m);
    }
    lmin = groupMin<8>(lmin);
    if (k == 0) sSlack[j] = __float_as_uint(lmin);
    statEnt += (lane == 0) ? unsigned(E) : 0u;
    __builtin_amdgcn_wave_barrier();
    // ---- level 2: sub-clusters, 16 entries x 4 per pass ----
    int NS = 0;
    for (int e0 = 0; e0 < E; e0 += 16) {
      const int e = e0 + (lane >> 2), u = lane & 3;
      bool keep = false;
      float smin = kInf;
      int first = 0, count = 0, jj = 0;
      if (e < E) {
        const int2 en = sEnt[e];
        jj = en.y >> 4;
        if (u < (en.y & 15)) {
          const ClusterF32 sc = P.subs32[en.x + u];
          const PairF32& fj = sF[jj];
          float gx, gy, gz, rho, slack;
          bool inside;
          keep = clusterGeomF32(fj, sc, gx, gy, gz, rho, inside, slack);
          // with the surrogate the network has decided on the whole cluster; the sub-cluster keeps
          // only its geometric tests then
          if (keep && inside && !(SUR && fj.slot >= 0) && P.sdfCull)
            keep = clusterSdfF32(P.sdf, fj, gx, gy, gz, rho, slack);
          if (!keep) smin = fmaxf(slack, 0.f);
          first = fj.nodeOff + sc.first;
          count = sc.count;
        }
      }
      smin = groupMin<4>(smin);  // the 4 lanes of an entry share its pair
      if (e < E && (lane & 3) == 0 && smin < kInf) atomicMin(&sSlack[jj], __float_as_uint(smin));
      const unsigned long long m = __ballot(keep);
      if (keep) sSub[NS + __popcll(m & ltMask)] = make_int2(first, count | (jj << 16));
      NS += __popcll(m);
    }
    __builtin_amdgcn_wave_barrier();
    // ---- level 3: nodes, 4 sub-entries x 16 per pass, two passes per iteration: the node loads,
    // then the grid reads of the nodes that pass the sphere and box tests, are issued for both
    // passes before either is used; the next iteration's node loads are issued before this
    // iteration's tests ----
    int total = 0;
    int jjn[2];
    bool liven[2];
    float4 ndn[2];
    auto loadNodes = [&](int e0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = e0 + 4 * h + q;
        jjn[h] = 0;
        liven[h] = false;
        ndn[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e < NS) {
          const int2 se = sSub[e];
          jjn[h] = se.y >> 16;
          liven[h] = b16 < (se.y & 0xFFFF);
          if (liven[h]) ndn[h] = P.nodes32[se.x + b16];
        }
      }
    };
    if (NS > 0) loadNodes(0);
    for (int e0 = 0; e0 < NS; e0 += 8) {
      int jjv[2];
      bool live[2], geo[2];
      float4 nd[2];
      float gx[2], gy[2], gz[2], sl[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        jjv[h] = jjn[h];
        live[h] = liven[h];
        nd[h] = ndn[h];
      }
      if (e0 + 8 < NS) loadNodes(e0 + 8);
#pragma unroll
      for (int h = 0; h < 2; ++h) geo[h] = live[h] && nodeGeomF32(sF[jjv[h]], nd[h], gx[h], gy[h], gz[h], sl[h]);
      float cc[2][8], fx[2], fy[2], fz[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (geo[h]) sdfCorners(P.sdf, sF[jjv[h]], gx[h], gy[h], gz[h], cc[h], fx[h], fy[h], fz[h]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = e0 + 4 * h + q;
        bool cand = false;
        float smin = kInf;
        if (live[h]) {
          float slack = sl[h];
          if (geo[h]) cand = nodeSdfF32(sF[jjv[h]], cc[h], fx[h], fy[h], fz[h], slack);
          smin = cand ? 0.f : fmaxf(slack, 0.f);
        }
        smin = groupMin<16>(smin);  // the 16 lanes of a sub-entry share its pair
        const unsigned long long m = __ballot(cand);
        const unsigned int mq = unsigned((m >> (16 * q)) & 0xFFFFull);
        if (b16 == 0 && e < NS) {
          sMask[e] = mq;
          atomicAdd(&sCnt[jjv[h]], __popc(mq));  // LDS: 4 groups may share a pair
          if (smin < kInf) atomicMin(&sSlack[jjv[h]], __float_as_uint(smin));
        }
        total += __popcll(m);
      }
    }
    __builtin_amdgcn_wave_barrier();
    // ---- one reservation per turn of the block, exact size, and the reads of what the exact tests need: in
    // flight together, used after the certificates and the list of slots are done.  (Returning atomics on one
    // address are served 11 ns apart: one per batch was 8.7 us of the kernel's 32 for 794 batches that arrive
    // together, now 25 in all; an ordered bed of 10,000 batches 157 -> 147.) ----
    if (lane == 0) sTotal[wl] = total;
    __syncthreads();
    int ahead = 0, blockTotal = 0, blockFirst = 0;
#pragma unroll
    for (int w = 0; w < kNarrowBlock / 64; ++w) {
      const int t = sTotal[w];
      ahead += w < wl ? t : 0;
      blockTotal += t;
    }
    if (blockTotal > 0 && threadIdx.x == 0) blockFirst = atomicAdd(&P.devInt[1], blockTotal);
    const bool mine = lane < nb && bi + lane * NB < nAct;
    const bool share = own && sCnt[j] > 0;
    PairShare part{};
    if (share) part = readShare<SEC>(P, sF[j].info, sF[j].A, k);
    // the pair's place in its master's list and in its partner's reaction list
    int masterFirst = 0, rcSlot = -1, rcFirst = 0;
    if (mine && sCnt[lane] > 0) {
      const uint32_t info = sF[lane].info, type = info >> 28;
      const int B = int(info & kPartnerMask);
      masterFirst = P.pairStart[sF[lane].A];
      if (type == PT_PP || (type >= PT_GX && B != sF[lane].A)) {
        rcSlot = P.rcSlot[sF[lane].pair];
        rcFirst = P.rcStart[B];
      }
    }
    if (mine) {
      const PairF32& fl = sF[lane];
      // separation certificate in world units, net of the motion since the build
      float sg = __uint_as_float(sSlack[lane]);
      bool surDep = false;  // the surrogate's slack is the smaller one
      if (SUR) {
        const float ss = P.surSlack[bi + lane * NB];
        if (ss < sg) {
          sg = ss;
          surDep = true;
        }
      }
      float sw = -1.f, s0 = -1.f;
      const float sgr = sg * (1.f - 1e-5f) - 1e-6f;  // g units; the map's rounding is in the thresholds
      if (sgr > 0.f && P.useCert) {
        s0 = sgr * fl.gToWorld * (1.f - 1e-5f);
        sw = (sgr * fl.gToWorld - fl.certD0) * (1.f - 1e-5f);
      }
      // (the sign of .z marks a certificate that rests on the surrogate's slack)
      P.cert[fl.pair] = make_float4(sw > 0.f ? sw : -1.f, fl.certCB, surDep ? -fl.certCA : fl.certCA,
                                    s0 > 0.f ? s0 : -1.f);
    }
    int contacts = 0;  // contacts of this lane's pair
    if (total > 0) {
      // ---- slots, relative to the batch's first: a pair's candidates are contiguous, in (cluster,
      // sub-cluster, node) order.  Lanes = sub-entries: an entry's first slot is its pair's next free one
      // plus the candidates of the pair's entries before it, counted bit by bit across the wavefront ----
      if (mine) {
        int off = 0;
        for (int jj = 0; jj < lane; ++jj) off += sCnt[jj];
        sOff[lane] = off;
        sHits[lane] = 0;
      }
      __builtin_amdgcn_wave_barrier();
      for (int e0 = 0; e0 < NS; e0 += 64) {
        const int e = e0 + lane;
        const unsigned int mq = e < NS ? sMask[e] : 0u;
        const int jj = e < NS ? sSub[e].y >> 16 : 0, n = __popc(mq);
        unsigned long long same = ~0ull;  // the lanes with an entry of the same pair
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const unsigned long long m = __ballot((jj >> b) & 1);
          same &= (jj >> b) & 1 ? m : ~m;
        }
        int before = 0, all = 0;
#pragma unroll
        for (int b = 0; b < 5; ++b) {
          const unsigned long long m = __ballot((n >> b) & 1) & same;
          before += __popcll(m & ltMask) << b;
          all += __popcll(m) << b;
        }
        const int base = sOff[jj] + before;
        if (e < NS) sMask[e] = mq | unsigned(base) << 16;
        __builtin_amdgcn_wave_barrier();
        if (e < NS && (same & ltMask) == 0) sOff[jj] += all;  // (the pair's first lane)
        __builtin_amdgcn_wave_barrier();
      }
      if (share) {
        writeShare(part, sF[j].info, k, sX[j]);
        __builtin_amdgcn_wave_barrier();
        pairLaw(sF[j].info, k, sX[j]);
      }
    }
    if (threadIdx.x == 0) sFirst = blockFirst;
    __syncthreads();
    const int first = __builtin_amdgcn_readfirstlane(sFirst + ahead);
    if (total > 0) {
      // (a negative first: more than 2^31 slots asked for this step)
      if (first < 0 || (long long)first + total > P.contactCap) {
        // the call halts with a capacity error; slots reserved below the capacity stay empty
        if (lane == 0) {
          atomicMax(&P.devInt[5], int(min((long long)first + total, 0x7fffffffll)));
          raiseError(P, kErrContacts);
        }
        for (int c = first + lane; first >= 0 && c < (int)P.contactCap; c += 64) {
          if (c - first >= total) break;
          P.cInfo[c] = kInvalidInfo;
          P.hashSlot[c] = -1;
        }
        total = 0;
      }
    }
    if (total > 0) {
      for (int e0 = 0; e0 < NS; e0 += 4) {
        const int e = e0 + q;
        if (e < NS) {
          const unsigned int mq = sMask[e];
          if ((mq >> b16) & 1u) {
            const int2 se = sSub[e];
            const int r = int(mq >> 16) + __popc(mq & lt16);
            if (r < kSlotStage) sStage[r] = make_int2(se.y >> 16, se.x + b16);
            else P.cNode[first + r] = se.x + b16;  // cluster-ordered node index until the exact test
          }
        }
      }
      // ---- the exact test and contact law of the batch's candidates, by the whole wavefront, 64 slots at
      // a time; a pair's contacts leave their terms side by side from the pair's first slot on ----
      __threadfence_block();
      __builtin_amdgcn_wave_barrier();
      for (int r0 = 0; r0 < total; r0 += 64) {
        const int r = r0 + lane;
        int jj = 0;
        bool hit = false;
        SlotTerms terms{};
        if (r < total) {
          int node;
          if (r < kSlotStage) {
            const int2 st = sStage[r];
            jj = st.x;
            node = st.y;
          } else {
            while (r >= sOff[jj]) ++jj;  // (sOff now holds each pair's end)
            node = P.cNode[first + r];
          }
          P.cPair[first + r] = sF[jj].pair;
          hit = exactSlot(P, first + r, sF[jj], sX[jj], sF[jj].info, node, terms, statQueries, statContacts);
        }
        const unsigned long long hits = __ballot(hit);
        // the hits among this chunk's slots of pair j
        auto hitsOf = [&](int j) {
          const int lo = max(sOff[j] - sCnt[j] - r0, 0), hi = min(sOff[j] - r0, 64);
          return hi > lo ? hits & (~0ull >> (64 - (hi - lo)) << lo) : 0ull;
        };
        if (hit) {
          const int at = first + sOff[jj] - sCnt[jj] + sHits[jj] + __popcll(hitsOf(jj) & ltMask);
          double* o = P.cTerm + (long long)at * kTermDoubles;
          o[0] = terms.F.x; o[1] = terms.F.y; o[2] = terms.F.z;
          o[3] = terms.TA.x; o[4] = terms.TA.y; o[5] = terms.TA.z;
          o[6] = terms.TB.x; o[7] = terms.TB.y; o[8] = terms.TB.z;
        }
        __builtin_amdgcn_wave_barrier();
        if (mine) sHits[lane] += __popcll(hitsOf(lane));
        __builtin_amdgcn_wave_barrier();
      }
      // each pair with a contact: the place of its terms to both bodies' lists, its bit to their masks
      if (mine) contacts = sHits[lane];
      if (contacts > 0) {
        const int2 span = make_int2(first + sOff[lane] - sCnt[lane], contacts);
        P.pairSpan[sF[lane].pair] = span;
        atomicOr(&P.hitMask[sF[lane].A].x, hitBit(sF[lane].pair - masterFirst));
        if (rcSlot >= 0) {
          P.rcSpan[rcSlot] = span;
          atomicOr(&P.hitMask[sF[lane].info & kPartnerMask].y, hitBit(rcSlot - rcFirst));
        }
      }
    }
    if (mine) P.pairCcnt[sF[lane].pair] = contacts;
    statCand += (lane == 0) ? unsigned(total) : 0u;
  }
  // (lane 0 counted the batches' candidates and entries; without a candidate no lane tested one)
  const unsigned int t = __builtin_amdgcn_readfirstlane(statCand), te = __builtin_amdgcn_readfirstlane(statEnt);
  if (!(t | te)) return;
  unsigned long long tq = 0, tc = 0;
  if (t) {
    tq = (unsigned long long)wsum(double(statQueries));
    tc = (unsigned long long)wsum(double(statContacts));
  }
  if (lane0 == 0) {
    const int slot = (blockIdx.x + wl) & (kStatSlots - 1);
    atomicAdd(statSlot(P, 0, slot), (unsigned long long)t);
    atomicAdd(statSlot(P, 1, slot), tq);
    atomicAdd(statSlot(P, 2, slot), tc);
    atomicAdd(statSlot(P, 3, slot), (unsigned long long)te);
  }
}

// Surrogate cluster decisions, one wavefront per batch of 8 candidate pairs (lanes = pair x
// cluster, as stage 1 of k_candidates): bit c of surMask[p] is 0 when the network culls cluster c
// of pair p.  Only clusters whose centre lies in a family partner's grid box are queried, packed
// 16 per network pass.
__global__ __launch_bounds__(kNarrowBlock) void k_sur_masks(Params P) {
  LSD_HALT(P);
  __shared__ int sQ[kNarrowBlock / 64][64];
  const int lane = threadIdx.x & 63, wl = threadIdx.x >> 6;
  const EvalRecords rec = evalRecords(P);
  const int nAct = rec.n;
  const int wave = __builtin_amdgcn_readfirstlane(int(blockIdx.x * (kNarrowBlock / 64) + wl));
  const int nWaves = int(gridDim.x * (kNarrowBlock / 64));
  const int iters = (P.maxClusters + 7) >> 3;
  const int j = lane >> 3, k = lane & 7;
  for (int base = wave * kBatch; base < nAct; base += nWaves * kBatch) {
    const int a = base + j;  // map record
    const bool own = a < nAct;
    PairF32 f;
    if (own) f = reinterpret_cast<const PairF32*>(P.pairMap)[rec.at(a)];
    unsigned long long mask = ~0ull;
    float smin = __builtin_huge_valf();  // smallest slack of the clusters the network culls
    for (int it = 0; it < iters; ++it) {
      const int c = it * 8 + k;
      float gx = 0.f, gy = 0.f, gz = 0.f, rho = 0.f, ux = 0.f, uy = 0.f, uz = 0.f;
      int qslot = -1;
      if (own && c < f.nClusters && f.slot >= 0) {
        const ClusterF32 cl = P.clusters32[f.clusterOff + c];
        bool inside;
        float slack;
        if (clusterGeomF32(f, cl, gx, gy, gz, rho, inside, slack) && inside) {
          qslot = f.slot;
          surQueryPoint(P, f, gx, gy, gz, ux, uy, uz);
        }
      }
      const float d = surInferPacked(P.sur, ux, uy, uz, qslot, lane, sQ[wl]);
      const bool cull = qslot >= 0 && !clusterSurKeep(P, f, d, rho);
      if (cull) smin = fminf(smin, fmaxf(clusterSurSlack(P, f, d, rho), 0.f));
      // collect this group's 8 decisions of pair j into its mask
      const unsigned long long b = __ballot(cull);
      const unsigned long long mine = (b >> (8 * j)) & 0xFFull;
      mask &= ~(mine << (8 * it));
    }
    smin = groupMin<8>(smin);
    if (own && k == 0) {
      P.surMask[a] = mask;
      P.surSlack[a] = smin;
    }
  }
}

// Exact audit of the surrogate: every contact of this (plain) step whose partner is in the
// family must lie in a cluster that the surrogate keeps; a culled one is a missed contact.
// One lane per contact slot, 64 per wave through the network.
__global__ __launch_bounds__(kNarrowBlock) void k_sur_audit(Params P) {
  LSD_HALT(P);
  __shared__ int sQ[kNarrowBlock / 64][64];
  const int lane = threadIdx.x & 63;
  const int n = min(P.devInt[1], (int)P.contactCap);
  const int nWaves = int(gridDim.x * (kNarrowBlock / 64));
  unsigned long long checked = 0, missed = 0;
  for (int base = int(blockIdx.x * (kNarrowBlock / 64) + (threadIdx.x >> 6)) * 64; base < n; base += nWaves * 64) {
    const int c = base + lane;
    bool q = false;
    PairF32 f;
    float gx = 0.f, gy = 0.f, gz = 0.f, rho = 0.f, ux = 0.f, uy = 0.f, uz = 0.f;
    if (c < n && P.cInfo[c] != kInvalidInfo) {
      const int p = P.cPair[c];
      f = reinterpret_cast<const PairF32*>(P.pairMap)[P.pairRec[p]];
      if (f.slot >= 0) {
        const int A = P.pairA[p];
        const int orig = P.cNode[c] - P.prop[A].nodeStart;
        const int cluster = P.nodeCluster[f.nodeOff + orig];
        const ClusterF32 cl = P.clusters32[f.clusterOff + cluster];
        bool inside;
        float slack;
        const bool geom = clusterGeomF32(f, cl, gx, gy, gz, rho, inside, slack);
        q = geom && inside;  // the only clusters the surrogate decides on
        if (q) surQueryPoint(P, f, gx, gy, gz, ux, uy, uz);
        checked++;
      }
    }
    const float d = surInferPacked(P.sur, ux, uy, uz, q ? f.slot : -1, lane, sQ[threadIdx.x >> 6]);
    if (q && !clusterSurKeep(P, f, d, rho)) missed++;
  }
  const unsigned long long tc = (unsigned long long)wsum(double(checked));
  const unsigned long long tm = (unsigned long long)wsum(double(missed));
  if (lane == 0 && (tc | tm)) {
    atomicAdd(&P.devStat[10], tc);
    atomicAdd(&P.devStat[11], tm);
  }
}

// ------------------------------------------------------------------------------------------
// Bonds (one thread per bond)
// ------------------------------------------------------------------------------------------
// Force and torque of a bond on one of its bodies, at the place where that body's sums read them.
__device__ __forceinline__ void bondEnd(const Params& P, int at, d3 F, d3 M) {
  double* o = P.bEnd + 6ll * at;
  o[0] = F.x; o[1] = F.y; o[2] = F.z;
  o[3] = M.x; o[4] = M.y; o[5] = M.z;
}
__global__ void k_bonds(Params P) {
  LSD_HALT(P);
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= P.nBonds) return;
  double* out = P.bOut + 6ll * k;
  if (P.bActive[k] == 0) {
    for (int t = 0; t < 6; ++t) out[t] = 0.;
    bondEnd(P, P.bEndAt[2 * k], mk3(0, 0, 0), mk3(0, 0, 0));
    bondEnd(P, P.bEndAt[2 * k + 1], mk3(0, 0, 0), mk3(0, 0, 0));
    return;
  }
  const double* C = P.bConst + 9ll * k;
  const double B1 = C[0], B2 = C[1], B3 = C[2], B4 = C[3], rad = C[4], L0 = C[5], sT = C[6], coh = C[7],
               bmu = C[8];
  const d3* L = P.bLocal + 8ll * k;
  const int i = P.bI[k], j = P.bJ[k];
  const q4 qi = P.quat[i], qj = P.quat[j];
  const d3 n1i = rot(qi, L[0]), n2i = rot(qi, L[1]), n3i = rot(qi, L[2]);
  const d3 n1j = rot(qj, L[4]), n2j = rot(qj, L[5]), n3j = rot(qj, L[6]);
  const d3 ri = P.pos[i], rj = P.pos[j];
  const d3 rbi = rot(qi, L[3]) + ri, rbj = rot(qj, L[7]) + rj;
  P.bPoint[k] = 0.5 * (rbi + rbj);
  d3 F = mk3(0, 0, 0), Mij = mk3(0, 0, 0), Mji = mk3(0, 0, 0);
  int active = 1;
  const d3 rbij = rbi - rbj;
  const double D = len(rbij);
  if (!isZero(D)) {
    const d3 nij = normalize(rbij);
    const d3 e = -nij;
    out[0] = 0.5 * B1 * (D - L0) * (D - L0);
    out[1] = B2 * (0.5 * dot((n1j - n1i), e) - 0.25 * dot(n1i, n1j) + 0.75);
    out[2] = (0.25 * B2 + B3 + 0.5 * B4) * (dot(n1i, n1j) + 1.);
    out[3] = -0.5 * B4 * (dot(n1i, n1j) + dot(n2i, n2j) + dot(n3i, n3j) - 1);
    F = B1 * (D - L0) * e + B2 / (2 * D) * ((n1j - n1i) - dot((n1j - n1i), e) * e);
    const d3 MTB = B3 * cross(n1j, n1i) - 0.5 * B4 * (cross(n2j, n2i) + cross(n3j, n3i));
    Mij = -0.5 * B2 * cross(e, n1i) + MTB;
    Mji = 0.5 * B2 * cross(e, n1j) - MTB;
    const double Fn = dot(F, nij);
    const d3 Fs = F - Fn * nij;
    const double Tt = dot(MTB, nij);
    const d3 Tb = MTB - Tt * nij;
    const double Ab = rad * rad * kPi;
    const double Ib = Ab * rad * rad / 4.;
    const double Jb = 2 * Ib;
    out[4] = -Fn / Ab + len(Tb) / Ib * rad;
    out[5] = len(Fs) / Ab + fabs(Tt) / Jb * rad;
    if (sT > 0. && out[4] > sT) active = 0;
    else if (coh > 0. && out[5] > coh - bmu * out[4]) active = 0;
  }
  P.bActive[k] = active;
  bondEnd(P, P.bEndAt[2 * k], F, Mij + cross(rbi - ri, F));
  bondEnd(P, P.bEndAt[2 * k + 1], -F, Mji + cross(rbj - rj, -F));
}

// ------------------------------------------------------------------------------------------
// Per-body segmented reduction + second half-kick
// ------------------------------------------------------------------------------------------
__device__ void stepEnd(const Params& P);
__device__ void stepEndWave(const Params& P, int l);

// Adds `n` terms to F and T in order: term k is 6 values at base + stride * k, a force and, `tOff` values
// further, a torque; the force counts with `sign`.  The reads of kTermsAtOnce terms are issued together
// (as many as the body pass has registers for beside the state it has already read).
constexpr int kTermsAtOnce = 3;
__device__ __forceinline__ void addTerms(const double* base, int n, int stride, int tOff, double sign, d3& F, d3& T) {
  for (int k0 = 0; k0 < n; k0 += kTermsAtOnce) {
    d3 f[kTermsAtOnce], t[kTermsAtOnce];
#pragma unroll
    for (int u = 0; u < kTermsAtOnce; ++u)
      if (k0 + u < n) {
        const double* r = base + (long long)stride * (k0 + u);
        f[u] = mk3(r[0], r[1], r[2]);
        t[u] = mk3(r[tOff], r[tOff + 1], r[tOff + 2]);
      }
#pragma unroll
    for (int u = 0; u < kTermsAtOnce; ++u)
      if (k0 + u < n) {
        F += sign * f[u];
        T += t[u];
      }
  }
}
// The contact terms of the pairs whose bits are set, in order; spans: the pairs' places in cTerm (those of
// four pairs are read together).  tOff: the torque's place in a term.
__device__ __forceinline__ void addSpans(const Params& P, const int2* spans, unsigned int bits, int tOff, double sign,
                                         d3& F, d3& T) {
  while (bits) {
    int2 sp[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sp[u] = make_int2(0, 0);
      if (bits) {
        sp[u] = spans[__ffs(int(bits)) - 1];
        bits &= bits - 1;
      }
    }
    for (int u = 0; u < 4; ++u) {
      const int2 q = u == 0 ? sp[0] : u == 1 ? sp[1] : u == 2 ? sp[2] : sp[3];
      addTerms(P.cTerm + (long long)q.x * kTermDoubles, q.y, kTermDoubles, tOff, sign, F, T);
    }
  }
}

// Contact and bond sums on body b in a fixed order: its master pairs contact by contact, the reactions of
// the pairs where it is the partner, its bonds.  The narrow phase left the places of the contact terms in
// each body's own order and set the bit of each pair with a contact in the body's mask, so a body reads
// its mask (zero for a body without contacts, whose sums stay exactly zero), then the places, then the
// terms: three round trips, where a walk over all its pairs took two per pair and one per candidate slot
// (body pass: 82 -> 31 us for an ordered bed of 27,000 bodies with 7.6 contacts each as master, 53 -> 14 us
// for 8,000 bodies with 6 bonds each, 26.7 -> 23.3 us for 200,000 falling bodies, of which few touch).
// Returns whether any term was summed (false: F and T are exactly zero).
__device__ __forceinline__ bool reduceBody(const Params& P, int b, d3& F, d3& T) {
  F = mk3(0., 0., 0.);
  T = mk3(0., 0., 0.);
  const uint2 hit = P.hitMask[b];
  bool any = (hit.x | hit.y) != 0;
  if (any) {
    P.hitMask[b] = make_uint2(0u, 0u);
    const int p0 = P.pairStart[b], p1 = int(min((long long)P.pairStart[b + 1], P.pairCap));
    addSpans(P, P.pairSpan + p0, hit.x & ~kHitRest, 3, 1.0, F, T);
    if (hit.x & kHitRest)
      for (int p = p0 + kHitBits; p < p1; ++p)
        if (P.pairCcnt[p] > 0) addSpans(P, P.pairSpan + p, 1u, 3, 1.0, F, T);
    const int q0 = P.rcStart[b], q1 = P.rcStart[b + 1];
    addSpans(P, P.rcSpan + q0, hit.y & ~kHitRest, 6, -1.0, F, T);
    if (hit.y & kHitRest)
      for (int q = q0 + kHitBits; q < q1; ++q)
        if (P.pairCcnt[P.rcPair[q]] > 0) addSpans(P, P.rcSpan + q, 1u, 6, -1.0, F, T);
  }
  if (P.nBonds > 0) {
    // the bond kernel left each end's terms in this order
    const int q0 = P.bcStart[b], q1 = P.bcStart[b + 1];
    any = any || q1 > q0;
    addTerms(P.bEnd + 6ll * q0, q1 - q0, 6, 3, 1.0, F, T);
  }
  return any;
}

// One thread per body.  The last block, which has no bodies of its own, closes the step's bookkeeping with its
// first wavefront (thread 0 before its body's sums: 9.2 us of 27 bodies' steps one by one, now 4.5; 9.8 and 4.6 for
// 3,000 with a hook).
__global__ void k_reduce_kick(Params P, int kick) {
  LSD_HALT(P);
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x < 64) stepEndWave(P, int(threadIdx.x));
  if (b >= P.nP) return;
  d3 F, T;
  reduceBody(P, b, F, T);
  P.force[b] = F;
  P.torque[b] = T;
  P.forceSet[b] = 1;  // an external-force hook may add to the stored sums
  if (kick) halfKick(P, b, F, T);
}

// The end of one step and the start of the next in one pass over the bodies: sums, second
// half-kick, then the next step's first half-kick and drift (one thread per particle, then one per
// wall).  H describes the next step; P is this step's.  Nothing here reads another body's state,
// and this step's flags and counters are closed by thread 0 before it clears the next step's.
template <bool SEC>
__global__ void k_reduce_drift(Params P, StepHead H) {
  LSD_HALT_LATCH(P)
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  BodyIn in;
  bool set = false;
  if (b < P.nP) {
    in = loadBody<SEC>(P, b);
    set = P.forceSet[b] != 0;
  }
  if (b == 0) stepEnd(P);
  stepHead(P, H, b, int(gridDim.x * blockDim.x));
  if (b >= P.nP) {
    if (b - P.nP < P.nW) wallDrift(P, b - P.nP, H.buf);
    return;
  }
  d3 F, T;
  const bool any = reduceBody(P, b, F, T);
  kickDrift<SEC>(P, b, in, F, T, 2, H.buf);
  // the stored sums of a body without terms are already zero unless written otherwise since
  if (any || set) {
    P.force[b] = F;
    P.torque[b] = T;
    P.forceSet[b] = any ? 1 : 0;
  }
}
// The same for a small simulation (up to kWaveEndBodies bodies), whose
// counters a wavefront of a block of its own closes (stepEndWave): its body pass is short, and thread 0's
// rounds of counter reads were its last wavefront's (256 drums of 19k bodies in all: 0.0472 -> 0.0433 ms per
// step; the wavefront beside the bodies instead of before them another 1 % for 1,000).  In the 200k-body pass
// thread 0's version is the faster, and the kernel above is left as it compiles alone (any change to it shifts
// its code generation).
template <bool SEC>
__global__ void k_reduce_drift_small(Params P, StepHead H) {
  LSD_HALT_LATCH(P)
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  BodyIn in;
  bool set = false;
  if (b < P.nP) {
    in = loadBody<SEC>(P, b);
    set = P.forceSet[b] != 0;
  }
  // (the last block's thread 0 clears what its wavefront has just summed)
  const int bs = int(blockDim.x), last = int(gridDim.x - 1) * bs;
  if (b >= last && threadIdx.x < 64) stepEndWave(P, int(threadIdx.x));
  stepHead(P, H, b >= last ? b - last : b + bs, last + bs);
  if (b >= P.nP) {
    if (b - P.nP < P.nW) wallDrift(P, b - P.nP, H.buf);
    return;
  }
  d3 F, T;
  const bool any = reduceBody(P, b, F, T);
  kickDrift<SEC>(P, b, in, F, T, 2, H.buf);
  if (any || set) {
    P.force[b] = F;
    P.torque[b] = T;
    P.forceSet[b] = any ? 1 : 0;
  }
}

// Close of the pre-loop build: step bookkeeping, and the contact masks of the candidate kernel
// cleared (no sums follow; the stored forces stay those of the last step).
__global__ void k_prime_end(Params P) {
  LSD_HALT(P);
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b == 0) stepEnd(P);
  if (b < P.nP) P.hitMask[b] = make_uint2(0u, 0u);
}

// ------------------------------------------------------------------------------------------
// Call snapshot (restart of a call that halted on an error)
// ------------------------------------------------------------------------------------------
__global__ void k_snap_save(Params P, SnapDev S) {
  const Span g = gridSpan();
  for (int i = g.tid; i < P.nP; i += g.nth) {
    S.pos[i] = P.pos[i]; S.vel[i] = P.vel[i]; S.ang[i] = P.angvel[i];
    S.force[i] = P.force[i]; S.torque[i] = P.torque[i]; S.quat[i] = P.quat[i]; S.forceSet[i] = P.forceSet[i];
  }
  for (int i = g.tid; i < P.nW; i += g.nth) { S.wpos[i] = P.wpos[i]; S.wquat[i] = P.wquat[i]; }
  for (int i = g.tid; i < P.nBonds; i += g.nth) S.bActive[i] = P.bActive[i];
  const int n = int(min((long long)P.devInt[10 + S.prevBuf], S.hCap));
  for (int c = g.tid; c < n; c += g.nth) {
    S.hNode[c] = S.prevNode[c]; S.hInfo[c] = S.prevInfo[c]; S.hSpring[c] = S.prevSpring[c];
  }
  if (g.tid == 0) S.meta[0] = n;
  if (g.tid < kDevStats) S.devStat[g.tid] = P.devStat[g.tid];
}

// Back to the call's start; the history tables must be empty (filled by the host before).  The
// previous pair list is dropped (no certificate is inherited from it) and the step flags cleared.
__global__ void k_snap_restore(Params P, SnapDev S) {
  const Span g = gridSpan();
  for (int i = g.tid; i < P.nP; i += g.nth) {
    P.pos[i] = S.pos[i]; P.posDet[i] = S.pos[i]; P.vel[i] = S.vel[i]; P.angvel[i] = S.ang[i];
    P.force[i] = S.force[i]; P.torque[i] = S.torque[i]; P.quat[i] = S.quat[i]; P.forceSet[i] = S.forceSet[i];
    P.hitMask[i] = make_uint2(0u, 0u);
  }
  for (int i = g.tid; i <= P.nP; i += g.nth) P.pairStart[i] = 0;
  for (int i = g.tid; i < P.nW; i += g.nth) { P.wpos[i] = S.wpos[i]; P.wquat[i] = S.wquat[i]; }
  for (int i = g.tid; i < P.nBonds; i += g.nth) P.bActive[i] = S.bActive[i];
  const int n = S.meta[0];
  for (int c = g.tid; c < n; c += g.nth) {
    S.prevNode[c] = S.hNode[c]; S.prevInfo[c] = S.hInfo[c]; S.prevSpring[c] = S.hSpring[c];
  }
  if (g.tid < kDevStats) P.devStat[g.tid] = S.devStat[g.tid];
  if (g.tid < 18) P.barrier[g.tid * kBarrierLine] = 0;  // (the grid barrier's words and evalCount)
  if (g.tid == 0) {
    P.devInt[10 + S.prevBuf] = n;  // the restored slots, cleared from their table two steps on
    P.devInt[11 - S.prevBuf] = 0;  // the other table is empty
    P.devInt[1] = 0;
    P.devInt[rebuildFlagIdx(0)] = 0; P.devInt[rebuildFlagIdx(1)] = 0;
    P.devInt[ghostCountIdx(0)] = 0; P.devInt[ghostCountIdx(1)] = 0;
    P.devInt[3] = 0;
    P.devInt[kHaltedIdx] = 0;
    P.devInt[kErrStepIdx] = -1;
  }
  for (int k = g.tid; k < 5 * kStatSlots; k += g.nth) P.statSlots[k * kStatStride] = 0;
}

// The history table of the restored slots: each contact slot's key inserted again (the table was
// emptied first), its table slot recorded for the clearing two steps on.
__global__ void k_hist_reinsert(Params P, SnapDev S, unsigned long long* key, int* val, int* slotOf) {
  const Span g = gridSpan();
  const int n = S.meta[0];
  for (int c = g.tid; c < n; c += g.nth) {
    const uint32_t info = S.prevInfo[c];
    int at = -1;
    if (info != kInvalidInfo) {
      const unsigned long long k = histKey(info >> 28, S.prevNode[c], int(info & kPartnerMask));
      unsigned long long slot = mix64(k) & P.hashMask;
      for (unsigned long long probe = 0; probe <= P.hashMask; ++probe) {
        const unsigned long long old = atomicCAS(&key[slot], kHashEmpty, k);
        if (old == kHashEmpty || old == k) {
          val[slot] = c;
          at = int(slot);
          break;
        }
        slot = (slot + 1) & P.hashMask;
      }
    }
    slotOf[c] = at;
  }
}

// Second half-kick from the stored sums (after an external-force hook has added to them).
__global__ void k_kick(Params P) {
  LSD_HALT(P);
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= P.nP) return;
  halfKick(P, b, P.force[b], P.torque[b]);
}

// ------------------------------------------------------------------------------------------
// Step bookkeeping
// ------------------------------------------------------------------------------------------
// stepEnd by one wavefront, the first of the launch's last block (lanes l < min(64, blockDim.x)): the lanes read the stat
// slots (a line each) together and sum them across lanes (in FP64, exact for counts below 2^53), where
// thread 0 alone takes 8 dependent rounds of scalar loads.  Totals, flags and counters as stepEnd.
__device__ void stepEndWave(const Params& P, int l) {
  const int nl = min(64, int(blockDim.x));
  double s[5] = {0., 0., 0., 0., 0.};
  for (int k = l; k < kStatSlots; k += nl) {
#pragma unroll
    for (int f = 0; f < 5; ++f) s[f] += double(*statSlot(P, f, k));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      const double o = __shfl(s[f], l + off, 64);
      if (l + off < nl) s[f] += o;
    }
  }
  if (l == 0) {
    const int np = P.pairStart[P.nP];
    P.devInt[4] = max(P.devInt[4], np);
    P.devInt[5] = max(P.devInt[5], P.devInt[1]);
    P.devInt[10 + P.curBuf] = min(P.devInt[1], (int)P.contactCap);
    const unsigned long long t = (unsigned long long)s[0], q = (unsigned long long)s[1],
                             c = (unsigned long long)s[2], e = (unsigned long long)s[3],
                             mn = (unsigned long long)s[4];
    P.devStat[12] += mn;
    P.devStat[14] += P.devInt[rebuildFlagIdx(P.curBuf)] != 0 ? 1ull : 0ull;
    P.devStat[0] = t;
    P.devStat[1] = q;
    P.devStat[2] = c;
    P.devStat[3] += (unsigned long long)np;
    P.devStat[4] += t;
    P.devStat[5] += q;
    P.devStat[6] += c;
    P.devStat[8] += e;
    P.devInt[rebuildFlagIdx(P.curBuf)] = 0;
    P.devInt[ghostCountIdx(P.curBuf)] = 0;
  }
  // (after every lane's loads: their sums were exchanged above)
  for (int k = l; k < 5 * kStatSlots; k += nl) P.statSlots[k * kStatStride] = 0;
}

// Step totals into the counters, then the per-step counters that the drift kernel accumulates into
// cleared for the next step.
__device__ void stepEnd(const Params& P) {
  {
    const int np = P.pairStart[P.nP];  // (an overflowing list halted the call in the broad phase)
    P.devInt[4] = max(P.devInt[4], np);
    P.devInt[5] = max(P.devInt[5], P.devInt[1]);
    P.devInt[10 + P.curBuf] = min(P.devInt[1], (int)P.contactCap);  // slots to clear two steps on
    unsigned long long t = 0, q = 0, c = 0, e = 0, mn = 0;
    for (int k = 0; k < kStatSlots; ++k) {
      t += *statSlot(P, 0, k);
      q += *statSlot(P, 1, k);
      c += *statSlot(P, 2, k);
      e += *statSlot(P, 3, k);
      mn += *statSlot(P, 4, k);
    }
    P.devStat[12] += mn;
    P.devStat[14] += P.devInt[rebuildFlagIdx(P.curBuf)] != 0 ? 1ull : 0ull;
    P.devStat[0] = t;
    P.devStat[1] = q;
    P.devStat[2] = c;
    // sums over steps (profiling)
    P.devStat[3] += (unsigned long long)np;
    P.devStat[4] += t;
    P.devStat[5] += q;
    P.devStat[6] += c;
    P.devStat[8] += e;
  }
  P.devInt[rebuildFlagIdx(P.curBuf)] = 0;  // rebuild flag (the drift kernel raises it)
  P.devInt[ghostCountIdx(P.curBuf)] = 0;  // valid ghost images at their source's own position
  for (int k = 0; k < 5 * kStatSlots; ++k) P.statSlots[k * kStatStride] = 0;
  // (the contact slot count [1] and the pair check's evalCount stay readable after the step; the
  // drift kernel clears them)
}


// ------------------------------------------------------------------------------------------
// The whole broad phase in one launch (rebuild steps only; every block returns at once
// otherwise).  Phases are separated by grid barriers; every block runs every phase, so all blocks
// reach every barrier.  The host sizes the grid so that all its blocks are resident together.
// A rebuild is a chain of short phases: a barrier costs 2.3 to 2.9 us, a phase at least its own few dependent
// reads, so phases share barriers where neither reads what the other writes (14 barriers, once 19), and the sorts
// of long buckets are passed over when there are none.  Whole rebuild (the longest launch of a pass), before -> now: 27
// bodies 113 -> 80 us, 1,000 162 -> 109, 4,000 in a quarter sector 520 -> 301, 20,000 of scattered sizes 508 -> 319,
// 27,000 packed 225 -> 206, 200,000 of scattered sizes 1,074 -> 683.
// ------------------------------------------------------------------------------------------
// Blocks of the single-launch broad phase: large, so that few blocks meet at each barrier (the
// cost of a barrier grows with the number of blocks) while many threads work between them.
constexpr int kBroadThreads = 1024;

// Grid-stride loop bounds of phase `n` (a constant), worked out there: kept from the kernel's start, the indices
// cost the phases between registers.
__device__ __forceinline__ Span phaseSpan(int n) {
  return Span{int(blockIdx.x) * kBroadThreads + inLoop(int(threadIdx.x), n), int(gridDim.x) * kBroadThreads};
}

// Grid barrier in two levels (its words are zeroed by the pair check, the launch that follows every
// broad phase, and by the host after a failed call): a block arrives on
// its group's counter (group = blockIdx mod 8, the XCD the block runs on when the dispatcher deals
// blocks round-robin over the XCDs); the last arrival of a group arrives on the groups' counter, and
// the last of those writes the release word, which the blocks poll.  A barrier then serialises about
// nBlocks / 8 + 8 atomics on any one word instead of nBlocks, and the polls read a word no arrival
// writes.  The wait is bounded (P.barrierSpin polls, about a second by default): a block that gives
// up raises kErrBarrier.  A block also stops waiting as soon as any error flag is up, and after
// every barrier all blocks read the flags: sync() returns true when the launch must be abandoned,
// so every block leaves at the same barrier and no phase runs on the incomplete results of an
// earlier one.
struct GridBarrier {
  const Params& P;
  int nBlocks, passed;
  __device__ bool sync() {
    __shared__ int abandon;
    __syncthreads();
    ++passed;  // (by every thread: a uniform value takes no vector register)
    if (threadIdx.x == 0) {
      const int g = int(blockIdx.x) & 7;
      const int nGroups = min(nBlocks, 8);
      const int inGroup = (nBlocks - g + 7) >> 3;  // blocks b < nBlocks with b mod 8 == g
      int* groupCount = P.barrier + g * kBarrierLine;
      int* groupsDone = P.barrier + 8 * kBarrierLine;
      int* release = P.barrier + 9 * kBarrierLine;
      __threadfence();  // this block's writes, before the arrival
      if (atomicAdd(groupCount, 1) == passed * inGroup - 1) {
        __threadfence();  // (the group's arrivals, before the group's)
        if (atomicAdd(groupsDone, 1) == passed * nGroups - 1) {
          __threadfence();
          __hip_atomic_store(release, passed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      // relaxed polling (an acquire per poll would invalidate the caches every time), then one
      // acquire fence
      for (unsigned int it = 0;
           __hip_atomic_load(release, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < passed; ++it) {
        if (__hip_atomic_load(P.devInt + 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
        if (it >= unsigned(P.barrierSpin)) {
          raiseFlag(P, kErrBarrier);
          break;
        }
        __builtin_amdgcn_s_sleep(10);  // ~640 cycles between polls of the release word
      }
      __threadfence();  // the other blocks' writes, after the wait
      abandon = __hip_atomic_load(P.devInt + 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    }
    __syncthreads();
    return abandon != 0;
  }
};

// No vector register of this kernel may spill (1024 threads have 128 each): the compiler has put a spill at the head
// of a join block, before the lanes of the other side are back, so that only some lanes' values were kept, and the
// search then ran on garbage indices.
__global__ __launch_bounds__(kBroadThreads) void k_broad_phase(Params P) {
  LSD_HALT_LATCHED(P);
  if (P.devInt[rebuildFlagIdx(P.curBuf)] == 0) return;  // written by the drift kernel before this launch: grid-uniform
  __shared__ int lds[kScanLds];
  __shared__ int queues[kBroadThreads / kFindLanes * kFindQueue], many[kBroadThreads + 1];
  GridBarrier grid{P, int(gridDim.x), 0};
  const int ncell = P.sg.ncell;
  int* const bigCells = P.devInt + kBigCellsIdx;  // any cell (any reaction list) of more than kSmallBucket items:
  int* const bigRc = P.devInt + kBigRcIdx;        // without one, the phase that sorts those is left out
  // counting sort of the particles by search cell
  {
    const Span g = phaseSpan(0);
    for (int i = g.tid; i < ncell; i += g.nth) P.cellCount[i] = 0;
    for (int i = g.tid; i < P.nP; i += g.nth) {
      P.rcCount[i] = 0;
      P.scell[i] = searchCellOf(P, i);
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    P.devInt[2] = 0;  // large-bucket list
    *bigCells = 0;
    *bigRc = 0;
  }
  if (grid.sync()) return;
  bucketCount(P.scell, P.nP, P.cellCount, P.rank, phaseSpan(1));
  if (grid.sync()) return;
  scanReduceTiles(P.cellCount, ncell, P.scanTiles, lds);
  if (grid.sync()) return;
  scanApplyTiles(P.cellCount, ncell, P.scanTiles, P.cellStart, lds, bigCells);
  if (grid.sync()) return;
  bucketScatter(P.scell, P.nP, P.cellStart, P.rank, P.sortTmp, phaseSpan(2));
  if (grid.sync()) return;
  bucketSortSmall(P.cellStart, ncell, P.sortTmp, P.sorted, nullptr, P.sortBig, P.devInt + 2, phaseSpan(3), P.nP);
  if (grid.sync()) return;
  if (*bigCells) {
    bucketSortBig(P.cellStart, P.sortTmp, P.sorted, nullptr, P.sortBig, P.devInt + 2, phaseSpan(4), ncell, P.nP);
    if (grid.sync()) return;
  }
  // particle data in sorted order; candidate pairs per master, prefix, pair list
  {
    const Span g = phaseSpan(5);
    for (int k = g.tid; k < P.nP; k += g.nth) gatherParticle(P, k);
    backupPairs(P, g);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) P.devInt[2] = 0;  // large-bucket list of the reaction sort
  if (grid.sync()) return;
  pairsFind<kBroadThreads>(P, queues, many);
  if (grid.sync()) return;
  scanReduceTiles(P.pairCount, P.nP, P.scanTiles, lds);
  if (grid.sync()) return;
  scanApplyTiles(P.pairCount, P.nP, P.scanTiles, P.pairStart, lds);
  if (grid.sync()) return;
  // every block reads the same total after the barrier: all leave together when it does not fit
  if (pairOverflow(P)) return;
  pairsEmit<kBroadThreads>(P, queues, many);
  if (grid.sync()) return;
  inheritCerts(P, phaseSpan(6));  // reads the motion records before they restart
  // reaction CSR: pairs by partner (counted as they were written), in pair order
  scanReduceTiles(P.rcCount, P.nP, P.scanTiles, lds);
  if (grid.sync()) return;
  markBuild(P, phaseSpan(7));
  scanApplyTiles(P.rcCount, P.nP, P.scanTiles, P.rcStart, lds, bigRc);
  if (grid.sync()) return;
  rcScatterPairs(P, phaseSpan(8));
  if (grid.sync()) return;
  const int nRc = min(P.rcStart[P.nP], int(P.pairCap));
  bucketSortSmall(P.rcStart, P.nP, P.rcTmp, P.rcPair, P.rcSlot, P.sortBig, P.devInt + 2, phaseSpan(9), nRc);
  if (!*bigRc) return;
  if (grid.sync()) return;
  bucketSortBig(P.rcStart, P.rcTmp, P.rcPair, P.rcSlot, P.sortBig, P.devInt + 2, phaseSpan(10), P.nP, nRc);
}

template __global__ void k_candidates<false, false>(Params P);
template __global__ void k_candidates<true, false>(Params P);
template __global__ void k_candidates<false, true>(Params P);
template __global__ void k_candidates<true, true>(Params P);
template __global__ void k_kick_drift<false>(Params P, int forceRebuild);
template __global__ void k_kick_drift<true>(Params P, int forceRebuild);
template __global__ void k_reduce_drift<false>(Params P, StepHead H);
template __global__ void k_reduce_drift<true>(Params P, StepHead H);
template __global__ void k_reduce_drift_small<false>(Params P, StepHead H);
template __global__ void k_reduce_drift_small<true>(Params P, StepHead H);
template __global__ void k_pair_check<false>(Params P, int full);
template __global__ void k_pair_check<true>(Params P, int full);

}  // namespace lsd
