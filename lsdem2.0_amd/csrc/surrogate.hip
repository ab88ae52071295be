// Training and evaluation kernels of the learned culling surrogate (network in surrogate.h).
//
//   k_sur_sample   training / validation samples from the shapes' own SDF grids: grid nodes
//                  (exact values) and uniform points of the grid box (FP32 trilinear values),
//                  targets clamped to [-clamp, clamp] in normalised units
//   k_sur_train    one optimizer step's forward + backward over 64 samples per block; per-block
//                  partial gradients (deterministic, no atomics)
//   k_sur_adam     sums the block partials in a fixed order, Adam update of the FP32 masters,
//                  refreshes the BF16 swizzled copies
//   k_sur_eval     outputs and |error| statistics of a sample set
#include <hip/hip_runtime.h>

#include "surrogate_train.h"

namespace lsd {



__device__ __forceinline__ unsigned long long surHash(unsigned long long x) {
  x += 0x9e3779b97f4a7c15ull;
  x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
  x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
  return x ^ (x >> 31);
}
__device__ __forceinline__ float surUnit(unsigned long long h) { return float(h >> 40) * (1.0f / 16777216.0f); }

// FP32 trilinear value of a grid at index coordinates g (inside the box).
__device__ __forceinline__ float surTri(const float* g0, int nx, int ny, float gx, float gy, float gz, int mx, int my,
                                        int mz) {
  const int i0 = min(max(int(floorf(gx)), 0), mx - 2), j0 = min(max(int(floorf(gy)), 0), my - 2),
            k0 = min(max(int(floorf(gz)), 0), mz - 2);
  const float x = fminf(fmaxf(gx - i0, 0.f), 1.f), y = fminf(fmaxf(gy - j0, 0.f), 1.f), z = fminf(fmaxf(gz - k0, 0.f), 1.f);
  const int sy = nx, sz = nx * ny;
  const float* g = g0 + i0 + j0 * sy + k0 * sz;
  const float a = (g[0] * (1.f - x) + g[1] * x) * (1.f - y) + (g[sy] * (1.f - x) + g[sy + 1] * x) * y;
  const float b = (g[sz] * (1.f - x) + g[sz + 1] * x) * (1.f - y) + (g[sz + sy] * (1.f - x) + g[sz + sy + 1] * x) * y;
  return a * (1.f - z) + b * z;
}

__global__ void k_sur_sample(SurFamily F, SurSamples S, unsigned long long seed) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < S.n;
       i += (long long)gridDim.x * blockDim.x) {
    const int slot = int(i % F.nShapes);
    const ShapeDev sh = F.shapes[F.famShape[slot]];
    const float* g0 = F.sdf + sh.sdfOff;
    const unsigned long long h0 = surHash(seed ^ (unsigned long long)i), h1 = surHash(h0), h2 = surHash(h1);
    float gx, gy, gz, phi;
    if (((i / F.nShapes) & 1) == 0) {  // a grid node, exact value
      const int ix = int(h0 % (unsigned long long)sh.nx), iy = int(h1 % (unsigned long long)sh.ny),
                iz = int(h2 % (unsigned long long)sh.nz);
      gx = float(ix); gy = float(iy); gz = float(iz);
      phi = g0[ix + sh.nx * (iy + sh.ny * iz)];
    } else {  // uniform in the grid box
      gx = surUnit(h0) * float(sh.nx - 1);
      gy = surUnit(h1) * float(sh.ny - 1);
      gz = surUnit(h2) * float(sh.nz - 1);
      phi = surTri(g0, sh.nx, sh.ny, gx, gy, gz, sh.nx, sh.ny, sh.nz);
    }
    S.x[3 * i + 0] = float(sh.ox + double(gx) * sh.h);
    S.x[3 * i + 1] = float(sh.oy + double(gy) * sh.h);
    S.x[3 * i + 2] = float(sh.oz + double(gz) * sh.h);
    S.slot[i] = slot;
    S.t[i] = fminf(fmaxf(phi * F.invLen, -F.clamp), F.clamp);
  }
}



// v + its sum over the 16 lanes of a DPP row, in the order xor 1, 2, 4, 8 (each half of a pair adds the same two
// values, so once the quads agree a mirrored lane holds what the xor partner does).
__device__ __forceinline__ float surSum16(float v) {
#define LSD_DPP_ADD(ctrl) \
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), ctrl, 0xF, 0xF, true))
  LSD_DPP_ADD(0xB1);   // quad_perm 1,0,3,2
  LSD_DPP_ADD(0x4E);   // quad_perm 2,3,0,1
  LSD_DPP_ADD(0x141);  // mirrored in 8 lanes
  LSD_DPP_ADD(0x140);  // mirrored in 16 lanes
#undef LSD_DPP_ADD
  return v;
}

// One step's forward and backward over 64 samples per block, 16 waves: wave w works on the samples 16 (w mod 4) + ..
// and, of every layer, on the 16 outputs of block w / 4; the layers meet in LDS.  Bound by that chain (nine
// barriers, each with an LDS round trip, an MFMA chain and four SiLUs behind it) and by its first loads, so every
// weight is asked for before the layer that needs it.  Activations and their gradients are also kept transposed
// ([feature][sample]): an operand of the weight gradients, whose K dimension is the samples, is then one 8-byte read.
// (Four waves per block, each a chain of all 64 outputs, sums by bpermute, operands of the weight gradients
// gathered in 2-byte reads, 19 tiles a wave: 42 us for a step of 4,096 samples; 19 now.)
__global__ __launch_bounds__(kSurTrainThreads) void k_sur_train(SurTrainArgs A) {
  constexpr int kPad = kSurRows + 4;  // a transposed row, 34 words: 16 rows spread over the banks
  __shared__ sur_v4s sIn[kSurRows][kSurIn / 4 + 1];
  __shared__ sur_v4s sAct[2][kSurRows][kSurHid / 4 + 1];
  __shared__ __align__(8) uint16_t tX[kSurIn][kPad], tH[3][kSurHid][kPad], tDZ[4][kSurHid][kPad];
  __shared__ float4 sProd[kSurRows][kSurHid / 4 + 1];
  __shared__ float sRed[4][4 * kSurHid + kSurHid + 2];  // per 16 samples: db1..db4, dw5, db5, loss
  __shared__ float sEmb[kSurRows][kSurEmb];
  __shared__ int sSlot[kSurRows];
  const SurNet& N = A.net;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, m16 = lane & 15;
  const int sg = w & 3, mb = w >> 2;
  const int row = 16 * sg + m16, f0 = 16 * mb + 4 * q;  // the lane's sample; its first output of a layer
  sur_v4s w1[kSurKB1], wf[3][4], wb[4][4];
  float bias[4][4], w5[4];
#pragma unroll
  for (int kb = 0; kb < kSurKB1; ++kb) w1[kb] = N.wF[(mb * kSurKB1 + kb) * 64 + lane];
#pragma unroll
  for (int l = 0; l < 3; ++l)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) wf[l][kb] = N.wF[(kSurTileBase[l + 1] + mb * 4 + kb) * 64 + lane];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int l = 0; l < 4; ++l) bias[l][i] = N.param[kSurOffB[l] + f0 + i];
    w5[i] = N.param[kSurOffW5 + f0 + i];
  }
  const long long r = (long long)blockIdx.x * kSurRows + row;
  const long long si = (A.data.n > 0) ? (A.start + r * A.stride) % A.data.n : 0;
  const float px = A.data.x[3 * si], py = A.data.x[3 * si + 1], pz = A.data.x[3 * si + 2];
  const int slot = A.data.slot[si];
  const float target = A.data.t[si];
  // ---- input: two of the seven blocks per wave, the embedding (asked for first) by the last ----
  uint16_t e[4];
  if (mb == 3)
#pragma unroll
    for (int i = 0; i < 4; ++i) e[i] = N.emb[slot * kSurEmb + 4 * q + i];
  const float ux = px * N.invLen, uy = py * N.invLen, uz = pz * N.invLen;
  auto transposed = [&](uint16_t(*t)[kPad], int f, sur_v4s v) {
    t[f][row] = uint16_t(v.x);
    t[f + 1][row] = uint16_t(v.y);
    t[f + 2][row] = uint16_t(v.z);
    t[f + 3][row] = uint16_t(v.w);
  };
#pragma unroll 1
  for (int kb = mb; kb < 6; kb += 4) {
    float v[4];
    const int k0 = 16 * kb + 4 * q;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = surFeature(k0 + i, ux, uy, uz);
    const sur_v4s x = surPack(v[0], v[1], v[2], v[3]);
    sIn[row][4 * kb + q] = x;
    transposed(tX, k0, x);
  }
  if (mb == 3) {
    const sur_v4s x = {short(e[0]), short(e[1]), short(e[2]), short(e[3])};
    sIn[row][4 * 6 + q] = x;
    transposed(tX, 96 + 4 * q, x);
    if (q == 0) sSlot[row] = slot;
  }
  __syncthreads();
  // ---- forward ----
  float ds[4][4], h4[4];  // SiLU's derivative at each layer's outputs; the last activations
#pragma unroll
  for (int layer = 0; layer < 4; ++layer) {
    const sur_v4f zero = {0.f, 0.f, 0.f, 0.f};
    const sur_v4f acc = layer == 0 ? surMfmaK<kSurKB1>([&](int kb) { return w1[kb]; },
                                                       [&](int kb) { return sIn[row][4 * kb + q]; }, zero)
                                   : surMfmaK<4>([&](int kb) { return wf[layer > 0 ? layer - 1 : 0][kb]; },
                                                 [&](int kb) { return sAct[(layer + 1) & 1][row][4 * kb + q]; }, zero);
    if (layer == 0) {
#pragma unroll
      for (int l = 1; l < 4; ++l)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) wb[l][kb] = N.wB[(kSurTileBase[l] + mb * 4 + kb) * 64 + lane];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) wb[0][kb] = N.wB[(kSurTileBase[0] + 6 * 4 + kb) * 64 + lane];  // embedding rows
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float z = acc[i] + bias[layer][i];
      h4[i] = surSilu(z);
      ds[layer][i] = surDSilu(z);
    }
    if (layer < 3) {
      const sur_v4s h = surPack(h4[0], h4[1], h4[2], h4[3]);
      sAct[layer & 1][row][4 * mb + q] = h;
      transposed(tH[layer], f0, h);
    } else {
      sProd[row][4 * mb + q] = make_float4(h4[0] * w5[0], h4[1] * w5[1], h4[2] * w5[2], h4[3] * w5[3]);
    }
    __syncthreads();
  }
  float out = 0.f;  // (by every wave of the samples, in the order of surForwardInfer)
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const float4 p = sProd[row][4 * m + q];
    out += p.x;
    out += p.y;
    out += p.z;
    out += p.w;
  }
  out += __shfl_xor(out, 16, 64);
  out += __shfl_xor(out, 32, 64);
  out += N.param[kSurOffB5];
  // ---- backward ----
  const float err = out - target;
  const float dout = 2.0f * err / float(A.batch);
  float dz[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    dz[i] = dout * w5[i] * ds[3][i];
    const float g5 = surSum16(h4[i] * dout);
    if (m16 == 0) sRed[sg][4 * kSurHid + f0 + i] = g5;
  }
  if (mb == 0) {
    const float g = surSum16(dout);
    const float l2 = surSum16(err * err);
    if (lane == 0) {
      sRed[sg][5 * kSurHid] = g;
      sRed[sg][5 * kSurHid + 1] = l2 / float(A.batch);
    }
  }
#pragma unroll
  for (int layer = 3; layer >= 0; --layer) {
    const sur_v4s d = surPack(dz[0], dz[1], dz[2], dz[3]);
    sAct[layer & 1][row][4 * mb + q] = d;
    transposed(tDZ[layer], f0, d);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float gb = surSum16(dz[i]);
      if (m16 == 0) sRed[sg][layer * kSurHid + f0 + i] = gb;
    }
    __syncthreads();
    // dh_prev^T = W dz^T, then through the previous SiLU; of layer 1's inputs the embedding (block 6)
    if (layer > 0 || mb == 3) {
      const sur_v4f acc = surMfmaK<4>([&](int kb) { return wb[layer][kb]; },
                                      [&](int kb) { return sAct[layer & 1][row][4 * kb + q]; },
                                      sur_v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (layer > 0) dz[i] = acc[i] * ds[layer > 0 ? layer - 1 : 0][i];
        else sEmb[row][4 * q + i] = acc[i];
    }
  }
  // ---- weight gradients over the block's 64 samples: dW = H^T dZ (samples are the K dimension) ----
  float* G = A.partial + (long long)blockIdx.x * (kSurNParam + N.nShapes * kSurEmb + 1);
  const int nb = w & 3, n = 16 * nb + m16;
#pragma unroll
  for (int layer = 0; layer < 4; ++layer) {
    sur_v4s b[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) b[p] = *reinterpret_cast<const sur_v4s*>(&tDZ[layer][n][16 * p + 4 * q]);
    for (int kb = w >> 2; kb < (layer == 0 ? kSurKB1 : 4); kb += 4) {
      const uint16_t* a = layer == 0 ? tX[16 * kb + m16] : tH[layer > 0 ? layer - 1 : 0][16 * kb + m16];
      const sur_v4f acc = surMfmaK<4>([&](int p) { return *reinterpret_cast<const sur_v4s*>(a + 16 * p + 4 * q); },
                                      [&](int p) { return b[p]; }, sur_v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 4; ++i) G[kSurOffW[layer] + (16 * kb + 4 * q + i) * kSurHid + n] = acc[i];
    }
  }
  // biases, w5, b5, loss: the partials of the four 16s in a fixed order
  if (threadIdx.x < 5 * kSurHid + 2) {
    const int k = threadIdx.x;
    const float v = sRed[0][k] + sRed[1][k] + sRed[2][k] + sRed[3][k];
    if (k < 4 * kSurHid) G[kSurOffB[k / kSurHid] + (k % kSurHid)] = v;
    else if (k < 5 * kSurHid) G[kSurOffW5 + (k - 4 * kSurHid)] = v;
    else if (k == 5 * kSurHid) G[kSurOffB5] = v;
    else G[kSurNParam + N.nShapes * kSurEmb] = v;
  }
  // embedding gradients per family slot, samples in row order (by the block's last waves: the first had the biases)
  __syncthreads();
  for (int k = kSurTrainThreads - 1 - int(threadIdx.x); k < N.nShapes * kSurEmb; k += kSurTrainThreads) {
    const int s = k / kSurEmb, e = k % kSurEmb;
    float v = 0.f;
#pragma unroll 8
    for (int rr = 0; rr < kSurRows; ++rr) {
      const float add = v + sEmb[rr][e];
      v = sSlot[rr] == s ? add : v;
    }
    G[kSurNParam + k] = v;
  }
}


// Swizzled positions of W_layer[k][n] in the forward and backward tile sets.
__device__ __forceinline__ void surSwizzle(int layer, int k, int n, int& fTile, int& fLane, int& bTile, int& bLane,
                                           int& i) {
  const int KB = layer == 0 ? kSurKB1 : 4;
  fTile = kSurTileBase[layer] + (n >> 4) * KB + (k >> 4);
  fLane = (n & 15) + 16 * ((k & 15) >> 2);
  bTile = kSurTileBase[layer] + (k >> 4) * 4 + (n >> 4);
  bLane = (k & 15) + 16 * ((n & 15) >> 2);
  i = -1;  // per operand below
}

__device__ __forceinline__ void surStoreWeight(sur_v4s* wF, sur_v4s* wB, int layer, int k, int n, float value) {
  int fT, fL, bT, bL, unused;
  surSwizzle(layer, k, n, fT, fL, bT, bL, unused);
  short* f = reinterpret_cast<short*>(wF + fT * 64 + fL);
  short* b = reinterpret_cast<short*>(wB + bT * 64 + bL);
  const short h = short(surBf16(value));
  f[k & 3] = h;
  b[n & 3] = h;
}

// A thread per parameter (and one for the loss): the blocks' partial gradients in block order, sixteen reads in
// flight together, then the update.  Bound by those reads, which the other kernel's XCDs wrote; blocks of one
// wave, so that the 20,000 parameters reach every CU.  (Read and added one at a time by 78 blocks of 256, and the
// loss after that by one of them: 22 us for 64 partials; 4.7 now.)
__global__ void k_sur_adam(SurAdamArgs A) {
  const int nAll = kSurNParam + A.nShapes * kSurEmb;
  const int stride = nAll + 1;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > nAll) return;
  const bool isLoss = p == nAll;
  float* const w = p < kSurNParam ? &A.param[p] : &A.embF[p - kSurNParam];
  float m = 0.f, v = 0.f, old = 0.f;
  if (!isLoss) {
    m = A.m[p];
    v = A.v[p];
    old = *w;
  }
  float g = 0.f;
  const float* part = A.partial + p;
  int b = 0;
  for (; b + 16 <= A.blocks; b += 16) {
    float t[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) t[u] = part[(long long)(b + u) * stride];
#pragma unroll
    for (int u = 0; u < 16; ++u) g += t[u];
  }
  for (; b < A.blocks; ++b) g += part[(long long)b * stride];
  if (isLoss) {
    *A.loss = g;
    return;
  }
  m = A.b1 * m + (1.f - A.b1) * g;
  v = A.b2 * v + (1.f - A.b2) * g * g;
  A.m[p] = m;
  A.v[p] = v;
  const float nw = old - A.lr * (m * A.c1) / (sqrtf(v * A.c2) + A.eps);
  *w = nw;
  if (p >= kSurNParam) {
    A.emb[p - kSurNParam] = surBf16(nw);
    return;
  }
  for (int layer = 0; layer < 4; ++layer) {
    const int K = layer == 0 ? kSurIn : kSurHid;
    if (p >= kSurOffW[layer] && p < kSurOffW[layer] + K * kSurHid) {
      const int k = (p - kSurOffW[layer]) / kSurHid, n = (p - kSurOffW[layer]) % kSurHid;
      surStoreWeight(A.wF, A.wB, layer, k, n, nw);
    }
  }
}

// Fill the swizzled BF16 copies from the FP32 masters (after set_params).
__global__ void k_sur_pack(const float* param, const float* embF, int nShapes, sur_v4s* wF, sur_v4s* wB,
                           uint16_t* emb) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < kSurNParam + nShapes * kSurEmb;
       p += gridDim.x * blockDim.x) {
    if (p >= kSurNParam) {
      emb[p - kSurNParam] = surBf16(embF[p - kSurNParam]);
      continue;
    }
    for (int layer = 0; layer < 4; ++layer) {
      const int K = layer == 0 ? kSurIn : kSurHid;
      if (p >= kSurOffW[layer] && p < kSurOffW[layer] + K * kSurHid)
        surStoreWeight(wF, wB, layer, (p - kSurOffW[layer]) / kSurHid, (p - kSurOffW[layer]) % kSurHid, param[p]);
    }
  }
}

// Outputs (normalised units) of a sample set and error statistics against its targets:
// stat[0] = max |out - t| (float bits), stat[1..] unused.
__global__ __launch_bounds__(256) void k_sur_eval(SurNet N, SurSamples S, float* out, unsigned int* maxErrBits, float* sumAbs) {
  const int lane = threadIdx.x & 63;
  const long long nWaves = (long long)gridDim.x * (blockDim.x >> 6);
  const long long nGroups = (S.n + 63) / 64;
  for (long long grp = blockIdx.x * (long long)(blockDim.x >> 6) + (threadIdx.x >> 6); grp < nGroups; grp += nWaves) {
    const long long i = grp * 64 + lane;
    const bool ok = i < S.n;
    const float px = ok ? S.x[3 * i] : 0.f, py = ok ? S.x[3 * i + 1] : 0.f, pz = ok ? S.x[3 * i + 2] : 0.f;
    const int slot = ok ? S.slot[i] : -1;
    const float o = surInfer64(N, px * N.invLen, py * N.invLen, pz * N.invLen, slot, lane);
    if (ok) {
      if (out) out[i] = o;
      if (maxErrBits) {
        const float e = fabsf(o - S.t[i]);
        atomicMax(maxErrBits, __float_as_uint(e));
        atomicAdd(sumAbs, e);
      }
    }
  }
}

}  // namespace lsd
