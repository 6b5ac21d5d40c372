// Learned proposal for model fitting: a 3-layer MLP (nin -> nh -> nh -> nout)
// with ReLU, trained on simulator-generated (spike-train features,
// parameters) pairs with a Gaussian negative log-likelihood.  No counterpart
// in the reference (which initialises the swarm uniformly at random,
// brian/library/modelfitting/modelfitting.py:232-518); plain PSO remains
// the fallback.
//
// Every product runs on gfx950's matrix cores (v_mfma_f32_32x32x16_bf16:
// BF16 operands, FP32 accumulation).  One training step is two kernels:
//   k_mlp_rows   one workgroup per 32 batch rows runs the whole forward
//                pass, the loss and the backward pass down to dZ1 with the
//                activations in LDS; weights stream from L2 as BF16 with the
//                reduction dimension contiguous.  It writes the operands of
//                the weight gradients transposed (feature-major, batch
//                contiguous) for the next kernel.
//   k_mlp_wgrad  dW = P^T Q and the bias sums, one workgroup per 32x32 output
//                tile with a wavefront per slice of the batch, the slices
//                added in a fixed order in LDS (no atomics); then Adam on the
//                FP32 master weights of the tile and the refresh of the BF16
//                copies the row kernel reads.
// The step counter and the batch position live on the device, so a chunk
// of steps is captured once in a hipGraph and replayed.
#include "common.hpp"
#include "../../include/brianmi.h"

#include <cmath>
#include <memory>
#include <mutex>
#include <random>
#include <vector>

namespace bm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int MR = 32;          // batch rows per k_mlp_rows workgroup
constexpr int RT = 512;         // threads of a k_mlp_rows workgroup (8 wavefronts)
constexpr int RW = RT / 64;
constexpr int NO = 32;          // padded output width (2 nu <= 32)
constexpr int MAXNI = 256, MAXNH = 256;
constexpr int WG_SLICES = 8;    // batch slices of the weight-gradient kernel

__host__ __device__ inline uint16_t f2bf(float f) {
  // round to nearest even (finite inputs)
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  const uint32_t lsb = (u >> 16) & 1u;
  u += 0x7FFFu + lsb;
  return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t b) {
  return __builtin_bit_cast(float, (uint32_t)b << 16);
}

__device__ inline bf16x8_t ld8(const uint16_t *p) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t *>(p));
}

// acc += A[32 x K] . B[K x 32], K = 16 NF: A row-major in LDS (row stride
// lda), B given as Bt[n][k] (k contiguous, row stride ldb) starting at output
// column n0.  Lane layout of v_mfma_f32_32x32x16_bf16: lane l supplies row
// l % 32 of A and column l % 32 of B at k = 8 (l / 32) .. +7 of each 16-wide K
// block.  The B fragments are loaded apart from the products, ahead of the
// phase that uses them.
template <int NF>
struct Frags {
  bf16x8_t f[NF];
  __device__ __forceinline__ void load(const uint16_t *Bt, int ldb, int n0, int lane) {
    const uint16_t *b = Bt + (size_t)(n0 + (lane & 31)) * ldb + (lane >> 5) * 8;
#pragma unroll
    for (int q = 0; q < NF; ++q) f[q] = ld8(b + q * 16);
  }
  __device__ __forceinline__ void mma(f32x16_t &acc, const uint16_t *A, int lda, int lane) const {
    const uint16_t *a = A + (lane & 31) * lda + (lane >> 5) * 8;
#pragma unroll
    for (int q = 0; q < NF; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(a + q * 16), f[q], acc, 0, 0, 0);
  }
};
// row and column of accumulator element q of a 32x32 tile
__device__ inline int acc_row(int q, int lane) { return 8 * (q >> 2) + (lane >> 5) * 4 + (q & 3); }

struct MlpDev {
  int nin, ni, nh, nu, nout;          // ni: nin rounded up to 32
  int64_t off[7];                     // master parameter offsets (W1 b1 W2 b2 W3 b3 end)
  const float *p;                     // FP32 master parameters
  const uint16_t *w1t, *w2t, *w3t;    // BF16 [nh][ni], [nh][nh], [NO][nh] (forward: k = input)
  const uint16_t *w2, *w3;            // BF16 [nh][nh], [nh][NO] (backward: k = output)
};

// LDS row strides (BF16 elements): 8 elements of padding keep the 16-byte
// operand reads aligned and spread rows over the banks
__host__ __device__ inline int lds_stride(int n) { return n + 8; }

// LDS elements of the dZ1 buffer, which holds the four partial tiles of the
// output layer's product first
__host__ __device__ constexpr int rows_z1(int nh) {
  return MR * (nh + 8) > 4 * MR * NO * 2 ? MR * (nh + 8) : 4 * MR * NO * 2;
}

// One workgroup: rows [r0, r0 + 32) of the batch.  X rows are gathered
// through idx (FP32 [n][nin]).  TRAIN: loss per row, and the transposed
// operands of the weight gradients, feature-major with the batch (ldb
// columns) contiguous: XT [ni][B], A1T / A2T / dZ2T / dZ1T [nh][B], dOT [NO][B].
// Forward only: the nout outputs per row into out [B][nout].
//
// NH = nh (64, 128, 192, 256): wavefront t computes column tile t of every
// 256-wide layer.  A batch of 1024 rows is 32 workgroups, each a chain of five
// MFMA phases: what a phase waits for is its weights from L2, so each
// wavefront loads the fragments of all its tiles ahead (the first two layers'
// with the input rows, the others' during the second layer; 168 registers at
// NH = 256, of the 256 that two wavefronts a SIMD leave).  The loss runs one
// thread per (row, output), the transposes one 16-byte store per thread and
// item.  Batch 1024, 64 -> 256 -> 256 -> 8: 24.2 us, now 17.7.
template <bool TRAIN, int NH>
__global__ __launch_bounds__(RT) void k_mlp_rows(const MlpDev m, const float *__restrict__ X,
                                                  const float *__restrict__ U, const int *__restrict__ idx,
                                                  const int64_t *__restrict__ d_batch, int B, float *out,
                                                  uint16_t *XT, uint16_t *A1T, uint16_t *A2T, uint16_t *dOT,
                                                  uint16_t *dZ2T, uint16_t *dZ1T, float *loss,
                                                  int64_t *d_step) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NT = NH / 32, sh = NH + 8, so = NO + 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ni = m.ni, sx = lds_stride(ni);
  uint16_t *sX = reinterpret_cast<uint16_t *>(smem);          // [32][sx]
  uint16_t *sA1 = sX + MR * sx;                                // [32][sh]
  uint16_t *sA2 = sA1 + MR * sh;                               // [32][sh], later dZ2
  uint16_t *sZ1 = sA2 + MR * sh;                               // [32][sh] dZ1 (TRAIN)
  uint16_t *sdO = sZ1 + rows_z1(NH);                           // [32][so]
  float *sO = reinterpret_cast<float *>(sdO + MR * so);        // [32][NO]
  const int r0 = blockIdx.x * MR;
  const int64_t boff = (TRAIN && d_batch) ? *d_batch * (int64_t)B : 0;
  const bool tile = wave < NT;                 // this wavefront holds a column tile
  const int tn = tile ? wave * 32 : 0;         // its first column
  const int tc = tn + (lane & 31);

  // weights and biases first: they depend on nothing
  Frags<NH / 16> fw2;
  const uint16_t *w1 = m.w1t + (size_t)tc * ni + (lane >> 5) * 8;
  // two fragments (32 inputs) of layer 1 at a time
  bf16x8_t f1a = ld8(w1), f1b = ld8(w1 + 16);
  const float b1 = m.p[m.off[1] + tc], b2 = m.p[m.off[3] + tc];
  fw2.load(m.w2t, NH, tn, lane);
  // the rows' inputs, 16 threads to a row, all of them in flight at once;
  // zero padding columns
  const int gr = tid >> 4;
  const int64_t gsrc = idx ? idx[boff + r0 + gr] : (int64_t)(r0 + gr);
  // the target of this thread's (row, output) of the loss
  const int lr = tid & (MR - 1), lk = tid / MR;
  float u = 0.f;
  if constexpr (TRAIN) {
    if (lk < m.nu) u = U[(idx ? (int64_t)idx[boff + r0 + lr] : (int64_t)(r0 + lr)) * m.nu + lk];
  }
  float xr[MAXNI / 16];
#pragma unroll
  for (int q = 0; q < MAXNI / 16; ++q) {
    const int k = (tid & 15) + 16 * q;
    xr[q] = k < m.nin ? X[gsrc * m.nin + k] : 0.f;
  }
#pragma unroll
  for (int q = 0; q < MAXNI / 16; ++q)
    if (q * 16 < ni) sX[gr * sx + (tid & 15) + 16 * q] = f2bf(xr[q]);
  if constexpr (TRAIN) {
    for (int e = tid; e < MR * so; e += RT) sdO[e] = 0;
  }
  // layer 1: A1 = relu(X W1 + b1) (BF16; A1 > 0 is the backward mask)
  f32x16_t acc1 = {};
  __syncthreads();
  if (TRAIN && d_step && blockIdx.x == 0 && tid == 0) *d_step += 1;   // Adam step of this batch
  {
    const uint16_t *a = sX + (lane & 31) * sx + (lane >> 5) * 8;
    for (int k0 = 0; k0 < ni; k0 += 32) {
      const bf16x8_t c0 = f1a, c1 = f1b;
      if (k0 + 32 < ni) {
        f1a = ld8(w1 + k0 + 32);
        f1b = ld8(w1 + k0 + 48);
      }
      acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(a + k0), c0, acc1, 0, 0, 0);
      acc1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(a + k0 + 16), c1, acc1, 0, 0, 0);
    }
  }
  if (tile) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const float z = acc1[q] + b1;
      sA1[acc_row(q, lane) * sh + tc] = f2bf(z > 0.f ? z : 0.f);
    }
  }
  // layer 3's reduction is split over four wavefronts
  constexpr int KQ = NH / 4;
  Frags<KQ / 16> fw3;
  if (wave < 4) fw3.load(m.w3t + wave * KQ, NH, 0, lane);
  const float b3 = m.p[m.off[5] + (tid & (NO - 1))];
  Frags<2> fb3;
  Frags<NH / 16> fb2;
  if constexpr (TRAIN) {
    fb3.load(m.w3, NO, tn, lane);
    fb2.load(m.w2, NH, tn, lane);
  }
  __syncthreads();
  // layer 2
  if (tile) {
    f32x16_t acc = {};
    fw2.mma(acc, sA1, sh, lane);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const float z = acc[q] + b2;
      sA2[acc_row(q, lane) * sh + tc] = f2bf(z > 0.f ? z : 0.f);
    }
  }
  __syncthreads();
  // layer 3: O = A2 W3 + b3 (one tile), partial tiles summed in a fixed
  // order (sZ1 is free here)
  float *part3 = reinterpret_cast<float *>(sZ1);               // [4][32][32]
  static_assert(4 * MR * NO * 4 <= rows_z1(NH) * 2, "the partial tiles fit the dZ1 buffer");
  if (wave < 4) {
    f32x16_t acc = {};
    fw3.mma(acc, sA2 + wave * KQ, sh, lane);
#pragma unroll
    for (int q = 0; q < 16; ++q) part3[wave * MR * NO + acc_row(q, lane) * NO + (lane & 31)] = acc[q];
  }
  __syncthreads();
  for (int e = tid; e < MR * NO; e += RT)
    sO[e] = ((part3[e] + part3[MR * NO + e]) + (part3[2 * MR * NO + e] + part3[3 * MR * NO + e])) + b3;
  __syncthreads();
  if constexpr (!TRAIN) {
    for (int e = tid; e < MR * m.nout; e += RT) {
      const int r = e / m.nout, k = e % m.nout;
      if (r0 + r < B) out[(int64_t)(r0 + r) * m.nout + k] = sO[r * NO + k];
    }
    return;
  } else {
    // Gaussian NLL over nu outputs: O = [mu | s], sigma = exp(s) with s
    // clamped to [-7, 3]; dO (BF16) scaled by 1/B
    float *sL = part3;                                         // [nu][32] terms of the loss
    if (lk < m.nu) {
      const float invB = 1.f / (float)B;
      const float mu = sO[lr * NO + lk];
      const float sr = sO[lr * NO + m.nu + lk];
      const float s = fminf(fmaxf(sr, -7.f), 3.f);
      const float iv = expf(-2.f * s);
      const float e = u - mu;
      sL[lk * MR + lr] = 0.5f * e * e * iv + s;
      sdO[lr * so + lk] = f2bf(-e * iv * invB);
      const float ds = (sr > -7.f && sr < 3.f) ? (1.f - e * e * iv) : 0.f;
      sdO[lr * so + m.nu + lk] = f2bf(ds * invB);
    }
    // transposed operands of the weight gradients: item = (feature, 8
    // consecutive batch columns), one 16-byte store
    auto store_t = [&](const uint16_t *S, int stride, int nfeat, uint16_t *dst) {
      for (int c = wave & 3; c < MR / 8; c += 4)
        for (int f = (wave >> 2) * 64 + lane; f < nfeat; f += 2 * 64) {
          u32x4_t wv;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            wv[q] = (uint32_t)S[(8 * c + 2 * q) * stride + f] | ((uint32_t)S[(8 * c + 2 * q + 1) * stride + f] << 16);
          reinterpret_cast<u32x4_t *>(dst + (int64_t)f * B + r0)[c] = wv;
        }
    };
    store_t(sX, sx, ni, XT);
    store_t(sA1, sh, NH, A1T);
    store_t(sA2, sh, NH, A2T);
    __syncthreads();
    if (tid < MR) {
      // the loss is indexed by the row's position in the batch
      float L = 0.f;
      for (int k = 0; k < m.nu; ++k) L += sL[k * MR + tid];
      loss[r0 + tid] = L;
    }
    store_t(sdO, so, NO, dOT);
    // dZ2 = (dO W3^T) * (A2 > 0), into the A2 buffer (each element's mask
    // is read by the lane that overwrites it)
    if (tile) {
      f32x16_t acc = {};
      fb3.mma(acc, sdO, so, lane);
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int at = acc_row(q, lane) * sh + tc;
        sA2[at] = sA2[at] != 0 ? f2bf(acc[q]) : (uint16_t)0;
      }
    }
    __syncthreads();
    store_t(sA2, sh, NH, dZ2T);
    // dZ1 = (dZ2 W2^T) * (A1 > 0)
    if (tile) {
      f32x16_t acc = {};
      fb2.mma(acc, sA2, sh, lane);
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int at = acc_row(q, lane) * sh + tc;
        sZ1[at] = sA1[at] != 0 ? f2bf(acc[q]) : (uint16_t)0;
      }
    }
    __syncthreads();
    store_t(sZ1, sh, NH, dZ1T);
  }
}

// Adam's state and the BF16 copies it refreshes; without adam the gradient is
// written to g.
struct AdamArgs {
  float *p, *g, *m, *v;
  float lr, b1, b2, eps;
  const int64_t *d_step;
  int64_t *d_batch;            // advanced by one (next batch) when non-null
  uint16_t *w1t, *w2t, *w3t, *w2, *w3;
  int adam;
};

struct AdamIn {
  float p, m, v;       // loaded ahead of the gradient
  __device__ __forceinline__ void load(const AdamArgs &a, int64_t i) {
    p = a.p[i];
    m = a.m[i];
    v = a.v[i];
  }
};
// The Adam step of parameter i with bias correction c1, c2 for the step
// counted on the device; returns the weight's BF16 copy.
__device__ __forceinline__ uint16_t adam_step(const AdamArgs &a, const AdamIn &in, int64_t i, float gi, float c1,
                                              float c2) {
  const float mi = a.b1 * in.m + (1.f - a.b1) * gi;
  const float vi = a.b2 * in.v + (1.f - a.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float w = in.p - a.lr * (mi / c1) / (sqrtf(vi / c2) + a.eps);
  a.p[i] = w;
  return f2bf(w);
}

// Weight gradients and, with them at hand, Adam.  Workgroup b < ntiles: the
// 32x32 tile b of dW1 | dW2 | dW3; wavefront s sums the products of batch slice
// s on the matrix cores, the eight partial tiles meet in LDS and are added in
// the order of the slices.  The workgroups after them: 64 biases each, thread
// (slice, bias).  One kernel: the partial sums of a step (8 x 92,000 floats)
// stay out of memory, and a launch less lies between the gradients and the
// weights (5.7 + 5.0 us in two kernels, 8.9 in one at batch 1024).
struct WgradArgs {
  const uint16_t *XT, *A1T, *A2T, *dOT, *dZ2T, *dZ1T;
  int B, ntiles1, ntiles2, ntiles3;
};
constexpr int WT = WG_SLICES * 64;

__global__ __launch_bounds__(WT) void k_mlp_wgrad(const MlpDev m, const WgradArgs a, const AdamArgs ad) {
  __shared__ float part[WG_SLICES][32][33];
  const int tid = threadIdx.x, lane = tid & 63, slice = tid >> 6;
  const int ks = a.B / WG_SLICES;
  const int ntiles = a.ntiles1 + a.ntiles2 + a.ntiles3;
  int t = blockIdx.x;
  if (ad.d_batch && t == 0 && tid == 0) *ad.d_batch += 1;
  float c1 = 1.f, c2 = 1.f;
  if (ad.adam) {
    const float st = (float)*ad.d_step;
    c1 = 1.f - powf(ad.b1, st);
    c2 = 1.f - powf(ad.b2, st);
  }
  if (t < ntiles) {
    const uint16_t *P, *Q;
    int np_out, rows, cols, which;     // matrix [rows][cols] at offset
    int64_t off;
    if (t < a.ntiles1) {
      P = a.XT; Q = a.dZ1T; rows = m.nin; cols = m.nh; off = m.off[0]; np_out = m.nh / 32; which = 1;
    } else if ((t -= a.ntiles1) < a.ntiles2) {
      P = a.A1T; Q = a.dZ2T; rows = m.nh; cols = m.nh; off = m.off[2]; np_out = m.nh / 32; which = 2;
    } else {
      t -= a.ntiles2;
      P = a.A2T; Q = a.dOT; rows = m.nh; cols = NO; off = m.off[4]; np_out = 1; which = 3;
    }
    const int ti = t / np_out, tj = t % np_out;
    AdamIn in[1024 / WT] = {};
    if (ad.adam) {
#pragma unroll
      for (int e = 0; e < 1024 / WT; ++e) {
        const int gi = ti * 32 + ((e * WT + tid) >> 5);
        if (gi < rows) in[e].load(ad, off + (int64_t)gi * cols + tj * 32 + (tid & 31));
      }
    }
    // C[i][j] = sum_b P[i][b] Q[j][b] over the slice: A = P rows (k = b), Bt = Q rows
    f32x16_t acc = {};
    const int r = lane & 31, kh = (lane >> 5) * 8;
    const uint16_t *pa = P + (int64_t)(ti * 32 + r) * a.B + slice * ks + kh;
    const uint16_t *pb = Q + (int64_t)(tj * 32 + r) * a.B + slice * ks + kh;
#pragma unroll 8
    for (int k0 = 0; k0 < ks; k0 += 16)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ld8(pa + k0), ld8(pb + k0), acc, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 16; ++q) part[slice][acc_row(q, lane)][lane & 31] = acc[q];
    __syncthreads();
    uint16_t wb[1024 / WT];
#pragma unroll
    for (int e = 0; e < 1024 / WT; ++e) {
      const int i = (e * WT + tid) >> 5, j = tid & 31;
      const int gi = ti * 32 + i, gj = tj * 32 + j;
      wb[e] = 0;
      if (gi >= rows) continue;
      float gsum = 0.f;
#pragma unroll
      for (int s = 0; s < WG_SLICES; ++s) gsum += part[s][i][j];
      const int64_t at = off + (int64_t)gi * cols + gj;
      if (!ad.adam) {
        ad.g[at] = gsum;
        continue;
      }
      wb[e] = adam_step(ad, in[e], at, gsum, c1, c2);
      // BF16 copies: backward layout [in][out] here, forward [out][in] below
      if (which == 2) ad.w2[(int64_t)gi * m.nh + gj] = wb[e];
      else if (which == 3) ad.w3[gi * NO + gj] = wb[e];
    }
    if (!ad.adam) return;
    // the transposed copies through LDS, 64 bytes of a row at a time
    uint16_t *sw = reinterpret_cast<uint16_t *>(&part[0][0][0]);      // [32][34]
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 1024 / WT; ++e) sw[(tid & 31) * 34 + ((e * WT + tid) >> 5)] = wb[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 1024 / WT; ++e) {
      const int j = (e * WT + tid) >> 5, i = tid & 31;
      const int gi = ti * 32 + i, gj = tj * 32 + j;
      if (gi >= rows) continue;
      const uint16_t w = sw[j * 34 + i];
      if (which == 1) ad.w1t[(int64_t)gj * m.ni + gi] = w;
      else if (which == 2) ad.w2t[(int64_t)gj * m.nh + gi] = w;
      else ad.w3t[(int64_t)gj * m.nh + gi] = w;
    }
    return;
  }
  // bias sums: (slice, bias over b1 | b2 | b3)
  const int nb = 2 * m.nh + NO;
  int j = (t - ntiles) * 64 + lane;
  const bool on = j < nb;
  const uint16_t *Q = a.dOT;
  int64_t off = m.off[5];
  if (j < m.nh) { Q = a.dZ1T; off = m.off[1]; }
  else if ((j -= m.nh) < m.nh) { Q = a.dZ2T; off = m.off[3]; }
  else j -= m.nh;
  float s = 0.f;
  if (on) {
    const uint16_t *q = Q + (int64_t)j * a.B + slice * ks;
    for (int b = 0; b < ks; b += 8) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t *>(q + b);
#pragma unroll
      for (int c = 0; c < 4; ++c) s += bf2f((uint16_t)(v[c] & 0xFFFFu)) + bf2f((uint16_t)(v[c] >> 16));
    }
  }
  part[slice][lane >> 5][lane & 31] = s;
  __syncthreads();
  if (slice != 0 || !on) return;
  float gsum = 0.f;
#pragma unroll
  for (int q = 0; q < WG_SLICES; ++q) gsum += part[q][lane >> 5][lane & 31];
  if (ad.adam) {
    AdamIn in;
    in.load(ad, off + j);
    (void)adam_step(ad, in, off + j, gsum, c1, c2);
  } else {
    ad.g[off + j] = gsum;
  }
}

// BF16 copies of the master weights in both layouts (W1T padding rows zero)
__global__ void k_mlp_cast(const MlpDev md, uint16_t *w1t, uint16_t *w2t, uint16_t *w3t, uint16_t *w2,
                           uint16_t *w3) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const float *p = md.p;
  if (i < (int64_t)md.nh * md.ni) {
    const int64_t c = i / md.ni, r = i % md.ni;       // w1t[c][r] = W1[r][c]
    w1t[i] = r < md.nin ? f2bf(p[md.off[0] + r * md.nh + c]) : (uint16_t)0;
  }
  if (i < (int64_t)md.nh * md.nh) {
    w2[i] = f2bf(p[md.off[2] + i]);
    const int64_t c = i / md.nh, r = i % md.nh;       // w2t[c][r] = W2[r][c]
    w2t[i] = f2bf(p[md.off[2] + r * md.nh + c]);
  }
  if (i < (int64_t)md.nh * NO) {
    w3[i] = f2bf(p[md.off[4] + i]);
    const int64_t c = i / md.nh, r = i % md.nh;       // w3t[c][r] = W3[r][c]
    w3t[i] = f2bf(p[md.off[4] + r * NO + c]);
  }
}

// Mean of the per-row losses (one workgroup, fixed summation order).
__global__ __launch_bounds__(256) void k_mlp_loss_mean(const float *__restrict__ loss, int B, float *out) {
  __shared__ float sh[256];
  float s = 0.f;
  for (int i = threadIdx.x; i < B; i += 256) s += loss[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = sh[0] / (float)B;
}

// Scratch of bm_mlp_grad_noalloc: the per-step buffers of a batch of up to
// NA_MAXB rows for nin <= NA_MAXNI and nh <= MAXNH, one copy per GPU for the
// life of the process.
constexpr int NA_MAXB = 1024, NA_MAXNI = 128;
constexpr size_t NA_BF16 = (size_t)NA_MAXB * (NA_MAXNI + 4 * MAXNH + NO);          // BF16 elements
constexpr size_t NA_BYTES = NA_BF16 * 2 + (size_t)NA_MAXB * 4;
static __device__ __align__(256) unsigned char scratch[NA_BYTES];

}  // namespace bm

using namespace bm;

struct bm_mlp {
  int nin = 64, ni = 64, nh = 256, nout = 8, nu = 4;
  // parameters (FP32 master) as one flat buffer: W1 b1 W2 b2 W3 b3 (W3/b3 padded to NO)
  int64_t off[7] = {};
  DevBuf p, g, m, v;
  DevBuf w1t, w2t, w3t, w2, w3;     // BF16 copies
  DevBuf data_x, data_u;
  int64_t ndata = 0;
  // per-batch operands for the batch capacity
  int cap = 0;
  DevBuf xb, ub, outb, XT, A1T, A2T, dOT, dZ2T, dZ1T, loss, idx;
  DevBuf d_step, d_batch;           // int64 counters
  int64_t step = 0;
  hipStream_t stream = nullptr;
  hipGraphExec_t graph = nullptr;
  int graph_batch = 0, graph_steps = 0;
  float graph_lr = 0.f;
  ~bm_mlp() {
    if (graph) (void)hipGraphExecDestroy(graph);
    if (stream) (void)hipStreamDestroy(stream);
  }
  MlpDev dev() const {
    MlpDev d{};
    d.nin = nin;
    d.ni = ni;
    d.nh = nh;
    d.nu = nu;
    d.nout = nout;
    for (int q = 0; q < 7; ++q) d.off[q] = off[q];
    d.p = p.as<float>();
    d.w1t = w1t.as<uint16_t>();
    d.w2t = w2t.as<uint16_t>();
    d.w3t = w3t.as<uint16_t>();
    d.w2 = w2.as<uint16_t>();
    d.w3 = w3.as<uint16_t>();
    return d;
  }
};

namespace {

int64_t nparams(const bm_mlp *h) {
  return (int64_t)h->nin * h->nh + h->nh + (int64_t)h->nh * h->nh + h->nh + (int64_t)h->nh * NO + NO;
}

size_t rows_shmem(const bm_mlp *h) {
  return (size_t)(MR * (lds_stride(h->ni) + 2 * lds_stride(h->nh) + lds_stride(NO)) + rows_z1(h->nh)) * 2 +
         (size_t)MR * NO * 4;
}

void drop_graph(bm_mlp *h) {
  if (h->graph) (void)hipGraphExecDestroy(h->graph);
  h->graph = nullptr;
  h->graph_steps = 0;
}

void ensure_cap(bm_mlp *h, int B) {
  if (B <= h->cap) return;
  drop_graph(h);           // a captured training chunk holds the old buffers
  const int c = (B + 255) / 256 * 256;
  h->xb.alloc((size_t)c * h->nin * 4);
  h->ub.alloc((size_t)c * h->nu * 4);
  h->outb.alloc((size_t)c * h->nout * 4);
  h->XT.alloc((size_t)c * h->ni * 2);
  h->A1T.alloc((size_t)c * h->nh * 2);
  h->A2T.alloc((size_t)c * h->nh * 2);
  h->dOT.alloc((size_t)c * NO * 2);
  h->dZ2T.alloc((size_t)c * h->nh * 2);
  h->dZ1T.alloc((size_t)c * h->nh * 2);
  h->loss.alloc((size_t)c * 4);
  h->cap = c;
}

void cast_weights(bm_mlp *h) {
  const int64_t n = std::max<int64_t>((int64_t)h->nh * h->ni, (int64_t)h->nh * h->nh);
  hipLaunchKernelGGL(k_mlp_cast, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, h->stream, h->dev(),
                     h->w1t.as<uint16_t>(), h->w2t.as<uint16_t>(), h->w3t.as<uint16_t>(), h->w2.as<uint16_t>(),
                     h->w3.as<uint16_t>());
}

// forward + loss + backward of one batch of B rows (B multiple of 256 for
// the batch slices, rows gathered from X through idx or taken in order),
// then either Adam (adam = 1, lr) or the summed gradient into g.
// Device buffers one step works in: the transposed operands of the weight
// gradients, the per-row loss and the gradient
// (written when the step does not apply Adam).
struct StepBufs {
  uint16_t *XT, *A1T, *A2T, *dOT, *dZ2T, *dZ1T;
  float *loss, *g;
};

StepBufs handle_bufs(bm_mlp *h) {
  return {h->XT.as<uint16_t>(), h->A1T.as<uint16_t>(), h->A2T.as<uint16_t>(), h->dOT.as<uint16_t>(),
          h->dZ2T.as<uint16_t>(), h->dZ1T.as<uint16_t>(), h->loss.as<float>(), h->g.as<float>()};
}

// the row kernel for the handle's hidden width
using RowsFn = void (*)(const MlpDev, const float *, const float *, const int *, const int64_t *, int, float *,
                        uint16_t *, uint16_t *, uint16_t *, uint16_t *, uint16_t *, uint16_t *, float *, int64_t *);
template <bool TRAIN>
RowsFn rows_kernel(int nh) {
  switch (nh) {
    case 64: return k_mlp_rows<TRAIN, 64>;
    case 128: return k_mlp_rows<TRAIN, 128>;
    case 192: return k_mlp_rows<TRAIN, 192>;
    default: return k_mlp_rows<TRAIN, 256>;
  }
}

void step(bm_mlp *h, const StepBufs &sb, const float *X, const float *U, const int *idx, const int64_t *d_batch,
          int B, int adam, float lr) {
  const MlpDev md = h->dev();
  hipLaunchKernelGGL(rows_kernel<true>(h->nh), dim3(B / MR), dim3(RT), rows_shmem(h), h->stream, md, X, U, idx,
                     d_batch, B, nullptr, sb.XT, sb.A1T, sb.A2T, sb.dOT, sb.dZ2T, sb.dZ1T, sb.loss,
                     adam ? h->d_step.as<int64_t>() : nullptr);
  WgradArgs w{};
  w.XT = sb.XT;
  w.A1T = sb.A1T;
  w.A2T = sb.A2T;
  w.dOT = sb.dOT;
  w.dZ2T = sb.dZ2T;
  w.dZ1T = sb.dZ1T;
  w.B = B;
  w.ntiles1 = (h->ni / 32) * (h->nh / 32);
  w.ntiles2 = (h->nh / 32) * (h->nh / 32);
  w.ntiles3 = h->nh / 32;
  AdamArgs a{};
  a.p = h->p.as<float>();
  a.g = sb.g;
  a.m = h->m.as<float>();
  a.v = h->v.as<float>();
  a.lr = lr;
  a.b1 = 0.9f;
  a.b2 = 0.999f;
  a.eps = 1e-8f;
  a.d_step = h->d_step.as<int64_t>();
  a.d_batch = adam && d_batch ? const_cast<int64_t *>(d_batch) : nullptr;
  a.w1t = h->w1t.as<uint16_t>();
  a.w2t = h->w2t.as<uint16_t>();
  a.w3t = h->w3t.as<uint16_t>();
  a.w2 = h->w2.as<uint16_t>();
  a.w3 = h->w3.as<uint16_t>();
  a.adam = adam;
  const int blocks = w.ntiles1 + w.ntiles2 + w.ntiles3 + (2 * h->nh + NO + 63) / 64;
  hipLaunchKernelGGL(k_mlp_wgrad, dim3(blocks), dim3(WT), 0, h->stream, md, w, a);
}

}  // namespace

extern "C" {

int bm_mlp_create(int nin, int nh, int nu, const float *params, bm_mlp **out) {
  return guard([&] {
    BM_REQUIRE(nin > 0 && nin <= MAXNI, "nin must be in [1, 256]");
    BM_REQUIRE(nh % 64 == 0 && nh > 0 && nh <= MAXNH, "nh must be a multiple of 64 in [64, 256]");
    BM_REQUIRE(nu > 0 && 2 * nu <= NO, "nu must be in [1, 16]");
    auto h = std::make_unique<bm_mlp>();
    h->nin = nin;
    h->ni = (nin + 31) / 32 * 32;
    h->nh = nh;
    h->nu = nu;
    h->nout = 2 * nu;
    BM_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    int64_t o = 0;
    h->off[0] = o; o += (int64_t)nin * nh;
    h->off[1] = o; o += nh;
    h->off[2] = o; o += (int64_t)nh * nh;
    h->off[3] = o; o += nh;
    h->off[4] = o; o += (int64_t)nh * NO;
    h->off[5] = o; o += NO;
    h->off[6] = o;
    BM_REQUIRE(rows_shmem(h.get()) <= 65536, "nin and nh too large for the row kernel's 64 KiB of LDS");
    const int64_t n = o;
    h->p.alloc(n * 4);
    h->g.alloc(n * 4);
    h->m.alloc(n * 4);
    h->v.alloc(n * 4);
    h->w1t.alloc((size_t)nh * h->ni * 2);
    h->w2t.alloc((size_t)nh * nh * 2);
    h->w3t.alloc((size_t)NO * nh * 2);
    h->w2.alloc((size_t)nh * nh * 2);
    h->w3.alloc((size_t)nh * NO * 2);
    h->d_step.alloc(8);
    h->d_batch.alloc(8);
    BM_HIP(hipMemcpyAsync(h->p.p, params, n * 4, hipMemcpyHostToDevice, h->stream));
    BM_HIP(hipMemsetAsync(h->m.p, 0, n * 4, h->stream));
    BM_HIP(hipMemsetAsync(h->v.p, 0, n * 4, h->stream));
    BM_HIP(hipMemsetAsync(h->g.p, 0, n * 4, h->stream));
    BM_HIP(hipMemsetAsync(h->d_step.p, 0, 8, h->stream));
    BM_HIP(hipMemsetAsync(h->d_batch.p, 0, 8, h->stream));
    cast_weights(h.get());
    BM_HIP(hipStreamSynchronize(h->stream));
    *out = h.release();
  });
}

int bm_mlp_num_params(int nin, int nh, int nu, int64_t *n) {
  return guard([&] {
    bm_mlp t;
    t.nin = nin;
    t.nh = nh;
    t.nu = nu;
    *n = nparams(&t);
  });
}

int bm_mlp_destroy(bm_mlp *h) {
  return guard([&] {
    if (!h) return;
    (void)hipStreamSynchronize(h->stream);
    delete h;
  });
}

int bm_mlp_forward(bm_mlp *h, const float *X, int B, float *out) {
  return guard([&] {
    BM_REQUIRE(B >= 0, "B must be >= 0");
    if (B == 0) return;
    const int Bp = (B + MR - 1) / MR * MR;
    ensure_cap(h, Bp);
    BM_HIP(hipMemsetAsync(h->xb.p, 0, (size_t)Bp * h->nin * 4, h->stream));
    BM_HIP(hipMemcpyAsync(h->xb.p, X, (size_t)B * h->nin * 4, hipMemcpyHostToDevice, h->stream));
    hipLaunchKernelGGL(rows_kernel<false>(h->nh), dim3(Bp / MR), dim3(RT), rows_shmem(h), h->stream, h->dev(),
                       h->xb.as<float>(), nullptr, nullptr, nullptr, B, h->outb.as<float>(), nullptr, nullptr,
                       nullptr, nullptr, nullptr, nullptr, nullptr, nullptr);
    BM_HIP(hipGetLastError());
    BM_HIP(hipMemcpyAsync(out, h->outb.p, (size_t)B * h->nout * 4, hipMemcpyDeviceToHost, h->stream));
    BM_HIP(hipStreamSynchronize(h->stream));
  });
}

int bm_mlp_grad(bm_mlp *h, const float *X, const float *U, int B, double *loss, float *grads) {
  return guard([&] {
    BM_REQUIRE(B > 0 && B % 256 == 0, "gradient batches must be a positive multiple of 256");
    ensure_cap(h, B);
    BM_HIP(hipMemcpyAsync(h->xb.p, X, (size_t)B * h->nin * 4, hipMemcpyHostToDevice, h->stream));
    BM_HIP(hipMemcpyAsync(h->ub.p, U, (size_t)B * h->nu * 4, hipMemcpyHostToDevice, h->stream));
    step(h, handle_bufs(h), h->xb.as<float>(), h->ub.as<float>(), nullptr, nullptr, B, 0, 0.f);
    BM_HIP(hipGetLastError());
    std::vector<float> l(B);
    BM_HIP(hipMemcpyAsync(l.data(), h->loss.p, (size_t)B * 4, hipMemcpyDeviceToHost, h->stream));
    BM_HIP(hipMemcpyAsync(grads, h->g.p, (size_t)h->off[6] * 4, hipMemcpyDeviceToHost, h->stream));
    BM_HIP(hipStreamSynchronize(h->stream));
    double s = 0;
    for (float x : l) s += x;
    *loss = s / B;
  });
}

int bm_mlp_set_data(bm_mlp *h, const float *X, const float *U, int64_t n) {
  return guard([&] {
    BM_REQUIRE(n > 0, "empty data set");
    h->data_x.alloc((size_t)n * h->nin * 4);
    h->data_u.alloc((size_t)n * h->nu * 4);
    h->idx.alloc((size_t)n * 4);
    BM_HIP(hipMemcpyAsync(h->data_x.p, X, (size_t)n * h->nin * 4, hipMemcpyHostToDevice, h->stream));
    BM_HIP(hipMemcpyAsync(h->data_u.p, U, (size_t)n * h->nu * 4, hipMemcpyHostToDevice, h->stream));
    BM_HIP(hipStreamSynchronize(h->stream));
    h->ndata = n;
    drop_graph(h);
  });
}

// Adam on shuffled mini-batches of the resident data set.  The batches of
// an epoch read consecutive slices of a device permutation; the batch
// position and step count advance on the device, so chunks of steps replay
// as one captured graph.
int bm_mlp_train(bm_mlp *h, int epochs, int batch, float lr, uint64_t seed, double *last_loss) {
  return guard([&] {
    BM_REQUIRE(batch > 0 && batch % 256 == 0 && h->ndata >= batch,
               "batch must be a positive multiple of 256, at most the data size");
    ensure_cap(h, batch);
    std::mt19937_64 rng(seed);
    std::vector<int> perm(h->ndata);
    const int64_t nb = h->ndata / batch;
    const int chunk = (int)std::min<int64_t>(nb, 64);
    if (h->graph && (h->graph_batch != batch || h->graph_steps != chunk || h->graph_lr != lr)) drop_graph(h);
    if (!h->graph) {
      hipGraph_t gr;
      BM_HIP(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
      for (int k = 0; k < chunk; ++k)
        step(h, handle_bufs(h), h->data_x.as<float>(), h->data_u.as<float>(), h->idx.as<int>(),
             h->d_batch.as<int64_t>(), batch, 1, lr);
      hipError_t e = hipStreamEndCapture(h->stream, &gr);
      BM_HIP(e);
      e = hipGraphInstantiate(&h->graph, gr, nullptr, nullptr, 0);
      hipGraphDestroy(gr);
      BM_HIP(e);
      h->graph_batch = batch;
      h->graph_steps = chunk;
      h->graph_lr = lr;
    }
    const int64_t zero = 0;
    for (int e = 0; e < epochs; ++e) {
      for (int64_t i = 0; i < h->ndata; ++i) perm[i] = (int)i;
      std::shuffle(perm.begin(), perm.end(), rng);
      BM_HIP(hipMemcpyAsync(h->idx.p, perm.data(), (size_t)h->ndata * 4, hipMemcpyHostToDevice, h->stream));
      BM_HIP(hipMemcpyAsync(h->d_batch.p, &zero, 8, hipMemcpyHostToDevice, h->stream));
      int64_t done = 0;
      for (; done + chunk <= nb; done += chunk) BM_HIP(hipGraphLaunch(h->graph, h->stream));
      for (; done < nb; ++done)
        step(h, handle_bufs(h), h->data_x.as<float>(), h->data_u.as<float>(), h->idx.as<int>(),
             h->d_batch.as<int64_t>(), batch, 1, lr);
      // the host copies above read perm and zero: finish before reuse
      BM_HIP(hipStreamSynchronize(h->stream));
      h->step += nb;
    }
    std::vector<float> l(batch);
    BM_HIP(hipMemcpyAsync(l.data(), h->loss.p, (size_t)batch * 4, hipMemcpyDeviceToHost, h->stream));
    BM_HIP(hipStreamSynchronize(h->stream));
    double s = 0;
    for (float x : l) s += x;
    *last_loss = s / batch;
  });
}

namespace {
// Device address of this GPU's copy of the scratch array, looked up once
// per device (the array's name is only a host-side handle).
unsigned char *scratch_ptr() {
  static std::mutex mu;
  static std::vector<unsigned char *> ptrs;
  int dev = 0;
  BM_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  if ((int)ptrs.size() <= dev) ptrs.resize(dev + 1, nullptr);
  if (!ptrs[dev]) {
    void *p = nullptr;
    BM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    BM_REQUIRE(p != nullptr, "no device address for the gradient scratch");
    ptrs[dev] = static_cast<unsigned char *>(p);
  }
  return ptrs[dev];
}
}  // namespace

int bm_mlp_grad_noalloc(bm_mlp *h, const float *X, const float *U, int B, float *loss, float *grads) {
  return guard([&] {
    BM_REQUIRE(h && X && U && loss && grads, "null argument");
    BM_REQUIRE(B > 0 && B % 256 == 0 && B <= NA_MAXB, "B must be a multiple of 256 in [256, 1024]");
    BM_REQUIRE(h->nin <= NA_MAXNI, "bm_mlp_grad_noalloc supports nin <= 128");
    unsigned char *base = scratch_ptr();
    // buffers at their size for this B, back to back in the scratch
    uint16_t *bf = reinterpret_cast<uint16_t *>(base);
    StepBufs sb;
    sb.XT = bf;
    sb.A1T = sb.XT + (size_t)h->ni * B;
    sb.A2T = sb.A1T + (size_t)h->nh * B;
    sb.dOT = sb.A2T + (size_t)h->nh * B;
    sb.dZ2T = sb.dOT + (size_t)NO * B;
    sb.dZ1T = sb.dZ2T + (size_t)h->nh * B;
    unsigned char *fl = base + NA_BF16 * 2;
    sb.loss = reinterpret_cast<float *>(fl);
    sb.g = grads;
    // every element the kernels read is written earlier in the same call
    // (all batch columns of the operands, all slices of every parameter),
    // so nothing is cleared
    step(h, sb, X, U, nullptr, nullptr, B, 0, 0.f);
    hipLaunchKernelGGL(k_mlp_loss_mean, dim3(1), dim3(256), 0, h->stream, sb.loss, B, loss);
    BM_HIP(hipGetLastError());
    BM_HIP(hipStreamSynchronize(h->stream));
  });
}

int bm_mlp_get_params(bm_mlp *h, float *out) {
  return guard([&] {
    BM_HIP(hipMemcpyAsync(out, h->p.p, (size_t)h->off[6] * 4, hipMemcpyDeviceToHost, h->stream));
    BM_HIP(hipStreamSynchronize(h->stream));
  });
}

}  // extern "C"
