// Pairwise squared distances of sampled traces on the device: the van Rossum
// metric's distance matrix (brian/monitor.py:1427-1486).  Row i of X holds
// neuron i's filtered spike train sampled every step (T samples);
//   D[i][j] = scale * sum_t (X[i][t] - X[j][t])^2,   scale = dt / tau,
// symmetric with a zero diagonal.  The differences are formed as the
// reference does (no |x|^2 + |y|^2 - 2 x.y expansion, which cancels, so the
// matrix cores have no part in it): n^2 T / 2 subtract/multiply-adds on the
// FP64 vector units.  A workgroup takes one 64x64 output tile of the lower
// triangle and a range of the samples, both row panels staged through LDS 32
// samples at a time (the next stage's loads in flight during the sums), 4x4
// adjacent outputs per thread so that each operand is a 16-byte LDS read.
// Few traces make few tiles (500: 36, on 256 compute units), so the samples
// are split until about SPLIT_BLOCKS workgroups run; the ranges' partial
// tiles are added in ascending order by a second kernel.  500 traces of 10,000
// samples: 2.66 ms with one workgroup per tile, now 0.149 ms and 0.029 ms for
// the sums (28 ranges; 25 TFLOP/s); the copy of the 40 MB to the device bounds
// the call (4.3 -> 2.2 ms).
#include "common.hpp"

#include <algorithm>

namespace bm {
namespace {

constexpr int TILE = 64;      // output tile edge
constexpr int TK = 32;        // samples per LDS stage
constexpr int MT = 256;       // threads per workgroup: 16 x 16, 4 x 4 outputs each
constexpr int LD = TILE + 2;  // LDS row stride: 16-byte aligned operand reads
constexpr int PER = TILE * TK / MT;   // samples of a panel staged per thread
// workgroups wanted (four fit a compute unit's LDS) and the most ranges: a
// range of fewer than 8 stages costs more in partial tiles than it gains
constexpr int SPLIT_BLOCKS = 1024, SPLIT_MAX = 32, SPLIT_STAGES = 8;

// lower-triangle tile (bi >= bj) from the linear tile index
__device__ inline void tile_of(int64_t b, int64_t &bi, int64_t &bj) {
  bi = (int64_t)((__builtin_sqrt(8.0 * (double)b + 1.0) - 1.0) * 0.5);
  while ((bi + 1) * (bi + 2) / 2 <= b) ++bi;
  while (bi * (bi + 1) / 2 > b) --bi;
  bj = b - bi * (bi + 1) / 2;
}

__device__ inline void store_pair(double *D, int64_t n, int64_t i, int64_t j, double v) {
  if (i >= n || j > i) return;
  if (i == j) v = 0.0;
  D[i * n + j] = v;
  D[j * n + i] = v;
}

// Samples [tspan * blockIdx.y, + tspan).  part == null: the only range,
// results straight into D; else the tile's sums to part[range][tile][64][64].
__global__ __launch_bounds__(MT) void k_pair_sqdist(const double *X, int64_t n, int64_t T, int64_t tspan,
                                                    double scale, double *D, double *part) {
  int64_t bi, bj;
  tile_of(blockIdx.x, bi, bj);
  const int64_t i0 = bi * TILE, j0 = bj * TILE;
  const int64_t tb = (int64_t)blockIdx.y * tspan, te = tb + tspan < T ? tb + tspan : T;

  __shared__ __align__(16) double As[TK][LD];
  __shared__ __align__(16) double Bs[TK][LD];
  const int tid = threadIdx.x;
  const int ty = tid >> 4, tx = tid & 15;
  double acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[a][c] = 0.0;

  // thread tid stages sample tid % TK of rows tid / TK + q * (MT / TK);
  // consecutive threads read consecutive samples of one row
  const int sk = tid % TK, sr = tid / TK;
  double pa[PER], pb[PER];
  auto fetch = [&](int64_t t0) {
    const int64_t t = t0 + sk;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int64_t ri = i0 + sr + q * (MT / TK), rj = j0 + sr + q * (MT / TK);
      pa[q] = (ri < n && t < te) ? X[ri * T + t] : 0.0;
      pb[q] = (rj < n && t < te) ? X[rj * T + t] : 0.0;
    }
  };
  if (tb < te) fetch(tb);
  for (int64_t t0 = tb; t0 < te; t0 += TK) {
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      As[sk][sr + q * (MT / TK)] = pa[q];
      Bs[sk][sr + q * (MT / TK)] = pb[q];
    }
    __syncthreads();
    if (t0 + TK < te) fetch(t0 + TK);
#pragma unroll 4
    for (int k = 0; k < TK; ++k) {
      double a[4], c[4];
      *reinterpret_cast<double2 *>(a) = *reinterpret_cast<const double2 *>(&As[k][ty * 4]);
      *reinterpret_cast<double2 *>(a + 2) = *reinterpret_cast<const double2 *>(&As[k][ty * 4 + 2]);
      *reinterpret_cast<double2 *>(c) = *reinterpret_cast<const double2 *>(&Bs[k][tx * 4]);
      *reinterpret_cast<double2 *>(c + 2) = *reinterpret_cast<const double2 *>(&Bs[k][tx * 4 + 2]);
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double d = a[p] - c[q];
          acc[p][q] = __builtin_fma(d, d, acc[p][q]);
        }
    }
    __syncthreads();
  }
  if (part != nullptr) {
    double *o = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (TILE * TILE);
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
      for (int q = 0; q < 4; ++q) o[(ty * 4 + p) * TILE + tx * 4 + q] = acc[p][q];
    return;
  }
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int q = 0; q < 4; ++q) store_pair(D, n, i0 + ty * 4 + p, j0 + tx * 4 + q, scale * acc[p][q]);
}

// One workgroup per tile and quarter: the ranges' sums in ascending order.
__global__ __launch_bounds__(MT) void k_pair_sum(const double *part, int64_t ntiles, int nranges, int64_t n,
                                                 double scale, double *D) {
  int64_t bi, bj;
  tile_of(blockIdx.x, bi, bj);
  for (int e = blockIdx.y * (TILE * TILE / 4) + threadIdx.x; e < (int)(blockIdx.y + 1) * (TILE * TILE / 4); e += MT) {
    double s = 0.0;
    for (int r = 0; r < nranges; ++r) s += part[((int64_t)r * ntiles + blockIdx.x) * (TILE * TILE) + e];
    store_pair(D, n, bi * TILE + e / TILE, bj * TILE + e % TILE, scale * s);
  }
}

}  // namespace
}  // namespace bm

using namespace bm;

extern "C" {

int bm_pairwise_sq_distance(const double *X, int64_t n, int64_t T, double scale, double *D) {
  return guard([&] {
    BM_REQUIRE(n >= 0 && T >= 0 && (n == 0 || (X && D)), "bad arguments");
    BM_REQUIRE(n <= (int64_t(1) << 20), "at most 2^20 traces");
    if (n == 0) return;
    hipStream_t st;
    BM_HIP(hipStreamCreate(&st));
    struct StreamGuard {
      hipStream_t s;
      ~StreamGuard() { hipStreamDestroy(s); }
    } sg{st};
    DevBuf x, d;
    x.alloc((size_t)(n * T) * 8);
    d.alloc((size_t)(n * n) * 8);
    if (T > 0) BM_HIP(hipMemcpyAsync(x.p, X, (size_t)(n * T) * 8, hipMemcpyHostToDevice, st));
    const int64_t nb = (n + TILE - 1) / TILE;
    const int64_t blocks = nb * (nb + 1) / 2;
    BM_REQUIRE(blocks < (int64_t(1) << 31), "too many traces");
    const int64_t stages = (T + TK - 1) / TK;
    const int64_t ranges =
        std::max<int64_t>(1, std::min({SPLIT_BLOCKS / blocks, (int64_t)SPLIT_MAX, stages / SPLIT_STAGES}));
    const int64_t tspan = (stages + ranges - 1) / ranges * TK;
    const int nr = ranges > 1 ? (int)((T + tspan - 1) / tspan) : 1;
    DevBuf part;
    if (nr > 1) {
      try {
        part.alloc((size_t)nr * blocks * TILE * TILE * 8);      // at most 32 MB
      } catch (const Error &) {
        (void)hipGetLastError();     // no room: one range
      }
    }
    if (part.p) {
      hipLaunchKernelGGL(k_pair_sqdist, dim3((unsigned)blocks, nr), dim3(MT), 0, st, x.as<double>(), n, T, tspan,
                         scale, d.as<double>(), part.as<double>());
      hipLaunchKernelGGL(k_pair_sum, dim3((unsigned)blocks, 4), dim3(MT), 0, st, part.as<double>(), blocks, nr, n,
                         scale, d.as<double>());
      BM_HIP(hipGetLastError());
      BM_HIP(hipStreamSynchronize(st));     // part is released here
    } else {
      hipLaunchKernelGGL(k_pair_sqdist, dim3((unsigned)blocks), dim3(MT), 0, st, x.as<double>(), n, T, T, scale,
                         d.as<double>(), static_cast<double *>(nullptr));
      BM_HIP(hipGetLastError());
    }
    BM_HIP(hipMemcpyAsync(D, d.p, (size_t)(n * n) * 8, hipMemcpyDeviceToHost, st));
    BM_HIP(hipStreamSynchronize(st));
  });
}

}  // extern "C"
