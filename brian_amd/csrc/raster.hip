// Spike rasters sorted on the device.  A group's raster is RSHARD append
// regions of entries step << 32 | index in no order (net_types.hpp); reading
// it (SpikeMonitor, brian/monitor.py:156-199) returns the entries sorted by
// (step, index).
//
// Up to SMALL entries: one workgroup gathers the regions into LDS and sorts
// them there (bitonic), one launch.  More: the entries are packed into keys
// (step - first) << index bits | index, 32 bits wide where they fit and 64
// otherwise, and sorted by a least-significant-digit radix sort of 8 bits a
// pass over only the bits in use.  A pass is three kernels: digit counts per
// tile of 4096 keys, a scan of each digit's counts over the tiles, and a
// stable scatter that ranks equal digits by wavefront ballots; the last
// scatter writes the steps and indices instead of keys.  1.2 million spikes of
// a 2^20-neuron network take four passes over 5 MB, about 0.12 ms in 13
// kernels, bound by their launches and by the copy to the host after them:
// running 2000 steps and reading raster and state takes 13.6 ms, and took
// 57.7 with the copied regions sorted on the host (std::sort).  4096 entries
// fill 32 KiB of LDS; up to there one workgroup is the faster way: a read with
// its copies takes 85 us so and 130 by radix passes for 100 entries, 114 and 150 to
// 174 (two to four passes) for 4096.  The 500 spikes of 200 steps of 4000
// neurons: 1.29 -> 1.08 ms for the run and its reading, most of it one copy in
// place of one per region.
#include "net_launch.hpp"

#include <algorithm>

namespace bm {
namespace {

constexpr int RT = 256;            // threads of a tile's workgroup
constexpr int RROUNDS = 16;        // keys per thread
constexpr int RTILE = RT * RROUNDS;
constexpr int SMALL = 4096;        // entries sorted by one workgroup in LDS
constexpr int SMALL_T = 1024;

struct Regions {
  const unsigned long long *base;
  int64_t stride;                  // entries between regions
  uint32_t off[RSHARD + 1];        // first entry of each region in the gathered list
};

__device__ inline unsigned long long region_entry(const Regions &g, uint32_t q) {
  int a = 0;                       // last region with off[a] <= q
#pragma unroll
  for (int step = RSHARD / 2; step > 0; step >>= 1)
    if (g.off[a + step] <= q) a += step;
  return g.base[(int64_t)a * g.stride + (q - g.off[a])];
}

__global__ __launch_bounds__(SMALL_T) void k_raster_small(const Regions g, int n, int np2, int32_t *steps,
                                                          int32_t *idx) {
  __shared__ unsigned long long e[SMALL];
  for (int q = threadIdx.x; q < np2; q += SMALL_T) e[q] = q < n ? region_entry(g, (uint32_t)q) : ~0ull;
  for (int k = 2; k <= np2; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      __syncthreads();
      for (int t = threadIdx.x; t < np2 / 2; t += SMALL_T) {
        const int i = 2 * t - (t & (j - 1)), p = i + j;
        const unsigned long long a = e[i], b = e[p];
        if ((a > b) == ((i & k) == 0)) {
          e[i] = b;
          e[p] = a;
        }
      }
    }
  __syncthreads();
  for (int q = threadIdx.x; q < n; q += SMALL_T) {
    steps[q] = (int32_t)(e[q] >> 32);
    idx[q] = (int32_t)(e[q] & 0xFFFFFFFFu);
  }
}

template <typename K>
__global__ __launch_bounds__(RT) void k_raster_keys(const Regions g, uint32_t n, int64_t first, int ib, K *keys) {
  const uint32_t q = blockIdx.x * RT + threadIdx.x;
  if (q >= n) return;
  const unsigned long long e = region_entry(g, q);
  keys[q] = (K)(((unsigned long long)((int64_t)(e >> 32) - first) << ib) | (e & 0xFFFFFFFFull));
}

// counts of each digit in each tile: hist[digit][tile]
template <typename K>
__global__ __launch_bounds__(RT) void k_radix_count(const K *in, uint32_t n, int shift, uint32_t *hist, int ntiles) {
  __shared__ uint32_t cnt[256];
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  const uint32_t b = blockIdx.x * RTILE;
#pragma unroll
  for (int r = 0; r < RROUNDS; ++r) {
    const uint32_t q = b + r * RT + threadIdx.x;
    if (q < n) atomicAdd(&cnt[(uint32_t)(in[q] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
}

// inclusive scan of one value per thread over a workgroup of RT threads
__device__ inline uint32_t block_scan(uint32_t v, uint32_t *wsum) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(v, o);
    if (lane >= o) v += y;
  }
  if (lane == 63) wsum[wv] = v;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (int q = 0; q < RT / 64; ++q)
    if (q < wv) before += wsum[q];
  __syncthreads();
  return v + before;
}

// workgroup d: exclusive scan of digit d's counts over the tiles, its total
__global__ __launch_bounds__(RT) void k_radix_scan(uint32_t *hist, uint32_t *total, int ntiles) {
  __shared__ uint32_t wsum[RT / 64];
  __shared__ uint32_t last;
  uint32_t *h = hist + (size_t)blockIdx.x * ntiles;
  uint32_t carry = 0;
  for (int b = 0; b < ntiles; b += RT) {
    const int i = b + threadIdx.x;
    const uint32_t v = i < ntiles ? h[i] : 0u;
    const uint32_t inc = block_scan(v, wsum);
    if (i < ntiles) h[i] = carry + inc - v;
    if (threadIdx.x == RT - 1) last = inc;
    __syncthreads();
    carry += last;
    __syncthreads();
  }
  if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// Stable scatter of a tile: wavefront w takes the keys [w * 1024, +1024) of
// the tile in order, 64 at a time.
template <typename K, bool LAST>
__global__ __launch_bounds__(RT) void k_radix_scatter(const K *in, uint32_t n, int shift, const uint32_t *hist,
                                                      const uint32_t *total, int ntiles, K *out, int64_t first,
                                                      int ib, int32_t *steps, int32_t *idx) {
  constexpr int NW = RT / 64;
  __shared__ uint32_t cnt[NW][256];
  __shared__ uint32_t wsum[NW];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t t = total[tid];
  const uint32_t base = block_scan(t, wsum) - t + hist[(size_t)tid * ntiles + blockIdx.x];
#pragma unroll
  for (int w = 0; w < NW; ++w) cnt[w][tid] = 0u;
  __syncthreads();
  K key[RROUNDS];
  const uint32_t b = blockIdx.x * RTILE + wv * (64 * RROUNDS) + lane;
#pragma unroll
  for (int r = 0; r < RROUNDS; ++r) {
    const bool on = b + r * 64 < n;
    key[r] = on ? in[b + r * 64] : (K)0;
    if (on) atomicAdd(&cnt[wv][(uint32_t)(key[r] >> shift) & 255u], 1u);
  }
  __syncthreads();
  // first position of each wavefront's keys of digit tid
  uint32_t run = base;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const uint32_t c = cnt[w][tid];
    cnt[w][tid] = run;
    run += c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RROUNDS; ++r) {
    const bool on = b + r * 64 < n;
    const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
    unsigned long long same = __ballot(on);    // lanes holding a key of this digit
    if (same == 0ull) break;                   // past the end, and so are the rounds after
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const bool one = (d >> bit) & 1u;
      const unsigned long long m = __ballot(on && one);
      same &= one ? m : ~m;
    }
    const int leader = on ? __ffsll((long long)same) - 1 : 0;
    uint32_t p = 0;
    if (on && lane == leader) p = atomicAdd(&cnt[wv][d], (uint32_t)__popcll(same));
    p = __shfl(p, leader);
    if (!on) continue;
    p += __popcll(same & ((1ull << lane) - 1ull));
    if constexpr (LAST) {
      steps[p] = (int32_t)(first + (int64_t)(key[r] >> ib));
      idx[p] = (int32_t)((unsigned long long)key[r] & ((1ull << ib) - 1ull));
    } else {
      out[p] = key[r];
    }
  }
}

template <typename K>
void radix(const Regions &g, uint32_t n, int64_t first, int ib, int bits, int32_t *steps, int32_t *idx, void *work,
           hipStream_t st) {
  const int ntiles = (int)((n + RTILE - 1) / RTILE);
  K *a = static_cast<K *>(work), *b = a + n;
  uint32_t *hist = reinterpret_cast<uint32_t *>(b + n), *total = hist + (size_t)256 * ntiles;
  hipLaunchKernelGGL(k_raster_keys<K>, dim3((n + RT - 1) / RT), dim3(RT), 0, st, g, n, first, ib, a);
  for (int shift = 0; shift < bits; shift += 8) {
    hipLaunchKernelGGL(k_radix_count<K>, dim3(ntiles), dim3(RT), 0, st, a, n, shift, hist, ntiles);
    hipLaunchKernelGGL(k_radix_scan, dim3(256), dim3(RT), 0, st, hist, total, ntiles);
    if (shift + 8 >= bits)
      hipLaunchKernelGGL((k_radix_scatter<K, true>), dim3(ntiles), dim3(RT), 0, st, a, n, shift, hist, total, ntiles,
                         b, first, ib, steps, idx);
    else
      hipLaunchKernelGGL((k_radix_scatter<K, false>), dim3(ntiles), dim3(RT), 0, st, a, n, shift, hist, total,
                         ntiles, b, first, ib, steps, idx);
    std::swap(a, b);
  }
}

int bits_of(uint64_t v) {        // bits that hold the values 0..v
  int b = 0;
  while (v >> b) ++b;
  return b;
}

}  // namespace

size_t raster_sort_bytes(int64_t n, int64_t first, int64_t end, int64_t N) {
  if (n <= SMALL) return (size_t)n * 8;
  const int bits = bits_of((uint64_t)(N - 1)) + bits_of((uint64_t)(end - 1 - first));
  const size_t ntiles = (size_t)((n + RTILE - 1) / RTILE);
  return (size_t)n * 8 + 2 * (size_t)n * (bits <= 32 ? 4 : 8) + (256 * ntiles + 256) * 4;
}

void launch_raster_sort(const unsigned long long *base, int64_t stride, const unsigned long long *counts,
                        int64_t first, int64_t end, int64_t N, void *work, hipStream_t st) {
  Regions g{};
  g.base = base;
  g.stride = stride;
  for (int r = 0; r < RSHARD; ++r) g.off[r + 1] = g.off[r] + (uint32_t)counts[r];
  const uint32_t n = g.off[RSHARD];
  if (n == 0) return;
  int32_t *steps = static_cast<int32_t *>(work), *idx = steps + n;
  if (n <= (uint32_t)SMALL) {
    int np2 = 2;
    while (np2 < (int)n) np2 <<= 1;
    hipLaunchKernelGGL(k_raster_small, dim3(1), dim3(SMALL_T), 0, st, g, (int)n, np2, steps, idx);
  } else {
    const int ib = bits_of((uint64_t)(N - 1));
    const int bits = std::max(ib + bits_of((uint64_t)(end - 1 - first)), 1);
    if (bits <= 32) radix<uint32_t>(g, n, first, ib, bits, steps, idx, idx + n, st);
    else radix<uint64_t>(g, n, first, ib, bits, steps, idx, idx + n, st);
  }
  BM_HIP(hipGetLastError());
}

}  // namespace bm
