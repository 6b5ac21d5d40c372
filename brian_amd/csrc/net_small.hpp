// Small networks that advance one step per launch (a connection without
// delay, or STDP), advanced instead by one workgroup through a whole run in
// one launch.  Compiled at run time (hipRTC) from the network's structure:
// net.hip:small_source generates a struct SG<i> per group (its model as code,
// as for k_lean), and the kernel body that calls the templates below for each
// group, connection and STDP in order.
//
// Everything a step touches stays on one compute unit: state and last spike
// steps in registers (thread t holds neurons t, t + 1024, ...), the rings of
// pending deliveries, the spike lists and the STDP traces in LDS; only rows of
// the connectivity, plastic weights and the raster go to memory.  Step n:
//   phase 1  per neuron: tail of step n-1 (deliveries of ring slot n-1, then
//            resets), head of step n (update, threshold); spikes to the
//            group's list; STDP traces decay
//   barrier
//   phase 2  the lists' rows, shared out over the wavefronts: deliveries into
//            ring slots n + d, STDP's pre updates of the same synapses (each
//            weight read for its delivery before its update, the order of
//            sweep and k_stdp_pre); raster
//   barrier
//   phase 3  only where a group with STDP spiked: post updates, barrier
// The per-neuron arithmetic is k_lean's (or the general sweep's, for groups
// that run it), the deliveries add the same counts: rasters and state equal
// the windowed kernels' bit for bit where deliveries are counts, and up to the
// order of the floating additions otherwise.
//
// Why one workgroup: a step is a chain of memory round trips and barriers, not
// work (4000 neurons: 2.4 spikes, 190 synapses).  A launch per step pays the
// launch and the loads of everything anew; here a step costs two barriers and
// the chain row pointer -> columns.
#pragma once
#include "net_kernels.hpp"

namespace bm {

constexpr int SMT = SMALL_THREADS;
constexpr int SMW = SMT / 64;

template <class G>
struct SmallRegs {
  typename G::T x[G::K][G::M > 0 ? G::M : 1];
  int32_t last[G::K];
};

// LDS of group G
template <class G>
__device__ inline uint32_t *small_words(unsigned char *sm, const SmallNet &sn, int r) {
  return reinterpret_cast<uint32_t *>(sm + sn.ring_off[G::GI][r]);
}
template <class G>
__device__ inline typename G::T *small_floats(unsigned char *sm, const SmallNet &sn, int r) {
  return reinterpret_cast<typename G::T *>(sm + sn.ring_off[G::GI][r]);
}

// State into registers, pending deliveries into the LDS rings.
template <class G>
__device__ inline void small_load(const GroupDev &g, SmallRegs<G> &r, unsigned char *sm, const SmallNet &sn, int tid) {
  const int N = (int)g.N;
#pragma unroll
  for (int k = 0; k < G::K; ++k) {
    const int i = k * SMT + tid;
    r.last[k] = i < N ? g.last[i] : NEVER;
#pragma unroll
    for (int j = 0; j < G::M; ++j)
      r.x[k][j] = i < N ? static_cast<const typename G::T *>(g.S)[(int64_t)j * N + i] : (typename G::T)0;
  }
#pragma unroll
  for (int q = 0; q < G::NRING; ++q) {
    const RingDev &rd = g.rings[q];
    for (int d = 0; d < g.D; ++d) {
      const unsigned char *slot = static_cast<const unsigned char *>(rd.base) + (int64_t)d * rd.slot_bytes;
      for (int i = tid; i < N; i += SMT) {
        if (G::RCOUNT[q]) small_words<G>(sm, sn, q)[d * N + i] = load_slice(slot, i, rd.sw);
        else small_floats<G>(sm, sn, q)[d * N + i] = reinterpret_cast<const typename G::T *>(slot)[i];
      }
    }
  }
}

template <class G>
__device__ inline void small_store(const GroupDev &g, SmallRegs<G> &r, unsigned char *sm, const SmallNet &sn, int tid) {
  const int N = (int)g.N;
#pragma unroll
  for (int k = 0; k < G::K; ++k) {
    const int i = k * SMT + tid;
    if (i >= N) continue;
    g.last[i] = r.last[k];
#pragma unroll
    for (int j = 0; j < G::M; ++j) static_cast<typename G::T *>(g.S)[(int64_t)j * N + i] = r.x[k][j];
  }
#pragma unroll
  for (int q = 0; q < G::NRING; ++q) {
    const RingDev &rd = g.rings[q];
    for (int d = 0; d < g.D; ++d) {
      unsigned char *slot = static_cast<unsigned char *>(rd.base) + (int64_t)d * rd.slot_bytes;
      for (int i = tid; i < N; i += SMT) {
        if (!G::RCOUNT[q]) {
          reinterpret_cast<typename G::T *>(slot)[i] = small_floats<G>(sm, sn, q)[d * N + i];
          continue;
        }
        const uint32_t w = small_words<G>(sm, sn, q)[d * N + i];
        if (rd.sw == 2) reinterpret_cast<uint16_t *>(slot)[i] = (uint16_t)w;
        else if (rd.sw == 1) slot[i] = (unsigned char)w;
        else reinterpret_cast<uint32_t *>(slot)[i] = w;
      }
    }
  }
  if (g.hist_count != nullptr)
    for (int q = tid; q < g.H; q += SMT) g.hist_count[q] = 0u;   // nothing pending: delays are 0
}

// Tail of step n-1 for neuron i, slot k: deliveries of ring slot sl, resets.
template <class G>
__device__ inline void small_tail(const GroupDev &g, const typename G::KV &kv, SmallRegs<G> &r, unsigned char *sm, const SmallNet &sn, int64_t n,
                                  int sl, int k, int i) {
  using T = typename G::T;
  uint32_t w[MAXRING];
  T f[MAXRING];
  const int at = sl * (int)g.N + i;
#pragma unroll
  for (int q = 0; q < G::NRING; ++q) {
    w[q] = 0u;
    f[q] = (T)0;
    if (G::RCOUNT[q]) {
      w[q] = small_words<G>(sm, sn, q)[at];
      small_words<G>(sm, sn, q)[at] = 0u;
    } else {
      f[q] = small_floats<G>(sm, sn, q)[at];
      small_floats<G>(sm, sn, q)[at] = (T)0;
    }
  }
  G::deliver(r.x[k], w, f, kv);
  if (r.last[k] == NEVER) return;
  if constexpr (G::REFR == 0) {
    if (r.last[k] == (int32_t)(n - 1)) G::reset(r.x[k], kv);
  } else if ((n - 1) - (int64_t)r.last[k] < (int64_t)g.period) {
    if constexpr (G::REFR == 2) {
      const double na = (double)r.last[k] * g.dt + g.refr_arr[i];
      if (na > ((double)(n - 1) * g.dt - g.dt * 0.25)) G::reset(r.x[k], kv);
    } else {
      G::reset(r.x[k], kv);
    }
  }
}

// Phase 1 of a group: tail of step n-1 (unless skipped), head of step n.
template <class G>
__device__ inline void small_sweep(const GroupDev &g, const typename G::KV &kv, SmallRegs<G> &r, unsigned char *sm, const SmallNet &sn, int64_t n,
                                   bool tail, int sl, int *cnt, int tid) {
  const int N = (int)g.N, lane = tid & 63;
  uint16_t *list = reinterpret_cast<uint16_t *>(sm + sn.list_off[G::GI]);
#pragma unroll
  for (int k = 0; k < G::K; ++k) {
    const int i = k * SMT + tid;
    bool sp = false;
    if (i < N) {
      if constexpr (G::POISSON) {
        uint64_t thr = g.pthr[i];
        const int64_t row = n - g.ptab_n0;
        if (g.ptab && row >= 0 && row < g.ptab_len) thr = g.ptab[g.ptab_per_neuron ? row * N + i : row];
        sp = (uint64_t)counter_u32(g.seed, (uint64_t)i, (uint64_t)n) < thr;
      } else {
        if (tail) small_tail<G>(g, kv, r, sm, sn, n, sl, k, i);
        G::update(r.x[k], kv);
        sp = G::spike(r.x[k], kv);
        if constexpr (G::REFR != 0) {
          if (sp && r.last[k] != NEVER) {
            // next allowed spike time in seconds, as the general sweep tests it
            const double t = (double)n * g.dt + 0.0;
            const double lt = (double)r.last[k] * g.dt + 0.0;
            sp = lt + (G::REFR == 2 ? g.refr_arr[i] : g.refr_time) <= t;
          }
        }
      }
      if (sp) r.last[k] = (int32_t)n;
    }
    const unsigned long long mask = __ballot(sp);
    if (mask == 0ull) continue;
    int base = 0;
    const int leader = __ffsll((long long)mask) - 1;
    if (lane == leader) base = atomicAdd(cnt, __popcll(mask));
    base = __shfl(base, leader);
    if (sp) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = (uint16_t)i;
  }
}

// The last tail of a run.
template <class G>
__device__ inline void small_finish(const GroupDev &g, const typename G::KV &kv, SmallRegs<G> &r, unsigned char *sm, const SmallNet &sn,
                                    int64_t n, int sl, int tid) {
  if constexpr (!G::POISSON) {
#pragma unroll
    for (int k = 0; k < G::K; ++k)
      if (k * SMT + tid < (int)g.N) small_tail<G>(g, kv, r, sm, sn, n, sl, k, k * SMT + tid);
  }
}

// Phase 2 of a connection from group GS to ring C::RING of group GT: the
// source's S spikes, RS lanes to a row, wavefront chunks dealt on from `turn`
// over the connections of a step.
template <class C>
__device__ inline void small_propagate(const OutDev &od, const StdpDev *sd, unsigned char *sm, const SmallNet &sn,
                                       int S, int slot_n, int Dt, int Nt, int &turn, int tid) {
  using T = typename C::T;
  constexpr int PER = 64 / C::RS;
  const int lane = tid & 63, wv = tid >> 6;
  const int sub = lane / C::RS, sl = lane & (C::RS - 1);
  const uint16_t *list = reinterpret_cast<const uint16_t *>(sm + sn.list_off[C::SRC]);
  const int j0 = (wv - turn) & (SMW - 1);
  turn += (S + PER - 1) / PER;
  for (int p = j0 * PER + sub; p < S; p += SMW * PER) {
    const int64_t r = (int64_t)list[p] - od.src_off;
    if (r < 0 || r >= od.src_n) continue;
    const int64_t lo = od.row_ptr[r], hi = od.row_ptr[r + 1];
    T *apost = nullptr;
    if constexpr (C::STDP >= 0) {
      T *apre = reinterpret_cast<T *>(sm + sn.pre_off[C::STDP]);
      apost = reinterpret_cast<T *>(sm + sn.post_off[C::STDP]);
      if (sl == 0)
        apre[r] = (sd->interactions == 0 || sd->interactions == 3) ? apre[r] + (T)sd->Ap : (T)sd->Ap;
    }
    for (int64_t q = lo + sl; q < hi; q += C::RS) {
      const int col = od.col[q];
      int d = od.hom_delay;
      if constexpr (C::DLY == 1) d = static_cast<const uint8_t *>(od.dly)[q];
      else if constexpr (C::DLY == 2) d = static_cast<const uint16_t *>(od.dly)[q];
      int s = slot_n + d;
      while (s >= Dt) s -= Dt;
      const int at = s * Nt + (int)od.tgt_off + col;
      if constexpr (C::COUNT) {
        atomicAdd(reinterpret_cast<uint32_t *>(sm + sn.ring_off[C::TGT][C::RING]) + at, 1u << C::SHIFT);
      } else {
        T *w = static_cast<T *>(const_cast<void *>(od.w));
        __hip_atomic_fetch_add(reinterpret_cast<T *>(sm + sn.ring_off[C::TGT][C::RING]) + at, w[q], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        if constexpr (C::STDP >= 0)
          stdp_apply<T>(*sd, w, q, apost[col], sd->pre_mode, sd->pre_off, sd->pre_scale, 1);
      }
    }
  }
}

template <class T>
__device__ inline void small_decay(const StdpDev &sd, unsigned char *sm, const SmallNet &sn, int s, int tid) {
#pragma clang fp contract(off)
  T *a = reinterpret_cast<T *>(sm + sn.pre_off[s]), *b = reinterpret_cast<T *>(sm + sn.post_off[s]);
  for (int i = tid; i < (int)sd.src_n; i += SMT) a[i] = (T)sd.decay_pre * a[i] + (T)0;
  for (int i = tid; i < (int)sd.tgt_n; i += SMT) b[i] = (T)sd.decay_post * b[i] + (T)0;
}

// Phase 3 of one STDP: the columns of the S post spikes, the whole workgroup
// on each while they are few, a wavefront each when they are many.
template <class T>
__device__ inline void small_post(const StdpDev &sd, unsigned char *sm, const SmallNet &sn, int s, int tgt, int S,
                                  int tid) {
#pragma clang fp contract(off)
  const T *apre = reinterpret_cast<const T *>(sm + sn.pre_off[s]);
  T *apost = reinterpret_cast<T *>(sm + sn.post_off[s]);
  const uint16_t *list = reinterpret_cast<const uint16_t *>(sm + sn.list_off[tgt]);
  T *w = static_cast<T *>(sd.w);
  const bool many = S >= SMW;
  const int first = many ? tid & 63 : tid, stride = many ? 64 : SMT;
  for (int p = many ? tid >> 6 : 0; p < S; p += many ? SMW : 1) {
    const int64_t j = (int64_t)list[p] - sd.tgt_off;
    if (j < 0 || j >= sd.tgt_n) continue;
    if (first == 0)
      apost[j] = (sd.interactions == 0 || sd.interactions == 4) ? apost[j] + (T)sd.Am : (T)sd.Am;
    for (int64_t q = sd.col_ptr[j] + first; q < sd.col_ptr[j + 1]; q += stride)
      stdp_apply<T>(sd, w, sd.col_perm[q], apre[sd.col_row[q]], sd.post_mode, sd.post_off, sd.post_scale, 1);
  }
}

// Traces between memory and LDS.
template <class T>
__device__ inline void small_traces(const StdpDev &sd, unsigned char *sm, const SmallNet &sn, int s, bool load,
                                    int tid) {
  T *a = reinterpret_cast<T *>(sm + sn.pre_off[s]), *b = reinterpret_cast<T *>(sm + sn.post_off[s]);
  T *ga = static_cast<T *>(sd.a_pre), *gb = static_cast<T *>(sd.a_post);
  for (int i = tid; i < (int)sd.src_n; i += SMT) {
    if (load) a[i] = ga[i];
    else ga[i] = a[i];
  }
  for (int i = tid; i < (int)sd.tgt_n; i += SMT) {
    if (load) b[i] = gb[i];
    else gb[i] = b[i];
  }
}

// Raster of a group: one wavefront stages entries in LDS and appends
// SMALL_RASTER of them at a time to the append region with the fewest (one
// workgroup fills them all; a region by its block index would take the whole
// raster, and one by the step most of it where runs are of 32 steps).
struct SmallRaster {
  int cnt;
};
__device__ inline void small_raster_flush(const GroupDev &g, const unsigned long long *buf, SmallRaster &rr, int lane) {
  if (rr.cnt == 0) return;
  unsigned long long least = ~0ull;
  if (lane < RSHARD)
    least = __hip_atomic_load(g.raster_count + lane * RSTRIDE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) * RSHARD + lane;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) least = min(least, (unsigned long long)__shfl_xor(least, o));
  const int shard = (int)(least % RSHARD);
  unsigned long long at = 0;
  if (lane == 0) at = atomicAdd(g.raster_count + shard * RSTRIDE, (unsigned long long)rr.cnt);
  at = __shfl(at, 0);
  for (int p = lane; p < rr.cnt; p += 64)
    if (at + p < (unsigned long long)g.raster_cap) g.raster[(int64_t)shard * g.raster_cap + (int64_t)(at + p)] = buf[p];
  rr.cnt = 0;
}
__device__ inline void small_raster(const GroupDev &g, unsigned char *sm, const SmallNet &sn, int gi, int S, int64_t n,
                                    SmallRaster &rr, int lane) {
  const uint16_t *list = reinterpret_cast<const uint16_t *>(sm + sn.list_off[gi]);
  unsigned long long *buf = reinterpret_cast<unsigned long long *>(sm + sn.raster_off[gi]);
  for (int b = 0; b < S;) {
    const int m = min(S - b, SMALL_RASTER - rr.cnt);
    for (int p = lane; p < m; p += 64) buf[rr.cnt + p] = ((uint64_t)n << 32) | (uint64_t)list[b + p];
    rr.cnt += m;
    b += m;
    if (rr.cnt == SMALL_RASTER) small_raster_flush(g, buf, rr, lane);
  }
}

}  // namespace bm
