// wedge.hip — patterns counted by wedges: 4-cycles (P1; single queries and
// every 4-cycle query of a batch in the same launches), P4, P6 and P8.
//
// A root has a set of lists; c_x is the number of them that hold the id x.
//  * P1.  The reference's per-edge value (edges (v0, v1), v1 < v0: sum over v2
//    in N(v0), v2 < v1, of |N(v1) ∩ N(v2) ∩ [0, v0)|;
//    src/message_passing_gpu_kernels.cuh:104-186) summed over a root's edges is
//      sum over x < v0 of C(c_x, 2),  lists N(v) ∩ [0, v0), v in N(v0), v < v0:
//    every pair v2 < v1 of the c_x such v with the common neighbour x is one
//    term.
//  * P8 (:734-818: v1, v2, v3 and x in N(v0), v2 and v3 adjacent to v1, x to v2's
//    and v3's side, v1 the largest and x < v2) is the 4-cycle count of the
//    graph that N(v0) induces, with v1 as its root.  The induced graphs of all
//    roots are laid out as one graph whose vertices are the directed edges
//    (v0, u) (launch_ego_build), so P8 is P1 on that graph.
//  * P6 (:573-652: pairs of S = N(v0) ∩ N(v1), v1 < v0, and a common
//    neighbour of the pair other than v0 and v1): a root is an edge, its lists
//    are N(v), v in S, and the value is sum over x of C(c_x, 2) less C(|S|, 2)
//    for each of x = v0 and x = v1, where c_x = |S|.
//  * P4 (:361-447): lists N(u), u in N(v0); the edge (v0, v1) with s common
//    neighbours adds s times sum over x in N(v1) of c_x (less terms of the
//    triangle counts alone, added elsewhere): a second pass over the lists.
// The sum of C(c_x, 2) needs no second pass over the counters: an increment
// that finds the value k closes k pairs, so adding up what the increments
// return gives it.
//
// Four launches:
//   k_p1_reset     counters and per-root sums to zero (a kernel: capturable)
//   k_p1_len       per list its length (P1, P8: of the part below the root),
//                  and per root the sum W (its wedges) and the number of lists
//   k_p1_classify  roots into lists by W: wave tasks, block tasks, and block
//                  tasks cut into P1_PARTS ranges of x
//   p1_kernel      persistent; block tasks first (the long ones), then wave
//                  tasks.
// All counters live in LDS.  A wave task (W up to 1024, or 512 where ids and
// counts do not share a word) counts in the wave's 8 KB slice, an
// open-addressing table.  A block task walks x downwards in windows that fit
// the block's tables: dense 16-bit counters when a window spans at most 32768
// ids (32-bit and half the ids when a count could pass 65535), else a hash of
// up to 8192 wedges, the window's width chosen from the wedges it holds.
//
// What bounds it: the latency of the list loads behind the LDS segment cursor
// and the LDS atomics; every list is read once (R-MAT 18 P1: 8.6e8 wedges, 3.5
// GB of list elements in 3.2 ms, 1.1 TB/s, 7.7 GB past L2 as whole lines; a
// bank conflict in two of three LDS cycles).  One wave per root with a 32 KB
// table of its own held a CU to 4 waves, and roots above 16384 wedges counted
// in global memory, twice: P1 on R-MAT 18 149 -> 3.2 ms, R-MAT 20 785 -> 17.6
// ms, 3.8M-vertex Chung-Lu 178 -> 6.2 ms.  With an intersection per pair of the
// nest: P4 on R-MAT 14 152 -> 1.1 ms, P6 on R-MAT 11 282 -> 0.59, P8 on R-MAT 12
// 384 -> 0.88, P10 on R-MAT 10 173 -> 0.46.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "clique_dev.hpp"  // seg_advance, wave_sum_u64, wave_take
#include "kernels.hpp"
#include "sym_dev.hpp"

namespace jk {

using symd::lane;
using symd::lb;

namespace {

// Waves per block, the CU's LDS holding 16 / P1_WAVES blocks: one block waits at
// its barriers while the others work.  16 / 8 / 4 waves: R-MAT 18 3.8 / 3.2 /
// 4.4 ms, R-MAT 20 20.9 / 17.6 / 29.9, 3.8M-vertex Chung-Lu 7.0 / 6.2 / 5.7
// (narrower dense windows and the last split roots' tail cost the 4-wave form).
constexpr int P1_WAVES = 8;
constexpr int P1_SLICE = 2048;         // 32-bit words of LDS counters per wave task (8 KB)
constexpr int P1_TAB = P1_SLICE * P1_WAVES;  // ... per block task
constexpr int P1_PARTS = 16;           // x ranges of a split root
// roots with more wedges are split: 16 blocks then share what would be the
// last block's work (R-MAT 18: its widest root holds 5.6M of 863M wedges, more
// than a CU's average share)
constexpr uint64_t P1_SPLIT = 1ull << 19;
constexpr uint32_t P1_EMPTY = 0xffffffffu;

enum { W_P1 = WEDGE_P1, W_P4 = WEDGE_P4, W_P6 = WEDGE_P6 };  // P8 is W_P1 on another graph
enum { C_WAVE = 0, C_BLOCK = 1, C_SPLIT = 2, C_POPB = 3, C_POPW = 4 };

// A table slot is one word (key << cb | count) when the ids of the window
// (span of them) and the counts (at most m, the root's neighbours below it)
// fit 32 bits together, else a key word and a count word.  Returns cb, or 0.
// (EMPTY would be the largest key with the count 2^cb - 1 > m.)
__device__ __forceinline__ int packed_bits(int64_t span, int m) {
  const int cb = 32 - __builtin_clz((unsigned)m + 1u);
  return cb < 32 && span <= ((int64_t)1 << (32 - cb)) ? cb : 0;
}
// most wedges of a table of `words` words (load <= 1/2)
__device__ __forceinline__ int table_cap(int words, int cb) { return cb ? words / 2 : words / 4; }

__device__ __forceinline__ int find_prefix(const int64_t* cs, int n, int64_t t) {
  int lo = 0, hi = n;  // last i with cs[i] <= t
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cs[mid] <= t) lo = mid; else hi = mid;
  }
  return lo;
}

// the ids x of a root: [first, end); its lists are sorted over them
__device__ __forceinline__ int64_t first_id(const P1Q& Q, int32_t root) {
  return Q.csrc ? Q.crp[Q.csrc[root]] - Q.cbase : Q.xmin;
}
template <int M>
__device__ __forceinline__ int64_t end_id(const P1Q& Q, int32_t root) { return M == W_P1 ? root : Q.xend; }

__global__ void k_p1_reset(P1Args a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 8) a.ctr[i] = 0;
  for (int64_t k = i; k < a.roots; k += (int64_t)gridDim.x * blockDim.x) {
    a.W[k] = 0;
    a.m0[k] = 0;
  }
}

template <int M>
__global__ void __launch_bounds__(256) k_p1_len(P1Args a) {
  const int64_t tile = blockIdx.x;
  const int qi = a.q ? find_prefix(a.tcs, a.nq, tile) : 0;
  const P1Q Q = a.q ? a.q[qi] : a.one;
  const int64_t k = (tile - (a.q ? a.tcs[qi] : 0)) * 256 + threadIdx.x;
  int32_t v0 = -1, len = 0;
  if (k < Q.ne) {
    const int64_t e = Q.e0 + k;
    v0 = Q.src[e];
    const int32_t v = Q.ci[e];
    if constexpr (M == W_P1) {
      if (v < v0) {
        const int64_t b = Q.rp[v];
        len = lb(Q.ci + b, (int)(Q.rp[v + 1] - b), v0);  // x < v0
        if (e + 1 == Q.rp[v0 + 1] || Q.ci[e + 1] > v0) a.m0[Q.roff + v0 - Q.rb] = (int32_t)(e + 1 - Q.rp[v0]);
      }
    } else if constexpr (M == W_P4) {  // every list; only roots with a triangle on an edge to a smaller id
      len = (int32_t)(Q.rp[v + 1] - Q.rp[v]);
      if (v < v0 && Q.weight[e] > 0) a.m0[Q.roff + v0 - Q.rb] = (int32_t)(Q.rp[v0 + 1] - Q.rp[v0]);
    } else {  // W_P6: v0 is an edge, v the edge to a member of S
      const int32_t s = (int32_t)(Q.rp[v0 + 1] - Q.rp[v0]);
      if (s >= 2 && Q.vid[v0] < Q.csrc[v0]) {
        const int32_t y = Q.vid[v];
        len = (int32_t)(Q.lrp[y + 1] - Q.lrp[y]);
        if (e == Q.rp[v0]) a.m0[Q.roff + v0 - Q.rb] = s;
      }
    }
    a.len[Q.eoff + k] = len;
  }
  // per-root sums: a suffix sum within each run of equal sources of the wave
  // (edges are grouped by source), one atomic per run
  const int ln = lane();
  int64_t s = len;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t y = (int64_t)__shfl_down((unsigned long long)s, o);
    const int32_t r = __shfl_down(v0, o);
    if (ln + o < 64 && r == v0) s += y;
  }
  const int32_t before = __shfl_up(v0, 1);
  if (v0 >= 0 && s && (ln == 0 || before != v0))
    atomicAdd((unsigned long long*)&a.W[Q.roff + v0 - Q.rb], (unsigned long long)s);
}

template <int M>
__global__ void __launch_bounds__(256) k_p1_classify(P1Args a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int ln = lane();
  int cls = -1;
  int2 item = make_int2(0, 0);
  if (t < a.roots) {
    const int64_t i = a.roots - 1 - t;  // a relabelled graph ranks its widest roots last: list them first
    const uint64_t w = a.W[i];
    const int m0 = a.m0[i];
    if (w >= (M == W_P4 ? 1 : 2) && m0 > 0) {  // else no two wedges share an endpoint
      item.y = a.q ? find_prefix(a.rcs, a.nq, i) : 0;
      const P1Q& Q = a.q ? a.q[item.y] : a.one;
      item.x = (int32_t)(Q.rb + i - Q.roff);
      const int64_t span = end_id<M>(Q, item.x) - (M == W_P1 && Q.csrc ? first_id(Q, item.x) : 0);
      const int cap = table_cap(P1_SLICE, packed_bits(span, m0));
      cls = w <= (uint64_t)cap ? C_WAVE : w <= P1_SPLIT ? C_BLOCK : C_SPLIT;
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const uint64_t m = __ballot(cls == c);
    if (!m) continue;
    const unsigned long long base = wave_take(a.ctr + c, (unsigned long long)__popcll(m));
    if (cls == c) {
      const int64_t k = (int64_t)base + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      // the wave list grows from the front and the block list from the back
      // of one array of `roots` items; no root is in both
      if (c == C_WAVE) a.list[k] = item;
      else if (c == C_BLOCK) a.list[a.roots - 1 - k] = item;
      else a.split[k] = item;
    }
  }
}

// The segments of up to 64 neighbours (lane l: len elements from ci[base]) as
// one flattened stream, four loads in flight per lane; f(x, i) for every
// element x of lane i's segment.
template <class F>
__device__ __forceinline__ void stream64(const int32_t* ci, int64_t base, int len, int32_t* off, int64_t* lbase, F f) {
  const int ln = lane();
  const int incl = wave_incl_scan(len);
  const int T = __shfl(incl, 63);
  __syncwarp();  // the arrays are free again
  off[ln] = incl - len;
  lbase[ln] = base - (incl - len);  // element f of the lane's segment is ci[lbase + f]
  if (ln == 63) off[64] = T;
  __syncwarp();
  int i = 0;
  for (int f0 = ln; f0 < T; f0 += 256) {
    int32_t x[4];
    int seg[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int fe = f0 + 64 * u;
      if (fe < T) {
        i = seg_advance(off, 64, i, fe);
        seg[u] = i;
        x[u] = ci[lbase[i] + fe];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (f0 + 64 * u < T) f(x[u], seg[u]);
  }
}

// one wedge to the id `x` of the window in an open-addressing table of 2^lt
// slots: the wedges to x counted before.  cb: packed_bits; otherwise the
// counts follow the keys.
__device__ __forceinline__ uint32_t table_count(uint32_t* tab, int lt, int cb, uint32_t x) {
  uint32_t h = (x * 2654435761u) >> (32 - lt);
  const uint32_t mask = (1u << lt) - 1;
  if (cb) {
    for (;;) {
      uint32_t k = tab[h];
      if (k == P1_EMPTY) {
        k = atomicCAS(&tab[h], P1_EMPTY, (x << cb) | 1u);
        if (k == P1_EMPTY) return 0;
      }
      if ((k >> cb) == x) return atomicAdd(&tab[h], 1u) & ((1u << cb) - 1);
      h = (h + 1) & mask;
    }
  }
  for (;;) {
    uint32_t k = tab[h];
    if (k == P1_EMPTY) {
      k = atomicCAS(&tab[h], P1_EMPTY, x);
      if (k == P1_EMPTY) k = x;
    }
    if (k == x) return atomicAdd(&tab[mask + 1 + h], 1u);
    h = (h + 1) & mask;
  }
}

// the wedges to x counted in such a table (x is in it)
__device__ __forceinline__ uint32_t table_get(const uint32_t* tab, int lt, int cb, uint32_t x) {
  uint32_t h = (x * 2654435761u) >> (32 - lt);
  const uint32_t mask = (1u << lt) - 1;
  while ((cb ? tab[h] >> cb : tab[h]) != x) h = (h + 1) & mask;
  return cb ? tab[h] & ((1u << cb) - 1) : tab[mask + 1 + h];
}

// empties such a table (t4: its words as 16-byte groups), thread t of nt
__device__ __forceinline__ void table_clear(uint4* t4, int lt, int cb, int t, int nt) {
  const int g = (1 << lt) / 4;
  for (int k = t; k < g; k += nt) {
    t4[k] = make_uint4(P1_EMPTY, P1_EMPTY, P1_EMPTY, P1_EMPTY);
    if (!cb) t4[g + k] = make_uint4(0u, 0u, 0u, 0u);
  }
}

// lower bounds of several ids in one list (n entries), their loads overlapping
template <int K>
__device__ __forceinline__ void lb_many(const int32_t* l, int n, const int32_t (&y)[K], int (&pos)[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) pos[k] = 0;
  int step = n > 0 ? 1 << (31 - __builtin_clz(n)) : 0;
  for (; step; step >>= 1) {
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (pos[k] + step <= n && l[pos[k] + step - 1] < y[k]) pos[k] += step;
  }
}

template <int M>
__global__ void __launch_bounds__(64 * P1_WAVES) p1_kernel(P1Args a) {
  constexpr bool TWO = M == W_P4;  // a second pass over the lists reads the counters

  __shared__ __attribute__((aligned(16))) uint32_t s_tab[P1_TAB];
  __shared__ int32_t s_off[P1_WAVES][65];
  __shared__ int64_t s_lb[P1_WAVES][64];
  __shared__ int32_t s_wt[TWO ? P1_WAVES : 1][64];
  __shared__ int64_t s_task;
  __shared__ unsigned long long s_tot[3];
  __shared__ int s_next;
  constexpr int NT = 64 * P1_WAVES;
  const int tid = threadIdx.x;
  const int wv = tid >> 6;
  const int ln = lane();
  int32_t* off = s_off[wv];
  int64_t* lbs = s_lb[wv];
  int32_t* const wts = s_wt[TWO ? wv : 0];
  uint64_t acc = 0;
  int slot = 0;  // the query that acc belongs to
  auto flush = [&](int next) {
    if (next == slot) return;
    const uint64_t s = wave_sum_u64(acc) * (uint64_t)(a.q ? 1 : a.one.scale);
    if (ln == 0 && s) atomicAdd((unsigned long long*)(a.out + slot), (unsigned long long)s);
    acc = 0;
    slot = next;
  };
  if (!a.q) slot = a.one.slot;

  // ---- block tasks
  const int64_t nsplit = (int64_t)a.ctr[C_SPLIT] * P1_PARTS, nblock = (int64_t)a.ctr[C_BLOCK];
  for (;;) {
    __syncthreads();
    if (tid == 0) s_task = (int64_t)atomicAdd(a.ctr + C_POPB, 1ull);
    __syncthreads();
    const int64_t t = s_task;
    if (t >= nsplit + nblock) break;
    const bool part = t < nsplit;
    const int2 it = part ? a.split[t / P1_PARTS] : a.list[a.roots - 1 - (t - nsplit)];
    const P1Q Q = a.q ? a.q[it.y] : a.one;
    flush(Q.slot);
    const int32_t* ci = M == W_P6 ? Q.lci : Q.ci;  // the lists' elements
    const int32_t v0 = it.x;
    const int64_t b0 = Q.rp[v0];
    const int32_t* N0 = Q.ci + b0;
    // start of the j-th list
    auto list_at = [&](int j) -> int64_t { return M == W_P6 ? Q.lrp[Q.vid[N0[j]]] : Q.rp[N0[j]]; };
    // neighbours below the window's end, per list; a root that is one task
    // moves them down as its windows descend
    int32_t* lens = a.len + Q.eoff + (b0 - Q.e0);
    const int m0 = a.m0[Q.roff + v0 - Q.rb];
    const uint64_t W = a.W[Q.roff + v0 - Q.rb];
    int64_t xlo = M == W_P6 ? 0 : first_id(Q, v0), xhi = end_id<M>(Q, v0);
    const int64_t xend = xhi;
    if (part) {
      const int64_t span = xhi - xlo;
      const int p = (int)(t % P1_PARTS);
      xhi = xlo + span * (p + 1) / P1_PARTS;
      xlo = xlo + span * p / P1_PARTS;
    }
    const bool wide = m0 > 65535;  // a count may not fit 16 bits
    const int64_t DW = wide ? P1_TAB : 2 * P1_TAB;
    const int cs = max(1, min(64, (m0 + P1_WAVES - 1) / P1_WAVES));
    uint64_t left = W;           // wedges below the window's end
    int64_t hi = xhi, step = DW;
    while (hi > xlo) {
      // the window [lo, hi): everything left if it fits a table; dense
      // counters if it spans at most DW ids; else the widest of three widths
      // whose wedges fit
      int64_t lo = max(xlo, hi - step);
      bool dense = hi - lo <= DW;
      uint64_t tot = left;
      if (!part && hi - xlo > DW) {
        const int cap_all = table_cap(P1_TAB, packed_bits(hi - xlo, m0));
        if (left <= (uint64_t)cap_all) {
          lo = xlo;
          dense = false;
        } else if (!dense) {
          int32_t y[3];
#pragma unroll
          for (int k = 0; k < 3; ++k) y[k] = (int32_t)max(xlo, hi - max(DW, step << (2 - k) >> 1));  // 2, 1, 1/2 steps
          __syncthreads();
          if (tid < 3) s_tot[tid] = 0;
          __syncthreads();
          int64_t c[3] = {0, 0, 0};
          for (int j = tid; j < m0; j += NT) {
            const int n = lens[j];
            if (!n) continue;
            int pos[3];
            lb_many<3>(ci + list_at(j), n, y, pos);
#pragma unroll
            for (int k = 0; k < 3; ++k) c[k] += n - pos[k];
          }
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const uint64_t w = wave_sum_u64((uint64_t)c[k]);
            if (ln == 0 && w) atomicAdd(&s_tot[k], (unsigned long long)w);
          }
          __syncthreads();
          int best = -1;
#pragma unroll
          for (int k = 2; k >= 0; --k)
            if (s_tot[k] <= (uint64_t)table_cap(P1_TAB, packed_bits(hi - y[k], m0))) best = k;
          if (best < 0) {
            if (step <= 2 * DW) step = DW;
            else step = max(DW, step >> 2);
            continue;
          }
          lo = y[best];
          tot = s_tot[best];
          step = hi - lo;
          dense = step <= DW;
        }
      }
      const int cb = packed_bits(hi - lo, m0);
      int lt = 6;
      if (!dense)
        while ((1ull << lt) < 2 * tot) ++lt;
      // clear what this window uses
      __syncthreads();
      uint4* t4 = reinterpret_cast<uint4*>(s_tab);
      if (dense) {
        const int words = (int)(wide ? hi - lo : (hi - lo + 1) / 2);
        for (int k = tid; k < (words + 3) / 4; k += NT) t4[k] = make_uint4(0u, 0u, 0u, 0u);
      } else {
        table_clear(t4, lt, cb, tid, NT);
      }
      if (tid == 0) {
        s_next = 0;
        s_tot[0] = 0;
      }
      __syncthreads();
      const int32_t lo32 = (int32_t)lo;
      for (int pass = 0; pass < (TWO ? 2 : 1); ++pass) {
        if (pass) {
          __syncthreads();
          if (tid == 0) s_next = 0;
          __syncthreads();
        }
        const bool last = !TWO || pass == 1;
        for (;;) {
          const int jb = wave_take(&s_next, cs);
          if (jb >= m0) break;
          const int j = jb + ln;
          int len = 0;
          int64_t base = 0;
          if (ln < cs && j < m0) {
            int n = lens[j];
            if (n) {
              base = list_at(j);
              if (part && hi < xend) n = lb(ci + base, n, (int32_t)hi);
              const int s = lo32 > 0 ? lb(ci + base, n, lo32) : 0;
              if (!part && last) lens[j] = s;
              len = n - s;
              base += s;
            }
          }
          if (!part && last) {
            const int w = (int)wave_sum_u64((uint64_t)len);
            if (ln == 0 && w) atomicAdd(&s_tot[0], (unsigned long long)w);
          }
          if (TWO && pass) {
            // the edge to a smaller id with s common neighbours: s times the
            // counts of its list's elements
            int32_t wt = 0;
            if (len && N0[j] < v0) wt = Q.weight[b0 + j];
            if (wt == 0) len = 0;
            wts[ln] = wt;
            stream64(ci, base, len, off, lbs, [&](int32_t x, int i) {
              const uint32_t k = (uint32_t)(x - lo32);
              const uint32_t c = !dense ? table_get(s_tab, lt, cb, k)
                                 : wide ? s_tab[k]
                                        : (s_tab[k >> 1] >> ((k & 1u) * 16u)) & 0xffffu;
              acc += (uint64_t)wts[i] * c;
            });
          } else if (dense) {
            if (wide) {
              stream64(ci, base, len, off, lbs, [&](int32_t x, int) {
                const uint32_t c = atomicAdd(&s_tab[x - lo32], 1u);
                if (!TWO) acc += c;
              });
            } else {
              stream64(ci, base, len, off, lbs, [&](int32_t x, int) {
                const uint32_t i = (uint32_t)(x - lo32), sh = (i & 1u) * 16u;
                const uint32_t c = (atomicAdd(&s_tab[i >> 1], 1u << sh) >> sh) & 0xffffu;
                if (!TWO) acc += c;
              });
            }
          } else {
            stream64(ci, base, len, off, lbs, [&](int32_t x, int) {
              const uint32_t c = table_count(s_tab, lt, cb, (uint32_t)(x - lo32));
              if (!TWO) acc += c;
            });
          }
        }
      }
      if (!part) {
        __syncthreads();
        const uint64_t did = s_tot[0];
        left -= did;
        // sparser further down: a wider window next
        if (did < (uint64_t)P1_TAB / 4) step *= 4;
      }
      hi = lo;
    }
  }

  // ---- wave tasks
  __syncthreads();
  uint32_t* tab = s_tab + wv * P1_SLICE;
  const int64_t nwave = (int64_t)a.ctr[C_WAVE];
  // tasks per grab: an atomic on one address takes about 12 ns, so 4 at a time
  // bound the launch on large sparse graphs (Chung-Lu, 3.8M vertices: 8.9 ms,
  // 6.8 so)
  const int64_t chunk = max((int64_t)4, min((int64_t)32, nwave / ((int64_t)gridDim.x * P1_WAVES * 12)));
  for (;;) {
    const int64_t tb = (int64_t)wave_take(a.ctr + C_POPW, (unsigned long long)chunk);
    if (tb >= nwave) break;
    for (int64_t t = tb; t < min(nwave, tb + chunk); ++t) {
      const int2 it = a.list[t];
      const P1Q Q = a.q ? a.q[it.y] : a.one;
      flush(Q.slot);
      const int32_t v0 = it.x;
      const int64_t b0 = Q.rp[v0];
      const int32_t* lens = a.len + Q.eoff + (b0 - Q.e0);
      const int m0 = a.m0[Q.roff + v0 - Q.rb];
      const int W = (int)a.W[Q.roff + v0 - Q.rb];
      const int32_t xlo = M == W_P1 && Q.csrc ? (int32_t)first_id(Q, v0) : 0;
      const int cb = packed_bits(end_id<M>(Q, v0) - xlo, m0);
      int lt = 6;
      while ((1 << lt) < 2 * W) ++lt;
      __syncwarp();
      table_clear(reinterpret_cast<uint4*>(tab), lt, cb, ln, 64);
      for (int pass = 0; pass < (TWO ? 2 : 1); ++pass) {
        for (int jb = 0; jb < m0; jb += 64) {
          const int j = jb + ln;
          int len = j < m0 ? lens[j] : 0;
          const int32_t v = len ? Q.ci[b0 + j] : 0;
          const int64_t base = len ? (M == W_P6 ? Q.lrp[Q.vid[v]] : Q.rp[v]) : 0;
          const int32_t* ci = M == W_P6 ? Q.lci : Q.ci;
          if (TWO && pass) {
            const int32_t wt = len && v < v0 ? Q.weight[b0 + j] : 0;
            if (wt == 0) len = 0;
            wts[ln] = wt;
            stream64(ci, base, len, off, lbs, [&](int32_t x, int i) {
              acc += (uint64_t)wts[i] * table_get(tab, lt, cb, (uint32_t)x);
            });
          } else {
            stream64(ci, base, len, off, lbs, [&](int32_t x, int) {
              const uint32_t c = table_count(tab, lt, cb, (uint32_t)(x - xlo));
              if (!TWO) acc += c;
            });
          }
        }
      }
    }
  }
  flush(-1);
}

}  // namespace

size_t p1_scratch_bytes(int64_t roots, int64_t edges) {
  return 64 + (size_t)roots * (sizeof(uint64_t) + 2 * sizeof(int2) + sizeof(int32_t)) + (size_t)edges * sizeof(int32_t);
}

void p1_bind_scratch(P1Args& a, void* p) {
  unsigned char* b = static_cast<unsigned char*>(p);
  a.ctr = reinterpret_cast<unsigned long long*>(b);
  b += 64;
  a.W = reinterpret_cast<uint64_t*>(b);
  b += sizeof(uint64_t) * (size_t)a.roots;
  a.list = reinterpret_cast<int2*>(b);
  b += sizeof(int2) * (size_t)a.roots;
  a.split = reinterpret_cast<int2*>(b);
  b += sizeof(int2) * (size_t)a.roots;
  a.m0 = reinterpret_cast<int32_t*>(b);
  b += sizeof(int32_t) * (size_t)a.roots;
  a.len = reinterpret_cast<int32_t*>(b);
}

template <int M>
static hipError_t launch_wedge_m(const P1Args& a, int num_cu, hipStream_t st) {
  if (a.tiles <= 0 || a.roots <= 0) return hipSuccess;
  const unsigned rblocks = (unsigned)((a.roots + 255) / 256);
  hipLaunchKernelGGL(k_p1_reset, dim3(rblocks < 1024u ? rblocks : 1024u), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_p1_len<M>, dim3((unsigned)a.tiles), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_p1_classify<M>, dim3(rblocks), dim3(256), 0, st, a);
  const int64_t want = (a.roots + P1_WAVES - 1) / P1_WAVES, most = (int64_t)num_cu * (16 / P1_WAVES);
  hipLaunchKernelGGL(p1_kernel<M>, dim3((unsigned)(want < most ? want : most)), dim3(64 * P1_WAVES), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_wedge(int mode, const P1Args& a, int num_cu, hipStream_t st) {
  switch (mode) {
    case WEDGE_P1: return launch_wedge_m<W_P1>(a, num_cu, st);
    case WEDGE_P4: return launch_wedge_m<W_P4>(a, num_cu, st);
    case WEDGE_P6: return launch_wedge_m<W_P6>(a, num_cu, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace jk
