// p1_wedge.hip — 4-cycles (P1) by wedge counting, for single queries and for
// every 4-cycle query of a batch in the same launches.
//
// The reference's per-edge value (edges (v0, v1), v1 < v0: sum over v2 in
// N(v0), v2 < v1, of |N(v1) ∩ N(v2) ∩ [0, v0)|;
// src/message_passing_gpu_kernels.cuh:104-186) summed over a root's edges is
//   sum over x < v0 of C(c_x, 2),  c_x = |{v in N(v0) : v < v0, x in N(v)}|:
// every pair v2 < v1 of the c_x such v with the common neighbour x is one
// term.  So a root needs one pass over its wedges (v0, v, x) with v, x < v0.
// The sum needs no second pass over the counters: an increment that finds the
// value k closes k pairs, so adding up what the increments return gives
// sum C(c_x, 2).
//
// Four launches:
//   k_p1_reset     counters and per-root sums to zero (a kernel: capturable)
//   k_p1_len       per edge (v0, v), v < v0: |{x in N(v): x < v0}|, and per
//                  root the sum W (its wedges) and the number of such v
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
// and the LDS atomics; every list is read once (R-MAT 18: 8.6e8 wedges, 3.5 GB
// of list elements in 3.1 ms, 1.1 TB/s).  One wave per root with a 32 KB table
// of its own held a CU to 4 waves, and roots above 16384 wedges counted in
// global memory, twice: R-MAT 18 149 -> 3.1 ms, R-MAT 20 785 -> 17.5 ms,
// 3.8M-vertex Chung-Lu 178 -> 10 ms.
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
// its barriers while the others work.  16 / 8 / 4 waves: R-MAT 18 3.9 / 3.1 /
// 4.8 ms, R-MAT 20 20.9 / 17.5 / 29.2, Chung-Lu 11.4 / 10.0 / 9.8 (narrower
// dense windows and the last split roots' tail cost the 4-wave form).
constexpr int P1_WAVES = 8;
constexpr int P1_SLICE = 2048;         // 32-bit words of LDS counters per wave task (8 KB)
constexpr int P1_TAB = P1_SLICE * P1_WAVES;  // ... per block task
constexpr int P1_PARTS = 16;           // x ranges of a split root
// roots with more wedges are split: 16 blocks then share what would be the
// last block's work (R-MAT 18: its widest root holds 5.6M of 863M wedges, more
// than a CU's average share)
constexpr uint64_t P1_SPLIT = 1ull << 19;
constexpr uint32_t P1_EMPTY = 0xffffffffu;

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

__global__ void k_p1_reset(P1Args a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 8) a.ctr[i] = 0;
  for (int64_t k = i; k < a.roots; k += (int64_t)gridDim.x * blockDim.x) a.W[k] = 0;
}

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
    if (v < v0) {
      const int64_t b = Q.rp[v];
      len = lb(Q.ci + b, (int)(Q.rp[v + 1] - b), v0);  // x < v0
      if (e + 1 == Q.rp[v0 + 1] || Q.ci[e + 1] > v0) a.m0[Q.roff + v0 - Q.rb] = (int32_t)(e + 1 - Q.rp[v0]);
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

__global__ void __launch_bounds__(256) k_p1_classify(P1Args a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int ln = lane();
  int cls = -1;
  int2 item = make_int2(0, 0);
  if (t < a.roots) {
    const int64_t i = a.roots - 1 - t;  // a relabelled graph ranks its widest roots last: list them first
    const uint64_t w = a.W[i];
    if (w >= 2) {  // else no two wedges share an endpoint
      item.y = a.q ? find_prefix(a.rcs, a.nq, i) : 0;
      const int64_t rb = a.q ? a.q[item.y].rb : a.one.rb, roff = a.q ? a.q[item.y].roff : a.one.roff;
      item.x = (int32_t)(rb + i - roff);
      const int cap = table_cap(P1_SLICE, packed_bits(item.x, a.m0[i]));
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
// one flattened stream, four loads in flight per lane; f(x) for every element.
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
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int fe = f0 + 64 * u;
      if (fe < T) {
        i = seg_advance(off, 64, i, fe);
        x[u] = ci[lbase[i] + fe];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (f0 + 64 * u < T) f(x[u]);
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

__global__ void __launch_bounds__(64 * P1_WAVES) p1_kernel(P1Args a) {
  __shared__ __attribute__((aligned(16))) uint32_t s_tab[P1_TAB];
  __shared__ int32_t s_off[P1_WAVES][65];
  __shared__ int64_t s_lb[P1_WAVES][64];
  __shared__ int64_t s_task;
  __shared__ unsigned long long s_tot[3];
  __shared__ int s_next;
  constexpr int NT = 64 * P1_WAVES;
  const int tid = threadIdx.x;
  const int wv = tid >> 6;
  const int ln = lane();
  int32_t* off = s_off[wv];
  int64_t* lbs = s_lb[wv];
  uint64_t acc = 0;
  int slot = 0;  // the query that acc belongs to
  auto flush = [&](int next) {
    if (next == slot) return;
    const uint64_t s = wave_sum_u64(acc);
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
    const int32_t* ci = Q.ci;
    const int32_t v0 = it.x;
    const int64_t b0 = Q.rp[v0];
    const int32_t* N0 = ci + b0;
    // neighbours below the window's end, per list; a root that is one task
    // moves them down as its windows descend
    int32_t* lens = a.len + Q.eoff + (b0 - Q.e0);
    const int m0 = a.m0[Q.roff + v0 - Q.rb];
    const uint64_t W = a.W[Q.roff + v0 - Q.rb];
    int64_t xlo = Q.xmin, xhi = v0;  // ids below xmin have one neighbour: they close no pair
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
            lb_many<3>(ci + Q.rp[N0[j]], n, y, pos);
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
      for (;;) {
        const int jb = wave_take(&s_next, cs);
        if (jb >= m0) break;
        const int j = jb + ln;
        int len = 0;
        int64_t base = 0;
        if (ln < cs && j < m0) {
          int n = lens[j];
          if (n) {
            base = Q.rp[N0[j]];
            if (part && hi < v0) n = lb(ci + base, n, (int32_t)hi);
            const int s = lo32 > 0 ? lb(ci + base, n, lo32) : 0;
            if (!part) lens[j] = s;
            len = n - s;
            base += s;
          }
        }
        if (!part) {
          const int w = (int)wave_sum_u64((uint64_t)len);
          if (ln == 0 && w) atomicAdd(&s_tot[0], (unsigned long long)w);
        }
        if (dense) {
          if (wide) {
            stream64(ci, base, len, off, lbs, [&](int32_t x) { acc += atomicAdd(&s_tab[x - lo32], 1u); });
          } else {
            stream64(ci, base, len, off, lbs, [&](int32_t x) {
              const uint32_t i = (uint32_t)(x - lo32), sh = (i & 1u) * 16u;
              acc += (atomicAdd(&s_tab[i >> 1], 1u << sh) >> sh) & 0xffffu;
            });
          }
        } else {
          stream64(ci, base, len, off, lbs, [&](int32_t x) { acc += table_count(s_tab, lt, cb, (uint32_t)(x - lo32)); });
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
  constexpr int CHUNK = 4;
  for (;;) {
    const int64_t tb = (int64_t)wave_take(a.ctr + C_POPW, (unsigned long long)CHUNK);
    if (tb >= nwave) break;
    for (int64_t t = tb; t < min(nwave, tb + CHUNK); ++t) {
      const int2 it = a.list[t];
      const P1Q Q = a.q ? a.q[it.y] : a.one;
      flush(Q.slot);
      const int32_t v0 = it.x;
      const int64_t b0 = Q.rp[v0];
      const int32_t* lens = a.len + Q.eoff + (b0 - Q.e0);
      const int m0 = a.m0[Q.roff + v0 - Q.rb];
      const int W = (int)a.W[Q.roff + v0 - Q.rb];
      const int cb = packed_bits(v0, m0);
      int lt = 6;
      while ((1 << lt) < 2 * W) ++lt;
      __syncwarp();
      table_clear(reinterpret_cast<uint4*>(tab), lt, cb, ln, 64);
      for (int jb = 0; jb < m0; jb += 64) {
        const int j = jb + ln;
        const int len = j < m0 ? lens[j] : 0;
        const int64_t base = len ? Q.rp[Q.ci[b0 + j]] : 0;
        stream64(Q.ci, base, len, off, lbs, [&](int32_t x) { acc += table_count(tab, lt, cb, (uint32_t)x); });
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

hipError_t launch_p1(const P1Args& a, int num_cu, hipStream_t st) {
  if (a.tiles <= 0 || a.roots <= 0) return hipSuccess;
  const unsigned rblocks = (unsigned)((a.roots + 255) / 256);
  hipLaunchKernelGGL(k_p1_reset, dim3(rblocks < 1024u ? rblocks : 1024u), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_p1_len, dim3((unsigned)a.tiles), dim3(256), 0, st, a);
  hipLaunchKernelGGL(k_p1_classify, dim3(rblocks), dim3(256), 0, st, a);
  const int64_t want = (a.roots + P1_WAVES - 1) / P1_WAVES, most = (int64_t)num_cu * (16 / P1_WAVES);
  hipLaunchKernelGGL(p1_kernel, dim3((unsigned)(want < most ? want : most)), dim3(64 * P1_WAVES), 0, st, a);
  return hipGetLastError();
}

}  // namespace jk
