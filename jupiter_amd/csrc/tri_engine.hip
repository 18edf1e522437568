// tri_engine.hip — per-edge triangle counts, the patterns that are sums over
// triangles (P5, P7, P9, P11 and P12, and parts of P4 and P10), and the graph
// of induced neighbourhoods that P6, P8 and P10 count wedges on.
//
// With t(u, v) = |N(u) ∩ N(v)| and q(T) = |N(a) ∩ N(x) ∩ N(y)| of a triangle
// T = {a, x, y}, the per-edge values of sym_kernels.hip's header, summed over
// the edges of a root range, are sums over triangles; a term belongs to the
// vertex its edge is credited to (the larger end for P5, the smaller for P9,
// P11 and P12, either for P7):
//   P5   sum over edges e of T of q (t(e) - 2) / 2     e's larger end in the range
//   P7   sum over vertices v of T of (t(v, w) - 1)(t(v, w') - 1) - q
//   P9   C(q, 2)                                       smallest id in the range
//   P11  abc - q (a + b + c) + 2q, a, b, c = t - 1     smallest id in the range
//   P12  sum over edges e of T of (t(e) - 3) C(q, 2)   e's smaller end in the range
// (src/message_passing_gpu_kernels.cuh:454-1109).  Every triangle is found
// once, at its source a in the degree order (its vertex of least degree):
// with M = N(a) and L the out-neighbours of a, row x (x in L) is the bitmap of
// N(x) ∩ M over the positions of M.  Then t(a, x) is the row's population, x
// and y in L are adjacent iff x's row has y's bit, and q is the population of
// two rows' intersection.
//
// A row word is one ballot: each lane tests one member of M against N(x).
// The test is one load for a hub x, whose neighbours are kept as a bitmap over
// all vertices (hub_bitmaps: the highest-degree vertices within
// tri_hub_bytes), and a binary search in the short list of any other x.  So a
// directed edge costs d(a) / 64 such steps, a being its end of less degree.
//
// What bounds it: the M and bitmap loads, past L2 with hubs enough (R-MAT 18
// P5: the small block tier reads 16.6 GB in 2.7 ms, 6.2 TB/s, the large one 15.9
// GB in 3.65 ms, which also waits for its pairs' LDS rows; the array's block
// launch 25.9 GB in 3.4 ms), several in flight per wave.  Per edge, with q(v2)
// counted by streaming N(v2) or by binary searches, the same counts cost R-MAT
// 18: P5 296 -> 7.9 ms, P7 349 -> 7.8, P9 121 -> 6.6, P11 163 -> 7.8, P12 350 ->
// 7.8; R-MAT 16 P5 28 -> 1.6; the triangle array (one intersection per edge by
// binary searches before) R-MAT 18 20.2 -> 4.6 ms, 3.8M-vertex Chung-Lu 16 -> 8.8.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "clique_dev.hpp"
#include "kernels.hpp"
#include "sym_dev.hpp"

namespace jk {

using symd::C2;
using symd::lane;
using symd::lb;

namespace {

// t_a counts of roots up to this degree are made by one wave
constexpr int TRI_WAVE_DEG = 64;

struct Adj {
  const int64_t* rp;
  const int32_t* ci;
  const int32_t* ord;
  const uint32_t* hub;  // bitmap h of the vertex with order nv - 1 - h
  int64_t hwords;       // words per bitmap
  int32_t nv, nhub;
  __device__ explicit Adj(const TriArgs& a)
      : rp(a.rp), ci(a.ci), ord(a.ord), hub(a.hub), hwords(a.hwords), nv(a.nv), nhub(a.nhub) {}
  // x's bitmap, or null when x is no hub
  __device__ const uint32_t* bitmap(int32_t x) const {
    const int32_t h = nv - 1 - ord[x];
    return h < nhub ? hub + h * hwords : nullptr;
  }
};

__device__ __forceinline__ bool bit(const uint32_t* w, int32_t y) { return (w[y >> 5] >> (y & 31)) & 1u; }

__device__ __forceinline__ bool in_list(const int32_t* l, int n, int32_t y) {
  const int p = lb(l, n, y);
  return p < n && l[p] == y;
}

// Hub bitmaps: a wave sets the bits of 65,536 ids of one hub in LDS and writes
// them once (R-MAT 18, 4,096 hubs: 2.25 ms by atomics on memory zeroed before,
// 0.06 so; the query 10.4 -> 7.8).
constexpr int HUB_SEG = 2048;  // words
__global__ void __launch_bounds__(256) k_hub_fill(TriArgs a, const int32_t* inv, uint32_t* hub) {
  __shared__ __attribute__((aligned(16))) uint32_t s_seg[4][HUB_SEG];
  uint32_t* const seg = s_seg[threadIdx.x >> 6];
  uint4* const seg4 = reinterpret_cast<uint4*>(seg);
  const int ln = lane();
  const int64_t nseg = (a.hwords + HUB_SEG - 1) / HUB_SEG;
  for (int64_t u = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); u < nseg * a.nhub; u += (int64_t)gridDim.x * 4) {
    const int64_t h = u / nseg, w0 = (u - h * nseg) * HUB_SEG;
    const int n4 = (int)(min((int64_t)HUB_SEG, a.hwords - w0) / 4);  // hwords is a multiple of 4
    const int32_t v = inv[h];
    const int32_t* l = a.ci + a.rp[v];
    const int d = (int)(a.rp[v + 1] - a.rp[v]);
    const int64_t id0 = w0 * 32, id1 = id0 + (int64_t)HUB_SEG * 32;
    const int lo = id0 > 0 ? lb(l, d, (int32_t)id0) : 0, hi = id1 < a.nv ? lb(l, d, (int32_t)id1) : d;
    for (int t = ln; t < n4; t += 64) seg4[t] = make_uint4(0u, 0u, 0u, 0u);
    __syncwarp();
    for (int k = lo + ln; k < hi; k += 256) {
      int32_t x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = k + 64 * i < hi ? l[k + 64 * i] - (int32_t)id0 : -1;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (x[i] >= 0) atomicOr(&seg[x[i] >> 5], 1u << (x[i] & 31));
    }
    __syncwarp();
    uint4* const dst = reinterpret_cast<uint4*>(hub + h * a.hwords + w0);
    for (int t = ln; t < n4; t += 64) dst[t] = seg4[t];
    __syncwarp();
  }
}

__global__ void k_tri_reset(unsigned long long* ctr) {
  if (threadIdx.x < 8) ctr[threadIdx.x] = 0;
}

// smallest power of two >= d, at least 4 (d <= 64)
__device__ __forceinline__ int group_lanes(int d) { return d <= 4 ? 4 : 1 << (32 - __builtin_clz((unsigned)(d - 1))); }

// Lane j's member x_j of L (dp <= 64 of them): its order, and where its
// neighbours are.
struct Member {
  int32_t x, ord, n;  // n: degree of an x that is no hub, else -1
  int64_t at;         // word of its bitmap in hub, or its list's start in ci
};
__device__ __forceinline__ Member member(const Adj& A, const int32_t* L, int dp) {
  Member w{0, 0, 0, 0};
  if (lane() < dp) {
    w.x = L[lane()];
    w.ord = A.ord[w.x];
    const int32_t h = A.nv - 1 - w.ord;
    if (h < A.nhub) {
      w.n = -1;
      w.at = h * A.hwords;
    } else {
      w.at = A.rp[w.x];
      w.n = (int)(A.rp[w.x + 1] - w.at);
    }
  }
  return w;
}

// The rows of a root with d <= 64 neighbours M: lane j returns x_j's row, one
// word.  Groups of g lanes test all of M against one x each, 64 / g of them at
// a time, four such steps' bitmap loads in flight.
__device__ __forceinline__ uint64_t wave_rows(const Adj& A, const int32_t* M, int d, const Member& mb, int dp) {
  const int ln = lane();
  const int g = uni(group_lanes(d)), per = 64 / g;
  const int p = ln & (g - 1), grp = ln / g;
  const int32_t m = p < d ? M[p] : 0;
  const uint64_t gmask = g == 64 ? ~0ull : (1ull << g) - 1;
  uint64_t row = 0;
  for (int xb = 0; xb < dp; xb += 4 * per) {
    uint32_t wd[4];
    int n[4];
    int64_t at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int xi = xb + u * per + grp;
      n[u] = __shfl(mb.n, xi & 63);
      at[u] = __shfl(mb.at, xi & 63);
      if (xi >= dp || p >= d) n[u] = 0;
      wd[u] = n[u] < 0 ? A.hub[at[u] + (m >> 5)] : 0u;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      bool f = (wd[u] >> (m & 31)) & 1u;
      if (n[u] > 0) f = in_list(A.ci + at[u], n[u], m);
      const uint64_t mk = __ballot(f);
      const int k = ln - (xb + u * per);  // lane j takes the word of x_j
      if (k >= 0 && k < per) row = (mk >> (k * g)) & gmask;
    }
  }
  return row;
}

// ---------------------------------------------------------------------------
// Triangles per DAG edge.  Roots of up to 64 neighbours here, one wave each;
// wider ones go to the list of k_dtri_block.
__global__ void __launch_bounds__(256) k_dtri_wave(TriArgs a, int32_t* dtri) {
  const Adj A(a);
  const int ln = lane();
  const int64_t nch = ((int64_t)a.nv + a.vchunk - 1) / a.vchunk;
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t c = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); c < nch; c += nw) {
    const int64_t v = c * a.vchunk + ln;
    int64_t b = 0, db = 0;
    int d = 0, dp = 0;
    if (ln < a.vchunk && v < a.nv) {
      b = a.rp[v];
      d = (int)(a.rp[v + 1] - b);
      db = a.drp[v];
      dp = (int)(a.drp[v + 1] - db);
    }
    const uint64_t wide = __ballot(dp > 0 && d > TRI_WAVE_DEG);
    if (wide) {
      const unsigned long long base = wave_take(a.ctr, (unsigned long long)__popcll(wide));
      if ((wide >> ln) & 1ull) a.list[base + __popcll(wide & ((1ull << ln) - 1))] = (int32_t)v;
    }
    uint64_t todo = __ballot(dp > 0 && d <= TRI_WAVE_DEG);
    while (todo) {
      const int k = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int64_t kb = __shfl(b, k), kdb = __shfl(db, k);
      const int kd = uni(__shfl(d, k)), kdp = uni(__shfl(dp, k));
      const uint64_t row = wave_rows(A, a.ci + kb, kd, member(A, a.dci + kdb, kdp), kdp);
      if (ln < kdp) dtri[kdb + ln] = __popcll(row);
    }
  }
}

// sum over M of [m in N(x)] for one (uniform) x: a wave's share of the lanes
__device__ __forceinline__ int edge_hits(const Adj& A, const int32_t* M, int d, int32_t x) {
  const int ln = lane();
  int c = 0;
  const uint32_t* bm = A.bitmap(x);
  if (bm) {
    int p = ln;
    for (; p + 192 < d; p += 256) {  // four members in flight
      const int32_t m0 = M[p], m1 = M[p + 64], m2 = M[p + 128], m3 = M[p + 192];
      const uint32_t w0 = bm[m0 >> 5], w1 = bm[m1 >> 5], w2 = bm[m2 >> 5], w3 = bm[m3 >> 5];
      c += ((w0 >> (m0 & 31)) & 1u) + ((w1 >> (m1 & 31)) & 1u) + ((w2 >> (m2 & 31)) & 1u) + ((w3 >> (m3 & 31)) & 1u);
    }
    for (; p < d; p += 64) c += bit(bm, M[p]);
  } else {
    const int64_t b = A.rp[x];
    const int n = (int)(A.rp[x + 1] - b);
    for (int p = ln; p < d; p += 64) c += in_list(A.ci + b, n, M[p]);
  }
  return c;
}

__global__ void __launch_bounds__(512) k_dtri_block(TriArgs a, int32_t* dtri) {
  __shared__ int64_t s_task;
  __shared__ int s_next;
  const Adj A(a);
  const int ln = lane();
  const int64_t n = (int64_t)a.ctr[0];
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) {
      s_task = (int64_t)atomicAdd(a.ctr + 1, 1ull);
      s_next = 0;
    }
    __syncthreads();
    const int64_t t = s_task;
    if (t >= n) break;
    const int32_t v = a.list[t];
    const int64_t b = a.rp[v], db = a.drp[v];
    const int d = (int)(a.rp[v + 1] - b), dp = (int)(a.drp[v + 1] - db);
    for (;;) {
      const int j = uni(wave_take(&s_next, 1));
      if (j >= dp) break;
      const int c = symd::wsum(edge_hits(A, a.ci + b, d, uni(a.dci[db + j])));
      if (ln == 0) dtri[db + j] = c;
    }
  }
}

// t of every symmetric edge from its DAG edge
__global__ void __launch_bounds__(256) k_tri_scatter(TriArgs a, const int32_t* dtri, const int32_t* src, int64_t ne,
                                                     int32_t* tri) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t u = src[e], v = a.ci[e];
    const bool up = a.ord[u] < a.ord[v];
    const int32_t s = up ? u : v, y = up ? v : u;
    const int64_t b = a.drp[s];
    tri[e] = dtri[b + lb(a.dci + b, (int)(a.drp[s + 1] - b), y)];
  }
}

// ---------------------------------------------------------------------------
// Sums over triangles.

template <int P>
constexpr bool needs_t() { return P != 9; }
template <int P>
constexpr bool is_twice() { return P == 5 || P == 10; }  // sums twice the value

// one triangle's terms whose owner lies in [rb, re); ids a, x, y; txy etc.
// the triangle counts of its edges (unused for P9)
template <int P>
__device__ __forceinline__ int64_t tri_term(const TriArgs& g, int32_t a, int32_t x, int32_t y, int64_t tax, int64_t tay,
                                            int64_t txy, int64_t q) {
  auto in = [&](int32_t v) { return (int64_t)(v >= g.rb && v < g.re); };
  if constexpr (P == 4) {
    // the part of P4 over triangles: less, for each edge as the (v0, v1) of
    // the nest, the (t - 1) of the triangle's two other edges
    return -(in(max(a, x)) * (tay + txy - 2) + in(max(a, y)) * (tax + txy - 2) + in(max(x, y)) * (tax + tay - 2));
  } else if constexpr (P == 10) {
    // sum over the edges (v0, x) of k (3 - 2 t), k the 4-cliques on the edge:
    // half of the q of the edge's triangles
    return q * ((in(a) + in(x)) * (3 - 2 * tax) + (in(a) + in(y)) * (3 - 2 * tay) + (in(x) + in(y)) * (3 - 2 * txy));
  } else if constexpr (P == 5) {  // twice the value: halved at the end
    return q * (in(max(a, x)) * (tax - 2) + in(max(a, y)) * (tay - 2) + in(max(x, y)) * (txy - 2));
  } else if constexpr (P == 7) {
    return in(a) * ((tax - 1) * (tay - 1) - q) + in(x) * ((tax - 1) * (txy - 1) - q) +
           in(y) * ((tay - 1) * (txy - 1) - q);
  } else if constexpr (P == 9) {
    return in(min(a, min(x, y))) * C2(q);
  } else if constexpr (P == 11) {
    const int64_t s = tax + tay + txy - 3;
    return in(min(a, min(x, y))) * ((tax - 1) * (tay - 1) * (txy - 1) - q * s + 2 * q);
  } else {  // P12
    return C2(q) * (in(min(a, x)) * (tax - 3) + in(min(a, y)) * (tay - 3) + in(min(x, y)) * (txy - 3));
  }
}

// t of the edge between two members x and y of L with orders ox, oy
__device__ __forceinline__ int32_t dag_t(const TriArgs& a, int32_t x, int32_t y, int32_t ox, int32_t oy) {
  const int32_t s = ox < oy ? x : y, z = ox < oy ? y : x;
  const int64_t b = a.drp[s];
  return a.dtri[b + lb(a.dci + b, (int)(a.drp[s + 1] - b), z)];
}

// Adds a wave's sum to the result.  P5's and P10's sums count every value
// twice: the half is added, and an odd sum pairs up with another through a
// flag (the total is even).
__device__ __forceinline__ void add_half(uint64_t acc, unsigned long long* flag, uint64_t* out) {
  acc = wave_sum_u64(acc);
  if (lane() != 0 || !acc) return;
  const uint64_t half = (uint64_t)((int64_t)acc >> 1);
  const uint64_t odd = (acc & 1) ? atomicXor(flag, 1ull) : 0;
  atomicAdd((unsigned long long*)out, (unsigned long long)(half + odd));
}
template <int P>
__device__ __forceinline__ void tri_add(const TriArgs& a, uint64_t acc) {
  if constexpr (is_twice<P>()) {
    add_half(acc, a.ctr + 6, a.out);
  } else {
    acc = wave_sum_u64(acc);
    if (lane() == 0 && acc) atomicAdd((unsigned long long*)a.out, (unsigned long long)acc);
  }
}

// Block tiers by the bytes of a root's rows: LDS of TRI_LDS_S, of TRI_LDS_L,
// or a slice of global scratch.
constexpr int TRI_LDS_S = 16 << 10;
constexpr int TRI_LDS_L = 128 << 10;

__device__ __forceinline__ int row_words(int d) { return ((d + 63) >> 6) | 1; }  // odd: rows on different banks

// Roots of up to 64 neighbours, one wave each; wider ones onto the lists of
// the block tiers.
template <int P>
__global__ void __launch_bounds__(256) k_tri_wave(TriArgs a) {
  __shared__ uint32_t s_queue[4][128];
  uint32_t* const queue = s_queue[threadIdx.x >> 6];
  const Adj A(a);
  const int ln = lane();
  const int64_t nch = ((int64_t)a.nv + a.vchunk - 1) / a.vchunk;
  const int64_t nw = (int64_t)gridDim.x * 4;
  uint64_t acc = 0;
  for (int64_t c = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); c < nch; c += nw) {
    const int64_t v = c * a.vchunk + ln;
    int64_t b = 0, db = 0;
    int d = 0, dp = 0;
    if (ln < a.vchunk && v < a.nv) {
      b = a.rp[v];
      d = (int)(a.rp[v + 1] - b);
      db = a.drp[v];
      dp = (int)(a.drp[v + 1] - db);
    }
    const int64_t bytes = (int64_t)dp * row_words(d) * 8;
    const int tier = dp < 2 || d <= TRI_WAVE_DEG ? -1 : bytes <= TRI_LDS_S ? 0 : bytes <= TRI_LDS_L ? 1 : 2;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint64_t m = __ballot(tier == t);
      if (!m) continue;
      const unsigned long long base = wave_take(a.ctr + t, (unsigned long long)__popcll(m));
      if (tier == t) a.list[(int64_t)t * a.nv + base + __popcll(m & ((1ull << ln) - 1))] = (int32_t)v;
    }
    uint64_t todo = __ballot(dp >= 2 && d <= TRI_WAVE_DEG);
    while (todo) {
      const int k = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int64_t kb = __shfl(b, k), kdb = __shfl(db, k);
      const int kd = uni(__shfl(d, k)), kdp = uni(__shfl(dp, k));
      const int32_t root = (int32_t)(c * a.vchunk + k);
      const int32_t* M = a.ci + kb;
      const Member mb = member(A, a.dci + kdb, kdp);
      const uint64_t row = wave_rows(A, M, kd, mb, kdp);
      const int pos = ln < kdp ? lb(M, kd, mb.x) : 0;
      // adjacent pairs (i, j) into the wave's queue; 64 of them at a time
      // are evaluated
      auto drain = [&](int cnt) {
        const uint32_t e = ln < cnt ? queue[ln] : 0u;
        const int i = (int)(e >> 16), j = (int)(e & 0xffffu);
        const uint64_t ri = __shfl((unsigned long long)row, i), rj = __shfl((unsigned long long)row, j);
        const int32_t xi = __shfl(mb.x, i), xj = __shfl(mb.x, j);
        const int32_t oi = __shfl(mb.ord, i), oj = __shfl(mb.ord, j);
        if (ln < cnt) {
          const int32_t txy = needs_t<P>() ? dag_t(a, xi, xj, oi, oj) : 0;
          acc += (uint64_t)tri_term<P>(a, root, xi, xj, __popcll(ri), __popcll(rj), txy, __popcll(ri & rj));
        }
      };
      int qn = 0;
      for (int i = 0; i + 1 < kdp; ++i) {
        const uint64_t ri = __shfl((unsigned long long)row, i);
        const bool hit = ln > i && ln < kdp && ((ri >> pos) & 1ull);
        const uint64_t mk = __ballot(hit);
        if (!mk) continue;
        if (hit) queue[qn + __popcll(mk & ((1ull << ln) - 1))] = ((uint32_t)i << 16) | (uint32_t)ln;
        qn += __popcll(mk);
        __syncwarp();
        if (qn >= 64) {
          drain(64);
          qn -= 64;
          __syncwarp();
          if (ln < qn) queue[ln] = queue[64 + ln];
          __syncwarp();
        }
      }
      if (qn) drain(qn);
      __syncwarp();
    }
  }
  tri_add<P>(a, acc);
}

// One block per root of list TIER.  LDS (TIER < 2): the rows; always: L's
// positions in M, and a queue of adjacent pairs per wave, so that the pairs
// found by 64 lanes are evaluated by full waves.
template <int P, int TIER>
__global__ void __launch_bounds__(TIER == 0 ? 256 : 1024) k_tri_block(TriArgs a) {
  constexpr int WAVES = TIER == 0 ? 4 : 16;
  constexpr int NT = 64 * WAVES;
  constexpr int LDS = TIER == 0 ? TRI_LDS_S : TIER == 1 ? TRI_LDS_L : 64;
  __shared__ __attribute__((aligned(16))) unsigned char s_rows[LDS];
  __shared__ uint32_t s_queue[WAVES][128];
  __shared__ int64_t s_task;
  __shared__ int s_next;
  const Adj A(a);
  const int tid = threadIdx.x, wv = tid >> 6, ln = lane();
  // per member of L: position in M, t(a, x), order (scratch of the block)
  int32_t* const Lp = a.lscr + (int64_t)blockIdx.x * 3 * a.lstride;
  int32_t* const Lt = Lp + a.lstride;
  int32_t* const Lo = Lt + a.lstride;
  uint64_t* const B = TIER < 2 ? reinterpret_cast<uint64_t*>(s_rows) : a.rows + (int64_t)blockIdx.x * a.rstride;
  uint32_t* queue = s_queue[wv];
  const int64_t n = (int64_t)a.ctr[TIER];
  uint64_t acc = 0;
  for (;;) {
    __syncthreads();
    if (tid == 0) {
      s_task = (int64_t)atomicAdd(a.ctr + 3 + TIER, 1ull);
      s_next = 0;
    }
    __syncthreads();
    const int64_t t = s_task;
    if (t >= n) break;
    const int32_t root = a.list[(int64_t)TIER * a.nv + t];
    const int64_t b = a.rp[root], db = a.drp[root];
    const int d = (int)(a.rp[root + 1] - b), dp = (int)(a.drp[root + 1] - db);
    const int32_t* M = a.ci + b;
    const int32_t* L = a.dci + db;
    const int W = (d + 63) >> 6, S = row_words(d);
    for (int j = tid; j < dp; j += NT) {
      const int32_t x = L[j];
      Lp[j] = lb(M, d, x);
      if constexpr (needs_t<P>()) {
        Lt[j] = a.dtri[db + j];
        Lo[j] = a.ord[x];
      }
    }
    // rows: the (64-member chunk of M, x) pairs in order of the chunk, dealt
    // to the waves in runs, four x at a time (their loads overlap)
    const int64_t items = (int64_t)W * ((dp + 3) / 4);
    const int64_t per = (items + WAVES - 1) / WAVES;
    int64_t it = wv * per;
    const int64_t ie = min(items, it + per);
    const int quads = (dp + 3) / 4;
    int w = (int)(it / quads), jq = (int)(it % quads);
    int32_t m = -1;
    int wm = -1;
    for (; it < ie; ++it) {
      if (w != wm) {
        const int p = w * 64 + ln;
        m = p < d ? M[p] : -1;
        wm = w;
      }
      uint32_t wd[4];
      bool f[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = jq * 4 + u;
        const int32_t x = uni(L[min(j, dp - 1)]);
        const uint32_t* bm = A.bitmap(x);
        f[u] = false;
        wd[u] = 0;
        if (m >= 0) {
          if (bm) {
            wd[u] = bm[m >> 5];
          } else {
            const int64_t xb = A.rp[x];
            f[u] = in_list(A.ci + xb, (int)(A.rp[x + 1] - xb), m);
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = jq * 4 + u;
        const uint64_t word = __ballot(f[u] || ((wd[u] >> (m & 31)) & 1u));
        if (j < dp && ln == u) B[(int64_t)j * S + w] = word;
      }
      if (++jq == quads) {
        jq = 0;
        ++w;
      }
    }
    if constexpr (TIER == 2) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __syncthreads();
    if constexpr (TIER == 2) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    // pairs: q of up to 64 queued ones
    auto drain = [&](int cnt) {
      uint32_t e = 0;
      int q = 0;
      if (W < 48) {  // a lane per pair
        if (ln < cnt) {
          e = queue[ln];
          const uint64_t* bi = B + (int64_t)(e >> 16) * S;
          const uint64_t* bj = B + (int64_t)(e & 0xffffu) * S;
          for (int k = 0; k < W; ++k) q += __popcll(bi[k] & bj[k]);
        }
      } else {  // long rows: the wave per pair
        if (ln < cnt) e = queue[ln];
        for (int k = 0; k < cnt; ++k) {
          const uint32_t ek = __shfl(e, k);
          const uint64_t* bi = B + (int64_t)(ek >> 16) * S;
          const uint64_t* bj = B + (int64_t)(ek & 0xffffu) * S;
          int c = 0;
          for (int u = ln; u < W; u += 64) c += __popcll(bi[u] & bj[u]);
          c = symd::wsum(c);
          if (ln == k) q = c;
        }
      }
      if (ln < cnt) {
        const int i = (int)(e >> 16), j = (int)(e & 0xffffu);
        const int32_t x = L[i], y = L[j];
        int64_t ti = 0, tj = 0, txy = 0;
        if constexpr (needs_t<P>()) {
          ti = Lt[i];
          tj = Lt[j];
          txy = dag_t(a, x, y, Lo[i], Lo[j]);
        }
        acc += (uint64_t)tri_term<P>(a, root, x, y, ti, tj, txy, q);
      }
    };
    int qn = 0;
    for (;;) {
      const int i = uni(wave_take(&s_next, 1));
      if (i + 1 >= dp) break;
      const uint64_t* bi = B + (int64_t)i * S;
      for (int jb = i + 1; jb < dp; jb += 64) {
        const int j = jb + ln;
        bool hit = false;
        if (j < dp) {
          const int p = Lp[j];
          hit = (bi[p >> 6] >> (p & 63)) & 1ull;
        }
        const uint64_t mk = __ballot(hit);
        if (hit)
          queue[qn + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mk >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mk, 0u))] =
              ((uint32_t)i << 16) | (uint32_t)j;
        qn += __popcll(mk);
        __syncwarp();
        if (qn >= 64) {
          drain(64);
          qn -= 64;
          __syncwarp();
          if (ln < qn) queue[ln] = queue[64 + ln];
          __syncwarp();
        }
      }
    }
    drain(qn);
    __syncwarp();
  }
  tri_add<P>(a, acc);
}

// blocks of the kernels whose waves take a.vchunk vertices at a time
unsigned wave_grid(const TriArgs& a, int num_cu) {
  const int64_t blocks = ((int64_t)a.nv + 4 * a.vchunk - 1) / (4 * a.vchunk);
  return (unsigned)(blocks < num_cu * 8 ? blocks : num_cu * 8);
}

// ---------------------------------------------------------------------------
// The graph of induced neighbourhoods: a vertex per directed edge (v0, u) of
// the edges [e0, e0 + n), numbered from 0, joined to (v0, y) for every common
// neighbour y of v0 and u.  Row (v0, u) has t(v0, u) entries; the rows of one
// v0 are the graph that N(v0) induces.

// exclusive prefix of tri over the rows: tile sums, their prefix, the rows
constexpr int SCAN_TILE = 2048;

__device__ __forceinline__ int64_t block_excl(int64_t v, int64_t* part, int64_t& total) {
  const int ln = lane(), wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
  int64_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t y = (int64_t)__shfl_up((unsigned long long)x, o);
    if (ln >= o) x += y;
  }
  __syncthreads();
  if (ln == 63) part[wv] = x;
  __syncthreads();
  int64_t base = 0;
  total = 0;
  for (int k = 0; k < nw; ++k) {
    if (k < wv) base += part[k];
    total += part[k];
  }
  return base + x - v;
}

__global__ void __launch_bounds__(256) k_scan_tiles(const int32_t* tri, int64_t n, int64_t* tiles) {
  __shared__ int64_t part[4];
  const int64_t b = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x * 8;
  int64_t s = 0, total;
  for (int k = 0; k < 8; ++k) s += b + k < n ? tri[b + k] : 0;
  block_excl(s, part, total);
  if (threadIdx.x == 0) tiles[blockIdx.x] = total;
}

__global__ void __launch_bounds__(1024) k_scan_tops(int64_t* tiles, int64_t nt) {
  __shared__ int64_t part[16];
  int64_t run = 0;
  for (int64_t b = 0; b < nt; b += 1024) {
    const int64_t i = b + threadIdx.x;
    int64_t total;
    const int64_t x = block_excl(i < nt ? tiles[i] : 0, part, total);
    if (i < nt) tiles[i] = run + x;
    run += total;
  }
}

__global__ void __launch_bounds__(256) k_scan_rows(const int32_t* tri, int64_t n, const int64_t* tiles, int64_t* rp) {
  __shared__ int64_t part[4];
  const int64_t b = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x * 8;
  int64_t s = 0, total;
  int32_t t[8];
  for (int k = 0; k < 8; ++k) {
    t[k] = b + k < n ? tri[b + k] : 0;
    s += t[k];
  }
  int64_t run = tiles[blockIdx.x] + block_excl(s, part, total);
  for (int k = 0; k < 8; ++k) {
    if (b + k < n) rp[b + k] = run;
    run += t[k];
    if (b + k == n - 1) rp[n] = run;
  }
}

// A wave per row: the members of M = N(v0) that N(u) holds, in order.  Tests
// M's members against u when u is a hub or its list is not much shorter than
// M, else searches u's list in M.
__global__ void __launch_bounds__(256) k_ego_fill(TriArgs a, EgoArgs g) {
  const Adj A(a);
  const int ln = lane();
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t k = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); k < g.n; k += nw) {
    const int64_t e = g.e0 + k;
    if (g.tri[e] == 0) continue;
    const int32_t v0 = uni(g.src[e]), u = uni(a.ci[e]);
    const int64_t b = a.rp[v0], ub = a.rp[u];
    const int d = (int)(a.rp[v0 + 1] - b), du = (int)(a.rp[u + 1] - ub);
    const int32_t* M = a.ci + b;
    const int32_t* N = a.ci + ub;
    const uint32_t* bm = A.bitmap(u);
    const bool over_m = bm ? d <= 16 * du : d <= 2 * du;
    const int32_t base = (int32_t)(b - g.e0);
    int64_t at = g.rp[k];
    const int n = over_m ? d : du;
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int i = i0 + ln;
      bool f = false;
      int p = i;
      if (i < n) {
        if (over_m) {
          f = bm ? bit(bm, M[i]) : in_list(N, du, M[i]);
        } else {
          const int32_t y = N[i];
          p = lb(M, d, y);
          f = p < d && M[p] == y;
        }
      }
      const uint64_t mk = __ballot(f);
      if (f) {
        const int64_t o = at + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mk >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)mk, 0u));
        g.ci[o] = base + p;
        g.row[o] = (int32_t)k;
      }
      at += __popcll(mk);
    }
  }
}

// P10's part over the rows: for (v0, u), the pairs x, y of its entries with
// (t(v0, x) - 1)(t(v0, y) - 1).  A wave per row.
__global__ void __launch_bounds__(256) k_p10_rows(EgoArgs g, uint64_t* out) {
  const int ln = lane();
  const int64_t nw = (int64_t)gridDim.x * 4;
  uint64_t acc = 0;
  for (int64_t k = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); k < g.n; k += nw) {
    const int64_t b = g.rp[k], e = g.rp[k + 1];
    if (e - b < 2) continue;
    uint64_t s = 0, s2 = 0;
    for (int64_t i = b + ln; i < e; i += 64) {
      const uint64_t x = (uint64_t)(g.tri[g.e0 + g.ci[i]] - 1);
      s += x;
      s2 += x * x;
    }
    s = wave_sum_u64(s);
    s2 = wave_sum_u64(s2);
    acc += (uint64_t)(((unsigned __int128)s * s - s2) >> 1);
  }
  if (ln == 0 && acc) atomicAdd((unsigned long long*)out, (unsigned long long)acc);
}

// The closed parts of P4 and P6 per edge (v0, v1), v1 < v0, with s common
// neighbours: P4 (mode 0) -s (d0 + d1 - 1), and for a whole graph (mode 1) the
// triangle part too, which then sums to -2 s (s - 1); P6 (mode 2) -2 C(s, 2).
__global__ void __launch_bounds__(256) k_edge_base(const int64_t* rp, const int32_t* ci, const int32_t* src,
                                                   const int32_t* tri, int64_t e0, int64_t e1, int mode, uint64_t* out) {
  uint64_t acc = 0;
  for (int64_t e = e0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < e1; e += (int64_t)gridDim.x * blockDim.x) {
    const int32_t v0 = src[e], v1 = ci[e];
    const int64_t s = tri[e];
    if (v1 >= v0 || s == 0) continue;
    if (mode == 2) {
      acc -= (uint64_t)(s * (s - 1));
    } else {
      const int64_t d = (rp[v0 + 1] - rp[v0]) + (rp[v1 + 1] - rp[v1]);
      acc -= (uint64_t)(s * (d - 1)) + (mode == 1 ? (uint64_t)(2 * s * (s - 1)) : 0ull);
    }
  }
  acc = wave_sum_u64(acc);
  if (lane() == 0 && acc) atomicAdd((unsigned long long*)out, (unsigned long long)acc);
}

// P3 and tailed triangles over the edges [e0, e1) of a root range, from the
// triangle counts alone.  P3's value of (v0, v1) sums, over the triangles v0
// v1 v2 with v2 > v1, D0 - d0 + 4 - (d1 + d2) - (t01 + t02), which is symmetric in
// v1 and v2: per vertex o with T = half the sum of t over its edges, it is
//   T (D - d + 4) - sum over its edges (o, p) of t (t + d(p)),
// D the sum of its neighbours' degrees.  Tailed triangles: T (d - 2).  Edge by
// edge, twice the value: three coalesced streams and, where t > 0, the degree
// of p (R-MAT 18 P3: 14.7 ms over triangles, an intersection per edge of the
// range below that, 0.1 ms so).
template <bool P3>
__global__ void __launch_bounds__(256) k_edge_sum(const int64_t* rp, const int32_t* ci, const int32_t* src,
                                                  const int32_t* tri, const int64_t* nsum, int64_t e0, int64_t e1,
                                                  unsigned long long* flag, uint64_t* out) {
  uint64_t acc = 0;
  for (int64_t e = e0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < e1; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = tri[e];
    if (t == 0) continue;
    const int32_t o = src[e];
    const int64_t d = rp[o + 1] - rp[o];
    if constexpr (P3) {
      const int32_t p = ci[e];
      const int64_t dp = rp[p + 1] - rp[p];
      acc += (uint64_t)(t * (nsum[o] - d + 4) - 2 * t * (t + dp));
    } else {
      acc += (uint64_t)(t * (d - 2));
    }
  }
  add_half(acc, flag, out);
}

// sum of tri over each vertex's edges
__global__ void __launch_bounds__(256) k_root_tri(const int64_t* rp, const int32_t* tri, int32_t nv, int64_t* sum) {
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t v = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); v < nv; v += nw) {
    int64_t s = 0;
    for (int64_t e = rp[v] + lane(); e < rp[v + 1]; e += 64) s += tri[e];
    s = symd::wsum64(s);
    if (lane() == 0) sum[v] = s;
  }
}

// What the edges of EDGE_WORK_BLOCK vertices cost the per-edge launches where
// they have triangles (ns): x and y over the edges to larger ids, z over those
// to smaller ones; w what the vertices' rows and triangles cost the triangle
// sums.  A block each: the first vertices of an R-MAT graph are its hubs.
__global__ void __launch_bounds__(512) k_edge_work(TriArgs a, const int32_t* src, const int32_t* tri, float4* work) {
  __shared__ float4 s_part[8];
  const int64_t v = (int64_t)blockIdx.x * EDGE_WORK_BLOCK, ve = min((int64_t)a.nv, v + EDGE_WORK_BLOCK), end = a.rp[ve];
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (v + threadIdx.x < ve) {
    const int64_t u = v + threadIdx.x;
    s.w = 0.0035f * (float)(a.rp[u + 1] - a.rp[u]) * (float)(a.drp[u + 1] - a.drp[u]);
  }
  for (int64_t e0 = a.rp[v] + threadIdx.x; e0 < end; e0 += 2048) {
    int32_t te[4];
    bool up[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t e = min(e0 + 512 * k, end - 1);
      te[k] = e0 + 512 * k < end ? tri[e] : 0;
      up[k] = a.ci[e] > src[e];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float t = (float)te[k];
      if (t == 0.f) continue;
      const float b = 8.f + 0.6f * t + 0.00045f * t * t;
      if (up[k]) {
        s.x += 5.f + 0.001f * t * t;
        s.y += b;
      } else {
        s.z += b;
        s.w += 0.0087f * t;
      }
    }
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    s.x += __shfl_xor(s.x, o);
    s.y += __shfl_xor(s.y, o);
    s.z += __shfl_xor(s.z, o);
    s.w += __shfl_xor(s.w, o);
  }
  if (lane() == 0) s_part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 8; ++k) {
      s.x += s_part[k].x;
      s.y += s_part[k].y;
      s.z += s_part[k].z;
      s.w += s_part[k].w;
    }
    work[blockIdx.x] = s;
  }
}

// grid of a kernel with a wave per item, 4 waves per block
unsigned item_grid(int64_t items, int num_cu) {
  const int64_t blocks = (items + 3) / 4;
  return (unsigned)(blocks < (int64_t)num_cu * 8 ? (blocks > 0 ? blocks : 1) : (int64_t)num_cu * 8);
}

template <int P>
hipError_t launch_sum(const TriArgs& a, int num_cu, int gblocks, hipStream_t st) {
  hipLaunchKernelGGL(k_tri_reset, dim3(1), dim3(64), 0, st, a.ctr);
  hipLaunchKernelGGL(k_tri_wave<P>, dim3(wave_grid(a, num_cu)), dim3(256), 0, st, a);
  if (gblocks > 0) hipLaunchKernelGGL((k_tri_block<P, 2>), dim3(gblocks), dim3(1024), 0, st, a);
  if (a.wide) {
    hipLaunchKernelGGL((k_tri_block<P, 1>), dim3(num_cu), dim3(1024), 0, st, a);
    hipLaunchKernelGGL((k_tri_block<P, 0>), dim3(num_cu * TRI_SMALL_PER_CU), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

}  // namespace

int64_t tri_row_words(int64_t d, int64_t dp) { return dp * (((d + 63) >> 6) | 1); }
bool tri_rows_global(int64_t d, int64_t dp) { return dp >= 2 && d > TRI_WAVE_DEG && tri_row_words(d, dp) * 8 > TRI_LDS_L; }

hipError_t launch_hub_bitmaps(const TriArgs& a, int num_cu, hipStream_t st) {
  if (a.nhub <= 0) return hipSuccess;
  uint32_t* hub = const_cast<uint32_t*>(a.hub);
  // the hubs' vertices, in the task lists' memory, which is free until then
  hipError_t e = launch_hub_places(a.ord, a.nv, a.nhub, a.list, num_cu, st);
  if (e != hipSuccess) return e;
  const int64_t blocks = ((a.hwords + HUB_SEG - 1) / HUB_SEG * a.nhub + 3) / 4;
  hipLaunchKernelGGL(k_hub_fill, dim3((unsigned)(blocks < num_cu * 5 ? blocks : num_cu * 5)), dim3(256), 0, st, a,
                     a.list, hub);
  return hipGetLastError();
}

hipError_t launch_tri_build(const TriArgs& a, int32_t* dtri, const int32_t* src, int64_t ne, int32_t* tri, int num_cu,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_tri_reset, dim3(1), dim3(64), 0, st, a.ctr);
  hipLaunchKernelGGL(k_dtri_wave, dim3(wave_grid(a, num_cu)), dim3(256), 0, st, a, dtri);
  if (a.wide) hipLaunchKernelGGL(k_dtri_block, dim3(num_cu * 4), dim3(512), 0, st, a, dtri);
  const int64_t blocks = (ne + 255) / 256;
  if (ne > 0)
    hipLaunchKernelGGL(k_tri_scatter, dim3((unsigned)(blocks < num_cu * 16 ? blocks : num_cu * 16)), dim3(256), 0, st, a,
                       dtri, src, ne, tri);
  return hipGetLastError();
}

int64_t ego_tiles(int64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE; }

hipError_t launch_ego_build(const TriArgs& a, const EgoArgs& g, int num_cu, hipStream_t st) {
  if (g.n <= 0) return hipSuccess;
  const int64_t nt = ego_tiles(g.n);
  const int32_t* tri = g.tri + g.e0;
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)nt), dim3(256), 0, st, tri, g.n, g.tiles);
  hipLaunchKernelGGL(k_scan_tops, dim3(1), dim3(1024), 0, st, g.tiles, nt);
  hipLaunchKernelGGL(k_scan_rows, dim3((unsigned)nt), dim3(256), 0, st, tri, g.n, g.tiles, g.rp);
  hipLaunchKernelGGL(k_ego_fill, dim3(item_grid(g.n, num_cu)), dim3(256), 0, st, a, g);
  return hipGetLastError();
}

hipError_t launch_p10_rows(const EgoArgs& g, uint64_t* out, int num_cu, hipStream_t st) {
  hipLaunchKernelGGL(k_p10_rows, dim3(item_grid(g.n, num_cu)), dim3(256), 0, st, g, out);
  return hipGetLastError();
}

hipError_t launch_edge_base(const int64_t* rp, const int32_t* ci, const int32_t* src, const int32_t* tri, int64_t e0,
                            int64_t e1, int mode, uint64_t* out, int num_cu, hipStream_t st) {
  if (e1 <= e0) return hipSuccess;
  const int64_t blocks = (e1 - e0 + 255) / 256;
  hipLaunchKernelGGL(k_edge_base, dim3((unsigned)(blocks < num_cu * 8 ? blocks : num_cu * 8)), dim3(256), 0, st, rp, ci,
                     src, tri, e0, e1, mode, out);
  return hipGetLastError();
}

hipError_t launch_edge_sum(bool p3, const int64_t* rp, const int32_t* ci, const int32_t* src, const int32_t* tri,
                           const int64_t* nsum, int64_t e0, int64_t e1, unsigned long long* flag, uint64_t* out,
                           int num_cu, hipStream_t st) {
  if (e1 <= e0) return hipSuccess;
  const int64_t blocks = (e1 - e0 + 255) / 256;
  const dim3 grid((unsigned)(blocks < num_cu * 8 ? blocks : num_cu * 8));
  if (p3)
    hipLaunchKernelGGL(k_edge_sum<true>, grid, dim3(256), 0, st, rp, ci, src, tri, nsum, e0, e1, flag, out);
  else
    hipLaunchKernelGGL(k_edge_sum<false>, grid, dim3(256), 0, st, rp, ci, src, tri, nsum, e0, e1, flag, out);
  return hipGetLastError();
}

hipError_t launch_root_tri(const int64_t* rp, const int32_t* tri, int32_t nv, int64_t* sum, int num_cu, hipStream_t st) {
  hipLaunchKernelGGL(k_root_tri, dim3(item_grid(nv, num_cu)), dim3(256), 0, st, rp, tri, nv, sum);
  return hipGetLastError();
}

hipError_t launch_edge_work(const TriArgs& a, const int32_t* src, const int32_t* tri, float4* work, hipStream_t st) {
  if (a.nv > 0)
    hipLaunchKernelGGL(k_edge_work, dim3((unsigned)edge_work_blocks(a.nv)), dim3(512), 0, st, a, src, tri, work);
  return hipGetLastError();
}

hipError_t launch_tri_sum(int p, const TriArgs& a, int num_cu, int gblocks, hipStream_t st) {
  switch (p) {
    case 4: return launch_sum<4>(a, num_cu, gblocks, st);
    case 10: return launch_sum<10>(a, num_cu, gblocks, st);
    case 5: return launch_sum<5>(a, num_cu, gblocks, st);
    case 7: return launch_sum<7>(a, num_cu, gblocks, st);
    case 9: return launch_sum<9>(a, num_cu, gblocks, st);
    case 11: return launch_sum<11>(a, num_cu, gblocks, st);
    case 12: return launch_sum<12>(a, num_cu, gblocks, st);
  }
  return hipErrorInvalidValue;
}

}  // namespace jk
