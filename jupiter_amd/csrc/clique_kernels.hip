// clique_kernels.hip — gfx950 kernels for triangle and k-clique counting
// (TC and P13..P16) on the degree-oriented DAG.
//
// Replaces the reference's P13_kernel..P16_kernel
// (src/message_passing_gpu_kernels.cuh:1208-1537) and the level-by-level
// pattern_task_generate / pattern_extend_pull_workloads path
// (src/gpu_kernels_codegen.cuh:6-95,261-410).  The count for root v0 equals
// the reference's sum over the DAG edges (v0, v1): the number of k-cliques
// whose DAG source is v0.
//
// Design (one root vertex v0 per task, L = N+(v0) sorted, d = |L|):
//  1. Build.  L is staged in LDS.  The members among the last places of the
//     DAG's order have their out-neighbourhoods as bitmaps (hub rows), so 64
//     pairs of members are one gather and a ballot, and ranked members need
//     the pairs above the diagonal only: on R-MAT 22, 1.1e8 gathers in place of
//     nine tenths of 2.9e10 streamed elements, each with its hash probes in LDS
//     (one quarter of the roots, P13: all builds 33 -> 7.5 ms, the query 36.0 ->
//     9.8; what is left waits on the gathers' cache lines).  The out-lists
//     N+(L[i]) of the other members i are streamed as one flattened, coalesced sequence (a thread's element knows
//     its list by a forward cursor over the LDS segment offsets); each element
//     is looked up in L (binary search for one-word roots, a 16-bit position
//     hash otherwise) and, if present at position p, bit p of row i is set
//     (LDS / L2 atomic OR).  Row i is then the bitmap of L ∩ N+(L[i]), in
//     DAG order of the members.  Lists much longer than d (ratio switch) are
//     not streamed: every element of L is binary-searched in them instead
//     (galloping side of the merge/gallop choice).
//  2. Count.  k-cliques with source v0 are v0 plus a (k-1)-clique of the
//     DAG on L given by the rows.  TC needs no rows (it counts the matches of
//     step 1).  With d <= 64 every row is one 64-bit word and lane i counts
//     the cliques starting at i with AND + popcount.  With d > 64, the rows
//     are multi-word; for each i the wave compacts S = row i, and counts with
//     word-wise AND/popcount (k = 4), fp4 matrix-core products (k = 5), or the
//     rows compressed to S in registers (k = 5 on the 128-wide tier, k >= 6),
//     the last set of a search being a lane mask (count_cliques).
// Counts are exact uint64 (the matrix-core products are exact integers
// below 2^24 in f32).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "clique_dev.hpp"

namespace jk {

// ----------------------------------------------------------------------------
// Hub rows.  First the vertices of the places (inv), then a wave per row: set
// in LDS, written once (65,536 rows of R-MAT 22: 272 MB).
__global__ void __launch_bounds__(256) k_hub_places(const int32_t* ord, int32_t nv, int32_t top, int32_t* inv) {
  for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < nv; v += (int64_t)gridDim.x * 256) {
    const int32_t p = nv - 1 - ord[v];
    if (p < top) inv[p] = (int32_t)v;
  }
}
__global__ void __launch_bounds__(256) k_hub_rows(const int64_t* rp, const int32_t* ci, const int32_t* ord, int32_t nv,
                                                  int32_t top, const int32_t* inv, uint32_t* bits) {
  __shared__ __attribute__((aligned(16))) uint32_t s_row[4][HUB_TOP_MAX / 32];
  uint32_t* const row = s_row[threadIdx.x >> 6];
  uint4* const row4 = reinterpret_cast<uint4*>(row);
  const int ln = lane_id();
  for (int p = uni((int)(blockIdx.x * 4 + (threadIdx.x >> 6))); p < top; p += (int)gridDim.x * 4) {
    const int32_t v = inv[p];
    const int64_t b = rp[v], e = rp[v + 1];
    const int n4 = 8 * ((p >> 10) + 1);
    for (int t = ln; t < n4; t += 64) row4[t] = make_uint4(0u, 0u, 0u, 0u);
    __syncwarp();
    for (int64_t k = b + ln; k < e; k += 64) {
      const int32_t q = nv - 1 - ord[ci[k]];
      if (q < p) atomicOr(&row[q >> 5], 1u << (q & 31));
    }
    __syncwarp();
    uint4* const dst = reinterpret_cast<uint4*>(bits + hub_row_word((uint32_t)p));
    for (int t = ln; t < n4; t += 64) dst[t] = row4[t];
    __syncwarp();
  }
}

// a test of place q in row p reads word q / 32 also where q > p: past the last
// row at most top / 32 words
size_t hub_rows_words(int top) { return (size_t)hub_row_word((uint32_t)top) + (size_t)top / 32 + 32; }

hipError_t launch_hub_places(const int32_t* ord, int32_t nv, int32_t top, int32_t* inv, int num_cu, hipStream_t st) {
  const int64_t vb = ((int64_t)nv + 255) / 256;
  hipLaunchKernelGGL(k_hub_places, dim3((unsigned)(vb < num_cu * 8 ? vb : num_cu * 8)), dim3(256), 0, st, ord, nv, top,
                     inv);
  return hipGetLastError();
}

hipError_t launch_hub_rows(const int64_t* rp, const int32_t* ci, const int32_t* ord, int32_t nv, int32_t top,
                           int32_t* inv, uint32_t* bits, int num_cu, hipStream_t st) {
  if (top < 1 || top > nv || top > HUB_TOP_MAX) return hipErrorInvalidValue;
  const hipError_t e = launch_hub_places(ord, nv, top, inv, num_cu, st);
  if (e != hipSuccess) return e;
  const int rb = (top + 3) / 4;
  hipLaunchKernelGGL(k_hub_rows, dim3((unsigned)(rb < num_cu * 5 ? rb : num_cu * 5)), dim3(256), 0, st, rp, ci, ord, nv,
                     top, inv, bits);
  return hipGetLastError();
}

// ----------------------------------------------------------------------------
// Kernel.  G waves per root; WPB roots (groups) per block when G == 1.
// WMAX words per row => roots with d <= 64 * WMAX.  LROWS: rows in LDS,
// otherwise in a per-block slice of global scratch.
// Waves per SIMD the kernel's registers are held to.  These kernels are
// bound by latency rather than by any one unit, so on the tiers below the
// registers are capped at the occupancy their LDS allows (measured faster on
// the 5-clique tiers and the 4-clique 512-wide tier, also where they spill a
// few bytes a lane);
// elsewhere the compiler's own choice stands (already at the LDS or hardware
// limit, or the cap would spill).
template <int WMAX, int K, bool BYTES>
constexpr int min_waves() {
  if (BYTES) return 1;
  if (WMAX == 1 && K < 6) return 8;  // all blocks of the grid resident: roots are dealt by index
  if (K == 4 && WMAX == 8) return 6;
  if (K == 5 && WMAX == 4) return 8;
  if (K == 5 && WMAX == 8) return 6;
  if (K == 6 && WMAX == 4) return 7;
  if (K == 7 && WMAX == 4) return 5;
  return 1;
}
template <int G, int WPB, int WMAX, int K, bool BYTES, bool LROWS, bool FAR>
__global__ void __launch_bounds__(64 * G * WPB) __attribute__((amdgpu_waves_per_eu(min_waves<WMAX, K, BYTES>())))
clique_kernel(CliqueArgs a) {
  using LY = Lay<G, WMAX, K, BYTES, LROWS>;
  constexpr int DM = LY::DM;
  constexpr int NT = 64 * G * WPB;
  constexpr bool SMALL = WMAX == 1 && K <= 5 && !BYTES;  // roots of few members many at a time
  constexpr size_t ARENA = SMALL && sizeof(SmallRoots) > LY::SLOT ? sizeof(SmallRoots) : LY::SLOT;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[WPB][ARENA];
  __shared__ int32_t s_wtot[G + 1];
  __shared__ uint32_t s_task;
  const int slot = (G == 1) ? (int)(threadIdx.x >> 6) : 0;
  unsigned char* ar = s_arena[slot];
  uint64_t* rowp = LROWS ? reinterpret_cast<uint64_t*>(ar + LY::R_OFF)
                         : (a.gscr + (int64_t)blockIdx.x * DM * WMAX);
  const int64_t* __restrict__ rp = a.rp;
  uint64_t acc = 0;
  const HubRows hub{a.hub, a.hub_top, a.nv};
  if constexpr (G == 1) {
    // Roots are dealt by index, without a counter (one address takes an atomic
    // every 12 ns or so: 8,192 waves that only learn that the queue is empty
    // would wait 100 us).  A wave looks at 64 roots at a time, a lane each, so
    // roots outside [dmin, dmax] cost nothing: a.chunk neighbours from each of
    // 64 / a.chunk places all over the range, turned by an odd number from place
    // to place, since R-MAT degrees follow the bits of the id.
    const int ln = lane_id();
    const uint32_t nw = gridDim.x * WPB, w = blockIdx.x * WPB + slot;  // waves, this one
    const int lg = __builtin_ctz(a.chunk);
    const int64_t nplace = (a.ntasks + a.chunk - 1) >> lg;
    const int per = 64 >> lg;  // places per look
    for (int64_t s0 = 0; s0 * nw < nplace; s0 += per) {
      const int64_t row = s0 + (ln >> lg);
      const int64_t place = row * nw + (uint32_t)(w + (uint32_t)row * 0x9e3779b1u) % nw;
      const int64_t task = (place << lg) + (ln & (a.chunk - 1));
      int64_t lb = 0;
      int ld = -1;
      if (task < a.ntasks) {
        const int32_t v0 = a.ids ? a.ids[task] : (int32_t)(a.rb + task);
        lb = rp[v0];
        ld = (int)(rp[v0 + 1] - lb);
      }
      uint64_t m = __ballot(ld >= a.dmin && ld <= a.dmax && ld <= DM && ld >= 0);
      if constexpr (SMALL) {
        const bool small = ((m >> ln) & 1) && ld <= SMALL_D;
        small_roots<K, FAR>(rp, a.ci, a.ord, hub, a.ratio, lb, small ? ld : 0, *reinterpret_cast<SmallRoots*>(ar), acc);
        m &= ~__ballot(small);
        __syncwarp();
      }
      while (m) {
        const int l = __builtin_ctzll(m);
        m &= m - 1;
        process_root<G, WMAX, K, BYTES, LROWS>(rp, a.ci, a.ord, (int64_t)readlane_u64((uint64_t)lb, l),
                                               __builtin_amdgcn_readlane(ld, l), a.ratio, ar, rowp, s_wtot, acc,
                                               nullptr, hub);
      }
    }
  } else if constexpr (WMAX == 1) {
    // 6- and 7-cliques of one-word roots differ too much to be dealt by index:
    // a.chunk neighbours at a time from the queue
    const int ln = lane_id();
    for (int64_t base = (int64_t)blockIdx.x * a.chunk; base < a.ntasks;) {
      int64_t lb = 0;
      int ld = -1;
      if (ln < a.chunk && base + ln < a.ntasks) {
        const int32_t v0 = (int32_t)(a.rb + base + ln);
        lb = rp[v0];
        ld = (int)(rp[v0 + 1] - lb);
      }
      uint64_t m = __ballot(ld >= a.dmin && ld <= a.dmax && ld <= DM);
      while (m) {
        const int l = __builtin_ctzll(m);
        m &= m - 1;
        process_root<G, WMAX, K, BYTES, LROWS>(rp, a.ci, a.ord, (int64_t)readlane_u64((uint64_t)lb, l),
                                               __builtin_amdgcn_readlane(ld, l), a.ratio, ar, rowp, s_wtot, acc,
                                               nullptr, hub);
      }
      if (threadIdx.x == 0) s_task = atomicAdd(a.qctr, (uint32_t)a.chunk);
      __syncthreads();
      base = (int64_t)gridDim.x * a.chunk + s_task;  // (near 2^31 roots it passes 31 bits)
      __syncthreads();
    }
  } else {
    // a group's first root is its own index, the queue deals the others: the
    // small launches end without a counter round trip
    for (bool first = true;; first = false) {
      int32_t task = (int32_t)blockIdx.x;  // (ids of roots wider than a wave's: far below 2^31 of them)
      if (!first) {
        if (threadIdx.x == 0) s_task = gridDim.x + atomicAdd(a.qctr, 1u);
        __syncthreads();
        task = (int32_t)s_task;
        __syncthreads();
      }
      if (task >= a.ntasks) break;
      const int32_t v0 = a.ids ? a.ids[task] : (int32_t)(a.rb + task);
      const int64_t b0 = rp[v0];
      const int d = (int)(rp[v0 + 1] - b0);
      if (d < a.dmin || d > a.dmax || d > DM) continue;
      process_root<G, WMAX, K, BYTES, LROWS>(rp, a.ci, a.ord, b0, d, a.ratio, ar, rowp, s_wtot, acc, nullptr, hub);
    }
  }
  block_add<NT>(acc, a.out);
}

// ---------------------------------------------------------------------------
// Split form of the 1024-wide tier: the build runs with 16 waves per root
// (twice the waves that the count's registers and per-wave lists allow) and
// leaves each root's rows in a global slot; the count kernel reloads them.
// Task t (of a.ids) uses slot t of a.gscr, ROWW words each.
constexpr int SPLIT_WMAX = 16;
constexpr size_t ROWW = (size_t)64 * SPLIT_WMAX * SPLIT_WMAX;

template <int K>
__global__ void __launch_bounds__(64 * 16) clique_build_kernel(CliqueArgs a) {
  constexpr int G = 16;
  using LY = Lay<G, SPLIT_WMAX, K, false, true, false>;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[LY::SLOT];
  __shared__ int32_t s_wtot[G + 1];
  __shared__ int64_t s_task;
  uint64_t* rowp = reinterpret_cast<uint64_t*>(s_arena + LY::R_OFF);
  uint64_t acc = 0;
  for (;;) {
    if (threadIdx.x == 0) s_task = (int64_t)atomicAdd(a.qctr, 1u);
    __syncthreads();
    const int64_t task = uni((int)s_task);
    __syncthreads();
    if (task >= a.ntasks) break;
    const int32_t v0 = uni(a.ids[task]);
    const int64_t b0 = a.rp[v0];
    const int d = uni((int)(a.rp[v0 + 1] - b0));
    if (d < a.dmin || d > a.dmax || d > LY::DM) continue;
    process_root<G, SPLIT_WMAX, K, false, true, 1>(a.rp, a.ci, a.ord, b0, d, a.ratio, s_arena, rowp, s_wtot, acc,
                                                   nullptr, HubRows{a.hub, a.hub_top, a.nv});
    const int n = d * RowLayout((d + 63) >> 6).S;
    uint64_t* dst = a.gscr + (size_t)task * ROWW;
    for (int t = threadIdx.x; t < n; t += 64 * G) dst[t] = rowp[t];
    __syncthreads();
  }
}

// Waves per root of the count kernel: 12 (three per SIMD, all the LDS
// allows beside the rows) where the count fits the registers of three waves;
// the 7-clique count would spill there, so it keeps 8.
template <int K>
constexpr int split_count_waves() { return (K == 7) ? 8 : 12; }

template <int K>
__global__ void __launch_bounds__(64 * split_count_waves<K>()) clique_count_kernel(CliqueArgs a) {
  constexpr int G = split_count_waves<K>();
  using LY = Lay<G, SPLIT_WMAX, K, false, true, true, false>;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[LY::SLOT];
  __shared__ int32_t s_wtot[G + 1];
  __shared__ int64_t s_task;
  uint64_t* rowp = reinterpret_cast<uint64_t*>(s_arena + LY::R_OFF);
  uint64_t acc = 0;
  for (;;) {
    if (threadIdx.x == 0) s_task = (int64_t)atomicAdd(a.qctr, 1u);
    __syncthreads();
    const int64_t task = uni((int)s_task);
    __syncthreads();
    if (task >= a.ntasks) break;
    const int32_t v0 = uni(a.ids[task]);
    const int64_t b0 = a.rp[v0];
    const int d = uni((int)(a.rp[v0 + 1] - b0));
    if (d < a.dmin || d > a.dmax || d > LY::DM) continue;
    const int n = d * RowLayout((d + 63) >> 6).S;
    const uint64_t* src = a.gscr + (size_t)task * ROWW;
    for (int t = threadIdx.x; t < n; t += 64 * G) rowp[t] = __builtin_nontemporal_load(src + t);
    if (threadIdx.x == 0) s_wtot[G] = 0;
    __syncthreads();
    process_root<G, SPLIT_WMAX, K, false, true, 2>(a.rp, a.ci, a.ord, b0, d, a.ratio, s_arena, rowp, s_wtot, acc);
  }
  block_add<64 * G>(acc, a.out);
}

template <int K>
static hipError_t launch_split_k(bool build, const CliqueArgs& a, int grid, hipStream_t st) {
  if (build) hipLaunchKernelGGL(clique_build_kernel<K>, dim3(grid), dim3(64 * 16), 0, st, a);
  else hipLaunchKernelGGL(clique_count_kernel<K>, dim3(grid), dim3(64 * split_count_waves<K>()), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_clique_split(int k, bool build, const CliqueArgs& a, int grid, hipStream_t st) {
  switch (k) {
    case 4: return launch_split_k<4>(build, a, grid, st);
    case 5: return launch_split_k<5>(build, a, grid, st);
    case 6: return launch_split_k<6>(build, a, grid, st);
    case 7: return launch_split_k<7>(build, a, grid, st);
  }
  return hipErrorInvalidValue;
}

size_t split_slot_words() { return ROWW; }

// ---------------------------------------------------------------------------
// Split form of the 128- to 512-wide tiers for 6- and 7-cliques.  A root's
// rows differ by orders of magnitude in the cliques below them, so a block per
// root ended with a few blocks at work (R-MAT 16 P15: 1,834 128-wide roots, the
// heaviest holding 0.3 % of the work, took 12.6 of 17 ms after the others).
// Here the build leaves each root's rows in a global slot and the count takes
// one (root, row) per wave, row by row over all roots: the heavy early rows
// first.  A row's set is compressed to registers straight from the slot (L2).
// P15 on R-MAT 16: 76 -> 12.9 ms, R-MAT 18: 528 -> 101 ms; an edge of a set costs
// about 90 cycles of a SIMD (8 VALU and 6 SALU instructions, their latency and
// the loop's branches), which bounds it.
constexpr size_t rows_slot(int wmax) { return (size_t)64 * wmax * wmax; }

template <int G, int WMAX>
__global__ void __launch_bounds__(64 * G) clique_rows_build_kernel(CliqueArgs a) {
  using LY = Lay<G, WMAX, 4, false, true, false>;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[LY::SLOT];
  __shared__ int32_t s_wtot[G + 1];
  uint64_t* rowp = reinterpret_cast<uint64_t*>(s_arena + LY::R_OFF);
  uint64_t acc = 0;
  for (int64_t task = blockIdx.x; task < a.ntasks; task += gridDim.x) {
    const int32_t v0 = uni(a.ids[task]);
    const int64_t b0 = a.rp[v0];
    const int d = uni((int)(a.rp[v0 + 1] - b0));
    if (d < a.dmin || d > a.dmax || d > LY::DM) continue;
    process_root<G, WMAX, 4, false, true, 1>(a.rp, a.ci, a.ord, b0, d, a.ratio, s_arena, rowp, s_wtot, acc, nullptr,
                                             HubRows{a.hub, a.hub_top, a.nv});
    const int n = d * RowLayout((d + 63) >> 6).S;
    uint64_t* dst = a.gscr + (size_t)task * rows_slot(WMAX);
    for (int t = threadIdx.x; t < n; t += 64 * G) dst[t] = rowp[t];
    __syncthreads();
  }
}

template <int K, int WMAX>
__global__ void __launch_bounds__(256) clique_rows_count_kernel(CliqueArgs a) {
  constexpr int DM = 64 * WMAX;
  constexpr bool LIST = K - 2 > 4;
  __shared__ int16_t s_J[4][DM];
  __shared__ uint64_t s_rc[LIST ? 4 : 1][LIST ? 256 : 1];
  __shared__ uint16_t s_list[LIST ? 4 : 1][LIST ? FLAT_LIST : 1];
  const int wv = threadIdx.x >> 6;
  const int ln = lane_id();
  int16_t* const J = s_J[wv];
  uint64_t* const rc = s_rc[LIST ? wv : 0];
  uint16_t* const list = s_list[LIST ? wv : 0];
  uint64_t acc = 0;
  // the first quarter of the rows, which hold the wide sets, by PARTS waves
  // each (a set of more than 64 members; else the first does it alone)
  constexpr int PARTS = 4;
  const int64_t nw = (int64_t)gridDim.x * 4, early = a.ntasks * (DM / 4) * PARTS;
  for (int64_t t = (int64_t)blockIdx.x * 4 + wv; t < early + a.ntasks * (DM - DM / 4); t += nw) {
    const int64_t u = t < early ? t / PARTS : t - early;
    const int part = t < early ? (int)(t % PARTS) : 0;
    const int i0 = (int)(u / a.ntasks);
    const int64_t task = u - (int64_t)i0 * a.ntasks;
    const int i = uni(t < early ? i0 : i0 + DM / 4);
    const int32_t v0 = uni(a.ids[task]);
    const int64_t b0 = a.rp[v0];
    const int d = uni((int)(a.rp[v0 + 1] - b0));
    if (i >= d || d < a.dmin || d > a.dmax || d > DM) continue;
    const int W = (d + 63) >> 6;
    const RowsCached R{a.gscr + (size_t)task * rows_slot(WMAX), RowLayout(W)};
    // S = row i: its members' positions
    const uint64_t myword = ln < W ? R(i, ln) : 0ull;
    __syncwarp();
    int n = 0;
    for (int w = 0; w < W; ++w) {
      const uint64_t word = readlane_u64(myword, w);
      if ((word >> ln) & 1ull) J[n + below(word)] = (int16_t)((w << 6) | ln);
      n += __popcll(word);
    }
    __syncwarp();
    if (n < K - 2 || (n <= 64 && part > 0)) continue;
    const int ps = t < early ? PARTS : 1;
    if (n <= 64) {
      uint64_t row[1][1];
      compress_rows<1>(R, J, n, row, LIST ? rc : nullptr);
      acc += count_cliques<K - 2, 1, true>(row, rc, list, n);
    } else if (n <= 128) {
      uint64_t row[2][2];
      compress_rows<2>(R, J, n, row, LIST ? rc : nullptr);
      acc += count_cliques<K - 2, 2, true>(row, rc, list, n, part, ps);
    } else if (K == 6 && n <= 256) {
      if constexpr (K == 6 && WMAX > 2) {
        uint64_t row[4][4];
        compress_rows<4>(R, J, n, row, nullptr);
        acc += count_cliques<4, 4, true>(row, nullptr, nullptr, n, part, ps);
      }
    } else if constexpr (WMAX > 2) {
      // lanes over the members: candidate sets in registers, rows from L2
      for (int q = 64 * part + ln; q < n; q += 64 * ps) {
        const int j = J[q];
        const int ws = (j + 1) >> 6;  // row j has no bits before its own position
        uint64_t c[WMAX];
#pragma unroll
        for (int w = 0; w < WMAX; ++w) c[w] = (w >= ws && w < W) ? (R(i, w) & R(j, w)) : 0ull;
        acc += recR<K - 3, WMAX, false>(c, 0, W, R, nullptr);
      }
    }
  }
  block_add<256>(acc, a.out);
}

template <int K, int WMAX>
static hipError_t launch_rows_w(bool build, const CliqueArgs& a, int num_cu, int maxgrid, hipStream_t st) {
  constexpr int G = WMAX == 8 ? 8 : 4;
  if (build)
    hipLaunchKernelGGL((clique_rows_build_kernel<G, WMAX>), dim3((unsigned)(a.ntasks < maxgrid ? a.ntasks : maxgrid)),
                       dim3(64 * G), 0, st, a);
  else
    hipLaunchKernelGGL((clique_rows_count_kernel<K, WMAX>), dim3(8 * num_cu), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_clique_rows(int k, int tier, bool build, const CliqueArgs& a, int num_cu, int maxgrid,
                              hipStream_t st) {
  switch (k * 8 + tier) {
    case 6 * 8 + TIER_LDS2: return launch_rows_w<6, 2>(build, a, num_cu, maxgrid, st);
    case 6 * 8 + TIER_LDS4: return launch_rows_w<6, 4>(build, a, num_cu, maxgrid, st);
    case 6 * 8 + TIER_LDS8: return launch_rows_w<6, 8>(build, a, num_cu, maxgrid, st);
    case 7 * 8 + TIER_LDS2: return launch_rows_w<7, 2>(build, a, num_cu, maxgrid, st);
    case 7 * 8 + TIER_LDS4: return launch_rows_w<7, 4>(build, a, num_cu, maxgrid, st);
    case 7 * 8 + TIER_LDS8: return launch_rows_w<7, 8>(build, a, num_cu, maxgrid, st);
  }
  return hipErrorInvalidValue;
}

size_t rows_slot_words(int tier) { return rows_slot(tier == TIER_LDS2 ? 2 : tier == TIER_LDS4 ? 4 : 8); }

// ---------------------------------------------------------------------------
// Split form of the 2048-wide tier for 5- to 7-cliques.  The fused kernel
// counts a root with one block of 8 waves (two per SIMD, the registers of
// the 2x2 matrix-core tiles), so the roots of a query run about one per CU
// and the densest ones leave the device waiting.  Here a build kernel with
// 16 waves per root leaves each root's rows (512 KiB) in a global slot, and
// the count kernel lets a.rep blocks take the rows of one root from a shared
// global row counter.  (4-cliques keep the fused kernel: their whole-root
// product is not split by rows.)
constexpr int GLB_WMAX = 32;
constexpr size_t GSLOT = (size_t)64 * GLB_WMAX * GLB_WMAX;

template <int K>
__global__ void __launch_bounds__(64 * 16) clique_glb_build_kernel(CliqueArgs a) {
  constexpr int G = 16;
  using LY = Lay<G, GLB_WMAX, K, false, false, false>;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[LY::SLOT];
  __shared__ int32_t s_wtot[G + 1];
  __shared__ int64_t s_task;
  uint64_t acc = 0;
  for (;;) {
    if (threadIdx.x == 0) s_task = (int64_t)atomicAdd(a.qctr, 1u);
    __syncthreads();
    const int64_t task = uni((int)s_task);
    __syncthreads();
    if (task >= a.ntasks) break;
    const int32_t v0 = uni(a.ids[task]);
    const int64_t b0 = a.rp[v0];
    const int d = uni((int)(a.rp[v0 + 1] - b0));
    if (d < a.dmin || d > a.dmax || d > LY::DM) continue;
    process_root<G, GLB_WMAX, K, false, false, 1>(a.rp, a.ci, a.ord, b0, d, a.ratio, s_arena,
                                                  a.gscr + (size_t)task * GSLOT, s_wtot, acc, nullptr,
                                                  HubRows{a.hub, a.hub_top, a.nv});
  }
}

template <int K>
__global__ void __launch_bounds__(64 * 8) clique_glb_count_kernel(CliqueArgs a) {
  constexpr int G = 8;
  using LY = Lay<G, GLB_WMAX, K, false, false, true, false>;
  __shared__ __attribute__((aligned(16))) unsigned char s_arena[LY::SLOT];
  __shared__ int32_t s_wtot[G + 1];
  __shared__ int64_t s_item;
  uint64_t acc = 0;
  // Workgroups are dealt to the 8 XCDs round robin, so block b runs on XCD
  // b % 8.  Queue q (counter a.rowctr[q - 8]) holds the roots q, q + 8, ...,
  // each as rep items that start together: the blocks sharing a root's
  // 512 KiB of rows are on one XCD and read them through its L2.  A block
  // drains its own XCD's queue, then helps the others.
  uint32_t* const qx = a.rowctr - 8;
  const int xcd = (int)(blockIdx.x & 7);
  for (int s = 0; s < 8; ++s) {
    const int q = (xcd + s) & 7;
    const int64_t nq = a.ntasks > q ? ((a.ntasks - 1 - q) / 8 + 1) * a.rep : 0;
    for (;;) {
      if (threadIdx.x == 0) s_item = (int64_t)atomicAdd(qx + q, 1u);
      __syncthreads();
      const int64_t item = uni((int)s_item);
      __syncthreads();
      if (item >= nq) break;
      const int64_t task = (item / a.rep) * 8 + q;
      const int32_t v0 = uni(a.ids[task]);
      const int64_t b0 = a.rp[v0];
      const int d = uni((int)(a.rp[v0 + 1] - b0));
      if (d < a.dmin || d > a.dmax || d > LY::DM) continue;
      process_root<G, GLB_WMAX, K, false, false, 2>(a.rp, a.ci, a.ord, b0, d, a.ratio, s_arena,
                                                    a.gscr + (size_t)task * GSLOT, s_wtot, acc, a.rowctr + task);
    }
  }
  block_add<64 * G>(acc, a.out);
}

template <int K>
static hipError_t launch_glb_split_k(bool build, const CliqueArgs& a, int grid, hipStream_t st) {
  if (build) hipLaunchKernelGGL(clique_glb_build_kernel<K>, dim3(grid), dim3(64 * 16), 0, st, a);
  else hipLaunchKernelGGL(clique_glb_count_kernel<K>, dim3(grid), dim3(64 * 8), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_clique_glb_split(int k, bool build, const CliqueArgs& a, int grid, hipStream_t st) {
  switch (k) {
    case 5: return launch_glb_split_k<5>(build, a, grid, st);
    case 6: return launch_glb_split_k<6>(build, a, grid, st);
    case 7: return launch_glb_split_k<7>(build, a, grid, st);
  }
  return hipErrorInvalidValue;
}

size_t glb_slot_words() { return GSLOT; }

// ---------------------------------------------------------------------------
// Host-side launch table.
// 6- and 7-clique roots up to this out-degree run one wave each.
constexpr int SMALL_ROOT = 24;

template <int G, int WPB, int WMAX, int K, bool BYTES, bool LROWS, bool FAR = false>
static hipError_t launch_one(const CliqueArgs& a, int grid, hipStream_t st) {
  hipLaunchKernelGGL((clique_kernel<G, WPB, WMAX, K, BYTES, LROWS, FAR>), dim3(grid), dim3(64 * G * WPB), 0, st, a);
  return hipGetLastError();
}

template <int K, bool BYTES>
static hipError_t launch_k(int tier, const CliqueArgs& a, int grid, hipStream_t st) {
  switch (tier) {
    case TIER_WAVE:
      // 6- and 7-cliques of the wider one-word roots: four waves share a root
      // (their subtrees would leave one wave running alone at the end)
      if constexpr (!BYTES && K >= 6)
        if (a.dmin > SMALL_ROOT) return launch_one<4, 1, 1, K, BYTES, true>(a, grid, st);
      if constexpr (!BYTES && K < 6)
        if (a.far) return launch_one<1, 4, 1, K, BYTES, true, true>(a, grid, st);
      return launch_one<1, 4, 1, K, BYTES, true>(a, grid, st);
    case TIER_LDS2:   return launch_one<4, 1, 2, K, BYTES, true>(a, grid, st);
    case TIER_LDS4:   return launch_one<4, 1, 4, K, BYTES, true>(a, grid, st);
    case TIER_LDS8:   return launch_one<8, 1, 8, K, BYTES, true>(a, grid, st);
    case TIER_LDS16:  return launch_one<8, 1, 16, K, BYTES, true>(a, grid, st);
    case TIER_GLB32:  return launch_one<8, 1, 32, K, BYTES, false>(a, grid, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_clique(int k, bool bytes, int tier, const CliqueArgs& a, int grid, hipStream_t st) {
  switch (k) {
    case 3: return bytes ? launch_k<3, true>(tier, a, grid, st) : launch_k<3, false>(tier, a, grid, st);
    case 4: return bytes ? launch_k<4, true>(tier, a, grid, st) : launch_k<4, false>(tier, a, grid, st);
    case 5: return bytes ? launch_k<5, true>(tier, a, grid, st) : launch_k<5, false>(tier, a, grid, st);
    case 6: return bytes ? launch_k<6, true>(tier, a, grid, st) : launch_k<6, false>(tier, a, grid, st);
    case 7: return bytes ? launch_k<7, true>(tier, a, grid, st) : launch_k<7, false>(tier, a, grid, st);
  }
  return hipErrorInvalidValue;
}

int clique_small_root() { return SMALL_ROOT; }

int tier_max_deg(int tier) {
  switch (tier) {
    case TIER_WAVE: return 64;
    case TIER_LDS2: return 128;
    case TIER_LDS4: return 256;
    case TIER_LDS8: return 512;
    case TIER_LDS16: return 1024;
    case TIER_GLB32: return 2048;
  }
  return 0;
}

size_t tier_scratch_words(int tier) {
  return tier == TIER_GLB32 ? (size_t)2048 * 32 : 0;
}

}  // namespace jk
