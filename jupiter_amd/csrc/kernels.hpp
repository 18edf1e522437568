// Device kernel entry points of libjgpm (host-callable launchers).
#pragma once
#include "plan.hpp"
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace jk {

// Root tiers of the clique engine, by DAG out-degree d of the root.
enum {
  TIER_WAVE = 0,   // d <= 64    one wave per root, one-word rows in LDS
  TIER_LDS2 = 1,   // d <= 128   block per root, rows in LDS
  TIER_LDS4 = 2,   // d <= 256
  TIER_LDS8 = 3,   // d <= 512
  TIER_LDS16 = 4,  // d <= 1024  (128 KB of rows in LDS, one block per CU)
  TIER_GLB32 = 5,  // d <= 2048  block per root, rows in a global scratch slice
  NUM_TIERS = 6
};

struct CliqueArgs {
  const int64_t* rp;     // DAG row pointers
  const int32_t* ci;     // DAG column indices
  const int32_t* ord;    // position of every vertex in a topological order of the DAG
  const int32_t* ids;    // task -> root vertex (NULL: root = rb + task)
  int64_t rb;
  int64_t ntasks;
  int32_t dmin, dmax;    // roots outside [dmin, dmax] are skipped by this launch
  int32_t ratio;         // a list longer than ratio * d is binary-searched, not streamed
  int32_t chunk;         // roots taken per queue grab (wave tier)
  uint32_t* qctr;        // work-queue counter (zero before launch)
  uint64_t* gscr;        // global row scratch (TIER_GLB32)
  uint64_t* out;         // uint64 accumulator
  uint32_t* rowctr;      // split 2048-wide count: one row counter per task, 8 queue
                         // counters before them (all zero before)
  int32_t rep;           // split 2048-wide count: blocks per task
  const uint32_t* hub;   // hub rows (launch_hub_rows), of the hub_top last places of ord
  int32_t hub_top;       // 0: none
  int32_t nv;
  int32_t far;           // some vertex may have a list that is long for a small root (small_roots)
};

// Out-neighbourhoods of the `top` last vertices of ord as bitmaps
// (hub_rows_words(top) 32-bit words at bits; inv: top entries of scratch).
constexpr int HUB_TOP_MAX = 65536;
size_t hub_rows_words(int top);
// inv[p] = the vertex p places from the end of ord, p < top
hipError_t launch_hub_places(const int32_t* ord, int32_t nv, int32_t top, int32_t* inv, int num_cu, hipStream_t st);
hipError_t launch_hub_rows(const int64_t* rp, const int32_t* ci, const int32_t* ord, int32_t nv, int32_t top,
                           int32_t* inv, uint32_t* bits, int num_cu, hipStream_t st);

// Query descriptor as the persistent kernel sees it.
struct BQ {
  const int64_t* rp;
  const int32_t* ci;
  const int32_t* ord;
  const int32_t* src;
  const int32_t* tri;
  const int64_t* nsum;
  int64_t base;    // first root (clique) or first edge id (P1..P12)
  int64_t ntasks;  // roots or edges
  int32_t kind;    // 3..7: clique size; 100 + P: symmetric pattern P
  int32_t chunk;   // roots / edges per chunk
};

hipError_t launch_clique(int k, bool bytes, int tier, const CliqueArgs& a, int grid, hipStream_t st);
// Split form of TIER_LDS16 for counting (k >= 4): build kernel (rows to
// a.gscr slots of split_slot_words() words per task), then count kernel.
hipError_t launch_clique_split(int k, bool build, const CliqueArgs& a, int grid, hipStream_t st);
size_t split_slot_words();
// Split form of TIER_LDS2 .. TIER_LDS8 for k >= 6: build kernel (rows to a.gscr
// slots of rows_slot_words(tier) words per task), then a count kernel with a
// wave per (task, row).
hipError_t launch_clique_rows(int k, int tier, bool build, const CliqueArgs& a, int num_cu, int maxgrid,
                              hipStream_t st);
size_t rows_slot_words(int tier);
// Split form of TIER_GLB32 for k >= 5: build kernel (16 waves per root, rows
// to a.gscr slots of glb_slot_words() words per task), then count kernel
// (a.rep blocks per task share the root's rows through a.rowctr[task]).
hipError_t launch_clique_glb_split(int k, bool build, const CliqueArgs& a, int grid, hipStream_t st);
size_t glb_slot_words();

// Symmetric-graph patterns P1..P12: one wave per directed edge of [e0, e0+ne).
struct SymArgs {
  const int64_t* rp;     // symmetric row pointers
  const int32_t* ci;     // symmetric column indices
  const int32_t* src;    // COO source of every directed edge
  const int32_t* tri;    // per directed edge |N(u) ∩ N(v)| (patterns that use it)
  const int64_t* nsum;   // per vertex sum of neighbour degrees (P3)
  int64_t e0, ne;        // edge range
  unsigned long long* qctr;
  int32_t chunk;         // edges per queue grab
  int32_t* scr;          // per-wave list scratch for lists longer than the LDS capacity
  int64_t scr_stride;    // ints per scratch list (>= max degree)
  uint64_t* out;
  // P5, P7, P9, P11, P12: edges with heavy_min < tri[e] <= sym_heavy_nmax()
  // go to launch_sym_heavy (0: every edge runs here; needs tri)
  int32_t heavy_min;
  int32_t heavy_stream;  // stream N(v2) when d(v2) <= heavy_stream * |S|, else binary searches
  int32_t nv;            // vertices (the heavy kernel keeps S as a bitmap on small graphs)
  // the wave-per-edge launch appends each heavy edge to list 0 (|S| <=
  // heavy_mid), 1 (|S| <= sym_heavy_nmax()) or 2 (beyond, on graphs of at
  // most 2^20 vertices), at hlist + list * hcap, counters hctr[0..2]; an edge
  // that finds its list full it counts itself.  The heavy launches pop with
  // hctr[3..5].
  int32_t* hlist;
  unsigned long long* hctr;
  int32_t hcap;
  int32_t heavy_mid;
};
hipError_t launch_sym(int p, const SymArgs& a, int grid, hipStream_t st);
// The heavy edges of P5, P7, P9, P11 and P12, one block per edge, popped
// from list `shape` (0, 1, 2 as above) that launch_sym filled; shape 2 keeps
// S in the block's slice of a.scr (a.scr_stride ints, grid slices).
bool sym_heavy_pattern(int p);
int sym_heavy_nmax();
int sym_heavy_stream();
int sym_heavy_mid(int p);  // |S| up to this: the narrow launch (more blocks per CU)
hipError_t launch_sym_heavy(int p, const SymArgs& a, int shape, int grid, hipStream_t st);

// Patterns counted by wedges (wedge.hip).  4-cycles (P1): every root range of
// one or more queries in one sequence of launches.
enum { WEDGE_P1 = 0, WEDGE_P4 = 1, WEDGE_P6 = 2 };
struct P1Q {
  const int64_t* rp;
  const int32_t* ci;
  const int32_t* src;    // source of every directed edge
  int64_t e0, ne;        // directed edges of the root range
  int64_t rb, nr;        // first root, number of roots
  int64_t eoff, roff;    // the query's first entry in the per-edge and per-root scratch
  int32_t xmin;          // ids below have at most one neighbour (0: unknown)
  int32_t slot;          // its accumulator is out[slot]
  // single queries only:
  int64_t scale = 1;     // what the count is multiplied by
  const int32_t* csrc = nullptr;  // P8, P6 (roots are directed edges): the edges' sources ...
  const int64_t* crp = nullptr;   // ... and row pointers: a P8 root's ids start at crp[csrc[root]] - cbase
  int64_t cbase = 0;
  const int32_t* vid = nullptr;   // P6: the edges' ends
  const int64_t* lrp = nullptr;   // P6: the lists
  const int32_t* lci = nullptr;
  const int32_t* weight = nullptr;  // P4: per edge its triangles
  int32_t xend = 0;      // P4, P6: ids end here
  int32_t pad = 0;
};
struct P1Args {
  P1Q one;               // the query, when q is null
  const P1Q* q;          // device table of nq queries
  int nq;
  const int64_t* tcs;    // prefix of the queries' 256-edge tiles (nq + 1)
  const int64_t* rcs;    // prefix of the queries' roots (nq + 1)
  int64_t tiles, roots, edges;  // totals
  unsigned long long* ctr;      // scratch: list and task counters (8)
  uint64_t* W;                  // per root its wedges
  int32_t* m0;                  // per root its neighbours below it
  int2* list;                   // roots (root, query) as wave tasks from the front, block tasks from the back
  int2* split;                  // roots taken by several blocks
  int32_t* len;                 // per edge (v0, v) the neighbours of v below v0
  uint64_t* out;
};
size_t p1_scratch_bytes(int64_t roots, int64_t edges);
void p1_bind_scratch(P1Args& a, void* p);  // a.roots and a.edges set
hipError_t launch_wedge(int mode, const P1Args& a, int num_cu, hipStream_t st);  // P4, P6: one query

// One wave per root vertex v_0 of [rb, re) on the symmetric CSR.
struct PlanArgs {
  const int64_t* rp;
  const int32_t* ci;
  int64_t rb, re;
  unsigned long long* qctr;
  int32_t* scr;                  // per wave (k + 1) lists of `stride` ints
  int64_t stride;                // >= maximum degree
  uint64_t* out;
  Plan plan;
};
constexpr int PLAN_WPB = 4;
hipError_t launch_plan(const PlanArgs& a, int grid, hipStream_t st);
// Per-edge triangle counts, and the patterns that are sums over triangles
// (tri_engine.hip).
struct TriArgs {
  const int64_t* rp;     // symmetric CSR
  const int32_t* ci;
  const int64_t* drp;    // degree DAG
  const int32_t* dci;
  const int32_t* ord;    // position of every vertex in the degree order
  const int32_t* dtri;   // triangles per DAG edge (sums only)
  int32_t nv;
  int32_t vchunk;        // vertices a wave takes at a time (1 .. 64)
  int32_t wide;          // some vertex has more neighbours than a wave task takes
  int32_t nhub;          // hubs: the last nhub vertices of the degree order
  const uint32_t* hub;   // their neighbours as bitmaps over the vertices
  int64_t hwords;        // words per bitmap (a multiple of 4)
  int64_t rb, re;        // root range
  unsigned long long* ctr;      // scratch: list and task counters (8)
  int32_t* list;                // 3 lists of nv roots
  int32_t* lscr;                // 3 arrays of lstride ints per block
  int64_t lstride;              // >= the DAG's maximum out-degree
  uint64_t* rows;               // rows of roots too wide for LDS, rstride words per block
  int64_t rstride;
  uint64_t* out;
};
constexpr int TRI_MAX_OUT = 1 << 16;   // out-neighbours of a root: the sums' pair queues hold 16-bit positions
constexpr int TRI_SMALL_PER_CU = 6;  // blocks per CU of the narrow block tier
int64_t tri_row_words(int64_t d, int64_t dp);  // words of the rows of a root (degree d, out-degree dp)
bool tri_rows_global(int64_t d, int64_t dp);   // ... which do not fit LDS
// the hubs' bitmaps, then with them:
hipError_t launch_hub_bitmaps(const TriArgs& a, int num_cu, hipStream_t st);
// triangles of every DAG edge and of every symmetric edge (src: their sources)
hipError_t launch_tri_build(const TriArgs& a, int32_t* dtri, const int32_t* src, int64_t ne, int32_t* tri, int num_cu,
                            hipStream_t st);
// P5, P7, P9, P11 or P12, or the triangle parts of P4 and P10, over [rb, re); gblocks blocks for the roots whose
// rows are in a.rows (0: none)
hipError_t launch_tri_sum(int p, const TriArgs& a, int num_cu, int gblocks, hipStream_t st);

// The graph of induced neighbourhoods over the directed edges [e0, e0 + n)
// (whole roots): a vertex per edge (v0, u), joined to (v0, y) for every common
// neighbour y of v0 and u; vertices are numbered from 0.
struct EgoArgs {
  const int32_t* src;   // the edges' sources, triangle counts (whole graph)
  const int32_t* tri;
  int64_t e0, n;
  int64_t* tiles;       // scratch, ego_tiles(n)
  int64_t* rp;          // out: n + 1 row pointers
  int32_t* ci;          // out: entries, ascending in each row
  int32_t* row;         // out: their rows
};
int64_t ego_tiles(int64_t n);
hipError_t launch_ego_build(const TriArgs& a, const EgoArgs& g, int num_cu, hipStream_t st);  // with the hub bitmaps
hipError_t launch_p10_rows(const EgoArgs& g, uint64_t* out, int num_cu, hipStream_t st);
// closed per-edge parts: P4 (mode 0: root range, 1: whole graph), P6 (mode 2)
hipError_t launch_edge_base(const int64_t* rp, const int32_t* ci, const int32_t* src, const int32_t* tri, int64_t e0,
                            int64_t e1, int mode, uint64_t* out, int num_cu, hipStream_t st);
// P3 (p3; needs nsum) or tailed triangles over the edges [e0, e1) of a root
// range; *flag zero before
hipError_t launch_edge_sum(bool p3, const int64_t* rp, const int32_t* ci, const int32_t* src, const int32_t* tri,
                           const int64_t* nsum, int64_t e0, int64_t e1, unsigned long long* flag, uint64_t* out,
                           int num_cu, hipStream_t st);
// what the edges of every EDGE_WORK_BLOCK vertices cost the per-edge launches of P4 to P12, and the triangle sums
// (a.rp, ci, drp and nv)
constexpr int EDGE_WORK_BLOCK = 16;
__host__ __device__ inline int64_t edge_work_blocks(int64_t nv) { return (nv + EDGE_WORK_BLOCK - 1) / EDGE_WORK_BLOCK; }
hipError_t launch_edge_work(const TriArgs& a, const int32_t* src, const int32_t* tri, float4* work, hipStream_t st);
hipError_t launch_root_tri(const int64_t* rp, const int32_t* tri, int32_t nv, int64_t* sum, int num_cu, hipStream_t st);

int sym_waves_per_block();
int sym_lists_per_wave();
hipError_t launch_aux_src(const int64_t* rp, int32_t nv, int32_t* src, int grid, hipStream_t st);
hipError_t launch_aux_nsum(const int64_t* rp, const int32_t* ci, int32_t nv, int64_t* nsum, int grid, hipStream_t st);
// 3-stars: sum of C(d, 3) over the vertices [rb, re)
hipError_t launch_star3(const int64_t* rp, int64_t rb, int64_t re, unsigned long long* out, int grid, hipStream_t st);
// Diamonds over the directed edges [e0, e1) from the per-edge triangle array.
hipError_t launch_p2_edges(const int32_t* src, const int32_t* ci, const int32_t* tri, int64_t e0, int64_t e1,
                           unsigned long long* out, int grid, hipStream_t st);
int tier_max_deg(int tier);
// TIER_WAVE of 6- and 7-cliques runs as two launches: roots up to this
// out-degree with a wave each, wider ones (a.dmin above it) with a block each
int clique_small_root();
size_t tier_scratch_words(int tier);

// Roots wider than the widest row tier (DAG out-degree > 2048): the level
// nest per root, lists in global scratch (clique_huge.hip).
struct HugeArgs {
  const int64_t* rp;     // DAG row pointers
  const int32_t* ci;     // DAG column indices
  const int32_t* ids;    // the roots
  int64_t ntasks;
  int32_t* scr;          // huge_lists_per_block(k) * grid lists of stride ints
  int64_t stride;        // >= the DAG's maximum out-degree
  uint64_t* out;
};
int huge_lists_per_block(int k);
hipError_t launch_clique_huge(int k, const HugeArgs& a, int grid, hipStream_t st);

}  // namespace jk
