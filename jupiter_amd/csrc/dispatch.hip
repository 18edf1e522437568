// dispatch.hip — pattern id -> kernels, and the combination of partial
// accumulators into the final count.
//
// The reference chooses kernels by string compare and asserts on an unknown
// name (src/jupiter_gpm.cu:391-433,435-873); here an id selects an enqueue
// routine and an unknown id is JGPM_E_PATTERN.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "jgpm_device.hpp"

namespace jgpm {

static int grid_for(jgpm_ctx_s* c, int per_cu) { return std::max(1, per_cu) * c->num_cu; }

static thread_local jgpm_ctx_s* t_exec = nullptr;

jgpm_ctx_s* exec_ctx(const jgpm_graph_s* g) { return t_exec ? t_exec : g->ctx; }
ExecScope::ExecScope(jgpm_ctx_s* c) : prev(t_exec) { t_exec = c; }
ExecScope::~ExecScope() { t_exec = prev; }

size_t ws_held(const jgpm_ctx_s* c) {
  return c->hub_bytes + c->ego_bytes + c->te_bytes + c->p1_bytes + sizeof(uint64_t) * c->scr_words +
         sizeof(int32_t) * (c->sscr_ints + 3 * (size_t)c->hcap);
}

void ws_release(jgpm_ctx_s* c) {
  void* p[] = {c->d_hub, c->d_ego, c->d_te, c->d_p1, c->d_scr, c->d_sscr, c->d_hlist};
  for (void* x : p)
    if (x) (void)hipFree(x);
  c->d_hub = c->d_ego = c->d_te = c->d_p1 = nullptr;
  c->d_scr = nullptr;
  c->d_sscr = c->d_hlist = nullptr;
  c->hub_bytes = c->ego_bytes = c->te_bytes = c->p1_bytes = c->scr_words = c->sscr_ints = 0;
  c->hcap = 0;
}

// Bytes a workspace that holds `have` may take under the context's cap.
static size_t ws_room(const jgpm_ctx_s* c, size_t have) {
  const size_t others = ws_held(c) - have;
  return c->ws_cap > others ? c->ws_cap - others : 0;
}

// Grows one of the context's scratch buffers to `need` bytes (allocates, never
// while capturing); its contents are lost.  More than `cap` bytes in all the
// workspaces together are JGPM_E_NOMEM, as where the device has no room.
static int grow(jgpm_ctx_s* c, void*& p, size_t& have, size_t need, size_t cap, hipStream_t st) {
  if (have >= need) return JGPM_OK;
  if (cap != SIZE_MAX && ws_held(c) - have + need > cap) return JGPM_E_NOMEM;
  prof_stale(c);
  if (c->capturing) return JGPM_E_STATE;
  if (p) {
    if (hipStreamSynchronize(st) != hipSuccess) return JGPM_E_HIP;
    (void)hipFree(p);
    p = nullptr;
    have = 0;
  }
  if (hipMalloc(&p, need) != hipSuccess) {
    (void)hipGetLastError();
    return JGPM_E_NOMEM;
  }
  have = need;
  return JGPM_OK;
}

// Hub bitmaps of the triangle launches: the highest-degree vertices whose
// bitmaps fit 16 bytes a directed edge, at least 128 and at most 512 MiB
// (R-MAT 18: its 4,096 widest vertices; twice the bytes cost 0.3 of 7.8 ms for
// P5.  R-MAT 20, 128 / 256 / 512 MiB: 92.5 / 81.4 / 75.4 ms).
static int64_t tri_hub_bytes(int64_t nnz) {
  return std::max<int64_t>((int64_t)128 << 20, std::min<int64_t>((int64_t)512 << 20, 16 * nnz));
}

// Scratch of the triangle launches: the hub bitmaps, the task lists, and what
// the sums keep of a block's root.
static int64_t tri_hwords(int64_t nv) { return ((nv + 31) / 32 + 3) & ~(int64_t)3; }
static int32_t tri_hubs(const jgpm_graph_s* g) {
  return (int32_t)std::min<int64_t>(g->hubs, tri_hub_bytes(g->sym.nnz) / (4 * tri_hwords(g->sym.nv)));
}
static size_t tri_list_bytes(const jgpm_graph_s* g) {
  return (sizeof(int32_t) * 3 * (size_t)g->sym.nv + 15) & ~(size_t)15;
}
static size_t tri_root_bytes(const jgpm_graph_s* g, const jgpm_ctx_s* c) {
  return g->sym.max_deg <= 64 ? 0 : sizeof(int32_t) * 3 * (size_t)std::max(1, g->dag.max_deg) *
                                        (size_t)(jk::TRI_SMALL_PER_CU * c->num_cu);
}

// Arguments of the triangle launches on g, their scratch on the executing
// context (the hub bitmaps still to be made by launch_hub_bitmaps).  build:
// only for the triangle array.
static int tri_args(jgpm_graph_s* g, hipStream_t st, jk::TriArgs& a, bool build = false) {
  jgpm_ctx_s* c = exec_ctx(g);
  const int32_t nv = g->sym.nv;
  a = jk::TriArgs{};
  a.rp = g->sym.rp;
  a.ci = g->sym.ci;
  a.drp = g->dag.rp;
  a.dci = g->dag.ci;
  a.ord = g->d_ord;
  a.dtri = g->d_dtri;
  a.nv = nv;
  a.wide = g->sym.max_deg > 64;
  // a wave works its vertices off one after another: no more per wave than
  // it takes to fill the device (32 waves per CU)
  a.vchunk = std::max(1, std::min(64, nv / (64 * c->num_cu)));
  a.hwords = tri_hwords(nv);
  a.nhub = tri_hubs(g);
  a.lstride = std::max(1, g->dag.max_deg);
  size_t hub_b = 4 * (size_t)a.hwords * (size_t)a.nhub;
  const size_t list_b = tri_list_bytes(g), lscr_b = tri_root_bytes(g, c);
  int rc = grow(c, c->d_te, c->te_bytes, 64 + hub_b + list_b + lscr_b, c->ws_cap, st);
  if (rc == JGPM_E_NOMEM) {  // without bitmaps: every row searched for
    a.nhub = 0;
    hub_b = 0;
    rc = grow(c, c->d_te, c->te_bytes, 64 + list_b + lscr_b, c->ws_cap, st);
    if (rc == JGPM_E_NOMEM && build) rc = grow(c, c->d_te, c->te_bytes, 64 + list_b, c->ws_cap, st);
  }
  if (rc) return rc;
  unsigned char* b = static_cast<unsigned char*>(c->d_te);
  a.ctr = reinterpret_cast<unsigned long long*>(b);
  a.hub = reinterpret_cast<const uint32_t*>(b + 64);
  a.list = reinterpret_cast<int32_t*>(b + 64 + hub_b);
  a.lscr = reinterpret_cast<int32_t*>(b + 64 + hub_b + list_b);
  return JGPM_OK;
}

// Hub rows for a clique launch over the roots [rb, re), made on the stream.
// None where the range holds too few edges to pay for two small launches
// (R-MAT 10, 10,000 edges: TC 23 us without and 26 with; R-MAT 12, 52,000: 66 and
// 38), where there is no room, or while capturing.  As many rows as take no more
// than four words an edge of the range, at least 16,384 (8 MiB at half the
// square), at most 65,536 (R-MAT 22, a quarter of the roots: 0.21 ms for 272
// MB; P13 9.75 ms, with 32,768 rows 10.2); triangle counts, whose streams are
// cheaper, at most 32,768 (TC 7.9 ms, with 65,536 rows 8.7).
int clique_hub_rows(jgpm_graph_s* g, int k, int64_t rb, int64_t re, hipStream_t st, jk::CliqueArgs& a) {
  jgpm_ctx_s* c = exec_ctx(g);
  const int32_t nv = g->dag.nv;
  const int64_t ne = g->dag_rp_h[re] - g->dag_rp_h[rb];
  if (c->capturing || ne < 16384) return JGPM_OK;
  const int32_t cap = std::min(nv, k == 3 ? jk::HUB_TOP_MAX / 2 : jk::HUB_TOP_MAX);
  int32_t top = std::min(cap, 16384);
  while (top < cap && (int64_t)jk::hub_rows_words(std::min(cap, 2 * top)) <= 4 * ne) top = std::min(cap, 2 * top);
  const size_t bits_b = sizeof(uint32_t) * jk::hub_rows_words(top);
  const int rc = grow(c, c->d_hub, c->hub_bytes, bits_b + sizeof(int32_t) * (size_t)top, c->ws_cap, st);
  if (rc == JGPM_E_NOMEM) return JGPM_OK;
  if (rc) return rc;
  uint32_t* bits = static_cast<uint32_t*>(c->d_hub);
  int32_t* inv = reinterpret_cast<int32_t*>(static_cast<unsigned char*>(c->d_hub) + bits_b);
  prof_begin(c, st, "hub_rows");
  const hipError_t e = jk::launch_hub_rows(g->dag.rp, g->dag.ci, g->d_ord, nv, top, inv, bits, c->num_cu, st);
  prof_end(c, st);
  a.hub = bits;
  a.hub_top = top;
  a.nv = nv;
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

// Lazily built per-graph arrays of the symmetric kernels.
static int build_sym_aux(jgpm_graph_s* g, bool need_tri, bool need_nsum, hipStream_t st) {
  jgpm_ctx_s* c = exec_ctx(g);
  const int64_t ne = g->sym.nnz;
  if (!g->d_src) {
    if (hipMalloc(&g->d_src, sizeof(int32_t) * std::max<int64_t>(ne, 1)) != hipSuccess) return JGPM_E_NOMEM;
    g->bytes += 4 * ne;
    if (jk::launch_aux_src(g->sym.rp, g->sym.nv, g->d_src, grid_for(c, 4), st) != hipSuccess) return JGPM_E_HIP;
  }
  if (need_tri && !g->d_tri) {
    const int64_t nd = g->dag.nnz;
    jk::TriArgs a;
    int rc = tri_args(g, st, a, true);
    if (rc) return rc;
    int32_t *tri = nullptr, *dtri = nullptr;
    if (hipMalloc(&tri, sizeof(int32_t) * std::max<int64_t>(ne, 1)) != hipSuccess ||
        hipMalloc(&dtri, sizeof(int32_t) * std::max<int64_t>(nd, 1)) != hipSuccess) {
      if (tri) (void)hipFree(tri);
      return JGPM_E_NOMEM;
    }
    prof_begin(c, st, "edge_triangles");
    hipError_t e = jk::launch_hub_bitmaps(a, c->num_cu, st);
    if (e == hipSuccess) e = jk::launch_tri_build(a, dtri, g->d_src, ne, tri, c->num_cu, st);
    prof_end(c, st);
    if (e != hipSuccess) {
      (void)hipStreamSynchronize(st);
      (void)hipFree(tri);
      (void)hipFree(dtri);
      return JGPM_E_HIP;
    }
    g->d_tri = tri;
    g->d_dtri = dtri;
    g->bytes += 4 * ne + 4 * nd;
  }
  if (need_nsum && !g->d_nsum) {
    if (hipMalloc(&g->d_nsum, sizeof(int64_t) * (g->sym.nv + 1)) != hipSuccess) return JGPM_E_NOMEM;
    g->bytes += 8 * (int64_t)g->sym.nv;
    if (jk::launch_aux_nsum(g->sym.rp, g->sym.ci, g->sym.nv, g->d_nsum, grid_for(c, 4), st) != hipSuccess)
      return JGPM_E_HIP;
  }
  return JGPM_OK;
}

// Makes sure of a graph's lazy arrays.  They are built on the graph's own
// context: its stream orders the build before every later reader there, and
// g->aux_pending says that a reader on another stream has to wait for it.  A
// context that runs a query of another's graph (a serving lane) would publish
// an array that its stream is still filling, so where one is missing it gets
// JGPM_E_NOMEM and does without, like a query that found no room.
int ensure_sym_aux(jgpm_graph_s* g, bool need_tri, bool need_nsum, hipStream_t st) {
  jgpm_ctx_s* c = exec_ctx(g);
  if (g->d_src && (!need_tri || g->d_tri) && (!need_nsum || g->d_nsum)) return JGPM_OK;
  if (c != g->ctx) return JGPM_E_NOMEM;
  prof_stale(c);
  g->aux_pending = true;
  return build_sym_aux(g, need_tri, need_nsum, st);
}

bool pattern_uses_tri(int p) { return p == 3 || p == 4 || p == 7 || p == 10 || p == 11; }

// Words of the widest root's rows among those that do not fit LDS (0: none):
// a slice of the row scratch per block.
static int64_t widest_rows(jgpm_graph_s* g) {
  if (g->tri_rows < 0) {
    g->tri_rows = 0;
    if (jk::tri_rows_global(g->sym.max_deg, g->dag.max_deg))
      for (int32_t v = 0; v < g->sym.nv; ++v) {
        const int64_t d = g->sym_rp_h[v + 1] - g->sym_rp_h[v], dp = g->dag_rp_h[v + 1] - g->dag_rp_h[v];
        if (jk::tri_rows_global(d, dp)) g->tri_rows = std::max(g->tri_rows, jk::tri_row_words(d, dp));
      }
  }
  return g->tri_rows;
}

// given: arguments the caller has already (a second tri_args could move the
// scratch that they point to).
static int enqueue_tri_sum(jgpm_graph_s* g, int p, int64_t rb, int64_t re, int slot, hipStream_t st,
                           const jk::TriArgs* given = nullptr) {
  jgpm_ctx_s* c = exec_ctx(g);
  if (g->dag.max_deg > jk::TRI_MAX_OUT) return JGPM_E_NOMEM;  // per edge
  int rc = ensure_sym_aux(g, true, false, st);
  if (rc) return rc;
  jk::TriArgs a;
  if (given) a = *given;
  else if ((rc = tri_args(g, st, a))) return rc;
  a.rb = rb;
  a.re = re;
  a.out = c->d_out + slot;
  int gblocks = 0;
  if (widest_rows(g) > 0) {
    a.rstride = g->tri_rows;
    const int64_t room = (int64_t)(ws_room(c, sizeof(uint64_t) * c->scr_words) / sizeof(uint64_t)) / a.rstride;
    if (room < 1) return JGPM_E_NOMEM;
    gblocks = (int)std::min(room, std::max<int64_t>(1, std::min<int64_t>(c->num_cu, ((int64_t)1 << 27) / a.rstride)));  // 1 GiB
    if ((rc = ensure_scratch(c, (size_t)a.rstride * (size_t)gblocks))) return rc;
    a.rows = c->d_scr;
  }
  static const char* const kName[13] = {"", "", "", "", "sym_p4_tri", "sym_p5_tri", "", "sym_p7_tri", "", "sym_p9_tri",
                                        "sym_p10_tri", "sym_p11_tri", "sym_p12_tri"};
  prof_begin(c, st, kName[p]);
  hipError_t e = jk::launch_hub_bitmaps(a, c->num_cu, st);
  if (e == hipSuccess) e = jk::launch_tri_sum(p, a, c->num_cu, gblocks, st);
  prof_end(c, st);
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

// An array of n entries that `launch` fills on the device, to the host (through
// the triangle launches' scratch).
template <class T, class F>
static int device_array(jgpm_ctx_s* c, size_t n, hipStream_t st, std::vector<T>& h, F launch) {
  const int rc = grow(c, c->d_te, c->te_bytes, sizeof(T) * std::max<size_t>(n, 1), SIZE_MAX, st);
  if (rc) return rc;
  try {
    h.resize(n);
  } catch (const std::bad_alloc&) {
    return JGPM_E_NOMEM;
  }
  const bool ok = launch(static_cast<T*>(c->d_te)) == hipSuccess &&
                  hipMemcpyAsync(h.data(), c->d_te, sizeof(T) * n, hipMemcpyDeviceToHost, st) == hipSuccess;
  return hipStreamSynchronize(st) == hipSuccess && ok ? JGPM_OK : JGPM_E_HIP;
}

int ensure_tri_prefix(jgpm_graph_s* g, hipStream_t st) {
  if (!g->tri_pre_h.empty()) return JGPM_OK;
  jgpm_ctx_s* c = exec_ctx(g);
  if (c != g->ctx) return JGPM_E_NOMEM;  // as in ensure_sym_aux
  if (c->capturing) return JGPM_E_STATE;
  int rc = ensure_sym_aux(g, true, false, st);
  if (rc) return rc;
  prof_stale(c);
  const int32_t nv = g->sym.nv;
  std::vector<int64_t> sum;
  rc = device_array(c, (size_t)nv, st, sum,
                    [&](int64_t* d) { return jk::launch_root_tri(g->sym.rp, g->d_tri, nv, d, c->num_cu, st); });
  if (rc) return rc;
  try {
    sum.push_back(0);
  } catch (const std::bad_alloc&) {
    return JGPM_E_NOMEM;
  }
  int64_t most = 0, run = 0;
  for (int32_t v = 0; v <= nv; ++v) {
    const int64_t x = sum[v];
    most = std::max(most, x);
    sum[v] = run;
    run += x;
  }
  g->tri_max = most;
  g->tri_pre_h.swap(sum);
  return JGPM_OK;
}

int ensure_edge_work(jgpm_graph_s* g, hipStream_t st) {
  if (!g->work_pre_h.empty()) return JGPM_OK;
  jgpm_ctx_s* c = exec_ctx(g);
  if (c != g->ctx) return JGPM_E_NOMEM;  // as in ensure_sym_aux
  if (c->capturing) return JGPM_E_STATE;
  int rc = ensure_sym_aux(g, true, false, st);
  if (rc) return rc;
  prof_stale(c);
  const int32_t nv = g->sym.nv;
  (void)widest_rows(g);  // while the device builds the triangle array
  const int64_t nb = jk::edge_work_blocks(nv);
  std::vector<float4> work;
  jk::TriArgs a{};
  a.rp = g->sym.rp;
  a.ci = g->sym.ci;
  a.drp = g->dag.rp;
  a.nv = nv;
  rc = device_array(c, (size_t)nb, st, work,
                    [&](float4* d) { return jk::launch_edge_work(a, g->d_src, g->d_tri, d, st); });
  if (rc) return rc;
  std::vector<jgpm_graph_s::EdgeWork> pre;
  try {
    pre.resize((size_t)nb + 1);
  } catch (const std::bad_alloc&) {
    return JGPM_E_NOMEM;
  }
  double pass = 0;
  pre[0] = {0, 0, 0};
  for (int64_t k = 0; k < nb; ++k) {
    pre[k + 1] = {pre[k].lo_a + work[k].x, pre[k].lo_b + work[k].y, pre[k].hi_b + work[k].z};
    pass += work[k].w;
  }
  // measured: R-MAT 12 / 14 / 16 / 18: P9 0.13 / 0.32 / 1.27 / 6.5 ms, P5 - / 0.38 / 1.57 / 7.8; Barabasi-Albert
  // (60,000 vertices, 12 a vertex) 0.30, 0.32; Erdos-Renyi (32,768, degree 40) 0.34, 0.34; Chung-Lu (200,000) 0.49, 0.53
  g->tri_pass_a = 100e3 + 0.8 * nv + 0.08 * (double)g->sym.nnz + pass;
  g->tri_pass_b = 150e3 + 1.1 * nv + 1.25 * pass;
  g->work_pre_h.swap(pre);
  return JGPM_OK;
}

// Whether P4, P5, P7, P9, P11 or P12 over a root range runs over all triangles
// of the graph (the terms of other roots left out) or per edge of the range.
// The pass takes the same time whatever the range; the per-edge launches take
// 1.45 ns for each edge of the range and, for the edges that the pattern
// credits to the range (P9, P11, P12 to the smaller end, P5 and P4 to the
// larger, P7 to both) and that lie in t > 0 triangles, what k_edge_work adds
// up: R-MAT ids fall with the degree, so the last eighth of the edges of R-MAT 18 takes P9
// 1.6 ms per edge (6.5 over triangles), the first eighth 64.  P4 per edge waits
// for one intersection after the other at an edge to a hub, about 3 us each.
// Over ranges of 1/2 to 1/2048 of the edges at both ends and in the middle, on
// those graphs, the route taken was at most 1.23 times slower than per edge
// (P4 1.33 at 0.08 ms), and than the better one 2 times (a range of R-MAT 12's
// first roots 2.8: 0.35 and 0.13 ms).  A share of the edges as the line (1/8 for P9, P11, P12, 1/32 for P5,
// P7, 1/1024 for P4) was up to 4.7, 3.9 and 16 times slower than per edge.
static int over_triangles(jgpm_graph_s* g, int p, int64_t rb, int64_t re, hipStream_t st, bool& yes) {
  const int64_t ne = g->sym_rp_h[re] - g->sym_rp_h[rb];
  yes = ne == g->sym.nnz;
  if (yes) return JGPM_OK;
  // not worth the triangle array if nothing has built it yet
  if (!g->d_tri && !edge_route_needs_tri(exec_ctx(g), p) && ne < g->sym.nnz / 64) return JGPM_OK;
  const int rc = ensure_edge_work(g, st);
  if (rc) return rc;
  // the prefix at a vertex: of its block's work the share of its edges
  const int64_t *rp = g->sym_rp_h.data(), nv = g->sym.nv, B = jk::EDGE_WORK_BLOCK;
  auto at = [&](int64_t v) {
    const int64_t k = std::min(v / B, (int64_t)g->work_pre_h.size() - 2);
    const int64_t e0 = rp[k * B], e1 = rp[std::min(nv, (k + 1) * B)];
    const double f = e1 > e0 ? (double)(rp[v] - e0) / (double)(e1 - e0) : 0.0;
    const jgpm_graph_s::EdgeWork &x = g->work_pre_h[k], &y = g->work_pre_h[k + 1];
    return jgpm_graph_s::EdgeWork{x.lo_a + f * (y.lo_a - x.lo_a), x.lo_b + f * (y.lo_b - x.lo_b),
                                  x.hi_b + f * (y.hi_b - x.hi_b)};
  };
  const jgpm_graph_s::EdgeWork x = at(rb), y = at(re);
  const double lo_a = y.lo_a - x.lo_a, lo_b = y.lo_b - x.lo_b;
  const double hi_b = re > 1 ? y.hi_b - x.hi_b : 0;  // (vertex 0 has no smaller neighbour)
  const double base = 120e3 + 1.45 * (double)ne;
  switch (p) {
    case 4:
      yes = 75e3 + (hi_b > 0 ? 3e3 * g->sym.max_deg : 0.0) + 1.7 * (double)ne > g->tri_pass_b + 100e3;
      break;
    case 5: yes = base + hi_b > g->tri_pass_b; break;
    case 7: yes = base + lo_b + hi_b > g->tri_pass_b; break;
    case 9: yes = base + lo_a > g->tri_pass_a; break;
    case 11: yes = base + lo_a > g->tri_pass_b; break;
    case 12: yes = base + lo_b > g->tri_pass_b; break;
  }
  return JGPM_OK;
}

// P6, P8 and P10 count wedges on the graph of induced neighbourhoods, which
// has a vertex per directed edge of the roots and 2 t entries per edge.  It is
// built per query, for as many roots at a time as EGO_CAP entries hold.
constexpr int64_t EGO_CAP = (int64_t)1 << 28;
// Workspace bytes for an entry and an edge: 28 and 4 of the wedge launches, 8
// and 8 of the graph, and some to spare.
constexpr size_t EGO_ENTRY_BYTES = 64;

// Whether the range runs on the induced neighbourhoods: every root fits the
// cap, for P10, whose triangle part covers all triangles, the range is not a
// sliver of the graph, and there are triangles enough to pay for the launches
// (Erdos-Renyi, 1,000 vertices, 640 triangles: P8 114 us per edge, 194 on the
// induced graph; Barabasi-Albert, 1,000 vertices: 1,040 and 221; R-MAT 12
// 384,000 and 357).
static bool ego_route(jgpm_graph_s* g, int p, int64_t rb, int64_t re) {
  if (p != 6 && p != 8 && p != 10) return false;
  const int64_t ne = g->sym_rp_h[re] - g->sym_rp_h[rb];
  if (g->tri_pre_h[re] - g->tri_pre_h[rb] < 16384 && g->tri_max < 256) return false;
  return g->tri_max <= EGO_CAP && g->sym.max_deg < EGO_CAP && (p != 10 || ne >= g->sym.nnz / 1024);
}

static int enqueue_ego(jgpm_graph_s* g, int p, int64_t rb, int64_t re, int slot, hipStream_t st) {
  jgpm_ctx_s* c = exec_ctx(g);
  uint64_t* const out = c->d_out + slot;
  const int64_t *rp = g->sym_rp_h.data(), *pre = g->tri_pre_h.data();
  // chunks of whole roots, and the scratch of the largest
  const size_t tri_b = std::max(c->te_bytes, 64 + tri_list_bytes(g) + tri_root_bytes(g, c)) +
                       (p == 10 ? sizeof(uint64_t) * (size_t)widest_rows(g) : 0);
  const size_t room = ws_room(c, c->te_bytes + c->ego_bytes + c->p1_bytes);
  const int64_t cap = std::min<int64_t>(EGO_CAP, (int64_t)((room > tri_b ? room - tri_b : 0) / EGO_ENTRY_BYTES));
  if (cap < 1) return JGPM_E_NOMEM;
  std::vector<int64_t> cut{rb};
  int64_t most_e = 0, most_n = 0;
  for (int64_t r = rb; r < re;) {
    int64_t r2 = std::upper_bound(pre + r + 1, pre + re + 1, pre[r] + cap) - pre - 1;
    r2 = std::min(r2, (int64_t)(std::upper_bound(rp + r + 1, rp + re + 1, rp[r] + cap) - rp - 1));
    r2 = std::max(r2, r + 1);
    most_e = std::max(most_e, pre[r2] - pre[r]);
    most_n = std::max(most_n, rp[r2] - rp[r]);
    cut.push_back(r = r2);
  }
  const size_t rp_b = sizeof(int64_t) * (size_t)(most_n + 1), tiles_b = sizeof(int64_t) * (size_t)jk::ego_tiles(most_n);
  const size_t ent_b = sizeof(int32_t) * (size_t)most_e;
  int rc = grow(c, c->d_ego, c->ego_bytes, rp_b + tiles_b + 2 * ent_b + 64, c->ws_cap, st);
  if (!rc) rc = ensure_p1_scratch(c, jk::p1_scratch_bytes(most_n, most_e), c->ws_cap, st);
  jk::TriArgs ta;
  if (!rc) rc = tri_args(g, st, ta);
  if (!rc && p == 10) rc = enqueue_tri_sum(g, 10, rb, re, slot, st, &ta);
  if (rc) return rc;  // (nothing is launched when there was no room)
  static const char* const kName[11] = {"", "", "", "", "", "", "sym_p6_wedge", "", "sym_p8_wedge", "", "sym_p10_wedge"};
  prof_begin(c, st, kName[p]);
  hipError_t e = jk::launch_hub_bitmaps(ta, c->num_cu, st);
  for (size_t k = 0; k + 1 < cut.size() && e == hipSuccess; ++k) {
    jk::EgoArgs ea{};
    ea.src = g->d_src;
    ea.tri = g->d_tri;
    ea.e0 = rp[cut[k]];
    ea.n = rp[cut[k + 1]] - ea.e0;
    const int64_t ents = pre[cut[k + 1]] - pre[cut[k]];
    if (ents == 0) continue;
    unsigned char* b = static_cast<unsigned char*>(c->d_ego);
    ea.rp = reinterpret_cast<int64_t*>(b);
    ea.tiles = reinterpret_cast<int64_t*>(b + rp_b);
    ea.ci = reinterpret_cast<int32_t*>(b + rp_b + tiles_b);
    ea.row = reinterpret_cast<int32_t*>(b + rp_b + tiles_b + ent_b);
    e = jk::launch_ego_build(ta, ea, c->num_cu, st);
    jk::P1Args a{};
    a.one.rp = ea.rp;
    a.one.ci = ea.ci;
    a.one.src = ea.row;
    a.one.ne = ents;
    a.one.nr = ea.n;
    a.one.slot = slot;
    a.one.csrc = g->d_src + ea.e0;
    a.one.crp = g->sym.rp;
    a.one.cbase = ea.e0;
    if (p == 6) {
      a.one.vid = g->sym.ci + ea.e0;
      a.one.lrp = g->sym.rp;
      a.one.lci = g->sym.ci;
      a.one.xend = g->sym.nv;
    }
    if (p == 10) a.one.scale = -4;
    a.nq = 1;
    a.tiles = (ents + 255) / 256;
    a.roots = ea.n;
    a.edges = ents;
    a.out = c->d_out;
    jk::p1_bind_scratch(a, c->d_p1);
    if (e == hipSuccess) e = jk::launch_wedge(p == 6 ? jk::WEDGE_P6 : jk::WEDGE_P1, a, c->num_cu, st);
    if (e == hipSuccess && p == 10) e = jk::launch_p10_rows(ea, out, c->num_cu, st);
    if (e == hipSuccess && p == 6)
      e = jk::launch_edge_base(g->sym.rp, g->sym.ci, g->d_src, g->d_tri, ea.e0, ea.e0 + ea.n, 2, out, c->num_cu, st);
  }
  prof_end(c, st);
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

static int enqueue_p4(jgpm_graph_s* g, int64_t rb, int64_t re, int slot, hipStream_t st) {
  jgpm_ctx_s* c = exec_ctx(g);
  int rc = ensure_sym_aux(g, true, false, st);
  if (rc) return rc;
  const bool whole = rb == 0 && re == g->sym.nv;
  const int64_t e0 = g->sym_rp_h[rb], e1 = g->sym_rp_h[re];
  jk::P1Args a{};
  a.one.rp = g->sym.rp;
  a.one.ci = g->sym.ci;
  a.one.src = g->d_src;
  a.one.e0 = e0;
  a.one.ne = e1 - e0;
  a.one.rb = rb;
  a.one.nr = re - rb;
  a.one.slot = slot;
  a.one.weight = g->d_tri;
  a.one.xend = g->sym.nv;
  a.nq = 1;
  a.tiles = (a.one.ne + 255) / 256;
  a.roots = a.one.nr;
  a.edges = a.one.ne;
  a.out = c->d_out;
  if ((rc = ensure_p1_scratch(c, jk::p1_scratch_bytes(a.roots, a.edges), c->ws_cap, st))) return rc;
  if (!whole && (rc = enqueue_tri_sum(g, 4, rb, re, slot, st))) return rc;  // (nothing is launched when there was no room)
  jk::p1_bind_scratch(a, c->d_p1);
  prof_begin(c, st, "sym_p4_wedge");
  hipError_t e = jk::launch_wedge(jk::WEDGE_P4, a, c->num_cu, st);
  if (e == hipSuccess)
    e = jk::launch_edge_base(g->sym.rp, g->sym.ci, g->d_src, g->d_tri, e0, e1, whole ? 1 : 0, c->d_out + slot, c->num_cu,
                             st);
  prof_end(c, st);
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

// The per-edge launches of P5, P7, P9, P11 and P12 read the triangle array
// to send their heavy edges to the block-per-edge kernel.
static bool heavy_split_on(const jgpm_ctx_s* c, int p) {
  return jk::sym_heavy_pattern(p) && c->tune.sym_heavy_min < jk::sym_heavy_nmax();
}

bool edge_route_needs_tri(const jgpm_ctx_s* c, int p) {
  return p == 2 || pattern_uses_tri(p) || heavy_split_on(c, p);
}

int ensure_p1_scratch(jgpm_ctx_s* c, size_t bytes, size_t cap, hipStream_t st) {
  return grow(c, c->d_p1, c->p1_bytes, bytes, cap, st);
}

int p1_query(jgpm_graph_s* g, int64_t rb, int64_t re, hipStream_t st, jk::P1Q& q) {
  q = jk::P1Q{};
  // a whole-graph count runs on the degree-ordered relabelling: the same
  // identity in another vertex order gives the same total, and the hubs,
  // ranked last, are no wedge's middle vertex
  const bool whole = rb == 0 && re == g->sym.nv;
  int rc = whole ? ensure_rank_csr(g, st) : ensure_sym_aux(g, false, false, st);
  if (rc) return rc;
  q.rp = whole ? g->rsym.rp : g->sym.rp;
  q.ci = whole ? g->rsym.ci : g->sym.ci;
  q.src = whole ? g->d_rsrc : g->d_src;
  q.e0 = whole ? 0 : g->sym_rp_h[rb];
  q.ne = whole ? g->sym.nnz : g->sym_rp_h[re] - q.e0;
  q.rb = rb;
  q.nr = re - rb;
  q.xmin = whole ? g->rank_min2 : 0;
  return JGPM_OK;
}

static int enqueue_p1(jgpm_graph_s* g, int64_t rb, int64_t re, int slot, hipStream_t st) {
  if (re <= rb) return JGPM_OK;
  jgpm_ctx_s* c = exec_ctx(g);
  jk::P1Args a{};
  int rc = p1_query(g, rb, re, st, a.one);
  if (rc) return rc;
  a.one.slot = slot;
  a.nq = 1;
  a.tiles = (a.one.ne + 255) / 256;
  a.roots = a.one.nr;
  a.edges = a.one.ne;
  a.out = c->d_out;
  if ((rc = ensure_p1_scratch(c, jk::p1_scratch_bytes(a.roots, a.edges), SIZE_MAX, st))) return rc;
  jk::p1_bind_scratch(a, c->d_p1);
  prof_begin(c, st, "sym_p1_wedge");
  hipError_t e = jk::launch_wedge(jk::WEDGE_P1, a, c->num_cu, st);
  prof_end(c, st);
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

int enqueue_sym(jgpm_graph_s* g, int p, int64_t rb, int64_t re, int slot, hipStream_t st) {
  if (!g->has_sym) return JGPM_E_GRAPHKIND;
  jgpm_ctx_s* c = exec_ctx(g);
  if (p == 1) return enqueue_p1(g, rb, re, slot, st);
  if (p == 2) {
    // diamonds from the per-edge triangle array, which every later diamond,
    // P3 or induced-motif query on the graph then only reads
    int rc = ensure_sym_aux(g, true, false, st);
    if (rc) return rc;
    const int64_t e0 = g->sym_rp_h[rb], e1 = g->sym_rp_h[re];
    if (e1 <= e0) return JGPM_OK;
    const int64_t quads = (e1 - e0 + 3) / 4;
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((int64_t)8 * c->num_cu, (quads + 255) / 256));
    prof_begin(c, st, "sym_p2");
    hipError_t e = jk::launch_p2_edges(g->d_src, g->sym.ci, g->d_tri, e0, e1, (unsigned long long*)(c->d_out + slot),
                                       grid, st);
    prof_end(c, st);
    return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
  }
  if (p == 3) {
    int rc = ensure_sym_aux(g, true, true, st);
    if (rc) return rc;
    prof_begin(c, st, "sym_p3");
    hipError_t e = jk::launch_edge_sum(true, g->sym.rp, g->sym.ci, g->d_src, g->d_tri, g->d_nsum, g->sym_rp_h[rb],
                                       g->sym_rp_h[re], c->d_q64 + slot, c->d_out + slot, c->num_cu, st);
    prof_end(c, st);
    return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
  }
  // patterns that run over triangles or wedges of the whole range; where
  // there is no room for their scratch (nothing launched), per edge
  if (g->sym_rp_h[re] > g->sym_rp_h[rb]) {
    int rr = JGPM_E_NOMEM;
    if (p == 4 || jk::sym_heavy_pattern(p)) {
      bool yes = false;
      rr = over_triangles(g, p, rb, re, st, yes);
      if (!rr) rr = !yes ? JGPM_E_NOMEM : p == 4 ? enqueue_p4(g, rb, re, slot, st) : enqueue_tri_sum(g, p, rb, re, slot, st);
    } else if (p == 6 || p == 8 || p == 10) {
      rr = ensure_tri_prefix(g, st);
      if (!rr) rr = ego_route(g, p, rb, re) ? enqueue_ego(g, p, rb, re, slot, st) : JGPM_E_NOMEM;
    }
    if (rr != JGPM_E_NOMEM) return rr;
    (void)hipGetLastError();
  }
  int rc = ensure_sym_aux(g, edge_route_needs_tri(c, p), false, st);
  if (rc) return rc;
  const int wpb = jk::sym_waves_per_block();
  const int grid = grid_for(c, 2);
  const size_t stride = (size_t)std::max(1, g->sym_mmin);
  const size_t need = (size_t)grid * wpb * jk::sym_lists_per_wave() * stride;
  // the heavy-edge split needs its three edge lists, each as long as the
  // range's edge count up to 2^26 (grown per context, so not while a launch
  // sequence is being captured; edges beyond a full list run in the
  // wave-per-edge launch), and edge indices of a range that fit 32 bits
  const int64_t ne_r = g->sym_rp_h[re] - g->sym_rp_h[rb];
  bool heavy = heavy_split_on(c, p) && ne_r < INT32_MAX;
  const int64_t hwant = std::min<int64_t>(std::max<int64_t>(ne_r, 1), (int64_t)1 << 26);
  // a capped context gives back what another route took before it found no room
  if (c->ws_cap != SIZE_MAX) {
    const size_t want = sizeof(int32_t) * (std::max(need, c->sscr_ints) + (heavy ? 3 * (size_t)std::max(hwant, c->hcap) : 0));
    if (ws_held(c) - sizeof(int32_t) * (c->sscr_ints + 3 * (size_t)c->hcap) + want > c->ws_cap) {
      if (hipStreamSynchronize(st) != hipSuccess) return JGPM_E_HIP;
      ws_release(c);
    }
  }
  if (heavy && c->hcap < hwant) {
    if (c->capturing) {
      heavy = c->d_hlist != nullptr;  // the lists it has
    } else {
      if (c->d_hlist) {
        if (hipStreamSynchronize(st) != hipSuccess) return JGPM_E_HIP;
        (void)hipFree(c->d_hlist);
        c->d_hlist = nullptr;
        c->hcap = 0;
      }
      if (hipMalloc(&c->d_hlist, sizeof(int32_t) * 3 * (size_t)hwant) != hipSuccess) return JGPM_E_NOMEM;
      c->hcap = hwant;
      if (!c->d_hctr && hipMalloc(&c->d_hctr, sizeof(unsigned long long) * 6) != hipSuccess) return JGPM_E_NOMEM;
    }
  }
  if (c->sscr_ints < need) {
    if (c->d_sscr) {
      if (hipStreamSynchronize(st) != hipSuccess) return JGPM_E_HIP;
      (void)hipFree(c->d_sscr);
      c->d_sscr = nullptr;
      c->sscr_ints = 0;
    }
    if (hipMalloc(&c->d_sscr, need * sizeof(int32_t)) != hipSuccess) return JGPM_E_NOMEM;
    c->sscr_ints = need;
  }
  jk::SymArgs a{};
  a.rp = g->sym.rp;
  a.ci = g->sym.ci;
  a.src = g->d_src;
  a.tri = g->d_tri;
  a.nsum = g->d_nsum;
  a.e0 = g->sym_rp_h[rb];
  a.ne = g->sym_rp_h[re] - a.e0;
  if (a.ne <= 0) return JGPM_OK;
  a.qctr = c->d_q64 + (slot % (CTX_SLOTS - 1));
  a.chunk = 8;
  a.scr = c->d_sscr;
  a.scr_stride = (int64_t)stride;
  a.out = c->d_out + slot;
  a.heavy_min = heavy ? c->tune.sym_heavy_min : 0;
  a.heavy_stream = jk::sym_heavy_stream();
  a.nv = g->sym.nv;
  a.hlist = c->d_hlist;
  a.hctr = c->d_hctr;
  a.hcap = (int32_t)c->hcap;
  a.heavy_mid = heavy ? jk::sym_heavy_mid(p) : 0;
  // list counters to zero (a kernel, so the sequence can be captured)
  if (heavy && zero_u64(reinterpret_cast<uint64_t*>(c->d_hctr), 6, st)) return JGPM_E_HIP;
  static const char* const kSymName[13] = {"", "", "", "", "sym_p4", "sym_p5", "sym_p6",
                                           "sym_p7", "sym_p8", "sym_p9", "sym_p10", "sym_p11", "sym_p12"};
  prof_begin(c, st, kSymName[p]);
  hipError_t e = jk::launch_sym(p, a, grid, st);
  prof_end(c, st);
  if (e != hipSuccess) return JGPM_E_HIP;
  if (heavy) {
    // the edges the wave-per-edge launch listed, in three shapes: |S| up to
    // sym_heavy_mid(p) with a small LDS table and several blocks per CU,
    // up to sym_heavy_nmax() one block per CU, wider ones (graphs of at
    // most 2^20 vertices) with S in the list scratch, one slice per block
    static const char* const kHeavyName[13] = {"", "", "", "", "", "sym_p5_heavy", "", "sym_p7_heavy", "",
                                               "sym_p9_heavy", "", "sym_p11_heavy", "sym_p12_heavy"};
    const int shapes = g->sym.nv <= (1 << 20) ? 3 : 2;
    for (int shape = 0; shape < shapes && e == hipSuccess; ++shape) {
      prof_begin(c, st, kHeavyName[p]);
      e = jk::launch_sym_heavy(p, a, shape, shape ? c->num_cu : 4 * c->num_cu, st);
      prof_end(c, st);
    }
  }
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

int enqueue_vertex_sum(jgpm_graph_s* g, int mode, int64_t rb, int64_t re, int slot, hipStream_t st) {
  if (!g->has_sym) return JGPM_E_GRAPHKIND;
  int rc = ensure_sym_aux(g, mode == 1, false, st);
  if (rc) return rc;
  if (re <= rb) return JGPM_OK;
  jgpm_ctx_s* c = exec_ctx(g);
  prof_stale(c);
  const hipError_t e =
      mode == 0 ? jk::launch_star3(g->sym.rp, rb, re, (unsigned long long*)(c->d_out + slot), grid_for(c, 4), st)
                : jk::launch_edge_sum(false, g->sym.rp, g->sym.ci, g->d_src, g->d_tri, nullptr, g->sym_rp_h[rb],
                                      g->sym_rp_h[re], c->d_q64 + slot, c->d_out + slot, c->num_cu, st);
  return e == hipSuccess ? JGPM_OK : JGPM_E_HIP;
}

// Induced 4-vertex motifs from non-induced counts (exact inverse of the
// conversion matrix): with S = 3-star, T = tailed triangle, C = 4-cycle (P1),
// D = diamond (P2), K = K4 (P13):
//   I_K = K, I_D = D - 6K, I_C = C - D + 3K, I_T = T - 4D + 12K,
//   I_S = S - T + 2D - 4K.
int pattern_slots(int pattern) {
  switch (pattern) {
    case JGPM_I_DIAMOND: return 2;
    case JGPM_I_C4: case JGPM_I_TAILTRI: return 3;
    case JGPM_I_STAR3: return 4;
  }
  return 1;
}

int enqueue_pattern(jgpm_graph_s* g, int pattern, int64_t rb, int64_t re, int s, hipStream_t st) {
  int k = clique_k(pattern);
  if (k) {
    if (!g->has_dag) return JGPM_E_GRAPHKIND;
    return enqueue_clique(g, k, false, rb, re, s, st);
  }
  if (pattern >= JGPM_P1 && pattern <= JGPM_P12) return enqueue_sym(g, pattern, rb, re, s, st);
  if (!g->has_sym) return JGPM_E_GRAPHKIND;
  int rc = JGPM_OK;
  switch (pattern) {
    case JGPM_STAR3: return enqueue_vertex_sum(g, 0, rb, re, s, st);
    case JGPM_TAILTRI: return enqueue_vertex_sum(g, 1, rb, re, s, st);
    case JGPM_I_DIAMOND:
      if ((rc = enqueue_sym(g, JGPM_P2, rb, re, s, st))) return rc;
      return enqueue_clique(g, 4, false, rb, re, s + 1, st);
    case JGPM_I_C4:
      if ((rc = enqueue_sym(g, JGPM_P1, rb, re, s, st))) return rc;
      if ((rc = enqueue_sym(g, JGPM_P2, rb, re, s + 1, st))) return rc;
      return enqueue_clique(g, 4, false, rb, re, s + 2, st);
    case JGPM_I_TAILTRI:
      if ((rc = enqueue_vertex_sum(g, 1, rb, re, s, st))) return rc;
      if ((rc = enqueue_sym(g, JGPM_P2, rb, re, s + 1, st))) return rc;
      return enqueue_clique(g, 4, false, rb, re, s + 2, st);
    case JGPM_I_STAR3:
      if ((rc = enqueue_vertex_sum(g, 0, rb, re, s, st))) return rc;
      if ((rc = enqueue_vertex_sum(g, 1, rb, re, s + 1, st))) return rc;
      if ((rc = enqueue_sym(g, JGPM_P2, rb, re, s + 2, st))) return rc;
      return enqueue_clique(g, 4, false, rb, re, s + 3, st);
  }
  return JGPM_E_PATTERN;
}

int64_t query_array_bytes(const jgpm_graph_s* g, const jgpm_ctx_s* c, int p, int64_t rb, int64_t re) {
  if (clique_k(p)) return 0;
  const int64_t nv = g->sym.nv, nnz = g->sym.nnz;
  int64_t b = g->d_src ? 0 : 4 * nnz;
  // P1: the relabelled graph, and the two key arrays that it is sorted in
  if (p == JGPM_P1) return rb == 0 && re == nv && !g->rsym.ci ? b + 24 * nv + 24 * nnz : b;
  if (!g->d_tri) b += 4 * nnz + 4 * g->dag.nnz + (int64_t)(64 + tri_list_bytes(g) + tri_root_bytes(g, c)) +
                      4 * tri_hwords(nv) * tri_hubs(g);
  if (p == JGPM_P3 && !g->d_nsum) b += 8 * nv;
  return b;
}

int64_t query_ws_bytes(const jgpm_graph_s* g, const jgpm_ctx_s* c, int p, int64_t rb, int64_t re, int64_t most) {
  if (const int k = clique_k(p)) {
    // row scratch of the widest tiers: slices of the fused 2048-wide kernel,
    // for 5- to 7-cliques the row slots of the split one (<= 1 GiB); those of
    // the split 1024-wide one.  The tiers use one buffer after the other.
    int64_t b = 0;
    if (g->dag.max_deg > jk::tier_max_deg(jk::TIER_LDS16)) {
      const int64_t fused = (int64_t)4 * c->num_cu * (int64_t)jk::tier_scratch_words(jk::TIER_GLB32) * 8;
      b = k >= 5 ? std::max<int64_t>(fused, (int64_t)1 << 30) : fused;
    }
    if (k >= 4)
      b = std::max<int64_t>(b, std::min<int64_t>((int64_t)1 << 30,
                                                 8 * (int64_t)jk::split_slot_words() * (int64_t)g->tier_h[jk::TIER_LDS16].size()));
    return b;
  }
  const bool whole = rb == 0 && re == g->sym.nv;
  const int64_t ne = g->sym_rp_h[re] - g->sym_rp_h[rb];
  const int64_t wedge = (int64_t)jk::p1_scratch_bytes(re - rb, ne);
  if (p == JGPM_P1) return wedge;
  if (p == JGPM_P2 || p == JGPM_P3) return 0;
  const int64_t tri = (int64_t)(64 + tri_list_bytes(g) + tri_root_bytes(g, c));
  const int64_t rows = jk::tri_rows_global(g->sym.max_deg, g->dag.max_deg)
                           ? 8 * jk::tri_row_words(g->sym.max_deg, g->dag.max_deg) : 0;
  // per edge: list scratch of every wave, and the heavy-edge lists
  int64_t edge = (int64_t)grid_for(const_cast<jgpm_ctx_s*>(c), 2) * jk::sym_waves_per_block() *
                 jk::sym_lists_per_wave() * std::max(1, g->sym_mmin) * 4;
  if (jk::sym_heavy_pattern(p)) edge += 12 * std::min<int64_t>(ne, (int64_t)1 << 26);
  int64_t b = p == JGPM_P4 ? wedge + (whole ? 0 : tri + rows)
              : jk::sym_heavy_pattern(p) ? tri + rows
                                         : tri + (p == JGPM_P10 ? rows : 0) + ((int64_t)EGO_ENTRY_BYTES << 18);
  if (b > most) return edge;
  // (a part of a graph, and one with few triangles, may run per edge)
  return whole && p != JGPM_P6 && p != JGPM_P8 && p != JGPM_P10 ? b : std::max(b, edge);
}

int prepare_pattern(jgpm_graph_s* g, int pattern, int64_t rb, int64_t re) {
  jgpm_ctx_s* c = g->ctx;
  std::lock_guard<std::mutex> lk(c->mu);
  if (hipSetDevice(c->dev) != hipSuccess) return JGPM_E_HIP;
  ExecScope own(c);
  prof_reset(c, nullptr);
  int rc = JGPM_OK;
  if (clique_k(pattern)) {
    if (g->has_dag) rc = ensure_huge_ids(g);
  } else if (pattern == JGPM_P1) {
    jk::P1Q q;
    if (g->has_sym && re > rb) rc = p1_query(g, rb, re, c->st, q);
  } else if (pattern >= JGPM_P2 && pattern <= JGPM_P12) {
    // every one of them reads the triangle array on one of its routes; what
    // there is no room for is left out where the per-edge launches do without
    if (g->has_sym) {
      rc = ensure_sym_aux(g, true, pattern == JGPM_P3, c->st);
      if (!rc && (pattern == JGPM_P6 || pattern == JGPM_P8 || pattern == JGPM_P10)) rc = ensure_tri_prefix(g, c->st);
      if (!rc && (pattern == JGPM_P4 || jk::sym_heavy_pattern(pattern)) && (rb > 0 || re < g->sym.nv))
        rc = ensure_edge_work(g, c->st);
      if (rc == JGPM_E_NOMEM && (g->d_tri || !edge_route_needs_tri(c, pattern))) {
        (void)hipGetLastError();
        rc = ensure_sym_aux(g, false, pattern == JGPM_P3, c->st);
      }
    }
  }
  if (hipStreamSynchronize(c->st) == hipSuccess) g->aux_pending = false;
  else if (!rc) rc = JGPM_E_HIP;
  return rc;
}

uint64_t finish_pattern(int pattern, const uint64_t* h) {
  // unsigned wrap-around arithmetic is exact for the non-negative result
  switch (pattern) {
    case JGPM_I_DIAMOND: return h[0] - 6 * h[1];
    case JGPM_I_C4: return h[0] - h[1] + 3 * h[2];
    case JGPM_I_TAILTRI: return h[0] - 4 * h[1] + 12 * h[2];
    case JGPM_I_STAR3: return h[0] - h[1] + 2 * h[2] - 4 * h[3];
  }
  return h[0];
}

}  // namespace jgpm
