// C ABI of the device engine: graph upload, BFS and plain s–t queries.
//
// fc_graph_create_* replaces cudaGraph::cudaGraph (BFS-4K/src/device/cudaGraph.cu:7-36):
// the CSR is uploaded once and every per-query buffer is allocated up front,
// sized for the graph (queues of V entries per colour and parity, three
// frontier bitmaps per colour, a hub queue sized by the number of vertices of
// degree >= hub_threshold) instead of the reference's free/2 frontier buffers.
// fc_bfs replaces Reset + cudaBFS4K (BFS-4K/src/device/BFS_WorkEfficient.cu:81-133);
// fc_stcon replaces make_stcon's single-GPU path (st-conn/make_stcon.c:730-1497).
//
// Queries run through the device-side phase machine of visit.hip: the host
// starts it with one small launch that writes the control block, then replays
// a captured hipGraph of identical phase launches (or launches them directly
// when only a few are needed). The launches write a query's result to pinned
// memory when it is finished, where the host looks between batches of
// launches. Lists of plain queries, and visits that stay narrow, run inside
// one launch instead (st_teams_run).
#include "engine.hpp"
#include "team.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

using fc::fail;

namespace fc {
fc_status validate_csr32(const int32_t* off, const int32_t* col, int64_t V, int64_t E, int64_t hub, int64_t* hubs);
fc_status validate_csr64(const int64_t* off, const int32_t* col, int64_t V, int64_t E, int64_t hub, int64_t* hubs);
void hub_first32(const int32_t* off, const int32_t* col, int64_t V, int32_t* out);
void hub_first64(const int64_t* off, const int32_t* col, int64_t V, int32_t* out);
void relabel32(const int32_t* off, const int32_t* col, int64_t V, bool keep_order, int32_t* perm, int32_t* iperm,
               int32_t* noff, int32_t* ncol);
void relabel64(const int64_t* off, const int32_t* col, int64_t V, bool keep_order, int32_t* perm, int32_t* iperm,
               int64_t* noff, int32_t* ncol);
}  // namespace fc

namespace fcd {

fc_status hip_fail(hipError_t e, const char* what) {
  return fail(e == hipErrorNoDevice || e == hipErrorNoBinaryForGpu || e == hipErrorInvalidDevice ? FC_ERR_NOGPU
                                                                                                  : FC_ERR_HIP,
              "%s: %s", what, hipGetErrorString(e));
}

// Every graph of the process, for dev_malloc. Never destroyed: graphs may be
// freed by the caller's own static destructors.
struct Graphs {
  std::mutex mu;
  std::vector<fc_graph*> all;
};
static Graphs& graphs() {
  static Graphs* g = new Graphs();
  return *g;
}
static void graphs_remove(fc_graph* g) {
  std::lock_guard<std::mutex> lock(graphs().mu);
  auto& a = graphs().all;
  a.erase(std::remove(a.begin(), a.end(), g), a.end());
}

TeamUse::TeamUse(fc_graph* g_) : g(g_) {
  for (;;) {
    int n = g->team_use.load();
    if (n >= 0 && g->team_use.compare_exchange_weak(n, n + 1)) return;
    if (n < 0) std::this_thread::yield();  // for as long as a few frees take
  }
}

hipError_t dev_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  int device = 0;
  (void)hipGetDevice(&device);
  bool freed = false;
  {
    std::lock_guard<std::mutex> lock(graphs().mu);
    for (fc_graph* g : graphs().all) {
      int idle = 0;
      if (g->device != device || !g->team_use.compare_exchange_strong(idle, -1)) continue;
      freed |= g->team || g->st_teams;
      team_free(g->team);
      st_teams_free(g->st_teams);
      g->team = nullptr;
      g->st_teams = nullptr;
      g->team_use.store(0);
    }
  }
  return freed ? hipMalloc(p, bytes) : e;
}

size_t team_budget(size_t total) {
  size_t free = 0, all = 0;
  if (hipMemGetInfo(&free, &all) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return std::min(total / 8, free / 4);
}

fc_status ensure_queries(fc_graph* g, int32_t n) {
  if (n <= g->q_cap) return FC_OK;
  // the captured launches take only the control block, whose parameters
  // are rewritten by every run, so the graph stays valid
  (void)hipFree(g->d_qs);
  (void)hipFree(g->d_qt);
  if (g->h_out) (void)hipHostFree(g->h_out);
  g->d_qs = g->d_qt = nullptr;
  g->h_out = nullptr;
  g->q_cap = 0;
  const int32_t cap = std::max<int32_t>(n, 1024);
  FC_HIP(dev_malloc((void**)&g->d_qs, sizeof(int32_t) * (size_t)cap));
  FC_HIP(dev_malloc((void**)&g->d_qt, sizeof(int32_t) * (size_t)cap));
  FC_HIP(hipHostMalloc((void**)&g->h_out, sizeof(VisitOut) * (size_t)cap, hipHostMallocDefault));
  g->q_cap = cap;
  return FC_OK;
}

template <typename OffT>
static VisitParams<OffT> make_params(fc_graph* g) {
  VisitParams<OffT> p;
  std::memset(&p, 0, sizeof(p));
  set_param(p.off, (const OffT*)g->d_off);
  set_param(p.col, g->d_col);
  p.V = (int32_t)g->V;
  p.E = g->E;
  p.hub_threshold = g->hub_threshold;
  set_param(p.state, g->d_state);
  set_param(p.sst, g->d_sst);
  set_param(p.parent, g->d_parent);
  set_param(p.visited, g->d_visited);
  for (int c = 0; c < 2; ++c) {
    for (int k = 0; k < 3; ++k) set_param(p.fbm[c][k], g->d_fbm[c][k]);
    for (int k = 0; k < 2; ++k) {
      set_param(p.q[c][k], g->d_q[c][k]);
      set_param(p.hq[c][k], g->d_hq[c][k]);
      set_param(p.hb[c][k], g->d_hb[c][k]);
    }
  }
  p.qcap = g->qcap;
  p.hcap = g->hcap;
  set_param(p.ctl, g->d_ctl);
  set_param(p.qs, g->d_qs);
  set_param(p.qt, g->d_qt);
  set_param(p.out, g->h_out);
  p.lazy_state = g->relabeled ? 1 : 0;
  p.v_active = (int32_t)g->v_active;
  p.bottom_up = g->symmetric ? 1 : 0;
  set_param(p.head, g->d_head);
  return p;
}

static hipError_t launch_raw(fc_graph* g, int parity) {
  const bool wide = g->E >= kWideEdges && !g->narrow && !(g->regular && g->surface < kWideSurface);
  if (g->off64) return launch_phase<int64_t>(g->d_ctl, parity, g->blocks, wide, g->stream);
  return launch_phase<int32_t>(g->d_ctl, parity, g->blocks, wide, g->stream);
}

static fc_status ensure_graph(fc_graph* g) {
  if (g->gexec) return FC_OK;
  FC_HIP(hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal));
  hipError_t le = hipSuccess;
  for (int i = 0; i < kGraphLaunches && le == hipSuccess; ++i) le = launch_raw(g, i & 1);  // parities 0, 1, ...
  hipGraph_t gr = nullptr;
  hipError_t ce = hipStreamEndCapture(g->stream, &gr);
  if (le != hipSuccess) return hip_fail(le, "phase kernel capture");
  if (ce != hipSuccess) return hip_fail(ce, "hipStreamEndCapture");
  g->graph = gr;
  FC_HIP(hipGraphInstantiate(&g->gexec, g->graph, nullptr, nullptr, 0));
  return FC_OK;
}

// ---------------------------------------------------------------------------
// Plain s–t queries by teams (st_team_kernel): one launch per call.
// ---------------------------------------------------------------------------
struct StTeams {
  char* mem = nullptr;   // kXcds machines' workspaces
  size_t stride = 0;
  size_t o_q = 0, q1 = 0, o_hq = 0, hq1 = 0, o_hb = 0, hb1 = 0;  // pieces of one (state words first); x1: one array
  int blocks = 0, narrow_blocks = 0;
  uint32_t epoch_next = 1;
  char* d_io = nullptr;  // what a run uploads and reads back, and its pinned copy
  char* h_io = nullptr;
  size_t io_bytes = 0;
  bool off = false;      // not available for this graph
};

void st_teams_free(StTeams* w) {
  if (!w) return;
  (void)hipFree(w->mem);
  (void)hipFree(w->d_io);
  if (w->h_io) (void)hipHostFree(w->h_io);
  delete w;
}

static size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

static fc_status st_teams_alloc(fc_graph* g) {
  if (!g->st_teams) g->st_teams = new StTeams();
  StTeams* w = g->st_teams;
  if (w->mem || w->off) return FC_OK;
  hipDeviceProp_t prop;
  FC_HIP(hipGetDeviceProperties(&prop, g->device));
  const size_t V = (size_t)g->V, hcap = g->hcap;
  w->q1 = al256(4 * V);
  w->hq1 = al256(4 * hcap);
  w->hb1 = al256(8 * hcap);
  w->o_q = al256(8 * V);
  w->o_hq = w->o_q + 4 * w->q1;
  w->o_hb = w->o_hq + 4 * w->hq1;
  w->stride = w->o_hb + 4 * w->hb1;
  const int occ = g->off64 ? st_team_occupancy<int64_t>() : st_team_occupancy<int32_t>();
  const int nocc = g->off64 ? narrow_occupancy<int64_t>() : narrow_occupancy<int32_t>();
  // (a 4096^2 grid takes 3.2 GB)
  if (occ < 1 || g->cus % kXcds != 0 || kXcds * w->stride > team_budget(prop.totalGlobalMem)) {
    w->off = true;
    return FC_OK;
  }
  char* mem = nullptr;
  if (hipMalloc((void**)&mem, kXcds * w->stride) != hipSuccess) {
    (void)hipGetLastError();
    w->off = true;
    return FC_OK;
  }
  // Only the state words are read before they are written. The memory is the
  // teams' once they are cleared: a call that fails here leaves none behind.
  for (int k = 0; k < kXcds; ++k) {
    const hipError_t e = hipMemsetAsync(mem + (size_t)k * w->stride, 0, 8 * V, g->stream);
    if (e != hipSuccess) {
      (void)hipFree(mem);
      return hip_fail(e, "clearing the teams' state words");
    }
  }
  w->mem = mem;
  // 1,024 queries at s22 took 18.1, 11.9, 10.1 and 9.3 ms with 1 to 4 blocks
  // per CU, 8 queries on a 4096^2 grid 32.9, 27.1 and 25.4 ms with 1, 2 and 4.
  w->blocks = std::min(occ, 4) * g->cus;
  w->narrow_blocks = nocc > 0 ? g->cus : 0;
  return FC_OK;
}

// A query that reaches a level of more than this many edges per query of its
// call is given up and run again by launches: an XCD takes about as long for
// such a level (3.4 G claims/s) as the launches for all of the call's queries.
// Unbounded, a few hub expansions held up whole calls: R-MAT s24, 3, 6, 16 and
// 64 queries 0.78, 0.68, 1.53 and 2.44 ms, given up at 2^17 0.18, 0.25, 0.63
// and 1.49, by launches alone 0.21, 0.34, 0.93 and 3.01; s22, 64 queries 2.21,
// 0.95 and 2.16; two queries between two random graphs of 1M vertices, which
// they exhaust, 2.49, 1.05 and 1.07. At 2^16 and 2^18 within 5% of that. Where
// more than half of a call's eight or more queries are given up (64 such
// queries: 38 ms, unbounded 23), the graph's next calls are not bounded.
constexpr int64_t kTeamLevelEdges = 1 << 17;

// Whether n queries go to the teams: several always (eight are visited at a
// time: R-MAT s22, 16 queries, 0.42 -> 0.23 ms); a single one where its
// frontiers are likely to stay narrow (random graph of 50K vertices and degree
// 3, 53 against 68 us a call, 100^2 grid 160 against 341), since a few wide
// levels take the whole GPU no longer (s16 47 us against 53, the random graph
// with degree 8 45 against 49).
static bool st_teams_take(const fc_graph* g, int32_t n) { return g->use_st_teams && (n > 1 || g->narrow); }

// Levels (and parents) of a narrow BFS in caller ids, from the state words of
// the machine that ran it (out->meet).
__global__ void narrow_levels_kernel(const int32_t* __restrict__ perm, const int32_t* __restrict__ iperm,
                                     const char* __restrict__ mem, size_t stride, const VisitOut* __restrict__ out,
                                     uint32_t epoch, const int32_t* par, int32_t* __restrict__ lv_out,
                                     int32_t* par_out, int64_t V) {  // par_out may be par (without perm)
  const unsigned long long* sst =
      reinterpret_cast<const unsigned long long*>(mem + (size_t)(out->meet & (kXcds - 1)) * stride);
  const int64_t n = (int64_t)gridDim.x * blockDim.x;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += n) {
    const int32_t k = perm ? perm[v] : (int32_t)v;
    const unsigned long long w = sst[k];
    const bool r = (uint32_t)(w >> 32) == epoch;
    lv_out[v] = r ? (int32_t)((uint32_t)w & (uint32_t)kLevelMask) : -1;
    if (par_out) {
      const int32_t q = r ? par[k] : -1;
      par_out[v] = iperm && (uint32_t)q < (uint32_t)V ? iperm[q] : q;
    }
  }
}

// What a launch by teams starts from, written by one small launch before it: a
// block per machine clears the machine's words and writes its parameters (those
// of machine 0, its workspace moved by the stride). As an upload from pinned
// memory, 40 KB, it took 10 us of a query's 58.
constexpr int kStartThreads = 256;
template <typename Params>
struct TeamStart {
  Params prm;
  int32_t s[kStartPairs], t[kStartPairs];
};
template <typename T>
__device__ __forceinline__ void clear_words(T* p) {
  static_assert(sizeof(T) % sizeof(uint4) == 0, "16 bytes a store");
  for (uint32_t i = threadIdx.x; i < sizeof(T) / sizeof(uint4); i += kStartThreads)
    reinterpret_cast<uint4*>(p)[i] = make_uint4(0, 0, 0, 0);
}
template <typename Params>
__global__ __launch_bounds__(kStartThreads) void team_start_kernel(const TeamStart<Params> v, StTeamRun tr, size_t stride,
                                                                   int32_t* qs, int32_t* qt, int n) {
  const int k = (int)blockIdx.x;
  clear_words(tr.sync + k);
  clear_words(tr.bar + k);
  clear_words(tr.ctl + k);
  __syncthreads();
  if (threadIdx.x == 0) {
    for (auto& b : tr.ctl[k].best) b[0] = b[1] = ~0ull;
    if (k == 0) *tr.ticket = 0;
    Params p = v.prm;
    const size_t by = (size_t)k * stride;
    set_param(p.sst, (unsigned long long*)((char*)p.sst + by));
    for (int c = 0; c < 2; ++c)
      for (int r = 0; r < 2; ++r) {
        set_param(p.q[c][r], (int32_t*)((char*)p.q[c][r] + by));
        set_param(p.hq[c][r], (int32_t*)((char*)p.hq[c][r] + by));
        set_param(p.hb[c][r], (int64_t*)((char*)p.hb[c][r] + by));
      }
    set_param(p.ctl, &tr.ctl[k].v);
    ((Params*)tr.params)[k] = p;
  }
  if (k == 0 && (int)threadIdx.x < n) {
    qs[threadIdx.x] = v.s[threadIdx.x];
    qt[threadIdx.x] = v.t[threadIdx.x];
  }
}

// Run n plain s–t queries by teams (narrow: as narrow visits), or with bfs one
// BFS from s[0] as a narrow visit, whose levels (and, with par_out, parents)
// go to lv_out; results in g->h_out. *ran is false when the teams are not
// available for this graph.
static fc_status st_teams_run(fc_graph* g, const int32_t* s, const int32_t* t, int32_t n, bool narrow, bool bfs,
                              int32_t* lv_out, int32_t* par_out, double* ms, bool* ran, const VisitTail& after = {}) {
  *ran = false;
  const TeamUse use(g);
  fc_status st = st_teams_alloc(g);
  if (st != FC_OK) return st;
  StTeams* w = g->st_teams;
  if (w->off || (narrow && !w->narrow_blocks)) return FC_OK;
  if ((uint64_t)w->epoch_next + (uint64_t)n >= 0xFFFFFFF0ull) {
    for (int k = 0; k < kXcds; ++k)
      FC_HIP(hipMemsetAsync(w->mem + (size_t)k * w->stride, 0, 8 * (size_t)g->V, g->stream));
    w->epoch_next = 1;
  }
  static_assert(sizeof(VisitParams<int32_t>) == sizeof(VisitParams<int64_t>), "one size of parameters");
  const size_t o_bar = al256(kXcds * sizeof(TeamSync)), o_tick = o_bar + al256(kXcds * sizeof(TeamBar));
  const size_t o_ctl = o_tick + 256, o_par = o_ctl + al256(kXcds * sizeof(StTeamCtl));
  const size_t o_qs = o_par + al256(kXcds * sizeof(VisitParams<int64_t>)), o_qt = o_qs + al256(4 * (size_t)n);
  const size_t o_err = o_qt + al256(4 * (size_t)n), o_out = o_err + 256, bytes = o_out + sizeof(VisitOut) * (size_t)n;
  if (bytes > w->io_bytes) {
    (void)hipFree(w->d_io);
    if (w->h_io) (void)hipHostFree(w->h_io);
    w->d_io = w->h_io = nullptr;
    w->io_bytes = 0;
    const size_t cap = std::max<size_t>(bytes, 1u << 17);
    FC_HIP(dev_malloc((void**)&w->d_io, cap));
    FC_HIP(hipHostMalloc((void**)&w->h_io, cap, hipHostMallocDefault));
    w->io_bytes = cap;
  }
  *(uint32_t*)(w->h_io + o_err) = 0;
  StTeamRun tr;
  tr.sync = (TeamSync*)w->d_io;
  tr.bar = (TeamBar*)(w->d_io + o_bar);
  tr.ctl = (StTeamCtl*)(w->d_io + o_ctl);
  tr.ticket = (uint32_t*)(w->d_io + o_tick);
  tr.err = (uint32_t*)(w->h_io + o_err);
  tr.params = w->d_io + o_par;
  tr.nq = n;
  tr.epoch0 = w->epoch_next;
  tr.vw_fixed = g->vw_fixed;
  if (narrow && tr.vw_fixed == 0) {  // published vertices: the graph's mean degree, rounded up to a power of two
    tr.vw_fixed = 4;
    while (tr.vw_fixed < 64 && (int64_t)tr.vw_fixed * g->V < g->E) tr.vw_fixed <<= 1;
  }
  const int blocks = narrow ? w->narrow_blocks : w->blocks;
  tr.expected = (uint32_t)(blocks / kXcds);
  tr.parents = par_out != nullptr;
  tr.max_edges = n >= kXcds && !g->st_limit ? INT64_MAX : (int64_t)n * kTeamLevelEdges;
  w->epoch_next += (uint32_t)n;
  const int few = n <= kStartPairs ? n : 0;
  if (!few) {
    std::memcpy(w->h_io + o_qs, s, 4 * (size_t)n);
    std::memcpy(w->h_io + o_qt, t, 4 * (size_t)n);
    FC_HIP(hipMemcpyAsync(w->d_io + o_qs, w->h_io + o_qs, o_err - o_qs, hipMemcpyHostToDevice, g->stream));
  }
  auto start = [&](auto prm) {
    TeamStart<decltype(prm)> v;
    for (int c = 0; c < 2; ++c)
      for (int r = 0; r < 2; ++r) {
        const size_t k = (size_t)(2 * c + r);
        set_param(prm.q[c][r], (int32_t*)(w->mem + w->o_q + k * w->q1));
        set_param(prm.hq[c][r], (int32_t*)(w->mem + w->o_hq + k * w->hq1));
        set_param(prm.hb[c][r], (int64_t*)(w->mem + w->o_hb + k * w->hb1));
      }
    set_param(prm.sst, (unsigned long long*)w->mem);
    set_param(prm.qs, (const int32_t*)(w->d_io + o_qs));
    set_param(prm.qt, (const int32_t*)(w->d_io + o_qt));
    set_param(prm.out, (VisitOut*)((bfs ? w->d_io : w->h_io) + o_out));  // a BFS's is read on the device too
    v.prm = prm;
    for (int i = 0; i < kStartPairs; ++i) {
      v.s[i] = i < few ? s[i] : 0;
      v.t[i] = i < few ? t[i] : 0;
    }
    hipLaunchKernelGGL(team_start_kernel<decltype(prm)>, dim3(kXcds), dim3(kStartThreads), 0, g->stream, v, tr, w->stride,
                       (int32_t*)(w->d_io + o_qs), (int32_t*)(w->d_io + o_qt), few);
    return hipGetLastError();
  };
  FC_HIP(g->off64 ? start(make_params<int64_t>(g)) : start(make_params<int32_t>(g)));
  FC_HIP(hipEventRecord(g->ev0, g->stream));
  if (narrow)
    FC_HIP(g->off64 ? launch_narrow<int64_t>(tr, bfs, blocks, g->stream)
                    : launch_narrow<int32_t>(tr, bfs, blocks, g->stream));
  else
    FC_HIP(g->off64 ? launch_st_team<int64_t>(tr, blocks, g->stream) : launch_st_team<int32_t>(tr, blocks, g->stream));
  if (bfs) {
    const int lb = (int)std::min<int64_t>((g->V + 255) / 256, (int64_t)g->cus * 8);
    hipLaunchKernelGGL(narrow_levels_kernel, dim3(lb), dim3(256), 0, g->stream, g->d_perm, g->d_iperm, w->mem,
                       w->stride, (const VisitOut*)(w->d_io + o_out), tr.epoch0, g->d_parent, lv_out, par_out,
                       (int64_t)g->V);
    FC_HIP(hipGetLastError());
  }
  FC_HIP(hipEventRecord(g->ev1, g->stream));
  if (bfs) {
    FC_HIP(hipMemcpyAsync(w->h_io + o_out, w->d_io + o_out, sizeof(VisitOut), hipMemcpyDeviceToHost, g->stream));
    if (after) FC_HIP(after());
  }
  FC_HIP(hipStreamSynchronize(g->stream));
  float fms = 0.f;
  FC_HIP(hipEventElapsedTime(&fms, g->ev0, g->ev1));
  *ms = fms;
  if (*(const volatile uint32_t*)(w->h_io + o_err)) {
    // queues and counters are in an unknown state: the next run takes new ones
    st_teams_free(w);
    g->st_teams = nullptr;
    return fail(FC_ERR_TIMEOUT, "s–t visit: a team's wait was given up");
  }
  std::memcpy(g->h_out, w->h_io + o_out, sizeof(VisitOut) * (size_t)n);
  g->h_out[0].launches = 1;
  *ran = true;
  return FC_OK;
}

// A run's control block and, of a few queries, their ends, as kernel arguments:
// one launch instead of three copies from pageable memory and the wait for
// them (25 us before the first level).
struct VisitStart {
  VisitCtl ctl;
  int32_t s[kStartPairs], t[kStartPairs];
};
__global__ __launch_bounds__(kWave) void visit_start_kernel(const VisitStart v, VisitCtl* ctl, int32_t* qs,
                                                            int32_t* qt, int n) {
  const int i = (int)threadIdx.x;
  reinterpret_cast<uint4*>(ctl)[i] = reinterpret_cast<const uint4*>(&v.ctl)[i];
  if (i < n) {
    qs[i] = v.s[i];
    qt[i] = v.t[i];
  }
}

// Run the queries among s, t whose visit was given up (kTooWide) again and put
// their results in place; *found: whether there were any.
template <typename Run>
static fc_status redo_wide(fc_graph* g, const int32_t* s, const int32_t* t, int32_t n, double* ms, bool* found, Run run) {
  std::vector<int32_t> idx, vs, vt;
  for (int32_t i = 0; i < n; ++i)
    if (g->h_out[i].status == kTooWide) {
      idx.push_back(i);
      vs.push_back(s[i]);
      vt.push_back(t[i]);
    }
  *found = !idx.empty();
  if (idx.empty()) return FC_OK;
  const std::vector<VisitOut> kept(g->h_out, g->h_out + n);
  double more = 0.0;
  const fc_status st = run(vs.data(), vt.data(), (int32_t)idx.size(), &more);
  if (st != FC_OK) return st;
  const std::vector<VisitOut> again(g->h_out, g->h_out + idx.size());
  std::copy(kept.begin(), kept.end(), g->h_out);
  for (size_t k = 0; k < idx.size(); ++k) {
    g->h_out[idx[k]] = again[k];
    g->h_out[idx[k]].launches += kept[(size_t)idx[k]].launches;  // the first call's one
  }
  *ms += more;
  return FC_OK;
}

static fc_status run_launches(fc_graph* g, int mode, const int32_t* s, const int32_t* t, int32_t n, bool parents,
                              double* ms, const VisitTail& tail, const VisitTail& after);

fc_status run_visits(fc_graph* g, int mode, const int32_t* s, const int32_t* t, int32_t n, bool parents,
                     double* ms, const VisitTail& tail, const VisitTail& after) {
  *ms = 0.0;
  if (n <= 0) return FC_OK;
  fc_status st = ensure_queries(g, n);
  if (st != FC_OK) return st;
  if (mode == kModePlainSt && !parents && st_teams_take(g, n)) {
    bool ran = false, found = false;
    const bool narrow = g->narrow && g->narrow_st;
    st = st_teams_run(g, s, t, n, narrow, false, nullptr, nullptr, ms, &ran);
    if (st != FC_OK) return st;
    if (ran && narrow) {
      st = redo_wide(g, s, t, n, ms, &found, [&](const int32_t* vs, const int32_t* vt, int32_t k, double* more) {
        return st_teams_run(g, vs, vt, k, false, false, nullptr, nullptr, more, &ran);
      });
      if (st != FC_OK) return st;
      if (found) g->narrow_st = false;  // the next calls on this graph do not try
    }
    if (ran)
      return redo_wide(g, s, t, n, ms, &found, [&](const int32_t* vs, const int32_t* vt, int32_t k, double* more) {
        if (n >= kXcds && k > n / 2) g->st_limit = false;
        return run_launches(g, mode, vs, vt, k, false, more, {}, {});
      });
  }
  return run_launches(g, mode, s, t, n, parents, ms, tail, after);
}

static fc_status run_launches(fc_graph* g, int mode, const int32_t* s, const int32_t* t, int32_t n, bool parents,
                              double* ms, const VisitTail& tail, const VisitTail& after) {
  fc_status st = FC_OK;
  if (g->use_graphs) {
    st = ensure_graph(g);
    if (st != FC_OK) return st;
  }
  // s–t queries tag the state words with one epoch each (0 = never
  // visited); before the counter would wrap, the words are cleared.
  uint32_t epoch0 = 0;
  if (mode == kModePlainSt) {
    if ((uint64_t)g->epoch_next + (uint64_t)n >= 0xFFFFFFF0ull) {
      FC_HIP(hipMemsetAsync(g->d_sst, 0, sizeof(unsigned long long) * (size_t)g->V, g->stream));
      g->epoch_next = 1;
    }
    epoch0 = g->epoch_next;
    g->epoch_next += (uint32_t)n;
  }
  VisitStart init;
  init.ctl = g->off64 ? visit_init(make_params<int64_t>(g), mode, n, s, t, epoch0, g->vw_fixed, parents)
                      : visit_init(make_params<int32_t>(g), mode, n, s, t, epoch0, g->vw_fixed, parents);
  const int few = n <= kStartPairs ? n : 0;
  for (int i = 0; i < kStartPairs; ++i) {
    init.s[i] = i < few ? s[i] : 0;
    init.t[i] = i < few ? t[i] : 0;
  }
  if (!few) {
    FC_HIP(hipMemcpyAsync(g->d_qs, s, sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice, g->stream));
    FC_HIP(hipMemcpyAsync(g->d_qt, t, sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice, g->stream));
    // pageable host memory: finish the copies before the caller's arrays can
    // go away, and before timing starts
    FC_HIP(hipStreamSynchronize(g->stream));
  }
  hipLaunchKernelGGL(visit_start_kernel, dim3(1), dim3(kWave), 0, g->stream, init, g->d_ctl, g->d_qs, g->d_qt, few);
  FC_HIP(hipGetLastError());
  // the launches write a query's result here when it is finished
  constexpr int32_t kRunning = INT32_MIN;
  volatile VisitOut* const out = g->h_out;
  for (int32_t i = 0; i < n; ++i) out[i].status = kRunning;

  // Launch budget: the running estimate of working launches per query, plus
  // the launch that notices the last query's end. A single BFS needs no
  // extra margin: a short budget costs one more host poll, and each surplus
  // launch of the full grid a few us. At most kPollLaunches are queued
  // between two polls: a high-diameter batch needs hundreds of thousands of
  // launches, and queueing them all at once holds that many dispatches (and
  // a profiler's record of each) in flight in the runtime. A poll costs one
  // host round trip per kPollLaunches launches of at least 1.6 us each.
  // Launches alternate parity 0, 1, 0, ... (the state a launch reads), and
  // the captured graphs hold an even number of launches starting at 0.
  const double est = g->est_launches[mode];
  int64_t expected = (int64_t)std::ceil((double)n * est) + 1;
  int64_t launched = 0;
  int32_t qi = 0;  // queries finished
  FC_HIP(hipEventRecord(g->ev0, g->stream));
  for (int round = 0;; ++round) {
    int64_t want = expected - launched;
    if (want < 1) want = 1;
    if (want > kPollLaunches) want = kPollLaunches;
    if (want < kGraphLaunches || !g->use_graphs) {
      for (int64_t i = 0; i < want; ++i) {
        hipError_t e = launch_raw(g, (int)(launched & 1));
        if (e != hipSuccess) return hip_fail(e, "phase kernel launch");
        ++launched;
      }
    } else {
      if (launched & 1) {
        hipError_t e = launch_raw(g, 1);
        if (e != hipSuccess) return hip_fail(e, "phase kernel launch");
        ++launched;
        --want;
      }
      const int64_t ng = (want + kGraphLaunches - 1) / kGraphLaunches;
      for (int64_t i = 0; i < ng; ++i) FC_HIP(hipGraphLaunch(g->gexec, g->stream));
      launched += ng * kGraphLaunches;
    }
    if (tail) FC_HIP(tail());
    FC_HIP(hipEventRecord(g->ev1, g->stream));
    if (after) FC_HIP(after());
    FC_HIP(hipStreamSynchronize(g->stream));
    while (qi < n && out[qi].status != kRunning) ++qi;
    if (qi == n) break;
    // Every query stops within V+2 levels (device guard), so this bound is
    // never reached by a working visit.
    if (launched > (int64_t)n * (g->V + 4) + 64)
      return fail(FC_ERR_CAPACITY, "phase machine did not finish after %lld launches", (long long)launched);
    // Not finished. While the budget lasts, keep to it; past it, budget the
    // remaining queries with a wider margin.
    if (launched < expected) continue;
    const int64_t remaining = std::max<int64_t>(n - qi, 1);
    expected = launched + (int64_t)std::ceil((double)remaining * (est + 1.0) * (1.0 + round)) + 1;
  }
  float fms = 0.f;
  FC_HIP(hipEventElapsedTime(&fms, g->ev0, g->ev1));
  *ms = fms;
  double wl = 0;
  for (int32_t i = 0; i < n; ++i) wl += g->h_out[i].launches;
  g->est_launches[mode] = 0.5 * g->est_launches[mode] + 0.5 * (wl / n);
  return FC_OK;
}

// Whether every edge is stored in both directions, by hash sums: the sum over
// all edges of h(u, v) - h(v, u) is 0 (mod 2^64) on a symmetric graph, and on
// another one with probability about 2^-64. An edge that a list repeats counts
// once (id-sorted lists hold the copies side by side; elsewhere such a graph
// may be taken for a directed one, which only costs speed). One pass over the
// columns (s22: 0.2 ms); a wave takes chunks of 2,048 edges and walks the
// source along.
__device__ __forceinline__ unsigned long long edge_hash(uint32_t a, uint32_t b) {
  unsigned long long z = ((unsigned long long)a << 32 | b) + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Each vertex's first two columns side by side (VisitParams::head).
template <typename OffT>
__global__ __launch_bounds__(256) void head_kernel(const OffT* __restrict__ off, const int32_t* __restrict__ col,
                                                   int64_t V, unsigned long long* __restrict__ head) {
  const int64_t n = (int64_t)gridDim.x * blockDim.x;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += n) {
    const OffT b = off[v], d = off[v + 1] - b;
    const uint32_t u0 = d > 0 ? (uint32_t)col[b] : 0xffffffffu, u1 = d > 1 ? (uint32_t)col[b + 1] : 0xffffffffu;
    head[v] = ((unsigned long long)u1 << 32) | u0;
  }
}

template <typename OffT>
__global__ __launch_bounds__(256) void symmetry_kernel(const OffT* __restrict__ off, const int32_t* __restrict__ col,
                                                       int64_t V, int64_t E, unsigned long long* __restrict__ out) {
  constexpr int64_t kChunk = 2048;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int64_t waves = ((int64_t)gridDim.x * blockDim.x) >> 6;
  unsigned long long sum = 0;
  for (int64_t c = wave * kChunk; c < E; c += waves * kChunk) {
    int64_t lo = 0, hi = V;  // the last vertex whose list starts at or before the lane's first edge
    const int64_t j0 = c + lane_id();
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)off[mid] <= j0)
        lo = mid;
      else
        hi = mid;
    }
    const int64_t end = c + kChunk < E ? c + kChunk : E;
    for (int64_t j = j0; j < end; j += kWave) {
      while (lo + 1 < V && (int64_t)off[lo + 1] <= j) ++lo;
      const uint32_t u = (uint32_t)lo, v = (uint32_t)col[j];
      if (j > (int64_t)off[lo] && (uint32_t)col[j - 1] == v) continue;
      sum += edge_hash(u, v) - edge_hash(v, u);
    }
  }
  const uint64_t tot = wave_sum_u64(sum);
  if (lane_id() == 0 && tot) atomicAdd(out, (unsigned long long)tot);
}

}  // namespace fcd

using fcd::hip_fail;

template <typename OffT>
static fc_status graph_create(const OffT* off, const int32_t* col, int64_t V, int64_t E, uint32_t flags,
                              fc_graph** out) {
  fc::clear_error();
  if (!out || !off || (E > 0 && !col) || V < 1 || V > INT32_MAX - 64 || E < 0)
    return fail(FC_ERR_INVALID, "fc_graph_create: invalid arguments (V=%lld E=%lld)", (long long)V, (long long)E);
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(FC_ERR_NOGPU, "no HIP device available");
  fc_graph* g = new fc_graph();
  g->V = V;
  g->E = E;
  g->off64 = sizeof(OffT) == 8;
  // Degree from which a frontier vertex goes to the edge-balanced hub
  // queue. 256 measured best at R-MAT s22 (batch 2.09 ms, plain 32.0K q/s,
  // BFS 0.235 ms, against 2.11 ms, 29.2K q/s and 0.237 ms at 512 and
  // 2.40 ms, 30.0K q/s and 0.244 ms at 64).
  const char* ht = std::getenv("FASTCON_HUB_THRESHOLD");
  const bool ht_set = ht && std::atoi(ht) > 0;
  g->hub_threshold = ht_set ? std::atoi(ht) : 256;
  const char* vwf = std::getenv("FASTCON_VW");
  if (vwf) g->vw_fixed = fcd::visit_width(std::atoi(vwf));
  // Direct launches instead of replayed hipGraphs, for profiler runs: under
  // rocprofv3's kernel trace a hipGraphLaunch of the visit's graph ended in
  // a host segmentation fault inside the runtime, while direct launches of
  // the same kernel trace normally.
  const char* pg = std::getenv("FASTCON_PLAIN_GRAPHS");
  if (pg && std::strcmp(pg, "0") == 0) g->use_graphs = false;
  const char* pt = std::getenv("FASTCON_PLAIN_TEAMS");
  if (pt && std::strcmp(pt, "0") == 0) g->use_st_teams = false;
  int64_t hubs = 0;
  fc_status st = sizeof(OffT) == 8
                     ? fc::validate_csr64((const int64_t*)off, col, V, E, g->hub_threshold, &hubs)
                     : fc::validate_csr32((const int32_t*)off, col, V, E, g->hub_threshold, &hubs);
  if (st != FC_OK) {
    delete g;
    return st;
  }
  // Hub-queue counters pack (entries << 40) | edges into 64 bits: at most
  // 2^24 - 1 hub entries per frontier. The default threshold doubles until
  // the hubs fit; a threshold the caller set is kept, and the graph refused.
  const int64_t hub_cap = (int64_t)(1ll << (64 - fcd::kHubEdgeBits));
  while (!ht_set && hubs >= hub_cap && g->hub_threshold < (1 << 30)) {
    g->hub_threshold *= 2;
    hubs = 0;
    for (int64_t v = 0; v < V; ++v) hubs += (int64_t)off[v + 1] - (int64_t)off[v] >= g->hub_threshold;
  }
  if (hubs >= hub_cap) {
    const int32_t thr = g->hub_threshold;
    delete g;
    return fail(FC_ERR_CAPACITY, "fc_graph_create: %lld vertices of degree >= %d exceed the hub queue's %lld entries",
                (long long)hubs, thr, (long long)((1ll << (64 - fcd::kHubEdgeBits)) - 1));
  }
  auto bail = [&](fc_status s) {
    fc_graph_destroy(g);
    return s;
  };
  {
    double d2 = 0.0;
    int64_t active = 0;
    for (int64_t v = 0; v < V; ++v) {
      const double d = (double)((int64_t)off[v + 1] - (int64_t)off[v]);
      d2 += d * d;
      active += d > 0.0;
    }
    g->branch = E > 0 ? d2 / (double)E : 0.0;
    const double mean = active > 0 ? (double)E / (double)active : 0.0;
    g->regular = E > 0 && g->branch < mean + 0.5;
    g->skewed = g->branch > 4.0 * mean;
    // a mesh of D dimensions, with 2 D neighbours or 3^D - 1
    const double dims = std::max(1.0, g->branch < 7.0 ? g->branch / 2.0 : std::log(1.0 + g->branch) / std::log(3.0));
    if (g->regular) g->surface = g->branch * std::pow((double)active, 1.0 - 1.0 / dims);
    g->f_branch = (float)(std::log2(1.0 + g->branch) / 16.0);
    // A vertex reached over an edge leads to at most five others on average:
    // frontiers grow slowly or, on a grid, hardly. Measured (start engine
    // against narrow visits, device time): 2048^2 grid (3.9), a BFS 30.4
    // against 10.4 ms; a random graph of mean degree 3 (4.0), 50K vertices, a
    // BFS 0.25 against 0.16 ms, 64 queries 0.32 against 0.29; of degree 8
    // (9.0), 64 queries 0.15 against 0.18.
    g->narrow = E > 0 && g->branch <= 6.0;
  }
#define CK(call)                                            \
  do {                                                      \
    hipError_t _e = (call);                                 \
    if (_e != hipSuccess) return bail(hip_fail(_e, #call)); \
  } while (0)
  CK(hipGetDevice(&g->device));
  hipDeviceProp_t prop;
  CK(hipGetDeviceProperties(&prop, g->device));
  g->cus = prop.multiProcessorCount;
  CK(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
  CK(hipEventCreate(&g->ev0));
  CK(hipEventCreate(&g->ev1));
  CK(fcd::dev_malloc(&g->d_off, sizeof(OffT) * (size_t)(V + 1)));
  CK(fcd::dev_malloc((void**)&g->d_col, sizeof(int32_t) * (size_t)std::max<int64_t>(E, 1)));
  if (!(flags & FC_GRAPH_KEEP_IDS)) {
    g->relabeled = true;
    g->h_perm.resize((size_t)V);
    g->h_iperm.resize((size_t)V);
    std::vector<OffT> noff((size_t)V + 1);
    std::vector<int32_t> ncol((size_t)std::max<int64_t>(E, 1));
    if (sizeof(OffT) == 8)
      fc::relabel64((const int64_t*)off, col, V, (flags & FC_GRAPH_KEEP_ORDER) != 0, g->h_perm.data(),
                    g->h_iperm.data(), (int64_t*)noff.data(), ncol.data());
    else
      fc::relabel32((const int32_t*)off, col, V, (flags & FC_GRAPH_KEEP_ORDER) != 0, g->h_perm.data(),
                    g->h_iperm.data(), (int32_t*)noff.data(), ncol.data());
    CK(fcd::dev_malloc((void**)&g->d_perm, sizeof(int32_t) * (size_t)V));
    CK(fcd::dev_malloc((void**)&g->d_iperm, sizeof(int32_t) * (size_t)V));
    CK(hipMemcpyAsync(g->d_perm, g->h_perm.data(), sizeof(int32_t) * (size_t)V, hipMemcpyHostToDevice, g->stream));
    CK(hipMemcpyAsync(g->d_iperm, g->h_iperm.data(), sizeof(int32_t) * (size_t)V, hipMemcpyHostToDevice, g->stream));
    CK(hipMemcpyAsync(g->d_off, noff.data(), sizeof(OffT) * (size_t)(V + 1), hipMemcpyHostToDevice, g->stream));
    if (E > 0) CK(hipMemcpyAsync(g->d_col, ncol.data(), sizeof(int32_t) * (size_t)E, hipMemcpyHostToDevice, g->stream));
    // decreasing degree: the vertices of degree > 0 are a prefix
    int64_t va = V;
    while (va > 0 && noff[(size_t)va] == noff[(size_t)va - 1]) --va;
    for (int64_t v = 0; v < va; ++v)
      if (noff[(size_t)v + 1] == noff[(size_t)v])
        return bail(fail(FC_ERR_INVALID, "internal: degree order broken at vertex %lld", (long long)v));
    g->v_active = va;
    g->lists_sorted = !(flags & FC_GRAPH_KEEP_ORDER);
    // 512 top vertices on 1/64 of the edge ends or more: R-MAT graphs; 2^-12 of them on a sparse random graph
    g->hub_steps = (int64_t)noff[(size_t)std::min<int64_t>(512, V)] >= E / 64;
  } else {
    g->v_active = V;
    CK(hipMemcpyAsync(g->d_off, off, sizeof(OffT) * (size_t)(V + 1), hipMemcpyHostToDevice, g->stream));
  }
  if (E > 0 && !g->relabeled) {
    if (flags & FC_GRAPH_KEEP_ORDER) {
      CK(hipMemcpyAsync(g->d_col, col, sizeof(int32_t) * (size_t)E, hipMemcpyHostToDevice, g->stream));
    } else {
      std::vector<int32_t> ordered((size_t)E);
      if (sizeof(OffT) == 8)
        fc::hub_first64((const int64_t*)off, col, V, ordered.data());
      else
        fc::hub_first32((const int32_t*)off, col, V, ordered.data());
      CK(hipMemcpyAsync(g->d_col, ordered.data(), sizeof(int32_t) * (size_t)E, hipMemcpyHostToDevice, g->stream));
    }
  }

  // Workspace layout (256-byte aligned pieces of one allocation).
  const size_t nw64 = (size_t)((V + 63) / 64);
  const size_t bm_bytes = nw64 * 2 * sizeof(uint32_t);
  g->qcap = (uint32_t)V;
  g->hcap = (uint32_t)std::max<int64_t>(hubs, 1);
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  size_t off_state = 0;
  size_t off_sst = off_state + al(sizeof(int32_t) * (size_t)V);
  size_t off_parent = off_sst + al(sizeof(unsigned long long) * (size_t)V);
  size_t off_vis = off_parent + al(sizeof(int32_t) * (size_t)V);
  size_t off_fbm = off_vis + al(bm_bytes);
  size_t off_q = off_fbm + 6 * al(bm_bytes);
  size_t off_hq = off_q + 4 * al(sizeof(int32_t) * (size_t)g->qcap);
  size_t off_hb = off_hq + 4 * al(sizeof(int32_t) * (size_t)g->hcap);
  size_t off_ctl = off_hb + 4 * al(sizeof(int64_t) * (size_t)g->hcap);
  g->ws_bytes = off_ctl + al(sizeof(fcd::VisitCtl));
  CK(fcd::dev_malloc((void**)&g->d_ws, g->ws_bytes));
  CK(hipMemsetAsync(g->d_ws, 0, g->ws_bytes, g->stream));
  g->d_state = (int32_t*)(g->d_ws + off_state);
  g->d_sst = (unsigned long long*)(g->d_ws + off_sst);
  g->d_parent = (int32_t*)(g->d_ws + off_parent);
  g->d_visited = (uint32_t*)(g->d_ws + off_vis);
  for (int c = 0; c < 2; ++c) {
    for (int k = 0; k < 3; ++k) g->d_fbm[c][k] = (uint32_t*)(g->d_ws + off_fbm + (size_t)(c * 3 + k) * al(bm_bytes));
    for (int k = 0; k < 2; ++k) {
      g->d_q[c][k] = (int32_t*)(g->d_ws + off_q + (size_t)(c * 2 + k) * al(sizeof(int32_t) * g->qcap));
      g->d_hq[c][k] = (int32_t*)(g->d_ws + off_hq + (size_t)(c * 2 + k) * al(sizeof(int32_t) * g->hcap));
      g->d_hb[c][k] = (int64_t*)(g->d_ws + off_hb + (size_t)(c * 2 + k) * al(sizeof(int64_t) * g->hcap));
    }
  }
  g->d_ctl = (fcd::VisitCtl*)(g->d_ws + off_ctl);
  // canonical parameters, then the copy in the batch kernel's layout
  CK(fcd::dev_malloc((void**)&g->d_mlp, 2 * sizeof(float) * fcd::kMlpParams));
  CK(hipMemsetAsync(g->d_mlp, 0, 2 * sizeof(float) * fcd::kMlpParams, g->stream));
  CK(hipHostMalloc((void**)&g->h_phase, 4 * sizeof(int32_t), hipHostMallocDefault));
  if (fcd::dev_malloc((void**)&g->d_head, sizeof(unsigned long long) * (size_t)std::max<int64_t>(V, 1)) == hipSuccess) {
    hipLaunchKernelGGL(fcd::head_kernel<OffT>, dim3(g->cus * 8), dim3(256), 0, g->stream, (const OffT*)g->d_off, g->d_col, V,
                       g->d_head);
    CK(hipGetLastError());
  } else {
    (void)hipGetLastError();  // a bottom-up level does without
    g->d_head = nullptr;
  }
  // the sum lands in the parameters' buffer, which is still unused
  hipLaunchKernelGGL(fcd::symmetry_kernel<OffT>, dim3(g->cus * 8), dim3(256), 0, g->stream, (const OffT*)g->d_off,
                     g->d_col, V, E, (unsigned long long*)g->d_mlp);
  CK(hipGetLastError());
  CK(hipMemcpyAsync(g->h_phase, g->d_mlp, sizeof(unsigned long long), hipMemcpyDeviceToHost, g->stream));
  CK(hipMemsetAsync(g->d_mlp, 0, sizeof(unsigned long long), g->stream));

  int occ = sizeof(OffT) == 8 ? fcd::phase_occupancy<int64_t>() : fcd::phase_occupancy<int32_t>();
  if (occ < 1) return bail(fail(FC_ERR_NOGPU, "phase kernel has no occupancy on this device (missing gfx950 code?)"));
  // 16 waves per CU, in blocks of four, measured best for BFS and plain s–t at
  // s22 (8: 345, 12: 384, 16: 401, 24: 392, 32: 348 GTEPS): more blocks add
  // contention on the launch's shared counters more than they hide latency.
  // Wide graphs run the same waves in larger blocks (kWideWaves).
  int per_cu = std::min(occ, 4);
  const char* bpc = std::getenv("FASTCON_BLOCKS_PER_CU");
  if (bpc && std::atoi(bpc) > 0) per_cu = std::min(occ, std::atoi(bpc));
  g->blocks = per_cu * g->cus;
  fc_status s2 = fcd::ensure_queries(g, 1024);
  if (s2 != FC_OK) return bail(s2);
  // the uploads and clears above are ordered on the graph's stream only:
  // finish them before any other stream (a batch lane's) can touch the graph
  CK(hipStreamSynchronize(g->stream));
  g->symmetric = g->h_phase[0] == 0 && g->h_phase[1] == 0;
#undef CK
  {
    std::lock_guard<std::mutex> lock(fcd::graphs().mu);
    fcd::graphs().all.push_back(g);
  }
  *out = g;
  return FC_OK;
}

// For tests on hosts without a GPU.
extern "C" int32_t fcd_visit_width(int32_t asked) { return fcd::visit_width(asked); }
extern "C" int32_t fcd_query_set(int32_t q) { return fcd::query_set(q); }
extern "C" int32_t fcd_team_admit(uint32_t k, uint32_t expected) { return fcd::team_admit(k, expected); }

extern "C" fc_status fc_graph_create_csr32(const int32_t* off, const int32_t* col, int32_t V, int64_t E,
                                           uint32_t flags, fc_graph** out) {
  return graph_create<int32_t>(off, col, V, E, flags, out);
}

extern "C" fc_status fc_graph_create_csr64(const int64_t* off, const int32_t* col, int64_t V, int64_t E,
                                           uint32_t flags, fc_graph** out) {
  return graph_create<int64_t>(off, col, V, E, flags, out);
}

extern "C" fc_status fc_graph_destroy(fc_graph* g) {
  if (!g) return FC_OK;
  fcd::graphs_remove(g);
  if (g->stream) (void)hipStreamSynchronize(g->stream);
  fcd::batch_free(g->batch);
  fcd::team_free(g->team);
  fcd::st_teams_free(g->st_teams);
  if (g->gexec) (void)hipGraphExecDestroy(g->gexec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  if (g->h_out) (void)hipHostFree(g->h_out);
  if (g->h_phase) (void)hipHostFree(g->h_phase);
  (void)hipFree(g->d_qs);
  (void)hipFree(g->d_qt);
  if (g->h_stage) (void)hipHostFree(g->h_stage);
  (void)hipFree(g->d_mlp);
  (void)hipFree(g->d_ws);
  (void)hipFree(g->d_col);
  (void)hipFree(g->d_head);
  (void)hipFree(g->d_off);
  (void)hipFree(g->d_perm);
  (void)hipFree(g->d_iperm);
  (void)hipFree(g->d_lv_out);
  (void)hipFree(g->d_par_out);
  if (g->ev0) (void)hipEventDestroy(g->ev0);
  if (g->ev1) (void)hipEventDestroy(g->ev1);
  if (g->stream) (void)hipStreamDestroy(g->stream);
  delete g;
  return FC_OK;
}

// Copy device results to the caller on the graph's stream. The graph's
// streams do not wait for the legacy null stream, so no plain hipMemcpy or
// hipMemset touches its memory.
static hipError_t read_back(void* dst, const void* src, size_t bytes, fc_graph* g) {
  hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g->stream);
  if (e != hipSuccess) return e;
  return hipStreamSynchronize(g->stream);
}

static void add_stats(const fcd::VisitOut& o, fc_stats* s) {
  s->levels += o.levels;
  s->depth += o.depth;
  s->visited_vertices += o.visited_vertices;
  s->visited_edges += o.visited_edges;
  s->expanded_vertices += o.expanded_vertices;
  s->expanded_edges += o.expanded_edges;
  s->topdown_levels += o.topdown;
  s->bottomup_levels += o.bottomup;
  s->max_frontier = std::max(s->max_frontier, o.max_frontier);
  s->launches += o.launches;
}

static fc_status check_out(const fcd::VisitOut& o) {
  if (o.status != 0) return fail(FC_ERR_CAPACITY, "visit kernel: frontier guard tripped (err=%d)", o.err);
  return FC_OK;
}

// Levels (and parents) of a BFS on a relabelled graph back in caller ids:
// out[v] = lv[perm[v]], parents mapped through iperm. One coalesced pass.
// Levels and parents back in caller ids. A BFS writes state and parent only
// for the vertices it reaches; the visited bitmap says which those are.
__global__ void unpermute_kernel(const int32_t* __restrict__ perm, const int32_t* __restrict__ iperm,
                                 const uint32_t* __restrict__ reached, const int32_t* __restrict__ lv,
                                 const int32_t* __restrict__ par, int32_t* __restrict__ lv_out,
                                 int32_t* __restrict__ par_out, int64_t V) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += stride) {
    const int32_t k = perm[v];
    const bool r = (reached[(uint32_t)k >> 5] >> (k & 31)) & 1u;
    lv_out[v] = r ? lv[k] : -1;
    if (par) {
      const int32_t q = r ? par[k] : -1;
      par_out[v] = (uint32_t)q < (uint32_t)V ? iperm[q] : q;
    }
  }
}

extern "C" fc_status fc_bfs(fc_graph* g, int32_t src, int32_t* levels_out, int32_t* parents_out, fc_stats* stats) {
  fc::clear_error();
  if (!g) return fail(FC_ERR_INVALID, "fc_bfs: null graph");
  if (src < 0 || src >= g->V) return fail(FC_ERR_INVALID, "fc_bfs: source %d out of range [0,%lld)", src, (long long)g->V);
  const bool par = parents_out != nullptr;
  const int32_t none = -1;
  const int32_t dsrc = g->relabeled ? g->h_perm[(size_t)src] : src;
  double ms = 0, tried = 0;
  g->levels_valid = g->parents_valid = false;
  const size_t bytes = sizeof(int32_t) * (size_t)g->V;
  if (g->relabeled && !g->d_lv_out) FC_HIP(fcd::dev_malloc((void**)&g->d_lv_out, bytes));
  if (g->relabeled && par && !g->d_par_out) FC_HIP(fcd::dev_malloc((void**)&g->d_par_out, bytes));
  int32_t* const lv = g->relabeled ? g->d_lv_out : g->d_state;
  int32_t* const pa = g->relabeled ? g->d_par_out : g->d_parent;
  // small results come back behind the visit, through pinned memory
  const int results = (levels_out ? 1 : 0) + (par ? 1 : 0);
  const bool staged = results > 0 && bytes * (size_t)results <= fcd::kStageBytes;
  if (staged && !g->h_stage) FC_HIP(hipHostMalloc((void**)&g->h_stage, fcd::kStageBytes, hipHostMallocDefault));
  fcd::VisitTail tail, after;
  if (g->relabeled)  // the results in caller ids are part of the BFS: timed with it
    tail = [&]() {
      const int blocks = (int)std::min<int64_t>((g->V + 255) / 256, (int64_t)g->cus * 8);
      hipLaunchKernelGGL(unpermute_kernel, dim3(blocks), dim3(256), 0, g->stream, g->d_perm, g->d_iperm, g->d_visited,
                         g->d_state, par ? g->d_parent : nullptr, g->d_lv_out, g->d_par_out, (int64_t)g->V);
      return hipGetLastError();
    };
  if (staged)
    after = [&]() {
      hipError_t e = hipSuccess;
      if (levels_out) e = hipMemcpyAsync(g->h_stage, lv, bytes, hipMemcpyDeviceToHost, g->stream);
      if (par && e == hipSuccess)
        e = hipMemcpyAsync(g->h_stage + (levels_out ? bytes : 0), pa, bytes, hipMemcpyDeviceToHost, g->stream);
      return e;
    };
  bool narrow = false;
  fc_status st;
  if (g->use_st_teams && g->narrow && g->narrow_bfs) {
    if ((st = fcd::ensure_queries(g, 1)) != FC_OK) return st;
    st = fcd::st_teams_run(g, &dsrc, &none, 1, true, true, lv, par ? pa : nullptr, &ms, &narrow, after);
    if (st != FC_OK) return st;
    if (narrow && g->h_out[0].status == fcd::kTooWide) {
      narrow = g->narrow_bfs = false;
      tried = ms;
    }
  }
  if (!narrow) {
    st = fcd::run_visits(g, fcd::kModeBfs, &dsrc, &none, 1, par, &ms, tail, after);
    if (st != FC_OK) return st;
    ms += tried;
  }
  const fcd::VisitOut o = g->h_out[0];
  st = check_out(o);
  if (st != FC_OK) return st;
  g->levels_valid = true;
  g->parents_valid = par;
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->time_ms = ms;
    add_stats(o, stats);
  }
  if (staged) {
    if (levels_out) std::memcpy(levels_out, g->h_stage, bytes);
    if (parents_out) std::memcpy(parents_out, g->h_stage + (levels_out ? bytes : 0), bytes);
    return FC_OK;
  }
  if (levels_out) FC_HIP(read_back(levels_out, lv, bytes, g));
  if (parents_out) FC_HIP(read_back(parents_out, pa, bytes, g));
  return FC_OK;
}

extern "C" fc_status fc_graph_levels(fc_graph* g, int32_t* levels_out) {
  fc::clear_error();
  if (!g || !levels_out) return fail(FC_ERR_INVALID, "fc_graph_levels: null argument");
  if (!g->levels_valid) return fail(FC_ERR_INVALID, "fc_graph_levels: no BFS result on the device");
  const int32_t* lv = g->relabeled ? g->d_lv_out : g->d_state;
  FC_HIP(read_back(levels_out, lv, sizeof(int32_t) * (size_t)g->V, g));
  return FC_OK;
}

extern "C" fc_status fc_graph_parents(fc_graph* g, int32_t* parents_out) {
  fc::clear_error();
  if (!g || !parents_out) return fail(FC_ERR_INVALID, "fc_graph_parents: null argument");
  if (!g->parents_valid) return fail(FC_ERR_INVALID, "fc_graph_parents: the last BFS did not record parents");
  const int32_t* pa = g->relabeled ? g->d_par_out : g->d_parent;
  FC_HIP(read_back(parents_out, pa, sizeof(int32_t) * (size_t)g->V, g));
  return FC_OK;
}

static fc_status stcon_run(fc_graph* g, const int32_t* s, const int32_t* t, int32_t n, int32_t* connected,
                           int32_t* dist, int32_t* meet, fc_stats* stats) {
  fc::clear_error();
  if (!g || (n > 0 && (!s || !t))) return fail(FC_ERR_INVALID, "s–t query: null argument");
  if (n < 0) return fail(FC_ERR_INVALID, "s–t query: negative count");
  for (int32_t i = 0; i < n; ++i)
    if (s[i] < 0 || s[i] >= g->V || t[i] < 0 || t[i] >= g->V)
      return fail(FC_ERR_INVALID, "s–t query %d: vertex out of range [0,%lld)", i, (long long)g->V);
  g->levels_valid = g->parents_valid = false;
  // s == t needs no visit: distance 0.
  std::vector<int32_t> vs, vt, idx;
  vs.reserve(n);
  vt.reserve(n);
  idx.reserve(n);
  for (int32_t i = 0; i < n; ++i)
    if (s[i] != t[i]) {
      vs.push_back(g->relabeled ? g->h_perm[(size_t)s[i]] : s[i]);
      vt.push_back(g->relabeled ? g->h_perm[(size_t)t[i]] : t[i]);
      idx.push_back(i);
    }
  double ms = 0;
  fc_status st = fcd::run_visits(g, fcd::kModePlainSt, vs.data(), vt.data(), (int32_t)vs.size(), false, &ms);
  if (st != FC_OK) return st;
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->time_ms = ms;
  }
  for (int32_t i = 0; i < n; ++i) {
    if (connected) connected[i] = 1;
    if (dist) dist[i] = 0;
    if (meet) meet[i] = s[i];
  }
  for (size_t k = 0; k < idx.size(); ++k) {
    const fcd::VisitOut o = g->h_out[k];
    st = check_out(o);
    if (st != FC_OK) return st;
    const int32_t i = idx[k];
    if (connected) connected[i] = o.dist >= 0 ? 1 : 0;
    if (dist) dist[i] = o.dist;
    if (meet) meet[i] = (g->relabeled && (uint32_t)o.meet < (uint32_t)g->V) ? g->h_iperm[(size_t)o.meet] : o.meet;
    if (stats) add_stats(o, stats);
  }
  return FC_OK;
}

extern "C" fc_status fc_stcon(fc_graph* g, int32_t s, int32_t t, int32_t* connected, int32_t* dist, int32_t* meet,
                              fc_stats* stats) {
  return stcon_run(g, &s, &t, 1, connected, dist, meet, stats);
}

extern "C" fc_status fc_stcon_many(fc_graph* g, const int32_t* s, const int32_t* t, int32_t n, int32_t* connected,
                                   int32_t* dist, fc_stats* stats) {
  return stcon_run(g, s, t, n, connected, dist, nullptr, stats);
}

// Shortest s–t path from the parents a plain visit recorded (one wave).
// The meeting vertex u has level lu in its own colour's tree; the other end
// of the meeting edge is a neighbour w of u of the other colour at level
// dist - 1 - lu. The lanes search u's adjacency for w; lane 0 then walks
// both parent chains (a root is its own parent) and writes the path, s
// first, into out[0..dist]. *status receives dist + 1, or a negative code:
// -1 no such neighbour, -2 a chain left the vertex range, -3 a chain did not
// end at a root.
template <typename OffT>
__global__ void path_kernel(const OffT* __restrict__ off, const int32_t* __restrict__ col,
                            const unsigned long long* __restrict__ sst, uint32_t epoch,
                            const int32_t* __restrict__ parent, int32_t V, int32_t u, int32_t dist,
                            int32_t* __restrict__ out, int32_t* __restrict__ status) {
  using namespace fcd;
  const int lane = lane_id();
  const unsigned long long wu = sst[u];
  const int32_t su = (int32_t)(uint32_t)wu;
  const bool tu = (su & kColorBit) != 0;  // u on the t side
  const int32_t lu = su & kLevelMask;
  const int32_t want = dist - 1 - lu;
  int32_t w = -1;
  const OffT e1 = off[u + 1];
  for (OffT b = off[u]; b < e1; b += kWave) {
    const OffT e = b + (OffT)lane;
    int32_t x = -1;
    bool hit = false;
    if (e < e1) {
      x = col[e];
      const unsigned long long wx = sst[x];
      const int32_t sx = (int32_t)(uint32_t)wx;
      hit = (uint32_t)(wx >> 32) == epoch && (((sx & kColorBit) != 0) != tu) && (sx & kLevelMask) == want;
    }
    const uint64_t m = ballot(hit);
    if (m) {
      w = __shfl(x, __ffsll((unsigned long long)m) - 1);
      break;
    }
  }
  if (lane != 0) return;
  if (w < 0 || want < 0 || (uint32_t)(wu >> 32) != epoch) {
    *status = -1;
    return;
  }
  const int32_t a = tu ? w : u, b = tu ? u : w;  // s-side and t-side ends
  const int32_t la = tu ? want : lu;             // level of a from s
  int32_t x = a;
  for (int32_t k = la; k >= 0; --k) {
    if ((uint32_t)x >= (uint32_t)V) {
      *status = -2;
      return;
    }
    out[k] = x;
    x = parent[x];
  }
  if (x != out[0]) {  // out[0] must be the s root, its own parent
    *status = -3;
    return;
  }
  x = b;
  for (int32_t k = la + 1; k <= dist; ++k) {
    if ((uint32_t)x >= (uint32_t)V) {
      *status = -2;
      return;
    }
    out[k] = x;
    x = parent[x];
  }
  if (x != out[dist]) {  // out[dist] must be the t root
    *status = -3;
    return;
  }
  *status = dist + 1;
}

extern "C" fc_status fc_stcon_path(fc_graph* g, int32_t s, int32_t t, int32_t* path_out, int32_t cap, int32_t* len_out,
                                   fc_stats* stats) {
  fc::clear_error();
  if (!g || !len_out || (cap > 0 && !path_out)) return fail(FC_ERR_INVALID, "fc_stcon_path: null argument");
  if (s < 0 || s >= g->V || t < 0 || t >= g->V)
    return fail(FC_ERR_INVALID, "fc_stcon_path: vertex out of range [0,%lld)", (long long)g->V);
  g->levels_valid = g->parents_valid = false;
  if (stats) std::memset(stats, 0, sizeof(*stats));
  *len_out = 0;
  if (s == t) {
    *len_out = 1;
    if (cap < 1) return fail(FC_ERR_CAPACITY, "fc_stcon_path: the path needs 1 entry, cap is %d", cap);
    path_out[0] = s;
    return FC_OK;
  }
  const int32_t ds = g->relabeled ? g->h_perm[(size_t)s] : s;
  const int32_t dt = g->relabeled ? g->h_perm[(size_t)t] : t;
  double ms = 0;
  fc_status st = fcd::run_visits(g, fcd::kModePlainSt, &ds, &dt, 1, true, &ms);
  if (st != FC_OK) return st;
  const uint32_t epoch = g->epoch_next - 1;  // the query's tag in the state words
  const fcd::VisitOut o = g->h_out[0];
  st = check_out(o);
  if (st != FC_OK) return st;
  if (stats) {
    stats->time_ms = ms;
    add_stats(o, stats);
  }
  if (o.dist < 0) return FC_OK;
  *len_out = o.dist + 1;
  if (o.dist + 1 > cap)
    return fail(FC_ERR_CAPACITY, "fc_stcon_path: the path needs %d entries, cap is %d", o.dist + 1, cap);
  if ((uint32_t)o.meet >= (uint32_t)g->V || o.dist + 1 > g->V)
    return fail(FC_ERR_CAPACITY, "fc_stcon_path: visit returned meet %d at distance %d", o.meet, o.dist);
  // The frontier queues are idle after the visit: the path goes to the
  // first, the status word to the second.
  int32_t* d_path = g->d_q[0][0];
  int32_t* d_status = g->d_q[1][0];
  FC_HIP(hipEventRecord(g->ev0, g->stream));
  if (g->off64)
    hipLaunchKernelGGL(path_kernel<int64_t>, dim3(1), dim3(fcd::kWave), 0, g->stream, (const int64_t*)g->d_off,
                       g->d_col, g->d_sst, epoch, g->d_parent, (int32_t)g->V, o.meet, o.dist, d_path, d_status);
  else
    hipLaunchKernelGGL(path_kernel<int32_t>, dim3(1), dim3(fcd::kWave), 0, g->stream, (const int32_t*)g->d_off,
                       g->d_col, g->d_sst, epoch, g->d_parent, (int32_t)g->V, o.meet, o.dist, d_path, d_status);
  FC_HIP(hipGetLastError());
  FC_HIP(hipEventRecord(g->ev1, g->stream));
  int32_t status = 0;
  FC_HIP(hipMemcpyAsync(&status, d_status, sizeof(int32_t), hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipMemcpyAsync(path_out, d_path, sizeof(int32_t) * (size_t)(o.dist + 1), hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipStreamSynchronize(g->stream));
  float pms = 0.f;
  FC_HIP(hipEventElapsedTime(&pms, g->ev0, g->ev1));
  if (stats) stats->time_ms += pms;
  if (status != o.dist + 1) return fail(FC_ERR_HIP, "fc_stcon_path: path assembly failed (code %d)", status);
  if (g->relabeled)
    for (int32_t k = 0; k <= o.dist; ++k) path_out[k] = g->h_iperm[(size_t)path_out[k]];
  if (path_out[0] != s || path_out[o.dist] != t)
    return fail(FC_ERR_HIP, "fc_stcon_path: assembled path runs %d..%d", path_out[0], path_out[o.dist]);
  return FC_OK;
}

// validate_stcon_bfs (st-conn/make_stcon.c:1578-1641) on one GPU: the BFS
// from mn runs on the device, the parent walks on the host.
extern "C" fc_status fc_validate_stcon(fc_graph* g, int32_t s, int32_t t, int32_t mn, int32_t depth) {
  fc::clear_error();
  if (!g) return fail(FC_ERR_INVALID, "fc_validate_stcon: null graph");
  if (s < 0 || s >= g->V || t < 0 || t >= g->V || mn < 0 || mn >= g->V)
    return fail(FC_ERR_INVALID, "fc_validate_stcon: vertex out of range [0,%lld)", (long long)g->V);
  std::vector<int32_t> lv((size_t)g->V), par((size_t)g->V);
  fc_status st = fc_bfs(g, mn, lv.data(), par.data(), nullptr);
  if (st != FC_OK) return st;
  int32_t dep[2] = {-1, -1};
  const int32_t from[2] = {t, s};  // blue path first, as the reference
  for (int k = 0; k < 2; ++k) {
    int32_t v = from[k], p = v;
    int64_t steps = -1;
    do {
      v = p;
      if (v < 0 || v >= g->V) return fail(FC_ERR_MISMATCH, "%s path leaves the graph", k ? "RED" : "BLUE");
      p = par[(size_t)v];
      ++steps;
    } while (v != p && steps <= g->V);
    if (v != mn)
      return fail(FC_ERR_MISMATCH, "WRONG MATCHING NODE: %s Path leaf = %d, Matching Node = %d", k ? "RED" : "BLUE", v,
                  mn);
    dep[k] = (int32_t)steps;
    if (steps > depth)
      return fail(FC_ERR_MISMATCH, "WRONG ST-CON depth on %s: ST-CON depth = %d, bfs depth = %d", k ? "RED" : "BLUE",
                  depth, dep[k]);
  }
  const int32_t mx = std::max(dep[0], dep[1]);
  if (mx != depth)
    return fail(FC_ERR_MISMATCH, "WRONG ST-CON MAX depth: ST-CON MAX depth = %d, bfs MAX depth = %d", depth, mx);
  return FC_OK;
}

extern "C" fc_status fc_stcon_sched_many(fc_graph* g, const int32_t* s, const int32_t* t, int32_t n, int32_t policy,
                                         int32_t* connected, int32_t* dist, fc_stats* stats) {
  if (policy == FC_POLICY_PLAIN) return fc_stcon_many(g, s, t, n, connected, dist, stats);
  if (policy != FC_POLICY_HEURISTIC && policy != FC_POLICY_LEARNED)
    return fail(FC_ERR_INVALID, "unknown policy %d", policy);
  // One-sided scheduled steps for single queries are not built: an earlier
  // persistent-kernel version of this path waited out its grid-barrier
  // bound on the GPU, that cause was not identified, and the code was
  // removed. Heuristic and learned scheduling run in the batched engine.
  return fail(FC_ERR_UNSUPPORTED,
              "scheduled single-query visits are switched off; use fc_stcon_batch for heuristic or "
              "learned scheduling");
}
