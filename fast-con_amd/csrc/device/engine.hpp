// Internal definition of fc_graph: the device copy of one CSR graph, its HIP
// stream, and all per-query workspace, allocated once at creation.
#pragma once

#include <atomic>
#include <functional>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "fastcon.h"
#include "visit.hpp"

namespace fcd {
struct BatchWorkspace;
struct TeamWorkspace;
struct StTeams;
}

struct fc_graph {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  int64_t V = 0, E = 0;
  bool off64 = false;
  void* d_off = nullptr;
  int32_t* d_col = nullptr;
  unsigned long long* d_head = nullptr;  // VisitParams::head
  int cus = 0;
  int blocks = 0;               // cooperative grid of the visit kernel
  int32_t hub_threshold = 4096;
  bool symmetric = false;       // every edge is stored in both directions (checked by hash sums)
  bool hub_steps = false;       // the top vertices are on enough edges for hub steps
  double branch = 0.0;          // sum d^2 / sum d: the mean degree of a vertex reached over an edge
  bool regular = false;         // degrees hardly differ: a grid, a mesh
  double surface = 0.0;         // regular: edges on the surface of a ball half the graph wide, as expected
  bool skewed = false;          // branch is several mean degrees: hubs
  float f_branch = 0.f;         // scheduler feature: log2(1 + branch) / 16
  uint32_t hcap = 1;
  uint32_t qcap = 1;

  // Visit workspace: one allocation.
  char* d_ws = nullptr;
  size_t ws_bytes = 0;
  int32_t* d_state = nullptr;
  unsigned long long* d_sst = nullptr;  // s–t state words: (epoch << 32) | colour | level
  uint32_t epoch_next = 1;              // epoch of the next s–t query (0 = never visited)
  int32_t* d_parent = nullptr;
  uint32_t* d_visited = nullptr;
  uint32_t* d_fbm[2][3] = {};
  int32_t* d_q[2][2] = {};
  int32_t* d_hq[2][2] = {};
  int64_t* d_hb[2][2] = {};
  fcd::VisitCtl* d_ctl = nullptr;

  // Query lists of the phase machine (device) and its results (pinned host
  // memory); capacity q_cap.
  int32_t* d_qs = nullptr;
  int32_t* d_qt = nullptr;
  fcd::VisitOut* h_out = nullptr;   // pinned; the visits' launches write it
  char* h_stage = nullptr;          // pinned: small read-backs (kStageBytes)
  int32_t q_cap = 0;
  int32_t* h_phase = nullptr;       // pinned: small words read back
  // Captured hipGraph of kGraphLaunches identical phase launches.
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  double est_launches[2] = {10.0, 3.0};  // working launches per query (running estimate, per mode)
  int32_t vw_fixed = 0;
  bool use_graphs = true;           // replay captured launches (FASTCON_PLAIN_GRAPHS=0: direct launches)

  // Degree relabelling (absent with FC_GRAPH_KEEP_IDS): the device graph
  // uses new ids; perm maps a caller id to its device id, iperm back.
  bool relabeled = false;
  bool lists_sorted = false;  // device adjacency lists in ascending id order (renumbered, not FC_GRAPH_KEEP_ORDER)
  int64_t v_active = 0;  // vertices [0, v_active) have degree > 0: the degree-ordered
                         // numbering puts every isolated vertex after them; V otherwise
  int32_t* d_perm = nullptr;
  int32_t* d_iperm = nullptr;
  std::vector<int32_t> h_perm, h_iperm;
  // The last BFS's levels and parents in caller ids (relabelled graphs).
  int32_t* d_lv_out = nullptr;
  int32_t* d_par_out = nullptr;

  bool parents_valid = false;
  bool levels_valid = false;
  float* d_mlp = nullptr;           // scheduler parameters (device): canonical, then in mlp_t_index order
  bool mlp_set = false;
  std::vector<float> h_mlp;

  fcd::BatchWorkspace* batch = nullptr;
  fcd::TeamWorkspace* team = nullptr;
  fcd::StTeams* st_teams = nullptr;  // plain s–t queries by teams (allocated on first use)
  bool use_st_teams = true;          // FASTCON_PLAIN_TEAMS=0: every visit through the launches
  bool narrow = false;               // even degrees: visits are likely to stay narrow (narrow_kernel)
  bool narrow_st = true, narrow_bfs = true;  // until one did not
  bool st_limit = true;              // wide levels are left to the whole GPU (kTeamLevelEdges), until most queries had one
  std::atomic<int> team_use{0};      // calls that use the two workspaces above; -1: they are being given back
};

namespace fcd {

constexpr int kGraphLaunches = 16;
constexpr int64_t kPollLaunches = 4096;  // launches queued between two looks of the host at the results

fc_status hip_fail(hipError_t e, const char* what);

// Device memory. The teams' workspaces (team, st_teams) are the one part of a
// graph that it can do without: when memory runs out, those of every graph on
// the device whose teams are not at work are given back and the allocation is
// tried again. Their owners allocate them anew when they next fit.
hipError_t dev_malloc(void** p, size_t bytes);
// What a graph's next teams may take: an eighth of the device's memory, and no
// more than a quarter of what is free.
size_t team_budget(size_t total);
// Held while a call uses its graph's team workspaces.
struct TeamUse {
  fc_graph* g;
  explicit TeamUse(fc_graph* g_);
  ~TeamUse() { g->team_use.fetch_sub(1); }
  TeamUse(const TeamUse&) = delete;
  TeamUse& operator=(const TeamUse&) = delete;
};
fc_status ensure_queries(fc_graph* g, int32_t n);

// Run n visits through the phase machine (s[i], t[i]; t = -1 for BFS) and
// leave their results in g->h_out[0..n). *ms receives the device time. tail:
// work to queue behind the visits, part of that time (and queued again if they
// needed more launches than expected); after: read-backs behind that.
typedef std::function<hipError_t()> VisitTail;
fc_status run_visits(fc_graph* g, int mode, const int32_t* s, const int32_t* t, int32_t n, bool parents,
                     double* ms, const VisitTail& tail = {}, const VisitTail& after = {});
constexpr size_t kStageBytes = 1u << 20;
constexpr int kStartPairs = 32;

// One launch of the visit kernel on the control block ctl (which carries the
// launch parameters); launches alternate parity 0, 1, 0, ...
template <typename OffT>
hipError_t launch_phase(VisitCtl* ctl, int parity, int blocks, bool wide, hipStream_t s);

// Control block for a run of n queries: s–t queries start directly in their
// level phase (query i has epoch epoch0 + i), a BFS starts with its reset.
template <typename OffT>
inline VisitCtl visit_init(const VisitParams<OffT>& prm, int mode, int32_t n, const int32_t* s, const int32_t* t,
                           uint32_t epoch0, int vw_fixed, bool parents) {
  VisitCtl c;
  std::memset(&c, 0, sizeof(c));
  std::memcpy(c.params, &prm, sizeof(prm));
  VisitState& st = c.st[0];
  st.phase = mode == kModeBfs ? kPhaseReset : kPhaseLevel;
  st.qi = 0;
  st.src = s[0];
  st.dst = t[0];
  st.nsrc = st.ndst = -1;
  st.epoch = epoch0;
  for (auto& b : c.best) b[0] = b[1] = ~0ull;
  c.nq = n;
  c.mode = mode;
  c.vw_fixed = vw_fixed;
  c.record_parents = parents ? 1 : 0;
  return c;
}
template <typename OffT>
int phase_occupancy();
template <typename OffT>
hipError_t launch_st_team(const StTeamRun& tr, int blocks, hipStream_t s);
template <typename OffT>
int st_team_occupancy();
template <typename OffT>
hipError_t launch_narrow(const StTeamRun& tr, bool bfs, int blocks, hipStream_t s);
template <typename OffT>
int narrow_occupancy();

void batch_free(BatchWorkspace* b);
void team_free(TeamWorkspace* w);
void st_teams_free(StTeams* w);

}  // namespace fcd

#define FC_HIP(call)                                              \
  do {                                                            \
    hipError_t _e = (call);                                       \
    if (_e != hipSuccess) return fcd::hip_fail(_e, #call);        \
  } while (0)
