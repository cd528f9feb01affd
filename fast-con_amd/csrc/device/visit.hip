// Visit engines for BFS and s–t connectivity on gfx950. Three kernels run the
// same expansion and claims:
//  * phase_kernel: one launch per level over the whole GPU, driven by a
//    device-side phase machine in VisitCtl (BFS of wide frontiers, single
//    queries, path output);
//  * st_team_kernel: one launch for a list of plain queries, eight at a time,
//    one per XCD (team.hpp);
//  * narrow_kernel: one launch for a BFS or queries whose frontiers stay
//    narrow over many levels, by one team each.
//
// Why launches where the whole GPU works on a level: a grid-wide software
// barrier with the agent-scope release/acquire that cross-XCD visibility
// needs costs 16-35 us, a cooperative launch ~20 us, while a back-to-back
// ordinary launch costs ~2.4 us (1.6 us inside a hipGraph) and its boundary
// already orders every block's writes. Inside one XCD a barrier costs 0.6 us,
// which is what the other two build on. The launch per level replaces the
// reference's host-driven level loop with a
// 16-byte readback per level (BFS-4K/src/device/BFS_WorkEfficient.cu:81-118)
// and ST-CON's ~12 host round trips per level (st-conn/make_stcon.c:968-1187).
//
// No block votes and no block finalises. Every block loads the 1 KB control
// block at the start of a launch (one 16-byte load per lane of one wave) and
// derives the same step from it: whether the query is finished (met, empty
// frontier, error), the direction and the virtual-warp width. Block 0 writes
// the machine state of the next launch into the other half of a buffer
// indexed by launch parity, which no block of this launch reads, and writes
// the results of a finished query. A level's critical path is therefore the
// level's own memory traffic, with no atomic ticket and no serial chain of
// loads by a finalising block after it. The price is that a query's end is
// noticed at the start of the launch after its last level: an s–t query
// spends that launch expanding the next query's roots, so n queries of d
// levels cost n*d + 1 launches.
//
// s–t state words are 64-bit: (epoch << 32) | colour | level, and a word of
// another epoch is an unvisited vertex. Each query has its own epoch, so no
// query clears the state array: the next query starts in the same launch
// that sees the last one finish. Its roots are never claimed through the
// array; a probe that reaches the other colour's root proposes a meeting at
// the root's level 0.
//
// Frontier expansion (per colour, per level):
//  * top-down: normal-queue vertices are expanded by virtual warps of VW lanes
//    (4..64, from the frontier's average degree): the reference's
//    BFS_KernelMainGLOB + EdgeVisit (BFS-4K/src/device/WorkEfficientKernel/BFS_WE_KernelMain.cu:2-53,
//    BFS_WE_Kernels1.cu:44-74) rebuilt for 64-lane waves. Vertices of degree >=
//    hub_threshold are routed at claim time to a hub queue whose concatenated
//    adjacency is cut into chunks spread over the whole grid: the device-side
//    work queue that replaces the dynamic-parallelism child grids
//    (BFS-4K/src/device/WorkEfficientKernel/BFS_WE_Dynamic.cu:4-50).
//  * bottom-up (BFS): each wave owns 64 vertices; unvisited ones look for a
//    parent in the current frontier bitmap (direction-optimising BFS,
//    Beamer et al. SC'12).
// Frontier slots are reserved through LDS stages, one atomic per block, the
// in-house replacement of FrontierWrite::Write (BFS-4K/src/device/Util/GlobalWrite.cu:49-105)
// and of ST-CON's Thrust exclusive_scan / remove_copy compaction
// (st-conn/mythrustlib.cu:25-34,175-185), which cost O(V) per level.
//
// s–t claims take ONE atomicCAS per vertex (ST-CON k_stcon_binary_mask_unique_large,
// st-conn/cudakernel/stcon_kernel.cu:128-196). A CAS (or read) that shows the
// other colour is a meeting edge (v,u) and proposes the path length
// level(v)+1+level(u); the query ends after the level in which the first
// proposal appears, and the minimum proposal is the exact distance.
#include "visit.hpp"
#include "hubstage.hpp"
#include "team.hpp"

#include <hip/hip_runtime.h>

namespace fcd {

template <typename OffT>
__device__ __forceinline__ OffT bcast_off(OffT v, int src) {
  return sizeof(OffT) == 4 ? (OffT)bcast((int32_t)v, src) : (OffT)bcast64((int64_t)v, src);
}

__device__ __forceinline__ bool test_bit(const uint32_t* bm, int32_t v) {
  return (bm[v >> 5] >> (v & 31)) & 1u;
}

// Loads of the workspace, which this launch writes: in a team other blocks may
// have written the word earlier in the same launch (team.hpp).
template <bool TEAM, typename T>
__device__ __forceinline__ T ldw(const T* q) {
  return TEAM ? ld_team(q) : *q;
}

// Next-frontier appender of one wave. Normal-queue entries are staged in
// this wave's LDS buffer; a full buffer is published by the wave with one
// atomic, and at the end of the level the whole block publishes its buffers,
// degree sums and best meeting candidate with one atomic each. A single
// frontier counter hit by every wave-iteration was the bottleneck of large
// levels (a contended word sustains only tens of millions of atomics/s).
constexpr uint32_t kStageCap = 1024;

template <typename OffT>
struct Appender {
  const VisitParams<OffT>* p;
  int c;
  int nxt_par;
  Ring* nxt;
  uint32_t* nfbm;
  unsigned long long* best_out;  // the query's best meeting candidate (device)
  bool bitmaps;                 // keep the visited and frontier bitmaps (BFS: bottom-up levels may follow)
  uint32_t epoch;               // s–t: tag of the current query
  int32_t root_own, root_other; // s–t: this colour's root and the other colour's
  int32_t* buf;                 // this wave's LDS stage, kStageCap entries
  uint32_t cnt;                 // staged entries (wave-uniform)
  uint64_t mf;                  // per-lane degree sum of claimed vertices
  unsigned long long best;      // per-lane best meeting candidate (distance << 32 | vertex)
  HubStage h;                   // this wave's staged hub entries
};

template <typename OffT>
__device__ __forceinline__ void wave_flush(Appender<OffT>& a) {
  if (a.cnt == 0) return;
  __builtin_amdgcn_wave_barrier();
  uint32_t base = 0;
  if (lane_id() == 0) base = atomicAdd(&a.nxt->n, a.cnt);
  base = (uint32_t)__shfl((int)base, 0);
  int32_t* q = a.p->q[a.c][a.nxt_par];
  for (uint32_t i = (uint32_t)lane_id(); i < a.cnt; i += kWave) {
    const uint32_t slot = base + i;
    if (slot < a.p->qcap)
      q[slot] = a.buf[i];
    else
      atomicOr(&a.p->ctl->err, 1u);
  }
  __builtin_amdgcn_wave_barrier();
  a.cnt = 0;
}

// Wave-collective: add every claimed vertex (degree deg) to the next frontier
// of the appender's colour: normal entries and hub entries (degree >=
// hub_threshold) through their LDS stages. A per-lane atomic on the one hub
// counter serialised whole levels when thousands of hubs were claimed.
template <typename OffT>
__device__ __forceinline__ void push_next(Appender<OffT>& a, bool claimed, int32_t u, int64_t deg, bool set_bitmap) {
  const VisitParams<OffT>& p = *a.p;
  const bool hub = claimed && deg >= p.hub_threshold;
  const bool norm = claimed && !hub;
  const uint64_t m = ballot(norm);
  if (m) {
    const uint32_t k = (uint32_t)__popcll(m);
    if (a.cnt + k > kStageCap) wave_flush(a);
    if (norm) a.buf[a.cnt + lane_rank(m)] = u;
    a.cnt += k;
  }
  hub_push(a.h, hub, u, deg, (unsigned long long*)&a.nxt->hub, p.hq[a.c][a.nxt_par], p.hb[a.c][a.nxt_par], p.hcap,
           &p.ctl->err);
  if (claimed) {
    a.mf += (uint64_t)deg;
    if (set_bitmap) atomicOr(a.nfbm + (u >> 5), 1u << (u & 31));
  }
}

// Block-collective publication of both colours' staged entries (all threads,
// uniform control flow, at the end of the level). One barrier publishes every
// wave's counts; then four waves each take one list with one atomic, at the
// same time: wave 0 colour 0's normal list (with its degree sum and best
// meeting candidate), wave 1 colour 1's, waves 2 and 3 the two hub lists;
// after a second barrier every wave writes its entries.
template <int W>  // waves of the block
struct BlockShared {
  uint32_t cnt[2][W];
  unsigned long long mf[2][W];
  unsigned long long best[2][W];
  uint32_t hcnt[2][W];
  unsigned long long hedges[2][W];
  uint32_t base[2];
  unsigned long long hbase[2];
};

template <int W, typename OffT>
__device__ __forceinline__ void block_flush(Appender<OffT>& a, int ncol, BlockShared<W>& sh, Ring* nxt0, Ring* nxt1) {
  static_assert(W >= 4, "one publishing wave per list");
  const int w = (int)(threadIdx.x >> 6);
  const int lane = lane_id();
  const int own = a.c;  // this wave staged entries of its own colour only
  {
    const unsigned long long mf = (unsigned long long)wave_reduce_full_nz_u64<kWaveSum>(a.mf);
    const unsigned long long best = wave_reduce_full_nz_u64<kWaveMin>(a.best);
    const unsigned long long hd =
        wave_reduce_full_nz_u64<kWaveSum>((uint32_t)lane < a.h.cnt ? (unsigned long long)a.h.d[lane] : 0ull);
    if (lane == 0) {
      sh.cnt[own][w] = a.cnt;
      sh.mf[own][w] = mf;
      sh.best[own][w] = best;
      sh.hcnt[own][w] = a.h.cnt;
      sh.hedges[own][w] = hd;
      sh.cnt[own ^ 1][w] = 0;
      sh.mf[own ^ 1][w] = 0;
      sh.best[own ^ 1][w] = ~0ull;
      sh.hcnt[own ^ 1][w] = 0;
      sh.hedges[own ^ 1][w] = 0;
    }
  }
  __syncthreads();
  const int pc = w & 1;  // the list this wave publishes: colour pc, normal (w < 2) or hub (w >= 2)
  if (lane == 0 && w < 4 && pc < ncol) {
    Ring* nxt = pc ? nxt1 : nxt0;
    if (w < 2) {
      uint32_t tot = 0;
      unsigned long long mft = 0, bt = ~0ull;
      for (int i = 0; i < W; ++i) {
        const uint32_t k = sh.cnt[pc][i];
        sh.cnt[pc][i] = tot;
        tot += k;
        mft += sh.mf[pc][i];
        bt = sh.best[pc][i] < bt ? sh.best[pc][i] : bt;
      }
      sh.base[pc] = tot ? atomicAdd(&nxt->n, tot) : 0u;
      if (mft) atomicAdd((unsigned long long*)&nxt->mf, mft);
      if (bt != ~0ull) atomicMin(a.best_out, bt);
    } else {
      uint32_t k = 0;
      unsigned long long e = 0;
      for (int i = 0; i < W; ++i) {
        const uint32_t ki = sh.hcnt[pc][i];
        const unsigned long long ei = sh.hedges[pc][i];
        sh.hcnt[pc][i] = k;
        sh.hedges[pc][i] = e;
        k += ki;
        e += ei;
      }
      sh.hbase[pc] = k ? atomicAdd((unsigned long long*)&nxt->hub, ((unsigned long long)k << kHubEdgeBits) | e)
                       : 0ull;
    }
  }
  __syncthreads();
  const uint32_t base = sh.base[own] + sh.cnt[own][w];
  int32_t* q = a.p->q[own][a.nxt_par];
  for (uint32_t i = (uint32_t)lane; i < a.cnt; i += kWave) {
    const uint32_t slot = base + i;
    if (slot < a.p->qcap)
      q[slot] = a.buf[i];
    else
      atomicOr(&a.p->ctl->err, 1u);
  }
  if (a.h.cnt) {
    const unsigned long long hb = sh.hbase[own];
    hub_write(a.h, (uint32_t)(hb >> kHubEdgeBits) + sh.hcnt[own][w], (hb & kHubEdgeMask) + sh.hedges[own][w],
              a.p->hq[own][a.nxt_par], a.p->hb[own][a.nxt_par], a.p->hcap, &a.p->ctl->err);
  }
}

template <typename OffT>
__device__ __forceinline__ void propose(Appender<OffT>& a, int32_t dist, int32_t u) {
  const unsigned long long cand = ((unsigned long long)dist << 32) | (uint32_t)u;
  a.best = cand < a.best ? cand : a.best;
}

// Top-down probe of edge (v -> u) for colour c whose frontier is at level
// lvl, in three parts, so that a lane has the loads and the atomics of
// several edges in flight together:
//   probe_look   loads u's visited-bitmap word (BFS) or state word (s–t);
//   probe_issue  when that word leaves u unlabelled, issues the claiming
//                atomic together with the loads of u's offsets, so that a
//                claimed vertex's degree arrives with the atomic's result
//                instead of one round trip later;
//   probe_done   returns whether this lane claimed u (with its degree); for
//                s–t a meeting edge lowers the lane's best candidate.
template <typename OffT>
struct Probe {
  unsigned long long w;    // the looked-up word
  unsigned long long old;  // the atomic's result
  OffT ob, oe;             // u's offsets (when the atomic was issued)
  bool tried;              // the atomic was issued
};

template <bool TEAM, typename OffT>
__device__ __forceinline__ Probe<OffT> probe_look(const Appender<OffT>& a, bool st, int32_t u, bool act) {
  const VisitParams<OffT>& p = *a.p;
  Probe<OffT> r;
  r.w = 0;
  r.old = 0;
  r.ob = r.oe = 0;
  r.tried = false;
  if (!act) return r;
  if (!st)
    r.w = ldw<TEAM>((const uint32_t*)p.visited + (u >> 5));
  else if (u != a.root_own && u != a.root_other)
    r.w = ldw<TEAM>((const unsigned long long*)p.sst + u);
  return r;
}

template <typename OffT>
__device__ __forceinline__ void probe_issue(const Appender<OffT>& a, bool st, int lvl, int32_t u, bool act,
                                            Probe<OffT>& r) {
  const VisitParams<OffT>& p = *a.p;
  if (!act) return;
  if (!st) {
    // BFS claims through the visited bitmap: one atomicOr per newly reached
    // vertex; the looked-up word filters most already-visited probes.
    const uint32_t bit = 1u << (u & 31);
    if ((uint32_t)r.w & bit) return;
    r.ob = p.off[u];
    r.oe = p.off[u + 1];
    r.old = atomicOr(p.visited + (u >> 5), bit);
    r.tried = true;
    return;
  }
  // A word of another epoch is unvisited.
  if (u == a.root_own || u == a.root_other || (uint32_t)(r.w >> 32) == a.epoch) return;
  r.ob = p.off[u];
  r.oe = p.off[u + 1];
  r.old = atomicCAS(&p.sst[u], r.w, st_word(a.epoch, a.c, lvl + 1));
  r.tried = true;
}

template <typename OffT>
__device__ __forceinline__ bool probe_done(Appender<OffT>& a, int32_t* parent, bool st, int lvl, int32_t v,
                                           int32_t u, bool act, const Probe<OffT>& r, int64_t& deg) {
  const VisitParams<OffT>& p = *a.p;
  deg = 0;
  if (!act) return false;
  if (!st) {
    if (!r.tried || ((uint32_t)r.old & (1u << (u & 31)))) return false;
    p.state[u] = lvl + 1;
    if (parent) parent[u] = v;
    deg = (int64_t)(r.oe - r.ob);
    return true;
  }
  if (u == a.root_own) return false;
  if (u == a.root_other) {
    propose(a, lvl + 1, u);
    return false;
  }
  unsigned long long cur = r.w;
  if (r.tried) {
    // The looked-up word may be stale, so a failed CAS retries with the value
    // it returns; within a launch the word only changes to this epoch, so
    // the second attempt settles it (three attempts in all).
    const unsigned long long mine = st_word(a.epoch, a.c, lvl + 1);
    cur = r.old;
    bool won = r.old == r.w;
    for (int k = 0; k < 2 && !won && (uint32_t)(cur >> 32) != a.epoch; ++k) {
      const unsigned long long old = atomicCAS(&p.sst[u], cur, mine);
      won = old == cur;
      cur = old;
    }
    if (won) {
      if (parent) parent[u] = v;
      deg = (int64_t)(r.oe - r.ob);
      return true;
    }
  }
  if ((uint32_t)(cur >> 32) != a.epoch) {
    atomicOr(&p.ctl->err, 4u);
    return false;
  }
  const int32_t w = (int32_t)(uint32_t)cur;
  if (((w & kColorBit) != 0) != (a.c != 0)) propose(a, lvl + 1 + (w & kLevelMask), u);
  return false;
}

// The width is a run-time value: a copy of the code per width had made the
// kernel 48 KB of the 64 KB of instruction cache that two CUs share. It is a
// power of two in [4, 64] (visit_width, degree_width): with another one lanes
// would skip edges, and above 64 the loop over the frontier would not advance.
// push(claimed, u, first edge, degree) takes the claimed vertices (wave-collective).
template <bool TEAM, typename OffT, typename Push>
__device__ __forceinline__ void td_normal(Appender<OffT>& a, int32_t* parent, bool st, int vw, int lvl, int cur_par,
                                          uint32_t n, int gwave, int nwaves, Push push) {
  const VisitParams<OffT>& p = *a.p;
  const int lane = lane_id();
  const int sh = 31 - __builtin_clz((uint32_t)vw);
  const int grp = lane >> sh, sub = lane & (vw - 1);
  const uint32_t G = (uint32_t)kWave >> sh;
  const int32_t* q = p.q[a.c][cur_par];
  if (n > p.qcap) n = p.qcap;
  for (uint32_t base = (uint32_t)gwave * G; base < n; base += (uint32_t)nwaves * G) {
    const uint32_t i = base + (uint32_t)grp;
    int32_t v = 0;
    OffT b = 0, e = 0;
    if (i < n) {
      v = ldw<TEAM>(q + i);
      if ((uint32_t)v < (uint32_t)p.V) {
        b = p.off[v] + (OffT)sub;
        e = p.off[v + 1];
      } else {
        atomicOr(&p.ctl->err, 2u);
      }
    }
    // two columns per lane per round: both loads are issued before either
    // probe, halving the dependent round trips of long lists
    while (ballot(b < e)) {
      const bool a0 = b < e, a1 = b + vw < e;
      const int32_t u0 = a0 ? p.col[b] : 0;
      const int32_t u1 = a1 ? p.col[b + vw] : 0;
      Probe<OffT> r0 = probe_look<TEAM>(a, st, u0, a0), r1 = probe_look<TEAM>(a, st, u1, a1);
      probe_issue(a, st, lvl, u0, a0, r0);
      probe_issue(a, st, lvl, u1, a1, r1);
      int64_t d0, d1;
      const bool c0 = probe_done(a, parent, st, lvl, v, u0, a0, r0, d0);
      const bool c1 = probe_done(a, parent, st, lvl, v, u1, a1, r1, d1);
      push(c0, u0, r0.ob, d0);
      push(c1, u1, r1.ob, d1);
      b += 2 * vw;
    }
  }
}

// Edge-parallel expansion of the hub queue: the concatenated adjacency of all
// hub vertices is cut into chunks handed out across waves. A chunk is 256
// edges (four passes of one edge per lane) when there are enough edges for
// every wave to get a chunk of that size, else 128 or 64: when the hub edges
// are few (the second level of a visit from one root), a wave's chain of
// dependent loads per pass, not the edge count, sets the level's time, and
// smaller chunks spread the passes over more waves.
constexpr int kHubChunkMax = 256;

template <bool TEAM, typename OffT, typename Push>
__device__ __forceinline__ void td_hubs(Appender<OffT>& a, int32_t* parent, bool st, int lvl, int cur_par,
                                        uint64_t hubpk, int gwave, int nwaves, Push push) {
  const VisitParams<OffT>& p = *a.p;
  uint32_t nh = (uint32_t)(hubpk >> kHubEdgeBits);
  if (nh > p.hcap) nh = p.hcap;
  const uint64_t H = hubpk & kHubEdgeMask;
  if (nh == 0 || H == 0) return;
  const int lane = lane_id();
  const int32_t* hq = p.hq[a.c][cur_par];
  const int64_t* hb = p.hb[a.c][cur_par];
  const uint64_t nw = (uint64_t)nwaves;
  const int chunk = H >= nw * kHubChunkMax ? kHubChunkMax : H >= nw * (kHubChunkMax / 2) ? kHubChunkMax / 2 : kWave;
  for (uint64_t cb = (uint64_t)gwave * (uint64_t)chunk; cb < H; cb += nw * (uint64_t)chunk) {
    // Last slot with hb[slot] <= cb (hb[0] == 0): a 64-ary search, each lane
    // testing one of 64 evenly spaced probes per round.
    uint32_t lo = 0, hi = nh;
    while (hi - lo > 1) {
      const uint32_t span = hi - lo;
      const uint32_t step = (span + 63u) / 64u;
      const uint32_t probe = lo + (uint32_t)lane * step;
      const bool le = probe < hi && (uint64_t)ldw<TEAM>(hb + probe) <= cb;
      const uint64_t m = ballot(le);  // a prefix of lanes (hb ascending); lane 0 always set
      const uint32_t k = 63u - (uint32_t)__builtin_clzll((unsigned long long)m);
      lo = lo + k * step;
      const uint32_t nhi = lo + step;
      hi = nhi < hi ? nhi : hi;
    }
    for (int k = 0; k < chunk; k += kWave) {
      const uint64_t g = cb + (uint64_t)k + (uint64_t)lane;
      const bool act = g < H;
      int32_t v = -1, u = 0;
      if (act) {
        uint32_t s = lo;
        while (s + 1 < nh && (uint64_t)ldw<TEAM>(hb + s + 1) <= g) ++s;
        v = ldw<TEAM>(hq + s);
        const uint64_t h0 = (uint64_t)ldw<TEAM>(hb + s);
        bool good = (uint32_t)v < (uint32_t)p.V && h0 <= g;
        OffT k2 = 0;
        if (good) {
          k2 = p.off[v] + (OffT)(g - h0);
          good = k2 < p.off[v + 1];
        }
        if (good) {
          u = p.col[k2];
        } else {
          atomicOr(&p.ctl->err, 2u);
          v = -1;
        }
      }
      const bool ok = act && v >= 0;
      Probe<OffT> r = probe_look<TEAM>(a, st, u, ok);
      probe_issue(a, st, lvl, u, ok, r);
      int64_t d;
      const bool cl = probe_done(a, parent, st, lvl, v, u, ok, r, d);
      push(cl, u, r.ob, d);
    }
  }
}

// Level 0 of an s–t query: the root's adjacency [b, e) cut into 64-edge
// chunks over the waves of the grid (one edge per lane), whatever its degree.
template <bool TEAM, typename OffT, typename Push>
__device__ __forceinline__ void td_root(Appender<OffT>& a, int32_t* parent, int32_t r, OffT b, OffT e, int gwave,
                                        int nwaves, Push push) {
  const VisitParams<OffT>& p = *a.p;
  for (OffT k = b + (OffT)gwave * kWave; k < e; k += (OffT)nwaves * kWave) {
    const OffT j = k + (OffT)lane_id();
    const bool act = j < e;
    const int32_t u = act ? p.col[j] : 0;
    Probe<OffT> pr = probe_look<TEAM>(a, true, u, act);
    probe_issue(a, true, 0, u, act, pr);
    int64_t d;
    const bool cl = probe_done(a, parent, true, 0, r, u, act, pr, d);
    push(cl, u, pr.ob, d);
  }
}

// Candidates of degree <= kBuLane scan their own list; longer lists are
// scanned by the whole wave, 64 edges at a time, after the lane's own first
// round of eight.
constexpr int kBuLane = 128;

// Per-chunk loads of a bottom-up step (64 consecutive vertices of one wave):
// the unvisited flags and the offset pair. They are issued for the next
// chunk before the current chunk's columns are scanned, so a chunk costs
// about two dependent memory round trips instead of three.
template <typename OffT>
struct BuChunk {
  bool unvis;
  OffT b, e;
  unsigned long long head;
  uint32_t vword;  // the lane's visited word (lanes 0..31: 2w, 32..63: 2w + 1)
};

template <typename OffT>
__device__ __forceinline__ BuChunk<OffT> bu_load(const VisitParams<OffT>& p, uint32_t w) {
  const int lane = lane_id();
  const int32_t v = (int32_t)(w * 64u + (uint32_t)lane);
  const uint32_t wi = 2u * w + ((uint32_t)lane >> 5);
  BuChunk<OffT> c;
  c.vword = p.visited[wi];
  c.unvis = v < p.V && !((c.vword >> (lane & 31)) & 1u);
  c.b = c.e = 0;
  c.head = ~0ull;
  if (c.unvis) {
    c.b = p.off[v];
    c.e = p.off[v + 1];
    if (p.head) c.head = p.head[v];
  }
  return c;
}

// Bottom-up BFS step: every unvisited vertex looks for a neighbour in the
// current frontier bitmap.
template <typename OffT>
__device__ __forceinline__ void bu_step(Appender<OffT>& a, int32_t* parent, int lvl, const uint32_t* cfbm, int gwave,
                                        int nwaves) {
  const VisitParams<OffT>& p = *a.p;
  uint32_t* nfbm = a.nfbm;
  const int lane = lane_id();
  // Isolated vertices (the tail of a degree-ordered numbering) can have no
  // parent: their chunks are skipped (43% of the vertices of R-MAT s22).
  const uint32_t nw64 = ((uint32_t)p.v_active + 63u) >> 6;
  const int32_t mine = lvl + 1;
  // The wave's chunks are w = gwave + i * nwaves. Lane j first reads the
  // visited words of the j-th of the next 64 of them, so that chunks without
  // an unvisited vertex (most of them after the big bottom-up level) cost
  // nothing beyond that one round trip; the others are processed in order,
  // each loading the next one's visited bits and offsets while it works.
  for (uint64_t g0 = (uint64_t)gwave; g0 < nw64; g0 += (uint64_t)kWave * (uint64_t)nwaves) {
    const uint64_t cj = g0 + (uint64_t)lane * (uint64_t)nwaves;
    bool work = false;
    if (cj < nw64) {
      const uint64_t vis = ((uint64_t)p.visited[2 * cj + 1] << 32) | p.visited[2 * cj];
      const int64_t left = (int64_t)p.V - (int64_t)cj * 64;  // vertices of the chunk below V
      const uint64_t valid = left >= 64 ? ~0ull : (1ull << left) - 1ull;
      work = (~vis & valid) != 0;
    }
    uint64_t todo = ballot(work);
    if (!todo) continue;
    uint32_t w = (uint32_t)(g0 + (uint64_t)__builtin_ctzll(todo) * (uint64_t)nwaves);
    todo &= todo - 1;
    BuChunk<OffT> cur = bu_load(p, w);
    for (;;) {
      const bool more = todo != 0;
      uint32_t wn = 0;
      BuChunk<OffT> nx;
      if (more) {
        wn = (uint32_t)(g0 + (uint64_t)__builtin_ctzll(todo) * (uint64_t)nwaves);
        todo &= todo - 1;
        nx = bu_load(p, wn);
      }
      const int32_t v = (int32_t)(w * 64u + (uint32_t)lane);
      const bool cand = cur.unvis;
      const OffT b = cur.b, e = cur.e;
      const bool small = cand && (e - b) <= (OffT)kBuLane;
      int32_t par = -1;
      // A long list's first eight entries are scanned in the lane's own first
      // round too: they hold the parent of nearly every candidate (lists are in
      // id order, which puts the hubs first), so few long lists need the wave.
      const OffT lim = small ? e : (b + 8 < e ? b + 8 : e);
      // A list's first two columns come from an array of their own: read in
      // vertex order, they take 8 bytes a vertex where the list takes a line
      // (R-MAT s22: 300 MB for the 2.4M vertices that are not isolated), and
      // nine vertices in ten need no more. BFS of s22 167 -> 147 us, of s24
      // 477 -> 388, of a random graph of 2M vertices and degree 16 259 -> 239.
      OffT j0 = b;
      if (cand && p.head) {
        const int32_t u0 = (int32_t)(uint32_t)cur.head, u1 = (int32_t)(uint32_t)(cur.head >> 32);
        const uint32_t f0 = u0 >= 0 ? cfbm[u0 >> 5] : 0u, f1 = u1 >= 0 ? cfbm[u1 >> 5] : 0u;
        if (u1 >= 0 && ((f1 >> (u1 & 31)) & 1u)) par = u1;
        if (u0 >= 0 && ((f0 >> (u0 & 31)) & 1u)) par = u0;
        j0 = b + 2;
      }
      if (cand) {
        // eight independent column loads per round, then the eight bitmap
        // words together, so a round costs two round trips whichever column
        // holds the parent; most candidates find one in the first round
        for (OffT j = j0; j < lim && par < 0; j += 8) {
          int32_t u[8];
  #pragma unroll
          for (int k = 0; k < 8; ++k) u[k] = j + k < lim ? p.col[j + k] : -1;
          uint32_t fw[8];
  #pragma unroll
          for (int k = 0; k < 8; ++k) fw[k] = u[k] >= 0 ? cfbm[u[k] >> 5] : 0u;
  #pragma unroll
          for (int k = 7; k >= 0; --k)
            if (u[k] >= 0 && ((fw[k] >> (u[k] & 31)) & 1u)) par = u[k];
        }
      }
      uint64_t big = ballot(cand && !small && par < 0);
      while (big) {
        const int l = __ffsll((unsigned long long)big) - 1;
        big &= big - 1;
        const OffT bb = bcast_off<OffT>(lim, l), ee = bcast_off<OffT>(e, l);
        int32_t fp = -1;
        for (OffT j0 = bb; j0 < ee; j0 += kWave) {
          const OffT j = j0 + (OffT)lane;
          bool hit = false;
          int32_t u = 0;
          if (j < ee) {
            u = p.col[j];
            hit = test_bit(cfbm, u);
          }
          const uint64_t hm = ballot(hit);
          if (hm) {
            fp = bcast(u, __ffsll((unsigned long long)hm) - 1);
            break;
          }
        }
        if (lane == l) par = fp;
      }
      const bool claimed = cand && par >= 0;
      if (claimed) {
        p.state[v] = mine;
        if (parent) parent[v] = par;
      }
      // Bitmap words of these 64 vertices belong to this wave during a
      // bottom-up level, so they are updated without atomics (and the
      // prefetched words of the wave's next chunk are not changed by others).
      const uint64_t cm = ballot(claimed);
      // (the visited words came with the chunk's loads: no load waits here)
      if (lane == 0 && (uint32_t)cm) {
        p.visited[2u * w] = cur.vword | (uint32_t)cm;
        nfbm[2u * w] = (uint32_t)cm;
      }
      if (lane == 32 && (uint32_t)(cm >> 32)) {
        p.visited[2u * w + 1u] = cur.vword | (uint32_t)(cm >> 32);
        nfbm[2u * w + 1u] = (uint32_t)(cm >> 32);
      }
      push_next(a, claimed, v, claimed ? (int64_t)(e - b) : 0, false);
      if (!more) break;
      cur = nx;
      w = wn;
    }
  }
}

// Width for a top-down level: the smallest power of two >= the average degree
// of the normal-queue entries, clamped to [4, 64].
// Every block decides this at launch start: vw < ceil(mf / n) exactly when
// vw * n < mf, so no 64-bit division.
__device__ __forceinline__ int degree_width(uint32_t n, uint64_t mf_normal) {
  if (n == 0) return 4;
  int vw = 4;
  while (vw < 64 && (uint64_t)vw * n < mf_normal) vw <<= 1;
  return vw;
}

// Beamer's switch thresholds for direction-optimising BFS. His alpha of 14
// left levels of 9M edges to a top-down step at s22, 130 us where the
// bottom-up step took 35. Mean of 48 roots with alpha 14, 30, 60 and 120: s16
// 79, 72, 69, 66 us, s22 161, 152, 147, 147, s24 401, 393, 389, 415, a random
// graph of 2M vertices and degree 16 273, 239, 239, 240.
constexpr double kAlpha = 60.0;
constexpr double kBeta = 24.0;

__device__ __forceinline__ uint32_t ring_size(const Ring& r) { return r.n + (uint32_t)(r.hub >> kHubEdgeBits); }

__device__ __forceinline__ void zero_ring(Ring* r) { *r = Ring{0u, 0u, 0ull, 0ull}; }

// Waves of colour 0, in proportion to the colours' edges; a colour with edges
// has at least one.
__device__ __forceinline__ int colour_split(double e0, double e1, int nwaves) {
  const int lo = e0 > 0 ? 1 : 0, hi = e1 > 0 ? nwaves - 1 : nwaves;
  const double f = e0 + e1 > 0 ? e0 / (e0 + e1) : 0.5;
  const int w0 = (int)((double)nwaves * f + 0.5);
  return w0 < lo ? lo : (w0 > hi ? hi : w0);
}

// BFS reset (one launch): clear the bitmaps (and, on the caller's numbering,
// the levels and parents), and block 0 seeds the root.
template <typename OffT>
__device__ void bfs_reset(const VisitParams<OffT>& p, const VisitState& S, VisitState* nxt, int32_t* parent) {
  const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nthr = (int64_t)gridDim.x * blockDim.x;
  const uint32_t nwords = (((uint32_t)p.V + 63u) >> 6) * 2u;
  const int32_t src = S.src;
  if (!p.lazy_state) {
    for (int64_t v = gtid; v < p.V; v += nthr) {
      p.state[v] = v == src ? 0 : -1;
      if (parent) parent[v] = v == src ? (int32_t)v : -1;
    }
  }
  for (int64_t w = gtid; w < nwords; w += nthr) {
    const uint32_t bs = ((uint32_t)src >> 5) == (uint32_t)w ? 1u << (src & 31) : 0u;
    p.visited[w] = bs;
    p.fbm[0][0][w] = bs;
    p.fbm[0][1][w] = 0u;
    p.fbm[0][2][w] = 0u;
  }
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  VisitCtl* ctl = p.ctl;
  if (p.lazy_state) {
    // renumbered graph: only reached vertices' state and parent are written
    // (the visited bitmap marks them), so only the root's here
    p.state[src] = 0;
    if (parent) parent[src] = src;
  }
  const int64_t d = (int64_t)(p.off[src + 1] - p.off[src]);
  Ring r0{0u, 0u, 0ull, (uint64_t)d};
  if (d >= p.hub_threshold) {
    p.hq[0][0][0] = src;
    p.hb[0][0][0] = 0;
    r0.hub = (1ull << kHubEdgeBits) | (uint64_t)d;
  } else {
    p.q[0][0][0] = src;
    r0.n = 1u;
  }
  ctl->ring[0][0][0] = r0;
  zero_ring(&ctl->ring[0][0][1]);
  zero_ring(&ctl->ring[0][0][2]);
  VisitState n = S;
  n.phase = kPhaseLevel;
  n.lvl = 0;
  n.steps = n.td = n.bu = n.maxf = 0;
  n.launches = 1;
  n.bu_mode = 0;
  n.seen_edges = (uint64_t)d;
  n.visited_v = 1;
  n.visited_e = d;
  n.expv = n.expe = 0;
  *nxt = n;
}

// W: waves of a block (W or kWideWaves)
template <typename OffT, int W>
__global__ __launch_bounds__(W * kWave) void phase_kernel(VisitCtl* ctl, int parity) {
  __shared__ VisitCtl h;
  __shared__ int32_t s_stage[W * kStageCap];
  __shared__ int32_t s_hub[2][W * kHubStage];
  __shared__ BlockShared<W> s_sh;
  __shared__ OffT s_root[4];
  static_assert(sizeof(VisitCtl) == kWave * sizeof(uint4), "one 16-byte load per lane");
  if (threadIdx.x < kWave)
    reinterpret_cast<uint4*>(&h)[threadIdx.x] = reinterpret_cast<const uint4*>(ctl)[threadIdx.x];
  __syncthreads();
  const VisitParams<OffT>& p = *reinterpret_cast<const VisitParams<OffT>*>(h.params);
  const VisitState& S = h.st[parity];
  VisitState* nxt = &ctl->st[parity ^ 1];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (S.phase == kPhaseIdle) {
    if (lead) nxt->phase = kPhaseIdle;
    return;
  }
  const bool st = h.mode != kModeBfs;
  int32_t* const parent = h.record_parents ? p.parent : nullptr;
  if (S.phase == kPhaseReset) {
    bfs_reset(p, S, nxt, parent);
    return;
  }

  // ---- level phase: every block takes the same decisions from S ----
  // (Scalars only below: a local copy of the state, or arrays indexed by the
  // colour, would be put in scratch memory.)
  int q = S.qi, L = S.lvl;
  int qp = query_set(q);
  int32_t src = S.src, dst = S.dst;
  uint32_t epoch = S.epoch;
  bool start = st && L == 0;  // s–t: this launch expands the roots of query q
  const int ncol = st ? 2 : 1;
  Ring cur[2];
  cur[0] = h.ring[qp][0][L % 3];
  cur[1] = h.ring[qp][1][L % 3];
  const uint32_t nf0 = ring_size(cur[0]), nf1 = st ? ring_size(cur[1]) : 0u;
  const uint64_t mf01 = cur[0].mf + (st ? cur[1].mf : 0ull);
  // the level-L frontier (built by the previous launch) counted as labelled
  const bool counted = L > 0;
  const uint64_t seen = S.seen_edges + (counted ? mf01 : 0ull);
  if (!start) {
    // see whether the query is finished
    const bool empty = counted && (nf0 == 0 || (st && nf1 == 0));
    const unsigned long long best = h.best[qp][(L + 1) & 1];  // the last level's
    const bool runaway = S.steps > p.V + 2;
    if ((st && best != ~0ull) || empty || h.err || runaway) {
      if (lead) {
        const bool met = st && best != ~0ull;
        VisitOut o;
        o.status = (h.err || runaway) ? FC_CAPACITY_STATUS : 0;
        o.levels = S.steps;
        o.depth = met ? S.steps : 0;
        o.dist = met ? (int32_t)(best >> 32) : -1;
        o.meet = met ? (int32_t)(uint32_t)best : -1;
        o.topdown = S.td;
        o.bottomup = S.bu;
        o.max_frontier = S.maxf;
        o.visited_vertices = S.visited_v + (counted ? (int64_t)nf0 + (int64_t)nf1 : 0);
        o.visited_edges = S.visited_e + (counted ? (int64_t)mf01 : 0);
        o.expanded_vertices = S.expv;
        o.expanded_edges = S.expe;
        o.err = (int32_t)h.err;
        // a BFS spends one more launch noticing its empty frontier; an s–t
        // query notices its end in the launch that starts the next query
        o.launches = S.launches + (st ? 0 : 1);
        p.out[q] = o;
      }
      if (!st || q + 1 >= h.nq) {
        if (lead) nxt->phase = kPhaseIdle;
        return;
      }
      // the next s–t query starts in this launch
      ++q;
      qp = query_set(q);
      src = S.nsrc;
      dst = S.ndst;
      epoch = S.epoch + 1;
      L = 0;
      start = true;
    }
  }

  const int64_t gtid = (int64_t)blockIdx.x * (W * kWave) + threadIdx.x;
  const int64_t nthr = (int64_t)gridDim.x * (W * kWave);
  const int gwave = (int)(blockIdx.x * W + (threadIdx.x >> 6));
  const int nwaves = (int)(gridDim.x * W);
  int strat = kTopDown;
  int vw0 = 4, vw1 = 4;
  if (start) {
    if (threadIdx.x < 4) s_root[threadIdx.x] = p.off[(threadIdx.x < 2 ? src : dst) + (threadIdx.x & 1)];
    __syncthreads();
    const uint64_t ds = (uint64_t)(s_root[1] - s_root[0]), dt = (uint64_t)(s_root[3] - s_root[2]);
    if (lead) {
      // the new query's machine state after this launch (its level 0)
      nxt->phase = kPhaseLevel;
      nxt->qi = q;
      nxt->src = src;
      nxt->dst = dst;
      nxt->nsrc = q + 1 < h.nq ? p.qs[q + 1] : -1;
      nxt->ndst = q + 1 < h.nq ? p.qt[q + 1] : -1;
      nxt->lvl = 1;
      nxt->epoch = epoch;
      nxt->steps = 1;
      nxt->td = 2;
      nxt->bu = 0;
      nxt->maxf = 1;
      nxt->launches = 1;
      nxt->bu_mode = 0;
      nxt->seen_edges = ds + dt;
      nxt->visited_v = 2;
      nxt->visited_e = (int64_t)(ds + dt);
      nxt->expv = 2;
      nxt->expe = (int64_t)(ds + dt);
      p.sst[src] = st_word(epoch, 0, 0);
      p.sst[dst] = st_word(epoch, 1, 0);
      if (parent) {
        parent[src] = src;
        parent[dst] = dst;
      }
      // the next query's counters (this query's level-1 ring was cleared when
      // the previous query started), and this query's level-2 ring
      const int nq = query_set(q + 1);
      for (int c = 0; c < 2; ++c) {
        for (int k = 0; k < 3; ++k) zero_ring(&ctl->ring[nq][c][k]);
        zero_ring(&ctl->ring[qp][c][2]);
      }
      ctl->best[nq][0] = ctl->best[nq][1] = ~0ull;
    }
  } else {
    const double mu = (double)p.E - (double)seen;
    vw0 = h.vw_fixed > 0 ? h.vw_fixed : degree_width(cur[0].n, cur[0].mf - (cur[0].hub & kHubEdgeMask));
    if (st) vw1 = h.vw_fixed > 0 ? h.vw_fixed : degree_width(cur[1].n, cur[1].mf - (cur[1].hub & kHubEdgeMask));
    int bu = S.bu_mode;
    if (!st) {
      if (!bu) {
        // (a list holds a vertex's parents only where edges go both ways)
        if (p.bottom_up && (double)cur[0].mf > mu / kAlpha) bu = 1;
      } else if ((double)nf0 * kBeta < (double)p.V) {
        bu = 0;
      }
      strat = bu ? kBottomUp : kTopDown;
    }
    if (lead) {
      nxt->phase = kPhaseLevel;
      nxt->qi = q;
      nxt->src = src;
      nxt->dst = dst;
      nxt->nsrc = S.nsrc;
      nxt->ndst = S.ndst;
      nxt->lvl = L + 1;
      nxt->epoch = epoch;
      nxt->steps = S.steps + 1;
      nxt->td = S.td + (strat == kTopDown ? ncol : 0);
      nxt->bu = S.bu + (strat == kTopDown ? 0 : ncol);
      const int32_t mx = (int32_t)(nf0 > nf1 ? nf0 : nf1);
      nxt->maxf = mx > S.maxf ? mx : S.maxf;
      nxt->launches = S.launches + 1;
      nxt->bu_mode = bu;
      nxt->seen_edges = seen;
      nxt->visited_v = S.visited_v + (counted ? (int64_t)nf0 + (int64_t)nf1 : 0);
      nxt->visited_e = S.visited_e + (counted ? (int64_t)mf01 : 0);
      nxt->expv = S.expv + (int64_t)nf0 + (int64_t)nf1;
      nxt->expe = S.expe + (int64_t)mf01;
      zero_ring(&ctl->ring[qp][0][(L + 2) % 3]);
      if (st) zero_ring(&ctl->ring[qp][1][(L + 2) % 3]);
    }
    if (!st) {
      // the BFS frontier bitmap two levels ahead is free: clear it for the
      // next level's appends
      uint32_t* far = p.fbm[0][(L + 2) % 3];
      const uint32_t nwords = (((uint32_t)p.V + 63u) >> 6) * 2u;
      for (int64_t w = gtid; w < nwords; w += nthr) far[w] = 0u;
    }
  }

  // The waves are split between the colours in proportion to their frontier
  // edges, so that both colours' chains of dependent loads run at the same
  // time; each wave expands one colour and stages into that colour's lists.
  const int cur_par = L & 1;
  const int w0 = ncol == 2 ? colour_split(start ? (double)(s_root[1] - s_root[0]) : (double)cur[0].mf,
                                          start ? (double)(s_root[3] - s_root[2]) : (double)cur[1].mf, nwaves)
                           : nwaves;
  const int cw = gwave < w0 ? 0 : 1;  // this wave's colour
  const int lw = cw ? gwave - w0 : gwave, nlw = cw ? nwaves - w0 : w0;
  Appender<OffT> a;
  a.p = &p;
  a.c = cw;
  a.nxt_par = cur_par ^ 1;
  a.nxt = &ctl->ring[qp][cw][(L + 1) % 3];
  a.nfbm = p.fbm[cw][(L + 1) % 3];
  a.best_out = &ctl->best[qp][L & 1];
  a.bitmaps = !st;
  a.epoch = epoch;
  a.root_own = cw ? dst : src;
  a.root_other = cw ? src : dst;
  a.buf = s_stage + (threadIdx.x >> 6) * kStageCap;
  a.cnt = 0;
  a.mf = 0;
  a.best = ~0ull;
  a.h.u = &s_hub[0][(threadIdx.x >> 6) * kHubStage];
  a.h.d = &s_hub[1][(threadIdx.x >> 6) * kHubStage];
  a.h.cnt = 0;
  auto push = [&](bool claimed, int32_t u, OffT, int64_t deg) { push_next(a, claimed, u, deg, a.bitmaps); };
  if (start) {
    td_root<false>(a, parent, cw ? dst : src, s_root[2 * cw], s_root[2 * cw + 1], lw, nlw, push);
  } else if (strat == kTopDown) {
    // selects, not indexing: a local array indexed by a runtime value
    // would live in scratch memory
    const int vwc = cw ? vw1 : vw0;
    const uint32_t nc = cw ? cur[1].n : cur[0].n;
    const uint64_t hc = cw ? cur[1].hub : cur[0].hub;
    td_normal<false>(a, parent, st, vwc, L, cur_par, nc, lw, nlw, push);
    td_hubs<false>(a, parent, st, L, cur_par, hc, lw, nlw, push);
  } else {
    bu_step(a, parent, L, p.fbm[cw][L % 3], lw, nlw);
  }
  block_flush(a, ncol, s_sh, &ctl->ring[qp][0][(L + 1) % 3], &ctl->ring[qp][1][(L + 1) % 3]);
}

// Plain s–t queries by teams (team.hpp): each XCD's blocks visit a query of
// their own, level after level with a barrier inside the XCD, until no query
// is left. The visit is phase_kernel's (the same expansion, claims, frontier
// counters and stop rule), and so are the answers and the counters. A level
// of a long path costs one chain of dependent loads and a barrier instead of a
// launch (a 4096^2 grid: 8 us a level with launches), and eight queries run
// at a time.
//
// A query with a level of more than max_edges edges is given up (kTooWide): the
// caller runs it again by launches, on the whole GPU.
//
// Query k of a machine uses the counters of parity k mod 4. Block 0 clears
// those of query k + 2 when query k starts: all blocks have then left query
// k - 2, whose counters they were (its last reader passed a barrier of query
// k - 1), and no block appends to query k + 2 before two more barriers.
template <typename OffT>
__global__ __launch_bounds__(kBlock) void st_team_kernel(StTeamRun tr) {
  // read with scalar loads (the launch does not write it)
  typedef __attribute__((address_space(4))) const VisitParams<OffT>* params_ptr;
  const VisitParams<OffT>& p = *(const VisitParams<OffT>*)((params_ptr)(uintptr_t)tr.params + xcc_id());
  __shared__ int32_t s_stage[kWavesPerBlock * kStageCap];
  __shared__ int32_t s_hub[2][kWavesPerBlock * kHubStage];
  __shared__ BlockShared<kWavesPerBlock> s_sh;
  __shared__ OffT s_root[4];
  __shared__ unsigned long long s_now[7];  // the level's rings and the best candidate of the last level
  __shared__ int s_num, s_size, s_q, s_ok;
  static_assert(sizeof(Ring) == 3 * sizeof(unsigned long long), "a ring is three words");
  const int machine = xcc_id();
  TeamSync* ts = tr.sync + machine;
  TeamBar* bar = tr.bar + machine;
  StTeamCtl* ctl = tr.ctl + machine;
  if (threadIdx.x == 0) {
    uint32_t members = 0;
    s_num = team_register(ts, tr.expected, &members);
    s_size = (int)members;
    if (s_num == 0) {
      st_team(&ctl->q[0], atomicAdd(tr.ticket, 1u));
      __builtin_amdgcn_s_waitcnt(0);
      st_team(&ts->size.v, members);
    } else if (s_num > 0) {
      s_size = team_wait(&ts->size.v, 1u) ? (int)ld_agent(&ts->size.v) : 0;
      if (!s_size) st_agent(tr.err, 1u);
    }
  }
  __syncthreads();
  const int bid = __builtin_amdgcn_readfirstlane(s_num), nb = __builtin_amdgcn_readfirstlane(s_size);
  if (bid < 0 || nb == 0) return;
  const bool lead = bid == 0 && threadIdx.x == 0;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int gwave = bid * kWavesPerBlock + w, nwaves = nb * kWavesPerBlock;
  uint32_t bars = 0;
  for (uint32_t k = 0;; ++k) {
    const int qp = (int)(k & 3u);
    if (threadIdx.x == 0) s_q = (int)ld_agent(&ctl->q[qp]);
    __syncthreads();
    const int q = __builtin_amdgcn_readfirstlane(s_q);
    if (q >= tr.nq) return;
    const int32_t src = p.qs[q], dst = p.qt[q];
    const uint32_t epoch = tr.epoch0 + (uint32_t)q;
    if (threadIdx.x < 4) s_root[threadIdx.x] = p.off[(threadIdx.x < 2 ? src : dst) + (int)(threadIdx.x & 1)];
    __syncthreads();
    const uint64_t ds = (uint64_t)(s_root[1] - s_root[0]), dt = (uint64_t)(s_root[3] - s_root[2]);
    if (lead) {
      st_team(&ctl->q[(k + 1) & 3u], atomicAdd(tr.ticket, 1u));
      const int far = (int)((k + 2) & 3u);
      for (int c = 0; c < 2; ++c)
        for (int r = 0; r < 3; ++r) zero_ring(&ctl->ring[far][c][r]);
      ctl->best[far][0] = ctl->best[far][1] = ~0ull;
      p.sst[src] = st_word(epoch, 0, 0);
      p.sst[dst] = st_word(epoch, 1, 0);
    }
    int steps = 0, td = 0, maxf = 1;
    int64_t vis_v = 2, vis_e = (int64_t)(ds + dt), expv = 2, expe = (int64_t)(ds + dt);
    bool wide = (int64_t)(ds + dt) > tr.max_edges;  // then the roots are not expanded, and level 1 ends the query
    for (int L = 0;; ++L) {
      Ring cur[2] = {{0u, 0u, 0ull, ds}, {0u, 0u, 0ull, dt}};
      int vw0 = 4, vw1 = 4;
      if (L > 0) {
        if (threadIdx.x < 7) {
          const int i = (int)threadIdx.x;
          s_now[i] = ld_team(i < 6 ? reinterpret_cast<const unsigned long long*>(&ctl->ring[qp][i / 3][L % 3]) + i % 3
                                   : &ctl->best[qp][(L - 1) & 1]);
        }
        __syncthreads();
        auto now = [&](int i) { return (uint64_t)bcast64((int64_t)s_now[i], 0); };
        const uint64_t best = now(6);
        cur[0] = Ring{(uint32_t)now(0), 0u, now(1), now(2)};
        cur[1] = Ring{(uint32_t)now(3), 0u, now(4), now(5)};
        const uint32_t nf0 = ring_size(cur[0]), nf1 = ring_size(cur[1]);
        const int64_t mf01 = (int64_t)(cur[0].mf + cur[1].mf);
        vis_v += (int64_t)nf0 + (int64_t)nf1;
        vis_e += mf01;
        // The stop decision rests on words that no block changes during the
        // level (the error bits can: they only colour the result; a guard that
        // trips drops entries, so the visit still ends).
        const bool met = best != ~0ull, runaway = steps > p.V + 2;
        const bool empty = nf0 == 0 || nf1 == 0;
        wide |= !met && !empty && mf01 > tr.max_edges;
        if (met || empty || wide || runaway) {
          if (lead) {
            const uint32_t err = ld_team(&ctl->v.err);
            VisitOut o;
            o.status = (err || runaway) ? FC_CAPACITY_STATUS : wide ? kTooWide : 0;
            o.levels = steps;
            o.depth = met ? steps : 0;
            o.dist = met ? (int32_t)(best >> 32) : -1;
            o.meet = met ? (int32_t)(uint32_t)best : -1;
            o.topdown = td;
            o.bottomup = 0;
            o.max_frontier = maxf;
            o.visited_vertices = vis_v;
            o.visited_edges = vis_e;
            o.expanded_vertices = expv;
            o.expanded_edges = expe;
            o.err = (int32_t)err;
            o.launches = 0;  // the one launch is the call's
            p.out[q] = o;
          }
          break;
        }
        expv += (int64_t)nf0 + (int64_t)nf1;
        expe += mf01;
        const int32_t mx = (int32_t)(nf0 > nf1 ? nf0 : nf1);
        maxf = mx > maxf ? mx : maxf;
        vw0 = tr.vw_fixed > 0 ? tr.vw_fixed : degree_width(cur[0].n, cur[0].mf - (cur[0].hub & kHubEdgeMask));
        vw1 = tr.vw_fixed > 0 ? tr.vw_fixed : degree_width(cur[1].n, cur[1].mf - (cur[1].hub & kHubEdgeMask));
        if (lead) {
          zero_ring(&ctl->ring[qp][0][(L + 2) % 3]);
          zero_ring(&ctl->ring[qp][1][(L + 2) % 3]);
        }
      }
      ++steps;
      td += 2;
      const int w0 = colour_split((double)cur[0].mf, (double)cur[1].mf, nwaves);
      const int cw = gwave < w0 ? 0 : 1;
      const int lw = cw ? gwave - w0 : gwave, nlw = cw ? nwaves - w0 : w0;
      Appender<OffT> a;
      a.p = &p;
      a.c = cw;
      a.nxt_par = (L & 1) ^ 1;
      a.nxt = &ctl->ring[qp][cw][(L + 1) % 3];
      a.nfbm = nullptr;
      a.best_out = &ctl->best[qp][L & 1];
      a.bitmaps = false;
      a.epoch = epoch;
      a.root_own = cw ? dst : src;
      a.root_other = cw ? src : dst;
      a.buf = s_stage + w * kStageCap;
      a.cnt = 0;
      a.mf = 0;
      a.best = ~0ull;
      a.h.u = &s_hub[0][w * kHubStage];
      a.h.d = &s_hub[1][w * kHubStage];
      a.h.cnt = 0;
      auto push = [&](bool claimed, int32_t u, OffT, int64_t deg) { push_next(a, claimed, u, deg, false); };
      if (L == 0) {
        if (!wide) td_root<true>(a, (int32_t*)nullptr, cw ? dst : src, s_root[2 * cw], s_root[2 * cw + 1], lw, nlw, push);
      } else {
        td_normal<true>(a, (int32_t*)nullptr, true, cw ? vw1 : vw0, L, L & 1, cw ? cur[1].n : cur[0].n, lw, nlw, push);
        td_hubs<true>(a, (int32_t*)nullptr, true, L, L & 1, cw ? cur[1].hub : cur[0].hub, lw, nlw, push);
      }
      block_flush(a, 2, s_sh, &ctl->ring[qp][0][(L + 1) % 3], &ctl->ring[qp][1][(L + 1) % 3]);
      if (!team_barrier(bar, bid, nb, bars, &s_ok)) {
        if (threadIdx.x == 0) st_agent(tr.err, 1u);
        return;
      }
    }
  }
}

template <typename OffT>
hipError_t launch_st_team(const StTeamRun& tr, int blocks, hipStream_t s) {
  hipLaunchKernelGGL(st_team_kernel<OffT>, dim3(blocks), dim3(kBlock), 0, s, tr);
  return hipGetLastError();
}

template <typename OffT>
int st_team_occupancy() {
  int nb = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, st_team_kernel<OffT>, kBlock, 0) != hipSuccess) return 0;
  return nb;
}

template hipError_t launch_st_team<int32_t>(const StTeamRun&, int, hipStream_t);
template hipError_t launch_st_team<int64_t>(const StTeamRun&, int, hipStream_t);
template int st_team_occupancy<int32_t>();
template int st_team_occupancy<int64_t>();

// ---------------------------------------------------------------------------
// Narrow visits: a query or BFS whose frontiers stay small over many levels
// (grids, road networks, sparse random graphs), by one team per query.
//
// On such a visit a level's time is its chain of dependent memory round trips,
// not its work: a frontier entry, its offsets, a column, the neighbour's state
// word, the claiming atomic, the list reservation, the barrier. st_team_kernel
// pays all of them (7.6 us a level on a 4096^2 grid), a launch per level 7.9.
// Here
//  * a block keeps the vertices it claims, up to kKeep of them, in its LDS,
//    with their offsets, and its waves expand them at the next level. A CU
//    takes about one scattered lane per clock, so the widest block sets the
//    pace: one with much more than its part of the frontier publishes the
//    rest in the frontier lists, from where all waves take their shares
//    (2048^2 grid, BFS: 15.5 -> 14.4 ms);
//  * between its arrival at the barrier and the barrier's end, when it would
//    wait anyway, a wave loads the first columns of these vertices and the
//    state words and offsets they lead to. A word that another wave changes
//    meanwhile is settled by the claim, as every stale look is;
//  * a level ends without an atomic: each block stores a word of its own with
//    the counts of its claimed vertices, and one wave per block, which does
//    nothing else, reads the words of all blocks until they carry the level's
//    tag. The store is a plain one: an agent-scope store writes through the
//    L2, and the level ended 1.3 us later (15.8 against 11.0 ms). From the
//    sums every block takes the stop decision; the lists' counters and the
//    best candidate are only read when a block has flagged them.
// What is left of a level is the claiming atomic, two block-wide steps, a
// store and the loads that see it: 2.5 us for 2,000 vertices. Measured
// against one launch a level (BFS) or st_team_kernel: BFS of a 2048^2 grid 30.4
// -> 9.7 ms, of 500^2 7.35 -> 2.22 ms, eight queries on a 4096^2 grid 22.9 ->
// 12.3 ms. (Loading a line of the columns after the next as well cost the
// queries 5%; two kept entries per lane group, which a query's half of the
// waves needs on grids of 4096^2, cost a BFS 5%.) A visit whose frontier reaches kNarrowMax vertices is given up
// (kTooWide): the caller runs it on the engine that uses the whole GPU.
// A BFS is a visit with one colour and no target. Levels, counters and answers
// are those of the other engines.
constexpr int kNarrowWaves = kNarrowThreads / kWave;
constexpr uint32_t kNarrowStage = 256;   // entries a wave stages for publication
constexpr uint32_t kNarrowSpill = 64;    // and room for what the block gives up
constexpr uint32_t kNarrowMax = 65535;

// Colours, waves per block and colour that expand, and entries a block can
// keep per colour.
template <bool BFS>
struct NarrowSplit {
  static constexpr int kColours = BFS ? 1 : 2, kWorkers = (kNarrowWaves - 1) / kColours;
  static constexpr int kSets = BFS ? 1 : 2;  // kept entries per lane group of four
  static constexpr uint32_t kKeep = 16u * kSets * kWorkers;
  static_assert(kKeep <= kNarrowSpill * kWorkers, "kNarrowSpill");
};

template <typename OffT, bool BFS>
struct NarrowKept {  // a block's kept vertices of one colour, by level parity
  static constexpr uint32_t kKeep = NarrowSplit<BFS>::kKeep;
  uint32_t n[2];  // may exceed kKeep: the rest was staged
  int32_t v[2][kKeep];
  int32_t d[2][kKeep];
  OffT b[2][kKeep];
};

struct NarrowShared {
  uint32_t cnt[2][kNarrowWaves];
  uint32_t hcnt[2][kNarrowWaves];
  unsigned long long hedges[2][kNarrowWaves];
  uint32_t base[2];
  unsigned long long hbase[2];
  uint32_t claims[kNarrowWaves];
  unsigned long long sums[2][kNarrowWaves];
  // the level's end, from the service wave: narrow_word sums, and after a look
  // per colour the lists' n and hub words and the best candidate
  unsigned long long sum, now[5];
  int look[2];                // by level parity: this block has something to look at
};

// Add the claimed vertices to the next frontier: kept by the block, staged for
// publication, or staged as hubs (wave-collective).
template <typename OffT, bool BFS>
__device__ __forceinline__ void push_kept(Appender<OffT>& a, NarrowKept<OffT, BFS>& kp, int par, uint32_t& claims,
                                          bool claimed, int32_t u, OffT b, int64_t deg) {
  const VisitParams<OffT>& p = *a.p;
  const bool hub = claimed && deg >= p.hub_threshold;
  const bool norm = claimed && !hub;
  const uint64_t m = ballot(norm);
  claims += (uint32_t)__popcll(ballot(claimed));
  if (m) {
    uint32_t base = 0;
    if (lane_id() == 0) base = atomicAdd(&kp.n[par], (uint32_t)__popcll(m));
    const uint32_t at = (uint32_t)bcast((int32_t)base, 0) + lane_rank(m);
    const bool over = norm && at >= kp.kKeep;
    if (norm && !over) {
      kp.v[par][at] = u;
      kp.d[par][at] = (int32_t)deg;
      kp.b[par][at] = b;
    }
    const uint64_t mo = ballot(over);
    if (mo) {
      const uint32_t k = (uint32_t)__popcll(mo);
      if (a.cnt + k > kNarrowStage) wave_flush(a);
      if (over) a.buf[a.cnt + lane_rank(mo)] = u;
      a.cnt += k;
    }
  }
  hub_push(a.h, hub, u, deg, (unsigned long long*)&a.nxt->hub, p.hq[a.c][a.nxt_par], p.hb[a.c][a.nxt_par], p.hcap,
           &p.ctl->err);
  if (claimed) a.mf += (uint64_t)deg;
}

// Block-collective publication of the staged entries, as block_flush (whose
// sums and candidates travel elsewhere here).
template <typename OffT>
__device__ __forceinline__ void narrow_flush(Appender<OffT>& a, NarrowShared& sh, Ring* nxt0, Ring* nxt1) {
  const int w = (int)(threadIdx.x >> 6), lane = lane_id(), own = a.c;
  {
    const unsigned long long hd =
        wave_reduce_full_nz_u64<kWaveSum>((uint32_t)lane < a.h.cnt ? (unsigned long long)a.h.d[lane] : 0ull);
    if (lane == 0) {
      sh.cnt[own][w] = a.cnt;
      sh.hcnt[own][w] = a.h.cnt;
      sh.hedges[own][w] = hd;
      sh.cnt[own ^ 1][w] = 0;
      sh.hcnt[own ^ 1][w] = 0;
      sh.hedges[own ^ 1][w] = 0;
    }
  }
  __syncthreads();
  if (lane == 0 && w < 4) {
    const int c = w & 1;
    Ring* nxt = c ? nxt1 : nxt0;
    uint32_t tot = 0;
    unsigned long long e = 0;
    for (int i = 0; i < kNarrowWaves; ++i) {
      uint32_t& k = w < 2 ? sh.cnt[c][i] : sh.hcnt[c][i];
      const uint32_t ki = k;
      k = tot;
      tot += ki;
      if (w >= 2) {
        const unsigned long long ei = sh.hedges[c][i];
        sh.hedges[c][i] = e;
        e += ei;
      }
    }
    if (w < 2)
      sh.base[c] = tot ? atomicAdd(&nxt->n, tot) : 0u;
    else
      sh.hbase[c] =
          tot ? atomicAdd((unsigned long long*)&nxt->hub, ((unsigned long long)tot << kHubEdgeBits) | e) : 0ull;
  }
  __syncthreads();
  const uint32_t base = sh.base[own] + sh.cnt[own][w];
  int32_t* q = a.p->q[own][a.nxt_par];
  for (uint32_t i = (uint32_t)lane; i < a.cnt; i += kWave) {
    if (base + i < a.p->qcap)
      q[base + i] = a.buf[i];
    else
      atomicOr(&a.p->ctl->err, 1u);
  }
  if (a.h.cnt) {
    const unsigned long long hb = sh.hbase[own];
    hub_write(a.h, (uint32_t)(hb >> kHubEdgeBits) + sh.hcnt[own][w], (hb & kHubEdgeMask) + sh.hedges[own][w],
              a.p->hq[own][a.nxt_par], a.p->hb[own][a.nxt_par], a.p->hcap, &a.p->ctl->err);
  }
}

// A block's word at the end of a level: 16 bits of the level's tag, look, and
// the block's claimed vertices of both colours (each at most 2^16 - 1, so that
// the sums over 64 blocks fit their 23 bits).
__device__ __forceinline__ unsigned long long narrow_word(uint32_t tag, bool look, uint32_t n0, uint32_t n1) {
  const uint32_t m0 = n0 < 0xffffu ? n0 : 0xffffu, m1 = n1 < 0xffffu ? n1 : 0xffffu;
  return ((unsigned long long)(tag & 0xffffu) << 48) | (look ? 1ull << 47 : 0ull) | ((unsigned long long)m1 << 23) | m0;
}

template <typename OffT, bool BFS>
__global__ __launch_bounds__(kNarrowThreads) void narrow_kernel(StTeamRun tr) {
  // read with scalar loads (the launch does not write it)
  typedef __attribute__((address_space(4))) const VisitParams<OffT>* params_ptr;
  const VisitParams<OffT>& p = *(const VisitParams<OffT>*)((params_ptr)(uintptr_t)tr.params + xcc_id());
  using Split = NarrowSplit<BFS>;
  constexpr int kColours = Split::kColours, kWorkers = Split::kWorkers, kSets = Split::kSets;
  __shared__ NarrowKept<OffT, BFS> s_kept[kColours];
  __shared__ int32_t s_stage[kNarrowWaves * (kNarrowStage + kNarrowSpill)];
  __shared__ int32_t s_hub[2][kNarrowWaves * kHubStage];
  __shared__ NarrowShared sh;
  __shared__ OffT s_root[4];
  __shared__ int s_num, s_size, s_q, s_ok;
  const int machine = xcc_id();
  TeamSync* ts = tr.sync + machine;
  TeamBar* bar = tr.bar + machine;
  StTeamCtl* ctl = tr.ctl + machine;
  if (threadIdx.x == 0) {
    uint32_t members = 0;
    s_num = team_register(ts, tr.expected, &members);
    if (s_num >= kWave) s_num = -1;  // a wave reads a word of each block
    members = members < kWave ? members : kWave;
    s_size = (int)members;
    if (s_num == 0) {
      st_team(&ctl->q[0], atomicAdd(tr.ticket, 1u));
      __builtin_amdgcn_s_waitcnt(0);
      st_team(&ts->size.v, members);
    } else if (s_num > 0) {
      s_size = team_wait(&ts->size.v, 1u) ? (int)ld_agent(&ts->size.v) : 0;
      if (!s_size) st_agent(tr.err, 1u);
    }
  }
  __syncthreads();
  const int bid = __builtin_amdgcn_readfirstlane(s_num), nb = __builtin_amdgcn_readfirstlane(s_size);
  if (bid < 0 || nb == 0) return;
  const bool lead = bid == 0 && threadIdx.x == 0;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = lane_id();
  // The last wave serves: it ends the levels. The others alternate between the
  // colours (with two, one is left over).
  const bool serve = w == kNarrowWaves - 1, work = w < kWorkers * kColours;
  const int cw = BFS ? 0 : w & 1;
  const int wi = w / kColours, lw = bid * kWorkers + wi, nlw = nb * kWorkers;
  int32_t* const parent = BFS && tr.parents ? p.parent : nullptr;
  NarrowKept<OffT, BFS>& kp = s_kept[cw];
  // this lane's kept entries are ent(0), ent(1), ...: each wave takes 16 in turn
  const int sub = lane & 3;
  auto keep_limit = [](uint32_t part) {
    const uint32_t k = part + part / 4 + 32;
    return k < Split::kKeep ? k : Split::kKeep;
  };
  auto ent = [&](int i) { return (uint32_t)(16 * (i * kWorkers + wi) + (lane >> 2)); };
  uint32_t bars = 0, tag = 0;
  for (uint32_t k = 0;; ++k) {
    const int qp = (int)(k & 3u);
    if (threadIdx.x == 0) {
      s_q = (int)ld_agent(&ctl->q[qp]);
      sh.look[0] = sh.look[1] = 0;
      for (int c = 0; c < kColours; ++c) s_kept[c].n[0] = s_kept[c].n[1] = 0;
    }
    __syncthreads();
    const int q = __builtin_amdgcn_readfirstlane(s_q);
    if (q >= tr.nq) return;
    const int32_t src = p.qs[q], dst = BFS ? -1 : p.qt[q];
    const uint32_t epoch = tr.epoch0 + (uint32_t)q;
    if (threadIdx.x < 2 * kColours)
      s_root[threadIdx.x] = p.off[(threadIdx.x < 2 ? src : dst) + (int)(threadIdx.x & 1)];
    __syncthreads();
    const uint64_t ds = (uint64_t)(s_root[1] - s_root[0]), dt = BFS ? 0ull : (uint64_t)(s_root[3] - s_root[2]);
    if (lead) {
      st_team(&ctl->q[(k + 1) & 3u], atomicAdd(tr.ticket, 1u));
      const int far = (int)((k + 2) & 3u);
      for (int c = 0; c < 2; ++c)
        for (int r = 0; r < 3; ++r) zero_ring(&ctl->ring[far][c][r]);
      ctl->best[far][0] = ctl->best[far][1] = ~0ull;
      ctl->sum[far][0] = ctl->sum[far][1] = 0ull;
      p.sst[src] = st_word(epoch, 0, 0);
      if (!BFS) p.sst[dst] = st_word(epoch, 1, 0);
      if (parent) parent[src] = src;
    }
    Appender<OffT> a;
    a.p = &p;
    a.c = cw;
    a.nfbm = nullptr;
    a.bitmaps = false;
    a.epoch = epoch;
    a.root_own = cw ? dst : src;
    a.root_other = BFS ? -1 : cw ? src : dst;
    a.buf = s_stage + w * (kNarrowStage + kNarrowSpill);
    a.cnt = 0;
    a.mf = 0;
    a.h.u = &s_hub[0][w * kHubStage];
    a.h.d = &s_hub[1][w * kHubStage];
    a.h.cnt = 0;
    int steps = 0, maxf = 1, status = 0;
    int64_t vis_v = kColours, expv = kColours;
    uint64_t mf_done = 0;  // this lane's claimed degrees, but for the last level's
    uint32_t nf0 = 1, nf1 = BFS ? 0u : 1u, kept = 0;
    unsigned long long best = ~0ull;
    bool look = false;
    // the first columns of this lane's kept vertices and what they lead to
    int32_t pu[kSets];
    unsigned long long pw[kSets];
    OffT pb[kSets], pe[kSets];
    auto fresh = [&](int32_t u, unsigned long long word) {
      return u != a.root_own && u != a.root_other && (uint32_t)(word >> 32) != a.epoch;
    };
    for (int L = 0;; ++L) {
      uint32_t n_pub = 0;
      uint64_t h_pub = 0;
      if (L > 0) {
        if (look) {
          auto now = [&](int i) { return (uint64_t)bcast64((int64_t)sh.now[i], 0); };
          best = now(4);
          n_pub = (uint32_t)now(2 * cw);
          h_pub = now(2 * cw + 1);
        }
        vis_v += (int64_t)nf0 + (int64_t)nf1;
        const bool met = !BFS && best != ~0ull;
        if (steps > p.V + 2) status = FC_CAPACITY_STATUS;
        if (!met && !status && (nf0 >= kNarrowMax || nf1 >= kNarrowMax)) status = kTooWide;
        if (met || nf0 == 0 || (!BFS && nf1 == 0) || status) break;
        expv += (int64_t)nf0 + (int64_t)nf1;
        const int32_t mx = (int32_t)(nf0 > nf1 ? nf0 : nf1);
        maxf = mx > maxf ? mx : maxf;
        if (lead) {
          zero_ring(&ctl->ring[qp][0][(L + 2) % 3]);
          if (!BFS) zero_ring(&ctl->ring[qp][1][(L + 2) % 3]);
        }
      }
      ++steps;
      ++tag;
      const int par = L & 1, npar = par ^ 1;
      uint32_t claims = 0;
      a.nxt_par = npar;
      a.nxt = &ctl->ring[qp][cw][(L + 1) % 3];
      a.best = ~0ull;
      a.best_out = &ctl->best[qp][par];
      mf_done += a.mf;
      a.mf = 0;
      auto push = [&](bool claimed, int32_t u, OffT b, int64_t deg) {
        push_kept(a, kp, npar, claims, claimed, u, b, deg);
      };
      if (!work) {
      } else if (L == 0) {
        td_root<true>(a, parent, cw ? dst : src, s_root[2 * cw], s_root[2 * cw + 1], lw, nlw, push);
      } else {
        // kept vertices: their first four columns are here already
        if (ent(0) - (uint32_t)(lane >> 2) < kept) {
          Probe<OffT> r[kSets];
          uint64_t more = 0;
#pragma unroll
          for (int i = 0; i < kSets; ++i) {
            r[i].w = pw[i];
            r[i].old = 0;
            r[i].ob = pb[i];
            r[i].oe = pe[i];
            r[i].tried = pu[i] >= 0 && fresh(pu[i], pw[i]);
            if (r[i].tried) r[i].old = atomicCAS(&p.sst[pu[i]], pw[i], st_word(a.epoch, a.c, L + 1));
            more |= ballot(ent(i) < kept && kp.d[par][ent(i) < kept ? ent(i) : 0] > 4);
          }
#pragma unroll
          for (int i = 0; i < kSets; ++i) {
            const int32_t v = parent && ent(i) < kept ? kp.v[par][ent(i)] : 0;
            int64_t d;
            const bool cl = probe_done(a, parent, true, L, v, pu[i], pu[i] >= 0, r[i], d);
            push(cl, pu[i], r[i].ob, d);
          }
          // and the rest of longer lists
          if (more) {
#pragma unroll 1
            for (int i = 0; i < kSets; ++i) {
              const uint32_t e = ent(i);
              const bool on = e < kept;
              const OffT b = on ? kp.b[par][e] : (OffT)0;
              const int32_t d = on ? kp.d[par][e] : 0, v = on ? kp.v[par][e] : 0;
              for (int32_t j = 4 + sub; ballot(j < d); j += 4) {
                const bool act = j < d;
                const int32_t u = act ? p.col[b + (OffT)j] : 0;
                Probe<OffT> pr = probe_look<true>(a, true, u, act);
                probe_issue(a, true, L, u, act, pr);
                int64_t dg;
                const bool cl = probe_done(a, parent, true, L, v, u, act, pr, dg);
                push(cl, u, pr.ob, dg);
              }
            }
          }
        }
        // Published vertices go to the waves one by one while there are few
        // (they and what they claim stay with their wave), from another wave
        // on at each level.
        if (n_pub) {
          int vw = kWave;
          while (vw > tr.vw_fixed && (uint64_t)n_pub * (uint64_t)vw > (uint64_t)nlw * kWave) vw >>= 1;
          const int at = (int)(((uint32_t)lw + 29u * (uint32_t)L) % (uint32_t)nlw);
          td_normal<true>(a, parent, true, vw, L, par, n_pub, at, nlw, push);
        }
        if (h_pub) td_hubs<true>(a, parent, true, L, par, h_pub, lw, nlw, push);
      }
      // end of the level: publish if a wave of this block has to
      const bool cand = ballot(a.best != ~0ull) != 0;
      if (cand) {
        const unsigned long long b = wave_reduce_full_u64<kWaveMin>(a.best);
        if (lane == 0) atomicMin(a.best_out, b);
      }
      if (lane == 0) {
        sh.claims[w] = claims;
        if (cand || a.cnt || a.h.cnt) sh.look[par] = 1;
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      kept = kp.n[npar];
      // a block with much more than its part of the colour's frontier (as it
      // was at this level) gives away all above that part
      const uint32_t nf = cw ? nf1 : nf0, part = nf / (uint32_t)nb;
      bool flag = __builtin_amdgcn_readfirstlane(sh.look[par]) != 0;
      for (int c = 0; c < kColours; ++c) flag |= s_kept[c].n[npar] > keep_limit((c ? nf1 : nf0) / (uint32_t)nb);
      flag = __builtin_amdgcn_readfirstlane((int)flag) != 0;
      if (serve && lane < kColours) s_kept[lane].n[par] = 0;
      if (kept > keep_limit(part)) {
        const uint32_t end = kept < Split::kKeep ? kept : Split::kKeep, low = part < end ? part : end;
        kept = low;
        const uint32_t e = low + kNarrowSpill * (uint32_t)wi;
        if (work && e < end) {
          const uint32_t k = end - e < kNarrowSpill ? end - e : kNarrowSpill;
          if ((uint32_t)lane < k) a.buf[a.cnt + (uint32_t)lane] = kp.v[npar][e + (uint32_t)lane];
          a.cnt += k;
        }
      }
      if (flag) {
        narrow_flush(a, sh, &ctl->ring[qp][0][(L + 1) % 3], &ctl->ring[qp][1][(L + 1) % 3]);
        a.cnt = 0;
        a.h.cnt = 0;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
      }
      if (serve) {
        __builtin_amdgcn_s_setprio(3);  // before its block's prefetches
        // lanes 0..15: a wave's claims each, colour 1's in the upper half
        const unsigned long long cl = lane < kNarrowWaves ? (unsigned long long)sh.claims[lane] : 0ull;
        const unsigned long long both = (unsigned long long)bcast64(
            (int64_t)row_reduce_u64<kWaveSum>(!BFS && (lane & 1) ? cl << 32 : cl), 15);
        if (lane == 0) {
          sh.look[npar] = 0;  // for the next level; this level's readers have passed
          st_team(&ctl->word[tag & 1][bid], narrow_word(tag, flag, (uint32_t)both, (uint32_t)(both >> 32)));
        }
        const bool on = lane < nb;
        const unsigned long long* const from = &ctl->word[tag & 1][on ? lane : 0];
        unsigned long long x = ld_agent(from);
        uint64_t t0 = 0;
        bool ok = true;
        for (uint32_t i = 1; ballot((uint32_t)(x >> 48) != (tag & 0xffffu)); ++i) {
          if (i % 4096 == 0) {
            if (!t0) t0 = wall_clock64();
            if (wall_clock64() - t0 > kTeamWaitTicks) {
              ok = false;
              break;
            }
          }
          x = ld_agent(from);
        }
        const bool any = ballot((x >> 47) & 1ull) != 0;
        x = on ? x & ((1ull << 46) - 1) : 0ull;
        const unsigned long long sum = (unsigned long long)wave_reduce_full_nz_u64<kWaveSum>(x);
        if (any && ok && lane < 5)
          sh.now[lane] = ld_team(lane < 4 ? reinterpret_cast<const unsigned long long*>(
                                                &ctl->ring[qp][lane >> 1][(L + 1) % 3]) + (lane & 1)
                                          : &ctl->best[qp][par]);
        if (lane == 0) {
          sh.sum = sum | (any ? 1ull << 47 : 0ull);
          s_ok = ok;
        }
      } else {
        // meanwhile the others load the next level's first columns and the
        // state words they lead to
#pragma unroll
        for (int i = 0; i < kSets; ++i) {
          const uint32_t e = ent(i);
          pu[i] = e < kept && sub < kp.d[npar][e] ? p.col[kp.b[npar][e] + (OffT)sub] : -1;
        }
#pragma unroll
        for (int i = 0; i < kSets; ++i) {
          pw[i] = probe_look<true>(a, true, pu[i], pu[i] >= 0).w;
          pb[i] = pe[i] = 0;
          if (pu[i] >= 0) {
            OffT o[2];  // in one load
            __builtin_memcpy(o, p.off + pu[i], sizeof(o));
            pb[i] = o[0];
            pe[i] = o[1];
          }
        }
      }
      __syncthreads();
      if (!__builtin_amdgcn_readfirstlane(s_ok)) {
        if (threadIdx.x == 0) st_agent(tr.err, 1u);
        return;
      }
      const unsigned long long g = (unsigned long long)bcast64((int64_t)sh.sum, 0);
      nf0 = (uint32_t)g & 0x7fffffu;
      nf1 = (uint32_t)(g >> 23) & 0x7fffffu;
      look = (g >> 47) & 1ull;
    }
    // the degree sums of the claimed vertices, all and without the last level's
    {
      const unsigned long long all = (unsigned long long)wave_reduce_full_nz_u64<kWaveSum>(mf_done + a.mf);
      const unsigned long long exp = (unsigned long long)wave_reduce_full_nz_u64<kWaveSum>(mf_done);
      if (lane == 0) {
        sh.sums[0][w] = all;
        sh.sums[1][w] = exp;
      }
      __syncthreads();
      if (threadIdx.x < 2) {
        unsigned long long t = 0;
        for (int i = 0; i < kNarrowWaves; ++i) t += sh.sums[threadIdx.x][i];
        if (t) atomicAdd(&ctl->sum[qp][threadIdx.x], t);
      }
      if (!team_barrier(bar, bid, nb, bars, &s_ok)) {
        if (threadIdx.x == 0) st_agent(tr.err, 1u);
        return;
      }
    }
    if (lead) {
      const bool met = !BFS && best != ~0ull;
      VisitOut o;
      const uint32_t err = ld_team(&ctl->v.err);
      o.status = status ? status : err ? FC_CAPACITY_STATUS : 0;
      o.levels = steps;
      o.depth = met ? steps : 0;
      o.dist = met ? (int32_t)(best >> 32) : -1;
      o.meet = BFS ? machine : met ? (int32_t)(uint32_t)best : -1;  // BFS: whose state words hold the levels
      o.topdown = kColours * steps;
      o.bottomup = 0;
      o.max_frontier = maxf;
      o.visited_vertices = vis_v;
      o.visited_edges = (int64_t)(ds + dt + ld_team(&ctl->sum[qp][0]));
      o.expanded_vertices = expv;
      o.expanded_edges = (int64_t)(ds + dt + ld_team(&ctl->sum[qp][1]));
      o.err = (int32_t)err;
      o.launches = 0;  // the one launch is the call's
      p.out[q] = o;
    }
  }
}

template <typename OffT>
hipError_t launch_narrow(const StTeamRun& tr, bool bfs, int blocks, hipStream_t s) {
  if (bfs)
    hipLaunchKernelGGL((narrow_kernel<OffT, true>), dim3(blocks), dim3(kNarrowThreads), 0, s, tr);
  else
    hipLaunchKernelGGL((narrow_kernel<OffT, false>), dim3(blocks), dim3(kNarrowThreads), 0, s, tr);
  return hipGetLastError();
}

template <typename OffT>
int narrow_occupancy() {
  int a = 0, b = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, narrow_kernel<OffT, true>, kNarrowThreads, 0) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, narrow_kernel<OffT, false>, kNarrowThreads, 0) != hipSuccess)
    return 0;
  return a < b ? a : b;
}

template hipError_t launch_narrow<int32_t>(const StTeamRun&, bool, int, hipStream_t);
template hipError_t launch_narrow<int64_t>(const StTeamRun&, bool, int, hipStream_t);
template int narrow_occupancy<int32_t>();
template int narrow_occupancy<int64_t>();

template <typename OffT>
hipError_t launch_phase(VisitCtl* ctl, int parity, int blocks, bool wide, hipStream_t s) {
  if (wide)
    hipLaunchKernelGGL((phase_kernel<OffT, kWideWaves>), dim3((blocks * kWavesPerBlock + kWideWaves - 1) / kWideWaves),
                       dim3(kWideWaves * kWave), 0, s, ctl, parity);
  else
    hipLaunchKernelGGL((phase_kernel<OffT, kWavesPerBlock>), dim3(blocks), dim3(kBlock), 0, s, ctl, parity);
  return hipGetLastError();
}

template <typename OffT>
int phase_occupancy() {
  int nb = 0, wide = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, phase_kernel<OffT, kWavesPerBlock>, kBlock, 0) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&wide, phase_kernel<OffT, kWideWaves>, kWideWaves * kWave, 0) !=
          hipSuccess)
    return 0;
  return wide < 1 ? 0 : nb;
}

template hipError_t launch_phase<int32_t>(VisitCtl*, int, int, bool, hipStream_t);
template hipError_t launch_phase<int64_t>(VisitCtl*, int, int, bool, hipStream_t);
template int phase_occupancy<int32_t>();
template int phase_occupancy<int64_t>();

}  // namespace fcd
