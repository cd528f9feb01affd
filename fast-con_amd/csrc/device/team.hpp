// Teams: the blocks of one launch that run on one XCD and work together
// without ending the launch.
//
// MI355X has eight XCDs of 32 CUs with an L2 each. A barrier over the whole
// grid needs agent-scope fences, which write back and invalidate every L2
// (16-35 us), so grid-wide steps are separate launches. Blocks of one XCD
// share its L2, and there a barrier needs neither: it costs a store per block
// and the loads that see it, 0.6 us, against 8-20 us from one dependent
// launch to the next. Measured on this card with data written
// by plain stores and atomics and read by other CUs of the XCD:
//  * stores and atomics go through the L1 to the L2 (atomics on to the
//    memory side, 27 G/s over the chip whatever their scope), and a wave's
//    are there when its memory counter is zero (s_waitcnt);
//  * a plain load may hit a line that its own CU's L1 has kept, an
//    agent-scope load (sc1) never does: it reads the L2 at the same cost as
//    any L1 miss (90 ns, 250 G/s over the chip). So a team loads whatever
//    another block may have written in this launch with ld_team, and only
//    arrays that the launch never writes (the graph, the queries) plainly.
// An invalidation of the L1 (buffer_inv sc1) at each barrier would allow
// plain loads, but costs 60 ns a block, one after another.
//
// Membership is decided by the hardware: a block reads the XCD it runs on
// and takes a number there; the first one closes the XCD's registration when
// the expected blocks are there, or after a short wait when other work holds
// the CUs. A block that comes later leaves at once. All members are then
// resident and running, so a team's barriers end whatever else the GPU does;
// all the same every wait is bounded by the clock.
#pragma once

#include "wave.hpp"

namespace fcd {

constexpr int kXcds = 8;                   // XCD numbers 0..7
constexpr uint32_t kTeamClosed = 0x80000000u;
constexpr uint32_t kTeamMax = 128;         // blocks of a team: two words per lane of the wave that waits for them
constexpr uint64_t kTeamJoinTicks = 2000;  // 20 us at 100 MHz: registration closes at the latest
constexpr uint64_t kTeamWaitTicks = 2000000000ull;  // 20 s: a wait that has failed

// One 128-byte line per word that blocks of a team poll or count on.
struct alignas(128) TeamWord {
  uint32_t v;
  uint32_t pad[31];
};

// Per XCD; cleared before each launch.
struct TeamSync {
  TeamWord reg;     // blocks registered; kTeamClosed once closed
  TeamWord size;    // members, published when the team's state is ready
};

// Blocks with blockIdx % kXcds = k run on one XCD; the number is read from
// the hardware register, so nothing depends on that.
__device__ __forceinline__ int xcc_id() {
  constexpr int kHwRegXccId = 20;
  return (int)__builtin_amdgcn_s_getreg(kHwRegXccId | (3 << 11)) & (kXcds - 1);  // bits 0..3
}

template <typename T>
__device__ __forceinline__ T ld_team(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A store that other blocks of the XCD see with ld_team: to the L2 and no
// further, in one piece. The compiler keeps it behind the accesses before it;
// that those are out is the caller's wait.
template <typename T>
__device__ __forceinline__ void st_team(T* p, T v) {
  asm volatile("" ::: "memory");
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The number of the block that counted k on the registration word of a team
// for which `expected` blocks were planned, or -1: closed, or full. What a
// team's blocks own (tables, state words) is laid out for `expected` of them,
// and no placement of a launch's blocks on the XCDs may put more to work.
__host__ __device__ constexpr uint32_t team_full(uint32_t expected) { return expected < kTeamMax ? expected : kTeamMax; }
__host__ __device__ constexpr int team_admit(uint32_t k, uint32_t expected) {
  return (k & kTeamClosed) || k >= team_full(expected) ? -1 : (int)k;
}

// Register with the XCD's team (one thread). Returns this block's number, or
// -1 when registration is closed. *members is set for number 0 only, which
// has closed the registration and publishes the size itself (team_publish).
__device__ __forceinline__ int team_register(TeamSync* ts, uint32_t expected, uint32_t* members) {
  const uint32_t k = __hip_atomic_fetch_add(&ts->reg.v, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int number = team_admit(k, expected);
  if (number == 0) {
    const uint64_t t0 = wall_clock64();
    while (ld_agent(&ts->reg.v) < expected && wall_clock64() - t0 < kTeamJoinTicks) __builtin_amdgcn_s_sleep(1);
    const uint32_t n =
        __hip_atomic_fetch_or(&ts->reg.v, kTeamClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ~kTeamClosed;
    *members = n < team_full(expected) ? n : team_full(expected);
  }
  return number;
}

// Wait until the counter *p has reached v (one thread; a difference, so that
// it may wrap). False when the wait was given up.
__device__ __forceinline__ bool team_wait(const uint32_t* p, uint32_t v) {
  uint64_t t0 = 0;
  for (uint32_t i = 1; (int32_t)(ld_team(p) - v) < 0; ++i) {
    if (i % 4096) continue;
    if (!t0) t0 = wall_clock64();
    if (wall_clock64() - t0 > kTeamWaitTicks) return false;
  }
  return true;
}

// A team's barriers. Block bid stores the count of barriers it has reached in
// a word of its own, and a wave of each block that waits reads the words of
// all nb blocks. Nothing is counted with atomics (300 ns each, 13 ns more for
// every other block's), and the store stays in the L2: a barrier of 64 blocks
// takes 0.6 us, where an atomic arrival and a polled word took 1.9.
struct alignas(128) TeamBar {
  uint32_t at[kTeamMax];
};
// The block's stores are out and all its threads have passed a __syncthreads
// (one thread).
__device__ __forceinline__ void team_arrive(TeamBar* bar, int bid, uint32_t passed) {
  st_team(&bar->at[bid], passed);
}
// Wait until all nb blocks have reached barrier `passed` (one wave). False when
// the wait was given up.
__device__ __forceinline__ bool team_all(const TeamBar* bar, int nb, uint32_t passed) {
  const int lane = lane_id();
  const uint32_t* const a = &bar->at[lane < nb ? lane : 0];
  const uint32_t* const b = &bar->at[lane + kWave < nb ? lane + kWave : 0];
  const bool two = nb > kWave;
  uint64_t t0 = 0;
  for (uint32_t i = 1;; ++i) {
    const int32_t da = (int32_t)(ld_team(a) - passed), db = two ? (int32_t)(ld_team(b) - passed) : 0;
    if (!ballot(da < 0 || db < 0)) return true;
    if (i % 4096 == 0) {
      if (!t0) t0 = wall_clock64();
      if (wall_clock64() - t0 > kTeamWaitTicks) return false;
    }
  }
}
// Every store of the nb blocks is in the L2 when one passes. ok: an LDS word of
// the block. Returns (to all threads) whether the barrier was reached by all.
__device__ __forceinline__ bool team_barrier(TeamBar* bar, int bid, int nb, uint32_t& passed, int* ok) {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  ++passed;
  if (threadIdx.x < kWave) {
    if (threadIdx.x == 0) team_arrive(bar, bid, passed);
    const bool all = team_all(bar, nb, passed);
    if (threadIdx.x == 0) *ok = all;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*ok) != 0;
}

}  // namespace fcd
