// Device code shared by the kernels that put several workgroups on an event:
// words in device memory, and which event a workgroup works on.
#pragma once

#include "eikonal_device.hpp"
#include "kernels.hpp"

namespace adt {

using words_t = gptr<int>;

__device__ __forceinline__ int ld_dev(gptr<const int> p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(words_t p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int add_dev(words_t p, int v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Words shared only within an event's XCD: plain stores (they reach its L2)
// and read-modify-writes at its L2.
__device__ __forceinline__ void st_xcd(words_t p, int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int add_xcd(words_t p, int v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
// Keeps the compiler from moving memory accesses across.
__device__ __forceinline__ void code_fence() { asm volatile("" ::: "memory"); }

// The XCD this workgroup runs on.
__device__ __forceinline__ unsigned xcd_id() {
  unsigned x;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
  return x & (kTeamXcds - 1);
}

// What thread 0 of a workgroup keeps between claims.  `rank`: the workgroup's
// arrival number on its XCD; consecutive ranks form groups of per_group, and a
// group takes one event at a time.
struct TeamClaim {
  unsigned xcd;
  int rank;
  unsigned long long* slot;  // the group's word: generation, 1 (being taken) or event + 2
  int gen = 0;               // the group generation this workgroup works on
  int help = -1;             // position in the XCD's list once no event is left to take
  __device__ TeamClaim(TeamShared* sh, unsigned x, int r, int per_group) : xcd(x), rank(r) {
    const int grp = r / per_group;
    slot = &sh->group[x][grp < kTeamGroups ? grp : kTeamGroups - 1];
  }
};

// The next event of thread 0's workgroup, or -1: the one its group has taken,
// else the next of all (the groups take them in order), else, when none is
// left, one of its XCD's that is not `gone(e)`.  `takes(e)`: is it one of this
// kernel's.  A group's word is `being taken` only while a running thread is
// between two instructions here, so the wait for it ends.
template <typename Takes, typename Gone>
__device__ int claim_event(TeamShared* sh, int nev, TeamClaim& C, Takes takes, Gone gone) {
  if (C.help < 0) {
    for (;;) {
      unsigned long long g = __hip_atomic_load(C.slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int gg = (int)(g >> 32);
      const unsigned lo = (unsigned)g;
      if (lo == 1u) {
        __builtin_amdgcn_s_sleep(2);
        continue;
      }
      if (gg > C.gen) {
        C.gen = gg;
        if (lo != 0xffffffffu) return (int)lo - 2;
        C.help = 0;
        break;
      }
      // the generation this workgroup has finished (or none yet): take the next event
      unsigned long long want = g;
      const unsigned long long claim = ((unsigned long long)gg << 32) | 1ull;
      if (__hip_atomic_compare_exchange_strong(C.slot, &want, claim, __ATOMIC_RELAXED,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        int e;
        do {
          e = add_dev((words_t)&sh->next, 1);
        } while (e < nev && !takes(e));
        const unsigned nlo = e < nev ? (unsigned)(e + 2) : 0xffffffffu;
        if (e < nev) {
          const int at = add_dev((words_t)&sh->owned[C.xcd * 16], 1);
          st_dev((words_t)&sh->list[C.xcd * nev + at], e + 1);
        }
        __hip_atomic_store(C.slot, ((unsigned long long)(gg + 1) << 32) | nlo, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  // help with the XCD's other events, starting at a place of its own
  const int n = ld_dev((words_t)&sh->owned[C.xcd * 16]);
  while (C.help < n) {
    const int at = (C.help + C.rank) % n;
    const int e = ld_dev((words_t)&sh->list[C.xcd * nev + at]) - 1;
    ++C.help;
    if (e >= 0 && !gone(e)) return e;
  }
  return -1;
}

}  // namespace adt
