// What the waves of a workgroup of fwd3_team_kernel decide together.  Plain C++
// (no device code), so that a test can run it on the CPU with waves that lag.
#pragma once

#if defined(__HIP__)
#define ADT_GATE __device__ __forceinline__
#else
#define ADT_GATE inline
#endif

namespace adt {

// What the workgroup does next, in LDS.  The leader writes team, ticket and quit
// before a barrier of its own, `over` in team_gate.
struct TDraw {
  int team;    // index of the event's team descriptor, -1: leave
  int ticket;
  int quit;    // the event was finished or aborted when the item was drawn
  int over;    // or while the item waited for the items before it
};

// Is the item dropped?  `end`: it lies past the last iteration; `waits`: it has
// to wait for others' items (the leader does: wait() is true if the event is gone).
// Every wave has to come to the same answer by the same barriers, so what the
// leader learns goes into a word of its own: a wave may read `quit` only after the
// leader has waited.  read(x): x in every lane; sync(): the workgroup's barrier.
template <typename Draw, typename Read, typename Wait, typename Sync>
ADT_GATE bool team_gate(Draw& d, bool end, bool waits, bool leader, Read read, Wait wait,
                        Sync sync) {
  if (read(d.quit) || end) return true;
  if (!waits) return false;
  if (leader) d.over = wait() ? 1 : 0;
  sync();
  return read(d.over) != 0;
}

}  // namespace adt
