// opo_handoff.h -- how the blocks of a team agree on their next instance.
//
// One block of the team, the leader, takes indices from the launch's queue and
// publishes one word per turn, (turn << 32) | index; an index past the last
// instance ends the pass.  The other blocks wait for the word of their own
// turn, so the leader must not publish a turn before all have read the one
// before.  The stage waits see to that: a block that has arrived at a stage
// has read its turn, and the leader waits for the first stage's arrivals
// before it ends the second.  Two things keep it so:
//   - only an instance that runs is published (hand_out passes the finished
//     ones over: a turn without stages would have no wait);
//   - a pass of a single stage waits for that stage's arrivals at its end
//     (ends_with_wait), since no later stage does.
// The memory operations come from `Q`, so that the same code runs on a CPU
// under every interleaving (tests/native/handoff_check.cpp).
#pragma once

#ifdef __HIPCC__
#define OPO_HANDOFF __host__ __device__ __forceinline__
#else
#define OPO_HANDOFF inline
#endif

namespace opo {

// Leader: the next running instance (or an index >= total), published as `turn`.
template <typename Q, typename Runs>
OPO_HANDOFF unsigned hand_out(Q &q, unsigned turn, unsigned total, Runs runs) {
  unsigned i = q.take();
  while (i < total && !runs(i)) i = q.take();
  q.publish(((unsigned long long)turn << 32) | i);
  return i;
}

// The others: the index published for `turn`; false on a time-out.  The word
// that was tested is the word that is used: a second read could be a later turn.
template <typename Q> OPO_HANDOFF bool hand_in(Q &q, unsigned turn, unsigned *i) {
  unsigned long long w = 0;
  if (!q.await(turn, &w)) return false;
  *i = (unsigned)w;
  return true;
}
OPO_HANDOFF bool is_turn(unsigned long long w, unsigned turn) { return (unsigned)(w >> 32) == turn; }

// Whether a pass of nz slices (2 nz - 1 stages) waits after its last stage.
OPO_HANDOFF bool ends_with_wait(int nz) { return nz == 1; }

}  // namespace opo
