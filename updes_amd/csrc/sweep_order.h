// Order in which the superblocks of a triangular sweep are counted solved
// (trsv.hip).  Plain C++ as well as device code: a CPU test drives it with
// chunks that count in any order.
#pragma once

#if defined(__HIPCC__)
#define RBFX_HD __host__ __device__
#else
#define RBFX_HD
#endif

namespace rbfx {

// A chunk of superblock s (in solve order) of nch chunks, once its solution
// has arrived in memory.  count_chunk() adds it to the superblock's chunks and
// returns the number before it; wait_solved(s) returns once s superblocks are
// counted solved (false: the sweep failed); set_solved(v) makes it v.
//
// Chunks start on the published values of their predecessor, not on its
// count, so the last chunk of superblock s may get here before the last one of
// s - 1: it waits, so that a count of v always stands for the superblocks
// 0 .. v-1, whose plain solution may then be read.
template <class CountChunk, class WaitSolved, class SetSolved>
RBFX_HD inline void count_solved(unsigned s, unsigned nch, CountChunk&& count_chunk, WaitSolved&& wait_solved,
                                 SetSolved&& set_solved) {
  if (count_chunk() != nch - 1) return;
  if (wait_solved(s)) set_solved(s + 1);
}

}  // namespace rbfx
