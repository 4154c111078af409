// CPU driver of updes_amd/csrc/sweep_order.h, built by tests/test_sweep_order.py:
// the chunks of a sweep, in random orders that the published values allow.
// Prints "ok" and exits 0 when the count of solved superblocks never ran
// ahead of a superblock whose solution is not all in memory.
#include <stdio.h>

#include <random>
#include <vector>

#include "../updes_amd/csrc/sweep_order.h"

struct Sweep {
  unsigned nsb, nch;
  std::mt19937 rng;
  std::vector<unsigned> published, stored, counted;  // chunks of each superblock
  unsigned solved = 0;
  bool ok = true;

  Sweep(unsigned nsb_, unsigned nch_, unsigned seed)
      : nsb(nsb_), nch(nch_), rng(seed), published(nsb_), stored(nsb_), counted(nsb_) {}

  // one random step of any chunk that can take one; false when there is none.
  // Chunks of superblocks from `below` on count later: they come after the
  // chunk that waits in this very call chain.
  bool step(unsigned below) {
    struct Event { unsigned s, kind; };
    std::vector<Event> can;
    for (unsigned s = 0; s < nsb; ++s) {
      // the tagged values of the whole predecessor are what a chunk waits for
      if (published[s] < nch && (s == 0 || published[s - 1] == nch)) can.push_back({s, 0});
      if (stored[s] < published[s]) can.push_back({s, 1});
      if (s < below && counted[s] < stored[s]) can.push_back({s, 2});
    }
    if (can.empty()) return false;
    const Event e = can[rng() % can.size()];
    if (e.kind == 0) {
      ++published[e.s];
    } else if (e.kind == 1) {
      ++stored[e.s];
    } else {
      rbfx::count_solved(
          e.s, nch, [&]() { return counted[e.s]++; },
          [&](unsigned want) {
            while (solved < want)
              if (!step(e.s)) return false;  // nothing left that could satisfy the wait
            return true;
          },
          [&](unsigned v) {
            solved = v;
            for (unsigned s = 0; s < v; ++s) ok = ok && stored[s] == nch;
          });
    }
    return true;
  }
};

int main() {
  for (unsigned seed = 0; seed < 2000; ++seed) {
    Sweep w(1 + seed % 7, 1 + seed % 5, seed);
    while (w.step(w.nsb)) {
    }
    if (!w.ok || w.solved != w.nsb) {
      fprintf(stderr, "seed %u: %s, solved %u of %u\n", seed, w.ok ? "in order" : "counted ahead", w.solved, w.nsb);
      return 1;
    }
  }
  printf("ok\n");
  return 0;
}
