// Replays the launches that plan_launches groups from a checkpointed pass on labelled buffers:
// every launch has to read the states that its steps need, and none may write the state it
// reads or a buffer twice. Arguments: none; prints "RESULT OK" at the end.
#include <cstdio>
#include <string>

#include "sweep_plan.hpp"

using namespace lbmx;

static const char* replay(int nsteps, bool naive, int slots, int mode, int fwd, int adj) {
  std::vector<char> storage(slots + 2);  // distinct addresses stand for buffers
  std::vector<void*> slotbuf(slots);
  for (int k = 0; k < slots; ++k) slotbuf[k] = &storage[k];
  const SweepLaunches l =
      plan_launches(nsteps, naive, slotbuf, &storage[slots], &storage[slots + 1], true, mode, fwd, adj);
  std::vector<int> label(l.buffers.size(), -1);
  int next = nsteps, functional = 0;
  for (const SweepGroup& g : l.groups) {
    if (g.steps() < 1 || g.steps() > (g.kind == SweepOp::kAdj ? adj : g.kind == SweepOp::kFwd ? fwd : 1))
      return "a launch of too many steps";
    if (g.kind == SweepOp::kFwd && label[g.src] != g.t - 1) return "forward steps read a wrong state";
    std::vector<char> written(l.buffers.size(), 0);
    for (int j = 0; j < g.steps(); ++j) {
      const int b = g.buffers[j];
      if (g.kind == SweepOp::kAdj) {
        if (label[b] != g.t - j - 1 || g.t - j != next) return "a reverse step reads a wrong state";
        --next;
        continue;
      }
      if (g.kind == SweepOp::kFwd && g.with_obj) ++functional;
      if (b < 0) {
        if (j + 1 == g.steps()) return "a launch without a result";
        continue;
      }
      if (b == g.src) return "a launch writes the state it reads";
      if (written[b]) return "a launch writes a buffer twice";
      written[b] = 1;
      label[b] = g.kind == SweepOp::kInit ? 0 : g.t + j;
    }
  }
  if (next != 0) return "reverse steps are missing";
  if (functional != nsteps) return "the functional is not accumulated once per step";
  return nullptr;
}

int main() {
  const int modes[3] = {LBMX_CHECKPOINT_DYNAMIC, LBMX_CHECKPOINT_STATIC, LBMX_CHECKPOINT_BINOMIAL};
  for (int n : {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 13, 37, 60, 100, 200, 1000, 3000})
    for (int slots : {0, 2, 3, 4, 5, 6, 8, 10, 16, 30, 48, 64})
      for (int mode : modes)
        for (int fwd = 1; fwd <= 4; ++fwd)
          for (int adj = 1; adj <= 4; ++adj) {
            if (n >= 1000 && (fwd < 3 || adj != 3)) continue;
            const bool naive = slots == 0;
            const int held = naive ? n : std::min(slots, std::max(2, n));
            if (const char* e = replay(n, naive, held, mode, fwd, adj)) {
              std::printf("steps %d slots %d mode %d groups of %d / %d: %s\n", n, slots, mode, fwd, adj, e);
              return 1;
            }
          }
  std::printf("RESULT OK\n");
  return 0;
}
