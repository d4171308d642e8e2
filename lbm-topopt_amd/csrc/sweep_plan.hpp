// The sweeps of a design-gradient pass as a list of operations on numbered buffers, so that
// consecutive forward steps (and consecutive reverse steps) can share a launch.
#pragma once
#include <unordered_map>
#include <utility>
#include <vector>

namespace lbmx {

struct SweepOp {
  enum Kind { kInit, kFwd, kAdj } kind;
  int src;         // buffer read (kFwd: p_{t-1}; kAdj: p_{t-1})
  int dst;         // buffer written (kInit, kFwd)
  int t;           // kFwd: time of the new state; kAdj: reverse step
  bool with_obj;   // kFwd: accumulate the functional
};

// A launch: forward steps t, t + 1, .. from src, whose states go to `buffers` (-1: not kept, the
// last always is); or reverse steps t, t - 1, .. on the states `buffers`; or the initial state
// into buffers[0].
struct SweepGroup {
  SweepOp::Kind kind;
  int src, t;
  bool with_obj;
  std::vector<int> buffers;
  int steps() const { return (int)buffers.size(); }
};

// Groups up to max_fwd consecutive forward steps, and up to max_adj consecutive reverse steps. A
// state in between that nothing but the next step reads is not kept. A group's last state
// goes to the buffer that its step names, unless that is the buffer the group starts from (a
// launch cannot write what its other workgroups still read): then the buffer of a state that
// is not kept takes it, and the two change names from there on.
inline std::vector<SweepGroup> group_sweeps(const std::vector<SweepOp>& ops, int nbuffers, int max_fwd, int max_adj) {
  const int n = (int)ops.size();
  // passing[i]: the state that operation i writes is read by operation i + 1 alone
  std::vector<char> passing((size_t)n, 0);
  {
    // per buffer, scanning backwards: the two nearest accesses (operation, whether it reads)
    struct Access {
      int op = -1;
      bool read = false;
    };
    std::vector<Access> first((size_t)nbuffers), second((size_t)nbuffers);
    auto note = [&](int buf, int op, bool read) {
      second[buf] = first[buf];
      first[buf] = {op, read};
    };
    for (int i = n - 1; i >= 0; --i) {
      const SweepOp& o = ops[i];
      if (o.kind != SweepOp::kAdj) {
        const Access &a = first[o.dst], &b = second[o.dst];
        passing[i] = a.op == i + 1 && a.read && (b.op < 0 || !b.read);
        note(o.dst, i, false);
      }
      if (o.kind != SweepOp::kInit) note(o.src, i, true);
    }
  }
  std::vector<int> name((size_t)nbuffers);  // the buffer that stands for each one now
  for (int b = 0; b < nbuffers; ++b) name[b] = b;
  std::vector<SweepGroup> out;
  for (int i = 0; i < n;) {
    const SweepOp& o = ops[i];
    SweepGroup g{o.kind, -1, o.t, o.with_obj, {}};
    int steps = 1;
    if (o.kind == SweepOp::kAdj) {
      while (steps < max_adj && i + steps < n && ops[i + steps].kind == SweepOp::kAdj && ops[i + steps].t == o.t - steps)
        ++steps;
      for (int k = 0; k < steps; ++k) g.buffers.push_back(name[ops[i + k].src]);
    } else if (o.kind == SweepOp::kInit) {
      g.buffers.push_back(name[o.dst]);
    } else {
      g.src = name[o.src];
      while (steps < max_fwd && i + steps < n) {
        const SweepOp &last = ops[i + steps - 1], &next = ops[i + steps];
        if (next.kind != SweepOp::kFwd || next.src != last.dst || next.t != last.t + 1 || next.with_obj != o.with_obj)
          break;
        ++steps;
      }
      // the longest group that writes no buffer twice and not the one it reads
      int spare = -1;
      for (; steps > 1; --steps) {
        auto kept = [&](int buf) {
          for (int k = 0; k + 1 < steps; ++k)
            if (!passing[i + k] && ops[i + k].dst == buf) return true;
          return false;
        };
        const int dst = ops[i + steps - 1].dst;
        spare = -1;
        if (kept(o.src) || kept(dst)) continue;
        if (dst != o.src) break;
        for (int k = 0; k + 1 < steps && spare < 0; ++k)
          if (passing[i + k] && ops[i + k].dst != o.src && !kept(ops[i + k].dst)) spare = ops[i + k].dst;
        if (spare >= 0) break;
      }
      for (int k = 0; k + 1 < steps; ++k) g.buffers.push_back(passing[i + k] ? -1 : name[ops[i + k].dst]);
      const int dst = ops[i + steps - 1].dst;
      if (steps > 1 && dst == o.src) std::swap(name[dst], name[spare]);
      g.buffers.push_back(name[dst]);
    }
    i += steps;
    out.push_back(std::move(g));
  }
  return out;
}

}  // namespace lbmx
