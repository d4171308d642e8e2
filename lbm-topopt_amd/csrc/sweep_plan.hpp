// The sweeps of a design-gradient pass: run in order over opaque buffers, or as a list of
// operations on numbered buffers, so that consecutive forward steps (and consecutive reverse
// steps) can share a launch. Host code only.
#pragma once
#include <algorithm>
#include <memory>
#include <unordered_map>
#include <utility>
#include <vector>

#include "checkpoint.hpp"
#include "lbmx.h"

namespace lbmx {

// The sweeps of one design-gradient pass, over opaque state buffers (a single lattice, a batch
// of lattices in lockstep, or labelled host buffers that check the schedule).
struct SweepOps {
  virtual ~SweepOps() = default;
  virtual void init(void* dst) = 0;                                              // p_0
  virtual void fwd(const void* src, void* dst, int t, bool with_obj) = 0;       // p_t from p_{t-1}
  virtual void adj(const void* fsrc, const void* lin, void* lout, int t) = 0;  // nu_{t-1} from nu_t
};

struct PassResult {
  long long recompute = 0;  // forward sweeps re-run in the reverse phase
  int max_slots = 0;        // slots in use at most
};

// Forward phase storing checkpoints in `slotbuf` (Wang dynamic checkpointing, or every state
// when naive), then the reverse phase: the adjoint sweep at step t needs p_{t-1}, restored from
// the nearest checkpoint and re-advanced (LBDynamicCheckpointing, src/topOpt/LBCheckpointing.cc:42-48;
// WangCheckpointing::getForwardSolution, src/topOpt/WangCheckpointing.cc:36-126). Storing a
// checkpoint swaps buffer handles (no copy). On return, lin holds the final adjoint nu_0.
inline PassResult checkpointed_pass(SweepOps& ops, int nsteps, bool naive, std::vector<void*>& slotbuf,
                                    void* work0, void* work1, void*& lin, void*& lout, bool with_obj,
                                    int mode = LBMX_CHECKPOINT_DYNAMIC) {
  const int slots = (int)slotbuf.size();
  void* work[2] = {work0, work1};
  auto other_work = [&](const void* src) -> void*& { return src == work[0] ? work[1] : work[0]; };
  std::unique_ptr<WangSchedule> sched;
  if (!naive) {
    sched.reset(new WangSchedule(slots));
    if (mode == LBMX_CHECKPOINT_STATIC) sched->plan_static(nsteps - 1);
    if (mode == LBMX_CHECKPOINT_BINOMIAL) sched->plan_binomial(nsteps);
  }
  PassResult r;
  auto used = [&]() { r.max_slots = std::max(r.max_slots, naive ? slots : slots - sched->free_slots()); };
  ops.init(work[0]);
  auto store = [&](int step, void*& holder) -> void* {
    int s = naive ? step : sched->make_checkpoint(step);
    if (s < 0) return holder;       // a static schedule does not keep this step
    std::swap(slotbuf[s], holder);  // the slot now owns the state; holder gets a spare buffer
    return slotbuf[s];
  };
  void* src = store(0, work[0]);
  used();
  const void* last_input = nullptr;  // p_{nsteps-1}, the input of the last forward sweep
  for (int k = 1; k <= nsteps; ++k) {
    void*& dst = other_work(src);
    if (k == nsteps) last_input = src;
    ops.fwd(src, dst, k, with_obj);
    if (k < nsteps) src = store(k, dst);
    else src = dst;
    used();
  }
  for (int step = nsteps; step >= 1; --step) {
    const int index = step - 1;
    const void* fsrc = nullptr;
    if (naive) {
      fsrc = slotbuf[index];
    } else {
      WangSchedule::Plan plan = sched->get_forward_solution(index);
      if (plan.stored()) {
        // a binomial plan may hand the first reverse step the forward pass's last input
        fsrc = plan.from_slot >= 0 ? slotbuf[plan.from_slot] : last_input;
      } else {
        const void* s2 = slotbuf[plan.from_slot];
        size_t next = 0;
        for (int c = plan.from_step + 1; c <= plan.index; ++c) {
          void*& dst = other_work(s2);
          ops.fwd(s2, dst, c, false);
          ++r.recompute;
          if (next < plan.stores.size() && plan.stores[next].first == c) {
            int s = plan.stores[next].second;
            std::swap(slotbuf[s], dst);
            s2 = slotbuf[s];
            ++next;
          } else {
            s2 = dst;
          }
        }
        fsrc = s2;
      }
      used();
    }
    ops.adj(fsrc, lin, lout, step);
    std::swap(lin, lout);
    if (!naive) sched->release();
  }
  return r;
}

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

// Lists the sweeps of a pass on numbered buffers instead of running them.
struct RecordSweeps : SweepOps {
  std::vector<SweepOp> ops;
  std::unordered_map<const void*, int> id;
  int of(const void* p) { return id.emplace(p, (int)id.size()).first->second; }
  void init(void* dst) override { ops.push_back({SweepOp::kInit, -1, of(dst), 0, false}); }
  void fwd(const void* src, void* dst, int t, bool with_obj) override {
    const int a = of(src), b = of(dst);
    ops.push_back({SweepOp::kFwd, a, b, t, with_obj});
  }
  void adj(const void* fsrc, const void*, void*, int t) override { ops.push_back({SweepOp::kAdj, of(fsrc), -1, t, false}); }
};

// A pass as launches: the checkpointed pass's sweeps, consecutive ones grouped. buffers[i] is
// the buffer that the groups call i.
struct SweepLaunches {
  std::vector<SweepGroup> groups;
  std::vector<void*> buffers;
  PassResult result;
};
inline SweepLaunches plan_launches(int nsteps, bool naive, std::vector<void*> slotbuf, void* work0, void* work1,
                                   bool with_obj, int mode, int max_fwd, int max_adj) {
  RecordSweeps rec;
  std::vector<void*> all(slotbuf);
  all.push_back(work0);
  all.push_back(work1);
  for (void* p : all) rec.of(p);
  SweepLaunches l;
  l.buffers = all;
  char lam[2];
  void *lin = &lam[0], *lout = &lam[1];
  l.result = checkpointed_pass(rec, nsteps, naive, slotbuf, work0, work1, lin, lout, with_obj, mode);
  l.groups = group_sweeps(rec.ops, (int)all.size(), max_fwd, max_adj);
  return l;
}

}  // namespace lbmx
