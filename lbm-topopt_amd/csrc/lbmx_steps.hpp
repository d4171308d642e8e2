// Several steps of a 2D sweep in one launch: a workgroup takes a tile of 64 x H nodes through K
// forward (or reverse) steps, with the field between the steps in LDS. Step j of K covers the
// tile and a ring of K - j nodes around it (clipped to the domain), so that the tile's own nodes
// find all they read; the rings' nodes belong to neighbouring tiles, which compute them too.
// Field traffic falls from K reads and K writes of every node to one of each (plus the ring),
// and a launch's fixed costs (dispatch, argument and boundary descriptor loads, the first
// load's latency) are paid once per K steps.
//
// One wave holds one row of the widest region, x0 .. x0 + 63, through all steps (row y0 - (K-1)
// + wave); the ring's columns left and right of those 64, 2 (K-1) per row, are packed into
// further waves. Every wave of a row inside the tile is then exactly one 64-node row segment,
// as in the single-step sweeps: the functional's segment sums add the same values in the same
// order, step after step, and a node's arithmetic, storage rounding and boundary pieces are
// those of the single-step sweeps (same stored bits).
//
// LDS holds the stored encoding S of each population, plane by plane over the widest region
// ((64 + 2(K-1)) x (H + 2(K-1)) cells); two such fields when K > 2, read and written in turn.
// Cells outside the domain hold the mid-way reflections, as the halo does in memory.
#pragma once
#include "lbmx_kernels.hpp"
#include "lbmx_steps_shape.hpp"

namespace lbmx {

// Barrier between steps: the waves wait for their LDS accesses only (loads of the next step's
// fields and stores of this one's results stay in flight).
__device__ __forceinline__ void steps_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// This thread's node.
struct StepsNode {
  int x, y, ring;       // ring: distance from the tile, 0 inside
  bool active;          // in the domain
  bool row;             // the wave holds a row of the tile (not of its ring)
  bool bnd;
  int cell;             // LDS cell
  unsigned int off;     // element offset in the padded layout
  unsigned long long pieces;  // boundary pieces that meet the wave's nodes
};

// Locates the node and, in waves with boundary nodes, stages the wave's boundary pieces in LDS
// (each wave copies what it reads itself; waves that copy the same piece write the same words).
template <class L>
__device__ __forceinline__ StepsNode steps_node(const StepsCommon& c, int x0, int y0, const double* tf, int tf_stride) {
  const int h = c.K - 1;
  const int lane = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  const StepsPlace p = steps_place(c.K, c.H, wave, lane);
  StepsNode n;
  n.row = p.row;
  n.x = x0 + p.dx;
  n.y = y0 + p.dy;
  n.active = p.held && n.x >= 0 && n.x < c.nx && n.y >= 0 && n.y < c.ny;
  n.ring = p.ring;
  n.cell = p.cell;
  n.off = n.active ? layout_off(c.ls, n.x, n.y, 0) : 0u;
  n.bnd = n.active && on_boundary<L>(n.x, n.y, 0, c.nx, c.ny, 1);
  n.pieces = 0;
  if (__ballot(n.bnd) != 0ull && c.nbc > 0) {
    bool meets = false;
    if (lane < c.nbc) {
      const int* b = c.bcs[lane].box;
      const int xa = p.side ? x0 - h : x0, xb = p.side ? x0 + kTileX - 1 + h : x0 + kTileX - 1;
      const int ya = p.side ? y0 - h : y0 + p.dy, yb = p.side ? y0 + c.H - 1 + h : y0 + p.dy;
      meets = (b[0] <= xb) & (b[1] >= xa) & (b[2] <= yb) & (b[3] >= ya);
    }
    n.pieces = __ballot(meets);
    constexpr int W = (int)(sizeof(DevBC) / 4);
    static_assert(sizeof(DevBC) % 8 == 0 && W + kMaxSteps <= kTileX, "a lane copies one word or one time factor");
    const unsigned int* s = reinterpret_cast<const unsigned int*>(c.bcs);
    unsigned int* d = reinterpret_cast<unsigned int*>(pieces_lds);
    double* t = reinterpret_cast<double*>(pieces_lds + (size_t)c.nbc * sizeof(DevBC));
    for (unsigned long long m = n.pieces; m != 0; m &= m - 1) {
      const int b = __builtin_ctzll(m);
      if (lane < W) d[b * W + lane] = s[b * W + lane];
      else if (lane < W + c.K) t[(lane - W) * c.nbc + b] = tf[(lane - W) * tf_stride + b];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  return n;
}
__device__ __forceinline__ const double* steps_tfac(const StepsCommon& c, int j) {  // step j = 1..K
  return reinterpret_cast<const double*>(pieces_lds + (size_t)c.nbc * sizeof(DevBC)) + (j - 1) * c.nbc;
}

template <class L, class T>
__device__ __forceinline__ void steps_bcs(T (&f)[L::Q], const StepsNode& n, const double* tfac) {
  const DevBC* sb = staged_pieces();
  for (unsigned long long m = n.pieces; m != 0; m &= m - 1) {  // increasing piece index
    const int b = __builtin_ctzll(m);
    const DevBC& e = sb[b];
    if (in_box(e.box, n.x, n.y, 0)) bc_node<L, T>(f, e, T(tfac[b]), n.x, n.y, 0);
  }
}
template <class L, class T>
__device__ __forceinline__ void steps_bcs_adj(T (&l)[L::Q], const StepsNode& n) {
  const DevBC* sb = staged_pieces();
  for (unsigned long long m = n.pieces; m != 0;) {  // decreasing piece index
    const int b = 63 - __builtin_clzll(m);
    m &= ~(1ull << b);
    const DevBC& e = sb[b];
    if (in_box(e.box, n.x, n.y, 0)) bc_node_adj<L, T>(l, e);
  }
}

// ---- forward ----
// Stored encodings of a node's post-collision populations into the LDS field at `to`, with the
// reflections of a boundary node where the next step's region reads them.
template <class L, class P, bool TW>
__device__ __forceinline__ void steps_put(typename P::S* to, int cells, int pitch, const StepsNode& n, bool reflect,
                                          const StepsCommon& c, const typename P::T (&f)[L::Q], int t) {
  using S = typename P::S;
  auto put = [&](auto&& enc) __attribute__((always_inline)) {
    static_for<0, L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      to[q * cells + n.cell] = enc(qc);
    });
    if (n.bnd && reflect) {
      static_for<1, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        if constexpr (L::ex[q] != 0 || L::ey[q] != 0) {
          if (leaves<L, q>(n.x, n.y, 0, c.nx, c.ny, 1))
            to[L::opp[q] * cells + n.cell + L::ex[q] + L::ey[q] * pitch] = enc(qc);
        }
      });
    }
  };
  if constexpr (P::stochastic) {
    unsigned int r0, r1;
    sr_words(n.off, t, r0, r1);
    unsigned int e[(L::Q + 1) / 2];
    static_for<0, (L::Q + 1) / 2>([&](auto pc) {
      constexpr int k = decltype(pc)::value, q = 2 * k;
      if constexpr (q + 1 < L::Q)
        e[k] = P::template enc_pair<L, q, q + 1, TW>(f[q], f[q + 1], sr_seed<q, P::kRandomBits>(r0, r1),
                                                     sr_seed<q + 1, P::kRandomBits>(r0, r1));
      else
        e[k] = P::template enc_sr<L, q, false, TW>(0u, f[q], sr_seed<q, P::kRandomBits>(r0, r1));
    });
    put([&](auto qc) -> S {
      constexpr int q = decltype(qc)::value;
      return (q & 1) ? P::template half_of<true>(e[q >> 1]) : P::template half_of<false>(e[q >> 1]);
    });
  } else {
    put([&](auto qc) -> S { return P::template enc<L, decltype(qc)::value>(f[decltype(qc)::value]); });
  }
}

// dst[j - 1]: where the tile's state after step j goes, or null
template <class L, int COLL, int DES, class P>
__device__ __forceinline__ void fwd_steps(const StepsCommon& c, const void* src, void* const* dst, int t0,
                                          const double* tf, int tf_stride, int x0, int y0) {
  using T = typename P::T;
  using S = typename P::S;
  constexpr bool tw = kStoreTwice<P, COLL, DES>;
  const int K = c.K, h = K - 1, pitch = kTileX + 2 * h, cells = pitch * (c.H + 2 * h);
  S* fields = reinterpret_cast<S*>(pieces_lds + steps_pieces_bytes(c.nbc, K));
  const int fstride = (int)((((size_t)cells * L::Q * sizeof(S) + 15) & ~(size_t)15) / sizeof(S));
  T f[L::Q];
  T gam = T(0);
  const StepsNode n = steps_node<L>(c, x0, y0, tf, tf_stride);
  if (n.active) {
    gam = T(static_cast<const typename P::G*>(c.gamma)[n.y * c.nx + n.x]);
    pull_node<L, P, 0>(src, c.ls, n.off, f);
  }
  const int ys = __builtin_amdgcn_readfirstlane(n.y);
  const bool objseg = n.row && c.obj.acc != nullptr && (ys < c.ny) & segment_meets_terms(c.obj, x0, ys, 0);
  const bool objnode = objseg && (n.active & in_some_term<true>(c.obj, n.x, n.y, 0));
  const long long seg = bc_row_index(c.nx, c.ny, x0, ys, 0);
  auto step = [&](int j) __attribute__((always_inline)) {
    if (n.bnd) steps_bcs<L, T>(f, n, steps_tfac(c, j));
    const T temp = objnode ? node_temperature<L>(f) : T(0);
    T rho, jm[3];
    collide<L, COLL, DES, T, tw>(f, gam, c.m, rho, jm);
    double v = 0.0;
    if (objnode) v = double(node_objective<COLL, T, true>(c.obj, rho, jm, temp, n.x, n.y, 0));
    if (dst[j - 1] != nullptr && n.ring == 0)
      store_node<L, P, tw>(dst[j - 1], c.ls, n.off, f, n.bnd, n.x, n.y, 0, c.nx, c.ny, 1, t0 + j - 1);
    return v;
  };
  auto fetch = [&](const S* from) __attribute__((always_inline)) {
    static_for<0, L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      f[q] = P::template dec<L, q>(from[q * cells + n.cell - L::ex[q] - L::ey[q] * pitch]);
    });
  };
  double v = 0.0;
  if (n.active) {
    v = step(1);
    steps_put<L, P, tw>(fields, cells, pitch, n, n.ring <= K - 2, c, f, t0);
  }
  if (objseg) add_segment_sum(c.obj.acc, seg, v, objnode);
  S* cur = fields;
  S* nxt = fields + fstride;
#pragma unroll 1
  for (int j = 2; j <= K; ++j) {
    steps_barrier();
    v = 0.0;
    if (n.active && n.ring <= K - j) {
      fetch(cur);
      v = step(j);
      if (j < K) steps_put<L, P, tw>(nxt, cells, pitch, n, n.ring <= K - j - 1, c, f, t0 + j - 1);
    }
    if (objseg) add_segment_sum(c.obj.acc, seg, v, objnode);
    S* const s = cur;
    cur = nxt;
    nxt = s;
  }
}

// ---- reverse ----
// Reverse steps t, t - 1, .. (step j of K is t - j + 1, on the state s of that time pulled from
// state[j - 1]); between the steps LDS holds the boundary-corrected adjoint m of each node, which
// the next step gathers from x + c_q (the node's own opposite plane where that lies outside).
// Each node's sensitivity terms are added in step order, as the single-step sweeps add them.
template <class L, int COLL, int DES, class P>
__device__ __forceinline__ void adj_steps(const StepsCommon& c, const Layout& ll, const void* const* state,
                                          const void* lam_in, void* lam_out, double* sens, const double* tf,
                                          int tf_stride, int x0, int y0) {
  using T = typename P::T;
  using LS = typename P::LS;
  const int K = c.K, h = K - 1, pitch = kTileX + 2 * h, cells = pitch * (c.H + 2 * h);
  LS* fields = reinterpret_cast<LS*>(pieces_lds + steps_pieces_bytes(c.nbc, K));
  const int fstride = (int)((((size_t)cells * L::Q * sizeof(LS) + 15) & ~(size_t)15) / sizeof(LS));
  T f[L::Q], lam[L::Q];
  T gam = T(0);
  double s = 0.0;
  StepsNode n = steps_node<L>(c, x0, y0, tf, tf_stride);
  const int node = n.y * c.nx + n.x;
  const bool own = n.active && n.ring == 0;
  const unsigned int offl = n.active ? layout_off(ll, n.x, n.y, 0) * (unsigned int)sizeof(LS) : 0u;
  if (n.active) {
    pull_node<L, P, 0>(state[0], c.ls, n.off, f);
    static_for<0, L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      lam[q] = T(ld<LS>(gather_base<L, q, LS>(lam_in, ll), offl));
    });
    gam = T(static_cast<const typename P::G*>(c.gamma)[node]);
    if (own) s = __builtin_nontemporal_load(sens + node);
    if (n.bnd) {
      static_for<1, L::Q>([&](auto qc) {
        constexpr int r = decltype(qc)::value;
        if constexpr (L::ex[r] != 0 || L::ey[r] != 0) {
          if (leaves<L, r>(n.x, n.y, 0, c.nx, c.ny, 1)) lam[r] = T(ld<LS>(own_base<L::opp[r], LS>(lam_in, ll), offl));
        }
      });
    }
  }
  const bool objnode = c.obj.nterm > 0 && (n.active & in_some_term<true>(c.obj, n.x, n.y, 0));
  auto step = [&](int j) __attribute__((always_inline)) {
    if (n.bnd) steps_bcs<L, T>(f, n, steps_tfac(c, j));
    T srcA = 0, srcB[3] = {0, 0, 0}, srcAT = 0;
    if (objnode) {
      T rho, jm[3];
      flow_macros<L>(f, rho, jm);
      const T temp = node_temperature<L>(f);
      static_for<0, kMaxTerms>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        if ((m < c.obj.nterm) & in_box(c.obj.tbox[m], n.x, n.y, 0))
          term_source<T>(c.obj.tkind[m], rho, jm, temp, T(c.obj.time_const * c.obj.tweight[m]), srcA, srcB, srcAT);
      });
    }
    T dg = 0;
    reverse_collide<L, COLL, DES, T>(f, gam, c.m, lam, dg, srcA, srcB, srcAT);
    s += double(dg);
    if (n.bnd) steps_bcs_adj<L, T>(lam, n);
  };
  LS* cur = fields;
  LS* nxt = fields + fstride;
  if (n.active) {
    step(1);
    static_for<0, L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      cur[q * cells + n.cell] = LS(lam[q]);
    });
  }
#pragma unroll 1
  for (int j = 2; j <= K; ++j) {
    const bool now = n.active && n.ring <= K - j;
    // what a step derives from the design value is worth fewer registers than it takes to hold:
    // without this the compiler keeps it across the loop, and the FP64 forms spill
    if constexpr (sizeof(T) == 8) asm volatile("" : "+v"(gam), "+v"(n.cell), "+v"(n.off), "+v"(n.x), "+v"(n.y));
    if (now) pull_node<L, P, 0>(state[j - 1], c.ls, n.off, f);
    steps_barrier();
    if (now) {
      static_for<0, L::Q>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const int at = n.cell + L::ex[q] + L::ey[q] * pitch;
        if constexpr (L::ex[q] != 0 || L::ey[q] != 0) {
          const bool out = n.bnd && leaves<L, q>(n.x, n.y, 0, c.nx, c.ny, 1);
          lam[q] = T(cur[out ? L::opp[q] * cells + n.cell : q * cells + at]);
        } else {
          lam[q] = T(cur[q * cells + at]);
        }
      });
      step(j);
      if (j < K)
        static_for<0, L::Q>([&](auto qc) {
          constexpr int q = decltype(qc)::value;
          nxt[q * cells + n.cell] = LS(lam[q]);
        });
    }
    LS* const x = cur;
    cur = nxt;
    nxt = x;
  }
  if (own) {
    __builtin_nontemporal_store(s, sens + node);
    static_for<0, L::Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      st_nt<LS>(own_base_w<q, LS>(lam_out, ll), offl, LS(lam[q]));
    });
  }
}

template <class L, int COLL, int DES, class P>
__global__ __launch_bounds__(steps_max_waves(0, false) * kTileX) void k_fwd_steps(FwdSteps a) {
  const int tile = xcd_remap(blockIdx.x, a.nblocks);
  fwd_steps<L, COLL, DES, P>(a.c, a.src, a.dst, a.t, a.tf, kMaxBC, (tile % a.nblk_x) * kTileX,
                             (tile / a.nblk_x) * a.c.H);
}
template <class L, int COLL, int DES, class P>
__global__ __launch_bounds__(steps_max_waves(1, sizeof(typename P::T) == 8) * kTileX) void k_adj_steps(AdjSteps a) {
  const int tile = xcd_remap(blockIdx.x, a.nblocks);
  adj_steps<L, COLL, DES, P>(a.c, a.ll, a.state, a.lam_in, a.lam_out, a.sens, a.tf, kMaxBC,
                             (tile % a.nblk_x) * kTileX, (tile / a.nblk_x) * a.c.H);
}

// The workgroup's member of a batch and its tile; fills what the steps need of it.
template <int DIR>
__device__ __forceinline__ ConstInst& steps_locate(const BatchSteps& st, StepsCommon& c, int& inst, int& x0, int& y0) {
  const int b = xcd_remap(blockIdx.x, st.nblocks);
  inst = st.blk_inst[b];
  ConstInst& I = *((ConstInst*)(st.inst) + inst);
  const int tile = b - I.steps_begin[DIR];
  x0 = (tile % I.g.nblk_x) * kTileX;
  y0 = (tile / I.g.nblk_x) * st.H;
  c.nx = I.g.nx;
  c.ny = I.g.ny;
  c.K = st.K;
  c.H = st.H;
  c.nbc = I.nbc;
  c.bcs = I.bcs;
  c.gamma = I.gamma;
  c.ls = from_const(I.ls);
  c.m = from_const(I.m);
  c.obj = from_const(I.obj);
  return I;
}

template <class L, int COLL, int DES, class P>
__global__ __launch_bounds__(steps_max_waves(0, false) * kTileX) void k_fwd_steps_batch(BatchSteps st) {
  StepsCommon c;
  int i, x0, y0;
  ConstInst& I = steps_locate<0>(st, c, i, x0, y0);
  if (!st.with_obj) c.obj.acc = nullptr;
  void* dst[kMaxSteps];
#pragma unroll
  for (int j = 0; j < kMaxSteps; ++j) dst[j] = st.dst[j] ? static_cast<char*>(st.dst[j]) + I.state_off : nullptr;
  fwd_steps<L, COLL, DES, P>(c, static_cast<const char*>(st.state[0]) + I.state_off, dst, st.t,
                             st.tfac + (long long)i * st.tf_stride, st.tf_step, x0, y0);
}
template <class L, int COLL, int DES, class P>
__global__ __launch_bounds__(steps_max_waves(1, sizeof(typename P::T) == 8) * kTileX) void k_adj_steps_batch(BatchSteps st) {
  StepsCommon c;
  int i, x0, y0;
  ConstInst& I = steps_locate<1>(st, c, i, x0, y0);
  c.obj.acc = nullptr;
  if (!st.with_obj) c.obj.nterm = 0;
  const Layout ll = from_const(I.ll);
  const void* state[kMaxSteps];
#pragma unroll
  for (int j = 0; j < kMaxSteps; ++j) state[j] = static_cast<const char*>(st.state[j]) + I.state_off;
  adj_steps<L, COLL, DES, P>(c, ll, state, static_cast<const char*>(st.lam_in) + I.lam_off,
                             static_cast<char*>(st.lam_out) + I.lam_off, I.sens,
                             st.tfac + (long long)i * st.tf_stride, st.tf_step, x0, y0);
}

// ---- host-side launchers ----
template <class L, int COLL, int DES, class P>
hipError_t launch_fwd_steps_t(const FwdSteps& a, hipStream_t s) {
  const size_t lds = steps_pieces_bytes(a.c.nbc, a.c.K) + steps_field_bytes(a.c.K, a.c.H, L::Q, sizeof(typename P::S));
  hipLaunchKernelGGL((k_fwd_steps<L, COLL, DES, P>), dim3(a.nblocks), dim3(kTileX, steps_waves(a.c.K, a.c.H), 1), lds, s,
                     a);
  return hipGetLastError();
}
template <class L, int COLL, int DES, class P>
hipError_t launch_adj_steps_t(const AdjSteps& a, hipStream_t s) {
  const size_t lds = steps_pieces_bytes(a.c.nbc, a.c.K) + steps_field_bytes(a.c.K, a.c.H, L::Q, sizeof(typename P::LS));
  hipLaunchKernelGGL((k_adj_steps<L, COLL, DES, P>), dim3(a.nblocks), dim3(kTileX, steps_waves(a.c.K, a.c.H), 1), lds, s,
                     a);
  return hipGetLastError();
}
template <class L, int COLL, int DES, class P>
hipError_t launch_steps_batch_t(int kind, const BatchSteps& st, hipStream_t s) {
  const size_t elem = kind == 0 ? sizeof(typename P::S) : sizeof(typename P::LS);
  const size_t lds = steps_pieces_bytes(st.tf_stride, st.K) + steps_field_bytes(st.K, st.H, L::Q, elem);
  const dim3 block(kTileX, steps_waves(st.K, st.H), 1);
  if (kind == 0) hipLaunchKernelGGL((k_fwd_steps_batch<L, COLL, DES, P>), dim3(st.nblocks), block, lds, s, st);
  else if constexpr (COLL == C_CASC) return hipErrorInvalidValue;  // (steps_shape: one step per launch)
  else hipLaunchKernelGGL((k_adj_steps_batch<L, COLL, DES, P>), dim3(st.nblocks), block, lds, s, st);
  return hipGetLastError();
}

}  // namespace lbmx
