"""Timed cases of the framework: what a topology optimisation program has it do.

Each case is one call sequence through the public entry points (lbmx.Solver, lbmx.Batch,
lbmx.Filter, lbmx.MMA, lbmx_torch): a forward run, a design gradient, the gradients of a robust
ensemble, the design filter chain with its sensitivities, or one design update. exact() gives
the same outputs from plain torch in 64 bits: the lattice Boltzmann step written out on dense
tensors, its gradient by automatic differentiation, the cone filter as a sum of shifted fields,
and the MMA update on whole vectors.
"""
import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lbm-topopt_amd"))

import lbmx  # noqa: E402
import lbmx_torch  # noqa: E402
import workloads  # noqa: E402

PRECISION = {"f64": lbmx.FP64, "f32": lbmx.FP32, "f16": lbmx.FP16_SHIFTED, "bf16": lbmx.BF16_SHIFTED}
MODE = {"dynamic": lbmx.CHECKPOINT_DYNAMIC, "static": lbmx.CHECKPOINT_STATIC, "binomial": lbmx.CHECKPOINT_BINOMIAL}
COLLISION = {"bgk": lbmx.BGK, "mrt": lbmx.MRT, "cascaded": lbmx.CASCADED}
LATTICE = {"channel": lbmx.D2Q9, "pump": lbmx.D2Q9, "thermal": lbmx.D2Q9_D2Q5, "duct": lbmx.D3Q19}
Q_OF = {"channel": 9, "pump": 9, "thermal": 14, "duct": 19}
OMEGA = {"channel": 1.0 / 0.8, "pump": 1.0 / 0.8, "thermal": 1.25, "duct": 1.6}


def listed():
    return [
        # a solver checked or tuned on a coarse channel: many steps on a grid that does not fill the GPU
        dict(name="forward_channel_256x128_f64", kind="forward", problem="channel", collision="bgk", precision="f64",
             nx=256, ny=128, nz=1, steps=1000),
        # the smallest gradient: the miniature channel, through the autograd binding, default checkpoints
        dict(name="gradient_channel_48x24_f64", kind="gradient", problem="channel", collision="mrt", precision="f64",
             nx=48, ny=24, nz=1, steps=60, slots=64, mode="dynamic", autograd=True),
        # the unsteady pump: modulated inlet, dissipated power, one optimisation iteration's gradient
        dict(name="gradient_pump_1024x512_f64", kind="gradient", problem="pump", collision="bgk", precision="f64",
             nx=1024, ny=512, nz=1, steps=200, slots=12, mode="dynamic", autograd=False),
        # the same pump in the 16-bit storage form
        dict(name="gradient_pump_1024x512_f16", kind="gradient", problem="pump", collision="bgk", precision="f16",
             nx=1024, ny=512, nz=1, steps=200, slots=12, mode="binomial", autograd=False),
        # thermal channel, double distribution, the largest 2D grid
        dict(name="gradient_thermal_2048x1024_f64", kind="gradient", problem="thermal", collision="mrt",
             precision="f64", nx=2048, ny=1024, nz=1, steps=60, slots=7, mode="binomial", autograd=False),
        # the headline duct: D3Q19 MRT with Brinkman drag, plain FP64
        dict(name="gradient_duct_384x192x192_f64", kind="gradient", problem="duct", collision="mrt", precision="f64",
             nx=384, ny=192, nz=192, steps=24, slots=5, mode="binomial", autograd=False),
        # the headline duct in the 16-bit storage form
        dict(name="gradient_duct_384x192x192_f16", kind="gradient", problem="duct", collision="mrt", precision="f16",
             nx=384, ny=192, nz=192, steps=24, slots=5, mode="binomial", autograd=False),
        # a small duct of odd sizes in single precision, every state stored
        dict(name="gradient_duct_101x47x53_f32", kind="gradient", problem="duct", collision="mrt", precision="f32",
             nx=101, ny=47, nz=53, steps=40, slots=64, mode="dynamic", autograd=False),
        # the robust ensemble: 3 projection realisations x 8 candidates on uneven grids
        dict(name="ensemble_24_cascaded_f32", kind="ensemble", collision="cascaded", precision="f32", candidates=8,
             scale=1.0, steps=48, slots=6, mode="binomial"),
        # robust pump filter chain (radii 8 and 4) on its 2D grid: design and sensitivities
        dict(name="filter_1024x512_r8_r4", kind="filter", nx=1024, ny=512, nz=1, radius0=8, radius1=4, stages=2,
             beta=2.0),
        # 3D projection filter of the duct
        dict(name="filter_384x192x192_r3", kind="filter", nx=384, ny=192, nz=192, radius0=3, radius1=1, stages=1,
             beta=2.0),
        # the design update of the robust pump: three realisations and a volume constraint
        dict(name="mma_524288_m4", kind="mma", n=524288, m=4, movlim=0.1),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["forward", "gradient", "gradient", "gradient", "ensemble", "filter", "mma"])
    if kind in ("forward", "gradient"):
        problem = rng.choice(["channel", "pump", "thermal", "duct"])
        collision = {"channel": rng.choice(["bgk", "mrt", "cascaded"]), "pump": rng.choice(["bgk", "mrt"]),
                     "thermal": rng.choice(["bgk", "mrt"]), "duct": rng.choice(["bgk", "mrt"])}[problem]
        largest = 1e6 if kind == "forward" else {"channel": 524288, "pump": 524288, "thermal": 2.0e6, "duct": 14.0e6}[problem]
        nodes = _log(rng, 1.2e3 if problem != "duct" else 6e3, largest)
        if problem == "duct":
            ny = max(8, int(round((nodes / 2) ** (1 / 3) * rng.uniform(0.8, 1.2))))
            nz = max(8, int(round((nodes / 2) ** (1 / 3) * rng.uniform(0.8, 1.2))))
            nx = max(8, int(nodes / (ny * nz)))
        else:
            ny = max(8, int(round(math.sqrt(nodes / 2) * rng.uniform(0.7, 1.4))))
            nz, nx = 1, max(8, int(nodes / ny))
        most = {"channel": 1e8, "pump": 1e8, "thermal": 1.2e8, "duct": 3.3e8}[problem]
        if kind == "forward":
            steps = int(max(4, min(_log(rng, 50, 1000), most / (nx * ny * nz))))
            return dict(kind=kind, problem=problem, collision=collision, precision=rng.choice(list(PRECISION)),
                        nx=nx, ny=ny, nz=nz, steps=steps)
        steps = int(max(4, min(_log(rng, 20, 200), most / (nx * ny * nz))))
        slots = rng.choice([64, max(3, steps // 4), max(3, steps // 12)])
        if nodes > 3e6:
            slots = min(slots, 8)
        return dict(kind=kind, problem=problem, collision=collision, precision=rng.choice(list(PRECISION)), nx=nx,
                    ny=ny, nz=nz, steps=steps, slots=slots, mode=rng.choice(list(MODE)), autograd=rng.random() < 0.25)
    if kind == "ensemble":
        return dict(kind=kind, collision=rng.choice(["cascaded", "mrt"]), precision=rng.choice(["f32", "f64", "f16"]),
                    candidates=rng.randint(1, 8), scale=rng.uniform(0.25, 1.0), steps=rng.randint(12, 48),
                    slots=rng.randint(4, 12), mode=rng.choice(list(MODE)))
    if kind == "filter":
        if rng.random() < 0.5:
            n = _log(rng, 2e3, 2e6)
            ny = max(16, int(math.sqrt(n / 2) * rng.uniform(0.7, 1.4)))
            return dict(kind=kind, nx=max(16, int(n / ny)), ny=ny, nz=1, radius0=rng.randint(2, 12),
                        radius1=rng.randint(1, 6), stages=rng.randint(1, 2), beta=rng.uniform(1.0, 8.0))
        n = _log(rng, 1e4, 14e6)
        ny = max(10, int((n / 2) ** (1 / 3) * rng.uniform(0.8, 1.2)))
        nz = max(10, int((n / 2) ** (1 / 3) * rng.uniform(0.8, 1.2)))
        return dict(kind=kind, nx=max(10, int(n / (ny * nz))), ny=ny, nz=nz, radius0=rng.randint(1, 3), radius1=1,
                    stages=1, beta=rng.uniform(1.0, 8.0))
    return dict(kind=kind, n=int(_log(rng, 1e3, 4e6)), m=rng.randint(1, 6), movlim=rng.choice([0.05, 0.1, 0.2]))


# ---- inputs -----------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 77)
    return g


def _design(nx, ny, nz, gen):
    """gamma: a uniform random field smoothed over 5 nodes per axis (truncated at the edges)."""
    g = torch.rand((1, 1, nz, ny, nx), generator=gen, device="cuda", dtype=torch.float64)
    k = (1 if nz == 1 else 5, 5, 5)
    g = F.avg_pool3d(g, k, stride=1, padding=tuple(v // 2 for v in k), count_include_pad=False)
    return g.reshape(-1).contiguous()


def _initial(case):
    return dict(u0=(0.03, 0.0, 0.0), T0=0.5) if case["problem"] == "thermal" else {}


def _solver(case):
    p, nx, ny, nz = case["problem"], case["nx"], case["ny"], case["nz"]
    pbb = case["collision"] == "cascaded"
    s = lbmx.Solver(lbmx.make_desc(
        nx, ny, nz, lattice=LATTICE[p], collision=COLLISION[case["collision"]],
        design=lbmx.DESIGN_PBB if pbb else lbmx.DESIGN_BRINKMAN, precision=PRECISION[case["precision"]],
        omega=OMEGA[p], interp_q=0.1, alpha_max=1.0 if pbb else 0.1, thermal_diffusivity=0.02, ramp_p=1.0, ramp_ck=0.1))
    tc = 1.0 / case["steps"]
    if p == "channel":
        workloads.channel2d(s, nx, ny, time_const=tc)
    elif p == "pump":
        workloads.modulated_channel(s, nx, ny, steps=case["steps"])
    elif p == "thermal":
        workloads.thermal_channel2d(s, nx, ny, time_const=tc)
    else:
        workloads.duct3d(s, nx, ny, nz, time_const=tc)
    return s


def _ensemble_grids(case):
    """The uneven candidate grids of the robust ensemble, scaled."""
    return [(max(48, int(nx * case["scale"])), max(24, int(ny * case["scale"])))
            for nx, ny in workloads.ENSEMBLE_GRIDS[8 - case["candidates"]:]]


def _ensemble_inputs(case, seed):
    """(nx, ny, projected design) of every member, candidate by candidate."""
    out = []
    for c, (nx, ny) in enumerate(_ensemble_grids(case)):
        raw = workloads.ensemble_candidate(nx, ny, 1000 * (seed + 1) + c)
        for eta in workloads.ENSEMBLE_ETAS:
            g = workloads.heaviside_project(raw, 8.0, eta)
            out.append((nx, ny, torch.as_tensor(g, dtype=torch.float64, device="cuda")))
    return out


def _filter_stages(case):
    st = [(case["radius0"], True, case["beta"], 0.5), (case["radius1"], True, 1.0, 0.5)]
    return st[:case["stages"]]


def _filter_inputs(case, seed):
    """A design over the inner box (a margin of the radius around it) and a full-grid sensitivity."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    mx, my, mz = min(nx // 16, 16), min(ny // 16, 16), (min(nz // 16, 16) if nz > 1 else 0)
    box = (mx, nx - 1 - mx, my, ny - 1 - my, mz, nz - 1 - mz)
    gen = _generator(seed)
    nd = (box[1] - box[0] + 1) * (box[3] - box[2] + 1) * (box[5] - box[4] + 1)
    design = torch.rand(nd, generator=gen, device="cuda", dtype=torch.float64)
    sens = torch.randn(nx * ny * nz, generator=gen, device="cuda", dtype=torch.float64)
    return box, design, sens


def _mma_inputs(case, seed):
    """Targets and weights of the realisations of a robust problem; the last of several constraints is the volume."""
    gen = _generator(seed)
    n, m = case["n"], case["m"]
    r = max(1, m - 1)
    targets = [0.2 + 0.6 * torch.rand(n, generator=gen, device="cuda", dtype=torch.float64) for _ in range(r)]
    weights = [1.0 + 0.3 * ((3 * k) % 5 - 2) / 2.0 for k in range(r)]
    return targets, weights


def _mma_problem(case, x, targets, weights):
    """dfdx, constraint values and their sensitivities at x."""
    n, m = case["n"], case["m"]
    rows, vals = [], []
    for t, w in list(zip(targets, weights))[:m if m == 1 else m - 1]:
        rows.append((2 * w / n) * (x - t))
        vals.append(w * ((x - t) ** 2).sum() / n)
    if m == 1:  # one objective under the volume constraint
        return rows[0] * n, [float(x.mean()) - 0.4], [torch.full_like(x, 1.0 / n)]
    rows.append(torch.full_like(x, 1.0 / n))
    vals.append(x.mean() - 0.45)
    return torch.zeros_like(x), [float(v) for v in vals], rows


def _mma_constants(case):
    m = case["m"]
    return [0.0] if m == 1 else [1.0] * (m - 1) + [0.0]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        s = _solver(case)
        gamma = _design(case["nx"], case["ny"], case["nz"], _generator(seed))
        if kind == "gradient":
            s.checkpoint_config(case["slots"], MODE[case["mode"]])
            if case["autograd"]:
                gamma.requires_grad_(True)
        return dict(case=case, solver=s, gamma=gamma, start=_initial(case))
    if kind == "ensemble":
        members, designs = [], []
        for nx, ny, g in _ensemble_inputs(case, seed):
            s = lbmx.Solver(lbmx.make_desc(nx, ny, lattice=lbmx.D2Q9, collision=COLLISION[case["collision"]],
                                           design=lbmx.DESIGN_PBB, precision=PRECISION[case["precision"]],
                                           omega=1.0 / 0.6, interp_q=0.1, alpha_max=1.0))
            workloads.channel2d(s, nx, ny, time_const=1.0 / case["steps"])
            members.append(s)
            designs.append(g)
        b = lbmx.Batch(members)
        b.checkpoint_config(case["slots"], MODE[case["mode"]])
        return dict(case=case, members=members, designs=designs, batch=b)
    if kind == "filter":
        box, design, sens = _filter_inputs(case, seed)
        f = lbmx.Filter(lbmx.make_filter_desc(case["nx"], case["ny"], case["nz"], lbmx.make_box(*box),
                                              stages=_filter_stages(case)))
        return dict(case=case, filter=f, design=design, sens=sens)
    # a running optimisation: three updates done, the next one's inputs in hand
    targets, weights = _mma_inputs(case, seed)
    mma = lbmx.MMA(case["n"], case["m"], a=_mma_constants(case))
    x = torch.full((case["n"],), 0.5, device="cuda", dtype=torch.float64)
    for _ in range(3):
        df, g, dg = _mma_problem(case, x, targets, weights)
        mma.update_device(x, df, g, dg, case["movlim"])
    df, g, dg = _mma_problem(case, x, targets, weights)
    return dict(case=case, mma=mma, x=x, new=torch.empty_like(x), dfdx=df, g=g, dgdx=dg)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "forward":
        s = state["solver"]
        s.set_design_device(state["gamma"])
        s.init_equilibrium(**state["start"])
        J = s.forward(case["steps"])
        return dict(J=J, macros=s.get_macros())
    if kind == "gradient":
        s, gamma = state["solver"], state["gamma"]
        if case["autograd"] and not state["start"]:
            gamma.grad = None
            J = lbmx_torch.objective(gamma, s, case["steps"])
            J.backward()
            return dict(J=J.detach(), dJ=gamma.grad)
        s.set_design_device(gamma.detach())
        J, _ = s.gradient(case["steps"], want_sens=False, **state["start"])
        return dict(J=float(J), dJ=s.sensitivity_device().clone())  # the view itself ends with the solver
    if kind == "ensemble":
        for s, g in zip(state["members"], state["designs"]):
            s.set_design_device(g)
        J, _ = state["batch"].gradient(case["steps"], want_sens=False)
        return dict(J=J, dJ=[s.sensitivity_device().clone() for s in state["members"]])
    if kind == "filter":
        f = state["filter"]
        return dict(physical=f.design_device(state["design"]), sens=f.sensitivities_device(state["sens"]))
    x = state["new"].copy_(state["x"])
    state["mma"].update_device(x, state["dfdx"], state["g"], state["dgdx"], case["movlim"])
    return dict(x=x, change=state["mma"].design_change_device())


# ---- what a pass cannot do without --------------------------------------------------------------

_STATE_BYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}
_ADJOINT_BYTES = {"f64": 8, "f32": 4, "f16": 4, "bf16": 4}
_FLOPS = {9: (250, 500), 14: (400, 800), 19: (600, 1200)}  # per node: forward step, reverse step


def _sweep_work(Q, precision, nodes, steps, gradient):
    sf, sl = _STATE_BYTES[precision], _ADJOINT_BYTES[precision]
    sg = 8 if precision == "f64" else 4
    b, f = 2 * Q * sf + sg, _FLOPS[Q][0]
    if gradient:
        b, f = b + Q * sf + 2 * Q * sl + sg + 16, f + _FLOPS[Q][1]
    return {"bytes": float(b) * nodes * steps, "flops": float(f) * nodes * steps}


def _taps(R, dim):
    r = range(-R, R + 1)
    return sum(1 for z in (r if dim == 3 else (0,)) for y in r for x in r if x * x + y * y + z * z <= R * R)


def work(case):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        N = case["nx"] * case["ny"] * case["nz"]
        return _sweep_work(Q_OF[case["problem"]], case["precision"], N, case["steps"], kind == "gradient")
    if kind == "ensemble":
        N = 3 * sum(nx * ny for nx, ny in _ensemble_grids(case))
        return _sweep_work(9, case["precision"], N, case["steps"], True)
    if kind == "filter":
        N, dim = case["nx"] * case["ny"] * case["nz"], 2 if case["nz"] == 1 else 3
        taps = sum(_taps(R, dim) for R, _, _, _ in _filter_stages(case))
        return {"bytes": 32.0 * N, "flops": 4.0 * taps * N}
    n, m = case["n"], case["m"]
    return {"bytes": 8.0 * n * (m + 8), "flops": float(n) * 18 * (40 + 12 * m + 2 * m * m)}


# ---- the same outputs from plain torch in 64 bits -----------------------------------------------

# velocities, opposites and weights of the lattices, in the framework's order
_C9 = np.array([(0, 0), (1, -1), (0, -1), (-1, -1), (-1, 0), (-1, 1), (0, 1), (1, 1), (1, 0)])
_W9 = [4 / 9] + [1 / 36, 1 / 9] * 4
_C19 = np.array([(0, 0, 0), (0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, -1, -1), (0, 1, -1), (-1, 0, -1), (1, 0, -1),
                 (-1, -1, 0), (1, -1, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0), (0, 1, 1), (0, -1, 1), (1, 0, 1),
                 (-1, 0, 1), (1, 1, 0), (-1, 1, 0)])
_W19 = [1 / 3] + ([1 / 18] * 3 + [1 / 36] * 6) * 2
_C5 = np.array([(0, 0), (0, -1), (-1, 0), (0, 1), (1, 0)])


def _opposites(c):
    return [next(i for i in range(len(c)) if (c[i] == -c[q]).all()) for q in range(len(c))]


def _moments(dim):
    """Moment rows, their relaxation (0: conserved, None: omega, a rate) and their equilibrium (a, b, C)."""
    z = np.zeros
    if dim == 2:
        x, y = _C9[:, 0].astype(float), _C9[:, 1].astype(float)
        e = x * x + y * y
        M = np.stack([x * 0 + 1, x, y, -4 + 3 * e, 4 - 10.5 * e + 4.5 * e * e, (-5 + 3 * e) * x, (-5 + 3 * e) * y,
                      x * x - y * y, x * y])
        rate = [0, 0, 0, 1.4, 1.4, 1.2, 1.2, None, None]
        a, b, C = z(9), z((9, 2)), z((9, 2, 2))
        a[0], b[1, 0], b[2, 1] = 1, 1, 1
        a[3], a[4] = -2, 1
        C[3], C[4] = 3 * np.eye(2), -3 * np.eye(2)
        b[5, 0] = b[6, 1] = -1
        C[7] = np.diag([1, -1])
        C[8] = [[0, 0.5], [0.5, 0]]
        return M, rate, a, b, C
    x, y, w = (_C19[:, k].astype(float) for k in range(3))
    e = x * x + y * y + w * w
    M = np.stack([x * 0 + 1, x, y, w, 19 * e - 30, (21 * e * e - 53 * e + 24) / 2, (5 * e - 9) * x, (5 * e - 9) * y,
                  (5 * e - 9) * w, 3 * x * x - e, (3 * e - 5) * (3 * x * x - e), y * y - w * w,
                  (3 * e - 5) * (y * y - w * w), x * y, y * w, x * w, (y * y - w * w) * x, (w * w - x * x) * y,
                  (x * x - y * y) * w])
    rate = [0, 0, 0, 0, 1.19, 1.4, 1.2, 1.2, 1.2, None, 1.4, None, 1.4, None, None, None, 1.4, 1.4, 1.4]
    a, b, C = z(19), z((19, 3)), z((19, 3, 3))
    a[0] = 1
    for k in range(3):
        b[1 + k, k], b[6 + k, k] = 1, -2 / 3
    a[4], a[5] = -11, 3
    C[4], C[5] = 19 * np.eye(3), -5.5 * np.eye(3)
    C[9], C[11] = np.diag([2.0, -1, -1]), np.diag([0.0, 1, -1])
    C[10], C[12] = -0.5 * C[9], -0.5 * C[11]
    for k, (i, j) in {13: (0, 1), 14: (1, 2), 15: (0, 2)}.items():
        C[k, i, j] = C[k, j, i] = 0.5
    return M, rate, a, b, C


class _Lattice:
    """One lattice Boltzmann problem on dense tensors f[q, z, y, x]."""

    def __init__(self, case, gamma):
        self.problem, self.collision = case["problem"], case["collision"]
        self.nx, self.ny, self.nz, self.steps = case["nx"], case["ny"], case["nz"], case["steps"]
        self.dim = 3 if self.problem == "duct" else 2
        self.c, self.w = (_C19, _W19) if self.dim == 3 else (_C9, _W9)
        self.opp = _opposites(self.c)
        self.omega = case.get("omega", OMEGA.get(self.problem))
        self.gamma = gamma.reshape(self.nz, self.ny, self.nx)
        self.dev = gamma.device
        self.thermal = self.problem == "thermal"
        self.T = lambda v: torch.as_tensor(v, dtype=torch.float64, device=self.dev)
        self.time_const = 1.0 / self.steps
        self.pbb = self.collision == "cascaded" or self.collision.startswith("pbb_")
        self.collision = self.collision.replace("pbb_", "")
        if self.collision == "mrt":
            M, rate, a, b, C = _moments(self.dim)
            n2 = (M * M).sum(1)
            s = np.array([self.omega if r is None else r for r in rate], dtype=float)
            self.M, self.back = self.T(M), self.T((M / n2[:, None]).T.copy())
            self.s, self.a, self.b, self.C = self.T(s), self.T(a), self.T(b), C
            self.half = self.T(1 - s / 2)
        self.ct = self.T(self.c.astype(float))  # [Q, dim]
        self.wt = self.T(self.w)
        self.walls = self._wall_pieces()

    # -- collision
    def drag(self, gamma):
        q = 0.1
        return 0.1 * (1 - gamma * (1 + q) / (q + gamma))

    def collide(self, f, gamma):
        flow = f[:len(self.c)]
        shape = flow.shape
        p = flow.reshape(shape[0], -1)
        g = gamma.reshape(-1)
        rho = p.sum(0)
        j = self.ct.t() @ p
        if self.collision == "cascaded":
            out = self._cascaded(p, rho, j)
        else:
            alpha = 0.0 * g if self.pbb else self.drag(g)
            v = j / (1 + 0.5 * alpha)
            u2 = (v * v).sum(0)
            cu = self.ct @ v
            if self.collision == "bgk":
                eq = self.wt[:, None] * (rho + 3 * cu + 4.5 * cu * cu - 1.5 * u2)
                src = self.wt[:, None] * (3 * cu + 9 * cu * cu - 3 * u2)
                out = (1 - self.omega) * p + self.omega * eq - (1 - 0.5 * self.omega) * alpha * src
            else:
                src = self.wt[:, None] * (3 * cu + 9 * cu * cu - 3 * u2)
                rows = []
                for k in range(len(self.w)):
                    r = self.a[k] * rho + (self.b[k][:, None] * v).sum(0)
                    for i, l in zip(*np.nonzero(self.C[k])):
                        r = r + self.C[k][i, l] * v[i] * v[l]
                    rows.append(r)
                dm = self.s[:, None] * (self.M @ p - torch.stack(rows))
                dm = dm + self.half[:, None] * alpha * (self.M @ src)
                out = p - self.back @ dm
        if self.pbb:  # partial bounce-back: the odd part of each opposite pair scaled by 1 - BP(gamma)
            back = out[self.opp]
            out = 0.5 * (out + back) + 0.5 * (out - back) * (1.1 * g / (0.1 + g))
        out = out.reshape(shape)
        if not self.thermal:
            return out
        t = f[9:]
        T = t.sum(0)
        ramp = (gamma * (0.1 * 2.0 - 1.0) + 1.0) / (0.1 * (1.0 + gamma))
        om = 1.0 / (5.0 * 0.02 * ramp + 0.5)
        jx, jy = j[0].reshape(shape[1:]), j[1].reshape(shape[1:])
        q1, q2 = t[4] - t[2], t[3] - t[1]
        e = t[1] + t[2] + t[3] + t[4] - 4 * t[0]
        pxx = t[2] + t[4] - t[1] - t[3]
        d1, d2 = om * (q1 - jx * T) / 2, om * (q2 - jy * T) / 2
        d3, d4 = 1.5 * (e + 2 * T) / 20, 1.5 * pxx / 4
        new = [t[0] + 4 * d3, t[1] + d2 - d3 + d4, t[2] + d1 - d3 - d4, t[3] - d2 - d3 + d4, t[4] - d1 - d3 - d4]
        return torch.cat([out, torch.stack(new)])

    def _cascaded(self, f, r, j):
        x, y, om = j[0], j[1], self.omega
        u2 = x * x + y * y
        k0 = (r * u2 - f[8] - f[6] - f[2] - f[4] - 2 * (f[1] + f[3] + f[7] + f[5] - r / 3)) / 12
        k1 = om * (f[6] + f[2] - f[8] - f[4] + r * (x * x - y * y)) / 4
        k2 = om * (f[7] + f[3] - f[5] - f[1] - r * x * y) / 4
        k3 = (-((f[1] + f[3] - f[7] - f[5] - 2 * r * x * x * y + y * (r - f[6] - f[2] - f[0])) / 4
                + 0.5 * x * (f[7] - f[5] - f[1] + f[3])) + 0.5 * y * (-3 * k0 - k1) + 2 * x * k2)
        k4 = (-((f[3] + f[5] - f[1] - f[7] - 2 * r * y * y * x + x * (r - f[4] - f[8] - f[0])) / 4
                + 0.5 * y * (f[7] + f[3] - f[1] - f[5])) + 0.5 * x * (-3 * k0 + k1) + 2 * y * k2)
        k5 = (0.25 * (r / 9 - f[7] - f[5] - f[1] - f[3]
                      + 2 * (x * (f[7] - f[5] + f[1] - f[3]) + y * (f[7] + f[5] - f[1] - f[3]))
                      + 4 * x * y * (f[5] - f[7] + f[1] - f[3])
                      - x * x * (f[6] + f[7] + f[5] + f[2] + f[1] + f[3])
                      + y * y * (3 * r * x * x - f[8] - f[7] - f[5] - f[1] - f[3] - f[4]))
              - 2 * k0 - 2 * x * k4 - 2 * y * k3 + 4 * x * y * k2 - 1.5 * k0 * u2 + 0.5 * k1 * (x * x - y * y))
        T = [(-4, 0, 0, 0, 0, 4), (2, 0, 1, 1, -1, 1), (-1, -1, 0, -2, 0, -2), (2, 0, -1, 1, 1, 1),
             (-1, 1, 0, 0, -2, -2), (2, 0, 1, -1, 1, 1), (-1, -1, 0, 2, 0, -2), (2, 0, -1, -1, -1, 1),
             (-1, 1, 0, 0, 2, -2)]
        return f + self.T(np.array(T, dtype=float)) @ torch.stack([k0, k1, k2, k3, k4, k5])

    # -- streaming with mid-way reflection at the domain edges
    def stream(self, p):
        out = []
        dims = (self.nx, self.ny, self.nz)
        for q in range(p.shape[0]):
            c = self.c[q] if q < len(self.c) else _C5[q - 9]
            o = self.opp[q] if q < len(self.c) else 9 + [0, 3, 4, 1, 2][q - 9]
            c = list(c) + [0] * (3 - len(c))
            if not any(c):
                out.append(p[q])
                continue
            s = torch.roll(p[q], shifts=(int(c[2]), int(c[1]), int(c[0])), dims=(0, 1, 2))
            for axis in range(3):
                if c[axis]:  # the source x - c lies outside on this face
                    at = [slice(None)] * 3
                    at[2 - axis] = slice(0, 1) if c[axis] > 0 else slice(dims[axis] - 1, dims[axis])
                    s[tuple(at)] = p[o][tuple(at)]
            out.append(s)
        return torch.stack(out)

    def _wall_pieces(self):
        """(slices, directions replaced by their opposite) of the on-grid bounce-back walls."""
        X, Y, Z = self.nx - 1, self.ny - 1, self.nz - 1
        pieces = []
        for iz in ((-1, 0, 1) if self.dim == 3 else (0,)):
            for iy in (-1, 0, 1):
                for ix in (-1, 0, 1):
                    if iy == 0 and iz == 0:
                        continue  # inside, inlet and outlet
                    at = tuple(slice(0, 1) if n < 0 else slice(m, m + 1) if n > 0 else (slice(1, m) if m else slice(0, 1))
                               for n, m in ((iz, Z), (iy, Y), (ix, X)))
                    n = np.array([ix, iy, iz][:self.dim])
                    turned = [q for q in range(1, len(self.c)) if self.c[q] @ n <= 0]
                    if self.dim == 3 and (ix, iy, iz) == (-1, -1, -1):
                        turned = [q for q in turned if q not in (9, 13)]
                    pieces.append((at, turned))
        return pieces

    def boundaries(self, f, t):
        for at, turned in self.walls:
            old = [f[(self.opp[q],) + at] for q in turned]
            new = torch.stack(old).clone()
            for k, q in enumerate(turned):
                f[(q,) + at] = new[k]
        Y, Z = self.ny - 1, self.nz - 1
        ins = (slice(1, Z) if self.dim == 3 else slice(0, 1), slice(1, Y))
        west, east = ins + (slice(0, 1),), ins + (slice(self.nx - 1, self.nx),)
        if self.dim == 2:
            mid = (self.ny - 1) / 2.0
            tf = 1.0 + 0.5 * math.sin(2 * math.pi * t / 1000.0) if self.problem == "pump" else 1.0
            yy = torch.arange(1, Y, device=self.dev, dtype=torch.float64)[None, :, None]
            ux = 0.05 * (mid * mid - (yy - mid) ** 2) / (mid * mid) * tf
            g = [f[(q,) + west].clone() for q in range(9)]
            f[(1,) + west] = 0.5 * (g[6] - g[2]) + g[5] + ux / 6
            f[(7,) + west] = 0.5 * (g[2] - g[6]) + g[3] + ux / 6
            f[(8,) + west] = g[4] + 2 / 3 * ux
            g = [f[(q,) + east].clone() for q in range(9)]
            u = g[0] + g[2] + g[6] + 2 * (g[1] + g[7] + g[8]) - 1.0
            f[(4,) + east] = g[8] - 2 / 3 * u
            f[(3,) + east] = g[7] - u / 6 + 0.5 * (g[6] - g[2])
            f[(5,) + east] = g[1] - u / 6 + 0.5 * (g[2] - g[6])
        else:
            ux = 0.04
            g = [f[(q,) + west].clone() for q in range(19)]
            ny_ = 0.5 * (g[5] + g[11] + g[13] - g[2] - g[4] - g[14])
            nz_ = 0.5 * (g[10] + g[13] + g[14] - g[1] - g[4] - g[5])
            for q, v in ((7, g[16] + ux / 6 + nz_), (9, g[18] + ux / 6 + ny_), (12, g[3] + ux / 3),
                         (15, g[6] + ux / 6 - nz_), (17, g[8] + ux / 6 - ny_)):
                f[(q,) + west] = v
            g = [f[(q,) + east].clone() for q in range(19)]
            u = (g[0] + g[1] + g[2] + g[4] + g[5] + g[10] + g[11] + g[13] + g[14]
                 + 2 * (g[7] + g[9] + g[12] + g[15] + g[17])) - 1.0
            ny_ = 0.5 * (g[5] + g[11] + g[13] - g[2] - g[4] - g[14])
            nz_ = 0.5 * (g[10] + g[13] + g[14] - g[1] - g[4] - g[5])
            for q, v in ((3, g[12] - u / 3), (6, g[15] - u / 6 + nz_), (8, g[17] - u / 6 + ny_),
                         (16, g[7] - u / 6 - nz_), (18, g[9] - u / 6 - ny_)):
                f[(q,) + east] = v
        if self.thermal:
            across = (slice(0, 1), slice(None), slice(1, self.nx - 1))
            south, north = across[:1] + (slice(0, 1),) + across[2:], across[:1] + (slice(Y, Y + 1),) + across[2:]
            for at, q, T in ((south, 3, 0.0), (north, 1, 0.0), (west, 4, 1.0)):
                g = [f[(9 + k,) + at].clone() for k in range(5)]
                f[(9 + q,) + at] = T - (g[0] + g[1] + g[2] + g[3] + g[4] - g[q])
            f[(11,) + east] = f[(13,) + east].clone()
        return f

    # -- functional
    def objective(self, f):
        Y, Z = self.ny - 1, self.nz - 1
        ins = (slice(None), slice(1, Z) if self.dim == 3 else slice(0, 1), slice(1, Y))
        a, b = f[ins + (0,)], f[ins + (self.nx - 1,)]
        Q = len(self.c)
        if self.problem in ("channel", "duct"):
            return self.time_const * (a[:Q].sum(0).mean() - b[:Q].sum(0).mean())
        if self.problem == "thermal":
            jx = (self.ct[:, 0][:, None, None] * b[:Q]).sum(0)
            return -self.time_const * (jx * b[Q:].sum(0)).sum()

        def power(g):
            rho = g.sum(0)
            jx, jy = ((self.ct[:, k][:, None, None] * g).sum(0) for k in (0, 1))
            return ((rho / 3 + 0.5 * (jx * jx + jy * jy)) * jx).sum()

        return self.time_const * (power(a) - power(b))

    def start(self):
        """s_0: the equilibrium of the initial macros."""
        ux, T0 = (0.03, 0.5) if self.thermal else (0.0, 0.0)
        cu = self.c[:, 0] * ux
        f = np.array(self.w) * (1.0 + 3 * cu + 4.5 * cu ** 2 - 1.5 * ux * ux)
        if self.thermal:
            q1, e = ux * T0, -2 * T0
            f = np.concatenate([f, [T0 / 5 - 4 * e / 20, T0 / 5 + e / 20, T0 / 5 - q1 / 2 + e / 20, T0 / 5 + e / 20,
                                    T0 / 5 + q1 / 2 + e / 20]])
        return self.T(f)[:, None, None, None].expand(-1, self.nz, self.ny, self.nx).contiguous()

    def state(self, p, t):
        return self.boundaries(self.stream(p), t)

    def forward(self):
        """J and the macros of the last state."""
        with torch.no_grad():
            p, J = self.collide(self.start(), self.gamma), 0.0
            for t in range(1, self.steps + 1):
                f = self.state(p, t)
                J = J + self.objective(f)
                if t < self.steps:
                    p = self.collide(f, self.gamma)
            Q = len(self.c)
            m = torch.zeros((self.nz * self.ny * self.nx, 5), dtype=torch.float64, device=self.dev)
            flow = f[:Q].reshape(Q, -1)
            m[:, 0] = flow.sum(0)
            m[:, 1:1 + self.dim] = (self.ct.t() @ flow).t()
            if self.thermal:
                m[:, 4] = f[Q:].sum(0).reshape(-1)
        return J, m

    def gradient(self):
        """J and dJ/dgamma, step by step backwards over the stored states."""
        with torch.no_grad():
            stored = [self.collide(self.start(), self.gamma)]
            for t in range(1, self.steps):
                stored.append(self.collide(self.state(stored[-1], t), self.gamma))
        J, dJ, lam = 0.0, torch.zeros_like(self.gamma), None
        for t in range(self.steps, 0, -1):
            p = stored.pop().requires_grad_(True)
            g = self.gamma.detach().clone().requires_grad_(True)
            with torch.enable_grad():
                f = self.state(p, t)
                Jt = self.objective(f)
                total = Jt if lam is None else Jt + (self.collide(f, g) * lam).sum()
                gp, gg = torch.autograd.grad(total, (p, g), allow_unused=True)
            J = J + Jt.detach()
            lam = gp
            if gg is not None:
                dJ += gg
        # p_0 = collide(s_0, gamma) is the initial state and not part of the reverse loop
        return J, dJ.reshape(-1)


def _cone(x, R, dim):
    """Sum of (R - |d|) x(. + d) over the offsets within R, zero outside the grid."""
    pz = R if dim == 3 else 0
    xp = F.pad(x, (R, R, R, R, pz, pz))
    nz, ny, nx = x.shape
    acc = torch.zeros_like(x)
    for dz in range(-pz, pz + 1):
        for dy in range(-R, R + 1):
            for dx in range(-R, R + 1):
                w = R - math.sqrt(dx * dx + dy * dy + dz * dz)
                if w > 0:
                    acc += w * xp[pz + dz:pz + dz + nz, R + dy:R + dy + ny, R + dx:R + dx + nx]
    return acc


def _exact_filter(case, seed):
    box, design, sens = _filter_inputs(case, seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    dim = 2 if nz == 1 else 3
    at = (slice(box[4], box[5] + 1), slice(box[2], box[3] + 1), slice(box[0], box[1] + 1))
    x = torch.ones((nz, ny, nx), dtype=torch.float64, device="cuda")
    x[at] = design.reshape(x[at].shape)
    inside = torch.zeros_like(x, dtype=torch.bool)
    inside[at] = True
    one = torch.ones_like(x)
    kept = []
    for R, _, beta, eta in _filter_stages(case):
        den = torch.where(inside, _cone(one, R, dim), one)
        x = torch.where(inside, _cone(x, R, dim) / den, x)
        kept.append((R, beta, eta, den, x))
        top = math.tanh(beta * eta) + math.tanh(beta * (1 - eta))
        x = torch.where(inside, (math.tanh(beta * eta) + torch.tanh(beta * (x - eta))) / top, x)
    s = sens.reshape(nz, ny, nx)
    for R, beta, eta, den, dens in reversed(kept):
        top = math.tanh(beta * eta) + math.tanh(beta * (1 - eta))
        s = torch.where(inside, s * beta * (1 - torch.tanh(beta * (dens - eta)) ** 2) / top, s) / den
        s = _cone(torch.where(inside, s, torch.zeros_like(s)), R, dim) + torch.where(inside, torch.zeros_like(s), s)
    return dict(physical=x.reshape(-1), sens=s[at].reshape(-1))


class _MMA:
    """Svanberg's subproblem around the design and its dual interior-point solution."""

    def __init__(self, n, a):
        self.n, self.m, self.a, self.k = n, len(a), np.array(a), 0

    def update(self, x, df, gx, dg, movlim):
        self.k += 1
        up, lo = (x + movlim).clamp(max=1.0), (x - movlim).clamp(min=0.0)
        if self.k < 3:
            L, U = x - 0.5 * (up - lo), x + 0.5 * (up - lo)
        else:
            trend = (x - self.x1) * (self.x1 - self.x2)
            g = 1.0 - 0.3 * (trend < 0).double() + 0.2 * (trend > 0).double()
            span = (up - lo).clamp(min=1e-5)
            L = torch.minimum(torch.maximum(x - g * (self.x1 - self.L), x - 10 * span), x - 0.01 * span)
            U = torch.minimum(torch.maximum(x + g * (self.U - self.x1), x + 0.01 * span), x + 10 * span)
        self.L, self.U = L, U
        alpha, beta = torch.maximum(lo, 0.9 * L + 0.1 * x), torch.minimum(up, 0.9 * U + 0.1 * x)
        ux, xl = U - x, x - L
        extra = 0.001 * df.abs() + 0.5e-6 / (U - L)
        p0, q0 = ux * ux * (df.clamp(min=0) + extra), xl * xl * ((-df).clamp(min=0) + extra)
        G = torch.stack(list(dg))
        P, Q = ux * ux * G.clamp(min=0), xl * xl * (-G).clamp(min=0)
        b = (P / ux + Q / xl).sum(1).cpu().numpy() - np.array(gx)
        self.x2, self.x1 = getattr(self, "x1", None), x
        m, a, c = self.m, self.a, np.full(self.m, 1000.0)
        lam, mu = c / 2, np.ones(m)
        tol, epsi, err = 1e-9 * math.sqrt(m + self.n), 1.0, 1.0

        def primal():
            np.maximum(lam, 0.0, out=lam)
            return np.maximum(0.0, lam - c), max(0.0, 10.0 * (lam @ a - 1.0))

        def point():
            l = torch.as_tensor(lam, dtype=x.dtype, device=x.device)
            pl, ql = p0 + l @ P, q0 + l @ Q
            sp, sq = pl.sqrt(), ql.sqrt()
            free = (sp * L + sq * U) / (sp + sq)
            new = torch.minimum(torch.maximum(free, alpha), beta)
            return new, free, pl, ql, (P / (U - new) + Q / (new - L)).sum(1).cpu().numpy()

        while epsi > tol:
            loop = 0
            while err > 0.9 * epsi and loop < 100:
                loop += 1
                y, z = primal()
                new, free, pl, ql, sums = point()
                d2 = -1.0 / (2 * pl / (U - new) ** 3 + 2 * ql / (new - L) ** 3)
                d2 = torch.where((free < alpha) | (free > beta), torch.zeros_like(d2), d2)
                PQ = P / (U - new) ** 2 - Q / (new - L) ** 2
                H = ((PQ * d2) @ PQ.t()).cpu().numpy().copy()
                grad = -(sums - b - a * z - y) - epsi / lam
                H[np.diag_indices(m)] += np.where(lam > c, -1.0, 0.0) - mu / lam
                if lam @ a > 0:
                    H -= 10.0 * np.outer(a, a)
                corr = 1e-4 * np.trace(H) / m
                H[np.diag_indices(m)] += -1e-7 if -corr < 1e-7 else corr
                s = np.linalg.solve(H, grad)
                sm = -mu + epsi / lam - s * mu / lam
                theta = 1.0 / max(1.005, (-1.01 * s / lam).max(), (-1.01 * sm / mu).max())
                lam += theta * s
                mu += theta * sm
                y, z = primal()
                new, _, _, _, sums = point()
                err = max(np.abs(sums - b - a * z - y + mu).max(), np.abs(mu * lam - epsi).max())
            epsi *= 0.1
        return new


def _exact_mma(case, seed):
    targets, weights = _mma_inputs(case, seed)
    o = _MMA(case["n"], _mma_constants(case))
    x = torch.full((case["n"],), 0.5, device="cuda", dtype=torch.float64)
    for _ in range(4):
        old = x
        df, g, dg = _mma_problem(case, x, targets, weights)
        x = o.update(x, df, g, dg, case["movlim"])
    return dict(x=x, change=float((x - old).abs().max()))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        lat = _Lattice(case, _design(case["nx"], case["ny"], case["nz"], _generator(seed)))
        if kind == "forward":
            J, m = lat.forward()
            return dict(J=float(J), macros=m.cpu().numpy())
        J, dJ = lat.gradient()
        return dict(J=J if case["autograd"] and case["problem"] != "thermal" else float(J), dJ=dJ)
    if kind == "ensemble":
        Js, dJs = [], []
        for nx, ny, g in _ensemble_inputs(case, seed):
            lat = _Lattice(dict(problem="channel", collision="pbb_" + case["collision"], omega=1.0 / 0.6, nx=nx, ny=ny,
                                nz=1, steps=case["steps"]), g)
            J, dJ = lat.gradient()
            Js.append(float(J))
            dJs.append(dJ)
        return dict(J=np.array(Js), dJ=dJs)
    if kind == "filter":
        return _exact_filter(case, seed)
    return _exact_mma(case, seed)
