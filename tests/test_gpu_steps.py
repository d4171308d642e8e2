"""Several steps of a 2D sweep in one launch, against the sweeps of one step per launch.

forward(n) and gradient(n) take tiles of the field through several steps per launch; forward(1)
and the stepwise reverse loop (adjoint_step) run one. Both do the same arithmetic on the same
stored values, so states, adjoint populations and sensitivities are the same bits. The sizes sit
at the edges of the tiles (64 columns; rows chosen by how many tiles there are): less than one
tile, exact multiples, one more, and a field of several hundred tiles, which takes the largest
ones. The step counts leave remainders of every group length; two slots more than half of the
steps make the reverse pass recompute and keep states inside a group.
"""
import numpy as np
import pytest

import lbmx
import workloads

pytestmark = pytest.mark.gpu

FORMS = [
    ("mrt brinkman fp64", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_BRINKMAN, lbmx.FP64),
    ("bgk brinkman fp32", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_BRINKMAN, lbmx.FP32),
    ("bgk pbb fp64", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_PBB, lbmx.FP64),
    ("bgk none fp16", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_NONE, lbmx.FP16_SHIFTED),
    ("mrt pbb bf16", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_PBB, lbmx.BF16_SHIFTED),
    ("cascaded pbb fp32", lbmx.D2Q9, lbmx.CASCADED, lbmx.DESIGN_PBB, lbmx.FP32),
    ("thermal mrt pbb fp64", lbmx.D2Q9_D2Q5, lbmx.MRT, lbmx.DESIGN_PBB, lbmx.FP64),
    ("thermal bgk brinkman fp64", lbmx.D2Q9_D2Q5, lbmx.BGK, lbmx.DESIGN_BRINKMAN, lbmx.FP64),
    ("thermal bgk brinkman fp16", lbmx.D2Q9_D2Q5, lbmx.BGK, lbmx.DESIGN_BRINKMAN, lbmx.FP16_SHIFTED),
]
SIZES = [(12, 6, 9), (64, 16, 5), (65, 17, 7), (200, 33, 6), (1283, 205, 7)]


def _solver(form, nx, ny, steps):
    _, lat, coll, des, prec = form
    s = lbmx.Solver(lbmx.make_desc(nx, ny, lattice=lat, collision=coll, design=des, precision=prec, omega=1.3,
                                   interp_q=0.1, alpha_max=1.0 if des == lbmx.DESIGN_PBB else 0.1,
                                   thermal_diffusivity=0.02, ramp_p=1.0, ramp_ck=0.1))
    if lat == lbmx.D2Q9_D2Q5:
        workloads.thermal_channel2d(s, nx, ny, time_const=1.0 / steps)
    else:
        workloads.channel2d(s, nx, ny, time_const=1.0 / steps, modulation=(5.0, 0.3))
    s.set_design(workloads.design_field(nx, ny, 1, seed=nx))
    return s


def _start(form):
    return dict(u0=(0.03, 0.0, 0.0), T0=0.5) if form[1] == lbmx.D2Q9_D2Q5 else dict(u0=(0.02, 0.0, 0.0))


@pytest.mark.parametrize("nx,ny,steps", SIZES)
@pytest.mark.parametrize("form", FORMS, ids=[f[0] for f in FORMS])
def test_steps_equal_single_sweeps(lbmx_mod, form, nx, ny, steps):
    s, kw = _solver(form, nx, ny, steps), _start(form)
    s.init_equilibrium(**kw)
    states, Js = [s.get_state()], []
    for _ in range(steps):
        Js.append(s.forward(1))
        states.append(s.get_state())
    s.adjoint_reset(0)
    s.adjoint_set_timestep(steps)
    for t in range(steps, 0, -1):
        s.set_state(states[t], t)
        s.adjoint_step(with_source=True)
    g, lam = s.get_sensitivity(), s.get_adjoint()

    s.init_equilibrium(**kw)
    J = s.forward(steps)
    assert np.array_equal(s.get_state(), states[-1])
    # the same per-segment values, added in another order: some 1e3 additions in double of terms
    # whose magnitudes add to at most 2 per column node
    assert abs(J - sum(Js)) <= 1e3 * 2.3e-16 * 2 * ny
    for slots in (0, steps // 2 + 2):
        s.checkpoint_config(slots)
        Jg, gg = s.gradient(steps, **kw)
        assert Jg == J
        assert np.array_equal(gg, g), slots
        assert np.array_equal(s.get_adjoint(), lam), slots


@pytest.mark.parametrize("form", FORMS, ids=[f[0] for f in FORMS])
def test_batched_steps_equal_single_instances(lbmx_mod, form):
    steps, kw = 7, _start(form)
    members = [_solver(form, nx, ny, steps) for nx, ny in ((65, 17), (12, 6), (643, 205), (700, 190))]
    ref = []
    for m in members:
        m.checkpoint_config(5)
        ref.append(m.gradient(steps, **kw))
    for sizes in ((0, 1), (0, 1, 2, 3)):  # one tile per CU, and the tiles of large fields
        b = lbmx.Batch([members[i] for i in sizes])
        b.checkpoint_config(5)
        J, sens = b.gradient(steps, **kw)
        for k, i in enumerate(sizes):
            assert J[k] == ref[i][0]
            assert np.array_equal(sens[k], ref[i][1])
        b.close()
