"""Which launches a 2D batch runs: several steps per launch by itself, one step per launch once a
tile is set, and whichever the autotuner finds faster. Results do not depend on it."""
import numpy as np
import pytest

import lbmx
import workloads

pytestmark = pytest.mark.gpu

STEPS = 11


def members(coll, prec, grids=((64, 32), (130, 50), (70, 21))):
    out = []
    for i, (nx, ny) in enumerate(grids):
        s = lbmx.Solver(lbmx.make_desc(nx, ny, lattice=lbmx.D2Q9, collision=coll, design=lbmx.DESIGN_PBB,
                                       precision=prec, omega=1.3, interp_q=0.1, alpha_max=1.0))
        workloads.channel2d(s, nx, ny, time_const=1.0 / STEPS)
        s.set_design(workloads.design_field(nx, ny, 1, seed=i))
        out.append(s)
    return out


def run(b):
    b.checkpoint_config(4)
    return b.gradient(STEPS, u0=(0.02, 0.0, 0.0))


@pytest.mark.parametrize("coll,prec,default", [(lbmx.MRT, lbmx.FP64, (4, 4)), (lbmx.CASCADED, lbmx.FP32, (4, 1))])
def test_a_set_tile_runs(lbmx_mod, coll, prec, default):
    ms = members(coll, prec)
    b = lbmx.Batch(ms)
    assert b.steps_per_launch() == default
    J, g = run(b)
    several = b.device_bytes()
    b.close()
    for rows, paired in ((1, False), (2, True), (4, False), (4, True)):
        b = lbmx.Batch(ms)
        b.set_tile(rows, paired)
        assert b.tile() == (rows, paired) and b.steps_per_launch() == (1, 1)
        J1, g1 = run(b)
        assert list(J1) == list(J) and all(np.array_equal(x, y) for x, y in zip(g, g1))
        # the launches of several steps have a workgroup map of their own
        assert b.device_bytes() < several if rows == 4 else True
        b.close()


def test_autotune_weighs_launches_of_several_steps(lbmx_mod):
    """On a batch of a few small members a step of four per launch takes about half of a launch of
    its own, so the autotuner keeps those launches, also after a tile was set."""
    b = lbmx.Batch(members(lbmx.MRT, lbmx.FP64))
    J, g = run(b)
    b.set_tile(1, False)
    rows, ms = b.autotune(20)
    assert rows in (1, 2, 4) and all(0 < v < 1e3 for v in ms)
    assert b.steps_per_launch() == (4, 4) and b.tile()[0] == rows
    J1, g1 = run(b)
    assert list(J1) == list(J) and all(np.array_equal(x, y) for x, y in zip(g, g1))
    b.close()


def test_time_sweeps_times_the_launches_of_a_pass(lbmx_mod):
    """time_sweeps makes the launches that forward and gradient make: the device time of n sweeps
    is within a quarter of the pass's wall time (a launch per step takes 1.6 times it here), and
    the state it leaves is that of forward."""
    n, nx, ny = 600, 256, 128
    s = lbmx.Solver(lbmx.make_desc(nx, ny, lattice=lbmx.D2Q9, collision=lbmx.MRT, design=lbmx.DESIGN_BRINKMAN,
                                   precision=lbmx.FP64, omega=1.3, interp_q=0.1, alpha_max=0.1))
    workloads.channel2d(s, nx, ny, time_const=1.0 / n)
    s.set_design(workloads.design_field(nx, ny, 1, seed=3))
    assert min(s.steps_per_launch()) > 1
    s.init_equilibrium(u0=(0.02, 0.0, 0.0))
    s.forward(n)
    after = s.get_state()
    s.init_equilibrium(u0=(0.02, 0.0, 0.0))
    s.time_sweeps(0, n)
    assert s.timestep() == n and np.array_equal(s.get_state(), after)
    wall, timed = [], []
    for _ in range(3):
        s.init_equilibrium(u0=(0.02, 0.0, 0.0))
        s.forward(n)
        wall.append(s.stats()["forward_phase_ms"])
        timed.append(s.time_sweeps(0, n))
    assert min(timed) < 1.25 * min(wall)
    s.checkpoint_config(0)
    wall, timed = [], []
    for _ in range(3):
        s.gradient(n, u0=(0.02, 0.0, 0.0))
        wall.append(s.stats()["reverse_phase_ms"])
        s.init_equilibrium(u0=(0.02, 0.0, 0.0))
        s.forward(8)
        timed.append(s.time_sweeps(1, n))
    assert min(timed) < 1.25 * min(wall)
    s.close()
