"""More forms and tile shapes of the sweeps that take several steps per launch, against one step
per launch (see test_gpu_steps): fields of one round of workgroups with tiles of many rows, a
field of several rounds, and every operator and storage form those sweeps are built for."""
import numpy as np
import pytest

import lbmx
import test_gpu_steps as steps_test

pytestmark = pytest.mark.gpu

MORE = [
    ("mrt none fp64", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_NONE, lbmx.FP64),
    ("mrt none fp32", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_NONE, lbmx.FP32),
    ("mrt brinkman fp32", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_BRINKMAN, lbmx.FP32),
    ("mrt brinkman fp16", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_BRINKMAN, lbmx.FP16_SHIFTED),
    ("mrt pbb fp64", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_PBB, lbmx.FP64),
    ("mrt pbb fp32", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_PBB, lbmx.FP32),
    ("bgk none fp64", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_NONE, lbmx.FP64),
    ("bgk none fp32", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_NONE, lbmx.FP32),
    ("bgk brinkman fp64", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_BRINKMAN, lbmx.FP64),
    ("bgk brinkman bf16", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_BRINKMAN, lbmx.BF16_SHIFTED),
    ("bgk pbb fp32", lbmx.D2Q9, lbmx.BGK, lbmx.DESIGN_PBB, lbmx.FP32),
    ("cascaded pbb fp64", lbmx.D2Q9, lbmx.CASCADED, lbmx.DESIGN_PBB, lbmx.FP64),
    ("cascaded none fp32", lbmx.D2Q9, lbmx.CASCADED, lbmx.DESIGN_NONE, lbmx.FP32),
    ("cascaded pbb fp16", lbmx.D2Q9, lbmx.CASCADED, lbmx.DESIGN_PBB, lbmx.FP16_SHIFTED),
    ("cascaded none bf16", lbmx.D2Q9, lbmx.CASCADED, lbmx.DESIGN_NONE, lbmx.BF16_SHIFTED),
    ("thermal mrt brinkman fp64", lbmx.D2Q9_D2Q5, lbmx.MRT, lbmx.DESIGN_BRINKMAN, lbmx.FP64),
    ("thermal mrt brinkman fp32", lbmx.D2Q9_D2Q5, lbmx.MRT, lbmx.DESIGN_BRINKMAN, lbmx.FP32),
    ("thermal bgk pbb fp32", lbmx.D2Q9_D2Q5, lbmx.BGK, lbmx.DESIGN_PBB, lbmx.FP32),
    ("thermal bgk none fp64", lbmx.D2Q9_D2Q5, lbmx.BGK, lbmx.DESIGN_NONE, lbmx.FP64),
    ("thermal mrt none fp16", lbmx.D2Q9_D2Q5, lbmx.MRT, lbmx.DESIGN_NONE, lbmx.FP16_SHIFTED),
    ("thermal mrt pbb bf16", lbmx.D2Q9_D2Q5, lbmx.MRT, lbmx.DESIGN_PBB, lbmx.BF16_SHIFTED),
]
FORWARD_ONLY = [
    ("standard bgk fp64", lbmx.D2Q9, lbmx.BGK_STANDARD, lbmx.DESIGN_NONE, lbmx.FP64),
    ("standard bgk pbb fp32", lbmx.D2Q9, lbmx.BGK_STANDARD, lbmx.DESIGN_PBB, lbmx.FP32),
    ("standard bgk fp16", lbmx.D2Q9, lbmx.BGK_STANDARD, lbmx.DESIGN_NONE, lbmx.FP16_SHIFTED),
    ("darcy mrt fp64", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_DARCY, lbmx.FP64),
    ("darcy mrt bf16", lbmx.D2Q9, lbmx.MRT, lbmx.DESIGN_DARCY, lbmx.BF16_SHIFTED),
]
# one round of tiles of 2, some 6 and some 8 rows; several rounds, with rows left over
SIZES = [(65, 17, 7), (640, 131, 6), (512, 256, 5), (900, 301, 7)]


@pytest.mark.parametrize("nx,ny,steps", SIZES)
@pytest.mark.parametrize("form", MORE, ids=[f[0] for f in MORE])
def test_more_forms(lbmx_mod, form, nx, ny, steps):
    steps_test.test_steps_equal_single_sweeps(lbmx_mod, form, nx, ny, steps)


@pytest.mark.parametrize("nx,ny,steps", SIZES[1:])
@pytest.mark.parametrize("form", steps_test.FORMS, ids=[f[0] for f in steps_test.FORMS])
def test_more_shapes(lbmx_mod, form, nx, ny, steps):
    steps_test.test_steps_equal_single_sweeps(lbmx_mod, form, nx, ny, steps)


@pytest.mark.parametrize("nx,ny,steps", SIZES)
@pytest.mark.parametrize("form", FORWARD_ONLY, ids=[f[0] for f in FORWARD_ONLY])
def test_forward_only_forms(lbmx_mod, form, nx, ny, steps):
    s, kw = steps_test._solver(form, nx, ny, steps), steps_test._start(form)
    s.init_equilibrium(**kw)
    Js = [s.forward(1) for _ in range(steps)]
    one = s.get_state()
    s.init_equilibrium(**kw)
    J = s.forward(steps)
    assert np.array_equal(s.get_state(), one)
    assert abs(J - sum(Js)) <= 1e3 * 2.3e-16 * 2 * ny
    s.close()


EVERY = steps_test.FORMS + MORE + FORWARD_ONLY


@pytest.mark.parametrize("form", EVERY, ids=[f[0] for f in EVERY])
def test_small_fields_take_several_steps(form):
    """These tests would compare a sweep with itself if the rule fell back to one step per launch."""
    s = steps_test._solver(form, 65, 17, 7)
    fwd, rev = s.steps_per_launch()
    cascaded = form[2] == lbmx.CASCADED
    assert fwd == 4 and (rev == 1 if cascaded else rev > 1)
    s.close()
