"""Cone filter kernels with the radius known to the compiler (2D radii 1..12, 3D radii 1..3) at
the edges of their tiles: bit for bit against the oracle's row loop, forward and transposed,
with filter boxes that leave identity rows inside the tiles."""
import numpy as np
import pytest

import lbmx
import oracle

pytestmark = pytest.mark.gpu

B = lbmx.make_box

CASES = [((129, 9, 1), (2, 126, 1, 7, 0, 0), R) for R in range(1, 13)]
CASES += [((128, 8, 1), (0, 127, 0, 7, 0, 0), 4), ((1, 1, 1), (0, 0, 0, 0, 0, 0), 3),
          ((257, 17, 1), (130, 200, 3, 12, 0, 0), 8), ((64, 40, 1), (5, 60, 4, 33, 0, 0), 13)]
CASES += [((129, 17, 5), (1, 127, 2, 15, 1, 3), R) for R in (1, 2, 3, 4)]
CASES += [((128, 16, 4), (0, 127, 0, 15, 0, 3), 3), ((37, 5, 9), (30, 36, 0, 4, 2, 8), 2)]


def chain(dims, fbox, R, project=False):
    nx, ny, nz = dims
    full = (0, nx - 1, 0, ny - 1, 0, nz - 1)
    dev = lbmx.Filter(lbmx.make_filter_desc(*dims, B(*full), B(*fbox), ((R, project, 2.0, 0.5),)))
    return dev, oracle.FilterChain(*dims, full, fbox, stages=((R, project, 2.0, 0.5),))


@pytest.mark.parametrize("dims,fbox,R", CASES)
def test_cone_tiles_bitwise(lbmx_mod, dims, fbox, R):
    dev, ref = chain(dims, fbox, R)
    rng = np.random.default_rng(R)
    x, s = rng.random(ref.n), rng.standard_normal(ref.n)
    assert np.array_equal(dev.design(x), ref.density(x, R))
    assert np.array_equal(dev.sensitivities(s), ref.density_transpose(s, R))
    dev.close()


@pytest.mark.parametrize("dims,R", [((70, 30, 1), 5), ((40, 20, 9), 3)])
def test_nonfinite_values_stay_within_the_radius(lbmx_mod, dims, R):
    dev, ref = chain(dims, (0, dims[0] - 1, 0, dims[1] - 1, 0, dims[2] - 1), R)
    x = np.random.default_rng(1).random(ref.n)
    x[ref.n // 2], x[ref.n // 3] = np.inf, np.nan
    assert np.array_equal(dev.design(x), ref.density(x, R), equal_nan=True)
    assert np.array_equal(dev.sensitivities(x), ref.density_transpose(x, R), equal_nan=True)
    dev.close()


@pytest.mark.parametrize("project", [False, True])
def test_design_and_result_in_one_array(lbmx_mod, project):
    import torch
    dims = (130, 21, 1)
    dev, _ = chain(dims, (3, 120, 2, 18, 0, 0), 6, project)
    x = torch.rand(dims[0] * dims[1], dtype=torch.float64, device="cuda")
    apart = dev.design_device(x.clone())
    together = x.clone()
    dev.design_device(together, out=together)
    assert torch.equal(apart, together)
    dev.close()


def test_projection_over_its_whole_range(lbmx_mod):
    """Sharp projections saturate and near-zero arguments keep their digits: the projected field
    against the definition in the host's arithmetic, to a few units of the last place."""
    nx = 4096
    beta = 40.0
    box = B(0, nx - 1, 0, 0, 0, 0)
    dev = lbmx.Filter(lbmx.make_filter_desc(nx, 1, 1, box, box, ((1, True, beta, 0.5),)))
    x = np.concatenate([np.linspace(0.0, 1.0, nx // 2), 0.5 + np.linspace(-1e-9, 1e-9, nx // 2)])
    dev.design(x)
    f, p = dev.field(0), dev.field(1)
    ref = (np.tanh(beta * 0.5) + np.tanh(beta * (f - 0.5))) / (np.tanh(beta * 0.5) + np.tanh(beta * 0.5))
    assert np.max(np.abs(p - ref)) <= 4 * np.finfo(float).eps
    dev.close()
