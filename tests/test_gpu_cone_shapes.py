"""Cone filter on grids either side of the line between the kernel of the radius and the kernel of
any radius: bit for bit against the oracle's row loop, at the edges of the former's tiles."""
import numpy as np
import pytest

import lbmx
from test_gpu_cone_tiles import chain

pytestmark = pytest.mark.gpu

# 3D: 3 x 2 workgroups of the kernel of any radius per slice; slices left over after fours
CASES = [((129, 17, nz), (1, 127, 2, 15, 1, nz - 2), R)
         for R, sizes in ((1, (266, 267, 583, 587)), (2, (149, 151, 247, 251)), (3, (115, 117, 183, 185))) for nz in sizes]
CASES += [((37, 5, 2), (30, 36, 0, 4, 0, 1), 3), ((16, 16, 16), (0, 15, 0, 15, 0, 15), 2)]
CASES += [((3, ny, 1), (0, 2, 1, ny - 2, 0, 0), 2) for ny in (524280, 524281, 700001)]  # tall 2D grids


@pytest.mark.parametrize("dims,fbox,R", CASES)
def test_cone_shapes_bitwise(lbmx_mod, dims, fbox, R):
    dev, ref = chain(dims, fbox, R)
    rng = np.random.default_rng(R)
    x, s = rng.random(ref.n), rng.standard_normal(ref.n)
    assert np.array_equal(dev.design(x), ref.density(x, R))
    assert np.array_equal(dev.sensitivities(s), ref.density_transpose(s, R))
    dev.close()
