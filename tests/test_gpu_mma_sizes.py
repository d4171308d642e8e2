"""MMA updates on the device at the sizes where its reductions change shape: one variable, one
workgroup more or less than full, more variables than one pass of the grid covers, every
number of constraints; and updates whose arrays share memory. Bars as for the other updates: the
interior-point tolerance's effect on the design stays below 1e-9 per update."""
import numpy as np
import pytest

import lbmx
import oracle

pytestmark = pytest.mark.gpu


def inputs(x, targets, weights):
    n = x.size
    g = [w * np.sum((x - t) ** 2) / n for t, w in zip(targets, weights)] + [x.mean() - 0.45]
    dg = [2 * w * (x - t) / n for t, w in zip(targets, weights)] + [np.full(n, 1.0 / n)]
    return np.zeros(n), np.array(g), np.stack(dg)


@pytest.mark.parametrize("n,m", [(1, 2), (63, 3), (256, 2), (257, 5), (5000, 8), (3000, 7), (20011, 6), (600001, 2)])
@pytest.mark.parametrize("modified", [False, True])
def test_updates_match_oracle(lbmx_mod, n, m, modified):
    rng = np.random.default_rng(n + m)
    targets = [0.2 + 0.6 * rng.random(n) for _ in range(m - 1)]
    weights = [1.0 + 0.1 * k for k in range(m - 1)]
    a = [1.0] * (m - 1) + [0.0]
    dev, ref = lbmx.MMA(n, m, a=a), oracle.MMA(n, m, a=a)
    dev.set_options(constraint_modification=modified)
    ref.set_options(constraint_modification=modified)
    xd = xr = np.full(n, 0.5)
    for _ in range(4):
        xd = dev.update(xd, *inputs(xd, targets, weights), 0.1)
        xr = ref.update(xr, *inputs(xr, targets, weights), 0.1)
        assert np.max(np.abs(xd - xr)) < 1e-9
        assert abs(dev.design_change() - ref.design_change(xr)) < 1e-9
        xd = xr.copy()  # (each update is compared by itself)
    dev.close()


def test_arrays_that_share_memory(lbmx_mod):
    """The design may be the objective's sensitivity array itself or overlap a constraint's."""
    import torch
    n = 4000
    gen = torch.Generator(device="cuda").manual_seed(3)
    pool = torch.rand(n + 100, dtype=torch.float64, device="cuda", generator=gen) * 0.5 + 0.2

    def update(x, df, dg):
        mma = lbmx.MMA(n, 1)
        mma.update_device(x, df, [0.1], [dg], 0.1)
        out = x.clone()
        mma.close()
        return out

    vol = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    apart = update(pool[:n].clone(), pool[:n].clone(), vol)
    shared = pool[:n].clone()
    assert torch.equal(apart, update(shared, shared, vol))
    apart = update(pool[:n].clone(), vol, pool[100:].clone())
    both = pool.clone()
    assert torch.equal(apart, update(both[:n], vol, both[100:]))
