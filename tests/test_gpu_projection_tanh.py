"""The projection's tanh on the device, digit by digit. A filter of radius 1 is the identity (its
only weight is the node's own), and with eta = 0 and beta = 64 the projected value is
(tanh(0) + tanh(64 x)) / (tanh(0) + tanh(64)) = tanh(64 x) exactly, with 64 x exact: the field is
the device's tanh itself. The reference is the host's 64-bit-mantissa tanh, whose own error is
about a thousandth of a unit of a double's last place."""
import numpy as np
import pytest

import lbmx

pytestmark = pytest.mark.gpu

N = 512


def project(x, eta, beta, eta_field=None):
    box = lbmx.make_box(0, N - 1, 0, N - 1, 0, 0)
    dev = lbmx.Filter(lbmx.make_filter_desc(N, N, 1, box, box, ((1, True, beta, eta),)))
    if eta_field is not None:
        dev.set_eta_field(0, eta_field)
    p = dev.design(x)
    assert np.array_equal(dev.field(0), x)
    dev.close()
    return p


def arguments():
    rng = np.random.default_rng(5)
    n = N * N // 4
    edges = (rng.integers(0, 40, n) + 0.5) * (np.log(2.0) / 2)  # where 2 |x| / ln 2 rounds up or down
    a = np.concatenate([10.0 ** rng.uniform(-290, 1.3, n), rng.uniform(0.0, 22.0, n), rng.uniform(0.1, 0.25, n),
                        edges * (1.0 + 1e-6 * rng.standard_normal(n))])
    return a * rng.choice([-1.0, 1.0], a.size)


def test_tanh_to_the_last_place(lbmx_mod):
    assert np.finfo(np.longdouble).nmant >= 63
    a = arguments()
    p = project(a / 64.0, 0.0, 64.0)
    ref = np.tanh(a.astype(np.longdouble))
    err = np.abs((p.astype(np.longdouble) - ref) / np.spacing(np.abs(ref.astype(np.float64)))).astype(np.float64)
    k = int(np.argmax(err))
    print(f"largest error {err[k]:.3f} units of the last place at {a[k]!r}, rms {np.sqrt(np.mean(err ** 2)):.3f}")
    assert err[k] < 1.0
    assert np.array_equal(np.signbit(p), np.signbit(a))


def test_per_node_thresholds(lbmx_mod):
    """Thresholds from a field: the same bits as the constant where they are equal, and the
    definition elsewhere. Units u = 2^-53: three tanh of 1 u at most and their two sums (values
    below 2: 1 u each), the argument's two roundings (|x| sech^2 x < 0.45 each) and the quotient
    with tsum > 0.9 leave less than 10 u of values up to 1."""
    rng = np.random.default_rng(6)
    a = arguments()
    assert np.array_equal(project(a / 64.0, 0.0, 64.0, np.zeros(N * N)), project(a / 64.0, 0.0, 64.0))
    x, eta, beta = rng.random(N * N), rng.uniform(0.3, 0.7, N * N), 4.0
    p = project(x, 0.5, beta, eta).astype(np.longdouble)
    xl, el = x.astype(np.longdouble), eta.astype(np.longdouble)
    tb = np.tanh(beta * el)
    ref = (tb + np.tanh(beta * (xl - el))) / (tb + np.tanh(beta * (1 - el)))
    assert float(np.max(np.abs(p - ref))) < 10 * 2.0 ** -53
