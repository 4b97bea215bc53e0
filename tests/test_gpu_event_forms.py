"""The fused producers' event loop and FP64 event form at the sizes where they
can go wrong: event counts around a wave, a workgroup and a round of the
grid, every precision and grid mode, and integration limits of extreme width.
"""
import numpy as np
import pytest

from oracle import vegas as ora
from tests.parity import assert_sigma, kappa_vegas
from tests.test_gpu_kernels import DEV, FAMILIES, _fused_once, dev, random_grid, rel
from vegasflow_amd import kernels

pytestmark = pytest.mark.gpu


def _plain_once(fam, d, n, precision, limits=None):
    kw = {}
    if limits is not None:
        xmin, xmax = limits
        kw = dict(xmin=dev(xmin), xdelta=dev(xmax - xmin), xdeltajac=float(np.prod(xmax - xmin)))
    step = kernels.make_step(d, n, precision=precision, train=False, seed=3, draw_id=1, xjac=1.0 / n, **kw)
    ws = kernels.Workspace(DEV, kernels.partial_stride(d, 1, False))
    ng = kernels.plain_fused(step, FAMILIES[fam][0].to_struct(d), ws)
    return kernels.vegas_finalize(d, 1, False, False, n, ws, ng, raw=True).cpu().numpy()


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("d,n", [(1, 63), (3, 64), (7, 65), (8, 257), (2, 262144 + 63), (15, 524288 + 1), (16, 1024)])
def test_every_event_is_taken_once(d, n, precision):
    """A constant integrand on the identity grid gives every event the weight
    2.5 / n: its sum is 2.5, its sum of squares 6.25 / n and every
    dimension's histogram adds up to that, if and only if each event is
    taken once. The weight's rounding is the bound: FP64 a few ulp per
    operation, mixed d FP32 products of 2^-24 each, doubled by the square."""
    tol = 1e-13 if precision == "f64" else 2 * (d + 4) * 2.0 ** -24
    for train in (False, True):
        out, hist, _ = _fused_once("const", d, n, ora.initial_grid(d), train, precision=precision)
        assert abs(out[0] / 2.5 - 1.0) < tol
        if train:
            np.testing.assert_allclose(hist.sum(axis=1), 6.25 / n, rtol=tol)
    res, res2 = _plain_once("const", d, n, precision)
    assert abs(res / 2.5 - 1.0) < tol and abs(res2 * n / 6.25 - 1.0) < tol


@pytest.mark.parametrize("train", [True, False])
@pytest.mark.parametrize("d", [3, 4])
def test_f64_jacobian_of_extreme_limits(d, train):
    """Widths from 1e-60 to 1e60: the Jacobian comes from the slopes times
    per-pair constants, which must neither overflow nor lose digits; a
    dimension of zero width gives an integral of exactly 0."""
    n = 20_011
    rng = np.random.default_rng(d)
    grid = random_grid(rng, d)
    width = np.array([1e-60, 1e60, 1e-60, 1e60])[:d]
    xmin = np.zeros(d)
    out, hist, _ = _fused_once("product", d, n, grid, train, seed=5, draw=2, limits=(xmin, width))
    u = ora.uniform_f64(5, 2, n, d)
    res, sig, arr, *_ = ora.vegas_iteration(grid, u, ora.product, n, train=train, xmin=xmin, xmax=width)
    assert rel(out[0], res) < 1e-12
    assert_sigma(out[1], sig, kappa_vegas(res, sig, n))
    if train:
        np.testing.assert_allclose(hist, arr, rtol=1e-12)
    width[1] = 0.0
    out, _, _ = _fused_once("product", d, n, grid, train, seed=5, draw=2, limits=(xmin, width))
    assert out[0] == 0.0 and out[1] == 0.0


@pytest.mark.parametrize("fam,d", [("product", 3), ("gauss_offc", 8), ("bw", 4)])
def test_plain_limits_match_oracle(fam, d):
    """PlainFlow's one-FMA coordinate with integration limits."""
    n = 30_011
    xmin, xmax = np.linspace(0.05, 0.2, d), np.linspace(0.8, 1.7, d)
    res, res2 = _plain_once(fam, d, n, "f64", (xmin, xmax))
    x, w = ora.apply_xjac_and_limits(ora.uniform_f64(3, 1, n, d), np.ones(1), 1.0 / n, xmin, xmax)
    tmp = FAMILIES[fam][1](x) * w
    assert rel(res, tmp.sum()) < 1e-12 and rel(res2, np.square(tmp).sum()) < 1e-12
