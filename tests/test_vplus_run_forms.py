"""The VEGAS+ run loop's cube arithmetic on the CPU, and the loop itself on the
GPU where it can go wrong: trips across no, one, a few and many cube
boundaries, empty cubes, partial last trips and runs across a multiple of
2^32 in the event counter.
"""
import numpy as np
import pytest
import torch

from oracle import vegas as ora


def _magic(n):
    """magic and shift of StrataPos (vplus_fused.hpp) for n_strat = n, with
    its FP64 division."""
    log = 0 if n <= 1 else (n - 1).bit_length()
    shift = max(0, log - 8)
    return (int(float(2 ** (32 + shift)) / float(n)) + 1) & 0xFFFFFFFF, shift


def test_cube_digits_by_multiplication_are_exact():
    """mulhi(c, magic) >> shift = c / n for every cube index below 2^24: around
    every multiple of n near both ends and at random indices, for every
    n_strat that n_dim >= 2 allows, and far beyond."""
    rng = np.random.default_rng(0)
    top = 1 << 24
    for n in list(range(2, 4097)) + [5000, 65535, 65536, 65537, (1 << 22) + 1, (1 << 23) - 1]:
        magic, shift = _magic(n)
        assert magic < 1 << 32
        k = np.unique(np.concatenate([np.arange(1, 20), rng.integers(1, top // n + 2, 50),
                                      np.arange(max(1, top // n - 20), top // n + 1)]))
        c = np.concatenate([k * n - 1, k * n, rng.integers(0, top, 50)])
        c = c[(c >= 0) & (c < top)].astype(np.uint64)
        q = (c * np.uint64(magic)) >> np.uint64(32 + shift)
        np.testing.assert_array_equal(q, c // np.uint64(n))


def test_position_by_fma_stays_inside_and_accurate():
    """base + per_draw * draw at the draws' extremes: never outside (0, 50), and
    as near to the real number (80-bit) as three roundings of values up to 50
    allow, 150 * 2^-53, the bound of the reference's three roundings too: the
    draw's term carries the two of its factor (and is at most 50 / n), the
    corner's term the two of base (at most 50 - 50 / n), and their sum one."""
    real = np.longdouble
    span, cut = (1.0 - 1e-8) - 1e-8, 1e-8
    r = np.array([0.0, 2.0 ** -52, 0.5, 1.0 - 2.0 ** -52]).astype(real)
    hw = np.array([0, 1, 2 ** 31, 2 ** 32 - 1]).astype(real)
    for n in list(range(1, 300)) + [1000, 2047, 4095]:
        c = 50.0 / n
        h = np.arange(n).astype(real)[:, None]
        base = (h * real(c) + real(c * cut)).astype(np.float64)
        f64 = (r * real(c * span) + base).astype(np.float64)
        mixed = (hw * real(c * 2.0 ** -32) + (h * real(c)).astype(np.float64)).astype(np.float64)
        assert f64.min() > 0.0 and f64.max() < 50.0
        assert mixed.min() >= 0.0 and mixed.max() < 50.0
        for got, u in ((f64, r * real(span) + real(cut)), (mixed, hw * real(2.0 ** -32))):
            assert np.abs(got - (h + u) * 50 / n).max() <= 150 * 2.0 ** -53


def _events(pattern, n_cubes, rng):
    if pattern == "boundary_counts":  # 64-event trips of 1 to 33 cubes, cubes of 1 to 200 events
        n_ev = np.concatenate([np.repeat(np.array([200, 63, 64, 65, 1, 30, 21, 16, 13, 12, 2]), 7),
                               rng.integers(1, 90, n_cubes)])[:n_cubes]
        return rng.permutation(n_ev)
    if pattern == "one_large":  # one wave's worth of events in one cube
        n_ev = np.full(n_cubes, 2)
        n_ev[n_cubes // 2] = 40_000
        return n_ev
    n_ev = rng.integers(2, 40, n_cubes)  # runs of empty cubes between others
    n_ev[rng.random(n_cubes) < 0.3] = 0
    n_ev[100:180] = 0
    return n_ev


CASES = [(2, 20, "boundary_counts", 0), (3, 7, "one_large", 0), (4, 5, "empty", 0),
         (2, 20, "boundary_counts", 2 ** 32 - 5_003), (5, 4, "boundary_counts", 2 ** 32 - 64)]


def _produce(precision, fn, d, n_strat, pattern, offset):
    """One producer call; the per-cube sums and the histograms, and the
    oracle's x, w (jacobian included), bins and cubes of the same draws."""
    from tests.test_gpu_vplus import DEV, _device_strata, dev, random_grid
    from vegasflow_amd import kernels

    rng = np.random.default_rng(d + n_strat)
    n_cubes = n_strat ** d
    n_ev = _events(pattern, n_cubes, rng).astype(np.int32)
    total = int(n_ev.sum())
    grid = random_grid(rng, d)
    _, _, strata = _device_strata({"n_strat": n_strat, "n_cubes": n_cubes, "n_ev": n_ev})
    ress = torch.zeros(n_cubes, dtype=torch.float64, device=DEV)
    ress2 = torch.zeros_like(ress)
    ws = kernels.Workspace(DEV, kernels.partial_stride(d, 1, True))
    step = kernels.make_step(d, total, precision=precision, train=True, seed=23, draw_id=5, event_offset=offset,
                             xjac=1.0 / n_cubes)
    ng = kernels.vplus_fused(step, strata, fn.to_struct(d), dev(grid), ress, ress2, ws)
    hist = torch.empty((d, 50), dtype=torch.float64, device=DEV)
    kernels.vegas_finalize(d, 1, True, False, total, ws, ng, hist_out=hist, raw=True)
    if precision == "f64":
        u = ora.uniform_f64(23, 5, total, d, event_offset=offset)
    else:
        u = ora.hi_words(23, 5, total, d, event_offset=offset).astype(np.float64) * 2.0 ** -32
    x, w, ind, seg = ora.generate_samples_in_hypercubes(u, n_strat, n_ev, ora.hypercubes(n_strat, d), grid)
    x, w = ora.apply_xjac_and_limits(x, w, 1.0 / n_cubes)
    return ress.cpu().numpy(), ress2.cpu().numpy(), hist.cpu().numpy(), x, w, ind, seg


@pytest.mark.gpu
@pytest.mark.parametrize("d,n_strat,pattern,offset", CASES)
def test_run_loop_matches_oracle(d, n_strat, pattern, offset):
    """FP64: per-cube sums and bin histograms of one producer call within
    1e-12 of each sum (for cubes of tiny sums, 1e-14 of the largest)."""
    from tests.test_gpu_vplus import MIX, mix_np

    ress, ress2, hist, x, w, ind, seg = _produce("f64", MIX, d, n_strat, pattern, offset)
    tmp = w * mix_np(x)
    for got, values in ((ress, tmp), (ress2, np.square(tmp))):
        want = np.bincount(seg, weights=values, minlength=n_strat ** d)
        np.testing.assert_allclose(got, want, rtol=1e-12, atol=1e-14 * want.max())
    want = ora.bin_histogram(np.square(tmp), ind, d)
    np.testing.assert_allclose(hist, want, rtol=1e-12, atol=1e-14 * want.max())


@pytest.mark.gpu
@pytest.mark.parametrize("d,n_strat,pattern,offset", CASES)
def test_mixed_run_loop_matches_oracle(d, n_strat, pattern, offset):
    """Mixed, with the product of the coordinates, whose FP32 rounding has a
    bound: a coordinate P + Q frac of positive terms carries at most three
    roundings and its product one, a Jacobian factor one and its product
    one, so an event 6 d of 2^-24, its square 12 d, and sums of positive
    terms no more."""
    from vegasflow_amd.integrands import Product

    ress, ress2, hist, x, w, ind, seg = _produce("mixed", Product(), d, n_strat, pattern, offset)
    tmp = w * ora.product(x)
    rtol = 12 * d * 2.0 ** -24 + 1e-12
    for got, values in ((ress, tmp), (ress2, np.square(tmp))):
        np.testing.assert_allclose(got, np.bincount(seg, weights=values, minlength=n_strat ** d), rtol=rtol)
    np.testing.assert_allclose(hist, ora.bin_histogram(np.square(tmp), ind, d), rtol=rtol)
