"""Independent iterations (a frozen grid, PlainFlow) in one launch: the same
draws, results and history as one after the other, to summation order."""
import numpy as np
import pytest
import torch

import vegasflow_amd as vf
from vegasflow_amd import kernels

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _close(a, b, n):
    """Sums of n terms in two orders: within n 2^-53 of each other at worst;
    sigma^2 (N sum f^2 - (sum f)^2, of a flat integrand) may cancel to 1e-4."""
    for (ra, ea, _), (rb, eb, _) in zip(a.history, b.history):
        assert abs(ra - rb) <= n * 2.0**-53 * abs(rb)
        assert abs(ea - eb) <= 1e4 * n * 2.0**-53 * abs(eb)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("cls,d,n,limits", [(vf.VegasFlow, 1, 2, False), (vf.VegasFlow, 3, 257, True),
                                            (vf.VegasFlow, 8, 100_003, False), (vf.VegasFlow, 16, 4096, False),
                                            (vf.PlainFlow, 2, 300_000, True), (vf.PlainFlow, 7, 63, False),
                                            (vf.PlainFlow, 20, 5000, False)])
def test_groups_match_single_iterations(cls, d, n, limits, dtype):
    box = {"xmin": [-0.5] * d, "xmax": [1.25] * d} if limits else {}
    runs = (1, 2, 5, 16, 17, 40)
    out = []
    for replayed in (False, True):
        inst = cls(d, n, seed=13, verbose=False, dtype=dtype, **box)
        inst.use_graphs = replayed
        inst.compile(vf.Product())
        if cls is vf.VegasFlow:
            inst.freeze_grid()
        for n_iter in runs:
            inst.run_integration(n_iter)
        out.append(inst)
    eager, grouped = out
    assert len(grouped.history) == len(eager.history) == sum(runs)
    assert grouped._draw_count == eager._draw_count
    _close(grouped, eager, n)


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_groups_across_the_counter_wrap(precision):
    """Events on both sides of 2^32: the pieces of every iteration meet in its
    own rows."""
    d, n, iters = 4, 5000, 3
    fn = vf.Product().to_struct(d)
    grid = torch.linspace(0, 1, 51, dtype=torch.float64, device=DEV).repeat(d, 1)
    rows = {}
    for group in (1, iters):
        counter = kernels.IterationCounter(DEV, 8)
        slot = counter.start(7, iters)
        for kind in ("vegas", "plain"):
            ws = kernels.Workspace(DEV, 2, group)
            for _ in range(iters // group):
                step = kernels.make_step(d, n, precision=precision, train=False, event_offset=(1 << 32) - 999, seed=3,
                                         xjac=1.0 / n, draw_dev=counter.draw, iterations=group)
                ng = kernels.vegas_fused(step, fn, grid, ws) if kind == "vegas" else kernels.plain_fused(step, fn, ws)
                kernels.vegas_finalize(d, 1, False, False, n, ws, ng, counter=counter, status=counter.status,
                                       iterations=group)
            assert float(ws.rows.abs().max()) == 0.0
            status, _, got = counter.read(7, slot, iters)
            rows[kind, group] = got.copy()
            assert status == 0
            counter.draw.fill_(7)
    for kind in ("vegas", "plain"):
        np.testing.assert_allclose(rows[kind, iters], rows[kind, 1], rtol=n * 2.0**-53 * 10)


def test_what_groups_refuse():
    d, n = 3, 100
    fn = vf.Product().to_struct(d)
    grid = torch.linspace(0, 1, 51, dtype=torch.float64, device=DEV).repeat(d, 1)
    ws = kernels.Workspace(DEV, kernels.partial_stride(d, 1, True), 2)
    train = kernels.make_step(d, n, train=True, xjac=1.0 / n, iterations=2)
    with pytest.raises(Exception, match="several iterations"):
        kernels.vegas_fused(train, fn, grid, ws)
    inject = torch.full((n, d), 0.5, dtype=torch.float64, device=DEV)
    with pytest.raises(Exception, match="several iterations"):
        kernels.plain_fused(kernels.make_step(d, n, train=False, xjac=1.0 / n, inject=inject, iterations=2), fn, ws)
    with pytest.raises(ValueError, match="rows for 1 iterations"):
        kernels.plain_fused(kernels.make_step(d, n, train=False, xjac=1.0 / n, iterations=2), fn,
                            kernels.Workspace(DEV, 2))
    with pytest.raises(Exception, match="several iterations need a counter"):
        kernels.vegas_finalize(d, 1, False, False, n, ws, 1, iterations=2)
    assert float(ws.rows.abs().max()) == 0.0
