"""The samplers with a compile-time n_dim against the runtime-n_dim kernels
(which take the same draws injected), bit by bit, and the pair-table digests
against numpy on values whose sums have no rounding."""
import numpy as np
import pytest
import torch

from oracle import vegas as ora
from vegasflow_amd import kernels

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
SEED, DRAW, OFFSET = 77, 4, (1 << 32) - 100  # the event counter's low word wraps


def _grid(rng, d):
    edges = np.zeros((d, 51))
    edges[:, 1:] = np.cumsum(rng.uniform(0.1, 1.0, (d, 50)), axis=1)
    return torch.tensor(edges / edges[:, -1:], device=DEV)


def _strata(rng, d, n_strat, largest):
    n_ev = rng.integers(2, largest + 1, size=n_strat**d).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(n_ev)]).astype(np.int32)
    n_ev_dev, off_dev = torch.tensor(n_ev, device=DEV), torch.tensor(off, device=DEV)
    return n_ev, off, kernels.make_strata(n_strat, n_strat**d, n_ev_dev, off_dev), (n_ev_dev, off_dev)


def _inject(precision, n, d):
    if precision == "f64":
        return torch.tensor(ora.uniform_f64(SEED, DRAW, n, d, event_offset=OFFSET), device=DEV)
    words = ora.hi_words(SEED, DRAW, n, d, event_offset=OFFSET).astype(np.uint32)
    return torch.tensor(words.view(np.int32), device=DEV)


def _outputs(precision, n, d, shift):
    """x, w, idx, seg buffers that start ``shift`` elements into an allocation."""
    ft = torch.float64 if precision == "f64" else torch.float32

    def buf(count, dtype):
        return torch.zeros(count + shift, dtype=dtype, device=DEV)[shift:]

    return buf(n * d, ft), buf(n, ft), buf(n * d, torch.uint8), buf(n, torch.int32)


@pytest.mark.parametrize("limits", [False, True])
@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("d,n,shift", [(1, 65, 0), (2, 64, 0), (3, 4097, 1), (4, 63, 0), (5, 1000, 0), (6, 20001, 0),
                                       (7, 130, 3), (8, 4096, 0), (13, 777, 0), (16, 1, 0)])
def test_samplers_match_runtime_dimension_kernels(d, n, shift, precision, limits):
    rng = np.random.default_rng(d)
    grid = _grid(rng, d)
    _, off, strata, _keep = _strata(rng, d, 2 if d > 3 else 5, 3 if d > 8 else 150)
    lim = {"xmin": torch.full((d,), -1.5, dtype=torch.float64, device=DEV),
           "xdelta": torch.full((d,), 2.25, dtype=torch.float64, device=DEV), "xdeltajac": 2.25**d} if limits else {}
    for kind in ("plain", "vegas", "vplus"):
        count = int(off[-1]) if kind == "vplus" else n
        inject = _inject(precision, count, d)
        got, want = _outputs(precision, count, d, shift), _outputs(precision, count, d, 0)
        for out, inj in ((got, None), (want, inject)):
            step = kernels.make_step(d, count, precision=precision, train=True, event_offset=OFFSET, seed=SEED,
                                     draw_id=DRAW, xjac=1.0 / count, inject=inj, **lim)
            x, w, idx, seg = out
            if kind == "plain":
                kernels.plain_sample(step, x)
            elif kind == "vegas":
                kernels.vegas_sample(step, grid, x, w, idx)
            else:
                kernels.vplus_sample(step, strata, grid, x, w, idx, seg)
        for name, a, b in zip(("x", "w", "idx", "seg"), got, want):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy(), err_msg=f"{kind} {name}")


@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("d,n,largest", [(2, 1, 3), (3, 63, 5), (4, 64, 12), (5, 65, 30), (6, 4097, 300), (9, 20000, 7),
                                         (14, 1000, 2)])
def test_digest_sums_are_exact_on_integers(d, n, largest, precision):
    """Weights 1 and 2, values -2..2: every square is at most 16 and all sums
    stay far below 2^53, so no order of additions rounds."""
    rng = np.random.default_rng(d)
    ft = torch.float64 if precision == "f64" else torch.float32
    n_ev, off, strata, _keep = _strata(rng, d, 2, largest)
    for cubes in (False, True):
        count = int(off[-1]) if cubes else n
        f, w = rng.integers(-2, 3, count), rng.integers(1, 3, count)
        idx = rng.integers(0, 50, (count, d)).astype(np.uint8)
        idx[: count // 3, 0] = 7  # many adds to the same cells
        seg = np.repeat(np.arange(len(n_ev)), n_ev).astype(np.int32)
        step = kernels.make_step(d, count, precision=precision, train=True)
        ws = kernels.Workspace(DEV, kernels.partial_stride(d, 1, True))
        args = [torch.tensor(f, dtype=ft, device=DEV), torch.tensor(w, dtype=ft, device=DEV), torch.tensor(idx, device=DEV)]
        tmp = (f * w).astype(np.float64)
        if cubes:
            ress, ress2 = (torch.zeros(len(n_ev), dtype=torch.float64, device=DEV) for _ in range(2))
            kernels.vplus_digest(step, strata, *args, torch.tensor(seg, device=DEV), ress, ress2, ws)
            np.testing.assert_array_equal(ress.cpu().numpy(), np.bincount(seg, tmp, len(n_ev)))
            np.testing.assert_array_equal(ress2.cpu().numpy(), np.bincount(seg, tmp * tmp, len(n_ev)))
        else:
            kernels.vegas_digest(step, *args, ws)
        row = ws.rows.reshape(-1, ws.stride).sum(dim=0).cpu().numpy()
        if not cubes:
            assert row[0] == tmp.sum() and row[1] == (tmp * tmp).sum()
        hist = row[2:2 + 50 * d].reshape(d, 50)
        for j in range(d):
            np.testing.assert_array_equal(hist[j], np.bincount(idx[:, j], tmp * tmp, 50))
