"""The pair kernels' split of a tile list: every event of every tile exactly
once, whatever the list looks like."""
import numpy as np
import pytest
import torch

from vegasflow_amd import Constant, _abi, kernels
from vegasflow_amd.batch import BatchVegas

pytestmark = pytest.mark.gpu


def _tiles(rows, device):
    arr = (_abi.BatchTile * len(rows))()
    for k, (item, count, first) in enumerate(rows):
        arr[k].item, arr[k].count, arr[k].first = item, count, first
    return torch.from_numpy(np.frombuffer(bytes(arr), dtype=np.uint8).copy()).to(device)


def _pieces(rng, item, n, size):
    cuts = np.unique(np.concatenate([[0, n], rng.integers(0, n, max(n // size, 0))]))
    return [(item, int(b - a), int(a)) for a, b in zip(cuts[:-1], cuts[1:])]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("sizes,piece,shuffle", [
    ([1 << 22], 1 << 30, False),                       # one tile, all workgroups
    ([2, 3, 64, 65, 127, 4096], 1 << 30, False),       # less than one workgroup's share each
    ([1 << 20, 3, 1 << 14, 77777, 1 << 18], 100, True),  # over 1e4 ragged tiles, no two in order
    ([1 << 20, 300001, 5000], 1000, False),            # over 1024 tiles that join
])
def test_every_event_counts_once(sizes, piece, shuffle, dtype):
    """With the integrand 1 and a uniform grid every event's w f / N is 1 / N to
    rounding. FP64: 14 factors with a few roundings each and sums of up to
    2^22 terms stay within 2^-46 + n 2^-53 of it, so a missing or repeated
    event shows. FP32: 14 factors of the map and 14 products within 2^-24
    each, 2^-19 altogether and twice that for squares, below one trip of 64
    events out of 2^22."""
    rng = np.random.default_rng(len(sizes))
    dims = [2, 3, 6, 7, 14, 9][: len(sizes)]
    b = BatchVegas([(Constant(1.0), d, n, 5 + i) for i, (d, n) in enumerate(zip(dims, sizes))], dtype=dtype,
                   events_per_tile=1024, pair_histograms=True)
    rows = [t for i, n in enumerate(sizes) for t in _pieces(rng, i, n, piece)]
    rows += [(0, 0, 0), (len(sizes) - 1, 0, 5)]  # empty tiles
    if shuffle:
        rng.shuffle(rows)
        rows = [tuple(int(v) for v in r) for r in rows]
    family, _, _, max_dim = b._launches[0]
    blocks = kernels.batch_pairs_blocks(family, max_dim, b.precision)
    for n_blocks in (1, 3, blocks):
        b.rows.zero_()
        kernels.batch_fused_pairs(b.items, b.n_items, _tiles(rows, b.device), len(rows), family, max_dim, b.draws,
                                  b.grids, b.rows, n_blocks, b.precision)
        out = b.rows.cpu().numpy()
        at = 0
        for d, n in zip(dims, sizes):
            row = out[at:at + 2 + 50 * d]
            at += 2 + 50 * d
            tol = n * (2.0**-18 if dtype == torch.float32 else 2.0**-45 + n * 2.0**-52)
            assert abs(row[0] * n - n) <= tol and abs(row[1] * n * n - n) <= tol
            hist = row[2:].reshape(d, 50) * n * n
            assert np.all(np.abs(hist.sum(axis=1) - n) <= tol)
            if dtype == torch.float64:
                assert np.all(np.abs(hist - np.round(hist)) <= tol)
