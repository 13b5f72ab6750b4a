"""The neighbour rows of few cells (one group of lanes per cell) and of many
(one thread per cell), 1-D to 8-D, dense and sparse grids: every label against
the oracle, the candidate sum and the neighbour-row count against a count over
the occupied cells."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    yield c
    c.close()


def expected(x, eps):
    """(sum of candidates, neighbour rows): cells by the reference's float
    product, their neighbourhoods by comparing every pair of cells; a row of
    cells differs along the dimension of fewest cells only."""
    rcp = x.dtype.type(1) / x.dtype.type(eps)
    v = (x - x.min(axis=0)) * rcp
    cells, counts = np.unique(np.floor(v).astype(np.int64), axis=0, return_counts=True)
    ncell = np.ceil(v.max(axis=0)).astype(np.int64) + 1
    near = (np.abs(cells[:, None, :] - cells[None, :, :]) <= 1).all(axis=2)
    cand = int((near @ counts * counts).sum())
    rest = [k for k in range(x.shape[1]) if k != int(np.argmin(ncell))]
    _, row = np.unique(cells[:, rest], axis=0, return_inverse=True)
    rows = sum(len(np.unique(row[m])) for m in near)
    return cand, rows


@pytest.mark.parametrize("d", range(1, 9))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 63, 900])
def test_small_grids(ctx, d, dtype, n):
    rng = np.random.default_rng(10 * d + n)
    x = np.concatenate([rng.normal(2, 0.3, (n - n // 3, d)), rng.uniform(0, 5, (n // 3, d))])
    x = x.astype(dtype)
    eps, mp = 0.5, 4
    print(f"[gpu-case] neighbour rows d={d} n={n} {np.dtype(dtype).name}", flush=True)
    got = ctx.cluster(x, eps, mp)
    st = ctx.stats()
    mismatches, bad = oracle.check(x, eps, mp, got)
    assert mismatches == 0 and bad == 0
    spans = np.ceil((x.max(axis=0) - x.min(axis=0)) / eps)
    if len(np.unique(spans)) == d:  # no tie in the dimension order
        assert (st["sum_candidates"], st["neighbor_rows"]) == expected(x, eps)
    else:
        assert st["sum_candidates"] == expected(x, eps)[0]


@pytest.mark.parametrize("d,n", [(3, 500_000), (4, 220_000), (5, 100_000)])
def test_one_thread_per_cell(ctx, d, n):
    """More cells than the group kernel takes (2^22 lanes)."""
    rng = np.random.default_rng(d)
    x = rng.uniform(0, {3: 44.0, 4: 15.0, 5: 10.0}[d], (n, d)).astype(np.float32)
    x[: n // 4] = x[: n // 4] * np.float32(0.1)
    eps, mp = 0.5, 5
    print(f"[gpu-case] neighbour rows, many cells d={d} n={n}", flush=True)
    got = ctx.cluster(x, eps, mp)
    assert ctx.stats()["occupied_cells"] * {3: 16, 4: 32, 5: 64}[d] > 1 << 22
    r = oracle.check_parallel(x, eps, mp, got, threads=16)
    assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
