"""Pairs of boxes of more than 2048 rows that only the exact union can join: the
single core pair within eps lies beyond the rows that the hook forest and the
root join look at (the first and last rows, the first 64 of the searching box,
the first 4096 of the other), so the pair goes by parts through the union's
list, and with the list cut short is tested in place."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

EPS = 1.0
MIN_POINTS = 40


def bridged(sizes, d, dtype, seed, bridge=True):
    """Two crowds of sizes[0] and sizes[1] rows in one sub-box each (eps / 2 wide),
    farther apart than eps but for one row of each, the 5000th of its crowd in
    input order; a third crowd apart from both."""
    rng = np.random.default_rng(seed)

    def block(n, x0):
        rows = rng.uniform(0.0, 0.01, (n, d))
        rows[:, 0] += x0
        return rows

    a, b = block(sizes[0], 0.0), block(sizes[1], 1.47)
    if bridge:
        a[4999, 0], b[4999, 0] = 0.43, 1.04
    third = block(3000, 4.2)
    # the crowds' rows take turns, each crowd in its own order
    which = rng.permutation(np.repeat([0, 1, 2], [len(a), len(b), len(third)]))
    x = np.empty((len(which), d))
    for k, rows in enumerate((a, b, third)):
        x[which == k] = rows
    corner = np.zeros((1, d))
    return np.concatenate([corner, x]).astype(dtype), np.concatenate([[0], which])


CASES = [((5001, 9000), 2, np.float32), ((9000, 5001), 3, np.float32), ((6000, 6000), 2, np.float64),
         ((7000, 5500), 3, np.float64)]


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,d,dtype", CASES)
def test_pairs_of_large_boxes(sizes, d, dtype):
    from hpdbscan_amd import _lib
    x, which = bridged(sizes, d, dtype, 7 + d)
    want = oracle.cluster(x, EPS, MIN_POINTS)
    assert len(np.unique(want[which < 2])) == 1 and len(np.unique(want)) == 2
    ctx = _lib.Context(0)
    try:
        # (2: no room for the parts of the larger box; 0: all of them)
        for limit in (0, 1, 2):
            print(f"[gpu-case] bridged boxes of {sizes} rows d={d} {np.dtype(dtype).name} "
                  f"limit={limit}", flush=True)
            ctx.set_open_pair_limit(limit)
            np.testing.assert_array_equal(ctx.cluster(x, EPS, MIN_POINTS), want)
            st = ctx.stats()
            assert st["box_union"] == 1 and st["open_box_pairs"] == 1
        ctx.set_graph(True)
        print("[gpu-case] the same, static pipeline", flush=True)
        np.testing.assert_array_equal(ctx.cluster(x, EPS, MIN_POINTS), want)
        assert ctx.graph_stats()["fallbacks"] == 0 and ctx.stats()["open_box_pairs"] == 1
        ctx.set_graph(False)
        # without the bridge the two stay apart
        y, _ = bridged(sizes, d, dtype, 7 + d, bridge=False)
        got = ctx.cluster(y, EPS, MIN_POINTS)
        np.testing.assert_array_equal(got, oracle.cluster(y, EPS, MIN_POINTS))
        assert len(np.unique(got)) == 3
    finally:
        ctx.close()
