"""Sub-boxes of more rows than one wave walks at once: rows at the rim of a box
of 16384 * k + r rows whose answer hangs on its far rows (core counts put off in
parts, border labels put off in parts), and box pairs that meet only there,
against the oracle's checker and with the box lists cut to one entry (every
walk in place)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

EPS = 1.0


@pytest.fixture(scope="module")
def ctx():
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    yield c
    c.close()


def rim(n, d, dtype, seed):
    """One crowd of n rows inside [0, 0.45]^d (one sub-box of eps / 2), nearly
    all of it in the near corner, and rows around it at distances near eps from
    the few far rows only."""
    rng = np.random.default_rng(seed)
    crowd = rng.uniform(0.0, 0.1, (n, d))
    far = rng.choice(n, 40, replace=False)
    crowd[far] = rng.uniform(0.3, 0.45, (40, d))
    around = rng.uniform(-1.6, 2.2, (3000, d))
    around = around[(around < 0.0).any(axis=1) | (around > 0.5).any(axis=1)]
    second = np.full((200, d), 1.9) + rng.uniform(0, 0.2, (200, d))
    x = np.concatenate([crowd, around, second, np.full((1, d), -2.0)])
    return x[rng.permutation(len(x))].astype(dtype)


@pytest.mark.parametrize("n", [16_384, 16_385, 50_001])
@pytest.mark.parametrize("d,dtype", [(2, np.float32), (3, np.float32), (2, np.float64)])
@pytest.mark.parametrize("min_points", [25, 60])
def test_rim_rows(ctx, n, d, dtype, min_points):
    x = rim(n, d, dtype, n + d)
    print(f"[gpu-case] rim of a box of {n} rows, d={d} {np.dtype(dtype).name} minPts={min_points}",
          flush=True)
    got = ctx.cluster(x, EPS, min_points)
    st = ctx.stats()
    assert st["noise_points"] == int((got == 0).sum())
    assert st["core_points"] == int((got < 0).sum())
    r = oracle.check_parallel(x, EPS, min_points, got, threads=16)
    assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    try:
        c.set_open_pair_limit(1)
        np.testing.assert_array_equal(c.cluster(x, EPS, min_points), got)
        c.set_open_pair_limit(0)
        c.set_graph(True)  # the static pipeline walks in place
        np.testing.assert_array_equal(c.cluster(x, EPS, min_points), got)
    finally:
        c.close()
