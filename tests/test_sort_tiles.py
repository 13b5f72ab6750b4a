"""Row counts around the edges where the sort changes its tiles (1024, 2048 and
4096 keys, up to 192 of them adding their own histograms) and the box table its
blocks: labels against the oracle's checker, and the same labels from the
static pipeline (whose sort runs on device-written key bits)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SELF = 192


@pytest.fixture(scope="module")
def ctx():
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    yield c
    c.close()


def blobs(n, d, seed):
    rng = np.random.default_rng(seed)
    centres = rng.uniform(0, 100, (60, d))
    x = centres[rng.integers(0, 60, n)] + rng.normal(0, 0.6, (n, d))
    far = rng.integers(0, n, n // 20)
    x[far] = rng.uniform(0, 100, (len(far), d))
    return x.astype(np.float32)


@pytest.mark.parametrize("tile", [1024, 2048, 4096])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("d", [1, 2, 3])  # 1, 2: the rows travel with the keys
def test_tile_edges(ctx, tile, off, d):
    n = SELF * tile + off
    x = blobs(n, d, n + d)
    eps, mp = {1: 2e-4, 2: 0.05, 3: 0.35}[d], 6
    print(f"[gpu-case] sort tiles n={n} d={d}", flush=True)
    got = ctx.cluster(x, eps, mp)
    r = oracle.check_parallel(x, eps, mp, got, threads=16)
    assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    try:
        c.set_graph(True)
        for _ in range(2):
            np.testing.assert_array_equal(c.cluster(x, eps, mp), got)
    finally:
        c.close()


@pytest.mark.parametrize("n", [6001, 6145, 7168, 7169, 12_289])
def test_few_tiles(ctx, n):
    for d in (1, 2, 3, 5):
        x = blobs(n, d, n + d)
        eps, mp = {1: 5e-3, 2: 0.3, 3: 0.9, 5: 1.2}[d], 6
        print(f"[gpu-case] sort tiles n={n} d={d}", flush=True)
        got = ctx.cluster(x, eps, mp)
        mismatches, bad = oracle.check(x, eps, mp, got)
        assert mismatches == 0 and bad == 0
