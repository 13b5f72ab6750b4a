"""4-D to 8-D rows beyond the all-pairs sizes (groups of 32 and 64 lanes per
chunk, box and row; neighbourhoods of up to 3^(D-1) rows), dense and sparse
clouds: every label against the oracle, the labels of the static pipeline and
with the pair lists cut to one entry."""
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


@pytest.mark.parametrize("d", range(4, 9))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("eps,spread", [(0.5, 0.1), (0.9, 0.45)])
def test_clouds(ctx, d, dtype, eps, spread):
    n = 13_001
    rng = np.random.default_rng(100 * d + int(10 * eps))
    centres = rng.uniform(0, 4, (12, d))
    x = centres[rng.integers(0, 12, n)] + rng.normal(0, spread, (n, d))
    # a dense core of one cluster: boxes of many rows beside boxes of one
    x[: n // 6] = centres[0] + rng.normal(0, spread / 6, (n // 6, d))
    far = rng.integers(0, n, n // 10)
    x[far] = rng.uniform(-1, 5, (len(far), d))
    x = x.astype(dtype)
    mp = 5
    print(f"[gpu-case] wide groups d={d} {np.dtype(dtype).name} eps={eps}", flush=True)
    got = ctx.cluster(x, eps, mp)
    r = oracle.check_parallel(x, eps, mp, got, threads=16)
    assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    try:
        c.set_open_pair_limit(1)
        np.testing.assert_array_equal(c.cluster(x, eps, mp), got)
        if d <= 6:  # (beyond, the static pipeline hands the run back)
            c.set_open_pair_limit(0)
            c.set_graph(True)
            np.testing.assert_array_equal(c.cluster(x, eps, mp), got)
    finally:
        c.close()


@pytest.mark.parametrize("d,eps", [(2, 0.06), (3, 0.4)])
def test_many_boxes(ctx, d, eps):
    """Above 250000 boxes the union looks at cells first in 2-D and 3-D too."""
    n = 700_000
    rng = np.random.default_rng(d)
    centres = rng.uniform(0, 60, (400, d))
    x = centres[rng.integers(0, 400, n)] + rng.normal(0, 1.2 if d == 2 else 0.9, (n, d))
    far = rng.integers(0, n, n // 10)
    x[far] = rng.uniform(0, 60, (len(far), d))
    x = x.astype(np.float32)
    print(f"[gpu-case] many boxes d={d}", flush=True)
    got = ctx.cluster(x, eps, 5)
    assert ctx.stats()["boxes"] > 250_000
    r = oracle.check_parallel(x, eps, 5, got, threads=16)
    assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
