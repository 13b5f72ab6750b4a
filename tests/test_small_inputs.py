"""Small inputs are clustered by comparing all pairs of rows, others (and every
run with timing on) through the sort and the index: both give the same labels
and the same counts, at the sizes around a wave, a block and the limit, and the
oracle's labels."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SAME = ("total_cells", "key_bits", "occupied_cells", "boxes", "neighbor_rows", "sum_candidates",
        "core_points", "noise_points", "ambiguous_borders")


@pytest.fixture(scope="module")
def contexts():
    from hpdbscan_amd import BORDER_ONE_THREAD, _lib
    small, general, one_thread = _lib.Context(0), _lib.Context(0), _lib.Context(0)
    general.set_timing(True)  # the general path whatever the size
    one_thread.set_border_rule(BORDER_ONE_THREAD)
    yield small, general, one_thread
    for c in (small, general, one_thread):
        c.close()


def cloud(n, d, dtype, seed, spread=1.0):
    rng = np.random.default_rng(seed)
    k = max(1, n // 150)
    centre = rng.uniform(-4, 4, (k, d)) * spread
    x = centre[rng.integers(0, k, n)] + rng.normal(0, 0.25, (n, d))
    noise = rng.random(n) < 0.15
    x[noise] = rng.uniform(-4, 4, (int(noise.sum()), d)) * spread
    return x.astype(dtype)


def check(contexts, x, eps, mp, what):
    small, general, one_thread = contexts
    print(f"[gpu-case] {what} n={len(x)} d={x.shape[1]} {x.dtype} eps={eps} minPts={mp}", flush=True)
    got = small.cluster(x, eps, mp)
    s = small.stats()
    np.testing.assert_array_equal(got, general.cluster(x, eps, mp))
    g = general.stats()
    assert {k: s[k] for k in SAME} == {k: g[k] for k in SAME}
    want = oracle.cluster(x, eps, mp)
    mismatches, bad = oracle.check(x, eps, mp, got)
    assert mismatches == 0 and bad == 0
    np.testing.assert_array_equal(one_thread.cluster(x, eps, mp), want)


@pytest.mark.parametrize("d", range(1, 9))
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 257, 4096, 6000, 6001])
def test_sizes(contexts, n, d, dtype):
    check(contexts, cloud(n, d, dtype, 100 * d + n), 0.2 + 0.1 * d, 5, "small")


@pytest.mark.parametrize("d,n", [(5, 12000), (6, 12001)])
def test_sizes_from_five_dimensions(contexts, n, d):
    check(contexts, cloud(n, d, np.float32, d), 0.6, 5, "small, 5-D and above")


@pytest.mark.parametrize("min_points", [0, 1, 2, 4000])
def test_min_points(contexts, min_points):
    check(contexts, cloud(3000, 3, np.float32, 1), 0.4, min_points, "small minPts")


@pytest.mark.parametrize("d", [1, 2, 3])
def test_duplicates_one_cell_and_negative(contexts, d):
    """Equal rows, all rows in one cell, rows that are all negative (the
    reference's maximum starts at the smallest positive value)."""
    rng = np.random.default_rng(d)
    x = rng.integers(-3, 4, (2000, d)).astype(np.float32)
    check(contexts, x, 1.0, 20, "duplicates")
    check(contexts, (x * np.float32(0.01)), 5.0, 20, "one cell")
    check(contexts, -cloud(1000, d, np.float64, 3) ** 2 - 1.0, 0.3, 5, "negative")


def test_grids_near_and_over_the_limits(contexts):
    """A dimension of 2^31 cells or more runs through the general path, a grid
    of more than 2^64 cells is refused, non-finite rows raise."""
    small, general, _ = contexts
    x = cloud(500, 2, np.float64, 5)
    x[0] = 0.0
    x[1] = (1.0e9, 1.0)
    check(contexts, x, 0.3, 3, "2^32 cells in one dimension")
    x[1] = 1.0e15
    for c in (small, general):
        with pytest.raises(NotImplementedError):
            c.cluster(np.concatenate([x, x, x], axis=1), 1e-3, 3)
    x[2, 1] = np.nan
    for c in (small, general):
        with pytest.raises(ValueError):
            c.cluster(x, 0.3, 3)


def test_replayed_with_new_data_and_parameters(contexts):
    """Graph mode captures the all-pairs kernels: replays with other rows, eps
    and minPts in the same buffers, other work in between."""
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    n, d = 2111, 3
    xd, ld = _lib.DeviceBuffer(c, 4 * n * d), _lib.DeviceBuffer(c, 8 * n)
    try:
        c.set_graph(True)
        for i in range(5):
            x = cloud(n, d, np.float32, 50 + i)
            eps, mp = 0.3 + 0.05 * i, 4 + i
            xd.copy_from(x)
            c.cluster_device(xd.ptr, n, d, np.float32, eps, mp, ld.ptr)
            np.testing.assert_array_equal(ld.to_array(np.int64, n), contexts[1].cluster(x, eps, mp))
            contexts[0].cluster(x[: 900 + i], eps, mp)
        assert c.graph_stats() == {"launches": 5, "captures": 1, "fallbacks": 0}
    finally:
        xd.close()
        ld.close()
        c.close()
