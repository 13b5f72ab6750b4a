"""Batches around the edges of the 64-way search of the job table: 1 to 4097
jobs of ragged sizes, empty ones between them, rows of many jobs in one wave;
every job's labels against those of a call of its own, and the whole batch
through the static pipeline."""
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


@pytest.mark.parametrize("njobs", [1, 2, 63, 64, 65, 4096, 4097])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_job_counts(ctx, njobs, dtype):
    rng = np.random.default_rng(njobs)
    sizes = rng.integers(0, 40, njobs)
    sizes[rng.integers(0, njobs, njobs // 8)] = 0
    sizes[rng.integers(0, njobs, min(njobs, 3))] = 3000
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(off[-1])
    x = rng.uniform(0, 40, (n, 2)) + rng.integers(0, 3, (n, 1)) * 30
    x = np.round(x).astype(dtype) if np.issubdtype(dtype, np.integer) else x.astype(dtype)
    eps = rng.uniform(1.5, 4.0, njobs).astype(np.float32)
    mp = rng.integers(2, 8, njobs).astype(np.uint64)
    print(f"[gpu-case] {njobs} jobs, {n} rows of {np.dtype(dtype).name}", flush=True)
    got = ctx.cluster_batch(x, off, eps, mp)
    for j in np.unique(np.concatenate([np.arange(min(njobs, 70)),
                                       np.arange(max(0, njobs - 70), njobs),
                                       np.flatnonzero(sizes == 3000)])):
        a, b = off[j], off[j + 1]
        if a == b:
            continue
        mismatches, bad = oracle.check(x[a:b], float(eps[j]), int(mp[j]), got[a:b])
        assert mismatches == 0 and bad == 0, f"job {j}"
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    try:
        c.set_graph(True)
        np.testing.assert_array_equal(c.cluster_batch(x, off, eps, mp), got)
    finally:
        c.close()
