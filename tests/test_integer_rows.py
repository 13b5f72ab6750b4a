"""Integer rows that float reproduces exactly run on boxes as float rows, the
others by the row-level union: both sides of every limit of that rule (the sum
of squares at 2^24 and at the type's largest value, the coordinates at 2^24)
against the oracle.  Which side ran shows in the run's box count."""
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


def clusters(n, d, dtype, lo, hi, sigma, seed):
    """Gaussian clusters and 10 % uniform rows of integers in [lo, hi], both
    ends taken by a row."""
    rng = np.random.default_rng(seed)
    centre = rng.uniform(lo, hi, (8, d))
    x = centre[rng.integers(0, 8, n)] + rng.normal(0, sigma, (n, d))
    noise = rng.random(n) < 0.1
    x[noise] = rng.uniform(lo, hi, (int(noise.sum()), d))
    x = np.clip(np.rint(x), lo, hi)
    x[0], x[1] = lo, hi
    return x.astype(dtype)


# (dtype, d, lo, hi, sigma, eps, runs on boxes)
CASES = [
    # 3 * (2 eps + 1)^2 around 2^24
    (np.int32, 3, -20_000, 20_000, 900, 1181.0, True),
    (np.int32, 3, -20_000, 20_000, 900, 1182.0, False),
    # coordinates and spans around 2^24
    (np.int64, 2, -(1 << 23), 1 << 23, 900, 700.0, True),
    (np.int64, 2, -(1 << 23), (1 << 23) + 1, 900, 700.0, False),
    (np.uint32, 2, (1 << 24) - 5000, 1 << 24, 60, 50.0, True),
    (np.uint32, 2, (1 << 24) - 5000, (1 << 24) + 1, 60, 50.0, False),
    # 3 * (2 eps + 1)^2 around the type's largest value
    (np.int16, 3, -1500, 1500, 40, 51.0, True),
    (np.int16, 3, -1500, 1500, 40, 52.0, False),
    (np.uint16, 3, 0, 3000, 60, 73.0, True),
    (np.uint16, 3, 0, 3000, 60, 74.0, False),
    (np.int8, 2, -100, 100, 2, 3.0, True),
    (np.int8, 2, -100, 100, 2, 3.6, False),
    (np.uint8, 1, 0, 255, 3, 7.4, True),
    # eps^2 truncates to 0: only equal rows are near
    (np.int32, 3, 0, 12, 2, 0.9, True),
    (np.uint64, 4, 0, 60, 3, 2.5, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{np.dtype(c[0]).name}-{c[1]}d-{c[5]}")
@pytest.mark.parametrize("min_points", [1, 5])
def test_against_oracle(ctx, case, min_points):
    dtype, d, lo, hi, sigma, eps, boxes = case
    x = clusters(4001, d, dtype, lo, hi, sigma, 7)
    print(f"[gpu-case] {np.dtype(dtype).name} d={d} [{lo}, {hi}] eps={eps} minPts={min_points}",
          flush=True)
    got = ctx.cluster(x, eps, min_points)
    assert (ctx.stats()["boxes"] > 0) == boxes
    mismatches, bad = oracle.check(x, eps, min_points, got)
    assert mismatches == 0 and bad == 0


def test_batch_takes_one_route(ctx):
    """One job of a batch outside the rule keeps the whole batch on the
    integer path; every job's labels equal the oracle's either way."""
    a = clusters(2500, 3, np.int32, -3000, 3000, 40, 1)
    b = clusters(3001, 3, np.int32, 0, 1 << 25, 90, 2)
    for parts, boxes in (((a, a[:700]), True), ((a, b), False)):
        x = np.concatenate(parts)
        off = np.cumsum([0, *map(len, parts)])
        got = ctx.cluster_batch(x, off, 60.0, 6)
        assert (ctx.stats()["boxes"] > 0) == boxes
        for j, rows in enumerate(parts):
            mismatches, bad = oracle.check(rows, 60.0, 6, got[off[j]:off[j + 1]])
            assert mismatches == 0 and bad == 0
