"""Clusters whose boxes hang together in long chains (1023 to 5000 boxes in a
line, alone and several interleaved in sort order): one cluster per line,
against the oracle, in both pipelines."""
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


@pytest.mark.parametrize("boxes", [1023, 1024, 1025, 5000])
@pytest.mark.parametrize("d,lines", [(1, 1), (2, 1), (2, 3), (3, 3)])
def test_lines(ctx, boxes, d, lines):
    rng = np.random.default_rng(boxes + d)
    # four rows in every half of a unit cell along the first axis, lines 7 apart
    at = np.repeat(np.arange(boxes) * 0.5, 4) + rng.uniform(0.05, 0.45, 4 * boxes)
    parts = []
    for k in range(lines):
        x = rng.uniform(0.0, 0.2, (len(at), d))
        x[:, 0] = at
        if d > 1:
            x[:, 1] += 7.0 * k
        parts.append(x)
    x = np.concatenate(parts)
    x = x[rng.permutation(len(x))].astype(np.float32)
    print(f"[gpu-case] {lines} lines of {boxes} boxes, d={d}", flush=True)
    got = ctx.cluster(x, 1.0, 4)
    mismatches, bad = oracle.check(x, 1.0, 4, got)
    assert mismatches == 0 and bad == 0
    assert len(np.unique(np.abs(got))) == lines
    from hpdbscan_amd import _lib
    c = _lib.Context(0)
    try:
        c.set_graph(True)
        for _ in range(2):
            np.testing.assert_array_equal(c.cluster(x, 1.0, 4), got)
    finally:
        c.close()
