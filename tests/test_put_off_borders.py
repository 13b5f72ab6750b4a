"""Border rows next to boxes of more than 16384 rows of two clusters, whose walks
are put off and run by several waves: the rule by which such a wave leaves its
walk out, over every interleaving of the waves' steps (on the CPU, the
library's own expression), and the labels and the number of ambiguous rows
under both border rules against the oracle."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

import oracle
from conftest import ROOT

CSRC = os.path.join(ROOT, "hpdbscan_amd", "csrc")

# Waves of one row: read one word, read the other, decide, publish into one
# word, publish into the other.  Every order of the reads and of the
# publications, every interleaving, every starting state that a walk in place
# can leave, hits and misses.
MODEL = r"""
#include <algorithm>
#include <array>
#include <climits>
#include <cstdio>
#include <vector>
#include "put_off.hpp"

struct Wave { int cl; bool hit, min_read_first, min_put_first; };
struct State { int best, worst; };
struct Local { int step = 0, best = 0, worst = 0; };
static long runs = 0, wrong = 0;

static bool step(const Wave& w, Local& l, State& s) {  // false: the wave is done
    switch (l.step++) {
        case 0: (w.min_read_first ? l.best : l.worst) = w.min_read_first ? s.best : s.worst; return true;
        case 1:
            (w.min_read_first ? l.worst : l.best) = w.min_read_first ? s.worst : s.best;
            return !hpd::cluster_settled(l.best, l.worst, w.cl) && w.hit;
        case 2:
            if (w.min_put_first) s.best = std::min(s.best, w.cl);
            else s.worst = std::max(s.worst, w.cl);
            return true;
        default:
            if (w.min_put_first) s.worst = std::max(s.worst, w.cl);
            else s.best = std::min(s.best, w.cl);
            return false;
    }
}

static void go(const std::vector<Wave>& w, std::array<Local, 3> l, State s, unsigned on, State want) {
    bool any = false;
    for (size_t i = 0; i < w.size(); ++i) {
        if (!(on >> i & 1)) continue;
        any = true;
        std::array<Local, 3> l2 = l;
        State s2 = s;
        const bool more = step(w[i], l2[i], s2);
        go(w, l2, s2, more ? on : on & ~(1u << i), want);
    }
    if (any) return;
    ++runs;
    // the label is the smallest cluster, the row is ambiguous with two of them
    if (s.best != want.best || (s.best != s.worst) != (want.best != want.worst)) ++wrong;
}

int main() {
    const State starts[] = {{INT_MAX, -1}, {5, 5}, {4, 6}};
    for (const State s : starts)
        for (int n = 2; n <= 3; ++n)
            for (int code = 0; code < (n == 2 ? 32 * 32 : 8 * 8 * 8); ++code) {
                std::vector<Wave> w;
                int c = code;
                for (int i = 0; i < n; ++i) {
                    const int k = n == 2 ? c % 32 : c % 8;
                    c /= n == 2 ? 32 : 8;
                    // (three waves: hits, published in the kernel's order)
                    if (n == 2) w.push_back({3 + 2 * (k & 3), (k & 4) != 0, (k & 8) != 0, (k & 16) != 0});
                    else w.push_back({3 + 2 * (k & 3), true, (k & 4) != 0, true});
                }
                State want = s;
                for (const Wave& x : w)
                    if (x.hit) want = {std::min(want.best, x.cl), std::max(want.worst, x.cl)};
                go(w, {}, s, (1u << n) - 1, want);
            }
    std::printf("%ld %ld\n", runs, wrong);
    return 0;
}
"""


def test_no_interleaving_loses_a_cluster(tmp_path):
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    runs, wrong = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                          text=True).stdout.split())
    assert runs > 1_000_000
    assert wrong == 0


EPS = 1.0
MIN_POINTS = 500


def two_crowds(d, dtype, seed):
    """Two crowds of 20000 and 17000 rows, each in one sub-box (eps / 2 wide),
    1.5 eps apart, with only 40 rows of either within eps of the 400 rows
    between them.  An arm of smaller crowds joins the second one from a
    later cell but starts in an earlier one than both, so that the second
    crowd's cluster is the smaller id, while at one thread the first crowd's
    rows carry the smaller provisional label.  Returns the rows (input order)
    and a mask of those between the crowds."""
    rng = np.random.default_rng(seed)

    def block(n, lo, hi):
        # the dimensions beyond the second stay in one sub-box of the grid
        rows = np.concatenate([np.asarray(lo, float), np.zeros(d - 2)])
        size = np.concatenate([np.asarray(hi, float) - lo, np.full(d - 2, 0.02)])
        return rows + size * rng.random((n, d))

    # (a corner row makes the grid start at (-1, -1, 0 ...): cells and
    # sub-boxes begin at whole and half numbers)
    first = np.concatenate([block(19_960, (0.01, 3.2), (0.08, 3.3)),
                            block(40, (0.40, 3.2), (0.44, 3.3))])
    second = np.concatenate([block(16_960, (2.43, 3.2), (2.48, 3.3)),
                             block(40, (2.03, 3.2), (2.06, 3.3))])
    between = block(400, (1.12, 2.9), (1.40, 3.6))
    path = [(4.2, 0.2 + 0.4 * k) for k in range(11)] + [(3.8 - 0.4 * k, 4.2) for k in range(4)]
    arm = [block(700, p, (p[0] + 0.05, p[1] + 0.05)) for p in path]
    corner = np.concatenate([[-1.0, -1.0], np.zeros(d - 2)])[None, :]
    x = np.concatenate([first, second, between, *arm, corner])
    mid = np.zeros(len(x), bool)
    mid[37_000:37_400] = True
    order = rng.permutation(len(x))
    return np.ascontiguousarray(x[order].astype(dtype)), mid[order]


@pytest.fixture(scope="module")
def crowds():
    kept = {}

    def get(d, dtype):
        key = (d, np.dtype(dtype).name)
        if key not in kept:
            x, mid = two_crowds(d, dtype, 17 + d)
            kept[key] = (x, mid, oracle.cluster(x, EPS, MIN_POINTS, full=True))
        return kept[key]

    return get


CASES = [(2, np.float32), (3, np.float32), (2, np.float64)]


def min_rule(r, x):
    """Labels under the smallest-cluster rule from the oracle's: an ambiguous row
    takes the smallest cluster among the cores within eps."""
    want = r["labels"].copy()
    cores = np.flatnonzero(r["core"])
    xc, lc = x[cores].astype(np.float64), -want[cores]
    for i in np.flatnonzero(r["ambiguous"]):
        d2 = ((xc - x[i].astype(np.float64)) ** 2).sum(axis=1)
        assert np.abs(d2 - EPS * EPS).min() > 1e-6  # no doubt in any rounding
        want[i] = lc[d2 <= EPS * EPS].min()
    return want


@pytest.mark.parametrize("d,dtype", CASES)
def test_crowds_are_what_they_are_meant_to_be(crowds, d, dtype):
    """Two boxes above 16384 rows, border rows next to both, and a label that
    the two rules choose differently."""
    x, mid, r = crowds(d, dtype)
    box = np.floor((x.astype(np.float64) - x.min(axis=0)) / (EPS / 2)).astype(int)
    _, counts = np.unique(box, axis=0, return_counts=True)
    assert sorted(counts[counts > 16_384]) == [17_000, 20_000]
    assert not r["core"][mid].any()
    assert r["ambiguous"][mid].sum() > 100 and not r["ambiguous"][~mid].any()
    assert (min_rule(r, x) != r["labels"]).sum() > 100


@pytest.mark.gpu
@pytest.mark.parametrize("d,dtype", CASES)
@pytest.mark.parametrize("rule", ["min", "one_thread"])
def test_put_off_borders_of_two_clusters(crowds, d, dtype, rule):
    from hpdbscan_amd import BORDER_MIN_CLUSTER, BORDER_ONE_THREAD, _lib
    x, mid, r = crowds(d, dtype)
    want = r["labels"] if rule == "one_thread" else min_rule(r, x)
    ctx = _lib.Context(0)
    try:
        ctx.set_border_rule(BORDER_ONE_THREAD if rule == "one_thread" else BORDER_MIN_CLUSTER)
        for k in range(3):
            print(f"[gpu-case] two crowds d={d} {np.dtype(dtype).name} rule={rule} run {k}",
                  flush=True)
            np.testing.assert_array_equal(ctx.cluster(x, EPS, MIN_POINTS), want)
            st = ctx.stats()
            assert st["ambiguous_borders"] == int(r["ambiguous"].sum())
            assert st["core_points"] == int(r["core"].sum())
            assert st["noise_points"] == int((want == 0).sum())
    finally:
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("limit", [1, 2, 5, 101])
@pytest.mark.parametrize("d,dtype", CASES)
def test_lists_that_overflow(crowds, d, dtype, limit):
    """The lists of put-off walks cut short: walks in place (1 holds no box of
    two parts), partly filled ranges, and rows with one crowd's walk put off and
    the other's in place, in the core count and in the border pass."""
    from hpdbscan_amd import BORDER_ONE_THREAD, _lib
    x, _, r = crowds(d, dtype)
    ctx = _lib.Context(0)
    try:
        ctx.set_open_pair_limit(limit)
        for rule, want in ((0, min_rule(r, x)), (BORDER_ONE_THREAD, r["labels"])):
            print(f"[gpu-case] two crowds d={d} {np.dtype(dtype).name} limit={limit} rule={rule}",
                  flush=True)
            ctx.set_border_rule(rule)
            np.testing.assert_array_equal(ctx.cluster(x, EPS, MIN_POINTS), want)
            st = ctx.stats()
            assert st["ambiguous_borders"] == int(r["ambiguous"].sum())
            assert st["core_points"] == int(r["core"].sum())
    finally:
        ctx.close()
