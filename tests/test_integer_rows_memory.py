"""Integer rows take more workspace as float rows than on the integer path: a call
that has room for the one only must still run.  A small shared object that
counts and bounds hipMalloc stands between the library and the runtime, in a
child process."""
from __future__ import annotations

import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static size_t held, peak, budget = ~(size_t)0;
static struct { void* p; size_t n; } all[1024];

static void* real(const char* name) {
    return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), name);
}
int hipMalloc(void** p, size_t n) {
    if (n > budget || held > budget - n) return 2; /* hipErrorOutOfMemory */
    int rc = ((int (*)(void**, size_t))real("hipMalloc"))(p, n);
    if (rc != 0) return rc;
    for (int i = 0; i < 1024; ++i)
        if (!all[i].p) {
            all[i].p = *p;
            all[i].n = n;
            break;
        }
    held += n;
    if (held > peak) peak = held;
    return 0;
}
int hipFree(void* p) {
    for (int i = 0; p && i < 1024; ++i)
        if (all[i].p == p) {
            held -= all[i].n;
            all[i].p = 0;
        }
    return ((int (*)(void*))real("hipFree"))(p);
}
size_t shim_held(void) { return held; }
size_t shim_peak(void) { return peak; }
void shim_reset_peak(void) { peak = held; }
void shim_budget(size_t n) { budget = n; }
"""

CHILD = r"""
import ctypes, json, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
for f in (shim.shim_held, shim.shim_peak):
    f.restype = ctypes.c_size_t
shim.shim_budget.argtypes = [ctypes.c_size_t]
import numpy as np
from hpdbscan_amd import BORDER_ONE_THREAD, _lib
x = np.load(sys.argv[2])
out = {}

def call(name, ctx):
    shim.shim_reset_peak()
    print("[gpu-case]", name, file=sys.stderr, flush=True)
    labels = ctx.cluster(x, 30.0, 8)
    np.save(f"{sys.argv[3]}_{name}.npy", labels)
    out[name] = {"box_union": ctx.stats()["box_union"], "peak": shim.shim_peak()}

for rule in (0, BORDER_ONE_THREAD):
    ctx = _lib.Context(0)
    ctx.set_border_rule(rule)
    call(f"free{rule}", ctx)
    ctx.close()
    assert shim.shim_held() == 0
    shim.shim_budget(out[f"free{rule}"]["peak"] - 1)
    ctx = _lib.Context(0)
    ctx.set_border_rule(rule)
    call(f"tight{rule}", ctx)
    shim.shim_budget((1 << 64) - 1)
    call(f"again{rule}", ctx)
    ctx.close()
    assert shim.shim_held() == 0
print(json.dumps(out))
"""


@pytest.mark.parametrize("dtype", [np.int16, np.int32])
def test_room_for_the_integer_path_only(tmp_path, dtype):
    rng = np.random.default_rng(5)
    n, hi = 200_000, 1000
    centres = rng.uniform(0.1 * hi, 0.9 * hi, (20, 3))
    x = centres[rng.integers(0, 20, n)] + rng.normal(0, 0.02 * hi, (n, 3))
    x[::10] = rng.uniform(0, hi, (n // 10, 3))
    x = np.clip(np.round(x), 0, hi).astype(dtype)
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), "-ldl"], check=True)
    np.save(tmp_path / "x.npy", x)
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), str(tmp_path / "x.npy"),
                        str(tmp_path / "labels")], cwd=ROOT, capture_output=True, text=True,
                       timeout=100, env={**os.environ, "PYTHONPATH": ROOT})
    print(r.stderr, flush=True)
    assert r.returncode == 0, r.stderr[-2000:]
    st = json.loads(r.stdout.splitlines()[-1])
    for rule in (0, 1):
        labels = {k: np.load(tmp_path / f"labels_{k}{rule}.npy") for k in ("free", "tight", "again")}
        r = oracle.check_parallel(x, 30.0, 8, labels["free"], threads=8)
        assert r["mismatches"] == 0 and r["bad_ambiguous"] == 0
        np.testing.assert_array_equal(labels["tight"], labels["free"])
        np.testing.assert_array_equal(labels["again"], labels["free"])
        assert [st[f"{k}{rule}"]["box_union"] for k in ("free", "tight", "again")] == [1, 0, 1]
