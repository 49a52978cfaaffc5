"""Device memory that runs out, without a GPU: the library's host code runs on a stand-in for the
HIP runtime (hip_stub.c) whose k-th allocation fails, for every k a call makes.  A call that
fails says so, leaves an engine without a state (no later call uses arrays that are gone or too
small), and the same engine or network takes the next."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, os, sys
import numpy as np
stub = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)    # before the library: its calls resolve here
stub.stub_fail.argtypes = [C.c_long]
stub.stub_outside.restype = stub.stub_live.restype = C.c_long
sys.path.insert(0, os.path.join(sys.argv[2], "osprey-dpd_amd"))
import dpd_amd as D
OOM, STATE = 2, 6
A, G = np.full((2, 2), 25.0), np.full((2, 2), 4.5)
rng = np.random.default_rng(1)

def state(cells, n):
    x = rng.uniform(0, 1, (n, 3)) * np.array(cells, float)
    return np.arange(1, n + 1, dtype=np.int32), np.zeros(n, np.int32), x, np.zeros((n, 3))

def code(f):
    try:
        f()
        return 0
    except D.DpdError as err:
        return err.code

def every_failure(call, after):
    # with the k-th allocation failing, k = 0, 1, ... until the call makes fewer
    k = 0
    while True:
        e = after(None)
        stub.stub_fail(k)
        rc = code(lambda: call(e))
        stub.stub_fail(-1)
        assert stub.stub_outside() == 0, (k, rc)
        if rc == 0:
            e.close()
            return k
        assert rc == OOM, (k, rc)
        assert code(lambda: e.step(2)) == STATE and code(lambda: e.slice_stress(4)) == STATE, k
        after(e)
        assert code(lambda: e.step(2)) == 0 and stub.stub_outside() == 0, k
        e.close()
        k += 1
"""

BEADS = PRELUDE + """
cells = (5, 4, 6)
for n0, n1 in ((300, 700), (700, 300)):
    def first(e):
        e = e or D.Engine(cells, A, G)
        e.upload(*state(cells, n0))
        return e
    print("allocations:", every_failure(lambda e: e.upload(*state(cells, n1)), first))
def first(e):
    e = e or D.Engine(cells, A, G)
    e.upload(*state(cells, 300))
    e.upload_topology(range(0, 99), range(1, 100), np.ones(99), np.ones(99))
    return e
n = every_failure(lambda e: e.upload_topology(range(0, 200), range(1, 201), np.ones(200), np.ones(200)), first)
print("allocations:", n)
assert n > 3
"""

BATCH = PRELUDE + """
cells = [(5, 4, 6), (3, 3, 4)]
def put(e, n):
    for b, c in enumerate(cells):
        e.upload_box(b, *state(c, n + b))
        e.upload_box_topology(b, range(0, n // 2), range(1, n // 2 + 1), np.ones(n // 2), np.ones(n // 2))
    e.commit()
def first(e):
    e = e or D.Batch([{"cells": c, "a": A, "gamma": G} for c in cells])
    put(e, 200)
    return e
n = every_failure(lambda e: put(e, 333), first)
print("allocations:", n)
assert n > 8
"""

NETWORK = PRELUDE + """
from dpd_amd.mlp import MLPError, Surrogate
X, Y = rng.normal(0, 1, (40, 7)), rng.normal(0, 1, (40, 2))
k = 0
while True:
    m = Surrogate(7, 32, 2)
    m.train(X[:20], Y[:20], iters=4)
    stub.stub_fail(k)
    try:
        m.train(X, Y, iters=9)
        done = True
    except MLPError:
        done = False
    stub.stub_fail(-1)
    # (fewer rows and iterations than the call that failed had made room for)
    m.train(X[:20], Y[:20], iters=4)
    m.gradients(X, Y)
    m.predict(X)
    assert stub.stub_outside() == 0, k
    m.close()
    if done:
        break
    k += 1
print("allocations:", k)
assert k > 10
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("stub") / "libstub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", "-o", path, os.path.join(HERE, "hip_stub.c")], check=True)
    return path


@pytest.mark.parametrize("script", [BEADS, BATCH, NETWORK], ids=["one-box", "batch", "network"])
def test_after_a_failed_call(stub, script):
    r = subprocess.run([sys.executable, "-c", script, stub, ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
