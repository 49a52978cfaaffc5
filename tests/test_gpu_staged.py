"""A batch goes on with what was committed while other boxes are staged: downloads, observables,
stress tables and energies are those of the committed state, with more and with fewer beads, bonds
and bond pairs staged than the device holds, until the next commit."""
import numpy as np
import pytest

import dpd_amd as D
from helpers import chain_state

pytestmark = pytest.mark.gpu
A3 = np.array([[25.0, 30.0, 35.0], [30.0, 10.0, 25.0], [35.0, 25.0, 40.0]])
G3 = np.full((3, 3), 4.5)
CELLS = [(6, 7, 8), (8, 6, 7), (5, 6, 6)]


def put(e, share, seed):
    for b, c in enumerate(CELLS):
        n = int(3 * np.prod(c) * share)
        ids, t, x, u, v, (h, tl, fi, se) = chain_state(c, n // 40, 10, n - 10 * (n // 40), seed=seed + b)
        e.upload_box(b, ids, t, x, v, unpbc=u)
        e.upload_box_topology(b, h, tl, np.full(len(h), 128.0), np.full(len(h), 0.4), fi, se, np.full(len(fi), 20.0),
                              np.zeros(len(fi)))


def seen(e):
    out = []
    for b in range(len(CELLS)):
        pair, bond = e.slice_stress(9, box=b)
        out += [*e.download_box(b), pair, bond, e.slice_stress_bondpairs(9, box=b), e.energy_output(b)]
    return out


@pytest.mark.parametrize("share", [1.5, 0.5])
def test_staged_boxes_take_effect_at_the_commit(share):
    e = D.Batch([{"cells": c, "a": A3, "gamma": G3, "seed": 3 + b} for b, c in enumerate(CELLS)])
    put(e, 1.0, 1)
    e.commit()
    e.step(3, observe=True)
    obs, n = e.observables(1), e.n
    before = seen(e)
    put(e, share, 50)
    print("staged", share, flush=True)
    after = seen(e)
    assert e.n == n and e.observables(1)["nbeads"] == obs["nbeads"] == len(before[8])
    for a, b in zip(before, after):
        # (tables and energies are sums of FP64 atomics, in any order)
        assert a.shape == b.shape and np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(a)
    e.step(2, observe=True)
    assert e.observables(1)["nbeads"] == obs["nbeads"]
    e.commit()
    assert e.n != n
    fresh = D.Batch([{"cells": c, "a": A3, "gamma": G3, "seed": 3 + b} for b, c in enumerate(CELLS)])
    put(fresh, share, 50)
    fresh.commit()
    for a, b in zip(seen(e), seen(fresh)):
        assert a.shape == b.shape and np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(a)
