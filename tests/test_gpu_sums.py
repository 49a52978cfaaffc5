"""Observables of batches whose boxes share wavefronts (down to seven beads a box, so that one
holds ten boxes), with one and with sixteen rows of accumulators a box (16 boxes and 17):
every box against an engine of its own, twice in a row, since a call leaves the accumulators
clear for the next."""
import numpy as np
import pytest

import dpd_amd as D
from helpers import random_state

pytestmark = pytest.mark.gpu
A2 = np.array([[25.0, 40.0], [40.0, 25.0]])
G2 = np.full((2, 2), 4.5)


@pytest.mark.parametrize("nbox", [1, 16, 17, 70])
@pytest.mark.parametrize("kernel", [D.PAIR_FULLSHELL, D.PAIR_HITLIST], ids=["fullshell", "hitlist"])
def test_observables_of_small_boxes(nbox, kernel):
    print("sums", nbox, kernel, flush=True)
    rng = np.random.default_rng(nbox)
    specs, states = [], []
    for i in range(nbox):
        cells = tuple(int(c) for c in rng.integers(3, 6, 3))
        n = int(rng.choice([7, 20, 64, 150, 300]))
        specs.append({"cells": cells, "a": A2, "gamma": G2, "seed": 40 + i, "dt": 0.01, "ntypes": 2})
        ids, t, x, v = random_state(cells, n, 2, seed=i)
        states.append((ids, t, x, v))
    # beads 0, 1 and 2 of every other box are a chain
    def chain(x, L):
        d = np.array([[0, 0, 0], [0.4, 0.1, 0], [0.5, 0.5, 0.2]])
        u = x.copy()
        u[:3] = u[0] + d
        x = np.mod(u, L)
        x[x >= L] = 0.0
        return x, u
    topo = ([0, 1], [1, 2], [90.0, 70.0], [0.4, 0.5], [1], [0], [15.0], [0.3])
    batch = D.Batch(specs, pair_kernel=kernel)
    singles = []
    for i, (s, (ids, t, x, v)) in enumerate(zip(specs, states)):
        x, u = chain(x, np.array(s["cells"], float))
        batch.upload_box(i, ids, t, x, v, unpbc=u)
        e = D.Engine(s["cells"], A2, G2, seed=s["seed"], dt=s["dt"], pair_kernel=kernel)
        e.upload(ids, t, x, v, unpbc=u)
        if i % 2 == 0:
            batch.upload_box_topology(i, *topo)
            e.upload_topology(*topo)
        singles.append(e)
    batch.commit(step0=0)
    for steps in (1, 4):
        batch.step(steps, observe=True)
        for i, e in enumerate(singles):
            e.step(steps, observe=True)
            a, b = batch.observables(i), e.observables()
            # the same terms but for the order of FP32 sums, whose rounding (1e-6 of a force) is that of
            # ten times the net stress at most; one bead or pair too few or too many is 3e-3 or more
            near = lambda p, q, scale: np.all(np.abs(np.asarray(p) - q) <= 1e-4 * scale)
            size = np.sqrt(len(states[i][0]) * b["sum_v2"].sum())   # of the largest momentum there could be
            assert near(a["kT"], b["kT"], b["kT"]) and near(a["sum_v2"], b["sum_v2"], b["sum_v2"].sum())
            assert near(a["momentum"], b["momentum"], size)
            assert near(a["stress"], b["stress"], np.abs(b["stress"]).max())
            assert near(a["pressure"], b["pressure"], max(abs(b["pressure"]), np.abs(b["stress"]).max()))
            assert near(a["pe"], b["pe"], b["pe"].sum())
