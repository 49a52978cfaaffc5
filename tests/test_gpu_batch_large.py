"""A batch of more beads than one round of wavefronts holds, with bonds and bond pairs: two beads a
thread in k_advance, which adds the bonded sums, in boxes whose border lies within a thread's pair
of beads and a workgroup.  Against the FP64 oracle, and the uploaded state's layout repeated."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import chain_state, force_errors

pytestmark = pytest.mark.gpu
A3 = np.array([[25.0, 30.0, 35.0], [30.0, 10.0, 25.0], [35.0, 25.0, 40.0]])
G3 = np.full((3, 3), 4.5)


@pytest.mark.parametrize("kernel", [D.PAIR_HITLIST, D.PAIR_FULLSHELL], ids=["hitlist", "fullshell"])
def test_steps_match_the_oracle(kernel):
    specs = [((40, 41, 42), 207001), ((47, 46, 45), 292010), ((20, 21, 22), 27719)]
    assert sum(n for _, n in specs) > 8192 * 64
    e = D.Batch([{"cells": c, "a": A3, "gamma": G3, "seed": 5 + b} for b, (c, _) in enumerate(specs)], pair_kernel=kernel)
    ref, first = [], []
    for b, (cells, n) in enumerate(specs):
        nch = n // 50
        ids, t, x, u, v, (h, tl, fi, se) = chain_state(cells, nch, 10, n - 10 * nch, seed=b)
        topo = (h, tl, np.full(len(h), 128.0), np.full(len(h), 0.4), fi, se, np.full(len(fi), 20.0), np.zeros(len(fi)))
        box = O.Box(cells, A3, G3, seed=5 + b, rng_mode=O.RNG_PHILOX)
        f0, _, _ = O.forces(box, ids, t, x, v, step=0, unpbc=u, topo=O.Topo(*topo))
        e.upload_box(b, ids, t, x, v, f=f0, unpbc=u)
        e.upload_box_topology(b, *topo)
        ref.append(O.System(box, ids, t, x, v, f0, unpbc=u, topo=O.Topo(*topo)))
        first.append((ids, t, topo))
    e.commit()
    print("large batch", e.n, kernel, flush=True)
    e.step(3, observe=True)
    states = []
    for b, s in enumerate(ref):
        s.run(3, step0=0)
        X, U, V, F = e.download_box(b)
        states.append((X, U, V, F))
        xr, ur, vr, fr = s.state()
        norm, _ = force_errors(F, fr)
        print(f"  box {b}: {norm:.2e}, |u - u_ref| max {np.abs(U - ur).max():.1e}", flush=True)
        assert norm < 1e-5 and np.abs(U - ur).max() < 1e-5
        assert abs(e.observables(b)["kT"] - (vr * vr).sum() / vr.size) < 1e-5
    f = e.compute_forces(step=7, thermostat=False)[0]
    for b, (ids, t, topo) in enumerate(first):
        X, U, V, F = states[b]
        e.upload_box(b, ids, t, X, V, f=F, unpbc=U)
        e.upload_box_topology(b, *topo)
    e.commit(3)
    # the conservative forces of the same state: positions are FP32 offsets in their cells and
    # come back the same
    assert np.array_equal(f, e.compute_forces(step=7, thermostat=False)[0])
