"""The counting sort of engines with dense cells (wide cells, or many beads in few), whose beads
are moved by slots rather than by groups of 64 cells: cells that reach over several workgroups'
256 slots and over the 1,024 counted at a time, a last workgroup of one slot, empty cells between
full ones, beads that gather past the room of their cell's bin, and a batch with bonds.  And a
group of more than 1,024 beads in an engine that is not dense, whose workgroup moves them alone.
The state reached is uploaded again: the layout is a function of the state, so the forces
are the same to the bit, and they match the FP64 oracle."""
import time

import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import chain_state, force_errors, random_state

pytestmark = pytest.mark.gpu
# weak forces and no thermostat: beads fly straight
A2 = np.array([[0.02, 0.03], [0.03, 0.02]])
G2 = np.zeros((2, 2))
DT = 0.02
# cells, width, beads, share of the box's x axis that holds them, gathering at step
STATES = [((3, 3, 3), 1.0, 1025, 1.0, 0), ((4, 4, 4), 2.0, 1536, 1.0, 0), ((5, 5, 5), 1.75, 4097, 1.0, 0),
          ((3, 4, 7), 3.0, 6805, 1.0, 0), ((7, 3, 3), 4.0, 9000, 0.4, 0), ((4, 4, 4), 1.0, 3000, 0.25, 1),
          ((4, 4, 4), 1.0, 3000, 1.0, 2), ((9, 8, 8), 1.0, 2900, 0.2, 0)]


@pytest.mark.parametrize("kernel", [D.PAIR_FULLSHELL, D.PAIR_HITLIST], ids=["fullshell", "hitlist"])
@pytest.mark.parametrize("cells,w,n,part,gather", STATES,
                         ids=["x".join(map(str, c)) + f"-w{w}-{n}-{p}-{g}" for c, w, n, p, g in STATES])
def test_layout_and_forces(cells, w, n, part, gather, kernel):
    print("dense", cells, w, n, part, gather, kernel, flush=True)
    widths = (w, w, w)
    ids, t, x, v = random_state(cells, n, 2, seed=n + gather, widths=widths, kT=0.25)
    L = np.array(cells) * w
    x[:, 0] *= part
    if gather:
        # beads less than `gather` cells from the target fly into it in that many steps
        rng = np.random.default_rng(n)
        goal = np.array([1.0, 2.0, 1.0]) + rng.uniform(0.3, 0.7, (n, 3))
        d = (goal - x + L / 2) % L - L / 2
        near = np.abs(d).max(axis=1) < gather
        v[near] = d[near] / (gather * DT)
    e = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=kernel, widths=widths)
    e.upload(ids, t, x, v)
    e.step(3)
    X, U, V, _ = e.download()
    assert (X >= 0).all() and (X < L).all()
    # (the forces of a cell of thousands move a bead by 0.1 at most)
    off = (X - x - 3 * DT * v + L / 2) % L - L / 2
    assert np.abs(off).max() < 0.1
    f, vir, _ = e.compute_forces(step=7, thermostat=False)
    fresh = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=kernel, widths=widths)
    fresh.upload(ids, t, X, V, unpbc=U)
    assert np.array_equal(f, fresh.compute_forces(step=7, thermostat=False)[0])
    fr, virr, _ = O.forces(O.Box(cells, A2, G2, seed=3, widths=widths), ids, t, X, V, step=7, thermostat=False)
    # FP32 sums of up to some hundred terms: a few hundred 2^-24 of the largest partial sum
    assert force_errors(f, fr)[0] < 2e-5
    assert np.linalg.norm(vir - virr) < 2e-5 * np.linalg.norm(virr)


def test_batch_with_bonds():
    """Boxes of wide cells and uneven sizes with chains and bond pairs, against the oracle."""
    a = np.array([[25.0, 30.0, 35.0], [30.0, 10.0, 25.0], [35.0, 25.0, 40.0]])
    g = np.full((3, 3), 4.5)
    specs = [((4, 4, 4), (2.0, 2.0, 2.0)), ((3, 5, 4), (3.0, 2.0, 2.0)), ((3, 3, 3), (3.0, 3.0, 3.0))]
    e = D.Batch([{"cells": c, "a": a, "gamma": g, "seed": 5 + b, "widths": w} for b, (c, w) in enumerate(specs)])
    ref = []
    for b, (c, w) in enumerate(specs):
        size = tuple(int(p * q) for p, q in zip(c, w))
        n = 3 * int(np.prod(size))
        ids, t, x, u, v, (h, tl, fi, se) = chain_state(size, n // 40, 10, n - 10 * (n // 40), seed=b)
        topo = (h, tl, np.full(len(h), 128.0), np.full(len(h), 0.4), fi, se, np.full(len(fi), 20.0), np.zeros(len(fi)))
        box = O.Box(c, a, g, seed=5 + b, widths=w, rng_mode=O.RNG_PHILOX)
        f0, _, _ = O.forces(box, ids, t, x, v, step=0, unpbc=u, topo=O.Topo(*topo))
        e.upload_box(b, ids, t, x, v, f=f0, unpbc=u)
        e.upload_box_topology(b, *topo)
        ref.append(O.System(box, ids, t, x, v, f0, unpbc=u, topo=O.Topo(*topo)))
    e.commit()
    e.step(5)
    for b, s in enumerate(ref):
        s.run(5, step0=0)
        X, U, V, F = e.download_box(b)
        xr, ur, vr, fr = s.state()
        norm, _ = force_errors(F, fr)
        print(f"  box {b}: {norm:.2e}, |u - u_ref| max {np.abs(U - ur).max():.1e}", flush=True)
        assert norm < 1e-5 and np.abs(U - ur).max() < 1e-5


def test_sort_is_a_small_part_of_a_step():
    """41,472 beads in 27 cells: a step costs little beyond its pair launch (2 to 4 ms here), as
    in boxes of unit cells, whose sort takes some 5 us.  A hundred times that is allowed."""
    cells, w = (3, 3, 3), 8.0
    n = 3 * 24 ** 3
    ids, t, x, v = random_state(cells, n, 1, seed=1, widths=(w, w, w))
    e = D.Engine(cells, np.array([[1.0]]), np.array([[4.5]]), dt=0.01, seed=3, widths=(w, w, w))
    e.upload(ids, t, x, v)
    e.step(20, graph=True)
    pair = min(e.time_pair(10) for _ in range(3))
    step = []
    for _ in range(3):
        t0 = time.perf_counter()
        e.step(20, graph=True)
        step.append((time.perf_counter() - t0) / 20 * 1e3)
    print(f"  step {min(step):.3f} ms, pair launch {pair:.3f} ms", flush=True)
    assert min(step) - pair < 0.5
