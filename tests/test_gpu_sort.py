"""The counting sort where it can go wrong: a group of 64 cell keys with one bead, with more
than the 256 that move at once and with more than the 1,024 whose order is found in LDS, box
sizes with a ragged last group, and beads that gather in one cell, past the room of its bin,
in the first step (filed by k_advance) and in the second (filed by the pair launch or by
k_advance).  The state reached is uploaded again: the layout is a function of the state, so
the conservative forces are the same to the bit, and they match the FP64 oracle."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import force_errors, random_state

pytestmark = pytest.mark.gpu
# weak forces and no thermostat: beads fly straight
A2 = np.array([[0.02, 0.03], [0.03, 0.02]])
G2 = np.zeros((2, 2))
DT = 0.02
# cells, beads, gathering at step
STATES = [((4, 4, 4), 1, 0), ((3, 3, 7), 190, 0), ((5, 5, 5), 530, 0), ((4, 4, 4), 1025, 0), ((8, 4, 4), 4000, 0),
          ((6, 5, 7), 630, 1), ((6, 5, 7), 630, 2), ((4, 5, 4), 2400, 1), ((4, 5, 4), 2400, 2)]


@pytest.mark.parametrize("kernel", [D.PAIR_FULLSHELL, D.PAIR_HITLIST], ids=["fullshell", "hitlist"])
@pytest.mark.parametrize("cells,n,gather", STATES, ids=["x".join(map(str, c)) + f"-{n}-{g}" for c, n, g in STATES])
def test_layout_and_forces(cells, n, gather, kernel):
    print("sort", cells, n, gather, kernel, flush=True)
    ids, t, x, v = random_state(cells, n, 2, seed=n + gather)
    L = np.array(cells, dtype=float)
    if gather:
        # beads less than `gather` cells from the target fly into it in that many steps
        rng = np.random.default_rng(n)
        goal = np.array([1.0, 2.0, 1.0]) + rng.uniform(0.3, 0.7, (n, 3))
        d = (goal - x + L / 2) % L - L / 2
        near = np.abs(d).max(axis=1) < gather
        v[near] = d[near] / (gather * DT)
    e = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=kernel)
    e.upload(ids, t, x, v)
    e.step(3)
    X, U, V, _ = e.download()
    assert (X >= 0).all() and (X < L).all()
    if gather:   # (the forces of a cell of thousands move a bead by 0.1 at most)
        off = (X - x - 3 * DT * v + L / 2) % L - L / 2
        assert np.abs(off).max() < 0.1
    f, vir, _ = e.compute_forces(step=7, thermostat=False)
    fresh = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=kernel)
    fresh.upload(ids, t, X, V, unpbc=U)
    assert np.array_equal(f, fresh.compute_forces(step=7, thermostat=False)[0])
    fr, virr, _ = O.forces(O.Box(cells, A2, G2, seed=3), ids, t, X, V, step=7, thermostat=False)
    # FP32 sums of up to some hundred terms: a few hundred 2^-24 of the largest partial sum
    if n > 1:
        assert force_errors(f, fr)[0] < 2e-5
        assert np.linalg.norm(vir - virr) < 2e-5 * np.linalg.norm(virr)


def test_graphs_after_an_odd_number_of_steps():
    """A captured sequence holds the buffers it was captured with: after an odd number of
    steps the state lies in the other ones."""
    cells, n = (7, 6, 9), 1134
    ids, t, x, v = random_state(cells, n, 2, seed=2)
    out = []
    for graph in (True, False):
        e = D.Engine(cells, A2 * 1000, G2 + 4.5, dt=DT, seed=3, pair_kernel=D.PAIR_HITLIST)
        e.upload(ids, t, x, v)
        for k in (3, 2, 4, 5, 2, 4):
            e.step(k, graph=graph)
        out.append(e.download())
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [8192 * 64, 8192 * 64 + 1, 8192 * 64 + 257])
def test_two_beads_a_thread(n):
    """Engines of more beads than the chip's wavefronts hold take two beads a thread in
    k_advance (every step's, with the full-shell kernel): at the line and one bead and one
    workgroup past it."""
    cells = (64, 56, 52)
    print("two beads", n, flush=True)
    ids, t, x, v = random_state(cells, n, 2, seed=n)
    L = np.array(cells, dtype=float)
    e = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=D.PAIR_FULLSHELL)
    e.upload(ids, t, x, v)
    e.step(3)
    X, U, V, _ = e.download()
    # weak forces: three steps of free flight but for some 1e-3 of a cell
    off = (X - x - 3 * DT * v + L / 2) % L - L / 2
    assert np.abs(off).max() < 0.01 and np.abs(U - x - 3 * DT * v).max() < 0.01
    f, _, _ = e.compute_forces(step=7, thermostat=False)
    fresh = D.Engine(cells, A2, G2, dt=DT, seed=3, pair_kernel=D.PAIR_FULLSHELL)
    fresh.upload(ids, t, X, V, unpbc=U)
    assert np.array_equal(f, fresh.compute_forces(step=7, thermostat=False)[0])
