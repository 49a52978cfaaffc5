"""The hit-list kernel's lists where they can go wrong: rows of three, four and five cells
(both faces in one wavefront, x indices modulo 4 across a face), rows longer than the 256
cells of a scan code's x field, a last wavefront with one bead, boxes so dense that every
list overflows within a row, and a cluster that leaves most lists empty while some overflow.
Forces, virial and energy of every schedule against the FP64 oracle."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import force_errors, random_state

pytestmark = pytest.mark.gpu
A2 = np.array([[25.0, 40.0], [40.0, 25.0]])
G2 = np.full((2, 2), 4.5)
HITLIST = [k for k in range(D.schedule_count()) if "hitlist" in D.schedule_name(k)]
# cells, beads, share of the beads in one cell
BOXES = [((3, 3, 3), 81, 0.0), ((4, 3, 5), 65, 0.0), ((5, 7, 3), 900, 0.0), ((6, 3, 4), 1300, 0.0),
         ((259, 3, 3), 7000, 0.0), ((21, 9, 4), 2305, 0.03), ((64, 4, 3), 2304, 0.0)]


@pytest.mark.parametrize("cells,n,clump", BOXES, ids=["x".join(map(str, c)) + f"-{n}" for c, n, _ in BOXES])
@pytest.mark.parametrize("sched", HITLIST, ids=[D.schedule_name(k) for k in HITLIST])
def test_lists_match_the_oracle(sched, cells, n, clump):
    ids, t, x, v = random_state(cells, n, 2, seed=sum(cells) + n)
    m = int(clump * n)
    if m:   # a clump beside the x face
        rng = np.random.default_rng(n)
        x[:m] = np.array([cells[0] - 0.7, 1.2, 1.4]) + rng.uniform(0.0, 0.65, (m, 3))
    print(D.schedule_name(sched), cells, n, flush=True)
    e = D.Engine(cells, A2, G2, seed=11, pair_kernel=D.PAIR_HITLIST)
    e.upload(ids, t, x, v)
    e.set_schedule(sched)
    F, vir, pe = e.compute_forces(step=4)
    fr, virr, per = O.forces(O.Box(cells, A2, G2, seed=11), ids, t, x, v, step=4)
    norm, _ = force_errors(F, fr)
    # FP32 sums of up to ~150 terms: 150 * 2^-24 = 9e-6 of their largest partial sum
    assert norm < 1e-5
    assert np.allclose(vir, virr, rtol=1e-5, atol=1e-6 * np.abs(virr).max())
    assert np.allclose(pe, per, rtol=1e-5)


@pytest.mark.parametrize("n,bonds,name", [
    (11000, 0, "hitlist-split9-t256-c8"), (11001, 0, "hitlist-split3-t256-c12"), (50000, 9, "hitlist-split9-t256-c8"),
    (50001, 9, "hitlist-split3-t256-c12"), (100000, 0, "hitlist-split3-t256-c12"), (100001, 9, "hitlist-t256-c32"),
    (262144, 0, "hitlist-t256-c32"), (262145, 0, "hitlist-t256-c24")])
def test_automatic_schedule_by_bead_count(n, bonds, name):
    cells = (40, 30, 30)
    ids, t, x, v = random_state(cells, n, 2, seed=5)
    u = x.copy()
    h, tl = np.arange(bonds), np.arange(bonds) + 20
    u[tl] = u[h] + [0.4, 0.1, 0.0]
    x = np.mod(u, np.array(cells, float))
    topo = (h, tl, np.full(bonds, 50.0), np.full(bonds, 0.5))
    e = D.Engine(cells, A2, G2, seed=3, pair_kernel=D.PAIR_AUTO)
    e.upload(ids, t, x, v, unpbc=u)
    if bonds:
        e.upload_topology(*topo)
    assert D.schedule_name(e.schedule) == name
    F, _, _ = e.compute_forces(step=2)
    T = O.Topo(*topo, [], [], [], []) if bonds else None
    fr, _, _ = O.forces(O.Box(cells, A2, G2, seed=3), ids, t, x, v, step=2, unpbc=u, topo=T)
    assert force_errors(F, fr)[0] < 1e-5
    if bonds:   # without the topology the choice is that of free beads
        e.upload(ids, t, x, v, unpbc=u)
        e.upload_topology()
        free = 6 if n <= 11000 else (5 if n <= 100000 else (3 if n <= 262144 else 2))
        assert e.schedule == free
