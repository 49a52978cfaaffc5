"""The slice-stress tables where their LDS windows can go wrong: one slice, fewer slices than
a window, slices much thinner than a cell layer (several windows of the bonded tables), a
window too large for LDS (global atomics), a wavefront of z layers with few beads, three
cells in z (a window over the whole box), and sixteen bead types (no window, no bonded
window).  Against the FP64 oracle."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import chain_state

pytestmark = pytest.mark.gpu

CASES = [((8, 8, 8), 3, 1536, 1), ((8, 8, 8), 3, 1536, 5), ((9, 7, 12), 3, 2268, 96), ((7, 9, 4), 3, 300, 33),
         ((5, 6, 3), 3, 270, 7), ((8, 8, 8), 3, 1536, 800), ((8, 8, 9), 16, 1728, 20), ((9, 7, 12), 1, 2268, 6000)]


@pytest.mark.parametrize("cells,nt,n,nslices", CASES,
                         ids=["x".join(map(str, c)) + f"-t{t}-{s}" for c, t, _, s in CASES])
def test_tables_match_the_oracle(cells, nt, n, nslices):
    nch = max(1, n // 60)
    ids, t, x, u, v, (h, tl, fi, se) = chain_state(cells, nch, 8, n - 8 * nch, seed=n + nslices)
    rng = np.random.default_rng(nslices)
    t = rng.integers(0, nt, len(ids)).astype(np.int32)
    a = rng.uniform(20, 60, (nt, nt))
    a, g = 0.5 * (a + a.T), np.full((nt, nt), 4.5)
    # (chain_state's bonds are 0.5 long: stretched ones, whose table is not zero)
    k, l0 = np.full(len(h), 128.0), np.full(len(h), 0.4)
    mod, ph = np.full(len(fi), 20.0), np.zeros(len(fi))
    print(cells, nt, len(ids), nslices, flush=True)
    e = D.Engine(cells, a, g, seed=9)
    e.upload(ids, t, x, v, unpbc=u)
    e.upload_topology(h, tl, k, l0, fi, se, mod, ph)
    pair, bond = e.slice_stress(nslices)
    bp = e.slice_stress_bondpairs(nslices) if nt < 16 else None
    box, topo = O.Box(cells, a, g, seed=9), O.Topo(h, tl, k, l0, fi, se, mod, ph)
    pr, br = O.slice_stress(box, ids, t, x, v, 0, nslices, unpbc=u, topo=topo)
    pr = pr.reshape(nslices, nt, nt, 9)
    pr = (0.5 * (pr + pr.transpose(0, 2, 1, 3))).reshape(nslices, nt * nt, 9)
    # FP32 pair forces within 1e-5 of the oracle's, and separations of single FP32 offsets
    # (2^-24 of a cell, over a bond's length of ~0.1 at the least)
    for got, ref in ((pair, pr), (bond, br)) + (() if bp is None else
                                               ((bp, O.slice_stress_bondpairs(box, ids, t, x, nslices, unpbc=u, topo=topo)),)):
        assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
        assert np.abs(got.sum(0) - ref.sum(0)).max() <= 1e-5 * np.abs(ref.sum(0)).max()


@pytest.mark.parametrize("nslices", [6, 560, 6000], ids=["long-lists", "short-lists", "no-window"])
def test_lists_that_overflow(nslices):
    """A clump of 600 beads in two cells beside the x face (some 150 partners a bead in the half
    shell, where a list holds 28 or 12) in a box that is thin elsewhere, with a window beside
    which the long lists fit, one beside which only the short do, and none."""
    cells, n = (6, 5, 8), 900
    rng = np.random.default_rng(3)
    L = np.array(cells, float)
    x = rng.uniform(0, 1, (n, 3)) * L
    x[:600] = (np.array([5.2, 2.1, 3.6]) + rng.uniform(0, 1, (600, 3)) * [1.2, 0.8, 0.9]) % L
    t = rng.integers(0, 3, n).astype(np.int32)
    v = rng.normal(0, 1, (n, 3))
    a = np.array([[25.0, 30.0, 40.0], [30.0, 20.0, 35.0], [40.0, 35.0, 15.0]])
    g = np.full((3, 3), 4.5)
    ids = np.arange(1, n + 1, dtype=np.int32)
    print("lists", nslices, flush=True)
    e = D.Engine(cells, a, g, seed=9)
    e.upload(ids, t, x, v)
    pair, _ = e.slice_stress(nslices)
    pr, _ = O.slice_stress(O.Box(cells, a, g, seed=9), ids, t, x, v, 0, nslices)
    pr = pr.reshape(nslices, 3, 3, 9)
    pr = (0.5 * (pr + pr.transpose(0, 2, 1, 3))).reshape(nslices, 9, 9)
    assert np.linalg.norm(pair - pr) <= 1e-5 * np.linalg.norm(pr)
