"""Slice stress of flat pairs: two beads with |dz| <= 1e-5 add half of their share to each
bead's own slice, under (its type, the other's), also where a slice border lies between them
or one of them lies on it.  Isolated pairs about slice borders, layer borders of the cells and
the periodic face, with a window in LDS beside either list length and without one, in cells of
unit and other heights.  Expected: the oracle's pair forces, split by the rule in FP64."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O

pytestmark = pytest.mark.gpu
A3 = np.array([[25.0, 40.0, 30.0], [40.0, 20.0, 35.0], [30.0, 35.0, 15.0]])
G3 = np.full((3, 3), 4.5)
# z of the two beads about a border: across it, across it and past the border rule, on it,
# both above, and both in the middle of a slice
ABOUT = [(-3e-6, 4e-6), (-5e-7, 9e-6), (-5e-6, 2e-6), (0.0, 0.0), (2e-6, 8e-6), (0.11, 0.11 + 4e-6)]


def own_slices(z, nslices, Lz):
    """(slice, share) of a bead that stands for both of a flat pair"""
    s = z * nslices / Lz
    k = min(int(s), nslices - 1)
    return [(k, 1.0)] if s - k > 1e-5 else [(k, 0.5), ((k - 1) % nslices, 0.5)]


@pytest.mark.parametrize("cells,width,nslices", [((8, 8, 8), 1.0, 16), ((8, 8, 8), 1.0, 560), ((8, 8, 8), 1.0, 6000),
                                                 ((8, 8, 8), 1.25, 20)],
                         ids=["long-lists", "short-lists", "no-window", "w_z-1.25"])
def test_halves_go_to_the_beads_own_slices(cells, width, nslices):
    L = np.array([8.0, 8.0, 8.0 * width])
    rng = np.random.default_rng(nslices)
    x = []
    for i, level in enumerate((0.0, 1.5, 3.0, 4.5, 6.0)):
        for j in range(24):
            a, b = ABOUT[(i + j) % len(ABOUT)]
            at = np.array([2.0 * (j % 4) - 0.4, 4.0 / 3.0 * (j // 4), level])
            pair = [at + [0.0, 0.0, a], at + [rng.uniform(0.4, 0.8), rng.uniform(-0.1, 0.1), b]]
            x += pair[::-1] if rng.random() < 0.5 else pair
    x = np.mod(np.array(x), L)
    n = len(x)
    order = rng.permutation(n)     # bead indices, and so slots of a cell, in any order
    mate = np.empty(n, int)
    place = np.argsort(order)
    mate[place] = place[np.arange(n) ^ 1]
    x = x[order]
    t = rng.integers(0, 3, n).astype(np.int32)
    v = rng.normal(0, 1, (n, 3))
    ids = np.arange(1, n + 1, dtype=np.int32)
    print("flat pairs", cells, width, nslices, flush=True)
    e = D.Engine(cells, A3, G3, seed=5, widths=(1.0, 1.0, width))
    e.upload(ids, t, x, v)
    got, _ = e.slice_stress(nslices, bonds=False)
    X = e.download()[0]
    F, _, _ = O.forces(O.Box(cells, A3, G3, seed=5, widths=(1.0, 1.0, width)), ids, t, X, v, step=0)
    want = np.zeros((nslices, 3, 3, 9))
    across = 0
    for i in range(n):
        d = X[i] - X[mate[i]]
        d -= L * np.round(d / L)
        assert abs(d[2]) <= 1e-5 and np.abs(F[i] + F[mate[i]]).max() < 1e-9 * np.abs(F[i]).max()
        across += own_slices(X[i, 2], nslices, L[2]) != own_slices(X[mate[i], 2], nslices, L[2])
        for s, share in own_slices(X[i, 2], nslices, L[2]):
            want[s, t[i], t[mate[i]]] += 0.5 * share * np.outer(F[i], d).ravel()
    assert across >= n // 4
    # FP32 pair forces within 1e-5 of the oracle's, entry by entry of the table
    got = got.reshape(want.shape)
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
