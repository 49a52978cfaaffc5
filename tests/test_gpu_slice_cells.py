"""Slice stress tables in boxes whose cells are wider than 1 and not as high as wide: the layers
that a workgroup's window follows, its first slice and its size are in units of the cells'
height.  Pairs, bonds and bond pairs against the FP64 oracle, with a window beside either list
length and without one."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import chain_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,widths,nslices", [
    ((8, 8, 8), (1.0, 1.0, 1.25), 5), ((8, 8, 8), (1.0, 1.0, 1.25), 77), ((4, 5, 3), (2.0, 1.0, 3.0), 16),
    ((5, 4, 4), (1.0, 2.0, 1.75), 320), ((4, 4, 6), (1.5, 2.0, 1.5), 6000), ((8, 6, 5), (1.0, 1.0, 1.6), 1)],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_tables_match_the_oracle(cells, widths, nslices):
    size = tuple(int(round(c * w)) for c, w in zip(cells, widths))
    assert np.allclose(size, np.array(cells) * widths)
    n = 3 * int(np.prod(size))
    ids, t, x, u, v, (h, tl, fi, se) = chain_state(size, n // 60, 8, n - 8 * (n // 60), seed=n + nslices)
    rng = np.random.default_rng(nslices)
    t = rng.integers(0, 3, n).astype(np.int32)
    a = rng.uniform(20, 60, (3, 3))
    a, g = 0.5 * (a + a.T), np.full((3, 3), 4.5)
    # (chain_state's bonds are 0.5 long: stretched ones, whose table is not zero)
    topo = (h, tl, np.full(len(h), 128.0), np.full(len(h), 0.4), fi, se, np.full(len(fi), 20.0), np.zeros(len(fi)))
    print("cells", cells, widths, n, nslices, flush=True)
    e = D.Engine(cells, a, g, seed=9, widths=widths)
    e.upload(ids, t, x, v, unpbc=u)
    e.upload_topology(*topo)
    pair, bond = e.slice_stress(nslices)
    bp = e.slice_stress_bondpairs(nslices)
    box, topo = O.Box(cells, a, g, seed=9, widths=widths), O.Topo(*topo)
    # at the positions the engine holds (FP32 offsets in their cells)
    X, U = e.download()[:2]
    pr, br = O.slice_stress(box, ids, t, X, v, 0, nslices, unpbc=U, topo=topo)
    pr = pr.reshape(nslices, 3, 3, 9)
    pr = (0.5 * (pr + pr.transpose(0, 2, 1, 3))).reshape(nslices, 9, 9)
    for got, ref, tol in ((pair, pr, 1e-5), (bond, br, 1e-9), (bp, O.slice_stress_bondpairs(box, ids, t, X, nslices, unpbc=U, topo=topo), 1e-9)):
        # FP32 pair forces within 1e-5 of the oracle's; bonds and bond pairs are FP64 on both sides
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
