"""Bonded terms by bead where they can go wrong: stars whose centre is in six bonds and nine
angles, rings, free dimers and angles with a preferred angle, 63 to 65 and 257 bonded beads (the
edges of a wavefront and a workgroup), molecules across the faces; one box with both pair
kernels (the terms in the pair launch and in their own) and a batch.  Forces, virial and
energies at the uploaded state, and the conservative forces of the state after three steps,
against the FP64 oracle."""
import numpy as np
import pytest

import dpd_amd as D
import oracle as O
from helpers import force_errors

pytestmark = pytest.mark.gpu
A2 = np.array([[25.0, 40.0], [40.0, 25.0]])
G2 = np.full((2, 2), 4.5)


def molecules(cells, nbonded, nfree, seed):
    rng = np.random.default_rng(seed)
    L = np.array(cells, dtype=float)
    u, bonds, pairs = [], [], []

    def step(p):
        d = rng.normal(size=3)
        return p + rng.uniform(0.35, 0.6) * d / np.linalg.norm(d)

    kind = 0
    while len(u) < nbonded:
        base, p = len(u), rng.uniform(0, 1, 3) * L
        left = nbonded - base
        u.append(p)
        if kind % 3 == 0 and left >= 7:     # a star: three bonds into the centre, three out of it
            u.extend(step(p) for _ in range(6))
            b = len(bonds)
            bonds.extend((base + 1 + i, base) for i in range(3))
            bonds.extend((base, base + 4 + i) for i in range(3))
            pairs.extend((b + 3 + o, b + i) for o in range(3) for i in range(3))
        elif kind % 3 == 1 and left >= 5:   # a ring of five
            for _ in range(4):
                u.append(step(u[-1]))
            b = len(bonds)
            bonds.extend((base + i, base + (i + 1) % 5) for i in range(5))
            pairs.extend((b + (i + 1) % 5, b + i) for i in range(5))
        elif left >= 2 and left != 3:       # a dimer
            u.append(step(p))
            bonds.append((base, base + 1))
        else:                               # three beads left, or one: a chain with the rest
            while len(u) < nbonded:
                u.append(step(u[-1]))
            b = len(bonds)
            bonds.extend((i, i + 1) for i in range(max(base - 1, 0) if left == 1 else base, nbonded - 1))
            pairs.extend((i + 1, i) for i in range(b, len(bonds) - 1))
        kind += 1
    u.extend(rng.uniform(0, 1, 3) * L for _ in range(nfree))
    u = np.array(u)
    x = np.mod(u, L)
    x[x >= L] = 0.0
    n = len(u)
    # the molecules are spread over the bead indices
    order = rng.permutation(n)
    place = np.argsort(order)
    h, t = (place[np.array(bonds)[:, k]] for k in (0, 1))
    first, second = ((np.array(pairs)[:, k] if pairs else np.zeros(0, int)) for k in (0, 1))
    topo = (h, t, rng.uniform(60, 130, len(h)), rng.uniform(0.3, 0.5, len(h)), first, second,
            rng.uniform(5, 20, len(first)), np.where(np.arange(len(first)) % 2, 0.0, np.radians(30.0)))
    types = (np.arange(n) < nbonded).astype(np.int32)[order]
    return np.arange(1, n + 1, dtype=np.int32), types, x[order], u[order], rng.normal(0, 1, (n, 3)), topo


def check(f, fr):
    # FP32 sums of up to ~150 pair terms and a bonded sum rounded once: 150 * 2^-24 of the
    # largest partial sum
    assert force_errors(f, fr)[0] < 1e-5


@pytest.mark.parametrize("kernel", [D.PAIR_FULLSHELL, D.PAIR_HITLIST], ids=["fullshell", "hitlist"])
@pytest.mark.parametrize("cells,nbonded,nfree", [((4, 5, 3), 2, 90), ((6, 5, 7), 63, 500), ((6, 5, 7), 64, 500),
                                                 ((5, 9, 4), 65, 400), ((8, 7, 6), 257, 700), ((9, 8, 7), 1500, 0)])
def test_terms_match_the_oracle(cells, nbonded, nfree, kernel):
    ids, types, x, u, v, topo = molecules(cells, nbonded, nfree, nbonded)
    print("bonded", cells, nbonded, kernel, flush=True)
    e = D.Engine(cells, A2, G2, seed=5, dt=0.01, pair_kernel=kernel)
    e.upload(ids, types, x, v, unpbc=u)
    e.upload_topology(*topo)
    box, T = O.Box(cells, A2, G2, seed=5, dt=0.01), O.Topo(*topo)
    f, vir, pe = e.compute_forces(step=3)
    fr, virr, per = O.forces(box, ids, types, x, v, step=3, unpbc=u, topo=T)
    check(f, fr)
    assert np.linalg.norm(vir - virr) < 1e-5 * np.linalg.norm(virr)
    assert np.allclose(pe, per, rtol=1e-5, atol=1e-6 * np.abs(per).max())
    e.step(3)
    X, U, V, _ = e.download()
    f, _, _ = e.compute_forces(step=8, thermostat=False)
    check(f, O.forces(box, ids, types, X, V, step=8, thermostat=False, unpbc=U, topo=T)[0])


def test_terms_of_a_batch_match_the_oracle():
    specs = [((4, 5, 3), 2, 90), ((6, 5, 7), 65, 500), ((5, 5, 5), 0, 300), ((8, 7, 6), 257, 700)]
    e = D.Batch([{"cells": c, "a": A2, "gamma": G2, "seed": 5 + i, "dt": 0.01, "ntypes": 2}
                 for i, (c, _, _) in enumerate(specs)], pair_kernel=D.PAIR_HITLIST)
    states = []
    for i, (cells, nb, nf) in enumerate(specs):
        if nb:
            st = molecules(cells, nb, nf, nb)
        else:
            st = molecules(cells, 2, nf, 9)[:5] + (None,)
        e.upload_box(i, st[0], st[1], st[2], st[4], unpbc=st[3])
        if nb:
            e.upload_box_topology(i, *st[5])
        states.append(st)
    e.commit(step0=0)
    for steps in (0, 3):
        if steps:
            e.step(steps)
        f, vir, pe = e.compute_forces(step=8, thermostat=False)
        off, sums = 0, np.zeros(3)
        for i, (cells, nb, _) in enumerate(specs):
            ids, types, x, u, v, topo = states[i]
            if steps:
                x, u, v, _ = e.download_box(i)
            T = O.Topo(*topo) if nb else None
            fr, _, per = O.forces(O.Box(cells, A2, G2, seed=5 + i, dt=0.01), ids, types, x, v, step=8,
                                  thermostat=False, unpbc=u, topo=T)
            check(f[off:off + len(ids)], fr)
            sums += per
            off += len(ids)
        assert np.allclose(pe, sums, rtol=1e-5)
