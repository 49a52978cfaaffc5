"""The hit-list kernel's candidate test on byte codes (code_dist2 in pair_kernels.hpp, scan_code
in engine_common.hpp), restated on the CPU with the kernel's FP32 and 32-bit arithmetic: no
pair inside the cut-off can be missed, in cubic and in unequal cells, across periodic faces of
any number of cells, at any cell index, with the borrows of the one subtraction; and of the
candidates of cubic cells only those within 1.03 of the cut-off pass."""
import numpy as np
import pytest

f32 = np.float32
U = 84


def scan_code(o, c, w):
    q = np.clip((o.astype(f32) * (f32(U) / w.astype(f32))).astype(np.int64), 0, U - 1) + U * c
    q &= 0xFF
    return (q[:, 0] | (q[:, 1] << 8) | (1 << 16) | (q[:, 2] << 24)).astype(np.uint32)


def bead_code(o, c, w):
    inv = f32(U) / w.astype(f32)
    t = o.astype(f32) * inv
    t[:, 1] -= f32(0.5)
    q = np.floor(t).astype(np.int64) + U * c
    return ((q[:, 0] & 0xFF) | ((q[:, 1] & 0xFF) << 8) | ((q[:, 2] & 0xFF) << 24)).astype(np.uint32)


def dist2(code, Q):
    d = (code - Q).astype(np.uint32)
    b = np.stack([(d >> s) & 0xFF for s in (0, 8, 16, 24)], -1).astype(np.int64)
    b = np.where(b > 127, b - 256, b)
    return (b * b).sum(axis=1)


def threshold(w):
    w = w.astype(f32)
    s2 = (w * w * np.array([1.0, 2.25, 1.0], f32)).sum(dtype=f32)
    t = (f32(1.0) + np.sqrt(s2) * f32(1.01 / U) + f32(1e-5)) * (f32(U) / w).max()
    return int(t * t) + 2


@pytest.mark.parametrize("w", [(1, 1, 1), (1.25, 1.25, 1.25), (1, 1.5, 2), (2.0, 1.0, 1.1), (1.0, 3.0, 1.0)])
@pytest.mark.parametrize("n", [(3, 4, 5), (64, 7, 300), (255, 256, 257)])
def test_no_pair_inside_the_cutoff_is_missed(w, n):
    rng = np.random.default_rng(int(10 * sum(w)) + sum(n))
    w, n = np.array(w, float), np.array(n)
    m = 200000
    c = rng.integers(0, n, (m, 3))
    edge = rng.random((m, 3)) < 0.2                       # beads in the first and last cells
    c = np.where(edge, np.where(rng.random((m, 3)) < 0.5, 0, n - 1), c)
    o = (rng.random((m, 3)) * w).astype(f32)
    o = np.where(rng.random((m, 3)) < 0.05, f32(0), np.minimum(o, (w * 0.99999994).astype(f32)))
    # partners on and inside the cut-off sphere
    d = rng.normal(size=(m, 3))
    d /= np.linalg.norm(d, axis=1)[:, None]
    d *= np.where(rng.random(m) < 0.5, 1.0, rng.random(m))[:, None]
    x = o.astype(float) + d
    step = np.floor(x / w).astype(int)
    po = np.clip(x - step * w, 0, None).astype(f32)
    po = np.minimum(po, (w * 0.99999994).astype(f32))
    keep = (np.abs(step) <= 1).all(axis=1)                # (a cell is no smaller than the cut-off)
    assert keep.mean() > 0.999
    pc = c + step
    wrap = np.where(pc < 0, 1, np.where(pc >= n, -1, 0))
    # the row across a face sees the bead a box's length away
    got = dist2(scan_code(po, pc + wrap * n, w), bead_code(o, c + wrap * n, w))
    # pairs in reach by the kernel's own FP32 positions
    diff = (po.astype(float) + step * w) - o
    inside = (diff * diff).sum(axis=1) < 1.0
    assert (got[keep & inside] < threshold(w)).all()


def test_candidates_that_pass_are_near():
    rng = np.random.default_rng(1)
    w, m = np.ones(3), 400000
    o, po = rng.random((m, 3)).astype(f32), rng.random((m, 3)).astype(f32)
    c, step = rng.integers(1, 50, (m, 3)), rng.integers(-1, 2, (m, 3))
    near = dist2(scan_code(po, c + step, w), bead_code(o, c, w)) < threshold(w)
    r = np.linalg.norm(po + step - o.astype(float), axis=1)
    # within the error of a code, sqrt(1 + 1.5^2 + 1) units, of the widened cut-off
    assert r[near].max() < 1.0 + 2 * 2.07 / U + 1e-3
    assert near.sum() < 1.12 * (r < 1.0).sum()
