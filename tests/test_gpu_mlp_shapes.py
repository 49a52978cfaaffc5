"""GPU tests of the surrogate network's kernels at the edges of their tiles: batches around a
16-row workgroup and a 128-row slab of the bias sums, hidden layers of one column tile, of a
ragged number of tiles per wavefront and of the largest size, the narrowest and widest inputs
and outputs, and batches of more than 256 workgroups (eight wavefronts instead of sixteen); and
where the update changes from four wavefronts to eight and to sixteen, with parts of its sums
of one to eight steps and longer."""
import numpy as np
import pytest

import mlp_oracle as M
from dpd_amd.mlp import Surrogate

pytestmark = pytest.mark.gpu

# Every operand of a product is rounded to BF16 (relative 2^-9).  Where the oracle's activation
# falls on the other side of a rounding boundary than the kernel's FP32 one it moves by a
# whole unit, 2^-8; a sum of many such terms is off by well under that unit.  One row and one
# tile leave a handful of terms, so the bound is the unit itself.
TOL = 2.0 ** -8


@pytest.mark.parametrize("nin,H,nout,n", [
    (1, 16, 1, 1), (7, 16, 2, 15), (16, 48, 16, 16), (3, 128, 5, 17), (6, 144, 2, 127), (6, 272, 2, 129),
    (7, 256, 2, 2100), (5, 528, 3, 40), (7, 1024, 2, 33), (2, 144, 1, 4112), (4, 272, 2, 4130),
    (4, 64, 2, 512), (6, 512, 2, 513), (3, 528, 2, 520), (7, 128, 2, 1024), (7, 128, 2, 1025), (5, 144, 2, 1030),
    (2, 32, 1, 1456), (2, 16, 1, 1100)])
def test_edges_of_the_tiles(nin, H, nout, n):
    rng = np.random.default_rng(nin + H + n)
    net = Surrogate(nin, H, nout, seed=4)
    scal = rng.normal(size=nin), rng.uniform(0.5, 2, nin), rng.normal(size=nout), rng.uniform(0.5, 2, nout)
    net.set_scaling(*scal)
    X, T = rng.normal(size=(n, nin)), rng.normal(size=(n, nout))
    xs, ts = (X - scal[0]) / scal[1], (T - scal[2]) / scal[3]
    theta = net.params().astype(np.float64)
    loss, g = net.gradients(X, T)
    lr, gr = M.loss_and_grad(theta, xs, ts, nin, H, nout, bf=True)
    assert abs(loss - lr) < TOL * lr
    for name, a, b in zip(("W1", "b1", "W2", "b2", "W3", "b3"), M.unpack(g, nin, H, nout), M.unpack(gr, nin, H, nout)):
        assert np.linalg.norm(a - b) < TOL * np.linalg.norm(b), name
    y = M.forward(theta, xs, nin, H, nout, bf=True)[2]
    assert np.linalg.norm((net.predict(X) - scal[2]) / scal[3] - y) < TOL * np.linalg.norm(y)
    # an iteration's loss is that of the parameters before it, and Adam's step follows the gradients
    losses = net.train(X, T, iters=2, lr=1e-5)
    assert abs(losses[0] - loss) < 1e-9 * loss and losses[1] < losses[0]
    m = np.zeros_like(theta)
    net.set_params(theta.astype(np.float32))
    net.train(X, T, iters=1, lr=1e-3)
    ref, _, _ = M.adam_step(theta, g.astype(np.float64), m, m, 1, 1e-3)
    assert np.max(np.abs(net.params() - ref)) < 1e-6
