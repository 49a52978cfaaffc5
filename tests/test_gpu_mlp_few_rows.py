"""Training of few rows of a wide network, whose forward and backward passes are two launches with
the columns of the large products spread over workgroups: one row, a ragged block of rows, a last
workgroup with fewer tiles than wavefronts, both sides of the line to the single launch, and that
twice the units do not cost far more than twice the time.  Against the FP64 oracle."""
import time

import numpy as np
import pytest

import mlp_oracle as M
from dpd_amd.mlp import Surrogate

pytestmark = pytest.mark.gpu
# operands rounded to BF16: one unit, as where one activation rounds the other way
TOL = 2.0 ** -8


@pytest.mark.parametrize("nin,H,nout,n", [(7, 1024, 2, 1), (7, 1008, 2, 17), (16, 528, 16, 100), (3, 640, 1, 16),
                                          (7, 1024, 2, 512), (7, 1024, 2, 513), (7, 528, 2, 816), (7, 528, 2, 817)])
def test_against_the_oracle(nin, H, nout, n):
    print("few rows", nin, H, nout, n, flush=True)
    rng = np.random.default_rng(nin + H + n)
    net = Surrogate(nin, H, nout, seed=4)
    X, T = rng.normal(size=(n, nin)), rng.normal(size=(n, nout))
    theta = net.params().astype(np.float64)
    loss, g = net.gradients(X, T)
    lr, gr = M.loss_and_grad(theta, X, T, nin, H, nout, bf=True)
    assert abs(loss - lr) < TOL * lr
    for name, a, b in zip(("W1", "b1", "W2", "b2", "W3", "b3"), M.unpack(g, nin, H, nout), M.unpack(gr, nin, H, nout)):
        assert np.linalg.norm(a - b) < TOL * np.linalg.norm(b), name
    # an iteration's loss is that of the parameters before it, and Adam's step follows the gradients
    losses = net.train(X, T, iters=2, lr=1e-5)
    assert abs(losses[0] - loss) < 1e-9 * loss and losses[1] < losses[0]
    m = np.zeros_like(theta)
    net.set_params(theta.astype(np.float32))
    net.train(X, T, iters=1, lr=1e-3)
    ref, _, _ = M.adam_step(theta, g.astype(np.float64), m, m, 1, 1e-3)
    assert np.max(np.abs(net.params() - ref)) < 1e-6


def test_time_follows_the_units():
    """16 rows: 1,024 units have four times the weights of 512.  Spread over the chip an iteration
    takes 1.4 times as long; one workgroup alone took 2.7 times."""
    rng = np.random.default_rng(1)
    X, T = rng.normal(size=(16, 7)), rng.normal(size=(16, 2))
    us = []
    for H in (512, 1024):
        net = Surrogate(7, H, 2, seed=4)
        net.train(X, T, iters=100)
        best = 1e9
        for _ in range(5):
            t = time.perf_counter()
            net.train(X, T, iters=100)
            best = min(best, time.perf_counter() - t)
        us.append(best * 1e4)
    print(f"  an iteration of 16 rows: {us[0]:.1f} us at 512 units, {us[1]:.1f} at 1,024", flush=True)
    assert us[1] < 2 * us[0]
