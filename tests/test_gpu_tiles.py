"""Device kernels at the sizes where their tiles, chunks and dispatch rules
change: edges and remainders of a tile, the smallest and the largest of a
kernel's range, against the FP64 oracle or a plain numpy statement."""
import sys

import numpy as np
import pytest

from . import cases, mlp_ref as M, orc
from .blgpu_import import blgpu
from .test_oracle_dsm import random_case

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def solver(x, y, z, nu=1e-5, **kw):
    eta, f, df = cases.load_blasius()
    return blgpu.Solver(x, y, z, nu, orc.blasius_tables(x, y, nu, eta, f, df), **kw)


# the stress march owns 30 x 6 cells of a 32 x 8 tile and a chunk of planes;
# nx - 1, ny - 1 cells and nz - 2 planes: one full tile, one cell more, two
# tiles and a remainder, the smallest grid, many planes.  Ghost planes that are
# no periodic copies exercise the index maps in every tile position.
@pytest.mark.parametrize("les", [2, 3])
@pytest.mark.parametrize("shape", [(31, 7, 9), (32, 8, 6), (62, 14, 23), (5, 4, 5), (95, 20, 70)])
def test_dsm_tile_edges(shape, les):
    say("dsm tiles", shape, les)
    x, y, z, U, V, W = random_case(sum(shape), *shape)
    rng = np.random.default_rng(9)
    for a in (U, V, W):
        a[:, :, 0] += 0.1 * rng.standard_normal(a[:, :, 0].shape)
        a[:, :, -1] += 0.1 * rng.standard_normal(a[:, :, -1].shape)
    o = orc.Oracle(x, y, z, 1e-5, les=les)
    o.set_fields(U, V, W)
    ref = o.eddy_viscosity()
    s = solver(x, y, z, les=les)
    s.set_fields(U, V, W)
    s.eddy_viscosity()
    # as the parity tests of the models: 1e-11 of the largest value (quotients
    # of sums of products of differences)
    err = np.abs(s.download(4) - ref).max() / np.abs(ref).max()
    say("nu_t err", err)
    assert err < 1e-11


# the gradient kernel takes tiles of 128 samples, one block per compute unit
# (256) looping over them: a part of a wave, one tile and its neighbours, and
# more tiles than blocks; FP32 sums to 1e-4 as in the closure's gradient tests
@pytest.mark.parametrize("n", [15, 127, 128, 129, 128 * 256 + 17, 128 * 300])
def test_mlp_gradient_tiles(n):
    say("mlp gradient", n)
    rng = np.random.default_rng(n)
    X = rng.uniform(-1, 1, (n, 10)).astype(np.float32)
    t = (0.05 * np.tanh(X[:, 0] * X[:, 1])).astype(np.float32)
    c = blgpu.Closure(capacity=16, batch_max=n)
    theta = M.init_params(3).astype(np.float32)
    c.params = theta
    g, loss = c.gradient(X, t)
    gr = M.grad(theta.astype(np.float64), X.astype(np.float64), t.astype(np.float64))
    y, _ = M.forward(theta.astype(np.float64), X.astype(np.float64))
    assert np.linalg.norm(g - gr) / np.linalg.norm(gr) < 1e-4
    assert np.abs(c.forward(X) - y).max() / np.abs(y).max() < 1e-5
    assert loss == pytest.approx(np.mean((y - t) ** 2), rel=1e-5)
    c.close()


@pytest.mark.parametrize("steps", [0, 1, 3])
def test_mlp_history_of_repeated_training(steps):
    """Every call returns its own steps' losses, longer or shorter than the last call's."""
    rng = np.random.default_rng(1)
    rows = np.zeros((500, 28), dtype=np.float32)
    rows[:, :10] = rng.uniform(-1, 1, (500, 10))
    rows[:, 10] = 0.1 * rows[:, 0]
    rows[:, 11] = 1.0
    one, two = (blgpu.Closure(capacity=500, batch_max=300) for _ in range(2))
    for c in (one, two):
        c.add_rows(rows)
        c.params = M.init_params(3).astype(np.float32)
    a = np.concatenate([one.train(4, 300, seed=5), one.train(steps, 300, seed=5)])
    b = two.train(4 + steps, 300, seed=5)
    np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(one.params, two.params)
