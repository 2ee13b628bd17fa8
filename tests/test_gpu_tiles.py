"""Device kernels at the sizes where their tiles, chunks and dispatch rules
change: edges and remainders of a tile, the smallest and the largest of a
kernel's range, against the FP64 oracle or a plain numpy statement."""
import sys

import numpy as np
import pytest

from . import cases, closure_ref as R, mlp_ref as M, orc
from .blgpu_import import blgpu, solver_for
from .test_gpu_mixed import mixed_solver
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


# statistics blocks: 64 columns by 4 plane groups, wall stress 64 by 16, monitor
# 8 rows of 256 columns: one column less and more than a block, fewer planes
# than groups, the smallest grid.  FP64 sums in another order: a few roundings
# of at most a few hundred terms, 1e-12 relative to the largest value.
@pytest.mark.parametrize("shape", [(64, 8, 18), (65, 9, 17), (5, 4, 5), (257, 18, 6), (258, 17, 40)])
def test_statistics_block_edges(shape):
    say("statistics", shape)
    x, y, z, U, V, W = random_case(sum(shape), *shape)
    rng = np.random.default_rng(2)
    n = (shape[0] + 1, shape[1] + 1, shape[2] + 1)
    P, N = (np.asfortranarray(rng.standard_normal(n)) for _ in range(2))
    s = solver(x, y, z)
    s.set_fields(U, V, W)
    s.upload(3, P)
    s.upload(4, N)
    st = s.statistics()
    _, yg = orc.centers(y)
    w0 = ((yg[1:] - y) / np.diff(yg))[None, :, None]
    u = w0 * U[:, :-1, 1:-1] + (1 - w0) * U[:, 1:, 1:-1]
    v = 0.5 * (V[:-1, :, 1:-1] + V[1:, :, 1:-1])
    w = 0.5 * (W[:-1, :, :-2] + W[1:, :, :-2])
    w = w0 * w[:, :-1] + (1 - w0) * w[:, 1:]
    p = P[:-1, :-1, 1:-1]
    nz = shape[2] - 2
    ref = dict(Umean=u.mean(2), Vmean=v.mean(2), Wmean=w.sum(2) / nz, U2mean=(u * u).mean(2), V2mean=(v * v).mean(2),
               W2mean=(w * w).sum(2) / nz, UVmean=(u * v).mean(2), Pmean=p.mean(2), P2mean=(p * p).mean(2))
    for k, r in ref.items():
        assert np.abs(st[k] - r).max() < 1e-12 * np.abs(r).max(), k
    nm = N[:-1, :-1, 1:-1].mean(2)
    assert np.abs(st["nu_t_mean"][:-1, :-1] - nm).max() < 1e-12 * np.abs(nm).max()
    dudy = (U[:, 1, 1:-1] - U[:, 0, 1:-1]).mean(1) / (yg[1] - yg[0])
    nm2 = np.zeros(n[:2])
    nm2[:-1, :-1] = nm
    tau = 0.25 * (nm2[:-1, 0] + nm2[:-1, 1] + nm2[1:, 0] + nm2[1:, 1]) * dudy
    cf = 2 * (1e-5 * dudy + tau - (u[:, 0] * v[:, 0]).mean(1))
    assert np.abs(st["Cf"] - cf).max() < 1e-12 * np.abs(cf).max()
    I = slice(1, -1)
    parts = [a[I, I, I] for a in (U, V, W, N)]
    scale = np.array([np.abs(a).sum() for a in parts])
    got = s.monitor()
    assert np.all(np.abs(got[:4] - [a.sum() for a in parts]) < 1e-13 * scale)
    np.testing.assert_array_equal(got[4:], [a.max() for a in parts])


# the z chunk of the stage march changes with the grid: one plane per block,
# two (with a remainder) and three
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(70, 9, 5), (131, 20, 13), (66, 25, 101), (300, 60, 40)])
def test_rhs_march_chunks(shape, precision):
    say("rhs march", shape, precision)
    x, y, z, U, V, W = random_case(sum(shape), *shape)
    if precision:
        U, V, W = (np.asfortranarray(a.astype(np.float32).astype(np.float64)) for a in (U, V, W))
    o = orc.Oracle(x, y, z, 1e-5)
    o.set_fields(U, V, W)
    ref = o.rhs()
    s = solver(x, y, z, precision=precision)
    s.set_fields(U, V, W)
    # FP64: the reference's rounding order differs in the last digits (1e-12 as
    # the parity tests); FP32 arithmetic: a few roundings of terms that cancel
    # against each other by less than a factor of ten on random fields
    tol = 1e-5 if precision else 1e-12
    for a, b in zip(s.rhs(), ref):
        assert np.linalg.norm(a - b) < tol * np.linalg.norm(b)


# the x transform: lengths of one factor pair each side of the 31 x 31 limit of
# the shared-area kernel, primes (one column per line), even factors (a pair
# index that is its own mirror), 32 x 32, and line counts that leave a part of a
# block; with many and with few lines (four or eight waves).  Solution against
# the oracle to the Poisson parity tests' 2e-11.
@pytest.mark.parametrize("n,ny,nz", [(4, 5, 6), (7, 4, 5), (22, 24, 10), (31, 9, 7), (127, 6, 8), (129, 75, 53), (197, 5, 6),
                                     (511, 12, 9), (961, 7, 6), (992, 6, 8), (1024, 5, 7), (146, 60, 66)])
def test_x_transform_lengths(n, ny, nz):
    say("x transform", n, ny, nz)
    rng = np.random.default_rng(n)
    nx = n + 2
    x = 1.0 + 0.001 * np.arange(nx)
    y = np.cumsum(np.r_[0, 0.002 + 0.0005 * rng.random(ny - 1)])
    z = 0.0015 * np.arange(nz)
    o = orc.Oracle(x, y, z, 1e-5)
    s = solver(x, y, z)
    r = np.asfortranarray(rng.standard_normal((nx + 1, ny + 1, nz + 1)))
    ref, got = o.poisson(r), s.poisson(r)
    I = (slice(1, n + 1), slice(1, ny), slice(1, nz - 1))
    err = np.linalg.norm((got - ref)[I]) / np.linalg.norm(ref[I])
    say("err", err)
    assert err < 2e-11
    s.close()


# the y solves: 32-row segments, with a last one of a single row and a full one,
# and more tiles of 64 systems than the blocks that reside at a time (8 / segments
# per CU), so that blocks take several; 1, 2, 3, 5 and 8 segments
@pytest.mark.parametrize("n,ny,nz", [(65, 5, 1032), (200, 34, 262), (140, 66, 182), (70, 130, 132), (66, 226, 130),
                                     (30, 33, 12), (30, 65, 12)])
def test_y_solve_segments(n, ny, nz):
    test_x_transform_lengths(n, ny, nz)


# the z transforms' tiles of 16 columns: one full round of the resident waves
# (2048 FP64 tiles, 4096 FP32), a part of a second one, and two rounds and a part
@pytest.mark.parametrize("n,ny,nz", [(128, 257, 8), (129, 257, 8), (268, 257, 7)])
def test_z_transform_rounds(n, ny, nz):
    test_x_transform_lengths(n, ny, nz)


@pytest.mark.parametrize("n,ny,nz", [(256, 257, 8), (258, 257, 8), (520, 257, 7)])
def test_z_transform_rounds_mixed(n, ny, nz):
    test_x_transform_lengths_mixed(n, ny, nz)


# transfers pass through a work array of (nx-2)(ny-1)(nz-2) values, planes of
# up to (nx+1)(ny+1): grids where it holds one plane, a part of the planes,
# and nearly all of them; both directions, exact (FP32 storage: rounded once)
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape", [(5, 4, 5), (6, 5, 40), (24, 16, 8), (300, 30, 20)])
def test_field_transfers(shape, precision):
    say("transfers", shape, precision)
    x, y, z, U, V, W = random_case(1, *shape)
    s = solver(x, y, z, precision=precision)
    rng = np.random.default_rng(4)
    fields = [np.asfortranarray(rng.standard_normal(sh)) for sh in s.shapes]
    for f, a in enumerate(fields):
        s.upload(f, a)
    for f, a in enumerate(fields):
        want = a.astype(np.float32).astype(np.float64) if precision else a
        np.testing.assert_array_equal(s.download(f), want)
    s.close()


# the FP32 x transform takes lengths up to 256 points per factor, the dense
# product the others: both sides of that rule, primes and 31 x 31.  The pressure
# recorded by one mixed projection against the FP64 one of the same FP32 fields.
# The largest errors on the way are those of the split-BF16 products along z: the
# two-term split of either operand and the dropped low x low product are 2^-18
# of a product each, 1.1e-5 in all if every term had the same sign, twice (forward
# and inverse); with the FP32 roundings of the x transforms and of what is stored
# between them (6e-8 each) 5e-5 of the norm is twice that.
@pytest.mark.parametrize("n,ny,nz", [(4, 5, 6), (127, 6, 8), (251, 7, 6), (257, 6, 7), (514, 5, 6), (961, 7, 6)])
def test_x_transform_lengths_mixed(n, ny, nz):
    say("mixed x transform", n, ny, nz)
    rng = np.random.default_rng(n)
    nx = n + 2
    x = 1.0 + 0.001 * np.arange(nx)
    y = np.cumsum(np.r_[0, 0.002 + 0.0005 * rng.random(ny - 1)])
    z = 0.0015 * np.arange(nz)
    shapes = [(nx, ny + 1, nz + 1), (nx + 1, ny, nz + 1), (nx + 1, ny + 1, nz)]
    f = [np.asfortranarray(rng.standard_normal(sh).astype(np.float32).astype(np.float64)) for sh in shapes]
    P = []
    for precision in (0, 1):
        s = solver(x, y, z, precision=precision)
        s.set_fields(*f)
        s.projection(1, 1e-4)
        P.append(s.download(3)[1:n + 1, 1:ny, 1:nz - 1])
        s.close()
    err = np.linalg.norm(P[1] - P[0]) / np.linalg.norm(P[0])
    say("err", err)
    assert err < 5e-5


# the closure's blocks take 256 cells each and loop once there are more than four
# per CU (262144 cells on 256 CUs); fewer cells than a wave's 64, and a remainder.
# Every cell against the row inference of the same network, which no loop is in.
# The features agree to FP64 rounding before the FP32 one, so a BF16 input of the
# network differs only where that rounding crosses a BF16 midpoint: fewer than 1 %
# of the cells, and there by no more than BF16 inference itself is off (5e-2).
@pytest.mark.parametrize("nx,ny,nz", [(5, 4, 5), (33, 12, 9), (162, 62, 40)])
def test_closure_blocks(nx, ny, nz):
    say("closure blocks", nx, ny, nz)
    x, y, z, U, V, W = random_case(nx + ny, nx, ny, nz)
    s = solver(x, y, z, les=4)
    s.set_fields(U, V, W)
    c = blgpu.Closure(capacity=16, batch_max=16)
    c.params = M.init_params(5).astype(np.float32)
    rows = np.ones((2, blgpu.MLP_ROW), dtype=np.float32)
    rows[1, :10] = -1.0
    c.add_rows(rows)
    d99 = 0.5 * y[-1]
    c.install(s, d99, 1e30)
    s.eddy_viscosity()
    got = s.download(4)[1:-1, 1:-1, 1:-1]
    f, _, _, scale = R.features(x, y, z, U, V, W, d99)
    X = f.reshape(10, -1, order="F").T.astype(np.float32)
    want = np.maximum(c.infer_bf16(X).reshape(f.shape[1:], order="F"), 0) * scale
    assert s.closure_fallback() == (got.size, 0)
    err = np.abs(got - want) / np.abs(want).max()
    say("cells", got.size, "largest", err.max(), "beyond 1e-6", (err > 1e-6).mean())
    assert err.max() < 5e-2
    assert (err > 1e-6).mean() < 1e-2
    c.close()
    s.close()


# the march accesses its fields past the caches where nine arrays exceed 256 MB:
# one step of grids just above that line (no model, a model with nu_t, RK2, FP32),
# to the bounds of the step parity tests (FP64 1e-10, mixed 1e-4 of |U|)
@pytest.mark.parametrize("nx,scheme,les,precision", [(130, 3, 0, 0), (130, 2, 0, 0), (130, 3, 1, 0), (260, 3, 0, 1),
                                                     (260, 2, 0, 1), (260, 3, 1, 1)])
def test_march_streams(nx, scheme, les, precision):
    say("streaming march", nx, scheme, les, precision)
    case = cases.laminar_small(nx=nx, ny=130, nz=250, Lz=0.15, noise=0.01, seed=5, scheme=scheme, les=les, cfl=-1e-5)
    o = case.oracle()
    s = (mixed_solver(case, o) if precision else solver_for(case, o)[0])
    o.compute_dt(), s.compute_dt()
    o.step()
    s.step()
    U = np.linalg.norm(o.fields()[0])
    for a, b in zip(s.fields(), o.fields()):
        err = np.linalg.norm(a - b) / U
        say("err", err)
        assert err < (1e-4 if precision else 1e-10)
    s.close()


# first factors of 2 to 7 points go through the vector units, in blocks of four
# waves (the last case: more than four blocks per CU) and of eight; the N2/2 + 1
# rows of the second factor leave 1, 3, 5, .. 14 rows of a tile of 16.  Both
# precisions, to the tolerances of the other lengths.
SHORT_FACTORS = [(194, 5, 6), (94, 9, 7), (159, 6, 8), (164, 7, 9), (185, 6, 5), (258, 12, 9), (343, 9, 11),
                 (502, 40, 34), (94, 97, 90)]


@pytest.mark.parametrize("n,ny,nz", SHORT_FACTORS)
def test_x_transform_short_factor(n, ny, nz):
    test_x_transform_lengths(n, ny, nz)


@pytest.mark.parametrize("n,ny,nz", SHORT_FACTORS)
def test_x_transform_short_factor_mixed(n, ny, nz):
    test_x_transform_lengths_mixed(n, ny, nz)


# with many lines a block takes as many as four products of the second factor
# hold: three of 16 x 32 points and four of 14 x 41, with a part of a block left
@pytest.mark.parametrize("n,ny,nz", [(512, 66, 99), (574, 70, 123)])
def test_x_transform_more_lines(n, ny, nz):
    test_x_transform_lengths(n, ny, nz)
    test_x_transform_lengths_mixed(n, ny, nz)


# the same marches by what a step changes, each component against its own change.
# With noise of 0.3 the eddy viscosity makes 0.15, 0.003 and 0.15 of the change of
# U, V and W (FP32 grid; 0.29, 0.0035 and 0.21 FP64), so a march without it, or with
# nu_t of another cell, is ten times past the bounds or more.  FP32: the z
# transforms' 5e-5 (as for the recorded pressure above) of the pressure gradient,
# whose norm is that of V's change at most, 2.7 times W's; the rounding of the RHS
# (1e-5) and of what is stored (6 times 3e-8 of |U|, 11 times W's change) are far
# below: 1.5e-4, and twice that.  FP64: 2e-11 of the pressure solution likewise,
# 6e-11, and twice that.
@pytest.mark.parametrize("nx,les,precision", [(130, 1, 0), (260, 0, 1), (260, 1, 1)])
def test_march_streams_increment(nx, les, precision):
    say("streaming march, increment", nx, les, precision)
    case = cases.laminar_small(nx=nx, ny=130, nz=250, Lz=0.15, noise=0.3, seed=5, les=les, cfl=-1e-5)
    o = case.oracle()
    if precision:
        o.set_fields(*[np.asfortranarray(a.astype(np.float32).astype(np.float64)) for a in o.fields()])
    old = [a.copy() for a in o.fields()]
    s = (mixed_solver(case, o) if precision else solver_for(case, o)[0])
    o.compute_dt(), s.compute_dt()
    o.step()
    s.step()
    for a, b, c in zip(s.fields(), o.fields(), old):
        err = np.linalg.norm(a - b) / np.linalg.norm(b - c)
        say("err", err)
        assert err < (3e-4 if precision else 1.2e-10)
    s.close()


# large launches of fewer than 128 planes: 385 tiles by 12, 12 and 11 planes in FP64,
# where no chunk keeps the launch to six blocks per compute unit at fewest plane steps;
# the same grid in FP32 takes a short last chunk by the rule of the smaller launches
@pytest.mark.parametrize("precision", [0, 1])
def test_rhs_march_large_launch(precision):
    test_rhs_march_chunks((642, 276, 36), precision)


# the spectral rows of the mixed path are padded to 32 values, and transfers pass
# through the same array: uploads whose low words are FP32 NaN patterns leave NaN in
# every other padding entry, and no solution entry may depend on it.  One length of each
# path: two-factor and dense x, folded and dense z (past 96 rows), partitioned and
# table y solve (past 256 rows).  To the bound of the mixed x transforms.
@pytest.mark.parametrize("n,ny,nz", [(37, 7, 6), (251, 7, 6), (257, 6, 7), (37, 5, 202), (257, 5, 202), (37, 260, 6)])
def test_mixed_padding_undefined(n, ny, nz):
    say("mixed padding", n, ny, nz)
    rng = np.random.default_rng(n)
    nx = n + 2
    x = 1.0 + 0.001 * np.arange(nx)
    y = np.cumsum(np.r_[0, 0.002 + 0.0005 * rng.random(ny - 1)])
    z = 0.0015 * np.arange(nz)
    P = []
    f = []
    for sh in [(nx, ny + 1, nz + 1), (nx + 1, ny, nz + 1), (nx + 1, ny + 1, nz)]:
        a = rng.standard_normal(sh)
        a.view(np.uint32).reshape(-1, 2)[:, 0] = 0x7FC00001
        f.append(np.asfortranarray(a))
    for precision in (0, 1):
        s = solver(x, y, z, precision=precision)
        s.set_fields(*(f if precision else [np.asfortranarray(a.astype(np.float32).astype(np.float64)) for a in f]))
        s.projection(1, 1e-4)
        P.append(s.download(3)[1:n + 1, 1:ny, 1:nz - 1])
        s.close()
    err = np.linalg.norm(P[1] - P[0]) / np.linalg.norm(P[0])
    say("err", err)
    assert err < 5e-5
