"""Device kernels at the sizes where their tiles, chunks and dispatch rules
change: edges and remainders of a tile, the smallest and the largest of a
kernel's range, against the FP64 oracle or a plain numpy statement."""
import sys

import numpy as np
import pytest

from . import cases, orc
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
