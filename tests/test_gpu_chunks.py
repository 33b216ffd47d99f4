"""Tile order of k_cg1s and k_mx1 where an XCD takes several tiles at a time (the
farthest column offset is no multiple of 8 tiles and spans 20 or more): boxes whose
planes give 3, 4 and 6 tiles an XCD, all with several whole spans and a remainder, by
one, two and four tiles a workgroup; and two planes only, where the rule is off.  CG and
mixed CG equal the oracle bit for bit."""
import numpy as np
import pytest

from cufoam_amd import mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def check(gpu, nx, ny, nz, coarsen):
    n = nx * ny * nz
    c = np.arange(n)
    i, j = c % nx, c // nx % ny
    nbr = np.stack([c + 1, c + nx, c + nx * ny], 1)
    ok = np.stack([i < nx - 1, j < ny - 1, c < n - nx * ny], 1)
    la = np.broadcast_to(c[:, None], nbr.shape)[ok].astype(np.int32)
    ua = nbr[ok].astype(np.int32)
    rng = np.random.default_rng(nx)
    up = -(1.0 + 0.5 * rng.random(len(la)))
    diag = mesh.row_abs_sum(n, la, ua, up, up) + 1e-2
    s = mesh.LduSystem(n, la, ua, diag, up, up, rng.uniform(-1, 1, n), np.zeros(n))
    gpu.set_system(s)
    A = O.ldu2csr(s)
    # the split form, also below 2^19 rows
    gpu.set_schedule(spmv64=6, fp64_direction=1, coarsen64=coarsen, coarsen32=coarsen)
    ref = O.solve("CG", A, s.b, s.x0, 0.0, 8)
    x, hist, st = gpu.solve("CG", s.b, s.x0, error=0.0, max_steps=8)
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)
    rx, rh, rit, rst = O.mixed_cg(A, s.b, s.x0, 1e-10, 1e-2, 9, 0)
    x, hist, it, rel, st = gpu.solve_mixed(s.b, s.x0, 1e-10, 1e-2, 9, 0)
    assert it == rit
    np.testing.assert_array_equal(hist, rh)
    np.testing.assert_array_equal(x, rx)


@pytest.mark.parametrize("nx,ny,nz", [(160, 161, 25), (250, 130, 18), (230, 226, 11), (301, 90, 4)])
def test_cg_and_mixed(gpu, nx, ny, nz):
    check(gpu, nx, ny, nz, 1)


@pytest.mark.parametrize("nx,ny,nz", [(160, 161, 25), (230, 226, 11), (301, 90, 4)])
@pytest.mark.parametrize("coarsen", [2, 4])
def test_several_tiles_a_workgroup(gpu, nx, ny, nz, coarsen):
    check(gpu, nx, ny, nz, coarsen)


@pytest.mark.parametrize("coarsen", [1, 4])
def test_two_planes(gpu, coarsen):
    check(gpu, 300, 300, 2, coarsen)
