"""Single-launch DIC / DILU sweeps (k_ilu_sweep): boxes of cells in lexicographic
order whose edges are no multiples of a brick, flat boxes (consecutive rows
instead of bricks), other orders, rows with more dependencies than are fetched
ahead, a pattern with a box's strides that wraps around (no box), and addressing
that is not upper triangular (level by level).  Histories and solutions equal
the oracle's face loops bit for bit."""
import numpy as np
import pytest

from cufoam_amd import mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def build(n, la, ua, seed, symmetric):
    order = np.lexsort((ua, la))
    la, ua = la[order].astype(np.int32), ua[order].astype(np.int32)
    rng = np.random.default_rng(seed)
    up = -(1.0 + 0.5 * rng.random(len(la)))
    lo = up.copy() if symmetric else up * (1.0 + 0.5 * rng.random(len(la)))
    diag = mesh.row_abs_sum(n, la, ua, lo, up) + 0.05
    return mesh.LduSystem(n, la, ua, diag, lo, up, rng.uniform(-1, 1, n), np.zeros(n))


def box(nx, ny, nz, seed, symmetric):
    c = np.arange(nx * ny * nz)
    i, j, k = c % nx, c // nx % ny, c // (nx * ny)
    la = np.concatenate([c[i < nx - 1], c[j < ny - 1], c[k < nz - 1]])
    ua = np.concatenate([c[i < nx - 1] + 1, c[j < ny - 1] + nx, c[k < nz - 1] + nx * ny])
    return build(nx * ny * nz, la, ua, seed, symmetric)


def wrapped(nx, ny, nz, seed, symmetric):
    """Offsets 1, nx and nx ny at every row: x and y run on into the next line."""
    n = nx * ny * nz
    c = np.arange(n)
    la = np.concatenate([c[:n - d] for d in (1, nx, nx * ny)])
    ua = np.concatenate([c[d:] for d in (1, nx, nx * ny)])
    return build(n, la, ua, seed, symmetric)


def dense_rows(n, seed, symmetric):
    """Each cell coupled to up to 12 earlier ones, in its own workgroup and others."""
    rng = np.random.default_rng(seed)
    pairs = {(int(a), i) for i in range(1, n)
             for a in np.concatenate([rng.integers(max(0, i - 40), i, 6), rng.integers(0, i, 6)])}
    la, ua = np.array(sorted(pairs)).T
    return build(n, la, ua, seed, symmetric)


def shuffled(nx, ny, nz, seed, symmetric):
    s = box(nx, ny, nz, seed, symmetric)
    return mesh.renumber(s, np.random.default_rng(seed).permutation(s.n_cells))


CASES = {
    "box_8": lambda sym: box(8, 8, 8, 1, sym),
    "box_ragged": lambda sym: box(19, 11, 23, 2, sym),
    "box_thin": lambda sym: box(40, 3, 9, 3, sym),
    "box_flat": lambda sym: box(60, 50, 1, 4, sym),
    "line": lambda sym: box(1500, 1, 1, 5, sym),
    "box_33": lambda sym: box(33, 33, 33, 6, sym),
    "wrapped": lambda sym: wrapped(16, 8, 10, 7, sym),
    "dense_rows": lambda sym: dense_rows(1300, 8, sym),
    "shuffled": lambda sym: shuffled(15, 13, 11, 9, sym),
}


@pytest.mark.parametrize("case", CASES)
def test_dic(gpu, case):
    s = CASES[case](True)
    gpu.set_system(s)
    for error, steps in ((0.0, 6), (1e-9 * np.linalg.norm(s.b), 800)):
        ref = O.pcg("DIC", s, s.b, s.x0, error, steps)
        x, hist, st = gpu.solve_pcg("DIC", s.b, s.x0, error=error, max_steps=steps)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("case", CASES)
def test_dilu(gpu, case):
    s = CASES[case](False)
    gpu.set_system(s)
    for error, steps in ((0.0, 6), (1e-8 * np.linalg.norm(s.b), 400)):
        ref = O.pbicg_ldu("DILU", s, s.b, s.x0, error, steps)
        x, hist, st = gpu.solve_pbicg("DILU", s.b, s.x0, error=error, max_steps=steps)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)


def test_addressing_not_upper_triangular(gpu):
    """A face whose owner is the larger cell: accepted, swept level by level."""
    la = np.array([0, 1, 2, 4, 5], np.int32)
    ua = np.array([1, 3, 3, 3, 6], np.int32)
    rng = np.random.default_rng(3)
    up = -rng.uniform(0.5, 1.0, 5)
    s = mesh.LduSystem(7, la, ua, np.full(7, 4.0), up.copy(), up, rng.uniform(-1, 1, 7),
                       np.zeros(7))
    gpu.set_system(s)
    ref = O.pcg("DIC", s, s.b, s.x0, 0.0, 4)
    x, hist, st = gpu.solve_pcg("DIC", s.b, s.x0, error=0.0, max_steps=4)
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("kind", ["DIC", "DILU"])
def test_long_chains_are_waited_for(gpu, kind):
    """40 workgroups in a chain, each slow (24 dependencies a row, most of them read
    one by one): a wave waits many times the polls after which it looks at the
    grid's progress, and gives up only if there is none."""
    n, bands = 40 * 512, 24
    c = np.arange(n)
    la = np.concatenate([c[:n - d] for d in range(1, bands + 1)])
    ua = np.concatenate([c[d:] for d in range(1, bands + 1)])
    s = build(n, la, ua, 11, kind == "DIC")
    gpu.set_system(s)
    gpu.set_sweep_polls(1 << 15)
    try:
        if kind == "DIC":
            ref = O.pcg("DIC", s, s.b, s.x0, 0.0, 2)
            x, hist, st = gpu.solve_pcg("DIC", s.b, s.x0, error=0.0, max_steps=2)
        else:
            ref = O.pbicg_ldu("DILU", s, s.b, s.x0, 0.0, 2)
            x, hist, st = gpu.solve_pbicg("DILU", s.b, s.x0, error=0.0, max_steps=2)
    finally:
        gpu.set_sweep_polls(0)
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("kind", ["DIC", "DILU"])
def test_sweep_failure_is_reported_and_recovers(gpu, kind):
    """The sweeps' bounded wait, forced from the host (gis_set_slot_fault): 1000
    rows are one reduction tile, which waits for nobody, but two workgroups of a
    sweep.  The factor's sweep and, with the factor kept, the solve's give up with
    GIS_ERR_SYNC; then the refilled vectors give the same bits again."""
    from cufoam_amd.gis import GisError
    s = dense_rows(1000, 12, kind == "DIC")
    ref = (O.pcg("DIC", s, s.b, s.x0, 0.0, 5) if kind == "DIC"
           else O.pbicg_ldu("DILU", s, s.b, s.x0, 0.0, 5))

    def solve():
        call = gpu.solve_pcg if kind == "DIC" else gpu.solve_pbicg
        return call(kind, s.b, s.x0, error=0.0, max_steps=5)
    gpu.set_system(s)
    for kept in (False, True):   # whether the factor is there already
        gpu.set_slot_fault(4)
        try:
            with pytest.raises(GisError) as e:
                solve()
            assert e.value.status == 13
        finally:
            gpu.set_slot_fault(0)
        for _ in range(2):
            x, hist, st = solve()
            np.testing.assert_array_equal(hist, ref.hist)
            np.testing.assert_array_equal(x, ref.x)
