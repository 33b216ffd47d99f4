"""Resident CG and BiCG (gis_resident.hip): one launch per solve where the system
fits the chip.  Sizes where the route or a tile remainder changes: a single
workgroup of one tile and of two, the first that exchange halos, ragged last
tiles and slices, the largest of one tile per workgroup and the first of two,
the first that does not fit; both slot forms; a halo too large for two tiles; rows
with too many entries.  Every result equals the launch-per-stage kernels' (the
schedule chosen explicitly) bit for bit, and the oracle's where that is quick."""
import numpy as np
import pytest

from cufoam_amd import mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def stages(g, f):
    """f(g) with the schedule in force chosen explicitly: the launch-per-stage loop."""
    g.set_schedule(spmv64=g.get_schedule()["spmv64"])
    return f(g)


@pytest.fixture
def fresh(gpu):
    """A handle of the test's own: no solve of it is held back."""
    from cufoam_amd.gis import Gis
    with Gis(0) as g:
        yield g


def counted(g, f):
    """f(g) and how much each of the handle's resident counts grew."""
    before = g.resident_counts()
    out = f(g)
    return out, {k: v - before[k] for k, v in g.resident_counts().items() if v != before[k]}


def banded(n, width, seed):
    """n cells on a line, each coupled to the next and to the one `width` on."""
    rng = np.random.default_rng(seed)
    c = np.arange(n)
    pairs = np.concatenate([np.stack([c[:-1], c[1:]], 1), np.stack([c[:-width], c[width:]], 1)])
    pairs = pairs[np.lexsort((pairs[:, 1], pairs[:, 0]))]
    la, ua = pairs[:, 0].astype(np.int32), pairs[:, 1].astype(np.int32)
    up = -(1.0 + 0.5 * rng.random(len(la)))
    lo = up * (1.0 + 0.5 * rng.random(len(la)))
    diag = mesh.row_abs_sum(n, la, ua, lo, up) + 0.1
    return mesh.LduSystem(n, la, ua, diag, lo, up, rng.uniform(-1, 1, n), np.zeros(n))


def symmetric(s):
    return mesh.LduSystem(s.n_cells, s.lower_addr, s.upper_addr,
                          mesh.row_abs_sum(s.n_cells, s.lower_addr, s.upper_addr, s.upper,
                                           s.upper) + 0.1, s.upper, s.upper, s.b, s.x0)


SIZES = [1, 3, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 3072, 4099, 65 * 1024 + 1,
         129 * 1024 - 3, 256 * 1024, 256 * 1024 + 1, 512 * 1024, 512 * 1024 + 1]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_resident_equals_stages(gpu, n, method):
    """Column offsets 1 and a large one: tables up to the remainders, far halos."""
    if n < 4:
        s = mesh.random_ldu(n, n, seed=n) if n > 1 else mesh.laplacian(1)
    else:
        s = banded(n, max(2, min(3001, n // 3)), seed=n)
    if method == "CG":
        s = symmetric(s)
    gpu.set_system(s)

    def run(g):
        return g.solve(method, s.b, s.x0, error=1e-9, max_steps=40)
    (x, hist, st), grew = counted(gpu, run)
    assert grew == ({"ran": 1} if n <= (512 if method == "CG" else 256) * 1024 else {})
    (x1, hist1, st1), grew = counted(gpu, lambda g: stages(g, run))
    assert grew == {}
    assert st == st1
    np.testing.assert_array_equal(hist, hist1)
    np.testing.assert_array_equal(x, x1)
    if n <= 5000:
        ref = O.solve(method, O.ldu2csr(s), s.b, s.x0, 1e-9, 40)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("n_cells,n_faces", [(900, 2500), (40000, 110000), (300000, 800000)])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_scattered_halos_and_long_rows(gpu, n_cells, n_faces, method):
    """Columns all over the vector: int32 slots, rows past 8 entries (not resident)."""
    s = mesh.random_ldu(n_cells, n_faces, seed=5, symmetric=method == "CG")
    gpu.set_system(s)

    def run(g):
        return g.solve(method, s.b, s.x0, error=1e-9, max_steps=25)
    (x, hist, _), grew = counted(gpu, run)
    assert grew == {}
    x1, hist1, _ = stages(gpu, run)
    np.testing.assert_array_equal(hist, hist1)
    np.testing.assert_array_equal(x, x1)


@pytest.mark.parametrize("n", [12, 40, 70])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_random_numbering(gpu, n, method):
    """Every neighbour in another workgroup; at 70^3 the halo of two tiles does not
    fit and the launch gives up before it starts."""
    s = mesh.laplacian(n, seed=3, shift=1e-2, symmetric=method == "CG")
    s = mesh.renumber(s, np.random.default_rng(1).permutation(s.n_cells))
    gpu.set_system(s)

    def run(g):
        return g.solve(method, s.b, s.x0, error=1e-6, max_steps=60)
    # 12^3: halos within 2 workgroups; 40^3: about 6000 rows, within CG's 8192, past
    # BiCG's 4096; 70^3: past CG's 5120 with two tiles, and more tiles than BiCG takes
    fits = n == 12 or (n == 40 and method == "CG")
    tries = {"ran": 1} if fits else {} if n == 70 and method == "BiCG" else {"unfit": 1}
    for want in (tries, tries if fits else {}):
        (x, hist, _), grew = counted(gpu, run)
        assert grew == want
    x1, hist1, _ = stages(gpu, run)
    np.testing.assert_array_equal(hist, hist1)
    np.testing.assert_array_equal(x, x1)


def line(n, shift, sym):
    """n cells on a line: CG and BiCG take thousands of iterations."""
    rng = np.random.default_rng(n)
    la = np.arange(n - 1, dtype=np.int32)
    up = -(1.0 + 0.5 * rng.random(n - 1))
    lo = up.copy() if sym else up * (1.0 + 1e-3 * rng.random(n - 1))
    diag = mesh.row_abs_sum(n, la, la + 1, lo, up) + shift
    return mesh.LduSystem(n, la, la + 1, diag, lo, up, rng.uniform(-1, 1, n), np.zeros(n))


@pytest.mark.parametrize("n", [5, 14, -900, -1900])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_chunks_continue(gpu, n, method):
    """More iterations than one launch makes: the next one goes on where it stopped.
    A box of 5^3 ends within one; 14^3 are three workgroups, lines of 900 and 1900
    cells a single one of one and of two tiles (BiCG: two workgroups)."""
    s = (mesh.laplacian(n, seed=9, shift=1e-3, symmetric=method == "CG") if n > 0
         else line(-n, 1e-6, method == "CG"))
    gpu.set_system(s)
    (x, hist, _), grew = counted(
        gpu, lambda g: g.solve(method, s.b, s.x0, error=-1.0, max_steps=4100))
    assert grew == {"ran": -(-(len(hist) - 1) // 2048)} and (grew["ran"] > 1 or n == 5)
    ref = O.solve(method, O.ldu2csr(s), s.b, s.x0, -1.0, 4100)
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)


def test_columns_and_transpose(gpu):
    """Few right-hand sides of a system that fits: the SpMM solve's bits."""
    s = mesh.laplacian(20, seed=4, shift=0.1, symmetric=False)
    gpu.set_system(s)
    B = np.random.default_rng(2).uniform(-1, 1, (3, s.n_cells))
    for transpose in (False, True):
        a, grew = counted(gpu, lambda g: g.solve_multi("BiCG", B, None, error=1e-8,
                                                       max_steps=300, transpose=transpose))
        assert grew == {"ran": 3}
        b = stages(gpu, lambda g: g.solve_multi("BiCG", B, None, error=1e-8, max_steps=300,
                                                transpose=transpose))
        gpu.set_system(s)
        for u, v in zip(a, b):
            np.testing.assert_array_equal(u, v)


def test_infinite_and_nan_inputs(gpu):
    """The stop rules' answers to infinities and NaN, and to a zero right-hand side."""
    s = mesh.laplacian(13, seed=6, shift=1e-2)
    for what in (np.inf, np.nan, 0.0):
        b = s.b.copy()
        if what == 0.0:
            b[:] = 0.0
        else:
            b[700] = what
        for method in ("CG", "BiCG"):
            gpu.set_system(s)

            def run(g):
                return g.solve(method, b, s.x0, error=1e-9, max_steps=6)
            (x, hist, st), grew = counted(gpu, run)
            assert grew == {"ran": 1}
            x1, hist1, st1 = stages(gpu, run)
            assert st == st1
            np.testing.assert_array_equal(hist, hist1)
            np.testing.assert_array_equal(x, x1)


@pytest.mark.parametrize("edges,launches", [([1, 2, 10, 11, 13], 1),
                                            ([40, 64, 3, 65, 17, 30, 30, 30], 2),
                                            ([20] * 40 + [8] * 30, 1)])
def test_batch(gpu, edges, launches):
    """One launch, several launches with systems of one and of two tiles per
    workgroup, and many small systems: every system its own solve's bits."""
    systems = [mesh.laplacian(n, seed=50 + i, shift=1e-3) for i, n in enumerate(edges)]
    err = np.array([1e-6 * np.linalg.norm(s.b) for s in systems])
    b = np.concatenate([s.b for s in systems])

    def run(g):
        return g.batch_solve(b, None, err, 70)
    gpu.batch_set_systems(systems)
    for _ in range(2):
        (x, it, nf, st), grew = counted(gpu, run)
        assert grew == {"ran": launches}
    gpu.batch_set_systems(systems)
    x1, it1, nf1, st1 = stages(gpu, run)
    np.testing.assert_array_equal(it, it1)
    np.testing.assert_array_equal(nf, nf1)
    np.testing.assert_array_equal(x, x1)
    off = 0
    for i, s in enumerate(systems):
        if s.n_cells <= 2200:
            ref = O.solve("CG", O.ldu2csr(s), s.b, s.x0, err[i], 70)
            assert it[i] == ref.iterations and nf[i] == ref.hist[-1]
            np.testing.assert_array_equal(x[off:off + s.n_cells], ref.x)
        off += s.n_cells


def test_batch_mixed_fit(gpu):
    """More iterations than a chunk, and a batch one of whose systems has long rows
    (the whole batch then runs stage by stage)."""
    small = [mesh.laplacian(n, seed=n, shift=1e-3) for n in (20, 3, 9)]
    b = np.concatenate([s.b for s in small])
    gpu.batch_set_systems(small)
    x, it, nf, st = gpu.batch_solve(b, None, -1.0, 2100)
    ref = O.solve("CG", O.ldu2csr(small[0]), small[0].b, small[0].x0, -1.0, 2100)
    assert it[0] == ref.iterations == 2100 and nf[0] == ref.hist[-1]
    np.testing.assert_array_equal(x[:8000], ref.x)
    mixed = small + [mesh.random_ldu(900, 9000, seed=1, symmetric=True)]
    b = np.concatenate([s.b for s in mixed])
    gpu.batch_set_systems(mixed)
    (x, it, nf, st), grew = counted(gpu, lambda g: g.batch_solve(b, None, 1e-8, 300))
    assert grew == {}
    off = 0
    for i, s in enumerate(mixed):
        ref = O.solve("CG", O.ldu2csr(s), s.b, s.x0, 1e-8, 300)
        assert it[i] == ref.iterations
        np.testing.assert_array_equal(x[off:off + s.n_cells], ref.x)
        off += s.n_cells


@pytest.mark.parametrize("first", ["CG", "BiCG"])
def test_one_form_that_does_not_fit_leaves_the_other(gpu, first):
    """About 6000 halo rows a workgroup: past BiCG's 4096, within CG's 8192.  The
    route of either does not depend on which ran first."""
    s = mesh.laplacian(40, seed=3, shift=1e-2)
    s = mesh.renumber(s, np.random.default_rng(1).permutation(s.n_cells))
    gpu.set_system(s)
    order = ["CG", "BiCG"] if first == "CG" else ["BiCG", "CG"]
    for rep in range(2):
        for method in order:
            (x, hist, _), grew = counted(
                gpu, lambda g: g.solve(method, s.b, s.x0, error=0.0, max_steps=20))
            if method == "CG":
                assert grew == {"ran": 1}
            else:
                assert grew == ({"unfit": 1} if rep == 0 else {})
            ref = O.solve(method, O.ldu2csr(s), s.b, s.x0, 0.0, 20)
            np.testing.assert_array_equal(hist, ref.hist)
            np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_late_grid_falls_back_and_holds_back(fresh, method):
    """A first launch that finds its grid late leaves the solve to the stages; the
    next 1, then 3 solves do not wait for theirs; a launch that runs ends that."""
    s = mesh.laplacian(14, seed=9, shift=1e-2, symmetric=method == "CG")
    fresh.set_system(s)
    ref = O.solve(method, O.ldu2csr(s), s.b, s.x0, 1e-9, 400)

    def solve(g):
        x, hist, _ = g.solve(method, s.b, s.x0, error=1e-9, max_steps=400)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)
    fresh.set_late_launches(0, 2)
    want = [{"late": 1}, {"skipped": 1}, {"late": 1}] + [{"skipped": 1}] * 3 + [{"ran": 1}] * 2
    for grew in want:
        assert counted(fresh, solve)[1] == grew


@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_late_grid_between_launches(fresh, method):
    """A launch in the middle of a solve that finds its grid late is tried again."""
    s = mesh.laplacian(14, seed=9, shift=1e-3, symmetric=method == "CG")
    fresh.set_system(s)
    ref = O.solve(method, O.ldu2csr(s), s.b, s.x0, -1.0, 4100)
    fresh.set_late_launches(1, 2)
    (x, hist, _), grew = counted(
        fresh, lambda g: g.solve(method, s.b, s.x0, error=-1.0, max_steps=4100))
    assert grew == {"ran": -(-(len(hist) - 1) // 2048), "late": 2} and grew["ran"] > 1
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("after,count", [(0, 1), (1, 1), (0, 9)])
def test_late_batch(fresh, use_graph, after, count):
    """Systems whose launch finds its grid late are left to the stage loop, beside
    those that ran."""
    systems = [mesh.laplacian(n, seed=60 + i, shift=1e-2) for i, n in enumerate([40, 64, 3, 65, 30])]
    err = np.array([1e-6 * np.linalg.norm(s.b) for s in systems])
    b = np.concatenate([s.b for s in systems])
    fresh.batch_set_systems(systems)

    def run(g):
        return g.batch_solve(b, None, err, 300, use_graph=use_graph)
    want, grew = counted(fresh, run)
    assert set(grew) == {"ran"} and grew["ran"] >= 2
    fresh.set_late_launches(after, count)
    got, late = counted(fresh, run)
    fresh.set_late_launches(0, 0)
    n = min(count, grew["ran"] - after)
    assert late == {k: v for k, v in (("late", n), ("ran", grew["ran"] - n)) if v}
    held, grew = counted(fresh, run)
    assert grew == {"skipped": 1}
    for u, v, w in zip(want, got, held):
        np.testing.assert_array_equal(u, v)
        np.testing.assert_array_equal(u, w)


def test_two_threads(gpu):
    """Two handles in two threads: while one's resident solve runs, a solve of the
    other goes stage by stage, with the same bits.  Either may come first."""
    import threading

    from cufoam_amd.gis import Gis
    s = mesh.laplacian(48, seed=12, shift=1e-3)
    ref = O.solve("CG", O.ldu2csr(s), s.b, s.x0, -1.0, 60)
    done = threading.Event()
    skipped = []

    def long_solves():
        with Gis(0) as g:
            g.set_system(s)
            for _ in range(4):
                g.solve("CG", s.b, s.x0, error=-1.0, max_steps=8000, hist_cap=1)
            skipped.append(g.resident_counts()["skipped"])
        done.set()
    gpu.set_system(s)
    before = gpu.resident_counts()["skipped"]
    t = threading.Thread(target=long_solves)
    t.start()
    while not done.is_set():
        x, hist, _ = gpu.solve("CG", s.b, s.x0, error=-1.0, max_steps=60)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)
    t.join()
    skipped.append(gpu.resident_counts()["skipped"] - before)
    assert len(skipped) == 2 and sum(skipped) > 0


@pytest.mark.parametrize("method", ["CG", "BiCG"])
@pytest.mark.parametrize("after", [0, 1, 2])
def test_columns_that_do_not_start_go_together(fresh, method, after):
    """From the first column whose launch finds its grid late, the columns are one
    SpMM solve: none of them tries a launch of its own."""
    s = mesh.laplacian(20, seed=4, shift=0.1, symmetric=method == "CG")
    fresh.set_system(s)
    A = O.ldu2csr(s)
    At = O.transpose(A)
    B = np.random.default_rng(2).uniform(-1, 1, (3, s.n_cells))
    fresh.set_late_launches(after, 1)
    (X, it, nf, st), grew = counted(
        fresh, lambda g: g.solve_multi(method, B, None, error=1e-8, max_steps=300))
    assert grew == {k: v for k, v in (("ran", after), ("late", 1)) if v}
    for k in range(3):
        ref = O.solve(method, A, B[k], np.zeros(s.n_cells), 1e-8, 300, At=At)
        assert it[k] == ref.iterations and nf[k] == ref.hist[-1]
        np.testing.assert_array_equal(X[k], ref.x)


def test_columns_that_do_not_fit_go_together(gpu):
    """A halo too large for BiCG: the first column gives up, then all are one solve."""
    s = mesh.laplacian(40, seed=3, shift=0.1, symmetric=False)
    s = mesh.renumber(s, np.random.default_rng(1).permutation(s.n_cells))
    gpu.set_system(s)
    A = O.ldu2csr(s)
    At = O.transpose(A)
    B = np.random.default_rng(2).uniform(-1, 1, (2, s.n_cells))
    for want in ({"unfit": 1}, {}):
        (X, it, nf, st), grew = counted(
            gpu, lambda g: g.solve_multi("BiCG", B, None, error=0.0, max_steps=40))
        assert grew == want
        for k in range(2):
            ref = O.solve("BiCG", A, B[k], np.zeros(s.n_cells), 0.0, 40, At=At)
            assert it[k] == ref.iterations and nf[k] == ref.hist[-1]
            np.testing.assert_array_equal(X[k], ref.x)


@pytest.mark.parametrize("edge", [12, 30, 48])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_few_steps_run_as_stages(gpu, edge, method):
    """Solves capped below the steps from which a resident launch pays: the stages,
    and for several columns one SpMM solve."""
    s = mesh.laplacian(edge, seed=13, shift=0.1, symmetric=method == "CG")
    gpu.set_system(s)
    A = O.ldu2csr(s)
    for steps, ran in ((1, {}), (2, {}), (3, {"ran": 1})):
        (x, hist, _), grew = counted(
            gpu, lambda g: g.solve(method, s.b, s.x0, error=0.0, max_steps=steps))
        assert grew == ran
        ref = O.solve(method, A, s.b, s.x0, 0.0, steps)
        np.testing.assert_array_equal(hist, ref.hist)
        np.testing.assert_array_equal(x, ref.x)
    B = np.random.default_rng(5).uniform(-1, 1, (3, s.n_cells))
    each = {12: 4, 30: 12, 48: 16}[edge]
    for nrhs in (1, 2, 3):
        line = max(3, each * (nrhs - 1))
        for steps, ran in ((line - 1, {}), (line, {"ran": nrhs})):
            (X, it, nf, _), grew = counted(
                gpu, lambda g: g.solve_multi(method, B[:nrhs], None, error=0.0, max_steps=steps))
            assert grew == ran
            for k in range(nrhs):
                ref = O.solve(method, A, B[k], np.zeros(s.n_cells), 0.0, steps)
                assert it[k] == ref.iterations and nf[k] == ref.hist[-1]
                np.testing.assert_array_equal(X[k], ref.x)


@pytest.mark.parametrize("method", ["CG", "BiCG"])
@pytest.mark.parametrize("edge", [14, 66])
def test_failed_launch_is_reported_and_recovers(fresh, method, edge):
    """The bounded waits inside a launch, forced from the host: every workgroup gives
    up after 4 polls and exits, the solve reports GIS_ERR_SYNC, and the next one has
    its bits again.  66^3: two tiles a workgroup (CG)."""
    from cufoam_amd.gis import GisError
    s = mesh.laplacian(edge, seed=15, shift=0.1, symmetric=method == "CG")
    if method == "BiCG" and edge == 66:
        s = mesh.laplacian(63, seed=15, shift=0.1, symmetric=False)
    fresh.set_system(s)
    A = O.ldu2csr(s)
    ref = O.solve(method, A, s.b, s.x0, 0.0, 40)
    B = np.stack([s.b, s.b[::-1]])
    fresh.set_resident_fault(4)
    for call in (lambda g: g.solve(method, s.b, s.x0, error=0.0, max_steps=40),
                 lambda g: g.solve_multi(method, B, None, error=0.0, max_steps=40)):
        with pytest.raises(GisError) as e:
            call(fresh)
        assert e.value.status == 13
    fresh.set_resident_fault(0)
    (x, hist, _), grew = counted(
        fresh, lambda g: g.solve(method, s.b, s.x0, error=0.0, max_steps=40))
    assert grew == {"ran": 1}
    np.testing.assert_array_equal(hist, ref.hist)
    np.testing.assert_array_equal(x, ref.x)
    X, it, nf, st = fresh.solve_multi(method, B, None, error=0.0, max_steps=40)
    np.testing.assert_array_equal(X[0], ref.x)


def test_failed_batch_launch_is_reported_and_recovers(fresh):
    """The same in a batch: systems of several workgroups fail, one of a single
    workgroup waits for nobody; then every system has its bits again."""
    from cufoam_amd.gis import GisError
    systems = [mesh.laplacian(n, seed=70 + i, shift=1e-2) for i, n in enumerate([14, 9, 40])]
    b = np.concatenate([s.b for s in systems])
    fresh.batch_set_systems(systems)
    fresh.set_resident_fault(4)
    with pytest.raises(GisError) as e:
        fresh.batch_solve(b, None, 1e-8, 300)
    assert e.value.status == 13
    fresh.set_resident_fault(0)
    (x, it, nf, st), grew = counted(fresh, lambda g: g.batch_solve(b, None, 1e-8, 300))
    assert set(grew) == {"ran"}
    off = 0
    for i, s in enumerate(systems):
        ref = O.solve("CG", O.ldu2csr(s), s.b, s.x0, 1e-8, 300)
        assert it[i] == ref.iterations and nf[i] == ref.hist[-1]
        np.testing.assert_array_equal(x[off:off + s.n_cells], ref.x)
        off += s.n_cells
