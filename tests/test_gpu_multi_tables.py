"""Multi-RHS SpMM over offset tables of 3 to 15 entries: tables shorter than a
batch, a whole batch, and one to three or more entries left over after it.  Every
column equals its single-RHS oracle solve bit for bit."""
import numpy as np
import pytest

from cufoam_amd import mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bands", [1, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_table_lengths(gpu, bands, method):
    n = 3000
    offs = [1, 2, 5, 70, 71, 200, 777][:bands]
    c = np.arange(n)
    la = np.concatenate([c[:n - d] for d in offs])
    ua = np.concatenate([c[d:] for d in offs])
    order = np.lexsort((ua, la))
    la, ua = la[order].astype(np.int32), ua[order].astype(np.int32)
    rng = np.random.default_rng(bands)
    up = -(1.0 + 0.5 * rng.random(len(la)))
    lo = up.copy() if method == "CG" else up * (1.0 + 0.5 * rng.random(len(la)))
    diag = mesh.row_abs_sum(n, la, ua, lo, up) + 0.1
    s = mesh.LduSystem(n, la, ua, diag, lo, up, rng.uniform(-1, 1, n), np.zeros(n))
    gpu.set_system(s)
    assert gpu.get_schedule()["spmv64"] == 6
    A = O.ldu2csr(s)
    B = rng.uniform(-1, 1, (4, n))
    X, it, nf, st = gpu.solve_multi(method, B, None, error=1e-8, max_steps=60)
    for k in range(4):
        ref = O.solve(method, A, B[k], np.zeros(n), 1e-8, 60)
        assert it[k] == ref.iterations and nf[k] == ref.hist[-1]
        np.testing.assert_array_equal(X[k], ref.x)


@pytest.mark.parametrize("bands,far,longest", [(12, 0, 25), (14, 0, 29), (15, 0, 31),
                                               (15, 1600, 32)])
@pytest.mark.parametrize("method", ["CG", "BiCG"])
def test_longest_tables(gpu, bands, far, longest, method):
    """The last batch of a long table reaches past the 32 bits of a row mask.  A
    far band of which each row has one side brings a table to 32 entries."""
    n = 3000
    offs = list(range(1, bands + 1)) + ([far] if far else [])
    c = np.arange(n)
    la = np.concatenate([c[:n - d] for d in offs])
    ua = np.concatenate([c[d:] for d in offs])
    order = np.lexsort((ua, la))
    la, ua = la[order].astype(np.int32), ua[order].astype(np.int32)
    rng = np.random.default_rng(longest)
    up = -(1.0 + 0.5 * rng.random(len(la)))
    lo = up.copy() if method == "CG" else up * (1.0 + 0.5 * rng.random(len(la)))
    diag = mesh.row_abs_sum(n, la, ua, lo, up) + 0.1
    s = mesh.LduSystem(n, la, ua, diag, lo, up, rng.uniform(-1, 1, n), np.zeros(n))
    gpu.set_system(s)
    sizes = []
    for a in range(0, n, 64):
        rows = np.arange(a, min(a + 64, n))
        sizes.append(sum(bool(((rows + d >= 0) & (rows + d < n)).any())
                         for d in [0] + offs + [-d for d in offs]))
    assert max(size for size in sizes if size <= 32) == longest
    lay = gpu.layout()
    assert lay["table_slices"] == sum(size <= 32 for size in sizes)
    assert lay["table_entries"] == sum(size for size in sizes if size <= 32)
    assert gpu.get_schedule()["spmv64"] == 6
    A = O.ldu2csr(s)
    B = rng.uniform(-1, 1, (4, n))
    X, it, nf, st = gpu.solve_multi(method, B, None, error=1e-8, max_steps=60)
    for k in range(4):
        ref = O.solve(method, A, B[k], np.zeros(n), 1e-8, 60)
        assert it[k] == ref.iterations and nf[k] == ref.hist[-1]
        np.testing.assert_array_equal(X[k], ref.x)
