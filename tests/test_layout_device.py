"""Set-up kernels (layout_kernels.hip): factors, residual and index arrays
between the caller's numbering and the internal one, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dataset(m, n, nnz, seed):
    """A uniform matrix with empty rows and columns; both copies in row /
    column order, as a caller hands them over."""
    from cdmf_amd import datadir
    r = np.random.default_rng(seed)
    cells = r.choice(m * n, size=min(nnz, m * n), replace=False)
    val = r.standard_normal(cells.size).astype(np.float32)
    return datadir.from_triplets(m, n, (cells // n, cells % n, val), (np.array([0]), np.array([0]), np.array([1.0])))


@pytest.mark.parametrize("m,n,nnz,k", [(1, 1, 1, 1), (255, 3, 300, 8), (256, 257, 900, 9), (2500, 61, 4000, 17)])
def test_factors_and_residual_round_trip(m, n, nnz, k):
    from cdmf_amd import solver as S
    ds = _dataset(m, n, nnz, seed=m + n)
    r = np.random.default_rng(k)
    with S.Solver(0) as s:
        s.upload(ds, with_test=False)
        for kk in (k, k + 1, 1):  # a second set_factors reuses or grows the staging
            W = r.standard_normal((kk, m)).astype(np.float32)
            H = r.standard_normal((kk, n)).astype(np.float32)
            s.set_factors(W, H)
            W2, H2 = s.factors()
            assert np.array_equal(W, W2) and np.array_equal(H, H2)
            a, b = s.residual()
            assert np.array_equal(a, ds.csr_val) and np.array_equal(b, ds.csc_val)


def _shuffled(ds, seed):
    """The same matrix with the elements of every row and column in another
    order (the order a caller may hand them over in is free)."""
    import dataclasses
    r = np.random.default_rng(seed)

    def mix(ptr, idx, val):
        row = np.repeat(np.arange(ptr.size - 1), np.diff(ptr.astype(np.int64)))
        o = np.lexsort((r.random(idx.size), row))
        return idx[o], val[o]

    ci, cv = mix(ds.csr_ptr, ds.csr_idx, ds.csr_val)
    ki, kv = mix(ds.csc_ptr, ds.csc_idx, ds.csc_val)
    return dataclasses.replace(ds, csr_idx=ci, csr_val=cv, csc_idx=ki, csc_val=kv)


def _degree_rows(lengths, n, seed):
    """One row per entry of `lengths`, distinct columns drawn uniformly."""
    from cdmf_amd import datadir
    r = np.random.default_rng(seed)
    rows = np.repeat(np.arange(len(lengths)), lengths)
    cols = np.concatenate([r.choice(n, size=d, replace=False) for d in lengths])
    val = r.integers(1, 6, rows.size).astype(np.float32)
    return datadir.from_triplets(len(lengths), n, (rows, cols, val), (np.array([0]), np.array([0]), np.array([1.0])))


EDGES = [0, 1, 2, 63, 64, 65, 127, 128, 255, 256, 257, 511, 513, 1023, 1024, 1025, 1500]


@pytest.mark.parametrize("n", [2000, 65536, 70001, (1 << 20) + 77])
def test_row_sort_ignores_the_callers_order(n):
    """Rows at the edges of every length class of the device sort, against
    one window of the long rows' bitmap and two, 16- and 32-bit indices: the
    order inside a row does not reach the results, and every element keeps
    its value and its place in the caller's arrays."""
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = _degree_rows(EDGES, n, seed=n)
    k = 3
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    got = []
    for one in (ds, _shuffled(ds, 1)):
        with S.Solver(0) as s:
            s.upload(one, with_test=False)
            s.set_factors(W0, H0)
            a, b = s.residual()
            assert np.array_equal(a, one.csr_val) and np.array_equal(b, one.csc_val)
            s.run(k, 0.05, 2, 2, variant=S.VARIANT_TILED)
            got.append(s.factors())
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


def test_row_sort_with_repeated_indices():
    """Rows that hold an index twice (every length class): each element keeps
    its value, and the solve matches the FP64 oracle as one with the
    elements in order does."""
    import dataclasses

    import oracle
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = _degree_rows([3, 40, 64, 200, 256, 300, 1200], 2000, seed=5)
    row = np.repeat(np.arange(ds.m), np.diff(ds.csr_ptr.astype(np.int64)))
    r = np.random.default_rng(6)
    rows, cols = np.concatenate([row, row[::3]]), np.concatenate([ds.csr_idx, ds.csr_idx[::3]]).astype(np.int64)
    vals = r.integers(1, 6, rows.size).astype(np.float32)
    o, q = np.lexsort((r.random(rows.size), rows)), np.lexsort((r.random(rows.size), cols))

    def ptr(i, size):
        return np.concatenate([[0], np.cumsum(np.bincount(i, minlength=size))]).astype(np.uint32)

    two = dataclasses.replace(ds, csr_ptr=ptr(rows, ds.m), csr_idx=cols[o].astype(np.uint32), csr_val=vals[o],
                              csc_ptr=ptr(cols, ds.n), csc_idx=rows[q].astype(np.uint32), csc_val=vals[q])
    k = 2
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    with S.Solver(0) as s:
        s.upload(two, with_test=False)
        s.set_factors(W0, H0)
        a, b = s.residual()
        assert np.array_equal(a, two.csr_val) and np.array_equal(b, two.csc_val)
        s.run(k, 0.05, 1, 2, variant=S.VARIANT_TILED)
        W, H = s.factors()
    Wo, Ho = oracle.ccd(two, W0, H0, k, 0.05, 1, 2, dtype="f64")[:2]
    # FP32 tree sums of at most 1,600 terms and 4 dependent sweeps: 1e-4 relative
    assert np.linalg.norm(W - Wo) <= 1e-4 * np.linalg.norm(Wo) and np.linalg.norm(H - Ho) <= 1e-4 * np.linalg.norm(Ho)


def test_refused_upload_leaves_the_context():
    from cdmf_amd import solver as S
    ds = _dataset(200, 100, 3000, seed=9)
    W, H = np.ones((2, 200), np.float32), np.ones((2, 100), np.float32)
    import dataclasses
    bad_i = ds.csr_idx.copy()
    bad_i[1234] = 100
    bad_k = ds.csc_idx.copy()
    bad_k[-1] = 200
    with S.Solver(0) as s:
        s.upload(ds, with_test=False)
        s.set_factors(W, H)
        for bad, text in ((dataclasses.replace(ds, csr_idx=bad_i), "CSR: index"),
                          (dataclasses.replace(ds, csc_idx=bad_k), "CSC: index")):
            with pytest.raises(S.CCDError, match=text):
                s.upload(bad, with_test=False)
        a, b = s.residual()
        assert np.array_equal(a, ds.csr_val) and np.array_equal(b, ds.csc_val)


@pytest.mark.parametrize("precision", [0, 1])
def test_larger_matrix_on_the_same_context(precision):
    """A second upload of a larger matrix at the same k gives what a new
    context gives (the factor buffers follow the new shape)."""
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    k = 5
    small, large = _dataset(60, 50, 900, seed=3), _dataset(3000, 2000, 40000, seed=4)

    def solve(s, ds):
        s.upload(ds, with_test=False)
        s.set_factors(D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32))
        s.run(k, 0.05, 2, 2, variant=S.VARIANT_TILED, precision=precision)
        return s.factors()

    with S.Solver(0) as s:
        solve(s, small)
        got = solve(s, large)
    with S.Solver(0) as s:
        want = solve(s, large)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_iteration_times_without_kernel_times():
    """profile_kinds "iter": the callback's times, none per kernel kind, and
    the same factors as without profiling."""
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = _dataset(500, 300, 9000, seed=8)
    k = 3
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    out = []
    with S.Solver(0) as s:
        s.upload(ds)
        for kw in (dict(profile=True, profile_kinds=("iter",)), dict()):
            recs = []
            s.set_factors(W0, H0)
            s.run(k, 0.05, 3, 2, variant=S.VARIANT_TILED, callback=recs.append, **kw)
            out.append(s.factors())
            assert len(recs) == 3
            for r in recs:
                assert (r.rank_time > 0 and r.update_time > 0 and r.rmse_time > 0) == bool(kw)
            if kw:
                assert s.loop_time() >= sum(r.rank_time + r.update_time + r.rmse_time for r in recs)
                assert all(v["launches"] == 0 for v in s.kernel_stats().values())
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
