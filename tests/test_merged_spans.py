"""Rows spanning tiles finished by the next sweep (MergedArgs) instead of
a launch of their own: bit for bit what the batched solver, which finishes
them between two barriers, computes for the same problem."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(lengths, n, seed):
    from cdmf_amd import datadir
    r = np.random.default_rng(seed)
    rows = np.repeat(np.arange(len(lengths)), lengths)
    cols = np.concatenate([r.choice(n, size=d, replace=False) for d in lengths])
    val = r.integers(1, 6, rows.size).astype(np.float32)
    return datadir.from_triplets(len(lengths), n, (rows, cols, val), (rows[:3], cols[:3], val[:3]))


def _uniform(m, n, per, seed):
    return _rows([per] * m, n, seed)


CASES = {
    # one tile and none spanning, two tiles and one span
    "one_tile": lambda: _uniform(20, 40, 10, 1),
    "two_tiles": lambda: _uniform(50, 60, 25, 2),
    # about 256 two-tile spans in the rows' layout (sigma 16), the bound of
    # the merge: just below and above
    "spans_252": lambda: _uniform(8900, 300, 30, 9),
    "spans_262": lambda: _uniform(9270, 300, 30, 10),
    # about 512 in the rows' layout, just below and above
    "spans_500": lambda: _uniform(17100, 300, 30, 3),
    "spans_530": lambda: _uniform(18100, 300, 30, 4),
    # 32 and 33 rows over more than two tiles
    "long_32": lambda: _rows([4000] * 32 + [7] * 500, 5000, 5),
    "long_33": lambda: _rows([4000] * 33 + [7] * 500, 5000, 6),
    # the gathered vector at the bound of the merge, and past it
    "wide_8192": lambda: _rows([1500] * 40 + [3] * 900, 8192, 11),
    "wide_8193": lambda: _rows([1500] * 40 + [3] * 900, 8193, 12),
    # past it, where the vector fills much of the LDS
    "wide_16384": lambda: _rows([1500] * 40 + [3] * 900, 16384, 7),
    "wide_16385": lambda: _rows([1500] * 40 + [3] * 900, 16385, 8),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("sigma", [8, 16])
def test_single_run_equals_batched(name, sigma):
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = CASES[name]()
    k, lam, outer, inner = 3, 0.05, 2, 3
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    with S.Solver(0) as s:
        s.set_plan(sigma=sigma, split_rows=0)
        s.upload(ds, with_test=False)
        out = []
        for graph in (False, True):
            s.set_factors(W0, H0)
            s.run(k, lam, outer, inner, variant=S.VARIANT_TILED, use_graph=graph)
            out.append(s.factors() + s.residual())
        s.set_factors(W0, H0)
        b = S.Batch(0)
        b.set_plan(sigma=sigma)
        b.add(s, k, lam, outer, inner)
        b.run()
        out.append(s.factors() + s.residual())
        b.close()
    assert np.all(np.isfinite(out[0][0]))
    for got in out[1:]:
        for x, y in zip(got, out[0]):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("precision,sigma", [(0, 32), (2, 16)])
def test_other_precisions_match_oracle(precision, sigma):
    """The merged sweeps with FP64 sums and at sigma 32.  FP32 sums of at most
    4,000 terms through 4 dependent sweeps: 1e-4 relative; FP64 sums 2e-5.
    (bfloat16: test_bf16_first_rank_matches_twin of test_gpu_parity.py runs
    merged sweeps.)"""
    import oracle
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = CASES["long_32"]()
    k, lam, outer, inner = 2, 0.1, 1, 2
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    Wo, Ho = oracle.ccd(ds, W0, H0, k, lam, outer, inner, dtype="f64")[:2]
    with S.Solver(0) as s:
        s.set_plan(sigma=sigma)
        s.upload(ds, with_test=False)
        s.set_factors(W0, H0)
        s.run(k, lam, outer, inner, variant=S.VARIANT_TILED, precision=precision)
        W, H = s.factors()
    tol = {0: 1e-4, 2: 2e-5}[precision]
    assert np.linalg.norm(W - Wo) <= tol * np.linalg.norm(Wo) and np.linalg.norm(H - Ho) <= tol * np.linalg.norm(Ho)


@pytest.mark.parametrize("name", ["two_tiles", "spans_252", "long_32", "wide_8192"])
@pytest.mark.parametrize("precision,sigma", [(1, 16), (2, 16), (0, 8), (0, 16), (0, 32)])
def test_merged_equals_finished_by_its_own_launch(name, precision, sigma):
    """The same matrix with empty rows and columns added until both gathered
    vectors are past the bound of the merge: the same tiles, each sweep's
    spanning rows finished by a launch of their own.  Every precision, bit
    for bit (with bfloat16 storage the merged rows are rounded as stored
    ones are)."""
    import dataclasses

    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = CASES[name]()
    k, lam, outer, inner = 2, 0.05, 2, 3
    m2, n2 = max(ds.m, 8300), max(ds.n, 8300)
    pad = lambda p, size: np.concatenate([p, np.full(size + 1 - p.size, p[-1], p.dtype)])
    wide = dataclasses.replace(ds, m=m2, n=n2, csr_ptr=pad(ds.csr_ptr, m2), csc_ptr=pad(ds.csc_ptr, n2))
    W0 = D.initial_col(k, ds.m)
    out = []
    for one in (ds, wide):
        W1 = np.zeros((k, one.m), np.float32)
        W1[:, :ds.m] = W0
        with S.Solver(0) as s:
            s.set_plan(sigma=sigma, split_rows=0)
            s.upload(one, with_test=False)
            s.set_factors(W1, np.zeros((k, one.n), np.float32))
            s.run(k, lam, outer, inner, variant=S.VARIANT_TILED, precision=precision)
            W, H = s.factors()
            out.append((W[:, :ds.m], H[:, :ds.n], *s.residual()))
    assert np.all(np.isfinite(out[0][0])) and np.any(out[0][0] != 0)
    for x, y in zip(*out):
        assert np.array_equal(x, y)
