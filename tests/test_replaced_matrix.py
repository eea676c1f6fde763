"""A test set that outlives its matrix: ccd_upload of another matrix on the
same context, without a new test set."""
import dataclasses
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = 3


def _data(m, n, nnz, seed):
    from cdmf_amd import data as D
    return D.gen_uniform(m, n, nnz, 200, seed=seed)


def _solve(S, s, ds, variant=3):
    from cdmf_amd import data as D
    s.set_factors(D.initial_col(K, ds.m), np.zeros((K, ds.n), np.float32))
    return s.run(K, 0.05, 2, 2, variant=variant).rmse, s.rmse()


@pytest.mark.parametrize("shape", [(300, 200), (500, 240), (300, 200, "same")])
def test_kept_where_it_fits(shape):
    """The entries mean the same cells in the new matrix, whatever order its
    rows have inside: what a new context with both uploads gives."""
    from cdmf_amd import solver as S
    first = _data(300, 200, 9000, 1)
    second = first if len(shape) == 3 else _data(*shape, 9000, 2)
    assert first.test_row.max() < second.m and first.test_col.max() < second.n
    with S.Solver(0) as s:
        s.upload(first)
        _solve(S, s, first)
        s.upload(second, with_test=False)
        s.upload(second, with_test=False)  # replaced twice before it is used again
        got = _solve(S, s, second)
        again = _solve(S, s, second)
    both = dataclasses.replace(second, test_row=first.test_row, test_col=first.test_col, test_val=first.test_val)
    with S.Solver(0) as s:
        s.upload(both)
        want = _solve(S, s, both)
    assert got == want and again == want and all(math.isfinite(x) for x in got[0])


@pytest.mark.parametrize("shape", [(100, 200), (300, 50), (30, 20)])
def test_dropped_where_it_does_not_fit(shape):
    """No RMSE, as without a test set; a new one is taken as usual."""
    from cdmf_amd import solver as S
    first, second = _data(300, 200, 9000, 1), _data(*shape, 300, 4)
    with S.Solver(0) as s:
        s.upload(first)
        _solve(S, s, first)
        s.upload(second, with_test=False)
        from cdmf_amd import data as D
        s.set_factors(D.initial_col(K, second.m), np.zeros((K, second.n), np.float32))
        assert all(math.isnan(x) for x in s.run(K, 0.05, 2, 2, variant=3).rmse)
        with pytest.raises(S.CCDError, match="no test set"):
            s.rmse()
        s.upload_test(np.array([0]), np.array([0]), np.ones(1))
        assert math.isfinite(s.rmse())
