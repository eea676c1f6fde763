"""Long rows that hold an index twice: their elements come out in (index,
caller's position) order, whatever order the caller interleaves the indices
in."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _both(lengths, n, seed, distinct=None):
    """Rows of random columns (below `distinct`) in random order, and the same
    rows with their elements sorted by column, equal ones in the first's
    order: equal inside, element for element."""
    from cdmf_amd import datadir
    r = np.random.default_rng(seed)
    m, nnz = len(lengths), sum(lengths)
    rows = np.repeat(np.arange(m), lengths)
    cols = r.integers(0, distinct or n, nnz) * (n // (distinct or n))
    vals = r.standard_normal(nnz).astype(np.float32)

    def ptr(i, size):
        return np.concatenate([[0], np.cumsum(np.bincount(i, minlength=size))]).astype(np.uint32)

    by_col = np.argsort(cols, kind="stable")  # columns hold their rows' elements in the first's order
    z = np.zeros(1, np.uint32)
    one = datadir.Dataset(m, n, ptr(rows, m), cols.astype(np.uint32), vals, ptr(cols, n),
                          rows[by_col].astype(np.uint32), vals[by_col], z, z, np.ones(1, np.float32))
    o = np.lexsort((np.arange(nnz), cols, rows))
    return one, dataclasses.replace(one, csr_idx=one.csr_idx[o], csr_val=vals[o])


# one, two, three and four digit passes (n up to 2^8, 2^16, 2^24 and past it)
# at their bounds; rows about the block's and a wave's steps of the sort;
# one column only, and a few that repeat often
@pytest.mark.parametrize("n,lengths,distinct", [
    (1, [257, 1024, 5000], None), (2, [300], None), (256, [257, 1023, 1024, 1025, 3000], None),
    (257, [300, 2049, 20000], None), (65536, [257, 70000], 9), (65536, [4096, 200000], None),
    (65537, [1025, 1088, 40000], 300), (1 << 24, [1025, 5000], 700), ((1 << 24) + 1, [2000, 300000], 50000),
    (70001, [3000000, 300, 5000], None)])
def test_order_inside_a_row(n, lengths, distinct):
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    out = []
    for ds in _both(lengths, n, n % 1000 + len(lengths), distinct):
        with S.Solver(0) as s:
            s.upload(ds, with_test=False)
            a, b = s.residual()
            assert np.array_equal(a, ds.csr_val) and np.array_equal(b, ds.csc_val)
            s.set_factors(D.initial_col(2, ds.m), np.zeros((2, n), np.float32))
            s.run(2, 0.05, 1, 2, variant=S.VARIANT_TILED)
            out.append(s.factors())
    assert np.all(np.isfinite(out[0][0])) and np.any(out[0][0] != 0)
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
