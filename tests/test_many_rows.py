"""Uploads of more rows than the set-up kernels have waves or blocks for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _regular(m, n, per, seed=0):
    """m rows of `per` ratings each: row i holds columns (i + j c) % n, j <
    per, in falling order of j; both copies by arithmetic, no sort.  n must
    divide m and c = n // per."""
    from cdmf_amd import datadir
    c = n // per
    assert m % n == 0 and c >= 1
    csr_idx = ((np.arange(m, dtype=np.int64)[:, None] + c * np.arange(per)[None, ::-1]) % n).astype(np.uint32).ravel()
    csr_ptr = (np.arange(m + 1, dtype=np.int64) * per).astype(np.uint32)
    # column x holds rows i = (x - j c) mod n + q n
    first = (np.arange(n, dtype=np.int64)[:, None] - c * np.arange(per)[None, :]) % n
    csc_idx = (first[:, :, None] + n * np.arange(m // n)[None, None, :]).astype(np.uint32).ravel()
    csc_ptr = (np.arange(n + 1, dtype=np.int64) * (per * (m // n))).astype(np.uint32)
    val = np.arange(m * per, dtype=np.uint32).view(np.float32)  # any bits: set-up only moves them
    z = np.zeros(1, np.uint32)
    return datadir.Dataset(m, n, csr_ptr, csr_idx, val, csc_ptr, csc_idx, val, z, z, np.ones(1, np.float32))


# 16,384 blocks of four waves: 65,536 short rows at once; 16,384 rows of more
# than 64 ratings; and more short rows than one launch has threads for at a
# wave a row (2^26)
@pytest.mark.parametrize("m,n,per", [(65600, 100, 1), (140000, 1000, 3), (16400, 100, 65), (33000, 1000, 70),
                                     ((1 << 26) + 4096, 2048, 1)])
def test_every_element_arrives(m, n, per):
    from cdmf_amd import solver as S
    ds = _regular(m, n, per)
    with S.Solver(0) as s:
        s.upload(ds, with_test=False)
        a, b = s.residual()
    assert np.array_equal(a.view(np.uint32), ds.csr_val.view(np.uint32))
    assert np.array_equal(b.view(np.uint32), ds.csc_val.view(np.uint32))


@pytest.mark.parametrize("m,n,per", [(140000, 1000, 3), (33000, 1000, 70)])
def test_rows_sorted_past_the_first_round(m, n, per):
    """The order inside the rows does not reach the results."""
    import dataclasses

    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    ds = dataclasses.replace(_regular(m, n, per), csr_val=np.ones(m * per, np.float32),
                             csc_val=np.ones(m * per, np.float32))
    flip = dataclasses.replace(ds, csr_idx=np.ascontiguousarray(ds.csr_idx.reshape(m, per)[:, ::-1]).ravel())
    out = []
    for one in (ds, flip):
        with S.Solver(0) as s:
            s.upload(one, with_test=False)
            s.set_factors(D.initial_col(2, m), np.zeros((2, n), np.float32))
            s.run(2, 0.05, 1, 2, variant=S.VARIANT_TILED)
            out.append(s.factors())
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
