"""Degree-binned sweeps (variant 1) at the edges of their work units: rows of
every remainder of a four-element group and of a 16-byte group's alignment,
the bounds of the lane groups, a whole number of groups in flight and one
more, and rows just below and above the split into pieces; small matrices,
where the units shrink to a pass each, against one whose units do not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(lengths, n, seed):
    from cdmf_amd import datadir
    r = np.random.default_rng(seed)
    lengths = r.permutation(lengths)
    rows = np.repeat(np.arange(len(lengths)), lengths)
    cols = np.concatenate([r.choice(n, size=d, replace=False) for d in lengths])
    val = r.integers(1, 6, rows.size).astype(np.float32)
    return datadir.from_triplets(len(lengths), n, (rows, cols, val), (rows[:7], cols[:7], val[:7]))


LENGTHS = list(range(0, 21)) + [31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 131, 255, 256, 257, 1023, 1024, 1025, 1027,
                                4096, 4099, 8191, 8192, 8193, 12289]


@pytest.mark.parametrize("copies,unit_elems", [(1, 4096), (1, 64), (40, 4096)])
@pytest.mark.parametrize("precision", [0, 2])
def test_row_lengths_match_oracle(copies, unit_elems, precision):
    """W, H and the residual against the FP64 oracle.  FP32 tree sums of up
    to 12,289 terms through two outer iterations of two sweeps: 1e-4
    relative (FP64 sums: the stored FP32 factors and residual only, 2e-5)."""
    import oracle
    from cdmf_amd import data as D
    from cdmf_amd import solver as S
    short = [d for d in LENGTHS if d <= 131]
    ds = _matrix(LENGTHS + short * (copies - 1), 16000, seed=copies)
    k, lam, outer, inner = 2, 0.1, 2, 2
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    Wo, Ho, _, ro, co = oracle.ccd(ds, W0, H0, k, lam, outer, inner, dtype="f64")
    with S.Solver(0) as s:
        s.set_plan(unit_elems=unit_elems)
        s.upload(ds)
        s.set_factors(W0, H0)
        s.run(k, lam, outer, inner, variant=S.VARIANT_NATIVE, precision=precision)
        W, H = s.factors()
        a, b = s.residual()
    tol = 1e-4 if precision == 0 else 2e-5
    for got, ref, what in ((W, Wo, "W"), (H, Ho, "H"), (a, ro, "CSR residual"), (b, co, "CSC residual")):
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err <= tol, "%s: %.3g" % (what, err)
