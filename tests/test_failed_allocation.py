"""A call that fails for want of device memory fails alone: the next call on
the same thread, on that object or another, is right."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_the_next_call_is_right():
    from cdmf_amd import data as D
    from cdmf_amd import foldin as F
    from cdmf_amd import solver as S
    ds = D.gen_uniform(300, 200, 3000, 100, seed=1)
    k = 4
    W0, H0 = D.initial_col(k, ds.m), np.zeros((k, ds.n), np.float32)
    ptr, idx, val = np.array([0, 3], np.uint32), np.array([1, 5, 9], np.uint32), np.ones(3, np.float32)

    def solve(s):
        s.upload(ds)
        s.set_factors(W0, H0)
        s.run(k, 0.05, 2, 2, variant=S.VARIANT_TILED)
        return s.factors()

    with S.Solver(0) as s, S.Solver(0) as other:
        want = solve(other)
        fold = F.FoldIn(want[1], 0.05)
        want_row = fold.rows(ptr, idx, val, 2)[0]

        def fail():
            with pytest.raises(S.CCDError, match="memory"):
                s.copy_probe(1 << 46)  # 64 TB

        for who in (s, other):
            fail()
            got = solve(who)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        fail()
        assert np.array_equal(fold.rows(ptr, idx, val, 2)[0], want_row)
        fail()
        b = S.Batch(0)
        s.set_factors(W0, H0)
        b.add(s, k, 0.05, 2, 2)
        b.run()
        b.close()
        fold.close()
        fail()  # nothing is left behind for torch either
        import torch
        assert float(torch.ones(8, device="cuda").sum()) == 8.0


def test_factors_that_do_not_fit():
    """ccd_set_factors of a rank too large for the device: the old factors are
    gone, so what needs factors says so; new ones are taken as usual."""
    import ctypes as C

    from cdmf_amd import data as D
    from cdmf_amd import datadir
    from cdmf_amd import solver as S
    m = n = 1 << 20
    i = np.arange(2000) * 500
    ds = datadir.from_triplets(m, n, (i, i[::-1].copy(), np.ones(i.size)), (i[:5], i[:5], np.ones(5)))
    W0, H0 = D.initial_col(2, m), np.zeros((2, n), np.float32)
    with S.Solver(0) as s:
        s.upload(ds)
        s.set_factors(W0, H0)
        s.run(2, 0.05, 1, 1, variant=S.VARIANT_TILED)
        want = s.factors()
        one = np.zeros(1, np.float32)  # not read: 800 GB of factors are refused first
        p = one.ctypes.data_as(C.POINTER(C.c_float))
        with pytest.raises(S.CCDError, match="memory"):
            s._check(s._lib.ccd_set_factors(s._ctx, 1 << 16, p, p))
        for call in (s.factors, s.rmse, lambda: s.objective(0.1), lambda: s.run(2, 0.05, 1, 1),
                     lambda: s.run(0, 0.05, 1, 1)):
            with pytest.raises(S.CCDError, match="factors"):
                call()
        s.set_factors(W0, H0)
        s.run(2, 0.05, 1, 1, variant=S.VARIANT_TILED)
        got = s.factors()
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_a_workspace_that_does_not_fit():
    """With the device nearly full, a training step whose workspace does not
    fit fails part way through its allocation; a small one after it is right."""
    import torch

    from cdmf_amd import foldin as F
    from cdmf_amd import solver as S
    r = np.random.default_rng(1)
    X, T = r.standard_normal((1 << 19, 34), dtype=np.float32), r.standard_normal((1 << 19, 16), dtype=np.float32)
    mlp = F.MLP(34, 256, 16, seed=1)
    want = mlp.loss_grad(X[:100], T[:100])
    torch.cuda.synchronize()
    # room for two or three of the six hidden-layer arrays of 512 MB
    full = torch.empty(torch.cuda.mem_get_info()[0] - (1400 << 20), dtype=torch.uint8, device="cuda")
    with pytest.raises(S.CCDError, match="memory"):
        mlp.loss_grad(X, T)
    got = mlp.loss_grad(X[:100], T[:100])
    assert got[0] == want[0] and np.array_equal(got[1], want[1])
    del full
    torch.cuda.empty_cache()
    mlp.close()
