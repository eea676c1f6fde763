"""GPU checks of the fold-in extension against the CPU oracle
(oracle/foldin_oracle.c, pinned in tests/test_oracle_foldin.py).

Bars:
  * features: FP64 sums in the same element order as the oracle, so
    relative 1e-6 (the float rounding of the same doubles);
  * fold-in sweeps: FP32 with a different summation order (wave
    reduction): Frobenius relative 1e-4 and elementwise 1e-3 relative +
    1e-4 rms, from zero and from a warm start, short rows (registers) and
    rows above 1024 ratings (streamed residual); 300 sweeps reach the ridge
    solve within 1e-3;
  * MLP: FP32 GPU forward and gradients against the FP64 oracle at the
    production shape (82 -> 256 -> 256 -> 40), on 96 rows and on 1024 rows
    (the weight-gradient products split K): relative Frobenius 1e-4 per
    parameter tensor, loss within 1e-5 relative; bfloat16-weight inference
    against the oracle run on the bfloat16-rounded weights, 1e-4;
  * training lowers the loss on a smooth regression target tenfold.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gpu():
    from cdmf_amd import foldin, solver
    if solver.device_count() < 1:
        pytest.fail("no HIP device visible: GPU tests need the MI355X")
    return foldin


def _say(msg):
    print(msg, flush=True)


def _rows(seed, rows, n, k, long_rows=0):
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 300, size=rows)
    deg[1] = 0
    for q in range(long_rows):
        deg[2 + q] = 1500 + 700 * q  # above 64 * 16: the streamed path
    deg = np.minimum(deg, n)
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    idx = np.concatenate([np.sort(rng.choice(n, size=d, replace=False)) for d in deg]).astype(np.uint32)
    val = rng.integers(1, 6, size=idx.size).astype(np.float32)
    H = (rng.random((k, n)) * 0.5).astype(np.float32)
    return ptr, idx, val, H


def _close(x, ref, what, frob=1e-4, rtol=1e-3):
    x = np.asarray(x, np.float64)
    ref = np.asarray(ref, np.float64)
    rms = float(np.sqrt(np.mean(ref * ref))) if ref.size else 0.0
    f = np.linalg.norm(x - ref) / max(np.linalg.norm(ref), 1e-300)
    assert f <= frob, "%s: Frobenius relative %.3g > %g" % (what, f, frob)
    np.testing.assert_allclose(x, ref, rtol=rtol, atol=1e-4 * rms, err_msg=what)


def test_features_match_oracle(oracle_lib):
    F = _gpu()
    ptr, idx, val, H = _rows(0, 500, 3000, 40, long_rows=2)
    fold = F.FoldIn(H, 0.05)
    got = fold.features(ptr, idx, val)
    ref = oracle_lib.fold_features(ptr, idx, val, H)
    np.testing.assert_allclose(got, ref, rtol=1e-6, atol=1e-7)
    fold.close()


@pytest.mark.parametrize("sweeps", [1, 5])
def test_fold_rows_match_oracle(oracle_lib, sweeps):
    F = _gpu()
    ptr, idx, val, H = _rows(1, 700, 4000, 40, long_rows=2)
    lam = 0.05
    fold = F.FoldIn(H, lam)
    W, t = fold.rows(ptr, idx, val, sweeps)
    _say("fold %d rows, %d sweeps: %.3f ms" % (ptr.size - 1, sweeps, 1e3 * t))
    _close(W, oracle_lib.fold_rows(ptr, idx, val, H, np.float32(lam), sweeps), "zero start, %d sweeps" % sweeps)
    assert np.all(W[1] == 0.0)
    W0 = (np.random.default_rng(2).normal(0, 0.3, W.shape)).astype(np.float32)
    Ww, _ = fold.rows(ptr, idx, val, sweeps, W0=W0)
    _close(Ww, oracle_lib.fold_rows(ptr, idx, val, H, np.float32(lam), sweeps, W0=W0), "warm start, %d sweeps" % sweeps)
    fold.close()


def test_fold_rows_very_long_row(oracle_lib):
    """A row above 16384 ratings: registers for the first 16384, the rest
    streamed through the global residual buffer."""
    F = _gpu()
    rng = np.random.default_rng(6)
    n, k = 20000, 8
    deg = [17000, 5, 0, 1100]
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    idx = np.concatenate([np.sort(rng.choice(n, size=d, replace=False)) for d in deg]).astype(np.uint32)
    val = rng.integers(1, 6, size=idx.size).astype(np.float32)
    H = (rng.random((k, n)) * 0.5).astype(np.float32)
    fold = F.FoldIn(H, 0.05)
    W, _ = fold.rows(ptr, idx, val, 3)
    _close(W, oracle_lib.fold_rows(ptr, idx, val, H, np.float32(0.05), 3), "very long row")
    np.testing.assert_allclose(fold.features(ptr, idx, val), oracle_lib.fold_features(ptr, idx, val, H), rtol=1e-6,
                               atol=1e-7)
    fold.close()


def _fold_f64(ptr, idx, val, H, lam, sweeps, W0):
    """The sweeps of plain fold-in in FP64, row by row."""
    k = H.shape[0]
    W = np.zeros((ptr.size - 1, k)) if W0 is None else W0.astype(np.float64)
    for i in range(ptr.size - 1):
        s, e = int(ptr[i]), int(ptr[i + 1])
        Ho = H[:, idx[s:e]].astype(np.float64)
        lamd = float(np.float32(lam) * np.float32(e - s))
        r = val[s:e] - W[i] @ Ho
        for _ in range(sweeps):
            for t in range(k):
                a = r + W[i, t] * Ho[t]
                W[i, t] = a @ Ho[t] / (lamd + Ho[t] @ Ho[t]) if e > s else 0.0
                r = a - W[i, t] * Ho[t]
    return W


@pytest.mark.parametrize("k", [1, 7, 8, 16, 17, 40, 63, 64, 65, 80, 81, 100, 127, 128])
def test_fold_rows_normal_equations(k):
    """Row lengths at the edges of a chunk of 64 ratings, of the one-wave
    rows (128) and of the long rows' eight chunks; ranks at the edges of the
    16-wide tiles, of the groups of tile pairs and of the two slots a lane
    holds; from zero and from a start, no sweep, one and three.  The sums
    and sweeps are FP64, so the result is the FP64 one but for its rounding
    to FP32 (6e-8) and, next to zero, 1e-9 of its size."""
    F = _gpu()
    deg = [0, 1, 2, 3, 4, 5, 15, 17, 63, 64, 65, 127, 128, 129, 191, 512, 513, 1025]
    rng = np.random.default_rng(k)
    n = 1200
    ptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    idx = np.concatenate([rng.choice(n, size=d, replace=False) for d in deg]).astype(np.uint32)
    val = rng.integers(1, 6, size=idx.size).astype(np.float32)
    H = rng.normal(0.1, 0.4, (k, n)).astype(np.float32)
    W0 = rng.normal(0, 0.3, (len(deg), k)).astype(np.float32)
    fold = F.FoldIn(H, 0.05)
    for sweeps in (0, 1, 3):
        for start in (None, W0):
            W, _ = fold.rows(ptr, idx, val, sweeps, W0=start)
            ref = _fold_f64(ptr, idx, val, H, 0.05, sweeps, start)
            size = max(float(np.abs(ref).max()), 1e-30)
            np.testing.assert_allclose(W, ref, rtol=6.1e-8, atol=1e-9 * size, err_msg="k=%d sweeps=%d" % (k, sweeps))
    fold.close()


@pytest.mark.parametrize("k", [1, 7, 8, 9, 57, 63, 65, 71, 100, 121])
def test_fold_rows_after_rows_without_a_number(k):
    """Ranks around a whole group of the chain, after rows whose products are
    NaN: what they left on the chip reaches no other call.  Bound as in
    test_fold_rows_normal_equations."""
    F = _gpu()
    rng = np.random.default_rng(k)
    rows, n = 4096, 50
    ptr = (2 * np.arange(rows + 1)).astype(np.uint32)
    idx = np.tile(np.array([0, 1], np.uint32), rows)
    val = np.ones(2 * rows, np.float32)
    wide = F.FoldIn(np.full((128, n), np.nan, np.float32), 0.05)
    H = rng.normal(0.1, 0.4, (k, n)).astype(np.float32)
    fold = F.FoldIn(H, 0.05)
    deg = [1, 5, 20, 40]
    p2 = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    i2 = np.concatenate([rng.choice(n, size=d, replace=False) for d in deg]).astype(np.uint32)
    v2 = rng.integers(1, 6, size=i2.size).astype(np.float32)
    ref = _fold_f64(p2, i2, v2, H, 0.05, 2, None)
    for call in (fold.rows, fold.rows_noalloc):
        bad, _ = wide.rows(ptr, idx, val, 1)
        assert np.isnan(bad).all()
        W, _ = call(p2, i2, v2, 2)
        np.testing.assert_allclose(W, ref, rtol=6.1e-8, atol=1e-9 * float(np.abs(ref).max()))
    wide.close()
    fold.close()


@pytest.mark.parametrize("nnz", [300, 65536, 70000])  # the index check on the host, and on the device
def test_fold_refuses_indices_out_of_range(nnz):
    from cdmf_amd.solver import CCDError
    F = _gpu()
    n = 500
    fold = F.FoldIn(np.ones((4, n), np.float32), 0.05)
    ptr = np.concatenate([np.arange(0, nnz, 250), [nnz]]).astype(np.uint32)
    idx = (np.arange(nnz) % n).astype(np.uint32)
    val = np.ones(nnz, np.float32)
    ok, _ = fold.rows(ptr, idx, val, 1)
    bad = idx.copy()
    bad[nnz // 2] = n
    for call in (fold.rows, fold.rows_noalloc):
        with pytest.raises(CCDError, match="out of range"):
            call(ptr, bad, val, 1)
    with pytest.raises(CCDError, match="out of range"):
        fold.features(ptr, bad, val)
    again, _ = fold.rows_noalloc(ptr, idx, val, 1)
    assert np.array_equal(ok, again)
    fold.close()


def test_fold_rows_reach_ridge_solution():
    F = _gpu()
    ptr, idx, val, H = _rows(3, 60, 500, 8)
    lam = 0.1
    fold = F.FoldIn(H, lam)
    W, _ = fold.rows(ptr, idx, val, 300)
    for i in range(ptr.size - 1):
        s, e = int(ptr[i]), int(ptr[i + 1])
        if e == s:
            continue
        Ho = H[:, idx[s:e]].astype(np.float64)
        ref = np.linalg.solve(Ho @ Ho.T + lam * (e - s) * np.eye(H.shape[0]), Ho @ val[s:e].astype(np.float64))
        np.testing.assert_allclose(W[i], ref, rtol=1e-3, atol=1e-4)
    fold.close()


def _split(P, dims):
    nin, hid, out = dims
    sizes = [hid * nin, hid, hid * hid, hid, out * hid, out]
    return np.split(np.asarray(P), np.cumsum(sizes)[:-1])


@pytest.mark.parametrize("rows", [96, 1024])  # 1024: the weight gradients split K over slices
def test_mlp_forward_and_gradients_match_oracle(oracle_lib, rows):
    F = _gpu()
    dims = (82, 256, 40)
    mlp = F.MLP(*dims, seed=7)
    P = mlp.get_params().astype(np.float64)
    rng = np.random.default_rng(4)
    Xn = rng.normal(0, 1, (rows, dims[0])).astype(np.float32)
    Tn = rng.normal(0, 1, (rows, dims[2])).astype(np.float32)
    loss, G = mlp.loss_grad(Xn, Tn)
    rloss, RG = oracle_lib.mlp_backward(P, Xn.astype(np.float64), Tn.astype(np.float64), dims)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss)
    for q, (g, r) in enumerate(zip(_split(G, dims), _split(RG, dims))):
        f = np.linalg.norm(g - r) / np.linalg.norm(r)
        _say("gradient tensor %d: relative %.2e" % (q, f))
        assert f <= 1e-4, "gradient tensor %d: %.3g" % (q, f)
    # forward with standardisation, FP32 and bfloat16 weights
    X = rng.normal(3, 2, (300, dims[0])).astype(np.float32)
    mu, sd = X.mean(0), X.std(0)
    omu, osd = rng.normal(0, 1, dims[2]).astype(np.float32), rng.uniform(0.5, 2, dims[2]).astype(np.float32)
    mlp.set_norm(mu, sd, omu, osd)
    Xn64 = (X.astype(np.float64) - mu) / sd.astype(np.float64)
    ref = oracle_lib.mlp_forward(P, Xn64, dims) * osd + omu
    _close(mlp.forward(X), ref, "forward fp32", frob=1e-5, rtol=1e-4)
    Pb = np.array([oracle_lib.bf16(float(x)) for x in P.astype(np.float32)])
    refb = oracle_lib.mlp_forward(Pb, Xn64, dims) * osd + omu
    _close(mlp.forward(X, bf16=True), refb, "forward bf16 weights", frob=1e-4, rtol=1e-3)
    mlp.close()


def test_mlp_training_lowers_loss():
    F = _gpu()
    rng = np.random.default_rng(5)
    X = rng.normal(0, 1, (8192, 12)).astype(np.float32)
    A = rng.normal(0, 0.5, (12, 4))
    T = (np.tanh(X @ A) + 0.1 * np.sin(3 * X[:, :4])).astype(np.float32)
    mlp = F.MLP(12, 64, 4, seed=1)
    mlp.set_norm(X.mean(0), X.std(0), T.mean(0), T.std(0))
    first = mlp.train(X, T, epochs=1, batch=256, lr=1e-3, seed=1)
    last = mlp.train(X, T, epochs=15, batch=256, lr=1e-3, seed=2)
    _say("training loss %.4f -> %.4f" % (first, last))
    assert last < 0.1 * first
    mlp.close()


@pytest.mark.parametrize("dims,rows", [((1, 1, 1), 1), ((1, 17, 3), 15), ((5, 16, 1), 16), ((18, 33, 8), 17),
                                       ((82, 256, 40), 513), ((30, 100, 14), 2049), ((82, 256, 40), 16400),
                                       ((12, 64, 5), 66000)])
def test_mlp_gemm_shapes(oracle_lib, dims, rows):
    """Products at the edges of the 16- and 64-wide tiles and of a step of 16
    K values, a single row, unit or output (every operand then has two unit
    strides), weight gradients over a K of one wave, of 16 and of several
    slices, inference in one chunk and in two: against the FP64 oracle.
    FP32 sums of up to 66,000 terms of mixed sign through three layers:
    relative Frobenius 2e-5 per tensor, loss 1e-5."""
    F = _gpu()
    rng = np.random.default_rng(rows)
    mlp = F.MLP(*dims, seed=3)
    nin, hid, nout = dims
    P = mlp.get_params()
    P += rng.normal(0, 0.05, P.size).astype(np.float32)
    mlp.set_params(P)
    P = P.astype(np.float64)
    X = rng.normal(0, 1, (rows, nin)).astype(np.float32)
    T = rng.normal(0, 1, (rows, nout)).astype(np.float32)
    loss, G = mlp.loss_grad(X, T)
    rloss, RG = oracle_lib.mlp_backward(P, X.astype(np.float64), T.astype(np.float64), dims)
    assert abs(loss - rloss) <= 1e-5 * abs(rloss)
    for q, (g, r) in enumerate(zip(_split(G, dims), _split(RG, dims))):
        f = np.linalg.norm(g - r) / max(np.linalg.norm(r), 1e-30)
        assert f <= 2e-5, "gradient tensor %d: %.3g" % (q, f)
    mu, sd = rng.normal(0, 1, nin).astype(np.float32), rng.uniform(0.5, 2, nin).astype(np.float32)
    omu, osd = rng.normal(0, 1, nout).astype(np.float32), rng.uniform(0.5, 2, nout).astype(np.float32)
    mlp.set_norm(mu, sd, omu, osd)
    ref = oracle_lib.mlp_forward(P, (X.astype(np.float64) - mu) / sd.astype(np.float64), dims) * osd + omu
    for mode, bar in ((0, 2e-6), (1, 1e-2)):  # 1: weights rounded to bfloat16 (2^-9)
        Y = mlp.forward(X, bf16=mode)
        f = np.linalg.norm(Y - ref) / np.linalg.norm(ref)
        assert f <= bar, "forward mode %d: %.3g" % (mode, f)
    mlp.close()


@pytest.mark.parametrize("k", [3, 65])
def test_fold_rows_past_one_grid_row(k):
    """More rows than one row of the sweeps' grid (2^20): the rows at its end
    and past it.  Bound as in test_fold_rows_normal_equations."""
    F = _gpu()
    rows, n = (1 << 20) + 5, 300
    rng = np.random.default_rng(k)
    ptr = np.arange(rows + 1, dtype=np.uint32)
    idx = rng.integers(0, n, rows).astype(np.uint32)
    val = rng.integers(1, 6, rows).astype(np.float32)
    H = rng.normal(0.1, 0.4, (k, n)).astype(np.float32)
    fold = F.FoldIn(H, 0.05)
    W, _ = fold.rows(ptr, idx, val, 2)
    fold.close()
    sel = np.r_[0:3, (1 << 20) - 3:rows]
    ref = _fold_f64(np.arange(sel.size + 1, dtype=np.uint32), idx[sel], val[sel], H, 0.05, 2, None)
    np.testing.assert_allclose(W[sel], ref, rtol=6.1e-8, atol=1e-9 * float(np.abs(ref).max()))


def test_warm_refused_after_the_upload():
    """A network or a mode that is refused once the batch is on its way: the
    caller may reuse its arrays at once, and the next call is right."""
    import torch

    from cdmf_amd.solver import CCDError
    F = _gpu()
    rng = np.random.default_rng(3)
    k, n, rows = 8, 500, 300
    ptr = (np.arange(rows + 1) * 20).astype(np.uint32)
    idx = rng.integers(0, n, rows * 20).astype(np.uint32)
    val = torch.empty(rows * 20, pin_memory=True).numpy()  # memory the device reads in place
    want_val = rng.integers(1, 6, rows * 20).astype(np.float32)
    H = rng.normal(0.1, 0.4, (k, n)).astype(np.float32)
    fold, narrow, wide = F.FoldIn(H, 0.05), F.MLP(2 * k + 2, 64, k, seed=1), F.MLP(2 * k + 2, 256, k, seed=1)
    val[:] = want_val
    want, _ = fold.warm(wide, ptr, idx, val, 2, bf16=2)
    for mlp, mode in ((narrow, 2), (wide, 3), (wide, -1)):
        val[:] = want_val
        with pytest.raises(CCDError):
            fold.warm(mlp, ptr, idx, val, 2, bf16=mode)
        val[:] = -1.0
        with pytest.raises(CCDError):
            mlp.forward(np.zeros((100, 2 * k + 2), np.float32), bf16=mode)
    val[:] = want_val
    got, _ = fold.warm(wide, ptr, idx, val, 2, bf16=2)
    assert np.array_equal(got, want)
    for x in (fold, narrow, wide):
        x.close()


def test_mlp_forward_gives_large_buffers_back():
    """1.1 GB of rows and outputs: what the device has free after the call is
    what it had before, and the rows are those of smaller calls."""
    import torch
    F = _gpu()
    mlp = F.MLP(82, 256, 40, seed=2)
    X = np.random.default_rng(1).standard_normal((1 << 16, 82), dtype=np.float32)
    want = mlp.forward(X, bf16=2)
    reps = 35  # 35 x 65,536 x 122 floats
    big = np.concatenate([X] * reps)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    got = mlp.forward(big, bf16=2)
    assert torch.cuda.mem_get_info()[0] >= before - (64 << 20)
    assert all(np.array_equal(got[i << 16:(i + 1) << 16], want) for i in (0, 17, reps - 1))
    assert np.array_equal(mlp.forward(X, bf16=2), want)
    mlp.close()


@pytest.mark.parametrize("k", [1, 8, 40, 65, 128])
def test_fold_rows_with_factors_that_are_not_finite(k):
    """An item factor that is NaN or infinite: the rows that rate the item are
    no number where the sweeps over the residual make them so (every rank: the
    residual starts as r - W0 h), the others are as without it."""
    F = _gpu()
    rng = np.random.default_rng(k)
    deg = [1, 5, 64, 70, 128, 129, 600]
    n = 700
    ptr = np.concatenate([[0], np.cumsum(2 * deg)]).astype(np.uint32)
    # the first seven rows rate item 0, the others do not
    idx = np.concatenate([np.append(0, 1 + rng.choice(n - 1, size=d - 1, replace=False)) for d in deg]
                         + [1 + rng.choice(n - 1, size=d, replace=False) for d in deg]).astype(np.uint32)
    val = rng.integers(1, 6, size=idx.size).astype(np.float32)
    H = rng.normal(0.1, 0.4, (k, n)).astype(np.float32)
    W0 = rng.normal(0, 0.3, (len(ptr) - 1, k)).astype(np.float32)
    for what in (np.nan, np.inf, -np.inf):
        for rank in sorted({0, k // 2, k - 1}):
            Hx = H.copy()
            Hx[rank, 0] = what
            fold = F.FoldIn(Hx, 0.05)
            for sweeps in (0, 1, 2):
                for start in (None, np.zeros_like(W0), W0):
                    W, _ = fold.rows(ptr, idx, val, sweeps, W0=start)
                    with np.errstate(all="ignore"):
                        ref = _fold_f64(ptr, idx, val, Hx, 0.05, sweeps, start)
                    assert np.array_equal(np.isfinite(W), np.isfinite(ref)), (what, rank, sweeps, start is None)
                    ok = np.isfinite(ref)
                    np.testing.assert_allclose(W[ok], ref[ok], rtol=6.1e-8, atol=1e-9 * max(1.0, np.abs(ref[ok]).max()))
            fold.close()
