"""Performance cases of the CCD++ framework: what its users run, from one
new user folded in by a serving loop to two outer iterations over a
480,189 x 17,770 matrix, through the Python entry points of
cdmf_amd.solver and cdmf_amd.foldin.

listed()            the named cases
draw(rng)           one more case of the same ranges
prepare(case, seed) what a user's program holds before the call
run(state)          one pass; returns the results a user would read
work(case)          bytes and operations one pass cannot do without
exact(case, seed)   the same results in 64 bits, without this package's
                    kernels (None where that takes too long)
"""
import dataclasses
import math

import numpy as np
import torch

from cdmf_amd import data as D
from cdmf_amd import foldin as F
from cdmf_amd import solver as S

HIDDEN = 256  # the warm-start network's hidden width (foldin.experiment's default)


def listed():
    return [
        # A serving loop folds in one new user (a couple of hundred ratings
        # against the large shape's items) without allocating: latency.
        dict(name="fold_one_user", kind="fold", entry="noalloc", rows=1, n=17770, k=40, nnz=206, sweeps=20),
        # A serving loop's batch of new users on the 26,744-item shape.
        dict(name="fold_serving_batch", kind="fold", entry="noalloc", rows=777, n=26744, k=64, nnz=101010, sweeps=10),
        # The held-out 10 % of the large shape's users, folded in from zero.
        dict(name="fold_heldout", kind="fold", entry="rows", rows=48019, n=17770, k=40, nnz=9907211, sweeps=20),
        # The same users through the learned warm start on the matrix cores.
        dict(name="warm_heldout", kind="warm", mode=2, rows=48019, n=17770, k=40, nnz=9907211, sweeps=7),
        # One training minibatch of the warm-start network: loss and gradients.
        dict(name="mlp_train_step", kind="mlp_grad", rows=1024, nin=82, nout=40),
        # The network over a large batch of feature rows in FP32.
        dict(name="mlp_forward", kind="mlp_forward", mode=0, rows=48019, nin=82, nout=40),
        # The small configuration, W first: launches and latency.
        dict(name="solve_small", kind="solve", m=2000, n=1000, nnz=45000, k=10, lam=0.05, outer=5, inner=5,
             variant=S.VARIANT_TILED, precision=S.PREC_FP32, order=S.ORDER_W_FIRST),
        # A medium matrix with Solver.run's default (degree-binned) sweeps.
        dict(name="solve_default", kind="solve", m=41871, n=16195, nnz=1500001, k=16, lam=0.05, outer=3, inner=5,
             variant=S.VARIANT_NATIVE, precision=S.PREC_FP32, order=S.ORDER_H_FIRST),
        # The precision study's shape with bfloat16-stored factors.
        dict(name="solve_ml20m_bf16", kind="solve", m=138493, n=26744, nnz=18000237, k=64, lam=0.05, outer=2, inner=5,
             variant=S.VARIANT_TILED, precision=S.PREC_BF16, order=S.ORDER_H_FIRST),
        # The large shape: the first two of the solve's outer iterations.
        dict(name="solve_netflix", kind="solve", m=480189, n=17770, nnz=99072112, k=40, lam=0.05, outer=2, inner=5,
             variant=S.VARIANT_TILED, precision=S.PREC_FP32, order=S.ORDER_H_FIRST),
        # A drop-in user's whole call from host arrays, with the reference's
        # default rank, iterations and lambda (Parameter).
        dict(name="onecall_csr5", kind="onecall", m=60235, n=9815, nnz=5000011, k=10, lam=0.1, outer=5, inner=5),
        # A grid of independent problems in one persistent launch.
        dict(name="batch", kind="batch", count=16, scale=0.5, shapes=4, outer=2),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fold", "fold", "warm", "mlp_grad", "mlp_forward", "solve", "solve", "solve", "onecall", "batch"])
    if kind in ("fold", "warm"):
        n = _logu(rng, 1000, 27000)
        k = rng.choice([8, 10, 16, 32, 40, 64, rng.randint(3, 100)])
        rows = _logu(rng, 1, 48019)
        # mean degree up to 206 as in the large shape, at most half the items
        nnz = min(_logu(rng, 10, 206) * rows, rows * n // 2)
        case = dict(kind=kind, rows=rows, n=n, k=k, nnz=max(nnz, rows), sweeps=_logu(rng, 1, 40))
        if kind == "warm":
            case["mode"] = rng.choice([0, 1, 2, 2])
        else:
            small = rows <= 4096 and nnz <= (1 << 20)
            case["entry"] = rng.choice(["rows", "noalloc"]) if small else "rows"
        return case
    if kind in ("mlp_grad", "mlp_forward"):
        k = rng.choice([8, 16, 32, 40, 64, rng.randint(3, 100)])
        case = dict(kind=kind, rows=_logu(rng, 64, 16384 if kind == "mlp_grad" else 48019), nin=2 * k + 2, nout=k)
        if kind == "mlp_forward":
            case["mode"] = rng.choice([0, 0, 1, 2])
        return case
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(3, 16), scale=rng.uniform(0.05, 0.5),
                    shapes=rng.randint(0, 9999), outer=rng.randint(1, 3))
    m, n = _logu(rng, 1000, 200000), _logu(rng, 500, 27000)
    nnz = min(_logu(rng, 10000, 18000000 if kind == "solve" else 5000000), m * n // 4)
    if nnz < 3 * m:
        m = max(500, nnz // 3)
        nnz = min(nnz, m * n // 4)
    case = dict(kind=kind, m=m, n=n, nnz=nnz, k=rng.choice([8, 10, 16, 32, 40, 64, rng.randint(2, 48)]),
                lam=rng.choice([0.01, 0.05, 0.1]), outer=rng.randint(1, 3), inner=rng.choice([1, 3, 5, 5]))
    if kind == "solve":
        case["variant"] = rng.choice([S.VARIANT_TILED, S.VARIANT_TILED, S.VARIANT_NATIVE, S.VARIANT_BATCHING])
        case["precision"] = rng.choice([S.PREC_FP32, S.PREC_FP32, S.PREC_FP32, S.PREC_BF16, S.PREC_FP64_SUMS])
        case["order"] = rng.choice([S.ORDER_H_FIRST, S.ORDER_H_FIRST, S.ORDER_W_FIRST])
    return case


# --------------------------------------------------------------- inputs ---
def _matrix(case, seed):
    """Power-law ratings 1..5 (the small configuration: uniform positions),
    a twentieth as many test entries, and the reference's start: W from
    initial_col and H = 0, or, W first, W = 0 and H uniform."""
    m, n, nnz, k = case["m"], case["n"], case["nnz"], case["k"]
    test = max(1, nnz // 20)
    if case.get("order") == S.ORDER_W_FIRST and nnz <= 50000:
        ds = D.gen_uniform(m, n, nnz, test, seed=seed)
    else:
        ds = D.gen_powerlaw(m, n, nnz, test, max_row_degree=min(n, 17000), rating_kind=1, seed=seed)
    if case.get("order") == S.ORDER_W_FIRST:
        return ds, np.zeros((k, m), np.float32), D.init_uniform((k, n), 1.0 / math.sqrt(k), seed)
    return ds, D.initial_col(k, m), np.zeros((k, n), np.float32)


def _problems(case, seed):
    """The batch's problems: shapes, k and lambda from the case, ratings from the seed."""
    specs = D.batch_specs(count=case["count"], seed=case["shapes"], scale=case["scale"])
    return [dataclasses.replace(q, seed=1000 * seed + i) for i, q in enumerate(specs)]


def _items(case, seed):
    """Item factors as a solve leaves them: a first rank that carries the
    mean rating, then ranks of falling size around zero."""
    k, n = case["k"], case["n"]
    r = np.random.default_rng([seed, 1])
    H = r.standard_normal((k, n), dtype=np.float32) * (0.5 / np.sqrt(1.0 + np.arange(k, dtype=np.float32)))[:, None]
    H[0] = 1.8 + 0.2 * H[0]
    return np.ascontiguousarray(H)


def _users(case, seed):
    """New users: CSR rows with power-law degrees, ratings 1..5."""
    rows, n, nnz = case["rows"], case["n"], case["nnz"]
    if rows < 8:  # too few rows for the generator's degree law
        r = np.random.default_rng([seed, 2])
        per = [nnz // rows + (1 if i < nnz % rows else 0) for i in range(rows)]
        p = 1.0 / np.arange(1.0, n + 1.0)
        idx = np.concatenate([np.sort(r.choice(n, d, replace=False, p=p / p.sum())) for d in per])
        ptr = np.concatenate([[0], np.cumsum(per)])
        return ptr.astype(np.uint32), idx.astype(np.uint32), r.integers(1, 6, nnz).astype(np.float32)
    ds = D.gen_powerlaw(rows, n, nnz, 1, max_row_degree=min(n, 17000), rating_kind=1, seed=seed)
    return ds.csr_ptr, ds.csr_idx, ds.csr_val


def _params(nin, nout, seed):
    """Flat network parameters (W1, b1, W2, b2, W3, b3), Glorot-uniform
    weights and small biases, as after some training."""
    r = np.random.default_rng([seed, 3])
    out = []
    for fo, fi in ((HIDDEN, nin), (HIDDEN, HIDDEN), (nout, HIDDEN)):
        out.append(r.uniform(-1.0, 1.0, fo * fi) * math.sqrt(6.0 / (fo + fi)))
        out.append(0.05 * r.standard_normal(fo))
    return np.concatenate(out).astype(np.float32)


def _warm_norm(case, H):
    """Feature and target statistics of the training users (their scale)."""
    k = case["k"]
    sd = H.std(axis=1)
    in_mean = np.concatenate([H.mean(axis=1), sd * sd, [4.0, 3.5]])
    in_std = np.concatenate([0.3 * sd, 0.5 * sd * sd, [1.2, 0.4]])
    out_mean = np.zeros(k)
    out_mean[0] = 1.5
    return [a.astype(np.float32) for a in (in_mean, in_std, out_mean, np.full(k, 0.3))]


def _features(rows, width, seed):
    """Raw feature rows for the network."""
    return np.random.default_rng([seed, 4]).standard_normal((rows, width), dtype=np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        ds, W0, H0 = _matrix(case, seed)
        s = S.Solver(0)
        s.upload(ds)
        return dict(case=case, solver=s, W0=W0, H0=H0)
    if kind == "onecall":
        ds, W0, H0 = _matrix(case, seed)
        return dict(case=case, ds=ds, W0=W0, H0=H0)
    if kind == "batch":
        b, solvers, init = S.Batch(0), [], []
        for q in _problems(case, seed):
            ds = D.batch_dataset(q)
            s = S.Solver(0)
            s.set_plan(sigma=16, split_rows=0)  # the batched kernel's tile layouts
            s.upload(ds)
            init.append((D.initial_col(q.solve.k, ds.m), np.zeros((q.solve.k, ds.n), np.float32)))
            s.set_factors(*init[-1])
            b.add(s, q.solve.k, q.solve.lam, case["outer"], q.solve.inner)
            solvers.append(s)
        return dict(case=case, batch=b, solvers=solvers, init=init)
    if kind in ("fold", "warm"):
        H = _items(case, seed)
        st = dict(case=case, fold=F.FoldIn(H, 0.05), users=_users(case, seed))
        if kind == "warm":
            k = case["k"]
            st["mlp"] = F.MLP(2 * k + 2, HIDDEN, k, seed=seed)
            st["mlp"].set_params(_params(2 * k + 2, k, seed))
            st["mlp"].set_norm(*_warm_norm(case, H))
        return st
    mlp = F.MLP(case["nin"], HIDDEN, case["nout"], seed=seed)
    mlp.set_params(_params(case["nin"], case["nout"], seed))
    st = dict(case=case, mlp=mlp, X=_features(case["rows"], case["nin"], seed))
    if kind == "mlp_grad":
        st["T"] = _features(case["rows"], case["nout"], seed + 7919)
    return st


# ----------------------------------------------------------------- pass ---
def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "solve":
        s = st["solver"]
        s.set_factors(st["W0"], st["H0"])
        r = s.run(c["k"], c["lam"], c["outer"], c["inner"], variant=c["variant"], precision=c["precision"],
                  order=c["order"])
        W, H = s.factors()
        return dict(W=W, H=H, rmse=r.rmse)
    if kind == "onecall":
        W, H = st["W0"].copy(), st["H0"].copy()  # the call updates them in place
        p = S.Parameter(k=c["k"], lambda_=c["lam"], maxiter=c["outer"], maxinneriter=c["inner"])
        S.cdmf_csr5(st["ds"], W, H, p)
        return dict(W=W, H=H)
    if kind == "batch":
        for s, (W0, H0) in zip(st["solvers"], st["init"]):
            s.set_factors(W0, H0)
        st["batch"].run()
        return [s.factors() for s in st["solvers"]]
    if kind == "fold":
        call = st["fold"].rows_noalloc if c["entry"] == "noalloc" else st["fold"].rows
        return call(*st["users"], c["sweeps"])[0]
    if kind == "warm":
        return st["fold"].warm(st["mlp"], *st["users"], c["sweeps"], bf16=c["mode"])[0]
    if kind == "mlp_forward":
        return st["mlp"].forward(st["X"], bf16=c["mode"])
    loss, grad = st["mlp"].loss_grad(st["X"], st["T"])
    return dict(loss=loss, grad=grad)


# ----------------------------------------------------------------- work ---
def _solve_work(m, n, nnz, k, outer, inner):
    """Every sweep depends on the one before it, so each reads the residual
    (FP32) and its indices (16 bits) again: 2 inner sweeps a rank, and per
    rank one update of both residual copies.  Per element a sweep takes four
    operations and the residual update of a rank four for each copy."""
    per_rank = (2 * inner * 6 + 2 * 4) * nnz + 4 * (2 * inner + 2) * (m + n)
    return dict(bytes=float(outer * k * per_rank), flops=float(outer * k * (2 * inner * 4 + 2 * 4) * nnz))


def _mlp_ops(rows, nin, nout):
    return 2.0 * rows * (nin * HIDDEN + HIDDEN * HIDDEN + HIDDEN * nout)


def work(case):
    kind = case["kind"]
    if kind in ("solve", "onecall"):
        return _solve_work(case["m"], case["n"], case["nnz"], case["k"], case["outer"], case["inner"])
    if kind == "batch":
        ws = [_solve_work(q.m, q.n, q.nnz - q.nnz // 10, q.solve.k, case["outer"], q.solve.inner)
              for q in _problems(case, 0)]
        return {a: sum(w[a] for w in ws) for a in ("bytes", "flops")}
    if kind in ("fold", "warm"):
        rows, k, nnz, sw = case["rows"], case["k"], case["nnz"], case["sweeps"]
        # the ratings and the item factors in, the user factors out; sweeps
        # over the ratings (8 operations an element and rank) or over the
        # users' normal equations, whichever takes fewer operations
        flops = min(8.0 * nnz * k * sw, 1.0 * nnz * k * (k + 3) + 2.0 * rows * sw * k * k)
        if kind == "warm":
            flops += 4.0 * nnz * k + _mlp_ops(rows, 2 * k + 2, k)
        return dict(bytes=8.0 * nnz + 4.0 * (rows + 1) + 4.0 * k * (case["n"] + rows), flops=flops)
    rows, nin, nout = case["rows"], case["nin"], case["nout"]
    np_ = HIDDEN * nin + HIDDEN * HIDDEN + nout * HIDDEN + 2 * HIDDEN + nout
    if kind == "mlp_forward":
        return dict(bytes=4.0 * (rows * (nin + nout) + np_), flops=_mlp_ops(rows, nin, nout))
    return dict(bytes=4.0 * (rows * (nin + nout) + 2 * np_),
                flops=3.0 * _mlp_ops(rows, nin, nout) - 2.0 * rows * nin * HIDDEN)


# ---------------------------------------------------------------- exact ---
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev()).to(dtype)


def _index(a):
    return torch.from_numpy(np.ascontiguousarray(a).astype(np.int64)).to(_dev())


def _sums(ptr, values):
    """Per-row sums of values in row order: differences of their running sum."""
    total = torch.cat([torch.zeros(1, dtype=torch.float64, device=values.device), values.cumsum(0)])
    return total[ptr[1:]] - total[ptr[:-1]]


def _ccd(ds, W0, H0, k, lam, outer, inner, w_first=False):
    """CCD++ in 64 bits; also the test RMSE after each outer iteration."""
    lam = float(np.float32(lam))
    rptr, cptr = _index(ds.csr_ptr), _index(ds.csc_ptr)
    nr, nc = rptr.diff(), cptr.diff()
    row, col = torch.repeat_interleave(nr), _index(ds.csr_idx)  # CSR order
    crow, ccol = _index(ds.csc_idx), torch.repeat_interleave(nc)  # CSC order
    res, cres = _t(ds.csr_val), _t(ds.csc_val)
    trow, tcol, tval = _index(ds.test_row), _index(ds.test_col), _t(ds.test_val)
    W, H = _t(W0), _t(H0)
    (W if w_first else H).zero_()

    def sweep(x, ptr, r, count):
        y = _sums(ptr, x * r) / (lam * count + _sums(ptr, x * x))
        return torch.where(count > 0, y, torch.zeros_like(y))

    rmse = []
    for o in range(outer):
        for t in range(k):
            u, v = W[t].clone(), H[t].clone()
            if o:
                res += u[row] * v[col]
                cres += u[crow] * v[ccol]
            for _ in range(inner):
                if w_first:
                    u = sweep(v[col], rptr, res, nr)
                v = sweep(u[crow], cptr, cres, nc)
                if not w_first:
                    u = sweep(v[col], rptr, res, nr)
            W[t], H[t] = u, v
            res -= u[row] * v[col]
            cres -= u[crow] * v[ccol]
        pred = sum(W[t][trow] * H[t][tcol] for t in range(k))
        rmse.append(float((pred - tval).square().mean().sqrt()))
    return W.cpu().numpy(), H.cpu().numpy(), rmse


def _gelu(z):
    return 0.5 * z * (1.0 + torch.erf(z * math.sqrt(0.5)))


def _layers(P, nin, nout):
    out, o = [], 0
    for fo, fi in ((HIDDEN, nin), (HIDDEN, HIDDEN), (nout, HIDDEN)):
        out += [P[o:o + fo * fi].reshape(fo, fi), P[o + fo * fi:o + fo * fi + fo]]
        o += fo * fi + fo
    return out


def _net(P, X, nin, nout):
    W1, b1, W2, b2, W3, b3 = _layers(P, nin, nout)
    return _gelu(_gelu(X @ W1.t() + b1) @ W2.t() + b2) @ W3.t() + b3


def _fold(case, seed):
    k, rows, lam = case["k"], case["rows"], float(np.float32(0.05))
    H32 = _items(case, seed)
    ptr, idx, val = _users(case, seed)
    H = _t(H32)
    ptr = _index(ptr)
    d = ptr.diff()
    row, col, r = torch.repeat_interleave(d), _index(idx), _t(val)
    W = torch.zeros((rows, k), dtype=torch.float64, device=_dev())
    if case["kind"] == "warm":
        S1 = _sums(ptr, r)
        ok = (d > 0) & (S1 != 0)
        Ss = torch.where(ok, S1, torch.ones_like(S1))
        X = torch.empty((rows, 2 * k + 2), dtype=torch.float64, device=_dev())
        for t in range(k):
            h = H[t][col]
            mean = torch.where(ok, _sums(ptr, r * h) / Ss, 0.0 * Ss)
            X[:, t] = mean
            X[:, k + t] = torch.where(ok, _sums(ptr, r * h * h) / Ss - mean * mean, 0.0 * Ss).clamp(min=0.0)
        X[:, 2 * k] = torch.log1p(d.double())
        X[:, 2 * k + 1] = S1 / d.clamp(min=1)
        im, isd, om, osd = (_t(a) for a in _warm_norm(case, H32))
        W = _net(_t(_params(2 * k + 2, k, seed)), (X - im) / isd, 2 * k + 2, k) * osd + om
    for t in range(k):
        r = r - W[row, t] * H[t][col]
    for _ in range(case["sweeps"]):
        for t in range(k):
            h = H[t][col]
            a = r + W[row, t] * h
            w = _sums(ptr, a * h) / (lam * d + _sums(ptr, h * h))
            w = torch.where(d > 0, w, torch.zeros_like(w))
            W[:, t] = w
            r = a - w[row] * h
    return W.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "onecall"):
        if float(case["nnz"]) * case["k"] * case["outer"] * case["inner"] > 1.5e9:
            return None
        ds, W0, H0 = _matrix(case, seed)
        W, H, rmse = _ccd(ds, W0, H0, case["k"], case["lam"], case["outer"], case["inner"],
                          case.get("order") == S.ORDER_W_FIRST)
        return dict(W=W, H=H, rmse=rmse) if kind == "solve" else dict(W=W, H=H)
    if kind == "batch":
        out, cost = [], 0.0
        for q in _problems(case, seed):
            cost += float(q.nnz) * q.solve.k * case["outer"] * q.solve.inner
            if cost > 1.5e9:  # the rest have no value here
                out.append((None, None))
                continue
            ds = D.batch_dataset(q)
            W0, H0 = D.initial_col(q.solve.k, ds.m), np.zeros((q.solve.k, ds.n), np.float32)
            out.append(_ccd(ds, W0, H0, q.solve.k, q.solve.lam, case["outer"], q.solve.inner)[:2])
        return out
    if kind in ("fold", "warm"):
        if float(case["nnz"]) * case["k"] * (case["sweeps"] + 2) > 1.2e10:
            return None
        return _fold(case, seed)
    P = _t(_params(case["nin"], case["nout"], seed))
    X = _t(_features(case["rows"], case["nin"], seed))
    if kind == "mlp_forward":
        return _net(P, X, case["nin"], case["nout"]).cpu().numpy()
    P.requires_grad_(True)
    T = _t(_features(case["rows"], case["nout"], seed + 7919))
    loss = (_net(P, X, case["nin"], case["nout"]) - T).square().mean()
    loss.backward()
    return dict(loss=float(loss.detach()), grad=P.grad.cpu().numpy())
