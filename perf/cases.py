"""What the engine is timed on: its public entry points over the range of workloads it is used for.

    listed()            the named cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the state a program holds before the call (engine, data, factors), from the seed alone
    run(state)          one pass, and its outputs
    work(case)          bytes and operations a pass cannot do without
    tolerance(case)     what another correct implementation at the same precision may differ by
    exact(case, seed)   the outputs in 64 bits, by plain torch

The rating matrices follow the package's workloads (toy_1k, ml10m_shape, ml_latest_shape, netflix_shape: the same
sizes, row laws, item popularity and rating scales), drawn on the GPU so that a state is quick to make. The factors
are those of a run under way: the planted model's, rotated into f columns, with noise.

Outputs that are factor matrices are the engine's own device buffers, on the stream of the state.
"""
import math

import numpy as np
import torch

import cuda_als_amd as ca
from cuda_als_amd.autograd import half_sweep
from cuda_als_amd.engine import Engine, Group, cg_update_x, make_config

LAM = 0.05
USERS, ITEMS = ca.ALS_SIDE_USERS, ca.ALS_SIDE_ITEMS
SOLVERS = {  # name: (solver, refinement steps, warm start)
    "lu": (ca.SolveType.LU, 0, False),
    "chol": (ca.SolveType.CHOL, 0, False),
    "refined": (ca.SolveType.CHOL, 2, False),
    "warm": (ca.SolveType.CHOL, 1, True),
    "cg": (ca.SolveType.CUMF_ALS_CG_FP32, 0, False),
    "cg16": (ca.SolveType.CUMF_ALS_CG_FP16, 0, False),
}
PRECS = {"fp32": ca.Prec.FP32, "bf16": ca.Prec.BF16, "fp16": ca.Prec.FP16}


def listed():
    return [
        # the smallest run there is: training with the error reported after each sweep (1,000 x 500, FP32, LU)
        dict(name="toy_train", kind="train", m=1000, n=500, nnz=18000, sigma=0.0, f=16, prec="fp32", solve="lu"),
        # the headline: mixed precision at the netflix shape, tuned, replayed from a graph
        dict(name="netflix_mixed", kind="sweep", m=480189, n=17770, nnz=99072112, sigma=1.2484, f=100, prec="fp16",
             solve="warm", tuned=True),
        # the plain FP32 Cholesky path that it is compared with, on a quarter of the users
        dict(name="netflix_fp32", kind="sweep", m=120047, n=17770, nnz=24768028, sigma=1.2484, f=100, prec="fp32",
             solve="chol"),
        # the reference's own configuration for this data: f = 80, 16-bit Gram, FP32 CG of 6 iterations
        dict(name="ml10m_cg_f80", kind="sweep", m=69878, n=10677, nnz=9000048, sigma=1.3, f=80, prec="fp16",
             solve="cg"),
        # its solver on the FP32 Gram
        dict(name="ml10m_cg_fp32", kind="sweep", m=69878, n=10677, nnz=9000048, sigma=1.3, f=100, prec="fp32",
             solve="cg"),
        # FP32 at a common rank, as a program trains that sets nothing but f
        dict(name="ml10m_fp32_f64", kind="sweep", m=69878, n=10677, nnz=9000048, sigma=1.3, f=64, prec="fp32",
             solve="chol"),
        # 16-bit Gram with two steps of classic refinement
        dict(name="ml10m_refined_f64", kind="sweep", m=69878, n=10677, nnz=9000048, sigma=1.3, f=64, prec="fp16",
             solve="refined"),
        # three models over one matrix, one launch per half-sweep
        dict(name="ml10m_group", kind="group", m=69878, n=10677, nnz=9000048, sigma=1.3, f=32, f2=64, f3=128,
             prec="bf16", solve="warm"),
        # forward and backward of the differentiable half-sweep, lambda per user
        dict(name="ml_latest_grad", kind="grad", m=283228, n=58098, nnz=24978100, sigma=1.5386, f=64, prec="fp16",
             solve="chol"),
        # folding in one batch of users: the exact solve of a range of rows
        dict(name="ml10m_rows", kind="rows", m=69878, n=10677, nnz=9000048, sigma=1.3, f=100, prec="fp32",
             solve="chol", first=20011, count=2000),
        # train and test error of a model
        dict(name="ml10m_rmse", kind="rmse", m=69878, n=10677, nnz=9000048, sigma=1.3, f=100, prec="fp32",
             solve="chol"),
        # batched CG on the caller's matrices, 6 iterations
        dict(name="cg_batch_f100", kind="cg_batch", batch=8192, f=100, half=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sweep", "sweep", "sweep", "sweep", "train", "group", "grad", "rows", "rmse", "cg_batch"])
    f = rng.choice([16, 32, 64, 80, 100, 128, rng.randint(5, 143), rng.randint(5, 143)])
    if kind == "cg_batch":
        return dict(kind=kind, batch=_log_int(rng, 20, 8192), f=f, half=rng.random() < 0.5)
    m, n = _log_int(rng, 500, 120000), _log_int(rng, 300, 30000)
    per_row = min(_log_int(rng, 8, 250), n // 6)
    case = dict(kind=kind, m=m, n=n, nnz=max(m * per_row, 2000), sigma=round(rng.uniform(0.0, 1.5), 3), f=f)
    case["prec"] = rng.choice(["fp32", "fp32", "bf16", "fp16"])
    case["solve"] = (rng.choice(["lu", "chol"]) if kind in ("rows", "rmse", "grad") else
                     rng.choice(["lu", "chol", "cg"]) if case["prec"] == "fp32" else
                     rng.choice(["chol", "refined", "warm", "warm", "cg", "cg16"]))
    if kind == "rows":
        case["first"] = rng.randint(0, m // 2)
        case["count"] = rng.randint(1, m // 2)
    if kind == "group":
        case["f2"], case["f3"] = rng.choice([16, 48, 64, 100]), rng.randint(5, 143)
    if kind == "grad":
        case["f"] = min(f, 100)
    return case


# ---------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _ratings(case, seed):
    """The rating matrix and test set of a case (host arrays) and the planted factors (m x 9 and n x 9, device)."""
    g = _generator(seed)
    m, n, nnz = case["m"], case["n"], case["nnz"]
    dev = torch.device("cuda")
    # row lengths: lognormal (uniform draws of users where sigma is 0), scaled to the total
    w = torch.exp(case["sigma"] * torch.randn(m, device=dev, generator=g, dtype=torch.float64))
    w *= nnz / w.sum()
    count = torch.clamp(torch.floor(w + torch.rand(m, device=dev, generator=g, dtype=torch.float64)), 1, 0.6 * n).long()
    # items by popularity (Zipf), a pair counted once: draw more than wanted, keep what is new up to each row's length
    cdf = torch.cumsum(1.0 / torch.arange(1, n + 1, device=dev, dtype=torch.float64), 0)
    cdf /= cdf[-1].clone()
    perm = torch.randperm(n, device=dev, generator=g)
    more = (count.double() * 1.15).long() + 1
    rows = torch.repeat_interleave(torch.arange(m, device=dev), more)
    items = perm[torch.searchsorted(cdf, torch.rand(rows.numel(), device=dev, generator=g, dtype=torch.float64)
                                    ).clamp_(max=n - 1)]
    key = torch.unique(rows * n + items)
    rows = key // n
    start = torch.searchsorted(rows, torch.arange(m, device=dev))
    place = torch.arange(key.numel(), device=dev) - start[rows]
    have = torch.bincount(rows, minlength=m)
    # a random run of a row's items rather than its first ones
    shift = (torch.rand(m, device=dev, generator=g) * have).long()
    key = key[(place - shift[rows]) % have[rows] < count[rows]]
    n_test = max(1, key.numel() // 10)
    rows, items = key // n, key % n
    # ratings: a planted model with a mean of 3, half stars from 0.5 to 5
    rank = 8
    pu = torch.cat([torch.full((m, 1), math.sqrt(3.0), device=dev),
                    torch.randn(m, rank, device=dev, generator=g) / math.sqrt(rank)], 1)
    pv = torch.cat([torch.full((n, 1), math.sqrt(3.0), device=dev),
                    torch.randn(n, rank, device=dev, generator=g) / math.sqrt(rank)], 1)

    def rated(r, c):
        s = torch.zeros(r.numel(), device=dev)
        for j in range(rank + 1):
            s += pu[r, j] * pv[c, j]
        s += 0.8 * torch.randn(r.numel(), device=dev, generator=g)
        return (torch.round(2 * s) / 2).clamp_(0.5, 5.0)

    val = rated(rows, items)
    t_rows = torch.sort(torch.randint(0, m, (n_test,), device=dev, generator=g))[0]
    t_items = torch.randint(0, n, (n_test,), device=dev, generator=g)
    t_val = rated(t_rows, t_items)
    order = torch.sort(items * m + rows)[1]

    def ptr(x, size):
        return torch.cat([torch.zeros(1, device=dev, dtype=torch.long), torch.cumsum(torch.bincount(x, minlength=size), 0)])

    def host(x):
        return x.to(torch.int32 if x.dtype == torch.int64 else torch.float32).cpu().numpy()

    data = ca.RatingData(m, n, host(ptr(rows, m)), host(items), host(val), host(ptr(items, n)), host(rows[order]),
                         host(val[order]), host(t_rows), host(t_items), host(t_val))
    return data, pu, pv


def _factors(case, f, seed, pu, pv):
    """Host factors of a run under way: the planted ones in f columns (an orthonormal mix of them), with noise."""
    g = _generator(seed * 7 + f)
    k = pu.shape[1]
    q = torch.linalg.qr(torch.randn(max(f, k), k, device="cuda", generator=g))[0][:f]

    def side(p):
        return (p @ q.T + 0.1 * torch.randn(p.shape[0], f, device="cuda", generator=g)).cpu().numpy()

    return side(pu), side(pv)


class _Buffer:
    """A device matrix of the engine, which it keeps alive."""

    def __init__(self, engine, side):
        self.engine = engine
        rows, ld = (engine.m if side == USERS else engine.n), engine.info().ld
        self.__cuda_array_interface__ = {"shape": (rows, engine.cfg.f), "strides": (4 * ld, 4), "typestr": "<f4",
                                         "data": (engine.device_factors(side), False), "version": 3}


def _matrix(engine, side):
    return torch.as_tensor(_Buffer(engine, side), device="cuda")


def _engine(case, f, seed, data, pu, pv, stream):
    solver, refine, warm = SOLVERS[case["solve"]]
    cfg = make_config(f, LAM, 1, solver, PRECS[case["prec"]], refine=refine, refine_warm=warm,
                      use_graph=bool(case.get("tuned")))
    e = Engine(cfg, data)
    e.set_stream(stream.cuda_stream)
    u, v = _factors(case, f, seed, pu, pv)
    e.set_factors(USERS, u)
    e.set_factors(ITEMS, v)
    if case.get("tuned"):
        e.autotune()
    return e


def _cg_systems(case, seed):
    """Regularised Gram matrices of rows with 2 f ratings, their right-hand sides and a start near the solution."""
    g = _generator(seed)
    b, f = case["batch"], case["f"]
    y = 0.3 * torch.randn(b, 2 * f, f, device="cuda", generator=g)
    a = torch.bmm(y.transpose(1, 2).contiguous(), y)
    a = 0.5 * (a + a.transpose(1, 2)) + LAM * 2 * f * torch.eye(f, device="cuda")
    rhs = torch.bmm(y.transpose(1, 2).contiguous(),
                    3.0 + torch.randn(b, 2 * f, 1, device="cuda", generator=g)).squeeze(2).contiguous()
    x0 = 0.1 * torch.randn(b, f, device="cuda", generator=g)
    return (a.half() if case["half"] else a).contiguous(), rhs, x0


def _gradient_inputs(case, seed):
    g = _generator(seed * 5 + 3)
    lam = LAM * torch.exp(0.3 * torch.randn(case["m"], device="cuda", generator=g))
    gx = 1e-3 * torch.randn(case["m"], case["f"], device="cuda", generator=g)
    return lam, gx


def _ranks(case):
    return [case["f"]] + [case[k] for k in ("f2", "f3") if k in case and case["kind"] == "group"]


def prepare(case, seed):
    state = dict(case=case, stream=torch.cuda.Stream())
    if case["kind"] == "cg_batch":
        state["A"], state["b"], state["x0"] = _cg_systems(case, seed)
        return state
    data, pu, pv = _ratings(case, seed)
    engines = [_engine(case, f, seed, data, pu, pv, state["stream"]) for f in _ranks(case)]
    state["engine"] = engines[0]
    state["factors"] = [(_matrix(e, USERS), _matrix(e, ITEMS)) for e in engines]
    if case["kind"] == "group":
        state["group"] = Group(engines)
    if case["kind"] == "grad":
        lam, state["gx"] = _gradient_inputs(case, seed)
        state["lam"] = lam.requires_grad_()
        state["Y"] = state["factors"][0][1].clone().requires_grad_()
    torch.cuda.synchronize()
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "cg_batch":
        x = state["x0"].clone()
        cg_update_x(state["A"], x, state["b"], 6, 1e-4)
        return x
    e = state["engine"]
    if kind == "sweep":
        e.sweep()
        return state["factors"][0]
    if kind == "train":
        return (e.train(1), *state["factors"][0])
    if kind == "group":
        state["group"].sweep()
        return state["factors"]
    if kind == "rows":
        e.set_stream(state["stream"].cuda_stream)
        _update_rows(e, case)
        return state["factors"][0][0][case["first"]:case["first"] + case["count"]]
    if kind == "rmse":
        return e.rmse(ca.ALS_RMSE_TEST), e.rmse(ca.ALS_RMSE_TRAIN)
    with torch.cuda.stream(state["stream"]):
        x = half_sweep(state["lam"], state["Y"], e, USERS)
        return (x.detach(), *torch.autograd.grad(x, (state["lam"], state["Y"]), state["gx"]))


def _update_rows(e, case):
    """One batch of the users' exact solve (als_update_rows of the C interface)."""
    rc = ca._capi.lib.als_update_rows(e.h, USERS, case["first"], case["count"], 1)
    if rc != 0:
        raise ca.AlsError(rc, "als_update_rows")


# ------------------------------------------------------------------ work
def work(case):
    f, kind = case["f"], case["kind"]
    if kind == "cg_batch":  # A, x and b once, x out; a product with A per iteration and one before
        b = case["batch"]
        return {"bytes": b * (f * f * (2 if case["half"] else 4) + 12 * f), "flops": b * 7 * 2.0 * f * f}
    m, n, nnz = case["m"], case["n"], float(case["nnz"])
    if kind == "rmse":
        t = nnz * 1.1
        return {"bytes": 12 * t + 4.0 * f * (m + n) * 2, "flops": 2 * f * t}
    total = {"bytes": 0.0, "flops": 0.0}
    share = case["count"] / m if kind == "rows" else 1.0
    halves = 2 if kind in ("sweep", "train", "group") else 1
    for f in _ranks(case):
        rows = (m + n) if halves == 2 else m * share
        # each side's ratings once, each factor matrix read and written once; Gram (one triangle) and solve
        total["bytes"] += halves * 8 * nnz * share + 4.0 * f * (m + n) * halves
        total["flops"] += halves * nnz * share * f * (f + 1) + rows * f ** 3 / 3.0
    if kind == "grad":  # the solve again for the adjoint, the ratings and both row matrices once more
        total["bytes"] += 8 * nnz + 4.0 * f * (3 * m + 2 * n)
        total["flops"] += 8.0 * f * nnz + 4.0 * f * f * m
    if kind == "train":
        total["bytes"] += 12 * nnz / 10
    return total


def tolerance(case):
    # four times the distance seen to exact(), or between the path and itself with its sums in another order
    kind, prec = case["kind"], case["prec"] if case["kind"] != "cg_batch" else "fp32"
    if kind == "cg_batch":
        return {"rel": 2e-6, "max": 2e-4}
    if kind == "rmse":
        return {"rel": 1e-6}
    if case["solve"] in ("cg", "cg16"):  # a row near the threshold stops an iteration earlier or later
        return {"rel": 2e-2, "max": 0.9}
    if prec == "fp32":  # plain FP32 solves of ill-conditioned rows
        return {"rel": 2e-4, "max": 0.2}
    if case["solve"] == "refined":
        return {"rel": 6e-4, "max": 0.3}
    return {"rel": 2e-3 if prec == "fp16" else 1.2e-2, "max": 0.9}


# ------------------------------------------------------------ in 64 bits
def _groups(ptr):
    """Rows in groups of like length: (rows, longest) with at most 2^27 padded ratings x 100 in a group."""
    length = np.diff(ptr)
    order = np.argsort(-length, kind="stable")
    i = 0
    while i < order.size and length[order[i]] > 0:
        top = int(length[order[i]])
        most = max(1, min(20000, 4_000_000 // top))
        j = i + int(np.searchsorted(-length[order[i:i + most]], -0.75 * top, side="right"))
        yield order[i:max(j, i + 1)], top
        i = max(j, i + 1)


def _padded(ptr, idx, val, Y, rows, top):
    """Rated rows of Y (zero past a row's end), ratings, indices and lengths of some rows."""
    r = torch.as_tensor(rows, device="cuda")
    start, length = ptr[r], ptr[r + 1] - ptr[r]
    at = torch.arange(top, device="cuda")
    inside = at[None, :] < length[:, None]
    pos = torch.where(inside, start[:, None] + at[None, :], 0)
    i = idx[pos]
    return r, Y[i] * inside[:, :, None], torch.where(inside, val[pos], 0.0), i, length


def _solve(A, b):
    return torch.cholesky_solve(b.unsqueeze(2), torch.linalg.cholesky(A)).squeeze(2)


def _cg(A, b, x, iters=6, tol=1e-4):
    r = b - torch.bmm(A, x.unsqueeze(2)).squeeze(2)
    p, old = r.clone(), (r * r).sum(1)
    live = torch.ones_like(old, dtype=torch.bool)
    for _ in range(iters):
        ap = torch.bmm(A, p.unsqueeze(2)).squeeze(2)
        pap = (p * ap).sum(1)
        live = live & (pap != 0)
        alpha = torch.where(live, old / torch.where(live, pap, 1.0), 0.0)
        x = x + alpha[:, None] * p
        r = r - alpha[:, None] * ap
        new = (r * r).sum(1)
        live = live & (new >= tol) & (new != 0)
        p = torch.where(live[:, None], r + (new / torch.where(live, old, 1.0))[:, None] * p, p)
        old = new
    return x


def _half(ptr, idx, val, Y, case, lam, X0=None, rows=None):
    """One half-sweep; with rows, of those alone (the others zero)."""
    if rows is not None:
        keep = np.zeros(ptr.size - 1, bool)
        keep[rows] = True
    p, i, v = (torch.as_tensor(a, device="cuda") for a in (ptr.astype(np.int64), idx.astype(np.int64), val))
    v = v.double()
    f = Y.shape[1]
    X = torch.zeros(ptr.size - 1, f, device="cuda", dtype=torch.float64)
    for rs, top in _groups(ptr):
        if rows is not None:
            rs = rs[keep[rs]]
            if not rs.size:
                continue
        r, y, w, _, length = _padded(p, i, v, Y, rs, top)
        yt = y.transpose(1, 2).contiguous()
        A = torch.bmm(yt, y)
        A.diagonal(dim1=1, dim2=2).add_((lam[r] * length)[:, None])
        b = torch.bmm(yt, w.unsqueeze(2)).squeeze(2)
        X[r] = _cg(A, b, X0[r]) if X0 is not None else _solve(A, b)
    return X


def _error(row, col, val, U, V):
    s, n = 0.0, row.size
    for a in range(0, n, 4_000_000):
        r, c, v = (torch.as_tensor(x[a:a + 4_000_000], device="cuda") for x in (row, col, val))
        s += float(((v.double() - (U[r.long()] * V[c.long()]).sum(1)) ** 2).sum())
    return math.sqrt(s / n)


def exact(case, seed):
    kind, f = case["kind"], case["f"]
    if kind == "cg_batch":
        A, b, x0 = _cg_systems(case, seed)
        return torch.cat([_cg(A[i:i + 1024].double(), b[i:i + 1024].double(), x0[i:i + 1024].double())
                          for i in range(0, case["batch"], 1024)])
    d, pu, pv = _ratings(case, seed)

    def start(f):
        u, v = _factors(case, f, seed, pu, pv)
        return torch.as_tensor(u, device="cuda").double(), torch.as_tensor(v, device="cuda").double()

    lam_u = torch.full((d.m,), float(np.float32(LAM)), device="cuda", dtype=torch.float64)
    lam_v = torch.full((d.n,), float(np.float32(LAM)), device="cuda", dtype=torch.float64)
    U0, V0 = start(f)
    if kind == "rmse":
        return (_error(d.t_row, d.t_col, d.t_val, U0, V0), _error(d.train_rows(), d.csr_idx, d.csr_val, U0, V0))
    if kind == "rows":
        rows = np.arange(case["first"], case["first"] + case["count"])
        return _half(d.csr_ptr, d.csr_idx, d.csr_val, V0, case, lam_u, rows=rows)[rows[0]:rows[-1] + 1]
    if kind == "grad":
        return _gradient(case, seed, d, V0)
    cg = case["solve"] in ("cg", "cg16")

    def sweep(U0, V0):
        U = _half(d.csr_ptr, d.csr_idx, d.csr_val, V0, case, lam_u, U0 if cg else None)
        return U, _half(d.csc_ptr, d.csc_idx, d.csc_val, U, case, lam_v, V0 if cg else None)

    if kind == "group":
        return [sweep(*start(f)) for f in _ranks(case)]
    U, V = sweep(U0, V0)
    return (np.array([_error(d.t_row, d.t_col, d.t_val, U, V)]), U, V) if kind == "train" else (U, V)


def _gradient(case, seed, d, Y):
    lam, gx = _gradient_inputs(case, seed)
    lam, gx = lam.double(), gx.double()
    p, i, v = (torch.as_tensor(a, device="cuda") for a in (d.csr_ptr.astype(np.int64), d.csr_idx.astype(np.int64),
                                                           d.csr_val))
    v = v.double()
    X, gl, gy = torch.zeros_like(gx), torch.zeros_like(lam), torch.zeros_like(Y)
    for rs, top in _groups(d.csr_ptr):
        r, y, w, at, length = _padded(p, i, v, Y, rs, top)
        yt = y.transpose(1, 2).contiguous()
        A = torch.bmm(yt, y)
        A.diagonal(dim1=1, dim2=2).add_((lam[r] * length)[:, None])
        both = torch.cat([torch.bmm(yt, w.unsqueeze(2)), gx[r].unsqueeze(2)], 2)
        x, xb = torch.cholesky_solve(both, torch.linalg.cholesky(A)).split(1, 2)
        inside = torch.arange(top, device="cuda")[None, :] < length[:, None]
        X[r] = x.squeeze(2)
        gl[r] = -length * (x * xb).sum((1, 2))
        e = w - torch.bmm(y, x).squeeze(2)
        c = (e[:, :, None] * xb.transpose(1, 2) - torch.bmm(y, xb) * x.transpose(1, 2)) * inside[:, :, None]
        gy.index_add_(0, at.reshape(-1), c.reshape(-1, Y.shape[1]))
    return X, gl, gy
