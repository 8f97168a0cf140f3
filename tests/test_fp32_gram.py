"""The FP32 Gram on BF16 matrix pipes: every operand is three BF16 parts
h + m + l, and a product is the six of their products that reach FP32's last
bits. The factors here are 1 + nearly 2^-8 + nearly 2^-17 (times a power of
two), where m and l are as large beside h as they get and always of its sign,
so that a product left out does not average away: it moves every entry of the
Gram by 2^-17 (h l, l h) or 2^-16 (m m) of its size. lambda is the factors'
squared norm, so the system's condition is 2 and half of that reaches the
solution: 3.8e-6 at least. What FP32 gives is some 17 roundings of 2^-24 at the
most: products and sums of a chunk's 32 ratings below 6, ten chunks added, the
factorisation and both substitutions at condition 2: 1e-6, which is the bar.
"""
import numpy as np
import pytest
import torch

import cuda_als_amd as ca
from cuda_als_amd import engine as E

BAR = 1e-6
LENGTHS = [1, 2, 31, 32, 33, 64, 65, 100, 300]
COLS = 320


def awkward(rng, *shape):
    """1 + m + l in FP32, m in (0.97 .. 1) 2^-8 and of 8 bits, l in (0.8 .. 0.98) 2^-17."""
    m = rng.integers(248, 256, shape) * 2.0 ** -16
    l = np.floor(rng.uniform(0.8, 0.98, shape) * 64) * 2.0 ** -23
    x = 1 + m + l
    assert (x.astype(np.float32) == x).all()
    return x.astype(np.float32)


def system(f):
    """Ratings' rows, indices, values and the fixed factors; each rating's sign is its item's."""
    rng = np.random.default_rng(f)
    sign = rng.choice([-1.0, 1.0], COLS).astype(np.float32)
    Y = awkward(rng, COLS, f) * sign[:, None] * 2.0 ** rng.integers(-2, 2, f).astype(np.float32)
    idx = np.concatenate([np.sort(rng.choice(COLS, n, replace=False)) for n in LENGTHS]).astype(np.int32)
    val = 4 * awkward(rng, idx.size) * sign[idx]
    lam = float(np.float32((Y[0].astype(np.float64) ** 2).sum()))
    return np.concatenate([[0], np.cumsum(LENGTHS)]), idx, val, Y, lam


def solve(f, gram):
    """The rows' solutions in 64 bits with gram(y, z) for the products y^T z."""
    ptr, idx, val, Y, lam = system(f)
    out = []
    for a, b in zip(ptr[:-1], ptr[1:]):
        y, r = Y[idx[a:b]], val[a:b, None]
        out.append(np.linalg.solve(gram(y, y) + lam * (b - a) * np.eye(f), gram(y, r)[:, 0]))
    return np.array(out)


def exact(y, z):
    return y.astype(np.float64).T @ z.astype(np.float64)


def rel(got, want):
    return (np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)).max()


def parts(x):
    out, rest = [], torch.tensor(x)
    for _ in range(3):
        p = rest.bfloat16().float()
        out.append(p.double().numpy())
        rest = rest - p
    assert not rest.any()
    return dict(zip("hml", out))


PRODUCTS = ["hh", "hm", "mh", "mm", "hl", "lh"]


@pytest.mark.parametrize("f", [1, 15, 64, 143])
def test_the_bar_tells_a_missing_product(f):
    """In 64 bits: the six products stay far below the bar, any five of them miss it."""
    def gram(keep):
        def of(y, z):
            py, pz = parts(y), parts(z)
            return sum(py[k[0]].T @ pz[k[1]] for k in keep)
        return of
    want = solve(f, exact)
    assert rel(solve(f, gram(PRODUCTS)), want) < BAR / 8
    for k in PRODUCTS:
        assert rel(solve(f, gram([p for p in PRODUCTS if p != k])), want) > 2 * BAR, k


@pytest.mark.gpu
@pytest.mark.parametrize("split_len", [1 << 30, 40])
@pytest.mark.parametrize("solver", [E.SolveType.CHOL, E.SolveType.CUMF_ALS_CG_FP32])
@pytest.mark.parametrize("f", [1, 15, 16, 31, 32, 47, 48, 63, 64, 79, 80, 95, 96, 111, 112, 127, 128, 129, 143])
def test_fp32_solutions(f, solver, split_len):
    """Every tile count, augmented and f = 16T, rows through the f x f system,
    whole and in parts. CG from the exact solution: at condition 2 its steps
    only follow the Gram's error."""
    ptr, idx, val, Y, lam = system(f)
    want = solve(f, exact)
    d = ca.from_arrays(len(LENGTHS), COLS, ptr, idx, val, [0], [0], [3.0])
    cfg = E.make_config(f, lam, 1, solver, E.Prec.FP32, split_len=split_len, cg_iters=12, cg_tol=0.0)
    with E.Engine(cfg, d) as e:
        if e.info().dual_max:
            e.set_dual_limit(ca.ALS_SIDE_USERS, 0)
        e.set_factors(ca.ALS_SIDE_USERS, want.astype(np.float32))
        e.set_factors(ca.ALS_SIDE_ITEMS, Y)
        e.update(ca.ALS_SIDE_USERS)
        got, info = e.get_factors(ca.ALS_SIDE_USERS), e.info()
    assert info.failures == 0 and info.dual_rows[0] == 0 and (info.nsplit_rows[0] > 0) == (split_len == 40)
    print(f, solver, split_len, rel(got, want))
    assert rel(got, want) <= BAR
