"""Ranks that fill their 16-column blocks (f = 16T): the systems are kept in T
blocks with the right-hand side beside them instead of an augmented row in a
block of its own. Every such rank, Gram precision and solver against the FP64
oracle, on rows that end at every place of a 32-rating chunk, whole and split
(so that b travels with the parts), and the neighbouring ranks 16T - 1 and
16T + 1 that keep the augmented form."""
import numpy as np
import pytest

import cuda_als_amd as ca
from cuda_als_amd import engine as E
from oracle import als_oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 63, 64, 65, 79, 80, 81, 96, 97, 128, 150, 193, 256, 300]
COLS = 320
ORACLE_PREC = {E.Prec.FP32: O.PREC_EXACT, E.Prec.BF16: O.PREC_BF16, E.Prec.FP16: O.PREC_FP16}


def matrix(f):
    rng = np.random.default_rng(f)
    idx = np.concatenate([np.sort(rng.choice(COLS, n, replace=False)) for n in LENGTHS]).astype(np.int32)
    val = rng.integers(1, 11, idx.size) / 2.0
    ptr = np.concatenate([[0], np.cumsum(LENGTHS)])
    d = ca.from_arrays(len(LENGTHS), COLS, ptr, idx, val, [0], [0], [3.0])
    return d, (0.4 * rng.standard_normal((len(LENGTHS), f))).astype(np.float32), \
        (0.4 * rng.standard_normal((COLS, f))).astype(np.float32)


def rel(got, want):
    return (np.abs(got - want).max(axis=1) / np.maximum(1.0, np.abs(want).max(axis=1))).max()


# (solver, refinement steps, warm): against the oracle on the Gram's own rounded inputs, but for the classic
# refinement, whose residual is restaged from the FP32 rows and which converges to the exact system's solution
SOLVES = {"chol": (E.SolveType.CHOL, 0, False), "warm": (E.SolveType.CHOL, 1, True),
          "refined": (E.SolveType.CHOL, 2, False), "cg": (E.SolveType.CUMF_ALS_CG_FP32, 0, False)}


# parts of split rows refine against the 16-bit system, so the refined solver runs unsplit
@pytest.mark.parametrize("solve,split_len", [(s, n) for s in SOLVES for n in (0, 40) if (s, n) != ("refined", 40)])
@pytest.mark.parametrize("prec", list(ORACLE_PREC))
@pytest.mark.parametrize("f", [15, 16, 17, 32, 40, 48, 63, 64, 65, 80, 90, 96, 100, 112, 127, 128, 129, 143])
def test_half_sweep(f, prec, solve, split_len):
    """Within 1e-4 of the FP64 oracle, as the other half-sweep tests ask (the
    oracle's system is formed from the same rounded factors, so the precision
    of the Gram's inputs is not in the difference; the FP32 solve of these
    rows is a few 1e-6 off, the refined one of BF16 rows, whose two steps
    each gain about two digits, a few 1e-5)."""
    d, U0, V0 = matrix(f)
    kind, refine, warm = SOLVES[solve]
    oprec = O.PREC_EXACT if solve == "refined" else ORACLE_PREC[prec]
    cfg = O.config(f, 0.05, O.SOLVE_CG if solve == "cg" else O.SOLVE_CHOL, cg_tol=0.0, gram_prec=oprec)
    want = O.update_rows(cfg, np.arange(d.m), d.csr_ptr, d.csr_idx, d.csr_val, V0.astype(np.float64),
                         U0.astype(np.float64) if solve == "cg" else None)
    with E.Engine(E.make_config(f, 0.05, 1, kind, prec, refine=refine, refine_warm=warm, cg_tol=0.0,
                                split_len=split_len), d) as e:
        if solve == "refined":
            e.set_schedule(ca.ALS_SIDE_USERS, 0, 0, 1 << 30)
        e.set_factors(ca.ALS_SIDE_USERS, U0)
        e.set_factors(ca.ALS_SIDE_ITEMS, V0)
        e.update(ca.ALS_SIDE_USERS)
        got = e.get_factors(ca.ALS_SIDE_USERS)
        info = e.info()
        assert info.failures == 0 and (info.nsplit_rows[0] > 0) == (split_len > 0)
    print(f, prec, solve, split_len, rel(got, want))
    assert not got[0].any() and rel(got, want) <= 1e-4


@pytest.mark.parametrize("prec", [E.Prec.FP32, E.Prec.FP16])
@pytest.mark.parametrize("f", [16, 64, 128])
def test_padding_of_caller_buffers(f, prec):
    """als_forward_dev writes whole rows of the caller's X, zeros past column
    f, whatever was there, and the adjoint does the same for its outputs."""
    import torch
    d, _, V0 = matrix(f)
    with E.Engine(E.make_config(f, 0.05, 1, E.SolveType.CHOL, prec), d) as e:
        ld = e.info().ld
        s = torch.cuda.Stream()
        e.set_stream(s.cuda_stream)
        Y = torch.zeros(d.n, ld, device="cuda")
        Y[:, :f] = torch.tensor(V0, device="cuda")
        X, xbar, ybar = (torch.full((r, ld), 7.0, device="cuda") for r in (d.m, d.m, d.n))
        g = torch.zeros(d.m, ld, device="cuda")
        g[:, :f] = 1e-2
        lbar = torch.zeros(d.m, device="cuda")
        torch.cuda.synchronize()
        e.forward_dev(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), None)
        e.adjoint_dev(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), g.data_ptr(), xbar.data_ptr(), lbar.data_ptr(),
                      ybar.data_ptr())
        torch.cuda.synchronize()
        for t in (X, xbar, ybar):
            assert not t[:, f:].any() and t[:, :f].any()


@pytest.mark.parametrize("f", [1, 16, 17, 48, 64, 100, 128, 143])
def test_saved_factors_fill_what_they_ask_for(f):
    """als_factor_save_bytes is what the forward pass stores, the tiles of the
    f x f system for every row that has ratings, to the last of them: nothing
    is written past it, and the adjoint from a buffer of just that size equals
    the one from the engine's own."""
    import torch
    d, _, V0 = matrix(f)
    with E.Engine(E.make_config(f, 0.05, 1, E.SolveType.CHOL, E.Prec.FP32), d) as e:
        ld, T = e.info().ld, (f + 15) // 16
        row = T * (T + 1) // 2 * 1024
        nbytes = e.factor_save_bytes(ca.ALS_SIDE_USERS)
        assert nbytes == d.m * row and e.factor_save_bytes(ca.ALS_SIDE_ITEMS) == d.n * row
        e.set_stream(torch.cuda.Stream().cuda_stream)
        save = torch.full((nbytes // 4 + 4096,), 7.0, device="cuda")
        Y = torch.zeros(d.n, ld, device="cuda")
        Y[:, :f] = torch.tensor(V0, device="cuda")
        g = torch.zeros(d.m, ld, device="cuda")
        g[:, :f] = 1e-2
        out = []
        for own in (False, True):
            X, xbar, ybar = (torch.empty(r, ld, device="cuda") for r in (d.m, d.m, d.n))
            lbar = torch.empty(d.m, device="cuda")
            torch.cuda.synchronize()
            if own:
                e.forward_dev(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), None)
                e.adjoint_dev(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), g.data_ptr(), xbar.data_ptr(),
                              lbar.data_ptr(), ybar.data_ptr())
            else:
                e.forward_dev_ws(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), None, save.data_ptr(), nbytes)
                e.adjoint_dev_ws(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), save.data_ptr(), nbytes, g.data_ptr(),
                                 xbar.data_ptr(), lbar.data_ptr(), ybar.data_ptr())
            torch.cuda.synchronize()
            out.append((X, xbar, ybar, lbar))
        with pytest.raises(ca.AlsError):
            e.forward_dev_ws(ca.ALS_SIDE_USERS, Y.data_ptr(), X.data_ptr(), None, save.data_ptr(), nbytes - 4)
    assert (save[nbytes // 4:] == 7.0).all() and (save[:nbytes // 4].view(d.m, row // 4)[1:, -256:] != 7.0).any(1).all()
    assert all(torch.equal(a, b) for a, b in zip(*out))


def test_fp32_factors_beyond_two_gib():
    """A fixed side past 2 GiB takes the FP32 Gram's 64-bit addresses instead
    of buffer offsets: users whose items lie at both ends of it, against the
    oracle (bar as above)."""
    import torch
    f, n = 100, (1 << 31) // (4 * 112) + 1000
    rng = np.random.default_rng(3)
    near = np.concatenate([np.arange(150), np.arange(n - 150, n)])
    lengths = [1, 31, 90, 200, 300]
    pos = np.concatenate([np.sort(rng.choice(near.size, k, replace=False)) for k in lengths])
    val = rng.integers(1, 6, pos.size).astype(np.float32)
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    d = ca.from_arrays(len(lengths), n, ptr, near[pos], val, [0], [0], [3.0])
    V0 = (0.4 * rng.standard_normal((near.size, f))).astype(np.float32)
    want = O.update_rows(O.config(f, 0.05, O.SOLVE_CHOL), np.arange(len(lengths)), ptr, pos, val, V0.astype(np.float64))
    with E.Engine(E.make_config(f, 0.05, 1, E.SolveType.CHOL, E.Prec.FP32), d) as e:
        class Rows:
            __cuda_array_interface__ = {"shape": (n, 112), "typestr": "<f4", "version": 3, "strides": None,
                                        "data": (e.device_factors(ca.ALS_SIDE_ITEMS), False)}
        Y = torch.as_tensor(Rows(), device="cuda")
        Y[torch.as_tensor(near, device="cuda"), :f] = torch.as_tensor(V0, device="cuda")
        torch.cuda.synchronize()
        e.set_dual_limit(ca.ALS_SIDE_USERS, 0)
        e.update(ca.ALS_SIDE_USERS)
        got = e.get_factors(ca.ALS_SIDE_USERS)
    assert rel(got, want) <= 1e-4


@pytest.mark.parametrize("side", [ca.ALS_SIDE_USERS, ca.ALS_SIDE_ITEMS])
@pytest.mark.parametrize("shape", [(40, 1500), (1500, 40)])
@pytest.mark.parametrize("prec", list(ORACLE_PREC))
@pytest.mark.parametrize("f", [64, 100])
def test_row_ranges_of_oblong_matrices(f, prec, shape, side):
    """als_update_rows on matrices with far more columns than rows and the
    other way round (a range's fixed side is as long as its own matrix's
    other dimension, whichever is larger): the rows of the range equal the
    whole half-sweep's, bit for bit, the others keep their values, and the
    half-sweep is within 1e-4 of the oracle."""
    from cuda_als_amd import _capi as A
    m, n = shape
    rng = np.random.default_rng(m + f)
    mask = rng.random((m, n)) < 0.12
    idx = np.nonzero(mask)[1]
    d = ca.from_arrays(m, n, np.concatenate([[0], np.cumsum(mask.sum(1))]), idx, rng.integers(1, 6, idx.size),
                       [0], [0], [3.0])
    U0, V0 = ((0.4 * rng.standard_normal((r, f))).astype(np.float32) for r in (m, n))
    rows = m if side == ca.ALS_SIDE_USERS else n
    first, count = rows // 3, rows // 2
    with E.Engine(E.make_config(f, 0.05, 1, E.SolveType.CHOL, prec), d) as e:
        out = []
        for ranged in (False, True):
            e.set_factors(0, U0)
            e.set_factors(1, V0)
            if ranged:
                assert A.lib.als_update_rows(e.h, side, first, count, 1) == 0
            else:
                e.update(side)
            out.append(e.get_factors(side))
    old = U0 if side == ca.ALS_SIDE_USERS else V0
    inside = np.zeros(rows, bool)
    inside[first:first + count] = True
    assert np.array_equal(out[1][inside], out[0][inside]) and np.array_equal(out[1][~inside], old[~inside])
    lists = (d.csr_ptr, d.csr_idx, d.csr_val, V0) if side == ca.ALS_SIDE_USERS else (d.csc_ptr, d.csc_idx, d.csc_val, U0)
    want = O.update_rows(O.config(f, 0.05, O.SOLVE_CHOL, gram_prec=ORACLE_PREC[prec]), np.arange(rows), *lists[:3],
                         lists[3].astype(np.float64))
    assert rel(out[0], want) <= 1e-4
