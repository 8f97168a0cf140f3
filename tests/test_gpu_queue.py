"""The update kernels' work queue where the batches just fill the launched
waves: as many batches as waves, one more, one fewer, a single wave and a
single batch. Each half-sweep runs several times on one engine (the ticket
counter has to be back at zero after every launch), directly and as replays
of a captured sweep, against the FP64 oracle."""
import numpy as np
import pytest

import cuda_als_amd as ca
from cuda_als_amd import _capi as A
from cuda_als_amd import engine as E
from oracle import als_oracle as O

pytestmark = pytest.mark.gpu

ROWS, COLS, PER_ROW = 96, 40, 9


def matrix(rows=ROWS):
    """Every user has PER_ROW ratings, so a batch of work 1 is one row."""
    rng = np.random.default_rng(5)
    idx = np.sort(rng.random((rows, COLS)).argsort(1)[:, :PER_ROW], 1).ravel()
    val = rng.integers(1, 6, idx.size)
    return ca.from_arrays(rows, COLS, np.arange(rows + 1) * PER_ROW, idx, val, [0], [0], [3.0])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("grid", [1, 2, ROWS - 1, ROWS, ROWS + 1])
@pytest.mark.parametrize("f,prec", [(16, E.Prec.FP32), (70, E.Prec.FP16)])
def test_batches_against_waves(f, prec, grid, graph):
    """f = 70 sends every row here through the dual kernel unless its limit is
    0; both are run (the dual kernel's waves are not the grid's: its own
    boundary is below). FP32 factors within 1e-4 of the oracle on the exact
    factors (as elsewhere for one half-sweep), FP16 within 1e-4 on the
    rounded ones."""
    d = matrix()
    V0 = np.random.default_rng(1).standard_normal((COLS, f)).astype(np.float32) * 0.3
    want = O.update_rows(O.config(f, 0.05, O.SOLVE_CHOL, gram_prec=O.PREC_FP16 if prec == E.Prec.FP16 else O.PREC_EXACT),
                         np.arange(ROWS), d.csr_ptr, d.csr_idx, d.csr_val, V0.astype(np.float64))
    with E.Engine(E.make_config(f, 0.05, 1, E.SolveType.CHOL, prec, use_graph=graph, batch_work=1), d) as e:
        for limit in {0, e.info().dual_max}:
            e.set_grid(ca.ALS_SIDE_USERS, grid)
            e.set_dual_limit(ca.ALS_SIDE_USERS, limit)
            if limit == 0:
                assert e.info().nbatches[0] == ROWS  # the batch size asked for, whatever the grid
            first = None
            for _ in range(4):
                e.set_factors(ca.ALS_SIDE_USERS, np.zeros((ROWS, f), np.float32))
                e.set_factors(ca.ALS_SIDE_ITEMS, V0)
                (e.sweep if graph else lambda: e.update(ca.ALS_SIDE_USERS))()
                U = e.get_factors(ca.ALS_SIDE_USERS)
                first = U if first is None else first
                assert np.array_equal(U, first)
            err = np.abs(first - want).max(axis=1) / np.maximum(1.0, np.abs(want).max(axis=1))
            assert e.info().failures == 0 and err.max() <= 1e-4, err.max()
            # one batch for all rows
            e.set_schedule(ca.ALS_SIDE_USERS, 0, 1 << 30)
            e.set_factors(ca.ALS_SIDE_ITEMS, V0)
            e.update(ca.ALS_SIDE_USERS)
            assert np.array_equal(e.get_factors(ca.ALS_SIDE_USERS), first)
            e.set_schedule(ca.ALS_SIDE_USERS, 0, 1)


def uneven():
    rng = np.random.default_rng(9)
    lengths = rng.integers(1, 200, 3000)
    idx = np.concatenate([np.sort(rng.choice(500, n, replace=False)) for n in lengths])
    return ca.from_arrays(3000, 500, np.concatenate([[0], np.cumsum(lengths)]), idx, rng.integers(1, 6, idx.size),
                          [0], [0], [3.0])


def test_batches_shrink_where_they_may():
    """On 64 waves this matrix's batches, three rows each by the scheduler's
    choice, shrink from larger ones unless a size is asked for, through the
    configuration or later; the flag brings the shrinking back, by itself with
    the scheduler's size, and rebuilds for another grid keep the mode."""
    d = uneven()

    def batches(cfg, *calls):
        with E.Engine(E.make_config(16, 0.05, 1, E.SolveType.CHOL, E.Prec.FP32, batch_work=cfg), d) as e:
            e.set_grid(ca.ALS_SIDE_USERS, 64)
            for c in calls:
                e.set_schedule(ca.ALS_SIDE_USERS, 0, c)
            n = e.info().nbatches[0]
            e.set_grid(ca.ALS_SIDE_USERS, 63)
            e.set_grid(ca.ALS_SIDE_USERS, 64)
            assert e.info().nbatches[0] == n
            return n

    shrinks = A.ALS_BATCH_SHRINKS
    assert batches(1) == batches(0, 1) == batches(0, shrinks, 1) == 3000
    assert batches(1, shrinks + 1) == batches(0, shrinks + 1) < 1500
    assert batches(1, shrinks) == batches(0, shrinks) < batches(0, 574)


@pytest.mark.parametrize("batch_work", [0, 500])
@pytest.mark.parametrize("prec", [E.Prec.FP32, E.Prec.FP16])
def test_a_stored_tuning_gives_the_batches_that_were_tuned(prec, batch_work):
    """als_autotune's result applied to a fresh engine in either order of the
    calls: the same batches as on the tuned engine, whether they shrink or
    not, and the same bits."""
    d = uneven()
    cfg = E.make_config(70, 0.05, 1, E.SolveType.CHOL, prec, batch_work=batch_work)
    V0 = np.random.default_rng(1).standard_normal((500, 70)).astype(np.float32) * 0.3

    def update(e):
        e.set_factors(ca.ALS_SIDE_ITEMS, V0)
        e.update(ca.ALS_SIDE_USERS)
        return list(e.info().nbatches), e.get_factors(ca.ALS_SIDE_USERS)

    with E.Engine(cfg, d) as e:
        e.init_factors()
        t = e.autotune()
        want = update(e)
    for order in (1, -1):
        with E.Engine(cfg, d) as e:
            for side in (0, 1):
                calls = [lambda: e.set_schedule(side, t["split_len"][side], t["batch_work"][side]),
                         lambda: e.set_grid(side, t["grid"][side]), lambda: e.set_dual_limit(side, t["dual_limit"][side])]
                for c in calls[::order]:
                    c()
                if t["gram_gather"][side]:
                    e.set_gram_gather(side, 1)
            got = update(e)
            assert got[0] == want[0] and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("prec", [E.Prec.FP32, E.Prec.FP16])
@pytest.mark.parametrize("rows", [-1, 0, 1, 2000, 30000])
def test_dual_batches_against_waves(rows, prec, graph):
    """The dual kernel's tickets: as many one-row batches as its waves (four a
    SIMD, 16 a CU), one fewer, one more and 2,000 more, and 30,000 rows in
    batches that shrink; the same bits from launch to launch, directly and
    from a graph, and within 1e-4 of the oracle."""
    import torch
    waves = 16 * torch.cuda.get_device_properties(0).multi_processor_count
    rows = rows if rows == 30000 else waves + rows
    d = matrix(rows)
    V0 = np.random.default_rng(1).standard_normal((COLS, 70)).astype(np.float32) * 0.3
    want = O.update_rows(O.config(70, 0.05, O.SOLVE_CHOL, gram_prec=O.PREC_FP16 if prec == E.Prec.FP16 else O.PREC_EXACT),
                         np.arange(rows), d.csr_ptr, d.csr_idx, d.csr_val, V0.astype(np.float64))
    with E.Engine(E.make_config(70, 0.05, 1, E.SolveType.CHOL, prec, use_graph=graph), d) as e:
        info = e.info()
        assert info.dual_rows[0] == rows
        assert info.nbatches[0] == rows if rows < 30000 else waves < info.nbatches[0] < rows
        first = None
        for _ in range(4):
            e.set_factors(ca.ALS_SIDE_USERS, np.zeros((rows, 70), np.float32))
            e.set_factors(ca.ALS_SIDE_ITEMS, V0)
            (e.sweep if graph else lambda: e.update(ca.ALS_SIDE_USERS))()
            U = e.get_factors(ca.ALS_SIDE_USERS)
            first = U if first is None else first
            assert np.array_equal(U, first)
        err = np.abs(first - want).max(axis=1) / np.maximum(1.0, np.abs(want).max(axis=1))
        assert e.info().failures == 0 and err.max() <= 1e-4, err.max()
