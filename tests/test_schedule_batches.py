"""The work schedule's batches (als_schedule_preview, no GPU): every rating of
every row in exactly one unit whatever the batch rule, fewer batches where an
average one would be small, the rule off where it would not."""
import ctypes as C

import numpy as np
import pytest

from cuda_als_amd import _capi as A


def preview(sizes, split_len, batch_work, grid, prec):
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    st = A.ScheduleStats()
    units = np.zeros((sizes.size + int(ptr[-1]) // 100 + 8, 4), np.int32)
    rc = A.lib.als_schedule_preview(sizes.size, ptr.ctypes.data_as(C.c_void_p), split_len, batch_work, grid, prec,
                                    C.byref(st), units.ctypes.data_as(C.c_void_p), units.shape[0])
    assert rc == 0
    return ptr, st, units[:st.nunits]


@pytest.mark.parametrize("grid", [1, 7, 64, 4096])
@pytest.mark.parametrize("rows,mean", [(1, 5), (3, 0), (500, 3), (3000, 40), (3000, 900)])
@pytest.mark.parametrize("prec", [A.ALS_PREC_FP32, A.ALS_PREC_FP16])
def test_units_cover_the_matrix(rows, mean, grid, prec):
    sizes = np.random.default_rng(rows + mean).poisson(mean, rows)
    ptr, st, u = preview(sizes, 1000, 0, grid, prec)
    for r in range(rows):
        mine = u[u[:, 0] == r]
        mine = mine[np.argsort(mine[:, 1], kind="stable")]
        assert mine[0, 1] == ptr[r] and mine[-1, 2] == ptr[r + 1] and (mine[1:, 1] == mine[:-1, 2]).all()
    assert 1 <= st.nbatches <= st.nunits


def test_small_batches_shrink_from_large_ones():
    """40,000 rows of 100 ratings on 64 waves, FP32: batches of one row would
    be 40,000; shrinking ones are at most two waves' worth per halving of what
    is left, and the last ones are still single rows' size. Rows of 6,000
    ratings keep one row a batch."""
    sizes = np.full(40000, 100)
    _, st, _ = preview(sizes, 0, 1, 64, A.ALS_PREC_FP32)
    assert st.nbatches <= 2 * 64 * np.log(40000 / 128) + 2 * 64 + 64
    _, st, _ = preview(np.full(4000, 6000), 0, 1, 64, A.ALS_PREC_FP16)
    assert st.nbatches == st.nunits
