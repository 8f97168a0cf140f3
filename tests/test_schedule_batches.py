"""The work schedule's batches (no GPU): every rating of every row in exactly
one unit whatever the batch rule, a caller's batch size kept as it is,
batches that may shrink doing so where they would be small and even where
they would not, and every unit in exactly one batch."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

from cuda_als_amd import _capi as A

SOLVE = {A.ALS_PREC_FP32: 96, A.ALS_PREC_FP16: 1024}  # cost of a solve in ratings


def preview(sizes, split_len, batch_work, grid, prec):
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    st = A.ScheduleStats()
    units = np.zeros((sizes.size + int(ptr[-1]) // 100 + 8, 4), np.int32)
    rc = A.lib.als_schedule_preview(sizes.size, ptr.ctypes.data_as(C.c_void_p), split_len, batch_work, grid, prec,
                                    C.byref(st), units.ctypes.data_as(C.c_void_p), units.shape[0])
    assert rc == 0
    return ptr, st, units[:st.nunits]


@pytest.fixture(scope="session")
def batches(tmp_path_factory):
    """(batch_work, batch_begin, cost of every unit) of a schedule without split rows."""
    exe, lib = tmp_path_factory.mktemp("sched") / "schedule_batches", A.LIB_PATH.parent
    cmd = ["g++", "-std=c++17", "-O1", f"-I{lib / 'csrc'}", str(Path(__file__).parent / "schedule_batches.cpp"), "-o",
           str(exe), f"-L{lib}", "-lals_mi355x", f"-Wl,-rpath,{lib}", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(sizes, batch_work, grid, prec, shrinks=False, slow=False):
        out = subprocess.run([str(exe), "1000000000", str(batch_work), str(grid), str(prec), str(int(shrinks)),
                              str(int(slow))],
                             input=" ".join(map(str, sizes)), capture_output=True, text=True, timeout=60, check=True)
        work, *begin = map(int, out.stdout.split())
        begin = np.array(begin)
        assert begin[0] == 0 and begin[-1] == sizes.size and (np.diff(begin) > 0).all()
        return work, begin, np.sort(sizes)[::-1] + SOLVE[prec]
    return run


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


@pytest.mark.parametrize("grid", [7, 2048])
@pytest.mark.parametrize("prec", [A.ALS_PREC_FP32, A.ALS_PREC_FP16])
def test_a_callers_batch_size_is_kept(prec, grid, batches):
    """Each batch ends with the unit that reaches the size asked for, so that
    a larger size never gives more batches."""
    sizes = np.random.default_rng(1).poisson(130, 20000)
    last = sizes.size
    for work in (1, 100, 200, 400, 700, 1600, 5000, 100000):
        got, begin, cost = batches(sizes, work, grid, prec)
        total = np.add.reduceat(cost, begin[:-1])
        before = total - cost[begin[1:] - 1]  # without its last unit
        assert got == work and (total[:-1] >= work).all() and (before < work).all()
        _, st, _ = preview(sizes, 1000000000, work, grid, prec)
        assert st.nbatches == begin.size - 1 <= last and st.batch_work == work
        last = st.nbatches


def test_small_batches_shrink_from_large_ones(batches):
    """40,000 rows of 100 ratings on 4,096 waves, FP32: batches of the chosen
    size would be one row each. They take half of an even share of what is
    left while that is more than a row: 2 waves' worth of them for every
    factor of e that the work left falls by until it is 2 waves' worth of
    rows, which go one by one. The same size asked for without shrinking is
    even. Rows of 6,000 ratings keep even batches."""
    sizes, waves = np.full(40000, 100), 4096
    work, begin, cost = batches(sizes, 0, waves, A.ALS_PREC_FP32, shrinks=True)
    rows = np.diff(begin)
    assert (np.diff(rows) <= 0).all() and rows[0] > 1 and rows[-1] == 1
    assert rows.size <= 2 * waves * (np.log(40000 / (2 * waves)) + 1) + 1 and work <= cost[0]
    assert (np.diff(batches(sizes, work, waves, A.ALS_PREC_FP32)[1]) == 1).all()
    assert np.array_equal(batches(sizes, work, waves, A.ALS_PREC_FP32, shrinks=True)[1], begin)
    _, begin, _ = batches(np.full(4000, 6000), 0, 64, A.ALS_PREC_FP16, shrinks=True)
    assert np.unique(np.diff(begin)[:-1]).size == 1


@pytest.mark.parametrize("slow", [False, True])
@pytest.mark.parametrize("prec,most", [(A.ALS_PREC_FP32, 1536), (A.ALS_PREC_FP16, 9216)])
def test_shrinking_batches_are_bounded(prec, most, slow, batches):
    """However few the waves, no shrinking batch is larger than what the
    counter asks for (half of that where ratings are slow) by more than its
    last row."""
    sizes = np.random.default_rng(2).poisson(120, 100000)
    work, begin, cost = batches(sizes, 0, 3072, prec, True, slow)
    total = np.add.reduceat(cost, begin[:-1])
    bound = most // (1 + slow)
    assert bound <= total.max() < bound + cost.max() and work < bound
    assert total[-2] < work + cost.max()


@pytest.mark.parametrize("prec", [A.ALS_PREC_FP32, A.ALS_PREC_FP16])
def test_split_length_does_not_fall_with_occupancy(prec):
    """The parts of long rows are no shorter where more waves fit on a SIMD:
    their number is a matter of the GPU's size and the work."""
    sizes = np.concatenate([np.full(20, 200000), np.full(9000, 3000)])
    lens = [preview(sizes, 0, 0, grid, prec)[1].split_len for grid in (1024, 2048, 3072, 8192)]
    assert len(set(lens)) == 1 and lens[0] > 2048 and preview(sizes, 0, 0, 256, prec)[1].split_len > lens[0]
