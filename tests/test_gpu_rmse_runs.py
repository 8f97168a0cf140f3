"""RMSE over runs of ratings: rating counts around a lane group's run and the
launch's group count (16,384 groups of 16 ratings at a time), sorted rows
(long and short stretches of one user), unsorted ones and a single user, for
every number of 64-column slices including the form for f > 192, with NaN in
the padding columns. The sum of squares within what FP32 dots may move it by:
a product passes through at most 20 roundings of 2^-24 on its way into a dot.
The same bits when called again."""
import ctypes as C

import numpy as np
import pytest

from cuda_als_amd import _capi as A

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("f", [1, 3, 63, 64, 65, 100, 128, 130, 192, 193, 300])
@pytest.mark.parametrize("n,order", [(1, "sorted"), (15, "sorted"), (17, "one"), (1000, "random"), (16384, "sorted"),
                                     (16385, "sorted"), (262144, "sorted"), (262145, "random"), (300001, "one"),
                                     (900000, "sorted")])
def test_runs(f, n, order):
    g = torch.Generator(device="cuda").manual_seed(n + f)
    users, items, ld = 700, 300, 4 * ((f + 3) // 4) + 4
    U, V = (torch.full((r, ld), float("nan"), device="cuda") for r in (users, items))
    U[:, :f] = torch.randn(users, f, device="cuda", generator=g) / f ** 0.25
    V[:, :f] = torch.randn(items, f, device="cuda", generator=g) / f ** 0.25
    row = torch.randint(0, users, (n,), device="cuda", generator=g, dtype=torch.int32)
    row = row.sort()[0] if order == "sorted" else torch.full_like(row, 699) if order == "one" else row
    col = torch.randint(0, items, (n,), device="cuda", generator=g, dtype=torch.int32)
    val = 3 + torch.randn(n, device="cuda", generator=g)
    out = torch.zeros(2, 2, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for k in range(2):
        rc = A.lib.als_rmse_dev_noalloc(*(C.c_void_p(t.data_ptr()) for t in (row, col, val)), n,
                                        *(C.c_void_p(t.data_ptr()) for t in (U, V)), f, ld,
                                        C.c_void_p(out[k].data_ptr()), None)
        assert rc == 0
    torch.cuda.synchronize()
    want = bound = 0.0
    for r, c, v in zip(row.split(100000), col.split(100000), val.split(100000)):
        p = U[r.long(), :f].double() * V[c.long(), :f].double()
        e, off = v.double() - p.sum(1), 20 * 2.0 ** -24 * p.abs().sum(1)
        want += float((e ** 2).sum())
        bound += float((2 * e.abs() * off + off ** 2).sum())
    got = out.cpu().numpy()
    assert (got[0] == got[1]).all() and abs(got[0, 0] - want) <= bound + 1e-12 * want, (got, want, bound)
    assert abs(got[0, 1] - np.sqrt(got[0, 0] / n)) <= 1e-12 * got[0, 1]
