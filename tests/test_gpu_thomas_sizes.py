"""The batched three-band solve and its adjoint at the sizes where its kernels
change: one row, the edges of the LDS kernels' batches of eight rows, of their
columns per block (64 and 65 rows) and of their row count (128 and 129), and
column counts that leave a block partly filled.  The reference is the same
recurrence (column_solvers.c:641-667) in numpy float64, one operation at a
time: the device forms every value with the same operations in the same order
and without contraction, so the results are equal, not close.  The bands' last
rows, which the solve does not use, hold NaN."""
import ctypes as C

import numpy as np
import pytest

from conftest import get_grid

pytestmark = pytest.mark.gpu


def thomas(c, d, e, r):
    n = d.shape[0]
    ep, x = np.zeros_like(d), np.zeros_like(d)
    if n > 1:
        ep[0] = e[0] / d[0]
    x[0] = r[0] / d[0]
    for j in range(1, n):
        den = d[j] - ep[j - 1] * c[j - 1]
        if j < n - 1:
            ep[j] = e[j] / den
        x[j] = (r[j] - x[j - 1] * c[j - 1]) / den
    for j in range(n - 2, -1, -1):
        x[j] = x[j] - ep[j] * x[j + 1]
    return x


@pytest.mark.parametrize("n", [1, 2, 8, 9, 26, 64, 65, 128, 129])
@pytest.mark.parametrize("ncol", [1, 47, 513])
def test_solve_and_adjoint_equal_the_recurrence(n, ncol):
    import torch
    from game_archived_amd.rkhevi import DeviceModel
    rng = np.random.default_rng(100 * n + ncol)
    c, e = (-rng.uniform(0.1, 1.0, (n, ncol)) for _ in range(2))
    d = 1.0 - c - e
    r, x_bar = rng.standard_normal((n, ncol)), rng.standard_normal((n, ncol))
    c[n - 1], e[n - 1] = np.nan, np.nan
    x = thomas(c, d, e, r)
    r_bar = thomas(e, d, c, x_bar)
    dm = DeviceModel(get_grid(3))
    try:
        lib = dm.lib
        dev = lambda a: torch.as_tensor(np.ascontiguousarray(a)).cuda()
        p = lambda t: C.c_void_p(t.data_ptr())
        new = lambda: torch.full((n, ncol), 7.0, dtype=torch.float64, device="cuda")
        tc, td, te, tr, tb = map(dev, (c, d, e, r, x_bar))
        tx, t_rb, t_cb, t_db, t_eb, work = (new() for _ in range(6))
        torch.cuda.synchronize()
        print(f"case: {n} rows, {ncol} columns", flush=True)
        dm._check(lib.game_gpu_op_thomas(n, ncol, p(tc), p(td), p(te), p(tr), p(tx), p(work)))
        dm._check(lib.game_gpu_op_thomas_adjoint(n, ncol, p(tc), p(td), p(te), p(tx), p(tb), p(t_rb), p(t_cb),
                                                 p(t_db), p(t_eb), p(work)))
        got = [t.cpu().numpy() for t in (tx, t_rb, t_cb, t_db, t_eb)]
    finally:
        dm.close()
    assert np.array_equal(got[0], x)
    assert np.array_equal(got[1], r_bar)
    assert np.array_equal(got[2][:-1], -r_bar[1:] * x[:-1])
    assert np.array_equal(got[3], -r_bar * x)
    assert np.array_equal(got[4][:-1], -r_bar[:-1] * x[1:])
    assert np.all(got[2][-1] == 7.0) and np.all(got[4][-1] == 7.0)
