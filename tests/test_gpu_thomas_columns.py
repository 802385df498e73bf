"""The three-band solve and its adjoint of three and four rows, where the
kernel with one column per lane and a work array gives way to the one with
quotients in LDS (against the recurrence, equal), and of more columns than a 32-bit byte
offset reaches (2^29 doubles): every column's solution is its own.  Bands of
zero and a diagonal of two make the solution half the right-hand side, which
counts the columns, so every value is exact and no two columns share one."""
import ctypes as C

import pytest

import test_gpu_thomas_sizes as sizes
from conftest import get_grid

pytestmark = pytest.mark.gpu

COLUMNS = (1 << 29) + 1077


@pytest.fixture(scope="module")
def lib():
    import torch
    from game_archived_amd.rkhevi import DeviceModel
    dm = DeviceModel(get_grid(3))
    yield dm
    dm.close()
    torch.cuda.empty_cache()


def p(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n", [1, 2])
def test_solve(lib, n):
    import torch
    filled = lambda v: torch.full((n, COLUMNS), v, dtype=torch.float64, device="cuda")
    zero, d, x, work = filled(0.0), filled(2.0), filled(7.0), filled(7.0)
    r = torch.arange(n * COLUMNS, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    print(f"case: {n} rows, {COLUMNS} columns", flush=True)
    lib._check(lib.lib.game_gpu_op_thomas(n, COLUMNS, p(zero), p(d), p(zero), p(r), p(x), p(work)))
    assert torch.equal(x.view(-1), r.mul_(0.5))


def test_adjoint(lib):
    import torch
    filled = lambda v: torch.full((COLUMNS,), v, dtype=torch.float64, device="cuda")
    bands, d, x, r_bar, d_bar, work = filled(0.0), filled(2.0), filled(0.5), filled(7.0), filled(7.0), filled(7.0)
    x_bar = torch.arange(1, COLUMNS + 1, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    print(f"case: adjoint, 1 row, {COLUMNS} columns", flush=True)
    # a single row has no bands: their cotangents are not written
    lib._check(lib.lib.game_gpu_op_thomas_adjoint(1, COLUMNS, p(bands), p(d), p(bands), p(x), p(x_bar), p(r_bar), p(bands),
                                                  p(d_bar), p(bands), p(work)))
    assert torch.equal(r_bar, x_bar.mul_(0.5))
    assert torch.equal(d_bar, x_bar.mul_(-0.5))
    assert not bands.any()


@pytest.mark.parametrize("n", [3, 4])
@pytest.mark.parametrize("ncol", [1, 513])
def test_few_rows(n, ncol):
    sizes.test_solve_and_adjoint_equal_the_recurrence(n, ncol)
