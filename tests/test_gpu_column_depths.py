"""The column solvers at the depths where their layout changes -- lanes per
block of the sound-wave solver (16 and 32 layers), rows and waves per block of
the tracer solve (9, 18 and 27 layers, multiples of seven beyond), chunks of
the sediment heat -- against the streaming forms with one column per lane and
the sediment heat box by box, bit for bit: the layout changes which thread
forms a value, never its arithmetic."""
import numpy as np
import pytest

from conftest import get_grid, oracle_state

pytestmark = pytest.mark.gpu


def run(grid, state, precision):
    from game_archived_amd.rkhevi import DeviceModel
    dm = DeviceModel(grid, precision=precision)
    try:
        dm.start(state)
        dm.run(2, 120.0)
        out = dict(dm.get_state().arrays())
        out.update(dm.get_irrev().arrays())
    finally:
        dm.close()
    return out


@pytest.mark.parametrize("res,layers", [(3, 4), (3, 5), (3, 9), (3, 10), (3, 16), (3, 17), (3, 18), (3, 19), (3, 27), (3, 28),
                                        (3, 32), (3, 33), (3, 35), (3, 36), (3, 56), (3, 57), (3, 63), (5, 41)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_depths_change_no_bit(monkeypatch, res, layers, precision):
    from game_archived_amd.rkhevi import FP64, MIXED
    prec = {"fp64": FP64, "mixed": MIXED}[precision]
    print(f"case: column solvers, res {res} x {layers} moist, {precision}", flush=True)
    grid = get_grid(res, "flat", moist=1, n_layers=layers, n_oro=layers - 2)
    state = oracle_state(grid, moist=True)
    got = run(grid, state, prec)
    for switch in ("GAME_GPU_VW_STREAMING", "GAME_GPU_GD_STREAMING", "GAME_GPU_SH_PER_BOX"):
        monkeypatch.setenv(switch, "1")
    want = run(grid, state, prec)
    for k in want:
        assert np.isfinite(got[k]).all(), k
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("layers", [26, 41])
def test_an_infinite_wind_spreads_alike(monkeypatch, layers):
    """an infinite vertical wind, up and down, in rows within and at the ends
    of a wave's rows: the same boxes become not-a-number"""
    print(f"case: infinite winds, res 3 x {layers} moist", flush=True)
    grid = get_grid(3, "flat", moist=1, n_layers=layers, n_oro=layers - 2)
    state, d = oracle_state(grid, moist=True), grid.dims
    for n, level in enumerate((3, 7, 8, 9, 10, 14, 18, layers - 1)):
        for cell, sign in ((40 * n + 20, 1.0), (40 * n + 330, -1.0)):
            state.wind[level * d.vpl + cell] = sign * np.inf
    from game_archived_amd.rkhevi import DeviceModel

    def tracers():
        dm = DeviceModel(grid)
        try:
            dm.start(state)
            dm.run(1, 120.0)
            return np.array(dm.get_state().rho)
        finally:
            dm.close()

    got = tracers()
    monkeypatch.setenv("GAME_GPU_GD_STREAMING", "1")
    want = tracers()
    assert np.isnan(want).any() and np.isfinite(want).any()
    assert np.array_equal(got, want, equal_nan=True)
