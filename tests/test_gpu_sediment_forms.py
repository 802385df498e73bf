"""The sediment heat in each form that the size of a grid chooses -- chunks of
two and of five layers, whole columns -- at depths that fill a chunk or a turn
of the column's loop and that leave a remainder, and at the least depth,
against one box per thread, bit for bit: the form changes which thread forms a
value, never its arithmetic."""
import numpy as np
import pytest

from conftest import get_grid, oracle_state
from test_gpu_parity import seeded_condensates

pytestmark = pytest.mark.gpu


def run(grid, state, precision):
    from game_archived_amd.rkhevi import FP64, MIXED, DeviceModel
    dm = DeviceModel(grid, precision={"fp64": FP64, "mixed": MIXED}[precision])
    try:
        dm.start(state)
        dm.run(2, 120.0)
        out = dict(dm.get_state().arrays())
        out.update(dm.get_irrev().arrays())
    finally:
        dm.close()
    return out


@pytest.mark.parametrize("layers", [3, 4, 5, 8, 9, 26, 41])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_form_changes_no_bit(monkeypatch, layers, precision):
    grid = get_grid(3, "gaussian", moist=1, n_layers=layers, n_oro=layers - 2)
    state = seeded_condensates(grid, oracle_state(grid, moist=True))
    monkeypatch.setenv("GAME_GPU_SH_LAYERS", "1")
    want = run(grid, state, precision)
    assert np.abs(want["condensates_sediment_heat"]).max() > 0
    for form in ("2", "5", "all"):
        print(f"case: sediment heat, res 3 x {layers}, {precision}, {form} layers per thread", flush=True)
        monkeypatch.setenv("GAME_GPU_SH_LAYERS", form)
        got = run(grid, state, precision)
        for k in want:
            assert np.array_equal(got[k], want[k]), (form, k)


def test_an_unknown_form_is_refused(monkeypatch):
    from game_archived_amd.rkhevi import DeviceModel, GameError
    monkeypatch.setenv("GAME_GPU_SH_LAYERS", "3")
    with pytest.raises(GameError, match="GAME_GPU_SH_LAYERS"):
        DeviceModel(get_grid(3, "gaussian", moist=1))
