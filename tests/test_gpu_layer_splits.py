"""The layer splits of the column-walking kernels: every chunk length that has
a kernel of its own (one, two and three layers per cell thread, the loop for
longer chunks) and uneven last chunks, over the mountain (chunks that begin in
and above the terrain layers) and with moisture, against the default splits,
bit for bit: the split changes which thread forms a value, never its
arithmetic."""
import numpy as np
import pytest

from conftest import get_grid, oracle_state

pytestmark = pytest.mark.gpu


def run(grid, state):
    from game_archived_amd.rkhevi import DeviceModel
    dm = DeviceModel(grid)
    try:
        dm.start(state)
        dm.run(2, 240.0)
        out = dict(dm.get_state().arrays())
        out.update(dm.get_forcings().arrays())
        out.update(dm.get_diagnostics().arrays())
    finally:
        dm.close()
    return out


@pytest.mark.parametrize("moist", [0, 1])
def test_splits_change_no_bit(monkeypatch, moist):
    grid = get_grid(3, "gaussian", moist=moist, n_layers=14, n_oro=11)
    state = oracle_state(grid, moist=bool(moist))
    want = run(grid, state)
    for split in (1, 2, 3, 5, 7, 13, 14):
        monkeypatch.setenv("GAME_GPU_SPLIT_CELL", str(split))
        monkeypatch.setenv("GAME_GPU_SPLIT_EDGE", str(split))
        print(f"case: res 3 x 14, moist {moist}, {split} chunks", flush=True)
        got = run(grid, state)
        for k in want:
            assert np.array_equal(got[k], want[k]), (split, k)
