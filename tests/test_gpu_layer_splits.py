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


@pytest.mark.parametrize("oro", ["flat", "gaussian"])
def test_splits_change_no_bit_of_the_operators(monkeypatch, oro):
    """the operators and their adjoints: chunks that carry the value of the
    layer above, with random fields"""
    import torch
    from adjoint_harness import Ops
    from game_archived_amd.rkhevi import DeviceModel
    from test_gpu_adjoint import OPS, rand
    grid = get_grid(3, oro, n_layers=14, n_oro=11)

    def results():
        dm = DeviceModel(grid)
        try:
            ops = Ops(dm)
            sz = ops.sizes()
            out = {}
            for name, nin, nout, nfix in OPS:
                x, y = rand(torch, sz[nin], 1), rand(torch, sz[nout], 2)
                fixed = [rand(torch, sz[nfix], 3)] if nfix else []
                ax, aty = ops.new(sz[nout]), ops.new(sz[nin])
                ops._run(name, x, *fixed, ax)
                ops._run(name + "_adjoint", *fixed, y, aty)
                out[name] = (ax.cpu().numpy(), aty.cpu().numpy())
        finally:
            dm.close()
        return out

    want = results()
    for split in (1, 2, 3, 5, 7, 13, 14):
        monkeypatch.setenv("GAME_GPU_SPLIT_CELL", str(split))
        monkeypatch.setenv("GAME_GPU_SPLIT_EDGE", str(split))
        print(f"case: operators, res 3 x 14 {oro}, {split} chunks", flush=True)
        got = results()
        for name, pair in want.items():
            for a, b in zip(pair, got[name]):
                assert np.array_equal(a, b), (split, name)
