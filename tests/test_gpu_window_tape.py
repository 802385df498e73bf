"""The window's tape: a step on it writes its results into the tape's buffers,
so neither the checkpoint interval (one step per segment, uneven last segments,
one segment) nor buffers left by an earlier window change a bit of the
gradient, and the resident states are afterwards those of the first segment's
steps taken one by one."""
import numpy as np
import pytest

from conftest import get_grid, oracle_state

pytestmark = pytest.mark.gpu

STEPS, DT = 5, 300.0
FIELDS = ("rho", "rhotheta_v", "theta_v_pert", "exner_pert", "wind")


@pytest.mark.parametrize("oro", ["flat", "gaussian"])
def test_checkpoint_interval_changes_no_bit(oro):
    from test_gpu_window import Window
    grid = get_grid(3, oro)
    a, b = oracle_state(grid), oracle_state(grid, seed=7)
    w = Window(grid)
    try:
        # a surface and top w that no step writes
        wind, d = np.array(a.wind), grid.dims
        rng = np.random.default_rng(3)
        wind[:d.nsh] = 1e-3 * rng.standard_normal(d.nsh)
        wind[-d.nsh:] = 1e-3 * rng.standard_normal(d.nsh)
        x = [w.dev(v) for v in (a.rho, a.rhotheta_v, wind)]
        target = w.dev(b.rho)
        want = None
        for k in (5, 2, 1, 3, 4, 7):
            print(f"case: window res 3 x 26 {oro}, {STEPS} steps, checkpoint every {k}", flush=True)
            cost, g = w.gradient(STEPS, DT, k, x, target)
            got = [np.array([cost])] + [t.cpu().numpy() for t in g]
            assert all(np.isfinite(v).all() for v in got)
            left = w.dm.get_state()
            left = [np.array(getattr(left, f)) for f in FIELDS]
            w.forward(min(k, STEPS), DT, x)
            steps = w.dm.get_state()
            for f, v in zip(FIELDS, left):
                assert np.array_equal(v, getattr(steps, f)), (k, f)
            if want is None:
                want = got
            for u, v in zip(want, got):
                assert np.array_equal(u, v), k
    finally:
        w.close()
