"""Initial pulses of any width, down to ones whose square underflows: the
density at a pulse's centre is its amplitude, and zero elsewhere for a width far
below the spacing."""
import numpy as np
import pytest

from tests.scenes import gpu_engine, grid_nodes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Q", [9, 27])
@pytest.mark.parametrize("width", [1e-3, 1e-150, 1e-155, 1e-160])
def test_narrow_pulse(oracle64, Q, width):
    h = 0.1
    nodes = grid_nodes(oracle64, 2 if Q == 9 else 3, h, 2 * h)
    eng = gpu_engine(nodes, Q, 16, h)
    eng.set_initial_pulse(nodes["points"][7].astype(np.float64), 1e-3, width)
    drho = eng.macroscopic(fresh=True)["drho"]
    assert abs(drho[7] - 1e-3) < 1e-9  # Q weights rounded to FP32
    assert np.abs(np.delete(drho, 7)).max() < 1e-9
