"""D2Q9 stencil passes at the edges of their blocks (128 nodes) and record
groups (four records): single RK4 stages against FP64 numpy, whole steps of
odd widths against the FP64 oracle and against the one-lane-per-distribution
kernels, and the saved state's rows."""
import struct

import numpy as np
import pytest

import naga_amd
from tests.scenes import gpu_engine, grid_nodes, oracle_engine, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,n_fluid,k", [(1, 1, 1), (127, 127, 3), (128, 128, 4), (129, 128, 5),
                                         (300, 257, 8), (700, 640, 13), (500, 0, 6),
                                         (1000, 999, 64)])
@pytest.mark.parametrize("stage", [1, 2, 3, 4])
def test_rk4_stage_block_edges(n, n_fluid, k, stage):
    rng = np.random.default_rng(n + k + stage)
    c, _, _, _ = naga_amd.lattice_tables(9)
    idx = rng.integers(0, n, (n_fluid, k)).astype(np.uint32)
    W = rng.standard_normal((n_fluid, k, 2)).astype(np.float32)
    y, f, y1, y2 = (rng.standard_normal((n, 9)).astype(np.float32) for _ in range(4))
    dt = 0.01
    got = naga_amd.rk4_stage(stage, y, idx, W, dt, n_fluid=n_fluid, stage_input=f, y1=y1, y2=y2)
    g = (y if stage == 1 else f).astype(np.float64)
    r = -np.einsum("ikd,ad,ika->ia", W.astype(np.float64), c, g[idx])
    want = y.astype(np.float64)
    Y = want[:n_fluid]
    if stage < 4:
        want[:n_fluid] = Y + (dt if stage == 3 else dt / 2) * r
    else:
        want[:n_fluid] = Y + ((y1[:n_fluid] - Y) + 2 * (y2[:n_fluid] - Y) +
                              (g[:n_fluid] - Y)) / 3 + dt / 6 * r
    # k products of unit size summed in FP32, scaled by dt
    assert np.abs(got - want).max() < 4e-7 * (8 + dt * k * 12)


@pytest.mark.parametrize("k", [12, 13, 15, 17, 22, 24, 31])
def test_odd_widths_against_the_oracle(oracle64, k):
    h = 0.04
    nodes = grid_nodes(oracle64, 2, h, 3 * h)
    eng, ref = gpu_engine(nodes, 9, k, h), oracle_engine(oracle64, nodes, 9, k, h)
    other = gpu_engine(nodes, 9, k, h)
    for e in (eng, ref, other):
        (e.set_pulse if e is ref else e.set_initial_pulse)([0.4, 0.6], 1e-3, 0.1)
    batch = naga_amd.SceneBatch([other])
    batch.set_q9_kernels(9)
    eng.step_forward(20)
    ref.step(20)
    batch.step_forward(20)
    a, b, c = eng.macroscopic(fresh=True), ref.get(fresh=True), other.macroscopic(fresh=True)
    for f in ("drho", "u"):
        assert rel_l2(a[f], b[f]) < 1e-5
        assert rel_l2(a[f], c[f]) < 1e-6
    batch.close()


def test_saved_state_rows(oracle64):
    """A saved state holds [N][9] rows in node order after its
    header, and loading it restores them."""
    h = 0.05
    nodes = grid_nodes(oracle64, 2, h, 3 * h)
    eng = gpu_engine(nodes, 9, 16, h)
    eng.set_initial_pulse([0.5, 0.5], 1e-3, 0.1)
    eng.step_forward(3)
    state, g = eng.save_state(), eng.distributions()["g"]
    N = eng.num_nodes
    assert state[:8] == b"NAGAST02" and struct.unpack("<3i", state[8:20]) == (9, 2, 9)
    head = len(state) - 4 * (2 * 9 * N + 4 * N + N + 2 * N)
    rows = np.frombuffer(state, np.float32, 9 * N, head).reshape(N, 9)
    assert np.array_equal(rows, g.T.astype(np.float32))
    eng.step_forward(2)
    want = eng.distributions()["g"]
    eng.load_state(state)
    assert np.array_equal(eng.distributions()["g"], g)
    eng.step_forward(2)
    assert np.array_equal(eng.distributions()["g"], want)
