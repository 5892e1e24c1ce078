"""D2Q9 stencil passes at the edges of their blocks (128 nodes) and record
groups (four records): single RK4 stages against FP64 numpy, whole steps of
odd widths against the FP64 oracle and against the one-lane-per-distribution
kernels, layers on both sides of the number of partial sums that the field
pass reads itself, and the saved state's rows."""
import struct
import time

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


def test_states_load_at_the_link_rate():
    """Loading a D2Q9 state takes about as long per byte as a D3Q27 one, whose
    rows lie on the device as they are saved."""
    per_byte = []
    for Q, h in ((27, 0.02), (9, 0.001)):
        D = 2 if Q == 9 else 3
        nodes = naga_amd.UniformGridProvider([0] * D, [1] * D, h, 8 * h, 0.5, jitter=0.25,
                                             seed=5).get()
        eng = naga_amd.SimulationEngine(lattice=Q, k=16)
        p = naga_amd.problem_parameters(Q, 0.6, 0.4 * h)
        eng.set_problem_parameters(p["nu"], 1.0, p["dt"], p["c"])
        eng.init_domain(nodes)
        state, t = eng.save_state(), []
        for _ in range(9):
            t0 = time.perf_counter()
            eng.load_state(state)
            t.append(time.perf_counter() - t0)
        per_byte.append(float(np.median(t)) / len(state))
        eng.close()
    print(per_byte, flush=True)
    assert per_byte[1] < 2.5 * per_byte[0]


# nodes per side with a layer over nearly the whole square: 96, 294 and
# 307 partial sums of 64 layer nodes (the field pass reads up to 300 itself)
LAYERS = (80, 139, 142)


def _wide_layer(oracle, side):
    h = 1.0 / (side - 1)
    return h, grid_nodes(oracle, 2, h, 0.49)


def test_wide_layers_against_the_oracle(oracle64):
    scenes = [_wide_layer(oracle64, side) for side in LAYERS]
    parts = [-(-(n["n_bulk"] + n["n_layer"]) // 64) - n["n_bulk"] // 64 for _, n in scenes]
    assert parts[0] < parts[1] <= 300 < parts[2]
    alone, batched = ([gpu_engine(n, 9, 16, h) for h, n in scenes] for _ in range(2))
    for e in alone + batched:
        e.set_initial_pulse([0.4, 0.6], 1e-3, 0.1)
    batch = naga_amd.SceneBatch(batched)
    batch.step_forward(10)
    for (h, nodes), e, b in zip(scenes, alone, batched):
        ref = oracle_engine(oracle64, nodes, 9, 16, h)
        ref.set_pulse([0.4, 0.6], 1e-3, 0.1)
        ref.step(10)
        e.step_forward(10)
        got, want = e.macroscopic(fresh=True), ref.get(fresh=True)
        assert rel_l2(got["drho"], want["drho"]) < 1e-5 and rel_l2(got["u"], want["u"]) < 1e-5
        assert np.array_equal(got["drho"], b.macroscopic(fresh=True)["drho"])
    batch.close()


def test_layer_means_are_linear_in_the_layer():
    """The field pass and the means, which move a fraction of the bytes that the
    collision and its PML terms do, take no longer than it does, whatever the
    layer's width (a million nodes)."""
    h = 0.001
    for layer in (0.03, 0.3):
        nodes = naga_amd.UniformGridProvider([0, 0], [1, 1], h, layer, 0.5, jitter=0.25,
                                             seed=5).get()
        eng = naga_amd.SimulationEngine(lattice=9, k=16)
        p = naga_amd.problem_parameters(9, 0.6, 0.4 * h)
        eng.set_problem_parameters(p["nu"], 1.0, p["dt"], p["c"])
        eng.init_domain(nodes)
        eng.set_initial_pulse([0.4, 0.6], 1e-3, 0.1)
        eng.step_forward(2)
        ms = [eng.profile_step() for _ in range(7)]
        t = {name: float(np.median([m[name] for m in ms])) for name in ms[0]}
        print(layer, t, flush=True)
        assert t["pm_layer_means"] + t["pf_pml_field"] < t["p1_collide"] + t["pl_pml_local"]
        eng.close()
