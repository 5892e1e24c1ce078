"""D3Q27 stencil widths between the kernels' own (padded to the next multiple
of 8): whole steps against the FP64 oracle with and without tile unions, single
RK4 stages against FP64 numpy, rows that no stencil names, and a batch that
mixes widths sharing a padded one."""
import numpy as np
import pytest

import naga_amd
from tests.scenes import gpu_engine, grid_nodes, oracle_engine, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [11, 12, 15, 17, 20, 24, 25, 31, 33, 40, 41, 47, 49])
@pytest.mark.parametrize("unions", ["1", "0"])
def test_padded_widths_against_the_oracle(oracle64, monkeypatch, k, unions):
    monkeypatch.setenv("NAGA_UNIONS", unions)
    h = 0.1
    nodes = grid_nodes(oracle64, 3, h, 2 * h)
    eng, ref = gpu_engine(nodes, 27, k, h, kb=20), oracle_engine(oracle64, nodes, 27, k, h, kb=20)
    eng.set_initial_pulse([0.4, 0.5, 0.6], 1e-3, 0.15)
    ref.set_pulse([0.4, 0.5, 0.6], 1e-3, 0.15)
    eng.step_forward(10)
    ref.step(10)
    a, b = eng.macroscopic(fresh=True), ref.get(fresh=True)
    assert rel_l2(a["drho"], b["drho"]) < 1e-5 and rel_l2(a["u"], b["u"]) < 1e-5
    p = eng.setup_products()  # the stencils themselves keep their width
    assert p["idx"].shape[1] == k and p["W"].shape[1] == k


def test_batch_of_widths_sharing_a_padded_one(oracle64):
    h = 0.1
    nodes = grid_nodes(oracle64, 3, h, 2 * h)
    ks = (32, 27, 24, 30, 21)
    alone, scenes = ([gpu_engine(nodes, 27, k, h, kb=20) for k in ks] for _ in range(2))
    for e in alone + scenes:
        e.set_initial_pulse([0.4, 0.5, 0.6], 1e-3, 0.15)
    batch = naga_amd.SceneBatch(scenes)
    batch.step_forward(8)
    for e in alone:
        e.step_forward(8)
    for a, b in zip(alone, scenes):
        assert np.array_equal(a.macroscopic()["drho"], b.macroscopic()["drho"])
    batch.close()


@pytest.mark.parametrize("n,n_fluid,k", [(1, 1, 12), (33, 31, 11), (65, 64, 12), (97, 95, 13),
                                         (301, 257, 15), (129, 127, 17), (333, 300, 20),
                                         (95, 95, 31), (257, 201, 33), (63, 61, 41),
                                         (131, 130, 47), (99, 77, 49)])
@pytest.mark.parametrize("stage", [1, 2, 3, 4])
def test_single_stages_of_any_width(n, n_fluid, k, stage):
    rng = np.random.default_rng(n + k + stage)
    c, _, _, _ = naga_amd.lattice_tables(27)
    idx = rng.integers(0, n, (n_fluid, k)).astype(np.uint32)
    W = rng.standard_normal((n_fluid, k, 3)).astype(np.float32)
    y, f, y1, y2 = (rng.standard_normal((n, 27)).astype(np.float32) for _ in range(4))
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
    # FP32 rounding of a sum of k products (three terms each) scaled by dt,
    # and of the sums of the four rows
    size = np.einsum("ikd,ad,ika->ia", np.abs(W).astype(np.float64), np.abs(c), np.abs(g)[idx])
    most = max(np.abs(v).max() for v in (y, f, y1, y2))
    assert np.abs(got - want).max() < 2.0 ** -24 * ((k + 6) * dt * size.max() + 16 * most)


@pytest.mark.parametrize("Q,k", [(9, 5), (9, 16), (27, 11), (27, 13), (27, 32)])
@pytest.mark.parametrize("stage", [2, 3])
def test_rows_outside_a_stencil_are_not_read(Q, k, stage):
    """Infinities in rows that no stencil entry names change nothing, also for
    those rows' own nodes (padding records must name entries of the stencil)."""
    rng = np.random.default_rng(k)
    n, D = 100, 2 if Q == 9 else 3
    idx = rng.integers(0, 90, (n, k)).astype(np.uint32)
    W = rng.standard_normal((n, k, D)).astype(np.float32)
    y = rng.standard_normal((n, Q)).astype(np.float32)
    f = y.copy()
    f[95:] = np.inf
    a, b = (naga_amd.rk4_stage(stage, y, idx, W, 0.01, stage_input=v) for v in (f, y))
    assert np.array_equal(a, b)
