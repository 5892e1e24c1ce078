"""D3Q27 stencil widths between the kernels' own (padded to the next multiple
of 8): whole steps against the FP64 oracle with and without tile unions, per
node widths, and a batch that mixes widths sharing a padded one."""
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
