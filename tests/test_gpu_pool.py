"""Device blocks kept between allocations: given back on request and within a
server's budget, and scenes rebuilt in memory that other scenes used, one after
another and from several threads at once, give the results of their first build
bit for bit."""
import threading

import numpy as np
import pytest
import torch

import naga_amd
from tests.scenes import gpu_engine, grid_nodes

pytestmark = pytest.mark.gpu

SCENES = [(27, 0.1, 32), (9, 0.04, 16), (27, 0.125, 20), (9, 0.03, 13), (27, 0.11, 32)]


def _solve(nodes, Q, k, h):
    eng = gpu_engine(nodes, Q, k, h, kb=16)
    eng.set_initial_pulse([0.4] * (2 if Q == 9 else 3), 1e-3, 0.15)
    eng.step_forward(12)
    out = eng.macroscopic(fresh=True)
    eng.close()
    return out


def test_kept_memory_is_given_back(oracle64):
    """Closed scenes' memory is kept for the next, and given back to the device by
    trim_memory."""
    nodes = grid_nodes(oracle64, 3, 0.04, 0.08)
    gpu_engine(nodes, 27, 32, 0.04, kb=16).close()  # the process' own memory: code, queues
    naga_amd.trim_memory()
    free = torch.cuda.mem_get_info()[0]
    gpu_engine(nodes, 27, 32, 0.04, kb=16).close()
    kept = naga_amd.trim_memory(1 << 40)
    assert kept > 10 << 20 and torch.cuda.mem_get_info()[0] < free
    assert naga_amd.trim_memory(kept // 2) <= kept // 2
    assert naga_amd.trim_memory() == 0
    assert torch.cuda.mem_get_info()[0] >= free - (2 << 20)


def test_server_keeps_within_its_budget(oracle64):
    """Memory kept from earlier scenes counts against a server's budget."""
    nodes = grid_nodes(oracle64, 3, 0.03, 0.06)
    gpu_engine(nodes, 27, 32, 0.03, kb=16).close()
    budget = 64 << 20
    assert naga_amd.trim_memory(1 << 40) > budget
    srv = naga_amd.SolveServer(hbm_budget_bytes=budget, max_active=4, chunk_steps=5)
    rid = srv.submit(naga_amd.make_request(9, 0.03125, 5))
    srv.drain()
    srv.result(rid)
    srv.close()
    assert naga_amd.trim_memory(1 << 40) <= budget


def _same(a, b):
    return all(np.array_equal(a[f], b[f]) for f in ("rho", "drho", "u"))


def test_rebuilt_scenes_and_threads(oracle64):
    nodes = [grid_nodes(oracle64, 2 if Q == 9 else 3, h, 2 * h) for Q, h, _ in SCENES]
    first = [_solve(n, Q, k, h) for n, (Q, h, k) in zip(nodes, SCENES)]
    for _ in range(2):  # now in blocks of the scenes before
        for n, (Q, h, k), want in reversed(list(zip(nodes, SCENES, first))):
            assert _same(_solve(n, Q, k, h), want)
    bad = []

    def work(t):
        for r in range(4):
            i = (t + r) % len(SCENES)
            Q, h, k = SCENES[i]
            try:
                if not _same(_solve(nodes[i], Q, k, h), first[i]):
                    bad.append((t, r, i))
            except Exception as e:  # a thread's error is the test's
                bad.append((t, r, i, str(e)))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
