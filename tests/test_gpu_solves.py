"""The wavefront solves at every register width's edges: batched systems
against numpy, and the stencil weights of narrow to widest stencils (on an
unjittered grid too, whose pivots tie) against the FP64 oracle."""
import numpy as np
import pytest

import naga_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 19, 20, 21, 28, 29, 36, 37, 44, 52, 53, 63, 64])
def test_batched_inverse_sizes(n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((40, n, n)) + np.eye(n)
    A[1] = np.eye(n)[rng.permutation(n)]  # every pivot moves, every tie is exact
    A[2] *= 1e-200
    A[3] *= 1e200
    inv, info = naga_amd.batched_matrix_inverse(A, return_info=True)
    assert not info.any()
    want = np.linalg.inv(A)
    err = np.abs(inv - want).max((1, 2)) / np.abs(want).max((1, 2))
    cond = np.linalg.cond(A)
    assert (err <= 1e-14 * n * cond).all()
    assert np.array_equal(inv[1], want[1])


@pytest.mark.parametrize("D,k", [(2, 8), (2, 12), (2, 17), (2, 24), (2, 25), (3, 12), (3, 16),
                                 (3, 24), (3, 32), (3, 33), (3, 48), (3, 60)])
@pytest.mark.parametrize("rbf", [0, 1])
@pytest.mark.parametrize("jitter", [0.25, 0.0])
def test_stencil_weights_every_width(oracle64, D, k, rbf, jitter):
    h = 0.08 if D == 2 else 0.15
    pts = oracle64.uniform_grid(D, [0] * D, [1] * D, h, jitter=jitter)["points"]
    d2, idx = oracle64.knn(pts, pts, k)
    W, info = oracle64.divergence_weights(pts, pts, idx, d2, rbf)
    try:
        op = naga_amd.DivergenceOperator.create(pts, k=k, rbf=rbf)
    except RuntimeError:  # stencils in one line or plane are singular for both
        assert np.any(info)
        return
    assert np.array_equal(op.support_indices(), idx)
    good = np.abs(W).max((1, 2)) < 1e3 / h  # near-singular stencils have no exact weights
    assert good.mean() > 0.5
    scale = np.abs(W[good]).max()
    assert np.abs(op.weights()[good] - W[good]).max() < 1e-7 * scale
