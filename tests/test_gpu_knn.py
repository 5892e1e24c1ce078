"""Exact kNN of clouds that each part of the search serves: boxes of cells
(evenly spread points), radii retried (clusters, edges of the cloud, ties),
narrow cells (crowded clouds), rings (points far apart, distances past the
largest float), against brute force with the same FP32 keys; and the time of
repeated points and crowded clouds against random ones."""
import time

import numpy as np
import pytest
import torch

import naga_amd

pytestmark = pytest.mark.gpu


def _brute(ref, query, k):
    """Keys (FP32 squared distance, index) in ascending order."""
    d2 = np.empty((len(query), len(ref)), np.float32)
    with np.errstate(over="ignore"):
        for b in range(0, len(query), 256):
            q = query[b:b + 256]
            s = (q[:, None, 0] - ref[None, :, 0]) ** 2
            for d in range(1, ref.shape[1]):
                s = (q[:, None, d] - ref[None, :, d]) ** 2 + s
            d2[b:b + 256] = s
    order = np.argsort(d2, axis=1, kind="stable")[:, :k]
    return np.take_along_axis(d2, order, 1), order.astype(np.uint32)


def _cloud(kind, D, n, rng):
    if kind == "uniform":
        return rng.random((n, D)).astype(np.float32)
    if kind == "cluster":  # most points in a ball of a hundredth of the box
        p = rng.random((n, D))
        p[: 3 * n // 4] = 0.4 + 0.01 * p[: 3 * n // 4]
        return p.astype(np.float32)
    if kind == "lattice":
        m = int(round(n ** (1.0 / D)))
        return np.stack(np.meshgrid(*[np.arange(m, dtype=np.float32)] * D, indexing="ij"),
                        -1).reshape(-1, D)
    if kind == "repeated":  # every point many times: ties at distance zero
        return np.repeat(rng.random((max(n // 100, 1), D)), 100, axis=0)[:n].astype(np.float32)
    if kind == "line":
        p = np.zeros((n, D), np.float32)
        p[:, 0] = rng.random(n)
        return p
    p = rng.random((n, D)).astype(np.float32)  # "huge": squares overflow to infinity
    p[::2] *= np.float32(1e20)
    return p


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("kind", ["uniform", "cluster", "lattice", "repeated", "line", "huge"])
@pytest.mark.parametrize("n,k", [(4096, 32), (4096, 1), (3000, 64), (3000, 17), (64, 64), (65, 33)])
def test_knn_matches_brute_force(D, kind, n, k):
    rng = np.random.default_rng(n + 10 * k + D)
    ref = _cloud(kind, D, n, rng)
    k = min(k, len(ref))
    lo, hi = ref.min(0), np.minimum(ref.max(0), 2.0)
    out = (lo + (hi - lo) * (1.4 * rng.random((200, D)) - 0.2)).astype(np.float32)
    query = np.concatenate([ref[:: max(1, len(ref) // 300)], out])
    print(f"kNN D={D} {kind} n={len(ref)} k={k} queries={len(query)}", flush=True)
    d2, idx = naga_amd.batched_nearest_neighbors(k, query, ref)
    want_d2, want_idx = _brute(ref, query, k)
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(d2.view(np.uint32), want_d2.view(np.uint32))


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("times", [65, 255, 257, 400, 1500])
@pytest.mark.parametrize("k", [1, 17, 64])
def test_repeated_points_match_brute_force(D, times, k):
    """Groups of equal points around the sizes of a wavefront and of a query's
    kept points, so that ties run through every bound: indices decide."""
    rng = np.random.default_rng(times + k)
    ref = np.repeat(rng.random((12, D)).astype(np.float32), times, axis=0)[rng.permutation(12 * times)]
    query = np.concatenate([ref[:40], rng.random((60, D)).astype(np.float32)])
    print(f"kNN D={D} times={times} k={k}", flush=True)
    d2, idx = naga_amd.batched_nearest_neighbors(k, query, ref)
    want_d2, want_idx = _brute(ref, query, k)
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(d2.view(np.uint32), want_d2.view(np.uint32))


def _device_time(ref, k):
    """Median time (s) of the search of ref's own neighbours, on device arrays."""
    n, D = ref.shape
    r = torch.from_numpy(ref).cuda()
    d2 = torch.empty(n, k, dtype=torch.float32, device="cuda")
    idx = torch.empty(n, k, dtype=torch.int32, device="cuda")
    t = []
    for _ in range(7):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        assert naga_amd.load().naga_knn_noalloc(
            r.data_ptr(), n, r.data_ptr(), n, D, k, d2.data_ptr(), idx.data_ptr(),
            torch.cuda.current_stream().cuda_stream) == 0
        torch.cuda.synchronize()
        t.append(time.perf_counter() - t0)
    return float(np.median(t))


@pytest.mark.parametrize("D", [2, 3])
def test_repeated_points_take_no_rings(D):
    """300-fold repeated points are searched in a few times the time of as many
    random ones (by rings of cells it was eight to fourteen times)."""
    rng = np.random.default_rng(D)
    p = rng.random((199800, D)).astype(np.float32)
    t = [_device_time(c, 16) for c in (p, np.repeat(p[:666], 300, axis=0))]
    print(t, flush=True)
    assert t[1] < 4.0 * t[0]


def _crowded(kind, D, n, rng):
    """Clouds that leave most of their bounding box empty."""
    if kind == "circle":
        p = rng.standard_normal((n, D))
        p[:, 2:] *= 0.01
        return (p / np.linalg.norm(p, axis=1, keepdims=True)).astype(np.float32)
    p = rng.random((n, D))  # "blob": nine tenths within about 0.05
    p[: 9 * n // 10] = 0.5 + 0.02 * rng.standard_normal((9 * n // 10, D))
    return p.astype(np.float32)


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("kind", ["circle", "blob"])
@pytest.mark.parametrize("k", [2, 9, 32, 64])
def test_crowded_clouds_match_brute_force(D, kind, k):
    rng = np.random.default_rng(k)
    ref = _crowded(kind, D, 6000, rng)
    query = np.concatenate([ref[::20], rng.uniform(-1.2, 1.2, (100, D)).astype(np.float32)])
    print(f"kNN D={D} {kind} k={k}", flush=True)
    d2, idx = naga_amd.batched_nearest_neighbors(k, query, ref)
    want_d2, want_idx = _brute(ref, query, k)
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(d2.view(np.uint32), want_d2.view(np.uint32))


@pytest.mark.parametrize("k", [32, 64])
def test_crowded_clouds_get_narrow_cells(k):
    """200,000 points on a circle are searched in less than three times the time
    of as many random ones (in cells sized for k points at the mean density it
    was four to five times)."""
    rng = np.random.default_rng(k)
    p = rng.random((200000, 2)).astype(np.float32)
    t = [_device_time(c, k) for c in (p, _crowded("circle", 2, 200000, rng))]
    print(t, flush=True)
    assert t[1] < 3.0 * t[0]


@pytest.mark.parametrize("approx", [1, 8, 64, 5000])
def test_knn_of_segmentations_matches_brute_force(approx):
    """Cells of any size given by the caller."""
    rng = np.random.default_rng(approx)
    ref = rng.random((5000, 3)).astype(np.float32)
    query = (rng.random((300, 3)) * 1.2 - 0.1).astype(np.float32)
    seg = naga_amd.NdCubicSegmentation(ref, approx_partition_size=approx)
    d2, idx = seg.batched_nearest_neighbors(32, query)
    want_d2, want_idx = _brute(ref, query, 32)
    assert np.array_equal(idx, want_idx) and np.array_equal(d2, want_d2)
