"""Neighbour queries at the edges of their kernels' buffers and lane groups, against brute force:
squared distances in FP64 in the kernels' own order of operations, so every comparison is exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _upload(ctx, x):
    import cuda_3d_amd as g

    return g.PointCloud.from_numpy(x, np.zeros_like(x), ctx=ctx)


def _dist2(q, p):
    d = q[:, None, :].astype(np.float64) - p[None, :, :].astype(np.float64)
    return (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]


def _cloud(kind, n, rng):
    if kind == "uniform":
        return rng.uniform(-0.1, 0.1, (n, 3)).astype(np.float32)
    if kind == "plane":
        x = rng.uniform(-0.1, 0.1, (n, 3))
        x[:, 2] = 1.0 + 1e-3 * rng.normal(size=n)
        return x.astype(np.float32)
    if kind == "lattice":  # equal distances everywhere
        return (rng.integers(-5, 6, (n, 3)) * np.float32(0.015625)).astype(np.float32)
    return np.tile(np.float32([[0.01, 0.02, 0.03]]), (n, 1))  # one place: only indices order them


@pytest.mark.parametrize("kind,n,r", [
    ("uniform", 1, 0.05), ("uniform", 63, 0.05), ("uniform", 700, 0.15), ("uniform", 3000, 0.15),
    ("plane", 2500, 0.03), ("plane", 2500, 0.4), ("lattice", 1900, 0.05), ("lattice", 1900, 0.3),
    ("place", 64, 0.01), ("place", 129, 0.01), ("place", 448, 0.01), ("place", 449, 0.01), ("place", 512, 0.01),
    ("place", 513, 0.01), ("place", 1500, 0.01)])
def test_neighbour_queries(ctx, kind, n, r):
    import cuda_3d_amd as g

    rng = np.random.default_rng(n)
    ref = _cloud(kind, n, rng)
    far = np.float32([[5, 5, 5], [-0.3, 0.0, 0.0], [0.1, 0.1, 0.1], [np.nan, 0, 0]])  # outside the grid, at its corner
    qry = np.concatenate([ref[rng.permutation(n)[:37]], _cloud(kind, 6, rng), far])
    d2, r2 = _dist2(qry, ref), np.float64(np.float32(r)) ** 2
    order = np.lexsort((np.broadcast_to(np.arange(n), d2.shape), d2), axis=1)
    cq, cr = _upload(ctx, qry), _upload(ctx, ref)
    for K in (0, 1, 30, 64, 128, 129, 447, 448, 449, 1000):
        off, idx = g.PointCloud.radius_search(cq, cr, r, K)
        for k in range(len(qry)):
            want = order[k][d2[k][order[k]] < r2]
            want = want[:K] if K else want
            np.testing.assert_array_equal(idx[off[k]:off[k + 1]], want, err_msg=f"K {K} query {k}")
    near = np.where(np.nan_to_num(d2, nan=np.inf).min(1) < r2, order[:, 0], -1)
    np.testing.assert_array_equal(g.PointCloud.nn_search(cq, cr, r), near)
    count = (_dist2(ref, ref) < r2).sum(1)
    for m in (-1, 0, 1, 8, int(np.median(count)), n):
        np.testing.assert_array_equal(cr.radius_outlier_removal(r, m).download()[0], ref[count > m], err_msg=f"min {m}")
