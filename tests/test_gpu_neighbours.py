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


@pytest.mark.parametrize("kind,n,r", [
    ("uniform", 2, 0.05), ("uniform", 65, 0.1), ("uniform", 1200, 0.09), ("plane", 2500, 0.02), ("plane", 2500, 0.04),
    ("lattice", 1900, 0.03), ("lattice", 1900, 0.08), ("place", 30, 0.01), ("place", 97, 0.01), ("place", 600, 0.01),
    ("uniform", 4200, 0.5)])
def test_normals_and_gradient(ctx, kind, n, r):
    """Normals and gradients with neighbourhoods around the group's buffer (96), the wavefront's
    (448) and the exact sums' bound (4096), and with ties: the oracle's FP64 operations on the
    same integer sums, so the same bits."""
    import cuda_3d_amd as g
    import oracle as O

    rng = np.random.default_rng(n)
    x = _cloud(kind, n, rng)
    pc = g.PointCloud.from_numpy(x, rng.uniform(0, 1, x.shape).astype(np.float32), ctx=ctx)
    xyzi = pc.download_xyzi()
    for K in ((0, 30, 1000) if n > 4000 else (0, 1, 3, 30, 95, 96, 97, 448, 449, 1000)):
        assert pc.estimate_normals(r, K)
        nrm = O.estimate_normals(xyzi, r, K)
        np.testing.assert_array_equal(pc.download_normals(), nrm[:, :3], err_msg=f"normals, {K} nearest")
        assert pc.compute_color_gradient(r, K)
        np.testing.assert_array_equal(pc.download_gradient(), O.color_gradient(xyzi, nrm, r, K)[:, :3],
                                      err_msg=f"gradient, {K} nearest")


@pytest.mark.parametrize("K", [0, 1, 30, 90, 500])
def test_pipeline_wide_normals(ctx, K):
    """The pipeline's joint walk (normals and gradient) with neighbourhoods on both sides of the
    group's buffer, against the separate calls: two frames, the same pose bit for bit."""
    import ctypes as C

    import cuda_3d_amd as g
    from cuda_3d_amd import _lib as L
    from cuda_3d_amd import scene
    from cuda_3d_amd.core import _ptr

    (td, tc), (sd, sc), _, cm = scene.frame_pair(5, 320, 240)
    cam, bil = g.make_camera(320, 240, cm.fx, cm.fy, cm.cx, cm.cy), g.bilateral(g.BILATERAL_FIXED, 2, 2.0, 30.0)
    dev = [(g.device_tensor(d.view(np.int16)), g.device_tensor(c)) for d, c in ((td, tc), (sd, sc))]
    lv = [g.level_params(v, 5.0 * v, K, 2.0 * v, 0, g.icp_params(5, 2.5 * v)) for v in (0.04, 0.02)]
    h, valid, T, reps = C.c_void_p(), C.c_int32(), np.zeros(16), (L.IcpReport * 2)()
    L.check(L.lib.gca_pipeline_create(ctx.handle, C.byref(cam), C.byref(bil), 0.2, 3.5, 2, (L.LevelParams * 2)(*lv),
                                      C.byref(h)), "create")
    try:
        for d, c in dev:
            L.check(L.lib.gca_pipeline_step(h, C.c_void_p(d.data_ptr()), C.c_void_p(c.data_ptr())), "step")
        L.check(L.lib.gca_pipeline_result(h, _ptr(T), reps, C.byref(valid)), "result")
    finally:
        L.lib.gca_pipeline_destroy(h)
    full = [g.PointCloud.create_from_rgbd(d, c, cam, bil, 0.2, 3.5, ctx=ctx) for d, c in dev]
    want, wreps = g.multiscale_icp(full[1], full[0], lv)
    np.testing.assert_array_equal(T.reshape(4, 4), want)
    assert [r.n_correspondences for r in reps] == [r.n_correspondences for r in wreps]


@pytest.mark.parametrize("kind,n,r", [("uniform", 1, 0.05), ("uniform", 64, 0.05), ("uniform", 65, 0.05), ("uniform", 900, 0.02),
                                      ("uniform", 2600, 0.02), ("plane", 2500, 0.006), ("plane", 2500, 0.02),
                                      ("lattice", 700, 0.02), ("place", 200, 0.01)])
def test_components(ctx, kind, n, r):
    """Clusters and residual segments where most points are in one component, in many, or in runs of
    neighbouring indices that end at a wavefront's edge; labels are whole numbers, so equal."""
    import cuda_3d_amd as g
    import oracle as O

    rng = np.random.default_rng(n)
    x = _cloud(kind, n, rng)
    x[: n // 5] += np.float32(0.5)   # a second region, and indices sorted in half of the cases
    if n % 2 == 0:
        x = x[np.lexsort(x.T)]
    if n > 100:
        x[n // 2] = 1.0  # far from everything
    pc = g.PointCloud.from_numpy(x, np.zeros_like(x), ctx=ctx)
    pc.set_normals(np.zeros_like(x))
    xyzi = pc.download_xyzi()
    res = rng.uniform(0, 0.02, n).astype(np.float32)
    res[: n // 2] = 0.001
    for residual in (None, res):
        for least in (1, 4):
            want = O.euclidean_clustering(xyzi, r, least, max(n, least), residual=residual)
            got = (pc.euclidean_clustering(r, least, max(n, least)) if residual is None else
                   pc.icp_residual_segmentation(r, residual, least, max(n, least)))
            assert len(got) == len(want)
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, np.sort(b))


@pytest.mark.parametrize("n,reverse,mx", [(1, False, 0), (63, True, 0), (1025, False, 0), (1025, True, 0),
                                          (6000, None, 0), (6000, None, 40)])
def test_clusters_are_numbered_by_their_lowest_point(ctx, n, reverse, mx):
    """Long chains in ascending, descending and shuffled order: the union-find's root is any of a
    component's points, the seed its lowest (and a capped search starts there)."""
    import cuda_3d_amd as g
    import oracle as O

    r = np.random.default_rng(n)
    k = np.arange(n)
    x = np.stack([0.009 * (k // 5), 0.1 * (k % 5), np.ones(n)], 1).astype(np.float32)  # five chains side by side
    x = x[::-1].copy() if reverse else x if reverse is False else x[r.permutation(n)]
    pc = g.PointCloud.from_numpy(x, np.zeros_like(x), ctx=ctx)
    pc.set_normals(np.zeros_like(x))
    xyzi = pc.download_xyzi()
    res = (0.001 * r.integers(0, 4, n)).astype(np.float32)
    for residual in (None, res):
        want = O.euclidean_clustering(xyzi, 0.01, 1, mx or n, residual=residual)
        got = (pc.euclidean_clustering(0.01, 1, mx or n) if residual is None else
               pc.icp_residual_segmentation(0.01, residual, 1, mx or n))
        assert len(got) == len(want)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, np.sort(b))


@pytest.mark.parametrize("n", [11999, 12000, 19999, 20000])
@pytest.mark.parametrize("kind,r", [("plane", 0.004), ("plane", 0.0012), ("blobs", 0.004), ("halves", 0.004), ("apart", 0.004)])
def test_components_on_both_sides_of_the_hook_rule(ctx, n, kind, r):
    """Clouds just below and above the sizes from which pairs and a big component come before the hook
    (12000, gated 20000), dense and too sparse for them, with one component of most points, with none and
    with one of about half."""
    import cuda_3d_amd as g
    import oracle as O

    rng = np.random.default_rng(n)
    x = rng.uniform(-0.1, 0.1, (n, 3))
    x[:, 2] = 1.0 + 1e-4 * rng.normal(size=n)
    if kind == "blobs":
        c = np.stack(np.meshgrid(np.arange(-5, 5), np.arange(-5, 5)), -1).reshape(-1, 2) * 0.02
        x[:, :2] = c[rng.integers(0, 100, n)] + rng.normal(0, 0.001, (n, 2))
    elif kind == "halves":   # half in one place, the rest in many
        c = np.stack(np.meshgrid(np.arange(-5, 5), np.arange(-5, 5)), -1).reshape(-1, 2) * 0.02
        k = n // 2 + (n % 3) - 1
        x[k:, :2] = c[rng.integers(0, 100, n - k)] + rng.normal(0, 0.001, (n - k, 2)) + 0.5
    elif kind == "apart":    # nothing is linked: every point is a component
        w = int(np.ceil(np.sqrt(n)))
        x[:, 0], x[:, 1] = 0.0041 * (np.arange(n) % w), 0.0041 * (np.arange(n) // w)
        x = x[rng.permutation(n)]
    x = x.astype(np.float32)
    pc = g.PointCloud.from_numpy(x, np.zeros_like(x), ctx=ctx)
    pc.set_normals(np.zeros_like(x))
    xyzi = pc.download_xyzi()
    res = rng.uniform(0, 0.02, n).astype(np.float32)
    for residual in (None, res):
        want = O.euclidean_clustering(xyzi, r, 1, n, residual=residual)
        got = (pc.euclidean_clustering(r, 1, n) if residual is None else pc.icp_residual_segmentation(r, residual, 1, n))
        assert len(got) == len(want)
        label = np.full(n, -1)
        for k, b in enumerate(want):
            label[b] = k
        have = np.full(n, -1)
        for k, a in enumerate(got):
            have[a] = k
        np.testing.assert_array_equal(have, label)
