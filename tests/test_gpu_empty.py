"""Neighbour calls and registrations with an empty cloud on either side: no neighbours, no points, the
initial pose; and with points that no grid holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clouds(ctx):
    import cuda_3d_amd as g

    r = np.random.default_rng(3)
    x = r.uniform(-0.2, 0.2, (500, 3)).astype(np.float32)
    return g.PointCloud(ctx), g.PointCloud.from_numpy(x, np.full_like(x, 0.5), ctx=ctx)


@pytest.mark.parametrize("radius", [1e-3, 0.05, 2.0])
def test_neighbour_calls(ctx, radius):
    import cuda_3d_amd as g

    e, some = _clouds(ctx)
    assert (g.PointCloud.nn_search(some, e, radius) == -1).all()
    assert len(g.PointCloud.nn_search(e, some, radius)) == 0
    for q, ref, n in ((some, e, 500), (e, some, 0), (e, e, 0)):
        for k in (0, 30):
            off, idx = g.PointCloud.radius_search(q, ref, radius, k)
            assert off.tolist() == [0] * (n + 1) and len(idx) == 0
    assert e.radius_outlier_removal(radius, 0).points_number() == 0
    for k in (0, 30):
        assert e.estimate_normals(radius, k) and e.compute_color_gradient(radius, k)
    assert e.euclidean_clustering(radius, 1, 10) == []
    assert e.icp_residual_segmentation(radius, np.zeros(0, np.float32), 1, 10) == []


@pytest.mark.parametrize("levels", [1, 3])
def test_registration(ctx, levels):
    import cuda_3d_amd as g

    e, some = _clouds(ctx)
    T0 = np.eye(4)
    T0[:3, 3] = 0.01, -0.02, 0.03
    lv = [g.level_params(v, icp=g.icp_params(5, 2.5 * v)) for v in (0.1, 0.05, 0.03)[:levels]]
    for src, tgt in ((some, e), (e, some), (e, e)):
        T, reps = g.multiscale_icp(src, tgt, lv, T0)
        np.testing.assert_array_equal(T, T0)
        assert all(r.n_correspondences == 0 for r in reps)


@pytest.mark.parametrize("far", [[np.inf, 0, 0], [0, -np.inf, 0], [np.inf, -np.inf, np.inf], [3e38, 0, -3e38]])
def test_points_beyond_any_grid(ctx, far):
    """A cloud with a point at (or near) infinity: one cell holds everything, the answers are the others'."""
    import cuda_3d_amd as g

    _, some = _clouds(ctx)
    x = some.download()[0]
    with_far = np.concatenate([x[:100], np.float32([far]), x[100:]])
    ref = g.PointCloud.from_numpy(with_far, np.full_like(with_far, 0.5), ctx=ctx)
    want = g.PointCloud.nn_search(some, some, 0.05)
    np.testing.assert_array_equal(g.PointCloud.nn_search(some, ref, 0.05), want + (want >= 100))
    want = some.radius_outlier_removal(0.05, 1).download()[0]
    np.testing.assert_array_equal(ref.radius_outlier_removal(0.05, 1).download()[0], want)
