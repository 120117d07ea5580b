"""The persistent launch's scheduler: many states, few and many work units, few workgroups.  Every
shape gives the bits of one launch per iteration."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _clouds(g, n, seed):
    r = np.random.default_rng(seed)
    x = r.uniform(-0.3, 0.3, (n, 3))
    x[:, 2] = 1.0 + 0.1 * np.sin(5 * x[:, 0]) * np.cos(4 * x[:, 1])
    c = 0.5 + 0.4 * np.sin(9 * x)
    src = (x + [0.004, -0.003, 0.005]).astype(np.float32)
    s, t = g.PointCloud.from_numpy(src, c.astype(np.float32)), g.PointCloud.from_numpy(x.astype(np.float32), c.astype(np.float32))
    t.estimate_normals(0.1, 30)
    t.compute_color_gradient(0.1, 0)
    return s, t


@pytest.mark.parametrize("pairs,levels,tune", [
    (2, 1, {}),                                            # two states
    (90, 3, {}),                                           # 270 states: more than one read of open words
    (90, 3, {"icp_persist_blocks": 1}),                    # one workgroup serves them all
    (7, 2, {"icp_max_units": 1}),                          # one sub-queue in use
    (7, 2, {"icp_lanes_batch": 64, "icp_max_units": 9}),   # one sub-queue of two units
    (40, 2, {"icp_lanes_batch": 64, "icp_max_units": 200, "icp_persist_blocks": 2000}),
])
def test_persistent_launch_equals_one_launch_per_iteration(pairs, levels, tune):
    import cuda_3d_amd as g

    ctx = g.default_context()
    made = [_clouds(g, n, n) for n in (1, 40, 700, 1500)]
    src = [[made[(k + l) % 4][0] for l in range(levels)] for k in range(pairs)]
    tgt = [[made[(k + l) % 4][1] for l in range(levels)] for k in range(pairs)]
    params = [g.icp_params((5, 9, 1)[l], 0.1) for l in range(levels)]
    T0 = np.tile(np.eye(4), (pairs, 1, 1))
    T0[:, 0, 3] = np.linspace(-0.01, 0.01, pairs)
    got = {}
    try:
        ctx.set_tuning(**tune)
        for launch in (1, 2):
            ctx.set_tuning(icp_launch=launch)
            T, reps = g.batch_multiscale_icp(src, tgt, params, T0, [0.1] * levels)
            got[launch] = T, [[(r.iterations, r.n_correspondences, r.rmse) for r in row] for row in reps]
    finally:
        ctx.set_tuning(icp_launch=0, **{k: 0 for k in tune})
    np.testing.assert_array_equal(got[1][0], got[2][0])
    assert got[1][1] == got[2][1]
    assert any(r[0] > 1 for row in got[1][1] for r in row)


@pytest.mark.parametrize("normal_r,max_nn,grad_r,grad_nn", [(2.5, 30, 2.0, 0),   # attributes from one walk
                                                            (2.5, 0, 2.5, 0),    # no cap, equal radii
                                                            (2.0, 30, 2.5, 0),   # the gradient reaches further
                                                            (2.5, 30, 2.0, 12)])  # a capped gradient
def test_multiscale_equals_its_steps(normal_r, max_nn, grad_r, grad_nn):
    import cuda_3d_amd as g

    src, tgt = _clouds(g, 20000, 5)
    voxels = (0.05, 0.03, 0.02)
    levels = [g.level_params(v, normal_radius=normal_r * v, normal_max_nn=max_nn, gradient_radius=grad_r * v,
                             gradient_max_nn=grad_nn, icp=g.icp_params(6, 2.5 * v)) for v in voxels]
    T, reps = g.multiscale_icp(src, tgt, levels)
    pose = np.eye(4)
    for v, rep in zip(voxels, reps):
        s, t = src.voxel_grid_down_sample(v), tgt.voxel_grid_down_sample(v)
        t.estimate_normals(normal_r * v, max_nn)
        t.compute_color_gradient(grad_r * v, grad_nn)
        Ts, one = g.batch_multiscale_icp([[s]], [[t]], [g.icp_params(6, 2.5 * v)], pose[None], [grad_r * v])
        pose = Ts[0]
        assert (rep.iterations, rep.n_correspondences, rep.rmse) == (one[0][0].iterations, one[0][0].n_correspondences,
                                                                     one[0][0].rmse)
    np.testing.assert_array_equal(T, pose)


@pytest.mark.parametrize("n,sizes,kinds,tune", [
    (20000, (0.04,), "j", {}),                                    # one level: no shared launch
    (20000, (0.08, 0.03), "jj", {}),                              # the smallest one
    (20000, (0.09, 0.06, 0.04, 0.02), "jjjj", {}),                # a full one
    (20000, (0.1, 0.08, 0.06, 0.05, 0.03), "jjjjj", {}),          # ... and one level over
    (20000, (0.08, 0.05, 0.03), "jsj", {}),                       # a level with walks of its own between
    (20000, (0.08, 0.05, 0.03), "sjj", {"grid_cell": 6}),
    (20000, (0.08, 0.05, 0.03), "jjj", {"voxel": 2}),             # the sorted path, size by size
    (20000, (0.08, 0.05, 0.00001), "jjj", {}),                    # a lattice beyond the bitmap
    (1, (0.08, 0.05, 0.03), "jjj", {}),
    (40, (0.3, 0.1), "jj", {}),
])
def test_multiscale_levels_built_together_equal_single_ones(n, sizes, kinds, tune):
    import cuda_3d_amd as g

    ctx = g.default_context()
    src, tgt = _clouds(g, n, 9)
    radii = [max(v, 0.02) for v in sizes]
    levels = [g.level_params(v, normal_radius=2.5 * r, normal_max_nn=30, gradient_radius=(2.0 if k == "j" else 3.0) * r,
                             gradient_max_nn=0, icp=g.icp_params(4, 2.5 * r)) for v, r, k in zip(sizes, radii, kinds)]
    old = ctx.get_tuning()
    try:
        ctx.set_tuning(**tune)
        for _ in range(2):  # the second call reuses the first one's scratch
            T, reps = g.multiscale_icp(src, tgt, levels)
            pose = np.eye(4)
            for v, r, k, rep in zip(sizes, radii, kinds, reps):
                s, t = src.voxel_grid_down_sample(v), tgt.voxel_grid_down_sample(v)
                t.estimate_normals(2.5 * r, 30)
                t.compute_color_gradient((2.0 if k == "j" else 3.0) * r, 0)
                Ts, one = g.batch_multiscale_icp([[s]], [[t]], [g.icp_params(4, 2.5 * r)], pose[None],
                                                 [(2.0 if k == "j" else 3.0) * r])
                pose = Ts[0]
                assert (rep.iterations, rep.n_correspondences, rep.rmse) == (
                    one[0][0].iterations, one[0][0].n_correspondences, one[0][0].rmse)
            np.testing.assert_array_equal(T, pose)
    finally:
        ctx.set_tuning(**old)


@pytest.mark.parametrize("blocks", [2, 3, 5, 7, 9])
@pytest.mark.parametrize("pairs,levels,units", [(1, 2, 3), (3, 3, 8), (12, 1, 40)])
def test_fewer_workgroups_than_sub_queues(blocks, pairs, levels, units):
    """Sub-queues that no workgroup has as its own, through many epochs: a workgroup that comes late to
    one is not held up there."""
    import cuda_3d_amd as g

    ctx = g.default_context()
    made = [_clouds(g, n, n) for n in (300, 1500)]
    src = [[made[(k + l) % 2][0] for l in range(levels)] for k in range(pairs)]
    tgt = [[made[(k + l) % 2][1] for l in range(levels)] for k in range(pairs)]
    params = [g.icp_params(40, 0.1, conv_rotation=-1.0)] * levels  # never converged: every iteration runs
    T0 = np.tile(np.eye(4), (pairs, 1, 1))
    got = {}
    try:
        ctx.set_tuning(icp_persist_blocks=blocks, icp_max_units=units, icp_lanes_batch=16, icp_lanes_small=16)
        for launch in (1, 2):
            ctx.set_tuning(icp_launch=launch)
            T, reps = g.batch_multiscale_icp(src, tgt, params, T0, [0.1] * levels)
            got[launch] = T, [[(r.iterations, r.n_correspondences, r.rmse) for r in row] for row in reps]
    finally:
        ctx.set_tuning(icp_launch=0, icp_persist_blocks=0, icp_max_units=0, icp_lanes_batch=0, icp_lanes_small=0)
    np.testing.assert_array_equal(got[1][0], got[2][0])
    assert got[1][1] == got[2][1]
    assert all(r[0] == 40 for row in got[1][1] for r in row)


def test_a_knob_that_nothing_reads_keeps_the_graphs(ctx):
    """Setting normals_lanes is accepted and changes nothing: the pipeline's graphs are not captured again."""
    import cuda_3d_amd as g
    from cuda_3d_amd import scene
    from cuda_3d_amd.pipeline import FramePipeline

    (td, tc), (sd, sc), _, cm = scene.frame_pair(5, 160, 120)
    dev = [(g.device_tensor(d.view(np.int16)), g.device_tensor(c)) for d, c in ((td, tc), (sd, sc))]
    pipe = FramePipeline(ctx, g.make_camera(160, 120, cm.fx, cm.fy, cm.cx, cm.cy), g.bilateral(), levels=(0.04,), iters=4)
    captures = []
    for k in range(16):
        if k == 8:
            pipe.ctx.set_tuning(normals_lanes=4)
            assert pipe.ctx.get_tuning()["normals_lanes"] == 4
        d, c = dev[k % 2]
        pipe.step(d.data_ptr(), c.data_ptr())
        pipe.result()
        captures.append(pipe.graph_stats()[0])
    assert captures[7] > 0 and captures[-1] == captures[7]
    pipe.close()
