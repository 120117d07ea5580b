"""The bilateral filter at the edges of its row segments, radii and weight tables: bit-equal to the
oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _frame(w, h, seed):
    """Depth in millimetres: smooth parts, steps of up to 3 m between neighbours (range weights far down
    the tables), holes, and a strip nearer than any staged part of a range table is long."""
    r = np.random.default_rng(seed)
    y, x = np.mgrid[0:h, 0:w]
    d = 900 + 1.5 * x + 2.0 * y + r.normal(0, 2, (h, w)) + 400.0 * ((x // 9 + y // 5) % 6)
    d = np.where(r.random((h, w)) < 0.1, 0, d)
    d = np.where(r.random((h, w)) < 0.1, r.integers(60, 3600, (h, w)), d)
    d[:, : max(w // 8, 1)] = r.integers(40, 130, (h, max(w // 8, 1)))
    return d.astype(np.uint16), r.integers(0, 256, (h, w, 3)).astype(np.uint8)


@pytest.mark.parametrize("w,h", [(1, 1), (5, 40), (255, 7), (256, 12), (257, 31), (530, 13)])
@pytest.mark.parametrize("mode,radius,ss,sd", [(2, 0, 1.0, 1.0), (1, 0, 2.0, 30.0), (1, 1, 2.0, 30.0), (1, 2, 2.0, 3.0),
                                               (1, 5, 2.0, 30.0), (1, 6, 3.0, 400.0), (1, 15, 8.0, 150.0),
                                               (1, 3, 2.0, 400.0)])
@pytest.mark.parametrize("frontend", [0, 1])
def test_filter_bits(w, h, mode, radius, ss, sd, frontend):
    import cuda_3d_amd as g

    depth, bgr = _frame(w, h, w + 3 * h + radius)
    cam, camo = (m.make_camera(w, h, 60.0, 60.0, w / 2, h / 2) for m in (g, O))
    ctx = g.default_context()
    try:
        ctx.set_tuning(frontend=frontend)
        pc = g.PointCloud.create_from_rgbd(depth, bgr, cam, g.bilateral(mode, radius, ss, sd), 0.03, 3.5)
    finally:
        ctx.set_tuning(frontend=0)
    xyz, rgb, _ = pc.download()
    ox, orgb, _, _ = O.cloud_from_rgbd(depth, bgr, camo, O.Bilateral(mode, radius, ss, sd), 0.03, 3.5)
    assert len(xyz) == len(ox)
    np.testing.assert_array_equal(xyz.view(np.uint32), np.ascontiguousarray(ox[:, :3]).view(np.uint32))
    np.testing.assert_array_equal(rgb, np.ascontiguousarray(orgb[:, :3]))
