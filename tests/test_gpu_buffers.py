"""Copies, appends and clouds made from buffers that other clouds gave back: exact values."""
import gc
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 2, 255, 257, 5000]


def _arrays(n, seed):
    r = np.random.default_rng(seed)
    return (r.uniform(-1, 1, (n, 3)).astype(np.float32), r.uniform(0, 1, (n, 3)).astype(np.float32),
            r.normal(size=(n, 3)).astype(np.float32))


def _cloud(g, n, seed, normals):
    x, c, m = _arrays(n, seed)
    pc = g.PointCloud.from_numpy(x, c)
    if normals:
        pc.set_normals(m)
    return pc, x, c, m


def _check(pc, x, c, m):
    got_x, got_c, _ = pc.download()
    np.testing.assert_array_equal(got_x, x)
    np.testing.assert_array_equal(got_c, c)
    assert pc.has_normals() == (m is not None)
    if m is not None:
        np.testing.assert_array_equal(pc.download_normals(), m)
    big = np.finfo(np.float32)
    np.testing.assert_array_equal(pc.get_min_bound(), x.min(0) if len(x) else np.full(3, big.max, np.float32))
    np.testing.assert_array_equal(pc.get_max_bound(),
                                  np.maximum(x.max(0), big.tiny) if len(x) else np.full(3, big.tiny, np.float32))


@pytest.mark.parametrize("na", SIZES)
@pytest.mark.parametrize("nb", SIZES)
def test_copy_and_append(na, nb):
    import cuda_3d_amd as g

    for normals in ((True, True), (True, False)):
        a, xa, ca, ma = _cloud(g, na, na + 1, normals[0])
        b, xb, cb, mb = _cloud(g, nb, 7 * nb + 2, normals[1])
        d = a.copy()
        _check(d, xa, ca, ma)
        both = np.concatenate([ma, mb]) if all(normals) else None
        d += b
        _check(d, np.concatenate([xa, xb]), np.concatenate([ca, cb]), both)
        d += b  # within the capacity of the first growth, or growing again
        both = np.concatenate([both, mb]) if all(normals) else None
        _check(d, np.concatenate([xa, xb, xb]), np.concatenate([ca, cb, cb]), both)
        d += d
        x = np.concatenate([xa, xb, xb] * 2)
        _check(d, x, np.concatenate([ca, cb, cb] * 2), None if both is None else np.concatenate([both, both]))
        T = np.eye(4)
        T[:3, 3] = 0.5, -0.25, 2.0
        a.transform(T)
        a += b  # the count is known, the bounds are not
        moved = (xa.astype(np.float64) + T[:3, 3]).astype(np.float32)
        _check(a, np.concatenate([moved, xb]), np.concatenate([ca, cb]),
               np.concatenate([ma, mb]) if all(normals) else None)


def test_headers_and_buffers_come_back_clean():
    import cuda_3d_amd as g

    kept = []
    for k in range(300):
        n = (0, 3, 9000)[k % 3]
        pc, x, c, _ = _cloud(g, n, k, False)
        if k % 50 == 0:
            kept.append((pc, x, c))
        del pc
        e = g.PointCloud()
        assert e.points_number() == 0 and e.device_arrays()[4]
        del e
    gc.collect()
    for pc, x, c in kept:
        _check(pc, x, c, None)
    e = g.PointCloud()
    down = e.voxel_grid_down_sample(0.1)  # an empty cloud in a used header
    assert down.points_number() == 0


def test_clouds_of_one_context_on_threads():
    import cuda_3d_amd as g

    g.default_context()
    bad = []

    def work(seed):
        r = np.random.default_rng(seed)
        for k in range(40):
            n = int(r.integers(0, 12000))
            pc, x, c, _ = _cloud(g, n, 1000 * seed + k, False)
            got = pc.copy().download()
            if not (np.array_equal(got[0], x) and np.array_equal(got[1], c)):
                bad.append((seed, k, n))

    ts = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_bounds_of_clouds_on_threads():
    """Each cloud's bounds are its own while clouds of the same context are made, moved and appended to
    on other threads."""
    import cuda_3d_amd as g

    g.default_context()
    bad = []

    def work(seed):
        r = np.random.default_rng(seed)
        T = np.eye(4)
        T[:3, 3] = 0.5, -0.25, 2.0
        for k in range(150):
            n = int(r.integers(1, 9000))
            x = (r.uniform(-1, 1, (n, 3)) + 10 * seed).astype(np.float32)
            pc = g.PointCloud.from_numpy(x, np.zeros_like(x))
            for step in range(3):
                if step == 1:
                    pc.transform(T)
                    x = (x.astype(np.float64) + T[:3, 3]).astype(np.float32)
                elif step == 2:
                    pc += pc
                if not (np.array_equal(pc.get_min_bound(), x.min(0)) and np.array_equal(pc.get_max_bound(), x.max(0))):
                    bad.append((seed, k, n, step))

    ts = [threading.Thread(target=work, args=(s,)) for s in range(1, 9)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, (len(bad), bad[:5])
