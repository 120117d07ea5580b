"""libgca.so's host code on a stand-in runtime (cpp/host_runtime.cpp): sizes it lays out and what it
does where memory ends.  No GPU, and the kernels do nothing, so device-made counts are zero."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import sys
sys.modules["torch"] = None  # it would bring a HIP runtime of its own
import ctypes as C
import numpy as np
import cuda_3d_amd as g
from cuda_3d_amd import _lib as L
rt = C.CDLL(sys.argv[1])
rt.host_runtime_budget.argtypes = [C.c_size_t]
rt.host_runtime_live.restype = C.c_size_t
MiB = 1 << 20
ctx = g.default_context()
def key(f):
    u = int(np.float32(f).view(np.uint32))
    return ~u & 0xffffffff if u >> 31 else u | 0x80000000
def bounds(pc, lowest, highest):         # what the kernels would have left
    hdr = (C.c_uint32 * 7).from_address(pc.device_arrays()[4])
    hdr[1:4], hdr[4:7] = [key(lowest)] * 3, [key(highest)] * 3
def cloud(n, seed=0):
    r = np.random.default_rng(seed)
    pc = g.PointCloud.from_numpy(r.uniform(-1, 1, (n, 3)), r.uniform(0, 1, (n, 3)))
    bounds(pc, -1, 1)
    return pc
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = tmp_path_factory.mktemp("rt") / "libhost_runtime.so"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", f"{rocm}/include",
                    os.path.join(ROOT, "tests", "cpp", "host_runtime.cpp"), "-o", str(so)], check=True)
    return str(so)


def _run(runtime, body):
    preload = [runtime] + [p for p in [os.environ.get("LD_PRELOAD")] if p]
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, runtime], cwd=ROOT, capture_output=True, text=True, timeout=60,
                       env=dict(os.environ, LD_PRELOAD=":".join(preload)))
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_grid_of_an_empty_cloud_is_one_cell(runtime):
    """An empty cloud's bounds are the fold's start values, lowest above highest."""
    out = _run(runtime, """
for q in (0, 6):
    ctx.set_tuning(grid_cell=q)
    for radius in (1e-3, 0.05, 1.0, 1e30):
        e, cells = g.PointCloud(), np.zeros(3, np.int32)
        dims, edge = np.zeros(3, np.int32), C.c_float()
        L.check(L.lib.gca_grid_cells(ctx.handle, e.handle, radius, cells.ctypes.data_as(C.c_void_p), None, C.byref(edge),
                                     dims.ctypes.data_as(C.c_void_p)), "gca_grid_cells")
        print(q, radius, dims.tolist())
        assert dims.tolist() == [1, 1, 1] and edge.value == np.float32(radius)
""")
    assert out.count("[1, 1, 1]") == 8


@pytest.mark.parametrize("lowest,highest", [(0.0, float("inf")), (float("-inf"), 1.0), (float("-inf"), float("inf")),
                                            (-3e38, 3e38)])
def test_grid_of_a_cloud_with_infinite_bounds_ends(runtime, lowest, highest):
    """The cell edge doubles until the cells are few enough, or it is infinite."""
    _run(runtime, f"""
pc = cloud(4)
bounds(pc, float("{lowest}"), float("{highest}"))
cells, dims = np.zeros((4, 3), np.int32), np.zeros(3, np.int32)
L.check(L.lib.gca_grid_cells(ctx.handle, pc.handle, 0.05, cells.ctypes.data_as(C.c_void_p), None, None,
                             dims.ctypes.data_as(C.c_void_p)), "gca_grid_cells")
assert (dims >= 1).all() and dims.astype(float).prod() <= 1 << 25
""")


def test_clouds_do_not_share_the_bounds_in_flight(runtime):
    """Upload, transform and append fold their workgroups' bounds in a second launch: what the two
    launches hand over is the cloud's own, whatever is enqueued between them for another cloud."""
    _run(runtime, """
rt.host_runtime_bounds.restype = C.c_void_p
used = []
T = np.ascontiguousarray(np.eye(4))
clouds = [cloud(n) for n in (1, 500, 70000)]
for pc in clouds:
    mine = set()
    L.check(L.lib.gca_transform(ctx.handle, pc.handle, T.ctypes.data_as(C.c_void_p)), "gca_transform")
    mine.add(rt.host_runtime_bounds())
    L.check(L.lib.gca_cloud_append(ctx.handle, pc.handle, pc.handle), "gca_cloud_append")
    mine.add(rt.host_runtime_bounds())
    xyz = np.zeros((3, 3), np.float32)
    L.check(L.lib.gca_cloud_upload(pc.handle, xyz.ctypes.data_as(C.c_void_p), xyz.ctypes.data_as(C.c_void_p), 3), "upload")
    mine.add(rt.host_runtime_bounds())
    assert len(mine) == 1 and None not in mine
    used += mine
assert len(set(used)) == len(clouds)
""")


def test_an_allocation_retried_without_the_pool_leaves_no_error(runtime):
    """The first try fails, the pool goes, the second succeeds: the call does, too, and so does the
    next one after a call that was refused for good."""
    _run(runtime, """
keep, a = cloud(1000), cloud(400_000)
del a                                    # its arrays are in the pool: 4 of 6.4 MB
rt.host_runtime_budget(rt.host_runtime_live() + MiB)
b = cloud(300_000)                       # another size class: no room beside the pool
assert b.points_number() == 300_000
try:
    cloud(2_000_000)
    raise SystemExit("room for 128 MB?")
except L.GcaError as e:
    assert e.status == L.GCA_ERR_OUT_OF_MEMORY
keep.transform(np.eye(4))
assert keep.points_number() == 1000
""")


def test_levels_built_one_by_one_where_the_lanes_do_not_fit(runtime):
    """A multi-scale call that cannot have the scratch of several levels at once still goes through."""
    _run(runtime, """
levels = [g.level_params(v, icp=g.icp_params(2, 2.5 * v)) for v in (0.1, 0.06, 0.04)]
src, tgt = cloud(200_000, 1), cloud(200_000, 2)
for pc in (src, tgt):
    for v in (0.1, 0.06, 0.04):
        pc.voxel_grid_down_sample(v)     # the scratch of one level at a time
one = rt.host_runtime_live()
other = g.Context(0)
tries = []
for extra in range(0, 200, 5):
    rt.host_runtime_budget(one + extra * MiB)
    try:
        g.multiscale_icp(src, tgt, levels)
        tries.append(extra)
        break
    except L.GcaError as e:
        assert e.status == L.GCA_ERR_OUT_OF_MEMORY
rt.host_runtime_budget(1 << 40)
g.multiscale_icp(src, tgt, levels)       # with all the memory it likes
print("one level at a time", one / MiB, "succeeds with", tries, "more; together takes", (rt.host_runtime_live() - one) / MiB)
# level by level, a walk each: the levels' clouds (as large as their inputs here, 3 x 2 x 12.2 MiB),
# the targets' grids (3 x 10.7) and one level's sums (22.9)
assert tries and tries[0] <= 135
""")


def test_memory_kept_for_reuse_gives_way(runtime):
    """What a context only keeps for its next calls (buffers of clouds that are gone, the scratch of a
    multi-scale call's further levels) is there for whatever does not fit otherwise: its own clouds, a
    batch plan, another context, a pipeline's."""
    _run(runtime, """
def level(n):
    s, t = cloud(n, 3), cloud(n, 4)
    t.estimate_normals(0.1, 30)
    t.compute_color_gradient(0.1, 0)
    return s, t
pairs = [level(2000) for _ in range(40)]
prm = [g.icp_params(3, 0.1)]
def plan():
    return g.BatchPlan([[s] for s, _ in pairs], [[t] for _, t in pairs], prm, np.tile(np.eye(4), (40, 1, 1)), [0.1])
def pipeline():
    cam, bil, h = g.make_camera(640, 480, 615.0, 615.0, 320, 240), g.bilateral(), C.c_void_p()
    lv = (L.LevelParams * 3)(*[g.level_params(v) for v in (0.04, 0.02, 0.01)])
    L.check(L.lib.gca_pipeline_create(ctx.handle, C.byref(cam), C.byref(bil), 0.2, 3.5, 3, lv, C.byref(h)), "pipeline")
    return h
def taken(make):
    rt.host_runtime_budget(1 << 40)
    before = rt.host_runtime_live()
    made = make()
    size = rt.host_runtime_live() - before
    if isinstance(made, C.c_void_p):
        L.lib.gca_pipeline_destroy(made)
    elif hasattr(made, "close"):
        made.close()
    return size
levels = [g.level_params(v, icp=g.icp_params(2, 2.5 * v)) for v in (0.1, 0.06, 0.04)]
src, tgt = cloud(400_000, 1), cloud(400_000, 2)
g.multiscale_icp(src, tgt, levels)       # its scratch stays
plan().close()                           # (so that the calls below find their small buffers)
other = g.Context(0)
wanted = {"cloud": lambda: cloud(600_000),
          "plan": plan,
          "other": lambda: g.PointCloud(other, 600_000),
          "pipeline": pipeline}
sizes = {k: taken(f) for k, f in wanted.items()}
for kept in ("pool", "lanes"):
    for k, make in wanted.items():
        rt.host_runtime_budget(1 << 40)
        if kept == "pool":
            bulk = [cloud(1_500_000) for _ in range(6)]
            del bulk
        else:
            g.multiscale_icp(src, tgt, levels)
        full = rt.host_runtime_live()
        rt.host_runtime_budget(full + sizes[k] // 4)  # a quarter of what it takes, the rest is kept memory
        made = make()
        print(kept, k, sizes[k] / MiB, full / MiB, "->", rt.host_runtime_live() / MiB)
        assert rt.host_runtime_live() <= full + sizes[k] // 4
        if k == "pipeline":
            L.lib.gca_pipeline_destroy(made)
        del made
""")


def test_large_arrays_take_what_they_hold(runtime):
    """Buffers too large for the pool are not rounded up to its classes."""
    _run(runtime, """
cloud(1)
for n in (9_000_001, 17_300_000):        # 137 and 264 MiB an array
    before = rt.host_runtime_live()
    pc = g.PointCloud(ctx, n)
    assert rt.host_runtime_live() - before == 4 * 16 * n
    del pc
    assert rt.host_runtime_live() == before
""")


def test_grid_attributes_are_both_there_or_neither(runtime):
    """A registration that ran out of memory between the target's sorted normals and its sorted
    gradients finds both on the next try."""
    _run(runtime, """
src, a, b = cloud(1000, 1), cloud(200_000, 2), cloud(200_000, 3)
def target(pc):
    pc.estimate_normals(0.1, 30)
    pc.compute_color_gradient(0.1, 0)
def align(pc):
    icp = g.ColorICP(3, 0.1, 0.1)
    icp.set_source_point_cloud(src)
    icp.set_target_point_cloud(pc)
    return icp.align()
def takes(pc):
    before = rt.host_runtime_live()
    assert align(pc)
    return rt.host_runtime_live() - before
target(a)
target(b)
warm = cloud(1000, 4)
target(warm)
assert align(warm)                       # the registration's own scratch
whole = takes(a)
assert whole >= 2 * 16 * 200_000         # normals and gradients in the grid's order
base, refused = rt.host_runtime_live(), 0
for room in range(0, whole + MiB, MiB // 4):
    rt.host_runtime_budget(base + room)
    try:
        assert align(b)
        break
    except L.GcaError as e:
        assert e.status == L.GCA_ERR_OUT_OF_MEMORY
        refused += 1
assert refused >= 8 and rt.host_runtime_live() - base == whole
""")


@pytest.mark.parametrize("room", [0, 5, 9, 14])
def test_a_cloud_that_could_not_grow_is_empty(runtime, room):
    """Its old arrays went before the new ones could not all be had: no call may find the old count."""
    _run(runtime, f"""
pc, full = cloud(30_000), cloud(400_000)
pc.estimate_normals(0.1, 30)
assert pc.points_number() == 30_000
rt.host_runtime_budget(rt.host_runtime_live() + {room} * MiB)
status = L.lib.gca_cloud_copy(ctx.handle, full.handle, pc.handle)
assert status == L.GCA_ERR_OUT_OF_MEMORY
count = C.c_int32.from_address(pc.device_arrays()[4]).value
assert (pc.points_number(), count, pc.has_normals()) == (0, 0, False)
assert all(pc.device_arrays())
rt.host_runtime_budget(1 << 40)
L.check(L.lib.gca_cloud_copy(ctx.handle, full.handle, pc.handle), "gca_cloud_copy")
""")
