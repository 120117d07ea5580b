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
def cloud(n, seed=0):
    r = np.random.default_rng(seed)
    return g.PointCloud.from_numpy(r.uniform(-1, 1, (n, 3)), r.uniform(0, 1, (n, 3)))
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
hdr = (C.c_uint32 * 7).from_address(pc.device_arrays()[4])  # count, lowest and highest as ordered keys
def key(f):
    u = int(np.float32(f).view(np.uint32))
    return ~u & 0xffffffff if u >> 31 else u | 0x80000000
lowest, highest = float("{lowest}"), float("{highest}")
hdr[1:4], hdr[4:7] = [key(lowest)] * 3, [key(highest)] * 3
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
