"""Performance cases: the work a user of cuda_3d_amd has it do, through the public entry points.

listed()            the cases that are timed; draw(rng) makes more of the same ranges
prepare(case, seed) what a program holds before the call (inputs, clouds, pipelines), from the seed
run(state)          one pass and its outputs
work(case)          the bytes and operations one pass cannot do without
exact(case, seed)   the values of run()'s outputs in 64 bits, by plain torch

Every input is a rendered RGB-D scene (three walls and four spheres at 0.4 to 3.4 m, sensor noise of
2 mm, 5 % holes, millimetre depth, colour noise), the framework's own kind of workload: a cloud's
neighbourhoods are surfaces of uneven density, in raster order.  Outputs of a size known only after the pass are arrays of the
largest size, zero beyond the count that is returned with them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import cuda_3d_amd as g
from cuda_3d_amd import autotune
from cuda_3d_amd.autograd import colored_icp_objective
from cuda_3d_amd.pipeline import FramePipeline

LAMBDA = 0.968
TMIN, TMAX = 0.2, 3.5
AREA = 8.0            # square metres of surface a camera sees, about
FILL = 0.9            # share of a frame's pixels that become points


# ---- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: a thumbnail frame to a cloud, where launches and the size read-back are all
        {"name": "cloud_160x120", "kind": "cloud", "w": 160, "h": 120, "filter": "fixed", "radius": 2},
        # the largest frame of the configurations through the reference's depth-adaptive filter
        {"name": "cloud_1280x720_adaptive", "kind": "cloud", "w": 1280, "h": 720, "filter": "adaptive", "radius": 5},
        # a registration target from a full frame: downsample, normals (30 nearest), colour gradient
        {"name": "target_640x480_1cm", "kind": "target", "w": 640, "h": 480, "voxel": 0.01, "max_nn": 30},
        # the reference's example program: one pair at 2 cm, 100 iterations at most, its own radii
        {"name": "align_424x240_2cm", "kind": "align", "w": 424, "h": 240, "voxel": 0.02, "iters": 100, "accum": 0},
        # one whole coarse-to-fine call on the largest frames
        {"name": "multiscale_1280x720", "kind": "multiscale", "w": 1280, "h": 720, "levels": 3, "iters": 30},
        # odometry where each pose is needed at once (a robot's control loop): read after every frame
        {"name": "odometry_640x480_each_pose", "kind": "odometry", "w": 640, "h": 480, "frames": 5, "overlap": False},
        # odometry of a recording: overlapped steps, the result read at the end
        {"name": "odometry_640x480_overlapped", "kind": "odometry", "w": 640, "h": 480, "frames": 16, "overlap": True},
        # many uneven pairs at once (loop closures, a dataset): one batched call over three levels
        {"name": "batch_64_pairs", "kind": "batch", "pairs": 64, "lo": 5000, "hi": 200000, "levels": 3, "iters": 30},
        # differentiable registration: the objective and its gradients, forward and backward
        {"name": "objective_100k", "kind": "objective", "n": 100000},
        # clean a scan, then the neighbourhoods of keypoints in it: outlier removal, capped radius search
        {"name": "neighbours_424x240", "kind": "neighbours", "w": 424, "h": 240, "radius_m": 0.03, "max_nn": 30, "min_nn": 8},
        # what moved and what stands: residuals against the previous frame, both segmentations
        {"name": "segment_424x240", "kind": "segment", "w": 424, "h": 240, "corr": 0.03, "tol": 0.02, "min_size": 20},
        # a SLAM map's update: the frame moved into the map, appended, downsampled at 8 mm
        {"name": "map_update_848x480", "kind": "map", "w": 848, "h": 480, "frames": 3, "voxel": 0.008},
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def size(lo, hi):  # odd and ragged sizes of the usual aspect ratios
        w = int(log(lo, hi))
        return {"w": w, "h": max(64, int(w * rng.choice((0.5625, 0.625, 0.75))))}

    kind = rng.choice(("cloud", "target", "align", "multiscale", "odometry", "batch", "objective", "neighbours",
                       "segment", "map"))
    if kind == "cloud":
        f = rng.choice(("fixed", "adaptive", "none"))
        return {"kind": kind, **size(120, 1280), "filter": f, "radius": rng.randint(1, 4) if f == "fixed" else 5}
    if kind == "target":
        return {"kind": kind, **size(160, 640), "voxel": round(log(0.01, 0.04), 4), "max_nn": rng.choice((0, 20, 30))}
    if kind == "align":
        return {"kind": kind, **size(160, 640), "voxel": round(log(0.015, 0.04), 4), "iters": rng.choice((30, 50, 100)),
                "accum": rng.choice((0, 0, 1, 2))}
    if kind == "multiscale":
        return {"kind": kind, **size(200, 1100), "levels": rng.randint(2, 3), "iters": rng.choice((15, 30))}
    if kind == "odometry":
        return {"kind": kind, **size(200, 640), "frames": rng.randint(3, 10), "overlap": rng.random() < 0.5}
    if kind == "batch":
        lo = int(log(2000, 10000))
        return {"kind": kind, "pairs": rng.randint(3, 40), "lo": lo, "hi": int(lo * rng.uniform(3, 12)),
                "levels": rng.randint(1, 3), "iters": rng.choice((15, 30))}
    if kind == "objective":
        return {"kind": kind, "n": int(log(3000, 300000))}
    if kind == "neighbours":
        return {"kind": kind, **size(160, 424), "radius_m": round(rng.uniform(0.015, 0.03), 4),
                "max_nn": rng.choice((0, 10, 30)), "min_nn": rng.randint(2, 12)}
    if kind == "segment":
        return {"kind": kind, **size(160, 640), "corr": round(rng.uniform(0.02, 0.04), 4),
                "tol": round(rng.uniform(0.012, 0.02), 4), "min_size": rng.randint(5, 50)}
    return {"kind": kind, **size(320, 848), "frames": rng.randint(1, 3), "voxel": round(rng.uniform(0.006, 0.012), 4)}


# ---- scenes ---------------------------------------------------------------------------------------

def _scene(seed, scale=1.0):
    rng = np.random.default_rng(seed)

    def tilted(n):
        v = np.asarray(n) + rng.uniform(-0.15, 0.15, 3)
        return v / np.linalg.norm(v)

    walls = [(tilted(n), d + rng.uniform(-0.1, 0.1)) for n, d in (((0, 0, 1.0), 2.8), ((0, 1.0, 0), 0.9), ((1.0, 0, 0), -1.1))]
    balls = []
    for _ in range(4):
        z = rng.uniform(1.0, 2.2)
        balls.append((np.array([rng.uniform(-0.45, 0.45) * z, rng.uniform(-0.3, 0.3) * z, z]), rng.uniform(0.12, 0.3)))
    return {"walls": [(n, d * scale) for n, d in walls], "balls": [(c * scale, r * scale) for c, r in balls],
            "scale": scale, "colours": rng.integers(30, 226, (7, 3))}


def _rigid(seed, degrees, metres):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=3)
    a /= np.linalg.norm(a)
    t = math.radians(rng.uniform(0.25, 1.0) * degrees)
    K = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
    G = np.eye(4)
    G[:3, :3] = np.eye(3) + math.sin(t) * K + (1 - math.cos(t)) * (K @ K)
    d = rng.normal(size=3)
    G[:3, 3] = d / np.linalg.norm(d) * metres * rng.uniform(0.25, 1.0)
    return G


def _focal(w):
    return 0.9609375 * w


def _render(scene, w, h, pose, seed):
    """(depth in metres, hit normal, colour bytes B G R, valid) per pixel, for a camera at `pose`."""
    dev = "cuda"
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    f, s = _focal(w), scene["scale"]
    xs = (torch.arange(w, dtype=torch.float64, device=dev) - 0.5 - w / 2) / f
    ys = (torch.arange(h, dtype=torch.float64, device=dev) - 0.5 - h / 2) / f
    y, x = torch.meshgrid(ys, xs, indexing="ij")
    rays = torch.stack([x, y, torch.ones_like(x)], -1)
    R = torch.tensor(pose[:3, :3], dtype=torch.float64, device=dev)
    o = torch.tensor(pose[:3, 3], dtype=torch.float64, device=dev)
    d = rays @ R.T
    best = torch.full((h, w), math.inf, dtype=torch.float64, device=dev)
    obj = torch.zeros((h, w), dtype=torch.int64, device=dev)
    nrm = torch.zeros((h, w, 3), dtype=torch.float64, device=dev)
    for k, (n, dist) in enumerate(scene["walls"]):
        n = torch.tensor(n, device=dev)
        t = (dist - o @ n) / (d @ n)
        hit = (t > 1e-6) & (t < best)
        best, obj, nrm = torch.where(hit, t, best), torch.where(hit, k, obj), torch.where(hit[..., None], n, nrm)
    for k, (c, r) in enumerate(scene["balls"]):
        oc = o - torch.tensor(c, device=dev)
        a, b = (d * d).sum(-1), d @ oc
        disc = b * b - a * (oc @ oc - r * r)
        t = torch.where(disc >= 0, (-b - disc.clamp(min=0).sqrt()) / a, math.inf)
        hit = (t > 1e-6) & (t < best)
        n = (oc + t.nan_to_num(posinf=0.0)[..., None] * d) / r
        best, obj, nrm = torch.where(hit, t, best), torch.where(hit, 3 + k, obj), torch.where(hit[..., None], n, nrm)
    z = best + torch.randn((h, w), generator=gen, dtype=torch.float64, device=dev) * 0.002
    valid = torch.isfinite(best) & (best >= 0.4 * s) & (best <= 3.4 * s)
    valid &= torch.rand((h, w), generator=gen, device=dev) >= 0.05
    col = torch.tensor(scene["colours"], device=dev)[obj]
    col = (col + torch.randint(-10, 11, (h, w, 3), generator=gen, device=dev)).clamp(0, 255).to(torch.uint8)
    return z, nrm @ R, col, valid


def _frame(scene, w, h, pose, seed):
    """A sensor frame: depth (millimetres, the bits of uint16) and BGR, on the GPU."""
    z, _, col, valid = _render(scene, w, h, pose, seed)
    mm = torch.where(valid, (z * 1000.0).round(), 0.0).to(torch.int16)
    return mm.contiguous(), col.contiguous()


def _points(scene, w, h, pose, seed):
    """FILL of a frame's pixels as points in raster order: (xyz [n, 3], rgb [n, 3], normals [n, 3]) in
    float32, and the pixel of each point."""
    z, nrm, col, valid = _render(scene, w, h, pose, seed)
    z = ((z * 1000.0).round() * 0.001).float()
    f = _focal(w)
    u = torch.arange(w, dtype=torch.float32, device="cuda") - 0.5 - w / 2
    v = torch.arange(h, dtype=torch.float32, device="cuda") - 0.5 - h / 2
    xyz = torch.stack([u[None, :] * z / f, v[:, None] * z / f, z], -1)
    rgb = col.flip(-1).float() * (1.0 / 255.0)
    nrm = torch.where(nrm[..., 2:] > 0, -nrm, nrm).float()
    pix = valid.flatten().nonzero().squeeze(1)
    n = int(FILL * w * h)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 3)
    pick = torch.randperm(len(pix), generator=gen, device="cuda")
    while len(pick) < n:  # a view past the walls: some pixels twice
        pick = torch.cat([pick, pick])
    pix = pix[pick[:n]].sort()[0]
    return xyz.reshape(-1, 3)[pix], rgb.reshape(-1, 3)[pix], nrm.reshape(-1, 3)[pix], pix


def _pair(seed, w, h, degrees=10.0, metres=0.1):
    """Points of a target frame and of a source frame from a camera moved by G (source -> target)."""
    scene, G = _scene(seed), _rigid(seed + 7919, degrees, metres)
    return _points(scene, w, h, np.eye(4), 2 * seed + 1), _points(scene, w, h, G, 2 * seed + 2), G


def _upload(xyz, rgb):
    return g.PointCloud.from_numpy(xyz.cpu().numpy(), rgb.cpu().numpy())


class _View:
    def __init__(self, owner, ptr, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n, 4), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _view(owner, ptr, n):
    """n float4 records of a cloud as a tensor, without a copy; the tensor keeps the cloud alive."""
    return torch.as_tensor(_View(owner, ptr, n), device="cuda")


def _out(cap):
    """A cloud of `cap` points, kept for a pass's output (an empty one would not be taken as `out`), and
    its arrays as they lie in memory."""
    pc = g.PointCloud.from_numpy(np.zeros((cap, 3), np.float32), np.zeros((cap, 3), np.float32))
    xyzi, rgb, normals, gradient = (_view(pc, p, cap).zero_() for p in pc.device_arrays()[:4])
    torch.cuda.synchronize()
    return pc, {"xyz": xyzi[:, :3], "intensity": xyzi[:, 3], "rgb": rgb[:, :3], "normals": normals[:, :3],
                "gradient": gradient[:, :3]}


def _cloud(pc, arrays, *names):
    return {"n": pc.points_number(), **{k: arrays[k] for k in ("xyz", "intensity", "rgb") + names}}


def _to(x, cap):
    return torch.cat([x, torch.zeros((cap - len(x),) + x.shape[1:], dtype=x.dtype, device=x.device)])


def _levels(case):
    return tuple(0.04 / 2 ** k for k in range(case["levels"]))


def _reports(rows):
    """The reports of registrations and their levels as arrays [registration, level]."""
    return {"iterations": np.array([[r.iterations for r in row] for row in rows]),
            "matches": np.array([[r.n_correspondences for r in row] for row in rows]),
            "rmse": np.array([[r.rmse for r in row] for row in rows]),
            "fitness": np.array([[r.fitness for r in row] for row in rows])}


# ---- prepare and run ------------------------------------------------------------------------------

def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["kind"]][1](state)


def _camera(w, h):
    return g.make_camera(w, h, _focal(w), _focal(w), w / 2, h / 2)


def _cloud_prepare(case, seed):
    w, h = case["w"], case["h"]
    depth, bgr = _frame(_scene(seed), w, h, np.eye(4), seed + 1)
    mode = {"fixed": g.BILATERAL_FIXED, "adaptive": g.BILATERAL_REFERENCE_ADAPTIVE, "none": g.BILATERAL_NONE}[case["filter"]]
    out, arrays = _out(w * h)
    return {"kind": "cloud", "depth": depth, "bgr": bgr, "cam": _camera(w, h),
            "filter": g.bilateral(mode, case["radius"], 2.0, 30.0), "out": out, "arrays": arrays}


def _cloud_run(s):
    pc = g.PointCloud.create_from_rgbd(s["depth"], s["bgr"], s["cam"], s["filter"], TMIN, TMAX, out=s["out"])
    return _cloud(pc, s["arrays"])


def _target_prepare(case, seed):
    xyz, rgb, _, _ = _points(_scene(seed), case["w"], case["h"], np.eye(4), seed + 1)
    out, arrays = _out(len(xyz))
    return {"kind": "target", "case": case, "full": _upload(xyz, rgb), "out": out, "arrays": arrays}


def _target_run(s):
    v = s["case"]["voxel"]
    t = s["full"].voxel_grid_down_sample(v, out=s["out"])
    t.estimate_normals(2.5 * v, s["case"]["max_nn"])
    t.compute_color_gradient(2.0 * v, 0)
    return _cloud(t, s["arrays"], "normals", "gradient")


def _align_prepare(case, seed):
    (tx, tr, _, _), (sx, sr, _, _), _ = _pair(seed, case["w"], case["h"])
    return {"kind": "align", "case": case, "src": _upload(sx, sr), "tgt": _upload(tx, tr)}


def _align_run(s):
    v = s["case"]["voxel"]
    src = s["src"].voxel_grid_down_sample(v)
    tgt = s["tgt"].voxel_grid_down_sample(v)
    tgt.estimate_normals(2.5 * v, 30)
    icp = g.ColorICP(s["case"]["iters"], 2.5 * v, 2.0 * v, s["case"]["accum"])
    icp.set_source_point_cloud(src)
    icp.set_target_point_cloud(tgt)
    icp.align()
    return {"T": icp.get_final_transformation_matrix(), **_reports([[icp.report]])}


def _multiscale_prepare(case, seed):
    s = _align_prepare(case, seed)
    s["kind"] = "multiscale"
    s["levels"] = [g.level_params(v, icp=g.icp_params(case["iters"], 2.5 * v)) for v in _levels(case)]
    return s


def _multiscale_run(s):
    T, reps = g.multiscale_icp(s["src"], s["tgt"], s["levels"])
    return {"T": T, **_reports([reps])}


def _odometry_prepare(case, seed):
    w, h, scene = case["w"], case["h"], _scene(seed)
    frames = [_frame(scene, w, h, _rigid(seed + 31 * k, 5.0, 0.05), seed + 1 + k) for k in range(case["frames"])]
    pipe = FramePipeline(g.default_context(), _camera(w, h), g.bilateral(g.BILATERAL_FIXED, 2, 2.0, 30.0),
                         overlap=case["overlap"])
    autotune.apply(pipe.ctx, workload="frame_overlapped" if case["overlap"] else "frame")
    torch.cuda.synchronize()
    return {"kind": "odometry", "overlap": case["overlap"], "pipe": pipe, "frames": frames}


def _odometry_run(s):
    # a pass steps the whole sequence; its first frame's pose depends on what was stepped before, so
    # the poses returned are those of the later frames
    pipe, poses, rows = s["pipe"], [], []
    for k, (depth, bgr) in enumerate(s["frames"]):
        pipe.step(depth.data_ptr(), bgr.data_ptr())
        if not s["overlap"]:
            T, reps = pipe.result()
            if k:
                poses.append(T)
                rows.append(_read(reps))
    if s["overlap"]:
        pipe.flush()
        T, reps = pipe.result()
        poses.append(T)
        rows.append(_read(reps))
    return {"T": np.stack(poses), "reports": np.array(rows)}


def _read(reps):
    # a pipeline's reports are its own buffers, written again by the next result
    return [[r.iterations, r.n_correspondences, r.rmse, r.fitness] for r in reps]


def _batch_prepare(case, seed):
    rng = np.random.default_rng(seed)
    # counts evenly spread over the logarithm of the range, so that every seed costs the same
    q = (np.arange(case["pairs"]) + 0.5) / case["pairs"]
    counts = np.rint(np.exp(math.log(case["lo"]) + q * math.log(case["hi"] / case["lo"]))).astype(int)
    rng.shuffle(counts)
    levels, src, tgt = _levels(case), [], []
    for k, n in enumerate(counts):
        w = int(max(64, math.sqrt(n * 4.0 / 3.0 / 0.85)))
        scene, G = _scene(seed + 17 * k, 2.0), _rigid(seed + 17 * k + 104729, 15.0, 0.2)
        rows = []
        for j, pose in enumerate((G, np.eye(4))):
            xyz, rgb, _, _ = _points(scene, w, w * 3 // 4, pose, seed + 17 * k + j)
            full = _upload(xyz[:n], rgb[:n])
            rows.append([full.voxel_grid_down_sample(v) for v in levels])
        for v, t in zip(levels, rows[1]):
            t.estimate_normals(2.5 * v, 30)
            t.compute_color_gradient(2.0 * v, 0)
        src.append(rows[0])
        tgt.append(rows[1])
    g.default_context().synchronize()
    return {"kind": "batch", "src": src, "tgt": tgt, "params": [g.icp_params(case["iters"], 2.5 * v) for v in levels],
            "T0": np.tile(np.eye(4), (len(counts), 1, 1)), "grad": [2.0 * v for v in levels]}


def _batch_run(s):
    T, reps = g.batch_multiscale_icp(s["src"], s["tgt"], s["params"], s["T0"], s["grad"])
    return {"T": T, **_reports(reps)}


def _objective_inputs(case, seed):
    """Source, target with normals and a tangential colour gradient, the pixel a source point falls on
    in the target's frame as its match (-1: none there), and a pose a little off the true one."""
    n = case["n"]
    w = int(max(64, math.sqrt(n * 4.0 / 3.0 / 0.8)))
    h = w * 3 // 4
    (tx, tr, tn, pix), (sx, sr, _, _), G = _pair(seed, w, h)
    sx, sr = sx[:n], sr[:n]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    grad = torch.randn((len(tx), 3), generator=gen, device="cuda")
    grad = grad - (grad * tn).sum(1, keepdim=True) * tn
    at = torch.full((w * h,), -1, dtype=torch.int32, device="cuda")
    at[pix] = torch.arange(len(pix), dtype=torch.int32, device="cuda")
    p = sx.double() @ torch.tensor(G[:3, :3].T, device="cuda") + torch.tensor(G[:3, 3], device="cuda")
    u = (p[:, 0] / p[:, 2] * _focal(w) + w / 2 + 0.5).round().long()
    v = (p[:, 1] / p[:, 2] * _focal(w) + h / 2 + 0.5).round().long()
    inside = (u >= 0) & (u < w) & (v >= 0) & (v < h)
    nn = torch.where(inside, at[(v.clamp(0, h - 1) * w + u.clamp(0, w - 1))], -1).to(torch.int32)
    T = _rigid(seed + 5, 0.5, 0.01) @ G
    xi = np.random.default_rng(seed).uniform(-0.005, 0.005, 6)
    I = (0.2126 * sr[:, 0].double() + 0.7152 * sr[:, 1].double() + 0.0722 * sr[:, 2].double()).float()
    return torch.cat([sx, I[:, None]], 1).contiguous(), tx, tr, tn, grad, nn, T, xi


def _objective_prepare(case, seed):
    src, tx, tr, tn, grad, nn, T, xi = _objective_inputs(case, seed)
    tgt = _upload(tx, tr)
    tgt.set_normals(tn.cpu().numpy())
    tgt.set_gradient(grad.cpu().numpy())
    return {"kind": "objective", "src": src, "tgt": tgt, "nn": nn, "T": T,
            "xi": torch.tensor(xi, dtype=torch.float64, device="cuda"), "work": g.PointCloud(None, len(src))}


def _objective_run(s):
    xi = s["xi"].clone().requires_grad_(True)
    p = s["src"].clone().requires_grad_(True)
    E = colored_icp_objective(xi, p, s["tgt"], s["nn"], s["T"], LAMBDA, s["work"])
    E.backward()
    return {"E": E.detach(), "dxi": xi.grad, "dpoints": p.grad}


def _neighbours_prepare(case, seed):
    xyz, rgb, _, _ = _points(_scene(seed), case["w"], case["h"], np.eye(4), seed + 1)
    keys = torch.arange(seed % 8, len(xyz), 8, device="cuda")[:len(xyz) // 8]
    most = len(keys) * (case["max_nn"] or int(40 * _density(case) * math.pi * case["radius_m"] ** 2))
    return {"kind": "neighbours", "case": case, "scan": _upload(xyz, rgb), "keys": _upload(xyz[keys], rgb[keys]),
            "idx": np.zeros(most, np.int32), "xyzi": torch.zeros((len(xyz), 4), device="cuda"),
            "rgb": torch.zeros((len(xyz), 4), device="cuda")}


def _neighbours_run(s):
    c = s["case"]
    clean = s["clean"] = s["scan"].radius_outlier_removal(c["radius_m"], c["min_nn"])
    offsets, idx = g.PointCloud.radius_search(s["keys"], clean, c["radius_m"], c["max_nn"])
    s["idx"][:len(idx)] = idx
    n, p = clean.points_number(), clean.device_arrays()
    s["xyzi"][:n] = _view(clean, p[0], n)
    s["rgb"][:n] = _view(clean, p[1], n)
    return {"n": n, "offsets": offsets, "idx": s["idx"], "xyzi": s["xyzi"], "rgb": s["rgb"]}


def _segment_inputs(case, seed):
    (tx, tr, tn, _), (sx, sr, sn, _), G = _pair(seed, case["w"], case["h"], 5.0, 0.05)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    grad = torch.randn((len(tx), 3), generator=gen, device="cuda")
    grad = 0.5 * (grad - (grad * tn).sum(1, keepdim=True) * tn)
    return tx, tr, tn, grad, sx, sr, sn, G


def _segment_prepare(case, seed):
    tx, tr, tn, grad, sx, sr, sn, G = _segment_inputs(case, seed)
    tgt, src = _upload(tx, tr), _upload(sx, sr)
    tgt.set_normals(tn.cpu().numpy())
    tgt.set_gradient(grad.cpu().numpy())
    src.set_normals(sn.cpu().numpy())
    return {"kind": "segment", "case": case, "src": src, "tgt": tgt, "T": G}


def _segment_run(s):
    c = s["case"]
    moved = s["src"].copy()
    moved.transform(s["T"])
    nn = g.PointCloud.nn_search(moved, s["tgt"], c["corr"], as_tensor=True)
    res, total = g.compute_residuals(moved, s["tgt"], nn, g.RESIDUAL_ABS, LAMBDA)
    big = moved.points_number()
    seg, n_seg, _ = moved.residual_segment_labels(c["tol"], res, c["min_size"], big)
    obj, n_obj, _ = moved.euclidean_cluster_labels(c["tol"], c["min_size"], big)
    return {"nn": nn, "residual": res, "total": total, "segments": seg, "n_segments": n_seg, "objects": obj,
            "n_objects": n_obj}


def _map_inputs(case, seed):
    scene = _scene(seed)
    poses = [_rigid(seed + 31 * k, 20.0, 0.3) for k in range(case["frames"] + 1)]
    clouds = [_points(scene, case["w"], case["h"], P, seed + 1 + k)[:2] for k, P in enumerate(poses)]
    world = [torch.cat([(x.double() @ torch.tensor(P[:3, :3].T, device="cuda") + torch.tensor(P[:3, 3], device="cuda")).float()
                        for (x, _), P in zip(clouds[1:], poses[1:])]), torch.cat([c for _, c in clouds[1:]])]
    return world, clouds[0], poses[0]


def _map_prepare(case, seed):
    (mx, mr), (fx, fr), P = _map_inputs(case, seed)
    out, arrays = _out(len(mx) + len(fx))
    return {"kind": "map", "map": _upload(mx, mr), "frame": _upload(fx, fr), "T": P, "voxel": case["voxel"],
            "out": out, "arrays": arrays}


def _map_run(s):
    grown = s["frame"].copy()
    grown.transform(s["T"])
    grown += s["map"]
    return _cloud(grown.voxel_grid_down_sample(s["voxel"], out=s["out"]), s["arrays"])


_KINDS = {"cloud": (_cloud_prepare, _cloud_run), "target": (_target_prepare, _target_run),
          "align": (_align_prepare, _align_run), "multiscale": (_multiscale_prepare, _multiscale_run),
          "odometry": (_odometry_prepare, _odometry_run), "batch": (_batch_prepare, _batch_run),
          "objective": (_objective_prepare, _objective_run), "neighbours": (_neighbours_prepare, _neighbours_run),
          "segment": (_segment_prepare, _segment_run), "map": (_map_prepare, _map_run)}


# ---- work -----------------------------------------------------------------------------------------

def _occupied(n, voxel, area=AREA):
    cells = area / voxel ** 2
    return cells * (1.0 - math.exp(-n / cells))


def _density(case):
    """Points per square metre of surface, about."""
    return FILL * case["w"] * case["h"] / AREA


def _target_work(n, voxels):
    # points and colours read once; per level its points, colours, normals and gradients written; per
    # point some 30 neighbours of 40 operations and the two small solves
    m = [_occupied(n, v) for v in voxels]
    return 32 * n + 64 * sum(m), 20 * n * len(m) + 1700 * sum(m)


def _icp_work(m, iters=4):
    # both clouds with the target's normals and gradient read once; per iteration and point a search
    # among some 10 candidates and 28 products
    return 16 * m + 48 * m, iters * m * 250


def work(case):
    k = case["kind"]
    n = int(FILL * case.get("w", 0) * case.get("h", 0))
    if k == "cloud":
        px = case["w"] * case["h"]
        taps = {"fixed": (2 * case["radius"] + 1) ** 2, "adaptive": 50, "none": 0}[case["filter"]]
        return {"bytes": 5 * px + 32 * n, "flops": px * (4 * taps + 40)}
    if k == "target":
        b, f = _target_work(n, [case["voxel"]])
        return {"bytes": b, "flops": f}
    if k in ("align", "multiscale"):
        levels = [case["voxel"]] if k == "align" else _levels(case)
        b, f = _target_work(n, levels)
        total, flops = b + 32 * n + 32 * sum(_occupied(n, v) for v in levels), f + 20 * n
        for v in levels:
            ib, jf = _icp_work(_occupied(n, v))
            total, flops = total + ib, flops + jf
        return {"bytes": total, "flops": flops}
    if k == "odometry":
        px = case["w"] * case["h"]
        levels = (0.04, 0.02, 0.01)
        b, f = _target_work(n, levels)
        for v in levels:
            ib, jf = _icp_work(_occupied(n, v))
            b, f = b + ib, f + jf
        return {"bytes": case["frames"] * (5 * px + 32 * n + b), "flops": case["frames"] * (140 * px + f)}
    if k == "batch":
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        m = case["pairs"] * sum(_occupied(mean, v, 4 * AREA) for v in _levels(case))
        b, f = _icp_work(m)
        return {"bytes": b, "flops": f}
    if k == "objective":
        return {"bytes": case["n"] * (16 + 4 + 48 + 16), "flops": case["n"] * 200}
    if k == "neighbours":
        near = min(case["max_nn"] or 1e9, _density(case) * math.pi * case["radius_m"] ** 2)
        return {"bytes": n * 64 + n / 8 * (16 + 4 + 4 * near), "flops": n * 10 * case["min_nn"] + n / 8 * 20 * near}
    if k == "segment":
        near = _density(case) * math.pi * case["tol"] ** 2
        return {"bytes": n * (48 + 48 + 4 + 4 + 8), "flops": n * (2 * 10 * near + 300)}
    total = n * (case["frames"] + 1)
    return {"bytes": 32 * total + 32 * _occupied(total, case["voxel"], 1.5 * AREA), "flops": 30 * total}


# ---- exact values ---------------------------------------------------------------------------------

def _near(q, p, r):
    """Pairs (query, point, squared distance) with distance below r, by query, distance, point."""
    q, p, out = q.double(), p.double(), []
    step = max(1, 60_000_000 // max(1, len(p)))
    for a in range(0, len(q), step):
        c = q[a:a + step]
        d2 = (c[:, 0, None] - p[None, :, 0]).square_()
        d2 += (c[:, 1, None] - p[None, :, 1]).square_()
        d2 += (c[:, 2, None] - p[None, :, 2]).square_()
        at = (d2 < float(np.float32(r)) ** 2).nonzero()
        out.append((at[:, 0] + a, at[:, 1], d2[at[:, 0], at[:, 1]]))
    i, j, d2 = (torch.cat(x) for x in zip(*out))
    o = torch.sort(d2, stable=True)[1]  # by query, then distance, then point
    o = o[torch.sort(i[o], stable=True)[1]]
    return i[o], j[o], d2[o]


def _nearest(q, p, r):
    """Index of each query's nearest point below r, -1 without one."""
    q, p, out = q.double(), p.double(), []
    step = max(1, 60_000_000 // max(1, len(p)))
    for a in range(0, len(q), step):
        c = q[a:a + step]
        d2 = (c[:, 0, None] - p[None, :, 0]).square_()
        d2 += (c[:, 1, None] - p[None, :, 1]).square_()
        d2 += (c[:, 2, None] - p[None, :, 2]).square_()
        d, j = d2.min(1)
        out.append(torch.where(d < float(np.float32(r)) ** 2, j, -1))
    return torch.cat(out)


def _luma(rgb):
    return 0.2126 * rgb[:, 0] + 0.7152 * rgb[:, 1] + 0.0722 * rgb[:, 2]


def _voxel_exact(xyz, rgb, v):
    """Means over the voxels of the points' own 32-bit lattice, in lattice order."""
    lo = xyz.amin(0)
    key = torch.floor((xyz - lo) / torch.tensor(v, dtype=torch.float32, device=xyz.device)).long()
    dims = key.amax(0) + 1
    _, inv, cnt = torch.unique((key[:, 0] * dims[1] + key[:, 1]) * dims[2] + key[:, 2], return_inverse=True, return_counts=True)
    mean = lambda a: torch.zeros((len(cnt), 3), dtype=torch.float64, device=a.device).index_add_(0, inv, a.double()) / cnt[:, None]  # noqa: E731
    return mean(xyz), mean(rgb)


def _segsum(i, x, m):
    return torch.zeros((m,) + x.shape[1:], dtype=torch.float64, device=x.device).index_add_(0, i, x)


def _normals_exact(p, r, k):
    m = len(p)
    i, j, _ = _near(p, p, r)
    if k:
        first = torch.searchsorted(i, torch.arange(m, device=p.device))
        keep = torch.arange(len(i), device=p.device) - first[i] < k
        i, j = i[keep], j[keep]
    u = p[j] - p[i]
    n = _segsum(i, torch.ones_like(u[:, 0]), m)
    mean = _segsum(i, u, m) / n[:, None]
    cov = _segsum(i, u[:, :, None] * u[:, None, :], m) / n[:, None, None] - mean[:, :, None] * mean[:, None, :]
    v = torch.linalg.eigh(cov.cpu())[1][:, :, 0].to(p.device)
    v = torch.where(v[:, 2:] > 0, -v, v)
    return torch.where((n >= 3)[:, None], v, 0.0)


def _gradient_exact(p, intensity, nrm, r):
    m = len(p)
    i, j, _ = _near(p, p, r)
    u = p[j] - p[i]
    u = u - (u * nrm[i]).sum(1, keepdim=True) * nrm[i]
    n = _segsum(i, torch.ones_like(u[:, 0]), m)
    A = _segsum(i, u[:, :, None] * u[:, None, :], m) + ((n - 1) ** 2)[:, None, None] * nrm[:, :, None] * nrm[:, None, :]
    A += 1e-6 * torch.eye(3, dtype=torch.float64, device=p.device)
    b = _segsum(i, u * (intensity[j] - intensity[i])[:, None], m)
    return torch.where((n >= 5)[:, None], torch.linalg.solve(A.cpu(), b.cpu()[:, :, None])[:, :, 0].to(p.device), 0.0)


def _cloud_exact(case, seed):
    # points by the filter's definition; a point's colour pixel hangs on the rounding of its 32-bit
    # projection (a projected pixel centre lies on the edge between two pixels), so it has no such value
    depth = _frame(_scene(seed), case["w"], case["h"], np.eye(4), seed + 1)[0].double()
    h, w = depth.shape
    scale = float(np.float32(0.001))
    tmin, tmax = float(np.float32(TMIN)), float(np.float32(TMAX))
    out = depth.clone()
    steps = [(case["radius"], 2.0, 30.0, None)] if case["filter"] == "fixed" else []
    if case["filter"] == "adaptive":
        steps = [(k, 8.0 + k, 100.0 + 10.0 * k, k) for k in range(6)]
    band = ((depth * scale - tmin) / 0.5).clamp(min=0).floor().clamp(max=5)
    for r, ss, sd, k in steps:
        pad = torch.nn.functional.pad(depth[None, None], (r, r, r, r))[0, 0]
        sw, swd = torch.zeros_like(depth), torch.zeros_like(depth)
        for dy in range(2 * r + 1):
            for dx in range(2 * r + 1):
                d = pad[dy:dy + h, dx:dx + w]
                wt = math.exp(-((dx - r) ** 2 + (dy - r) ** 2) / ss ** 2) * torch.exp(-(d - depth).square() / sd ** 2)
                wt = torch.where(d > 0, wt, 0.0)
                sw += wt
                swd += wt * d
        f = swd / sw
        out = torch.where(band == k, f, out) if k is not None else f
    z = out * scale
    ok = (depth > 0) & (depth * scale >= tmin) & (depth * scale <= tmax) & (z >= tmin) & (z <= tmax)
    f = float(np.float32(_focal(w)))
    x = (torch.arange(w, dtype=torch.float64, device="cuda") - 0.5 - w / 2)[None, :] * z / f
    y = (torch.arange(h, dtype=torch.float64, device="cuda") - 0.5 - h / 2)[:, None] * z / f
    return {"n": None, "xyz": _to(torch.stack([x, y, z], -1)[ok], w * h), "intensity": None, "rgb": None}


def _target_exact(case, seed):
    v = case["voxel"]
    xyz, rgb, _, _ = _points(_scene(seed), case["w"], case["h"], np.eye(4), seed + 1)
    p, c = _voxel_exact(xyz, rgb, v)
    # later stages start from the points and colours as a cloud holds them, in 32 bits
    q, I = p.float().double(), _luma(c.float().double()).float().double()
    nrm = _normals_exact(q, 2.5 * v, case["max_nn"])
    out = {"xyz": p, "intensity": _luma(c), "rgb": c, "normals": nrm, "gradient": _gradient_exact(q, I, nrm, 2.0 * v)}
    return {"n": None, **{k: _to(x, len(xyz)) for k, x in out.items()}}


def _register_exact(src, tgt, voxels, iters):
    """Coarse-to-fine colored ICP in 64 bits: the pose, and per level the mean square and the share matched."""
    dev = "cuda"
    T, got = torch.eye(4, dtype=torch.float64, device=dev), []
    for v in voxels:
        (s, sc), (t, tc) = _voxel_exact(*src, v), _voxel_exact(*tgt, v)
        s, t = s.float().double(), t.float().double()
        sI, tI = (_luma(c.float().double()).float().double() for c in (sc, tc))
        nrm = _normals_exact(t, 2.5 * v, 30)
        grd = _gradient_exact(t, tI, nrm, 2.0 * v)
        for _ in range(iters):
            p = s @ T[:3, :3].T + T[:3, 3]
            j = _nearest(p, t, 2.5 * v)
            on = j >= 0
            p, j, I = p[on], j[on], sI[on]
            q, n, d = t[j], nrm[j], grd[j]
            rg = ((p - q) * n).sum(1)
            gt = d - (d * n).sum(1, keepdim=True) * n
            rc = tI[j] + (d * (p - rg[:, None] * n - q)).sum(1) - I
            lam = float(np.float32(LAMBDA))
            J = torch.cat([math.sqrt(lam) * torch.cat([torch.linalg.cross(p, n), n], 1),
                           math.sqrt(1 - lam) * torch.cat([torch.linalg.cross(p, gt), gt], 1)])
            r = torch.cat([math.sqrt(lam) * rg, math.sqrt(1 - lam) * rc])
            x = torch.linalg.solve((J.T @ J).cpu(), -(J.T @ r).cpu()).numpy()
            (a, b, c) = x[:3]
            Rx = np.array([[1, 0, 0], [0, math.cos(a), -math.sin(a)], [0, math.sin(a), math.cos(a)]])
            Ry = np.array([[math.cos(b), 0, math.sin(b)], [0, 1, 0], [-math.sin(b), 0, math.cos(b)]])
            Rz = np.array([[math.cos(c), -math.sin(c), 0], [math.sin(c), math.cos(c), 0], [0, 0, 1]])
            D = np.eye(4)
            D[:3, :3], D[:3, 3] = Rz @ Ry @ Rx, x[3:]
            T = torch.tensor(D, device=dev) @ T
            last = (float((r * r).sum()) / len(s), len(j) / len(s))
            if 0.5 * (np.trace(D[:3, :3]) - 1) >= 1 - 1e-6 and (x[3:] ** 2).sum() <= 1e-6:
                break
        got.append(last)
    return {"T": T.cpu().numpy(), "iterations": None, "matches": None, "rmse": np.array([[r for r, _ in got]]),
            "fitness": np.array([[f for _, f in got]])}


def _align_exact(case, seed):
    (tx, tr, _, _), (sx, sr, _, _), _ = _pair(seed, case["w"], case["h"])
    return _register_exact((sx, sr), (tx, tr), [case["voxel"]], case["iters"])


def _multiscale_exact(case, seed):
    if case["w"] * case["h"] > 500_000:  # all distances of the finest level: too long
        return None
    (tx, tr, _, _), (sx, sr, _, _), _ = _pair(seed, case["w"], case["h"])
    return _register_exact((sx, sr), (tx, tr), _levels(case), case["iters"])


def _objective_exact(case, seed):
    src, tx, tr, tn, grad, nn, T, x = _objective_inputs(case, seed)
    xi = torch.tensor(x, dtype=torch.float64, device="cuda", requires_grad=True)
    p4 = src.double().requires_grad_(True)
    zero, one = torch.zeros_like(xi[0]), torch.ones_like(xi[0])
    c, s = torch.cos(xi[:3]), torch.sin(xi[:3])
    Rx = torch.stack([one, zero, zero, zero, c[0], -s[0], zero, s[0], c[0]]).reshape(3, 3)
    Ry = torch.stack([c[1], zero, s[1], zero, one, zero, -s[1], zero, c[1]]).reshape(3, 3)
    Rz = torch.stack([c[2], -s[2], zero, s[2], c[2], zero, zero, zero, one]).reshape(3, 3)
    on = nn >= 0
    j = nn[on].long()
    T = torch.tensor(T, device="cuda")
    p = (p4[on, :3] @ T[:3, :3].T + T[:3, 3]) @ (Rz @ Ry @ Rx).T + xi[3:]
    q, n, d = tx.double()[j], tn.double()[j], grad.double()[j]
    I = _luma(tr.double()).float().double()[j]
    rg = ((p - q) * n).sum(1)
    rc = I + (d * (p - rg[:, None] * n - q)).sum(1) - p4[on, 3]
    lam = float(np.float32(LAMBDA))
    E = lam * rg.square().sum() + (1 - lam) * rc.square().sum()
    E.backward()
    return {"E": E.detach(), "dxi": xi.grad, "dpoints": p4.grad}


def _segment_exact(case, seed):
    tx, tr, tn, grad, sx, sr, sn, G = _segment_inputs(case, seed)
    p = (sx.double() @ torch.tensor(G[:3, :3].T, device="cuda") + torch.tensor(G[:3, 3], device="cuda")).float().double()
    j = _nearest(p, tx, case["corr"])
    q, n, d = tx.double()[j], tn.double()[j], grad.double()[j]
    I, J = _luma(sr.double()).float().double(), _luma(tr.double()).float().double()[j]
    rg = ((p - q) * n).sum(1)
    rc = J + (d * (p - rg[:, None] * n - q)).sum(1) - I
    lam = float(np.float32(LAMBDA))
    res = torch.where(j >= 0, math.sqrt(lam) * rg.abs() + math.sqrt(1 - lam) * rc.abs(), 0.0)
    return {"nn": None, "residual": res, "total": float(res.sum()), "segments": None, "n_segments": None,
            "objects": None, "n_objects": None}


def _map_exact(case, seed):
    (mx, mr), (fx, fr), P = _map_inputs(case, seed)
    x = (fx.double() @ torch.tensor(P[:3, :3].T, device="cuda") + torch.tensor(P[:3, 3], device="cuda")).float()
    p, c = _voxel_exact(torch.cat([x, mx]), torch.cat([fr, mr]), case["voxel"])
    return {"n": None, **{k: _to(v, len(x) + len(mx)) for k, v in (("xyz", p), ("intensity", _luma(c)), ("rgb", c))}}


def exact(case, seed):
    # odometry and batches: discrete choices in 32 bits (which voxel a point falls in, when a level
    # stops) chain through whole sequences and levels of many pairs, so poses have no value in 64 bits
    # that could be had in seconds; neighbours: whole numbers and copies of the inputs only
    f = {"cloud": _cloud_exact, "target": _target_exact, "align": _align_exact, "multiscale": _multiscale_exact,
         "objective": _objective_exact, "segment": _segment_exact, "map": _map_exact}.get(case["kind"])
    return f(case, seed) if f else None
