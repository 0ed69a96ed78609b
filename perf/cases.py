"""The calls whose speed is kept in view, through the public entry points.

A case is a dict of plain values; ``listed()`` gives the named ones and
``draw(rng)`` further ones of the same ranges.  Kinds:

* ``fps``      nsfps_fps_device: device-resident points, a given range
* ``noalloc``  nsfps_fps_device_noalloc: the same with no device allocation
* ``host``     yuezu_fps_module.fps: a NumPy array in, a NumPy array out
* ``batched``  nsfps_fps_batched_device: clouds of one size, range=None or given
* ``plan``     nsfps_plan_sample on a plan that the program keeps
* ``group``    gather_points and ball_query on the samples' indices

Clouds (``cloud``): ``gauss`` N(0,1) in a +-100 range, ``cube`` uniform in
[-1,1]^3, ``lidar`` a rotating-LiDAR scan with box-shaped objects, ``shapes``
half ball, half jittered sphere with 1 % exact duplicates, ``clusters``
axis-aligned Gaussian clusters.  All results are indices or copied
coordinates, so every case is compared exactly.
"""

import math

import numpy as np
import torch

from ns_fps_amd import capi

_lib = None
_yf = None


def _capi():
    global _lib
    if _lib is None:
        _lib = capi.Lib()
    return _lib


def _module():
    global _yf
    if _yf is None:
        import yuezu_fps.yuezu_fps_module as yf
        _yf = yf
    return _yf


# ------------------------------------------------------------------ the cases

def _case(kind, cloud, n, m, grid, batch=1, ranged=True, radius=0.0, nsample=0):
    return {"kind": kind, "cloud": cloud, "n": n, "m": m, "batch": batch,
            "xb": grid[0], "yb": grid[1], "zb": grid[2], "ranged": ranged,
            "radius": radius, "nsample": nsample}


def listed():
    return [
        # one small object cloud, where launches and waits count
        dict(_case("fps", "cube", 1024, 256, (16, 16, 16)), name="object_1k"),
        # the reference's own quickstart (README, test.py)
        dict(_case("fps", "gauss", 10000, 1000, (16, 16, 16)), name="quickstart_10k"),
        # the drop-in call on host arrays: a scan's 16,384-point cut
        dict(_case("host", "lidar", 16384, 1024, (128, 128, 2)), name="host_cut_16k"),
        # a whole rotating-LiDAR scan
        dict(_case("fps", "lidar", 120000, 16384, (32, 32, 8)), name="lidar_120k"),
        # a scan's structure built once and sampled per request
        dict(_case("plan", "lidar", 124668, 16384, (128, 128, 2)), name="plan_lidar_125k"),
        # the headline: a dense cube, block counts that are powers of two
        dict(_case("fps", "cube", 1048576, 65536, (32, 32, 32)), name="uniform_1m"),
        # the same where cells share buckets
        dict(_case("fps", "cube", 1048576, 65536, (30, 30, 30)), name="uniform_1m_30"),
        # the first set-abstraction layer of a training batch
        dict(_case("batched", "shapes", 1024, 512, (16, 16, 16), batch=32, ranged=False),
             name="batch_32x1k"),
        # large set-abstraction clouds, 64 at once
        dict(_case("batched", "shapes", 16384, 4096, (16, 16, 16), batch=64, ranged=False),
             name="batch_64x16k"),
        # a map-scale cloud of clusters: the largest call
        dict(_case("fps", "clusters", 8388608, 524288, (64, 64, 64)), name="clustered_8m"),
        # grouping after sampling: a layer's worth of centers, and a whole scan's
        dict(_case("group", "shapes", 16384, 1024, (16, 16, 16), radius=0.2, nsample=32),
             name="group_16k"),
        dict(_case("group", "cube", 1048576, 65536, (32, 32, 32), radius=0.05, nsample=32),
             name="group_1m"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fps", "fps", "fps", "noalloc", "host", "batched", "batched", "plan", "group"])
    if kind == "batched":
        batch = _log_int(rng, 2, 64)
        n = _log_int(rng, 512, 16384)
        m = max(16, n // rng.randint(2, 16))
        return _case(kind, rng.choice(["shapes", "cube"]), n, m, rng.choice([(16, 16, 16), (8, 8, 8)]),
                     batch=batch, ranged=rng.random() < 0.3)
    cloud = rng.choice(["gauss", "cube", "lidar", "shapes", "clusters"])
    if kind == "group":
        n = _log_int(rng, 4096, 1048576)
        m = max(64, n // rng.randint(8, 32))
        # a radius of about nsample points for points that fill their volume
        unit = {"gauss": 1.0, "cube": 1.0, "lidar": 8.0, "shapes": 1.0, "clusters": 60.0}[cloud]
        nsample = rng.choice([16, 32, 64])
        return _case(kind, cloud, n, m, (16, 16, 16), radius=unit * (nsample / n) ** (1.0 / 3.0),
                     nsample=nsample)
    n = _log_int(rng, 600, {"fps": 4000000, "noalloc": 400000, "host": 400000, "plan": 1000000}[kind])
    m = max(32, n // rng.randint(4, 32))
    grids = {"gauss": [(16, 16, 16)], "cube": [(16, 16, 16), (32, 32, 32), (30, 30, 30), (17, 17, 17)],
             "lidar": [(32, 32, 8), (128, 128, 2)], "shapes": [(16, 16, 16), (32, 32, 32)],
             "clusters": [(64, 64, 64), (32, 32, 32)]}[cloud]
    return _case(kind, cloud, n, m, rng.choice(grids))


# ------------------------------------------------------------------ the inputs

_LIMITS = {"gauss": (-100.0, 100.0, -100.0, 100.0, -100.0, 100.0),
           "cube": (-1.0, 1.0, -1.0, 1.0, -1.0, 1.0),
           "lidar": (-80.0, 80.0, -80.0, 80.0, -4.0, 4.0),
           "shapes": (-1.1, 1.1, -1.1, 1.1, -1.1, 1.1),
           "clusters": (-600.0, 600.0, -600.0, 600.0, -600.0, 600.0)}


def _uniform(g, lo, hi, *size):
    return torch.rand(*size, generator=g, device=g.device) * (hi - lo) + lo


def _lidar(g, n):
    """64 beams, log-normal ranges, a ground plane at -1.7 m, and a fifth of
    the points on 40 boxes of 1 to 5 m standing on it."""
    per_box = n // 200
    ns = n - 40 * per_box
    beams = torch.deg2rad(_uniform(g, -25.0, 3.0, 64))
    e = beams[torch.randint(0, 64, (ns,), generator=g, device=g.device)]
    az = _uniform(g, 0.0, 2.0 * math.pi, ns)
    far = torch.exp(math.log(15.0) + 0.6 * torch.randn(ns, generator=g, device=g.device)).clamp(2.0, 80.0)
    ground = torch.where(e < 0, -1.7 / torch.sin(e), torch.full_like(e, math.inf))
    hit = ground < far
    t = torch.where(hit, ground, far)
    z = torch.where(hit, -1.7 + 0.03 * torch.randn(ns, generator=g, device=g.device), t * torch.sin(e))
    scan = torch.stack([t * torch.cos(e) * torch.cos(az), t * torch.cos(e) * torch.sin(az), z], 1)
    sides = _uniform(g, 1.0, 5.0, 40, 1, 3)
    centre = torch.cat([_uniform(g, -60.0, 60.0, 40, 1, 2), torch.full((40, 1, 1), -1.7, device=g.device)], 2)
    u = torch.rand(40, per_box, 3, generator=g, device=g.device)
    face = torch.randint(0, 5, (40, per_box), generator=g, device=g.device)
    u[..., 0] = torch.where(face == 0, 0.0, torch.where(face == 1, 1.0, u[..., 0]))
    u[..., 1] = torch.where(face == 2, 0.0, torch.where(face == 3, 1.0, u[..., 1]))
    u[..., 2] = torch.where(face == 4, 1.0, u[..., 2])
    u[..., :2] -= 0.5
    return torch.cat([scan, (centre + u * sides).reshape(-1, 3)], 0)


def _shapes(g, n):
    h = n // 2
    d = torch.randn(n, 3, generator=g, device=g.device)
    d = d / d.norm(dim=1, keepdim=True)
    d[:h] *= torch.rand(h, 1, generator=g, device=g.device) ** (1.0 / 3.0)
    d[h:] += 0.01 * torch.randn(n - h, 3, generator=g, device=g.device)
    dup = n // 100
    at = torch.randperm(n, generator=g, device=g.device)
    d[at[:dup]] = d[at[dup:2 * dup]]
    return d


def _clusters(g, n):
    centre = _uniform(g, -500.0, 500.0, 256, 3)
    sigma = torch.exp(_uniform(g, 0.0, math.log(30.0), 256, 3))
    k = torch.randint(0, 256, (n,), generator=g, device=g.device)
    return centre[k] + sigma[k] * torch.randn(n, 3, generator=g, device=g.device)


def _points(cloud, n, g):
    if cloud == "gauss":
        p = torch.randn(n, 3, generator=g, device=g.device)
    elif cloud == "cube":
        p = _uniform(g, -1.0, 1.0, n, 3)
    else:
        p = {"lidar": _lidar, "shapes": _shapes, "clusters": _clusters}[cloud](g, n)
    return p[torch.randperm(n, generator=g, device=g.device)].float().contiguous()


class _Plan:
    """A plan handle, given back with the state that holds it."""

    def __init__(self, points, n, rng):
        self.handle = _capi().plan_create(points.data_ptr(), n, rng, on_device=True)

    def __del__(self):
        _capi().plan_destroy(self.handle)


def prepare(case, seed):
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    kind, n, m, batch = case["kind"], case["n"], case["m"], case["batch"]
    blocks = (case["xb"], case["yb"], case["zb"])
    rng = capi.Range.of(_LIMITS[case["cloud"]] + blocks)
    pts = torch.stack([_points(case["cloud"], n, g) for _ in range(batch)])
    s = {"kind": kind, "n": n, "m": m, "batch": batch, "blocks": blocks, "pts": pts,
         "stream": torch.cuda.current_stream().cuda_stream or None}
    s["range"] = [rng] * batch if kind == "batched" and case["ranged"] else None if kind == "batched" else rng
    if kind == "group":
        s["idx"] = torch.randperm(n, generator=g, device=dev)[:m].int().contiguous()
        s["cen"] = torch.empty(m, 3, device=dev)
        s["out"] = torch.empty(m, case["nsample"], dtype=torch.int32, device=dev)
        s["radius"], s["nsample"] = case["radius"], case["nsample"]
    elif kind == "host":
        s["pts"] = pts[0].cpu().numpy()
        s["range"] = _module().make_range(*_LIMITS[case["cloud"]], *blocks)
    else:
        s["out"] = torch.full((batch, m), -1, dtype=torch.int32, device=dev)
    torch.cuda.synchronize()
    if kind == "plan":
        s["plan"] = _Plan(pts, n, rng)
    return s


# ------------------------------------------------------------------ the calls

def run(s):
    kind, n, m = s["kind"], s["n"], s["m"]
    if kind == "host":
        return {"idx": _module().fps(s["pts"], m, s["range"])}
    lib, stream, xyz = _capi(), s["stream"], s["pts"].data_ptr()
    if kind == "group":
        cen, out = s["cen"], s["out"]
        lib.gather_points_device(xyz, n, s["idx"].data_ptr(), m, cen.data_ptr(), stream)
        lib.ball_query_device(xyz, n, cen.data_ptr(), m, s["radius"], s["nsample"], out.data_ptr(), stream)
        return {"cen": cen, "idx": out}
    out = s["out"]
    if kind == "batched":
        lens = lib.fps_batched_device(xyz, s["batch"], n, m, out.data_ptr(), s["range"], s["blocks"], stream)
        return {"idx": out, "len": np.asarray(lens)}
    if kind == "plan":
        got = lib.plan_sample(s["plan"].handle, m, out.data_ptr(), stream)
    elif kind == "noalloc":
        got = lib.fps_device_noalloc(xyz, n, m, s["range"], out.data_ptr(), stream)
    else:
        got = lib.fps_device(xyz, n, m, s["range"], out.data_ptr(), stream)
    return {"idx": out, "len": got}


def work(case):
    """Each point read once and each result written once; every point's
    distance (8 operations) to at least one sample, or every neighbour's to
    its center."""
    n, m, b = case["n"], case["m"], case["batch"]
    if case["kind"] == "group":
        return {"bytes": 12 * n + 4 * m + 12 * m + 4 * m * case["nsample"], "flops": 8 * m * case["nsample"]}
    return {"bytes": b * (12 * n + 4 * m), "flops": 8 * b * n}


def tolerance(case):
    """Indices and copied coordinates: nothing may differ."""
    return "exact"


def exact(case, seed):
    """The gathered centers are copies of input rows; indices have no value in
    64 bits of their own."""
    if case["kind"] != "group":
        return None
    s = prepare(case, seed)
    return {"cen": s["pts"][0][s["idx"].long()].double(), "idx": None}
