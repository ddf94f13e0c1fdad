"""The work that users of this package have it do, as timed cases through its public entry points.

A mapper program takes lidar scans and turns them into cost maps: `Gvom` with host arrays (the reference's
calling pattern), the same with device-resident points, several scans per call, captured launch sequences,
the ROS node around it, and the differentiable map loss.  Map sizes, sensors and drop-out rates are those of
`gvom_synth.workload` and `bench.py` (16 x 512 to 128 x 2048 points, 64 x 64 x 32 to 512 x 512 x 64 voxels,
rings of 1 to 8 scans) and odd sizes between them.

`prepare` is a program in its steady state: a mapper whose ring is full and whose previous combined map
exists, and the next scans.  `run` is one pass: the next scan (or scans) in, the maps out.
"""
import math
import os
import random
import sys
from types import SimpleNamespace

import numpy as np
import torch   # before the package: both then use one HIP runtime, which map_loss needs

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "g-vom_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

XY_RES, Z_RES, MIN_DISTANCE = 0.4, 0.2, 1.0
W_HEIGHT = 0.1


def _case(**kw):
    c = dict(kind="device", rings=64, az=1024, batch=1, frames=1, xy=256, z=64, buffer=8, dropout=0.0, f64=False,
             transform="f32", overlap=False, ring_hint=False, ex=1, ez=1, debug=False)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a 16-ring sensor, one scan into a small local map, host arrays in and out
        _case(name="host small map", kind="host", rings=16, az=512, xy=64, z=32, buffer=1, dropout=0.05),
        # the reference's calling pattern at the headline size: numpy scan in, four numpy maps out
        _case(name="host frame", kind="host", rings=128, az=1024),
        # ros_numpy's float64 arrays (dropped returns removed) with tf's float64 matrix, an odd map size
        _case(name="host float64 ragged", kind="host", rings=64, az=1024, xy=250, z=60, buffer=4, dropout=0.25,
              f64=True, transform="f64"),
        # the ROS node with its default parameters: PointCloud2 in, OccupancyGrids and the debug clouds out
        _case(name="node tick", kind="node", rings=64, az=1024, buffer=4, dropout=0.05, debug=True),
        # points already on the GPU, maps stay there: default settings, no hint about the scan's order
        _case(name="device frame", rings=128, az=1024),
        # the same with what a caller with organised scans turns on: scan/combine overlap and the ring hint
        _case(name="device frame overlapped", rings=128, az=1024, overlap=True, ring_hint=True),
        # eight such frames captured once and replayed with new poses
        _case(name="graph of 8 frames", kind="graph", rings=128, az=1024, frames=8, overlap=True, ring_hint=True),
        # three sensors in one call, 10-40 % of the returns dropped, then one combine
        _case(name="batch of 3 sensors", kind="batch", rings=128, az=1024, batch=3, dropout=0.25),
        # the largest map and scan
        _case(name="large map", rings=128, az=2048, xy=512, z=64, dropout=0.10),
        # an odd tall map, world-frame points without a transform, a wider neighbourhood
        _case(name="tall odd map", rings=32, az=1800, xy=151, z=100, buffer=3, dropout=0.10, transform="none", ex=2),
        # training: the loss and its gradients through autograd on one scan
        _case(name="loss and gradients", kind="loss", rings=64, az=1024, buffer=1, dropout=0.05, f64=True,
              transform="f64"),
        # the same on a small scan and map, where the launches count
        _case(name="loss small", kind="loss", rings=16, az=512, xy=64, z=32, buffer=1, dropout=0.05, f64=True,
              transform="f64"),
    ]


def draw(rng):
    kind = rng.choice(["host", "host", "node", "device", "device", "device", "graph", "batch", "loss"])

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    rings, az = log(16, 128), log(512, 2048)
    c = _case(kind=kind, rings=rings, az=az, xy=log(64, 400), z=rng.randint(20, 96), buffer=rng.randint(1, 8),
              dropout=round(rng.choice([0.0, rng.uniform(0.0, 0.4)]), 3), f64=rng.random() < 0.3,
              transform=rng.choice(["f32", "f32", "f64", "none"]), ex=rng.choice([1, 1, 1, 2]))
    if kind == "node":
        c.update(transform="f64", f64=False, debug=rng.random() < 0.5, rings=max(rings, 32))
    elif kind == "loss":
        c.update(buffer=1, f64=True, transform="f64", ex=1)
    elif kind == "graph":
        c.update(frames=rng.randint(2, 4), overlap=True)
    elif kind == "batch":
        c.update(buffer=rng.randint(3, 8), batch=rng.randint(2, 3))
    elif kind == "device":
        c.update(overlap=rng.random() < 0.5)
    if kind in ("device", "graph") and c["dropout"] == 0.0 and c["rings"] >= 64:
        c.update(ring_hint=True)
    # the most expensive draw stays below the largest listed case
    while _voxels(c) * (c["buffer"] + 2) * c["frames"] > 500 * 500 * 64 * 10:
        c["xy"] = c["xy"] * 3 // 4
    return c


def _voxels(c):
    return c["xy"] * c["xy"] * c["z"]


# ---- scans: a spinning lidar over procedural terrain, made on the GPU from the seed ---------------------------

def _terrain(seed):
    """A raster of rolling ground with boxes and pits, 0.25 m cells over +-128 m, zero at the start pose."""
    r = random.Random(seed)
    n, res, half = 1024, 0.25, 128.0
    ax = -half + res * torch.arange(n, device="cuda", dtype=torch.float32)
    x, y = ax[:, None], ax[None, :]
    h = torch.zeros(n, n, device="cuda")
    for _ in range(8):
        a, lam, th, ph = r.uniform(0.05, 0.5), r.uniform(4, 24), r.uniform(0, 6.2832), r.uniform(0, 6.2832)
        h += a * torch.sin((x * math.cos(th) + y * math.sin(th)) * (6.2832 / lam) + ph)
    for _ in range(25):
        cx, cy = r.uniform(-40, 40), r.uniform(-40, 40)
        sx, sy, d = r.uniform(0.6, 3.0), r.uniform(0.6, 3.0), r.choice([-1.0, 1.0, 1.0]) * r.uniform(0.5, 2.0)
        if math.hypot(cx, cy) < 6.0:
            continue
        i, j, wi, wj = (int((v + o) / res) for v, o in ((cx, half), (cy, half), (sx, 0), (sy, 0)))
        h[i:i + wi + 1, j:j + wj + 1] += d
    return h - h[n // 2, n // 2].clone()


def _height(h, x, y):
    i = ((x + 128.0) * 4.0).long().clamp_(0, 1023)
    j = ((y + 128.0) * 4.0).long().clamp_(0, 1023)
    return h[i, j]


def _scans(case, seed, count):
    """`count` consecutive scans 0.4 m apart: per scan the sensor-frame points (kept returns, ring by ring), the
    vehicle position, the sensor-to-world matrix, and all rays' points with NaN where a return was dropped."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    h = _terrain(seed)
    rings, az = case["rings"], case["az"]
    span = 15.0 if rings <= 16 else 22.5
    el = torch.deg2rad(torch.linspace(-span, span, rings, device="cuda"))
    az0 = 6.2832 * torch.rand(1, device="cuda", generator=gen)
    a = az0 + (2 * math.pi / az) * torch.arange(az, device="cuda", dtype=torch.float32)
    d = torch.stack([torch.cos(el)[:, None] * torch.cos(a), torch.cos(el)[:, None] * torch.sin(a),
                     torch.sin(el)[:, None].expand(rings, az)], -1).reshape(-1, 3)
    n = d.shape[0]
    out = []
    for f in range(count):
        yaw, px = 0.02 * f, 0.4 * f
        o = torch.tensor([px, 0.0, 1.0], device="cuda") + torch.tensor([0.0, 0.0, 1.0], device="cuda") * h[
            512 + int(px * 4), 512]
        c, s = math.cos(yaw), math.sin(yaw)
        R = torch.tensor([[c, -s, 0.0], [s, c, 0.0], [0.0, 0.0, 1.0]], device="cuda", dtype=torch.float64)
        w = d @ R.float().T
        hit = torch.full((n,), float("nan"), device="cuda")
        t_prev = 1.0
        for k in range(1, 121):
            t = 1.0 * 100.0 ** (k / 120.0)
            p = o + t * w
            below = (p[:, 2] <= _height(h, p[:, 0], p[:, 1])) & hit.isnan()
            u = torch.rand(n, device="cuda", generator=gen)
            hit = torch.where(below, t_prev + u * (t - t_prev), hit)
            t_prev = t
        far = 50.0 + 50.0 * torch.rand(n, device="cuda", generator=gen)
        hit = torch.where(hit.isnan(), far, hit) + 0.02 * torch.randn(n, device="cuda", generator=gen)
        # a fixed share of the returns is dropped, at random
        order = torch.randperm(n, device="cuda", generator=gen)
        keep = torch.ones(n, dtype=torch.bool, device="cuda")
        keep[order[:int(n * case["dropout"])]] = False
        rel = hit.clamp(1.0, 100.0)[:, None].double() * d.double()   # sensor frame
        T = torch.eye(4, dtype=torch.float64, device="cuda")
        T[:3, :3], T[:3, 3] = R, o.double()
        if case["transform"] == "none":
            rel = rel @ R.T + o.double()
        rel = rel if case["f64"] else rel.float()
        tdt = torch.float64 if case["transform"] == "f64" else torch.float32
        rows = torch.where(keep[:, None], rel, torch.full_like(rel, float("nan")))
        out.append(SimpleNamespace(points=rel[keep].contiguous(), ego=o.double().cpu().numpy(), rows=rows,
                                   T=None if case["transform"] == "none" else T.to(tdt).cpu().numpy(), yaw=yaw))
    return out


# ---- states -----------------------------------------------------------------------------------------------------

def _mapper(case):
    import gvom
    return gvom.Gvom(XY_RES, Z_RES, case["xy"], case["z"], case["buffer"], MIN_DISTANCE, 0.5, 0.5, 0.3, 2.0, 4.0,
                     1.0, case["ex"], case["ez"])


class _DeviceMap:
    """One of a mapper's device maps; a tensor made from it keeps the mapper alive."""

    def __init__(self, owner, ptr, xy, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=(xy, xy), typestr=typestr, version=2)


def _device_maps(g):
    """The mapper's four device maps as tensors (gvom_device_maps)."""
    import ctypes
    import gvom_native as nat
    p = [ctypes.c_void_p() for _ in range(4)]
    nat.check(nat.load().gvom_device_maps(g._h, *[ctypes.byref(v) for v in p]), g._h)
    names = ("positive", "negative", "roughness", "visibility")
    types = ("<i4", "<i4", "<f8", "<i4")
    return {k: torch.as_tensor(_DeviceMap(g, v.value, g.xy_size, t), device="cuda")
            for k, v, t in zip(names, p, types)}


def _quaternion(yaw):
    return (0.0, 0.0, math.sin(yaw / 2), math.cos(yaw / 2))


def _message(case, s):
    """The scan as an organised PointCloud2: rows of `az` points, x y z intensity as float32, NaN where no return."""
    rows = torch.cat([s.rows, torch.zeros(s.rows.shape[0], 1, device="cuda")], 1)
    fields = [SimpleNamespace(name=k, offset=4 * i, datatype=7) for i, k in enumerate(("x", "y", "z", "intensity"))]
    return SimpleNamespace(height=case["rings"], width=case["az"], point_step=16, row_step=16 * case["az"],
                           is_bigendian=False, fields=fields, data=rows.cpu().numpy().tobytes())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "loss":
        from gvom_torch import MapLoss
        s = _scans(case, seed, 1)[0]
        loss = MapLoss(XY_RES, Z_RES, case["xy"], case["z"], MIN_DISTANCE, case["ex"], case["ez"], W_HEIGHT)
        pts = s.points.requires_grad_(True)
        xi = torch.zeros(6, dtype=torch.float64, requires_grad=True)
        return SimpleNamespace(kind=kind, loss=loss, points=pts, xi=xi, T=s.T, ego=s.ego)
    per = case["batch"] if kind == "batch" else 1
    count = case["frames"] if kind == "graph" else 4
    scans = _scans(case, seed, count * per)
    st = SimpleNamespace(kind=kind, k=0, count=count, case=case, graph=None)
    n_max = max(s.points.shape[0] for s in scans)
    if kind == "node":
        from gvom_node import GvomNode
        st.node = GvomNode(xy_resolution=XY_RES, z_resolution=Z_RES, width=case["xy"], height=case["z"],
                           buffer_size=case["buffer"], xy_eigen_dist=case["ex"], z_eigen_dist=case["ez"])
        st.steps = [(_message(case, s), tuple(s.ego), _quaternion(s.yaw)) for s in scans]
    else:
        g = st.g = _mapper(case)
        if kind == "host":
            st.steps = [(s.points.cpu().numpy(), tuple(s.ego), s.T) for s in scans]
        else:
            st.steps = []
            for b in range(count):
                group = scans[b * per:(b + 1) * per]
                off = np.cumsum([0] + [s.points.shape[0] for s in group]).astype(np.int64)
                T = None if group[0].T is None else np.stack([s.T for s in group])
                st.steps.append((torch.cat([s.points for s in group]), off, np.stack([s.ego for s in group]), T))
            g.reserve(n_max, max(p[1][-1] for p in st.steps))
            g.set_overlap(case["overlap"])
            if case["ring_hint"]:
                g.set_ray_rings(case["az"], 64 if case["rings"] >= 64 else 16)
                g.set_raycast_config(256, 1, False, False, False, False)
            st.maps = _device_maps(g)
            torch.cuda.synchronize()   # the points are complete before the library reads them
    # the ring is full and a previous combined map exists, as after the first second of driving
    fill = SimpleNamespace(**{**vars(st), "kind": "device" if kind == "graph" else kind})
    for _ in range(max(2, -(-case["buffer"] // per))):
        run(fill)
    if kind == "graph":
        g.graph_begin(count)
        for p, off, ego, T in st.steps:
            g.process_pointcloud_device(p.data_ptr(), int(off[-1]), ego[0], None if T is None else T[0], _np(p))
            g.combine_maps_device()
        st.graph = g.graph_end()
        st.egos = np.concatenate([q[2] for q in st.steps])
        st.Ts = None if scans[0].T is None else np.concatenate([q[3] for q in st.steps])
    return st


def _np(t):
    return np.float64 if t.dtype == torch.float64 else np.float32


def run(state):
    if state.kind == "loss":
        from gvom_torch import map_loss
        loss = map_loss(state.points, state.xi, state.T, state.ego, state.loss)
        g_points, g_xi = torch.autograd.grad(loss, (state.points, state.xi))
        return {"loss": loss.detach(), "grad_points": g_points, "grad_xi": g_xi}
    if state.kind == "graph":
        state.graph.launch(state.egos, state.Ts)
        return state.maps
    step = state.steps[state.k % state.count]
    state.k += 1
    if state.kind == "host":
        state.g.Process_pointcloud(*step)
        origin, pos, neg, rough, vis = state.g.combine_maps()
        return {"origin": origin, "positive": pos, "negative": neg, "roughness": rough, "visibility": vis}
    if state.kind == "node":
        message, ego, quat = step
        state.node.cb_odom(ego)
        state.node.cb_lidar(message, ego, quat)
        out = state.node.cb_timer(debug=state.case["debug"])
        # the voxel cloud is made too; its rows are as many as the map has cells
        clouds = {k: {n: v[n] for n in v.dtype.names} for k, v in out.debug.items() if k != "voxel"}
        return {"grids": out.grids, "origin": out.info.origin_position, "clouds": clouds}
    points, off, ego, T = step
    if state.kind == "batch":
        state.g.process_batch_device(points.data_ptr(), off, ego, T, _np(points))
    else:
        state.g.process_pointcloud_device(points.data_ptr(), int(off[-1]), ego[0], None if T is None else T[0],
                                          _np(points))
    state.g.combine_maps_device()
    return state.maps


# ---- what a pass cannot do without ----------------------------------------------------------------------------

def work(case):
    n = case["rings"] * case["az"] * (1.0 - case["dropout"])
    v, x = float(_voxels(case)), float(case["xy"] ** 2)
    per_point = 24.0 if case["f64"] else 12.0
    if case["kind"] == "loss":
        # points read, gradients written; per point 27 neighbour voxels' terms each way
        return {"bytes": 48.0 * n + 200.0, "flops": 27 * 60.0 * n}
    if case["kind"] == "node":
        per_point = 16.0 / (1.0 - case["dropout"])
    scans = case["batch"] if case["kind"] == "batch" else 1
    # a ray visits about a third of the map's side and a step is about 12 operations
    steps = n * case["xy"] / 3.0
    scan = {"bytes": per_point * n + 4 * v, "flops": 12 * steps}
    # the combine reads the ring's tables and the previous map and writes the new map and the four 2D maps
    combine = {"bytes": 4 * v * (case["buffer"] + 2) + 20 * x, "flops": 2 * v * (case["buffer"] + 1)}
    if case["kind"] == "node" and case["debug"]:
        combine["bytes"] += 40 * x
    return {k: case["frames"] * (scans * scan[k] + combine[k]) for k in scan}


# ---- 64-bit values ----------------------------------------------------------------------------------------------

def exact(case, seed):
    """The loss and its gradients in plain float64 torch.  The maps' only computed numbers are the roughness
    (the logarithm of a plane fit's residual, zero but for rounding wherever the ground is a plane or three cells
    are known: no such value) and the debug clouds' columns (decided voxel by voxel by the whole map's history)."""
    if case["kind"] != "loss":
        return None
    s = _scans(case, seed, 1)[0]
    xy, z, ex, ez = case["xy"], case["z"], case["ex"], case["ez"]
    T = torch.as_tensor(s.T, device="cuda")
    p = s.points
    w = (p @ T[:3, :3].T + T[:3, 3]).detach().requires_grad_(True)
    res = torch.tensor([XY_RES, XY_RES, Z_RES], dtype=torch.float64, device="cuda")
    size = torch.tensor([xy, xy, z], dtype=torch.float64, device="cuda")
    origin = torch.floor(torch.as_tensor(s.ego, device="cuda") / res - size / 2)
    q = w / res - origin
    own = torch.floor(q.detach()).long()
    far = (w.detach() ** 2).sum(1) >= MIN_DISTANCE ** 2
    lim, rad = size.long(), torch.tensor([ex, ex, ez], device="cuda")
    inside = far & ((own >= 0) & (own < lim)).all(1)
    near = far & ((own >= -rad) & (own < lim + rad)).all(1)
    voxels, cell = torch.unique((own[:, 0] * xy + own[:, 1])[inside] * z + own[inside, 2], return_inverse=True)
    table = torch.full((xy * xy * z,), -1, dtype=torch.long, device="cuda")
    table[voxels] = torch.arange(voxels.numel(), device="cuda")
    pt, vox, loc = [], [], []
    idx = torch.nonzero(near)[:, 0]
    for dx in range(-ex, ex + 1):
        for dy in range(-ex, ex + 1):
            for dz in range(-ez, ez + 1):
                u = own[idx] + torch.tensor([dx, dy, dz], device="cuda")
                ok = ((u >= 0) & (u < lim)).all(1)
                uu = u[ok]
                t = table[(uu[:, 0] * xy + uu[:, 1]) * z + uu[:, 2]]
                pt.append(idx[ok][t >= 0])
                vox.append(t[t >= 0])
                loc.append(uu[t >= 0])
    pt, vox, loc = torch.cat(pt), torch.cat(vox), torch.cat(loc)
    C = voxels.numel()
    r = q[pt] - loc
    cnt = torch.zeros(C, dtype=torch.float64, device="cuda").index_add_(0, vox, torch.ones_like(r[:, 0]))
    mean = torch.zeros(C, 3, dtype=torch.float64, device="cuda").index_add(0, vox, r) / cnt[:, None]
    e = r - mean[vox]
    cov = torch.zeros(C, 9, dtype=torch.float64, device="cuda").index_add(
        0, vox, (e[:, :, None] * e[:, None, :]).reshape(-1, 9)) / cnt[:, None]
    cov = cov.reshape(C, 3, 3)
    # lambda_min = v' C v with its unit eigenvector held (its own derivative drops out of the gradient)
    vec = torch.linalg.eigh(cov.detach().cpu())[1][:, :, 0].to(cov.device)
    rough = torch.einsum("ni,nij,nj->", vec, cov, vec)
    # the height of a column is that of its lowest point (of the lowest occupied voxel, which holds it)
    col = (own[:, 0] * xy + own[:, 1])[inside]
    zs = w[inside, 2]
    low = torch.full((xy * xy,), float("inf"), dtype=torch.float64, device="cuda")
    low = low.scatter_reduce(0, col, zs.detach(), "amin")
    is_low = zs.detach() == low[col]
    hs = zs[is_low]
    loss = rough + W_HEIGHT * ((hs - hs.mean()) ** 2).mean()
    gw, = torch.autograd.grad(loss, w)
    wd = w.detach()
    g_xi = torch.cat([gw.sum(0), torch.linalg.cross(wd, gw).sum(0)])
    return {"loss": loss.detach(), "grad_points": gw @ T[:3, :3], "grad_xi": g_xi.cpu()}
