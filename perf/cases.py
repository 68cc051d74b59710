"""The work a reconstruction program asks of this package, as measurable cases.

The package serves the frame loop of dynamic reconstruction: a depth frame is
filtered and back-projected (ingest), the motion graph is fitted to it (icp),
the frame is integrated into the volume through the warp (frame, batch,
dropin; plain for the first frame), and the surface is extracted (mesh) and
warped (points).  Each case is one such call with the sizes of the package's
own workloads (volumefusion_amd/scenes.py, tests, bench.py) or generic odd ones.

Kinds:
  frame   vf_warped_integrate of one frame (LBS or dual-quaternion blend)
  batch   one recorded plan over many volumes of mixed sizes
  dropin  the reference's nine separate calls on its own buffers
  plain   the first frame's integration, without a warp
  ingest  depth filter, bilateral filter, vertices, normals, centroid
  points  knn, weights and blend of free points (the extracted mesh)
  mesh    marching cubes into device buffers, or to host arrays
  icp     one ICP iteration: solver creation, five Gauss-Newton steps

Scenes are two intersecting ellipsoids seen by one pinhole camera, with depth
noise and dropout, nodes spread over the surfaces in random order, and a
smooth field of small rigid motions.  Everything follows from the seed.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from volumefusion_amd import _lib as L
from volumefusion_amd import ops
from volumefusion_amd.device import DeviceArray

DEV = "cuda"
F32, F64 = torch.float32, torch.float64
DELTA, MAX_WEIGHT = 0.012, 64.0
IDENTITY3 = (1.0, 0.0, 0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 1.0)


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # a coarse preview volume: the smallest frame, where launches count
        dict(name="frame_preview", kind="frame", x=72, y=60, z=84, voxel=0.005, nodes=160, k=4, width=320, height=288,
             blend="lbs", brick=0),
        # one object at 3 mm with a 640x576 sensor, dims off every brick size
        dict(name="frame_250", kind="frame", x=250, y=262, z=246, voxel=0.003, nodes=2048, k=8, width=640, height=576,
             blend="lbs", brick=0),
        # the large volume: 512^3 at 2 mm, 4096 nodes, a megapixel frame, the
        # brick shape that tuning picks for it
        dict(name="frame_512", kind="frame", x=512, y=512, z=512, voxel=0.002, nodes=4096, k=8, width=1024,
             height=1024, blend="lbs", brick=2),
        # dual-quaternion blending, the option for strong rotations
        dict(name="frame_dqb", kind="frame", x=192, y=200, z=180, voxel=0.004, nodes=1200, k=6, width=640, height=576,
             blend="dqb", brick=0),
        # many reconstructions on one device: 16 volumes of mixed resolution
        dict(name="batch_16", kind="batch", count=16, lo=64, hi=384, nodes_lo=128, nodes_hi=4096, k=8, width=640,
             height=576),
        # a program that keeps the reference's call sequence and buffers
        dict(name="dropin_k4", kind="dropin", x=160, y=144, z=168, voxel=0.004, nodes=900, k=4, width=640, height=576),
        # the first frame into an empty large volume, rows off the wave size
        dict(name="plain_500", kind="plain", x=500, y=480, z=512, voxel=0.002, width=1024, height=1024, camera=False),
        # every frame starts with its ingest: a megapixel depth frame
        dict(name="ingest_1024", kind="ingest", width=1024, height=1024, radius=5),
        # the extracted mesh through the motion graph, each frame
        dict(name="points_900k", kind="points", points=900001, nodes=4096, k=8, blend="lbs"),
        # the large volume's surface for the next step on the device
        dict(name="mesh_512", kind="mesh", x=512, y=512, z=512, voxel=0.002, width=1024, height=1024, faces=True,
             host=False),
        # a preview mesh for the program's own use on the host
        dict(name="mesh_host_128", kind="mesh", x=128, y=126, z=131, voxel=0.005, width=320, height=288, faces=False,
             host=True),
        # the motion fit of a large graph
        dict(name="icp_4096", kind="icp", nodes=4096, points=300000, k=6, reg_k=4, iterations=5),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["frame", "frame", "batch", "dropin", "plain", "ingest", "points", "mesh", "icp"])
    sensor = rng.choice([(320, 288), (640, 576), (640, 480), (1024, 1024), (513, 431)])
    w, h = sensor
    if kind == "icp":
        return dict(kind=kind, nodes=_log(rng, 60, 3600), points=_log(rng, 4000, 250000), k=rng.choice([4, 6, 8]),
                    reg_k=rng.choice([4, 6]), iterations=rng.randint(2, 6))
    if kind == "points":
        return dict(kind=kind, points=_log(rng, 900, 900000), nodes=_log(rng, 40, 4096), k=rng.choice([4, 6, 8]),
                    blend=rng.choice(["lbs", "lbs", "dqb"]))
    if kind == "ingest":
        return dict(kind=kind, width=w - rng.randint(0, 9), height=h - rng.randint(0, 9), radius=rng.choice([3, 5, 7]))
    if kind == "batch":
        lo = _log(rng, 48, 128)
        return dict(kind=kind, count=rng.randint(2, 20), lo=lo, hi=_log(rng, lo + 16, 352), nodes_lo=100,
                    nodes_hi=_log(rng, 400, 4000), k=rng.choice([4, 8]), width=640, height=576)
    side = _log(rng, 56, 176 if kind == "dropin" else 480)
    x, y, z = (max(40, side + rng.randint(-side // 10, side // 12)) for _ in range(3))
    voxel = round(rng.uniform(0.5, 1.0) / side, 5)
    base = dict(kind=kind, x=x, y=y, z=z, voxel=voxel, width=w, height=h)
    if kind == "plain":
        return dict(base, camera=rng.random() < 0.5)
    if kind == "mesh":
        host = side <= 136 and rng.random() < 0.5
        return dict(base, faces=rng.random() < 0.7, host=host)
    nodes = _log(rng, 100, 200 + side * 8)
    if kind == "dropin":
        return dict(base, nodes=nodes, k=rng.choice([4, 6, 8]))
    return dict(base, nodes=nodes, k=rng.choice([4, 6, 8]), blend=rng.choice(["lbs", "lbs", "lbs", "dqb"]),
                brick=rng.choice([0, 0, 2]))


# ---------------------------------------------------------------------------
# Scenes
# ---------------------------------------------------------------------------

def _rotation(rng) -> np.ndarray:
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]])


def _t(a, dtype=F64) -> torch.Tensor:
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


class Scene:
    """Two ellipsoids inside a box of edge e around (0, 0, zc)."""

    def __init__(self, seed: int, e: float, salt: int = 0):
        self.rng = np.random.default_rng([seed, salt])
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(int(self.rng.integers(1 << 40)))
        rng = self.rng
        self.e, self.zc = e, max(0.5, e)
        c = np.array([0.0, 0.0, self.zc])
        self.parts = [(c + e * np.array([-0.09, rng.uniform(-0.03, 0.03), 0.0]), e * rng.uniform(0.19, 0.30, 3),
                       _rotation(rng)),
                      (c + e * np.array([0.12, rng.uniform(0.0, 0.06), 0.05]), e * rng.uniform(0.18, 0.27, 3),
                       _rotation(rng))]

    def area(self) -> float:
        p = 1.6075
        return sum(4 * math.pi * (((a * b) ** p + (a * c) ** p + (b * c) ** p) / 3) ** (1 / p)
                   for _, (a, b, c), _ in self.parts)

    def uniform(self, *shape) -> torch.Tensor:
        return torch.rand(*shape, generator=self.gen, device=DEV, dtype=F64)

    def normal(self, *shape) -> torch.Tensor:
        return torch.randn(*shape, generator=self.gen, device=DEV, dtype=F64)

    def camera(self, width: int, height: int) -> tuple:
        """Column-major intrinsics."""
        f = float(np.float32(0.85 * min(width, height) / 0.9))
        return (f, 0.0, 0.0, 0.0, f, 0.0, float(np.float32(width / 2)), float(np.float32(height / 2)), 1.0)

    def depth(self, width: int, height: int) -> torch.Tensor:
        """A frame [height, width]: the nearest surface's z, 0 where there is
        none, 1.5 mm noise, 5 % dropout."""
        K = self.camera(width, height)
        u = (torch.arange(width, device=DEV, dtype=F64) - K[6]) / K[0]
        v = (torch.arange(height, device=DEV, dtype=F64) - K[7]) / K[4]
        d = torch.stack([u[None, :].expand(height, width), v[:, None].expand(height, width),
                         torch.ones(height, width, device=DEV, dtype=F64)], -1)
        best = torch.full((height, width), math.inf, device=DEV, dtype=F64)
        for c, axes, R in self.parts:
            M = _t(R / axes[None, :])  # row vector times M: body coordinates over the axes
            a, b = d @ M, _t(c) @ M
            A, B = (a * a).sum(-1), (a * b).sum(-1)
            disc = B * B - A * ((b * b).sum() - 1.0)
            t = (B - disc.clamp(min=0).sqrt()) / A
            best = torch.where((disc > 0) & (t > 1e-3), torch.minimum(best, t), best)
        hit = torch.isfinite(best)
        noisy = torch.where(hit, best, torch.zeros_like(best)) + 0.0015 * self.normal(height, width)
        keep = hit & (self.uniform(height, width) > 0.05)
        return torch.where(keep, noisy, torch.zeros_like(noisy)).to(F32)

    def on_surface(self, n: int, even: bool) -> tuple:
        """n points and unit normals over both surfaces: evenly spread with
        some jitter, in random order (nodes), or independent, in the order
        marching cubes visits 2 mm cubes (a mesh)."""
        pts, nrm = [], []
        n0 = max(1, n // 2) if n > 1 else 1
        for (c, axes, R), m in zip(self.parts, (n0, n - n0)):
            if m == 0:
                continue
            if even:
                i = torch.arange(m, device=DEV, dtype=F64) + 0.5
                z, phi = 1.0 - 2.0 * i / m, i * (math.pi * (3.0 - math.sqrt(5.0)))
                r = (1.0 - z * z).clamp(min=0).sqrt()
                u = torch.stack([r * torch.cos(phi), r * torch.sin(phi), z], -1) + 0.6 / math.sqrt(m) * self.normal(m, 3)
            else:
                u = self.normal(m, 3)
            u = u / u.norm(dim=1, keepdim=True)
            pts.append(_t(c) + (u * _t(axes)) @ _t(R).T)
            g = (u / _t(axes)) @ _t(R).T
            nrm.append(g / g.norm(dim=1, keepdim=True))
        p, q = torch.cat(pts), torch.cat(nrm)
        if even:
            order = torch.randperm(n, generator=self.gen, device=DEV)
        else:
            cell = ((p - p.min(0).values) / 0.002).to(torch.int64)
            order = torch.sort((cell[:, 2] * 4096 + cell[:, 1]) * 4096 + cell[:, 0], stable=True).indices
        return p[order], q[order]

    def motions(self, nodes: torch.Tensor, angle_deg: float = 5.0, shift: float = 0.010) -> torch.Tensor:
        """Rigid motions about the nodes from a smooth field: column-major
        float32 [n, 16]."""
        a = 2.0 * self.uniform(2, 3) - 1.0
        B = self.normal(2, 3, 3) * (3.0 / self.e)
        ph = 6.3 * self.uniform(2, 3)
        w = math.radians(angle_deg) * a[0] / a[0].norm() * torch.sin(nodes @ B[0].T + ph[0])
        t = shift * a[1] / a[1].norm() * torch.sin(nodes @ B[1].T + ph[1])
        th = w.norm(dim=1).clamp(min=1e-12)
        k = w / th[:, None]
        z = torch.zeros_like(th)
        K = torch.stack([z, -k[:, 2], k[:, 1], k[:, 2], z, -k[:, 0], -k[:, 1], k[:, 0], z], -1).view(-1, 3, 3)
        eye = torch.eye(3, device=DEV, dtype=F64)
        R = eye + torch.sin(th)[:, None, None] * K + (1 - torch.cos(th))[:, None, None] * (K @ K)
        T = torch.zeros(nodes.shape[0], 4, 4, device=DEV, dtype=F64)
        T[:, :3, :3] = R
        T[:, :3, 3] = nodes + t - (R @ nodes[:, :, None])[:, :, 0]
        T[:, 3, 3] = 1.0
        return T.transpose(1, 2).reshape(-1, 16).to(F32).contiguous()

    def graph(self, n: int) -> tuple:
        """Nodes [n, 3], the common radius, transforms [n, 16]."""
        p, _ = self.on_surface(n, True)
        p = p.to(F32)
        radius = float(np.float32(max(0.020, 0.5 * math.sqrt(self.area() / n))))
        return p, radius, self.motions(p.to(F64))


class Box:
    """A volume's geometry in float32, as DeviceTsdf derives it."""

    def __init__(self, x: int, y: int, z: int, voxel: float, zc: float):
        self.dim = (x, y, z)
        self.size = tuple(float(np.float32(d * voxel)) for d in self.dim)
        self.vs = tuple(float(np.float32(s) / np.float32(d)) for s, d in zip(self.size, self.dim))
        self.center = (0.0, 0.0, float(np.float32(zc)))
        self.n = x * y * z

    def corner(self, i: torch.Tensor, axis: int, dtype) -> torch.Tensor:
        """Voxel positions along an axis, volume frame."""
        half = float(np.float32(self.size[axis]) * np.float32(0.5))
        return i.to(dtype) * torch.tensor(self.vs[axis], dtype=dtype, device=DEV) - half

    def tsdf(self, start: tuple | None = None) -> ops.DeviceTsdf:
        t = ops.DeviceTsdf(self.size, self.dim, center=self.center, delta=DELTA)
        if start is not None:
            view(t.tsdf).copy_(start[0].view(-1))
            view(t.weights).copy_(start[1].view(-1))
        return t


# ---------------------------------------------------------------------------
# Device buffers
# ---------------------------------------------------------------------------

class _Span:
    def __init__(self, d: DeviceArray):
        self.owner = d
        self.__cuda_array_interface__ = {"shape": d.shape, "typestr": d.dtype.str, "data": (d.ptr, False),
                                         "version": 3, "strides": None}


def view(d: DeviceArray) -> torch.Tensor:
    """The buffer's memory as a tensor, which keeps the buffer alive."""
    return torch.as_tensor(_Span(d), device=DEV)


def buffer(shape, dtype=np.float32) -> DeviceArray:
    d = DeviceArray(shape, dtype)
    d.fill(0)
    return d


def on_device(t: torch.Tensor) -> DeviceArray:
    d = DeviceArray(tuple(t.shape), np.float32 if t.dtype == F32 else np.int32)
    view(d).copy_(t)
    return d


# ---------------------------------------------------------------------------
# Reference arithmetic: decisions in float32, values in the asked precision
# ---------------------------------------------------------------------------

def _sample(p, q, depth, K):
    """The projective update of points: p three float32 tensors, q the same
    points in the value precision.  (updated, new sample)."""
    h, w = depth.shape
    zi = 1.0 / p[2]
    px = (((K[0] * p[0]) * zi + K[6]) + 0.5).clamp(-2e9, 2e9).to(torch.int64)
    py = (((K[4] * p[1]) * zi + K[7]) + 0.5).clamp(-2e9, 2e9).to(torch.int64)
    ok = (p[2] >= 1e-4) & (px >= 0) & (px < w) & (py >= 0) & (py < h)
    d = depth.reshape(-1)[torch.where(ok, py * w + px, torch.zeros_like(px))]
    delta = float(np.float32(DELTA))
    s = p[2] - d
    ok = ok & (d >= 1e-4) & ~(s > delta)
    val = (q[2] - d.to(q[2].dtype)) / delta
    return ok, torch.where(s < -delta, torch.full_like(val, -1.0), val)


def _blend(t, w, ok, sample):
    """Running average of the updated voxels."""
    wn = w + 1.0
    return (torch.where(ok, (t * w + sample) / wn, t),
            torch.where(ok, wn.clamp(max=MAX_WEIGHT), w))


def _plain(box: Box, depth, K, dtype, start=None, pose=None, cap=MAX_WEIGHT):
    """The frame integrated without a warp, slab by slab."""
    X, Y, Z = box.dim
    if start is None:
        start = (torch.full((Z, Y, X), -1.0, device=DEV, dtype=dtype), torch.zeros(Z, Y, X, device=DEV, dtype=dtype))
    t, w = start[0].to(dtype).clone(), start[1].to(dtype).clone()
    for z0 in range(0, Z, 64):
        z1 = min(Z, z0 + 64)
        shape = (z1 - z0, Y, X)
        idx = (torch.arange(X, device=DEV).view(1, 1, X), torch.arange(Y, device=DEV).view(1, Y, 1),
               torch.arange(z0, z1, device=DEV).view(-1, 1, 1))

        def points(dt):
            p = [(box.corner(i, a, dt) + box.center[a]).expand(shape) for a, i in enumerate(idx)]
            if pose is not None:
                R, tr = pose
                p = [R[a] * p[0] + (R[3 + a] * p[1] + R[6 + a] * p[2]) + tr[a] for a in range(3)]
            return p

        p = points(F32)
        ok, s = _sample(p, p if dtype == F32 else points(dtype), depth, K)
        wn = w[z0:z1] + 1.0
        t[z0:z1] = torch.where(ok, (t[z0:z1] * w[z0:z1] + s) / wn, t[z0:z1])
        w[z0:z1] = torch.where(ok, wn.clamp(max=cap), w[z0:z1])
    return t, w


def _weight(d, r):
    """exp(-d^2 / 2 r^2), rounded once when d is float32."""
    x = -(d * d) / (2.0 * (r * r))
    return torch.exp(x.to(F64)).to(d.dtype)


def _lbs(T, p, w, idx, voxel_order=True):
    """sum_s w_s (T_s p): T [G, 16], p [n, 3], w [n, K] (0: no slot)."""
    out = [torch.zeros_like(p[:, 0]) for _ in range(3)]
    for s in range(idx.shape[1]):
        M = T[idx[:, s]]
        for a in range(3):
            a0, a1, a2, a3 = M[:, a] * p[:, 0], M[:, 4 + a] * p[:, 1], M[:, 8 + a] * p[:, 2], M[:, 12 + a]
            v = (a0 + (a1 + a2)) + a3 if voxel_order else (a0 + a1) + (a2 + a3)
            out[a] = out[a] + w[:, s] * v
    return torch.stack(out, -1)


def _dual(T):
    """Unit dual quaternions (real, dual) of small rotations."""
    tr = (T[:, 0] + T[:, 5]) + T[:, 10]
    s = (tr + 1.0).sqrt() * 2.0
    q = torch.stack([(T[:, 6] - T[:, 9]) / s, (T[:, 8] - T[:, 2]) / s, (T[:, 1] - T[:, 4]) / s, 0.25 * s], -1)
    q = q / (((q[:, 0] * q[:, 0] + q[:, 1] * q[:, 1]) + q[:, 2] * q[:, 2]) + q[:, 3] * q[:, 3]).sqrt()[:, None]
    x, y, z, w = q.unbind(-1)
    a, b, c = T[:, 12], T[:, 13], T[:, 14]
    d = torch.stack([0.5 * (w * a + (b * z - c * y)), 0.5 * (w * b + (c * x - a * z)),
                     0.5 * (w * c + (a * y - b * x)), 0.5 * -((a * x + b * y) + c * z)], -1)
    return q, d


def _cross(a, b):
    return torch.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1], a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                        a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], -1)


def _dqb(T, p, w, idx):
    """Blend of the slots' dual quaternions, applied to p."""
    qr, qd = _dual(T)
    f = qr[idx[:, 0]]
    br, bd = torch.zeros_like(f), torch.zeros_like(f)
    for s in range(idx.shape[1]):
        r, d = qr[idx[:, s]], qd[idx[:, s]]
        dot = ((r[:, 0] * f[:, 0] + r[:, 1] * f[:, 1]) + r[:, 2] * f[:, 2]) + r[:, 3] * f[:, 3]
        ws = torch.where(dot < 0, -w[:, s], w[:, s])[:, None]
        br, bd = br + ws * r, bd + ws * d
    il = 1.0 / (((br[:, 0] * br[:, 0] + br[:, 1] * br[:, 1]) + br[:, 2] * br[:, 2]) + br[:, 3] * br[:, 3]).sqrt()
    br, bd = br * il[:, None], bd * il[:, None]
    rv, dv = br[:, :3], bd[:, :3]
    turn = _cross(rv, _cross(rv, p) + br[:, 3:] * p)
    shift = 2.0 * ((br[:, 3:] * dv - bd[:, 3:] * rv) + _cross(rv, dv))
    return (p + 2.0 * turn) + shift


def _cube(radius: float, vs) -> tuple:
    return tuple(2 * (int(np.float32(radius) / np.float32(v)) + 1) + 1 for v in vs)


def _candidates(box: Box, nodes, radius: float, cube, k: int):
    """Each supported voxel's k nearest candidate nodes (cube and dist <= 2r),
    in (distance, index) order: voxel [S], node [S, k], slots used [S, k]."""
    X, Y, Z = box.dim
    m = nodes - torch.tensor(box.center, device=DEV)
    half = torch.tensor([np.float32(s) * np.float32(0.5) for s in box.size], device=DEV)
    inv = torch.tensor([np.float32(1.0 / float(v)) for v in box.vs], device=DEV)
    lo = ((m + half) * inv).to(torch.int64) - torch.tensor([(c - 1) // 2 for c in cube], device=DEV)
    off = torch.cartesian_prod(*(torch.arange(c, device=DEV) for c in cube))
    vox, dist, node = [], [], []
    step = max(1, 8_000_000 // off.shape[0])
    for g in range(0, nodes.shape[0], step):
        v = lo[g:g + step, None, :] + off[None]
        ok = ((v >= 0) & (v < torch.tensor(box.dim, device=DEV))).all(-1)
        d = [box.corner(v[..., a], a, F32) - m[g:g + step, None, a] for a in range(3)]
        r = (d[0] * d[0] + (d[1] * d[1] + d[2] * d[2])).sqrt()
        ok = ok & ~(r > float(np.float32(radius) * np.float32(2.0)))
        i = ok.nonzero(as_tuple=True)
        v = v[i]
        vox.append((v[:, 2] * Y + v[:, 1]) * X + v[:, 0])
        dist.append(r[i])
        node.append(i[0] + g)
    vox, dist, node = torch.cat(vox), torch.cat(dist), torch.cat(node)
    order = torch.sort((dist.view(torch.int32).to(torch.int64) << 32) | node).indices
    order = order[torch.sort(vox[order], stable=True).indices]
    vox, node = vox[order], node[order]
    uniq, count = torch.unique_consecutive(vox, return_counts=True)
    first = count.cumsum(0) - count
    s = torch.arange(k, device=DEV)[None, :]
    used = s < count[:, None]
    return uniq, node[(first[:, None] + torch.where(used, s, torch.zeros_like(s)))], used


def _warp(box: Box, vox, idx, used, nodes, radius, T, blend, dtype):
    """Warped camera-frame positions of the supported voxels."""
    X, Y, _ = box.dim
    p = torch.stack([box.corner(vox % X, 0, dtype), box.corner((vox // X) % Y, 1, dtype),
                     box.corner(vox // (X * Y), 2, dtype)], -1)
    c = torch.tensor(box.center, device=DEV, dtype=dtype)
    m = nodes.to(dtype) - c
    w = torch.zeros(idx.shape, device=DEV, dtype=dtype)
    total = torch.zeros(idx.shape[0], device=DEV, dtype=dtype)
    for s in range(idx.shape[1]):
        d = p - m[idx[:, s]]
        r = (d[:, 0] * d[:, 0] + (d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])).sqrt()
        w[:, s] = torch.where(used[:, s], _weight(r, torch.tensor(radius, device=DEV, dtype=dtype)), w[:, s])
        total = total + w[:, s]
    w = w / total[:, None]
    blend_fn = _dqb if blend == "dqb" else _lbs
    return blend_fn(T.to(dtype), p + c, w, idx)


def _warped_frame(box: Box, nodes, radius, T, depth, K, k, blend, start):
    """One warped frame in binary64 (decisions as in float32): tsdf, weight,
    the supported voxels, their warped positions, the collision counts."""
    X, Y, Z = box.dim
    vox, idx, used = _candidates(box, nodes, radius, _cube(radius, box.vs), k)
    n = box.n
    count = torch.zeros(n, device=DEV, dtype=torch.int32)
    target, fine = torch.empty_like(vox), torch.empty(vox.shape[0], 3, device=DEV, dtype=F64)
    coarse = torch.empty(vox.shape[0], 3, device=DEV, dtype=F32)
    for i in range(0, vox.shape[0], 1 << 20):
        j = slice(i, i + (1 << 20))
        p = _warp(box, vox[j], idx[j], used[j], nodes, radius, T, blend, F32)
        u = []
        for a in range(3):
            half = float(np.float32(box.size[a]) * np.float32(0.5))
            u.append((((p[:, a] - box.center[a]) + half) * float(np.float32(1.0 / float(box.vs[a])))).to(torch.int64))
        inside = torch.stack([(u[a] >= 0) & (u[a] < box.dim[a]) for a in range(3)]).all(0)
        target[j] = torch.where(inside, (u[2] * Y + u[1]) * X + u[0], torch.full_like(u[0], -1))
        coarse[j] = p
        fine[j] = _warp(box, vox[j], idx[j], used[j], nodes, radius, T, blend, F64)
    hit = target[target >= 0]
    count.index_add_(0, hit, torch.ones_like(hit, dtype=torch.int32))
    ok, s = _sample(list(coarse.unbind(-1)), list(fine.unbind(-1)), depth, K)
    ok = ok & (target >= 0) & (count[target.clamp(min=0)] <= 1)
    t, w = start[0].reshape(-1).to(F64).clone(), start[1].reshape(-1).to(F64).clone()
    v = vox[ok]
    t[v], w[v] = _blend(t[v], w[v], torch.ones_like(v, dtype=torch.bool), s[ok])
    return t, w, vox, fine, count


def _nearest(points, nodes, k: int, skip_self: bool = False):
    """The k nearest nodes by (float32 distance, index), chunked brute force."""
    out_d, out_i = [], []
    kk = min(k + (1 if skip_self else 0), nodes.shape[0])
    for i in range(0, points.shape[0], 8192):
        p = points[i:i + 8192]
        d = [p[:, None, a] - nodes[None, :, a] for a in range(3)]
        r = ((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]).sqrt()
        key = (r.view(torch.int32).to(torch.int64) << 32) | torch.arange(nodes.shape[0], device=DEV)[None]
        best = torch.topk(key, kk, dim=1, largest=False, sorted=True).values[:, kk - min(k, kk):]
        out_d.append((best >> 32).to(torch.int32).view(F32))
        out_i.append(best & 0xFFFFFFFF)
    return torch.cat(out_d), torch.cat(out_i)


# ---------------------------------------------------------------------------
# Inputs of each kind
# ---------------------------------------------------------------------------

def _frame_inputs(case, seed, salt=0):
    box = Box(case["x"], case["y"], case["z"], case["voxel"], 0.0)
    sc = Scene(seed, min(box.size), salt)
    box = Box(case["x"], case["y"], case["z"], case["voxel"], sc.zc)
    nodes, radius, T = sc.graph(case["nodes"])
    w, h = case["width"], case["height"]
    K = sc.camera(w, h)
    first, depth = sc.depth(w, h), sc.depth(w, h)
    return box, nodes, radius, T, K, depth, _plain(box, first, K, F32)


def _batch_cases(case):
    # sizes belong to the case, contents to the seed
    rng = np.random.default_rng([77, case["count"], case["lo"], case["hi"]])
    out = []
    for i in range(case["count"]):
        f = i / max(1, case["count"] - 1)
        d = int(round(case["lo"] * (case["hi"] / case["lo"]) ** f))
        g = int(round(case["nodes_lo"] * (case["nodes_hi"] / case["nodes_lo"]) ** f * rng.uniform(0.8, 1.0)))
        x, y, z = (max(40, d - int(rng.integers(0, 6))) for _ in range(3))
        out.append(dict(x=x, y=y, z=z, voxel=0.8 / d, nodes=g, width=case["width"], height=case["height"]))
    return out


def _points_inputs(case, seed):
    sc = Scene(seed, 1.0)
    nodes, radius, T = sc.graph(case["nodes"])
    p, q = sc.on_surface(case["points"], False)
    return nodes, radius, T, (p + 0.002 * sc.normal(case["points"], 1) * q).to(F32)


def _mesh_room(box: Box) -> int:
    """Vertices that a dozen sheets through the box may have."""
    return 16 * max(box.dim[a] * box.dim[b] for a, b in ((0, 1), (1, 2), (0, 2)))


def _mesh_inputs(case, seed):
    box = Box(case["x"], case["y"], case["z"], case["voxel"], 0.0)
    sc = Scene(seed, min(box.size))
    box = Box(case["x"], case["y"], case["z"], case["voxel"], sc.zc)
    K = sc.camera(case["width"], case["height"])
    v = None
    for _ in range(2):
        v = _plain(box, sc.depth(case["width"], case["height"]), K, F32, v)
    return box, v


def _icp_inputs(case, seed):
    sc = Scene(seed, 1.0)
    G, M, k = case["nodes"], case["points"], min(case["k"], case["nodes"])
    nodes = sc.on_surface(G, True)[0].to(F32)
    canon, normals = (t.to(F32) for t in sc.on_surface(M, False))
    radius = 3.0 * math.sqrt(sc.area() / G)
    d, idx = _nearest(canon, nodes, k)
    w = torch.where(d < radius, torch.exp(-(d * d) / (2 * radius * radius)), torch.zeros_like(d))
    w = w / w.sum(1, keepdim=True).clamp(min=1e-20)
    gknn = _nearest(nodes, nodes, case["reg_k"], skip_self=True)[1]
    gknn = torch.cat([gknn, torch.full((G, case["reg_k"] - gknn.shape[1]), -1, device=DEV, dtype=gknn.dtype)], 1)
    T = sc.motions(nodes.to(F64), 2.0, 0.004)
    target = _lbs(T.to(F64), canon.to(F64), w.to(F64), idx, False) + 0.0005 * sc.normal(M, 3)
    seen = (sc.uniform(M) < 0.9).nonzero()[:, 0]
    corr = torch.stack([seen, seen], 1).to(torch.int32).contiguous()
    eye = torch.eye(4, device=DEV, dtype=F32).reshape(1, 16).repeat(G, 1)
    return dict(corr=corr, canon=canon, knn=idx.to(torch.int32), kw=w.to(F32).contiguous(), normals=normals,
                graph=nodes, gknn=gknn.to(torch.int32).contiguous(), target=target.to(F32).contiguous(), T0=eye, k=k)


def _pose(seed):
    a, b = np.random.default_rng([seed, 5]).uniform(0.01, 0.05, 2)
    Ry = np.array([[math.cos(a), 0, math.sin(a)], [0, 1, 0], [-math.sin(a), 0, math.cos(a)]])
    Rx = np.array([[1, 0, 0], [0, math.cos(b), -math.sin(b)], [0, math.sin(b), math.cos(b)]])
    R = (Ry @ Rx).T.reshape(9).astype(np.float32)
    return tuple(float(v) for v in R), tuple(float(np.float32(v)) for v in (0.01, -0.006, 0.004))


def _plain_inputs(case, seed):
    box = Box(case["x"], case["y"], case["z"], case["voxel"], 0.0)
    sc = Scene(seed, min(box.size))
    box = Box(case["x"], case["y"], case["z"], case["voxel"], sc.zc)
    return box, sc.camera(case["width"], case["height"]), sc.depth(case["width"], case["height"])


def _graph_object(nodes, radius, T) -> ops.DeviceMotionGraph:
    return ops.DeviceMotionGraph(nodes.cpu().numpy(), T.cpu().numpy(), np.full(nodes.shape[0], radius, np.float32))


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

def prepare(case: dict, seed: int):
    return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def _prepare_frame(case, seed):
    box, nodes, radius, T, K, depth, start = _frame_inputs(case, seed)
    tsdf = box.tsdf(start)
    graph = _graph_object(nodes, radius, T)
    ws = ops.Workspace()
    if case["brick"]:
        ws.set_tuning(case["brick"], 0)
    return dict(ws=ws, tsdf=tsdf, graph=graph, depth=on_device(depth), K=K, k=case["k"],
                cube=_cube(radius, box.vs), blend=L.BLEND_DQB if case["blend"] == "dqb" else L.BLEND_LBS,
                out={"tsdf": view(tsdf.tsdf), "weights": view(tsdf.weights), "nodes": view(graph.points)})


def _run_frame(s):
    ops.warped_integrate(s["ws"], s["tsdf"], s["graph"], s["depth"], s["K"], s["k"], DELTA, MAX_WEIGHT, s["cube"],
                         blend=s["blend"])
    return s["out"]


def _prepare_batch(case, seed):
    tsdfs, graphs, depths, Ks, cubes = [], [], [], [], []
    for i, c in enumerate(_batch_cases(case)):
        box, nodes, radius, T, K, depth, start = _frame_inputs(c, seed, 100 + i)
        tsdfs.append(box.tsdf(start))
        graphs.append(_graph_object(nodes, radius, T))
        depths.append(on_device(depth))
        Ks.append(K)
        cubes.append(_cube(radius, box.vs))
    plan = ops.Plan(tsdfs, graphs, depths, Ks, case["k"], DELTA, MAX_WEIGHT, cubes, graph=True)
    return dict(plan=plan, out={"tsdf": [view(t.tsdf) for t in tsdfs], "weights": [view(t.weights) for t in tsdfs],
                                "nodes": [view(g.points) for g in graphs]})


def _run_batch(s):
    s["plan"].launch()
    return s["out"]


def _prepare_dropin(case, seed):
    box, nodes, radius, T, K, depth, start = _frame_inputs(case, seed)
    n, k = box.n, case["k"]
    tsdf = box.tsdf(start)
    s = dict(box=box, tsdf=tsdf, graph=_graph_object(nodes, radius, T), depth=on_device(depth), K=K,
             cube=_cube(radius, box.vs), size=(case["width"], case["height"]), idx=buffer((n, k), np.int32),
             dist=buffer((n, k)), w=buffer((n, k)), cnt=buffer((n,), np.int32), col=buffer((n,), np.int32),
             verts=buffer((n, 3)))
    s["out"] = {"tsdf": view(tsdf.tsdf), "weights": view(tsdf.weights), "vertices": view(s["verts"]),
                "counts": view(s["col"])}
    return s


def _run_dropin(s):
    # the reference's frame loop, its buffers cleared as it clears them
    t, g, box = s["tsdf"], s["graph"], s["box"]
    c, vs, n = t.center, t.voxel_size(), box.n
    s["cnt"].fill(0)
    s["col"].fill(0)
    ops.run_translate_kernel(g.points, g.count, tuple(-v for v in c))
    ops.run_tsdf_knn_graph(s["idx"], s["dist"], s["cnt"], g.points, g.radii, g.count, vs, box.size, box.dim, s["cube"])
    ops.run_compute_tsdf_warp_weights_kernel(s["w"], g.radii, s["idx"], s["dist"], s["cnt"], n)
    ops.run_generate_tsdf_vertices_kernel(s["verts"], vs, box.size, box.dim)
    ops.run_translate_kernel(g.points, g.count, c)
    ops.run_translate_kernel(s["verts"], n, c)
    ops.run_warp_tsdf_kernel(s["verts"], g.transforms, s["idx"], s["w"], s["cnt"], vs, box.size, box.dim)
    ops.run_count_collisions_per_voxel_kernel(s["col"], s["verts"], s["cnt"], vs, box.size, box.dim, IDENTITY3, c)
    ops.run_integrate_warped_tsdf_from_frame_kernel(t.tsdf, t.weights, s["verts"], s["col"], s["cnt"], s["depth"],
                                                    s["size"], DELTA, vs, box.size, box.dim, IDENTITY3, c, s["K"],
                                                    MAX_WEIGHT)
    return s["out"]


def _prepare_plain(case, seed):
    box, K, depth = _plain_inputs(case, seed)
    tsdf = box.tsdf()
    return dict(tsdf=tsdf, depth=on_device(depth), K=K, pose=_pose(seed) if case["camera"] else None,
                out={"tsdf": view(tsdf.tsdf), "weights": view(tsdf.weights)})


def _run_plain(s):
    t, d = s["tsdf"], s["depth"]
    if s["pose"] is None:
        t.integrate(d, s["K"], MAX_WEIGHT)
    else:
        h, w = d.shape
        ops.run_integrate_tsdf_from_camera_frame_kernel(t.tsdf, t.weights, d, (w, h), t.delta, t.vol_dim,
                                                        t.voxel_size(), t.vol_size, s["pose"][0], s["pose"][1],
                                                        t.rotation, t.center, s["K"], MAX_WEIGHT)
    return s["out"]


INGEST = dict(threshold=2.0, sigma_i=75.0, sigma_s=75.0, step=0.025, angles=(1.3, 2.1))


def _prepare_ingest(case, seed):
    sc = Scene(seed, 1.0)
    w, h = case["width"], case["height"]
    raw = on_device(sc.depth(w, h))
    depth, verts, normals = buffer((h, w)), buffer((h * w, 3)), buffer((h * w, 3))
    return dict(ws=ops.Workspace(), raw=raw, depth=depth, verts=verts, normals=normals, K=L.m3(sc.camera(w, h)), w=w,
                h=h, r=case["radius"], out=(view(depth), view(verts), view(normals)))


def _run_ingest(s):
    # the frame loop's buffers are kept; a frame arrives in `raw`
    s["depth"].copy_from(s["raw"])
    c, n = L.Float3(), C.c_uint64(0)
    L.call("vf_ingest_depth", s["ws"].handle, s["depth"].ptr, s["w"], s["h"], s["K"], INGEST["threshold"], s["r"],
           INGEST["sigma_i"], INGEST["sigma_s"], INGEST["step"], INGEST["angles"][0], INGEST["angles"][1],
           s["verts"].ptr, s["normals"].ptr, C.byref(c), C.byref(n), None)
    depth, verts, normals = s["out"]
    return {"depth": depth, "vertices": verts, "normals": normals, "centroid": np.array([c.x, c.y, c.z], np.float32),
            "count": int(n.value)}


def _prepare_points(case, seed):
    nodes, radius, T, p = _points_inputs(case, seed)
    out = buffer(tuple(p.shape))
    return dict(ws=ops.Workspace(), k=case["k"], points=on_device(p), graph=_graph_object(nodes, radius, T), buf=out,
                blend=L.BLEND_DQB if case["blend"] == "dqb" else L.BLEND_LBS, out={"warped": view(out)})


def _run_points(s):
    ops.warp_points(s["ws"], s["k"], s["points"], s["graph"], s["buf"], s["blend"])
    return s["out"]


def _prepare_mesh(case, seed):
    box, v = _mesh_inputs(case, seed)
    tsdf = box.tsdf(v)
    cap = _mesh_room(box)
    s = dict(ws=ops.Workspace(), tsdf=tsdf, box=box, faces=case["faces"], host=case["host"])
    if case["host"]:
        # the program's own arrays, which it draws from
        s["out"] = {"vertices": np.zeros((cap, 3), np.float32)}
        if case["faces"]:
            s["out"]["faces"] = np.zeros((cap // 3, 3), np.int32)
    else:
        s.update(cap=cap, verts=buffer((cap, 3)), tris=buffer((cap // 3, 3), np.int32), n=buffer((2,), np.int32))
        s["out"] = {"vertices": view(s["verts"]), "counts": view(s["n"])}
        if case["faces"]:
            s["out"]["faces"] = view(s["tris"])
    return s


def _run_mesh(s):
    t, box = s["tsdf"], s["box"]
    if s["host"]:
        v, f = ops.marching_cubes(s["ws"], t.tsdf, t.weights, box.dim, t.voxel_size(), box.size, full=s["faces"])
        s["out"]["vertices"][:len(v)] = v
        if s["faces"]:
            s["out"]["faces"][:len(f)] = f
        return dict(s["out"], count=len(v))
    s["n"].fill(0)
    geom = (L.i3(box.dim), L.f3(t.voxel_size()), L.f3(box.size), 0.0, None)
    if s["faces"]:
        L.call("vf_marching_cubes_full", s["ws"].handle, s["verts"].ptr, s["n"].ptr, s["cap"], s["tris"].ptr,
               s["n"].ptr + 4, s["cap"] // 3, t.tsdf.ptr, t.weights.ptr, *geom)
    else:
        L.call("vf_marching_cubes_mesh", s["ws"].handle, s["verts"].ptr, s["n"].ptr, s["cap"], t.tsdf.ptr,
               t.weights.ptr, *geom)
    return s["out"]


def _prepare_icp(case, seed):
    i = _icp_inputs(case, seed)
    d = {k: on_device(v) for k, v in i.items() if isinstance(v, torch.Tensor)}
    G, M = case["nodes"], case["points"]
    s = dict(d, G=G, M=M, k=i["k"], iterations=case["iterations"], T=buffer((G, 16)), pending=buffer((G, 16)),
             warped=buffer((M, 3)))
    s["problem"] = L.GNProblem(d["corr"].ptr, i["corr"].shape[0], d["canon"].ptr, i["k"], d["knn"].ptr, d["kw"].ptr,
                               d["normals"].ptr, d["graph"].ptr, G, d["gknn"].ptr, case["reg_k"], 1.0, 0.5)
    s["out"] = {"transforms": view(s["T"]), "pending": view(s["pending"]), "warped": view(s["warped"])}
    return s


def _run_icp(s):
    s["T"].copy_from(s["T0"])
    L.call("vf_warp_mesh", s["k"], s["warped"].ptr, s["canon"].ptr, s["T"].ptr, s["knn"].ptr, s["kw"].ptr, s["M"],
           s["G"], None)
    solver, report = C.c_void_p(), L.GNReport()
    L.call("vf_gn_solver_create", C.byref(solver), C.byref(s["problem"]), None)
    try:
        L.call("vf_gn_solver_iterate", solver, s["T"].ptr, s["pending"].ptr, s["warped"].ptr, s["canon"].ptr, s["M"],
               s["target"].ptr, s["iterations"], -1e30, C.byref(report), None)
    finally:
        L.call("vf_gn_solver_destroy", solver)
    return s["out"]


_PREPARE = dict(frame=_prepare_frame, batch=_prepare_batch, dropin=_prepare_dropin, plain=_prepare_plain,
                ingest=_prepare_ingest, points=_prepare_points, mesh=_prepare_mesh, icp=_prepare_icp)
_RUN = dict(frame=_run_frame, batch=_run_batch, dropin=_run_dropin, plain=_run_plain, ingest=_run_ingest,
            points=_run_points, mesh=_run_mesh, icp=_run_icp)


# ---------------------------------------------------------------------------
# The work of one pass
# ---------------------------------------------------------------------------

def _band(case) -> tuple:
    """About how many voxels a frame updates, and how many have a node near
    that could collide with them: the camera sees half of the surfaces, the
    update reaches delta to both sides of it."""
    e = case["voxel"] * min(case["x"], case["y"], case["z"])
    area = 2 * 4 * math.pi * (0.235 * e) ** 2
    v3 = case["voxel"] ** 3
    updated = min(0.5 * area * 2 * DELTA / v3, 0.5 * case["x"] * case["y"] * case["z"])
    return updated, 2 * updated


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "batch":
        each = [dict(work(dict(c, kind="frame", k=case["k"]))) for c in _batch_cases(case)]
        return {"bytes": sum(w["bytes"] for w in each), "flops": sum(w["flops"] for w in each)}
    pixels = case.get("width", 0) * case.get("height", 0)
    if kind == "ingest":
        # raw frame in; depth, vertices and normals out; the neighbourhood's products
        return {"bytes": pixels * (4 + 4 + 12 + 12), "flops": pixels * (2 * case["radius"] + 1) ** 2 * 4}
    if kind == "points":
        return {"bytes": case["points"] * 24 + case["nodes"] * 80, "flops": case["points"] * case["k"] * 60}
    if kind == "icp":
        rows = 0.9 * case["points"]
        per = case["iterations"]
        inputs = case["points"] * (8 * case["k"] + 12 + 12 + 12 + 8) + case["nodes"] * (64 * 2 + 12 + 4 * case["reg_k"])
        return {"bytes": inputs + 12 * case["points"],
                "flops": rows * (case["k"] * (case["k"] + 1) / 2 * 72 + per * case["k"] * 60)}
    n = case["x"] * case["y"] * case["z"]
    updated, reach = _band(case)
    if kind == "plain":
        # every voxel in view and in front of the surface is updated: about half
        return {"bytes": 4 * pixels + 16 * 0.45 * n, "flops": n * 20}
    if kind == "mesh":
        return {"bytes": 8 * n + 36 * updated * case["voxel"] / DELTA, "flops": n}
    if kind == "dropin":
        # counts, collisions and vertices are outputs over the whole volume,
        # knn slots and weights over the voxels near a node
        return {"bytes": 20 * n + 4 * pixels + 80 * case["nodes"] + reach * 12 * case["k"] + 16 * updated,
                "flops": reach * case["k"] * 60}
    return {"bytes": 4 * pixels + 80 * case["nodes"] + 16 * updated, "flops": reach * case["k"] * 60}


# ---------------------------------------------------------------------------
# The same results in binary64
# ---------------------------------------------------------------------------

def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](case, seed)


def _exact_frame(case, seed, salt=0):
    box, nodes, radius, T, K, depth, start = _frame_inputs(case, seed, salt)
    t, w, _, _, _ = _warped_frame(box, nodes, radius, T, depth, K, case["k"], case.get("blend", "lbs"), start)
    return {"tsdf": t, "weights": w, "nodes": nodes.to(F64)}


def _exact_batch(case, seed):
    each = [_exact_frame(dict(c, k=case["k"]), seed, 100 + i) for i, c in enumerate(_batch_cases(case))]
    return {key: [e[key] for e in each] for key in ("tsdf", "weights", "nodes")}


def _exact_dropin(case, seed):
    box, nodes, radius, T, K, depth, start = _frame_inputs(case, seed)
    t, w, vox, p, count = _warped_frame(box, nodes, radius, T, depth, K, case["k"], "lbs", start)
    X, Y, Z = box.dim
    v = torch.empty(Z, Y, X, 3, device=DEV, dtype=F64)
    for a, shape in ((0, (1, 1, X)), (1, (1, Y, 1)), (2, (Z, 1, 1))):
        v[..., a] = box.corner(torch.arange(box.dim[a], device=DEV).view(shape), a, F64) + box.center[a]
    v = v.view(-1, 3)
    v[vox] = p
    return {"tsdf": t, "weights": w, "vertices": v, "counts": count}


def _exact_plain(case, seed):
    box, K, depth = _plain_inputs(case, seed)
    t, w = _plain(box, depth, K, F64, pose=_pose(seed) if case["camera"] else None)
    return {"tsdf": t.view(-1), "weights": w.view(-1)}


def _normals(v, dtype):
    """Normals of the inner pixels' back-projected neighbours."""
    v = v.to(dtype)
    gx, gy = v[1:-1, 2:] - v[1:-1, :-2], v[2:, 1:-1] - v[:-2, 1:-1]
    gx = gx / (gx[..., :1] * gx[..., :1] + gx[..., 1:2] * gx[..., 1:2]).sqrt()
    gy = gy / (gy[..., :1] * gy[..., :1] + gy[..., 1:2] * gy[..., 1:2]).sqrt()
    q = _cross(gy.reshape(-1, 3), gx.reshape(-1, 3))
    q = q / (q[:, :1] * q[:, :1] + (q[:, 1:2] * q[:, 1:2] + q[:, 2:] * q[:, 2:])).sqrt()
    return q.view(gx.shape)


def _exact_ingest(case, seed):
    sc = Scene(seed, 1.0)
    W, H, r = case["width"], case["height"], case["radius"]
    d = sc.depth(W, H)
    K = sc.camera(W, H)
    d = torch.where((d > INGEST["threshold"]) | (d < 1e-4), torch.full_like(d, math.inf), d)
    # bilateral filter: spatial and intensity weights from their tables
    g = [np.float32(math.exp(float(np.float32(-float(i - r) ** 2 / (2 * INGEST["sigma_s"] ** 2)))))
         for i in range(2 * r + 1)]
    table = [np.float32(math.exp(-((i / 10.0) ** 2) / 2)) for i in range(31)]
    color = torch.tensor([int(c / table[30]) for c in table], device=DEV, dtype=F32)
    norm = float(np.float32(30 / (3 * INGEST["sigma_i"])))
    pad = torch.nn.functional.pad(d[None, None], (r, r, r, r), mode="replicate")[0, 0]
    frames = {}
    for dtype in (F32, F64):
        acc, tot = torch.zeros(H, W, device=DEV, dtype=dtype), torch.zeros(H, W, device=DEV, dtype=dtype)
        for a in range(2 * r + 1):
            for b in range(2 * r + 1):
                p = pad[b:b + H, a:a + W]
                diff = (d - p).abs()
                ok = torch.isfinite(p) & ~(diff > float(np.float32(INGEST["step"])))
                q = torch.where(ok, (diff * norm).abs(), torch.zeros_like(d)).to(torch.int64).clamp(max=30)
                wgt = (float(g[b] * g[a]) * color[q]).to(dtype)
                acc = torch.where(ok, acc + p.to(dtype) * wgt, acc)
                tot = torch.where(ok, tot + wgt, tot)
        f = torch.where(torch.isfinite(d), acc / tot, torch.full_like(acc, math.inf))
        z = torch.where(torch.isfinite(f) & (f >= 1e-4), f, torch.zeros_like(f))
        rf = torch.tensor([1.0 / K[0], 1.0 / K[4]], device=DEV, dtype=dtype)
        x0 = (torch.arange(W, device=DEV, dtype=dtype) - K[6]) * rf[0]
        y0 = (torch.arange(H, device=DEV, dtype=dtype) - K[7]) * rf[1]
        frames[dtype] = f, torch.stack([x0[None] * z, y0[:, None] * z, z], -1)
    v32 = frames[F32][1]
    f, v = frames[F64]
    ok = (v32[1:-1, 1:-1, 2] >= 1e-4) & (v32[1:-1, 2:, 2] >= 1e-4) & (v32[1:-1, :-2, 2] >= 1e-4)
    ok = ok & (v32[2:, 1:-1, 2] >= 1e-4) & (v32[:-2, 1:-1, 2] >= 1e-4)
    lo, hi = (math.cos(float(np.float32(a))) for a in INGEST["angles"])
    q32 = _normals(v32, F32)
    nz = q32[..., 2].to(F64)
    ok = ok & ~((nz < lo) & (nz > hi))
    n = torch.zeros_like(v)
    n[1:-1, 1:-1] = torch.where(ok[..., None], _normals(v, F64), torch.zeros_like(n[1:-1, 1:-1]))
    gone = torch.zeros(H, W, device=DEV, dtype=torch.bool)
    gone[1:-1, 1:-1] = ~ok | (q32.abs() <= 1e-4).all(-1)
    v = torch.where(gone[..., None], torch.zeros_like(v), v)
    f = torch.where(gone, torch.full_like(f, math.inf), f)
    count = int((v[..., 2] > 1e-4).sum())
    c = (v.reshape(-1, 3).sum(0) / count).cpu().numpy()
    return {"depth": f, "vertices": v.reshape(-1, 3), "normals": n.reshape(-1, 3), "centroid": c, "count": count}


def _exact_points(case, seed):
    nodes, radius, T, p = _points_inputs(case, seed)
    d, idx = _nearest(p, nodes, case["k"])
    use = ~(d >= float(np.float32(radius)))
    p, m = p.to(F64), nodes.to(F64)
    r = float(np.float32(radius))
    w = torch.stack([torch.exp(-((p - m[idx[:, s]]) ** 2).sum(1) / (2 * r * r)) for s in range(idx.shape[1])], 1)
    w = torch.where(use, w, torch.zeros_like(w))
    total = w.sum(1, keepdim=True)
    w = torch.where(total > 0, w / total, w)
    near = use.any(1)
    out = p.clone()
    if case["blend"] == "dqb":
        out[near] = _dqb(T.to(F64), p[near], w[near], idx[near])
    else:
        out[near] = _lbs(T.to(F64), p[near], w[near], idx[near], False)
    return {"warped": out}


_EDGES = ((0, 1), (1, 2), (2, 3), (3, 0), (4, 5), (5, 6), (6, 7), (7, 4), (0, 4), (1, 5), (2, 6), (3, 7))
_CORNERS = ((1, 1, 0), (1, 0, 0), (0, 0, 0), (0, 1, 0), (1, 1, 1), (1, 0, 1), (0, 0, 1), (0, 1, 1))


def _exact_mesh(case, seed):
    # with faces the vertices follow the triangle table's order, which plain
    # tensor code does not give; the edge points themselves are those of the
    # mode without faces
    if case["faces"] or case["x"] * case["y"] * case["z"] > 40_000_000:
        return None
    box, (t, w) = _mesh_inputs(case, seed)
    X, Y, Z = box.dim
    cut = lambda a, o: a[o[2]:o[2] + Z - 2, o[1]:o[1] + Y - 2, o[0]:o[0] + X - 2]  # noqa: E731
    c = torch.stack([cut(t, o) for o in _CORNERS], -1).view(-1, 8)
    seen = torch.stack([cut(w, o) != 0 for o in _CORNERS], -1).all(-1).view(-1)
    above = c > 0.0
    crossed = torch.stack([above[:, a] ^ above[:, b] for a, b in _EDGES], 1) & seen[:, None]
    cube, edge = crossed.nonzero(as_tuple=True)
    ea, eb = (_t(np.array(_EDGES)[:, i], torch.int64)[edge] for i in (0, 1))
    t0, t1 = (c[cube, e].to(F64) for e in (ea, eb))
    off = _t(np.array(_CORNERS), torch.int64)
    at = torch.stack([cube % (X - 2), (cube // (X - 2)) % (Y - 2), cube // ((X - 2) * (Y - 2))], -1)
    p0, p1 = (torch.stack([box.corner((at + off[e])[:, a], a, F64) for a in range(3)], -1) for e in (ea, eb))
    mu = ((0.0 - t0) / (t1 - t0)).clamp(0.0, 1.0)
    mu = torch.where(t1.abs() < 1e-7, torch.ones_like(mu), mu)
    mu = torch.where((t0.abs() < 1e-7) | ((t1.abs() >= 1e-7) & ((t0 - t1).abs() < 1e-7)), torch.zeros_like(mu), mu)
    v = p0 + mu[:, None] * (p1 - p0)
    full = torch.zeros(_mesh_room(box), 3, device=DEV, dtype=F64)
    full[:v.shape[0]] = v
    if case["host"]:
        return {"vertices": full, "count": v.shape[0]}
    return {"vertices": full, "counts": None}


def _exact_icp(case, seed):
    i = _icp_inputs(case, seed)
    G, k, R = case["nodes"], i["k"], case["reg_k"]
    wD, wR = 1.0, 0.5
    canon, kw, knn = i["canon"].to(F64), i["kw"].to(F64), i["knn"].to(torch.int64)
    rows = i["corr"][:, 0].to(torch.int64)
    p, n, w, j = canon[rows], i["normals"].to(F64)[rows], kw[rows], knn[rows]
    target = i["target"].to(F64)[rows]
    graph, gknn = i["graph"].to(F64), i["gknn"].to(torch.int64)
    w = torch.where(i["kw"][rows] < 1e-4, torch.zeros_like(w), w)
    twist = torch.cat([torch.linalg.cross(p, n), n], 1) * wD  # n^T grad(p)
    A = torch.zeros(G * G, 36, device=DEV, dtype=F64)
    outer = (twist[:, :, None] * twist[:, None, :]).view(-1, 36)
    for a in range(k):
        for b in range(k):
            A.index_add_(0, j[:, a] * G + j[:, b], outer * (w[:, a] * w[:, b])[:, None])
    grad = torch.zeros(G, 3, 6, device=DEV, dtype=F64)
    x, y, z = graph.unbind(-1)
    grad[:, 0, 1], grad[:, 0, 2], grad[:, 1, 0], grad[:, 1, 2], grad[:, 2, 0], grad[:, 2, 1] = z, -y, -z, x, y, -x
    grad[:, 0, 3] = grad[:, 1, 4] = grad[:, 2, 5] = 1.0
    grad = grad * wR
    gg = (grad.transpose(1, 2) @ grad).view(G, 36)
    own, nb = torch.arange(G, device=DEV)[:, None].expand(G, R).reshape(-1), gknn.reshape(-1)
    have = nb >= 0
    own, nb = own[have], nb[have]
    for a, b, s in ((own, own, 1.0), (nb, nb, 1.0), (own, nb, -1.0), (nb, own, -1.0)):
        A.index_add_(0, a * G + b, s * gg[own])
    A = A.view(G, G, 6, 6).permute(0, 2, 1, 3).reshape(6 * G, 6 * G)
    A.diagonal()[A.diagonal() == 0] = 1.0  # a node without rows
    fac = torch.linalg.cholesky(A)
    del A
    T = i["T0"].to(F64).clone()
    warped = _lbs(T, canon, kw, knn, False)
    before = T
    for _ in range(case["iterations"]):
        before = T
        rd = wD * (n * (warped[rows] - target)).sum(1)
        M = T.view(G, 4, 4).transpose(1, 2)
        h = torch.cat([graph, torch.ones(G, 1, device=DEV, dtype=F64)], 1)
        rr = wR * ((M[own] @ h[own][:, :, None]) - (M[nb] @ h[own][:, :, None]))[:, :3, 0]
        b = torch.zeros(G, 6, device=DEV, dtype=F64)
        for s in range(k):
            b.index_add_(0, j[:, s], twist * (w[:, s] * rd)[:, None])
        gr = (grad[own].transpose(1, 2) @ rr[:, :, None])[:, :, 0]
        b.index_add_(0, own, gr)
        b.index_add_(0, nb, -gr)
        u = torch.cholesky_solve(b.view(-1, 1), fac).view(G, 6)
        U = torch.zeros(G, 4, 4, device=DEV, dtype=F64)
        U[:, 0, 1], U[:, 0, 2], U[:, 0, 3] = -u[:, 2], u[:, 1], u[:, 3]
        U[:, 1, 0], U[:, 1, 2], U[:, 1, 3] = u[:, 2], -u[:, 0], u[:, 4]
        U[:, 2, 0], U[:, 2, 1], U[:, 2, 3] = -u[:, 1], u[:, 0], u[:, 5]
        T = T - U.transpose(1, 2).reshape(G, 16)
        warped = _lbs(T, canon, kw, knn, False)
    return {"transforms": before, "pending": T, "warped": warped}


_EXACT = dict(frame=_exact_frame, batch=_exact_batch, dropin=_exact_dropin, plain=_exact_plain, ingest=_exact_ingest,
              points=_exact_points, mesh=_exact_mesh, icp=_exact_icp)
