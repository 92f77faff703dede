"""Performance cases: the work that a user of this framework has it do, through its public entry
points, each with the inputs it meets in use.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a
program holds before the call (device tensors, the geometry, a network), ``run`` is one pass,
``work`` the bytes and operations a pass cannot do without, and ``exact`` the same result in plain
64-bit torch, where that takes seconds.

Sizes are those of the workload configurations (128^3 x 180 views, 512^3 x 720, the 512^2 x 256
helix, 256^3 x 360, the warm-start training and inference geometries) and odd ones around them.
Lengths are in voxels; a voxel with index g along an axis of N voxels sits at g - N // 2, a detector
pixel with index g at (g - N // 2) pitches from the detector centre.
"""
import math

import numpy as np
import torch

from fastcone_amd import fastcone as cone
from fastcone_amd import ops, phantom
from fastcone_amd.geometry import Geometry
from fastcone_amd.katsevich import HelixScan, katsevich
from fastcone_amd.unet import UNet3D

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def _ct(name, kind, nz, ny, nx, nv, nh, nw, pw, D, step=0.5, dtype="f32", mode=2, tilt=0.0):
    c = dict(kind=kind, nz=nz, ny=ny, nx=nx, nv=nv, nh=nh, nw=nw, pw=pw, D=D, step=step,
             dtype=dtype, mode=mode, tilt=tilt)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a quick look at a small specimen: launches and host latency count
        _ct("project small", "project", 64, 64, 64, 60, 96, 96, 0.75, 250.0, step=1.0),
        # the headline projector: 512^3, 720 views, 768^2 detector, half-voxel steps
        _ct("project 512x720", "project", 512, 512, 512, 720, 768, 768, 0.75, 1200.0),
        # a cropped block stored in 16 bits, odd sizes, few views
        _ct("project ragged bf16", "project", 203, 250, 301, 181, 288, 437, 0.8, 700.0,
            dtype="bf16"),
        # the matched transpose inside an iterative solver (256^3, 360 views)
        _ct("adjoint 256x360", "adjoint", 256, 256, 256, 360, 384, 384, 0.6, 500.0),
        # one gradient of |A x - b|^2 / 2 through autograd, at the warm-start training geometry
        _ct("gradient 128x90", "gradient", 128, 128, 128, 90, 192, 192, 0.75, 500.0),
        # filtered backprojection of a small scan, as a preview or a network's input
        _ct("fdk small", "fdk", 64, 64, 64, 60, 96, 96, 0.75, 250.0),
        # the headline reconstruction
        _ct("fdk 512x720", "fdk", 512, 512, 512, 720, 768, 768, 0.75, 1200.0),
        # unweighted backprojection of a misaligned detector, 16-bit projections, odd sizes
        _ct("backproject tilted f16", "backproject", 150, 333, 290, 275, 251, 470, 0.8, 800.0,
            dtype="f16", mode=0, tilt=0.01),
        # the whole helical reconstruction: 512^2 x 256, three turns of 1440 views
        dict(name="katsevich helix", kind="katsevich", nz=256, ny=512, nx=512, turns=3,
             per_turn=1440, nh=64, nw=512, R=1140.0, SDD=2080.0, dgamma=0.8 / 1040.0, drow=2.0,
             pitch=0.8, dtype="f32"),
        # the warm-start network: inference on one volume, and one training step's gradients
        dict(name="unet infer 256", kind="infer", n=1, nz=256, ny=256, nx=256),
        dict(name="unet train 4x128", kind="train", n=4, nz=128, ny=128, nx=128),
        # the drop-in calls on host arrays: forward projection, then backprojection
        _ct("host pair 128x180", "host", 128, 128, 128, 180, 192, 192, 0.75, 500.0, step=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["project", "adjoint", "gradient", "fdk", "backproject", "katsevich",
                       "infer", "train", "host"])
    if kind in ("infer", "train"):
        # sides are multiples of four; a training step holds a batch
        top = 256 if kind == "infer" else 128
        side = [4 * _log(rng, 8, top // 4) for _ in range(3)]
        return dict(kind=kind, n=1 if kind == "infer" else rng.randint(1, 4), nz=side[0],
                    ny=side[1], nx=side[2])
    if kind == "katsevich":
        nxy = _log(rng, 64, 384)
        nw, nh = int(1.1 * nxy), rng.choice([16, 24, 33, 48, 64])
        per_turn = rng.randrange(300, 1100)
        R, SDD = 2.2 * nxy, 4.0 * nxy
        drow = rng.choice([1.0, 1.5, 2.0])
        return dict(kind=kind, nz=_log(rng, 24, 96), ny=nxy, nx=nxy + rng.randrange(0, 9),
                    turns=rng.randint(2, 3), per_turn=per_turn, nh=nh, nw=nw, R=R, SDD=SDD,
                    dgamma=1.5 / nw * nxy / R, drow=drow, pitch=0.8,
                    dtype=rng.choice(["f32", "f32", "bf16", "f16"]))
    top = {"project": 384, "adjoint": 200, "gradient": 160, "fdk": 400, "backproject": 400,
           "host": 160}[kind]
    n = _log(rng, 48, top)
    nz, ny, nx = (max(24, int(n * rng.uniform(0.7, 1.1))) for _ in range(3))
    pw = rng.uniform(0.6, 0.9)
    nw = int(1.15 * math.hypot(nx, ny) / pw * rng.uniform(0.8, 1.0))
    nh = int(1.2 * nz / pw)
    D = round(n * rng.uniform(2.3, 4.0), 1)
    nv = _log(rng, 30, 400)
    dtype = "f32" if kind in ("gradient", "host") else rng.choice(["f32", "f32", "bf16", "f16"])
    step = 1.0 if kind == "host" else rng.choice([0.5, 0.5, 1.0, 0.4])
    mode = rng.choice([0, 1, 2]) if kind == "backproject" else 2
    tilt = rng.choice([0.0, 0.01]) if mode == 0 else 0.0
    return _ct(None, kind, nz, ny, nx, nv, nh, nw, pw, D, step=step, dtype=dtype, mode=mode,
               tilt=tilt)


# ---- inputs ---------------------------------------------------------------------------------


def _ellipsoids(c, seed, count=10):
    """Random ellipsoids that fill a block of the case's size (axes and densities as the
    configurations', scaled with the block)."""
    n = min(c["nz"], c["ny"], c["nx"])
    return phantom.random_ellipsoids(seed, count, (0.04 * n, 0.3 * n), (0.005, 0.02), 0.25 * n)


def _misalign(c):
    t = c["tilt"]
    return None if t == 0.0 else np.array([1.5, -2.0, 3.0, t, -0.5 * t, 0.75 * t], np.float32)


def _angles(c):
    return 2 * np.pi * np.arange(c["nv"]) / c["nv"]


def _geometry(c):
    return Geometry.circular(_angles(c), c["D"], c["pw"], (c["nz"], c["ny"], c["nx"]),
                             (c["nh"], c["nw"]), misalign=_misalign(c))


def _helix(c):
    height = c["nh"] * c["drow"] * c["R"] / c["SDD"]       # detector height at the axis
    hp = c["pitch"] * height / (2 * math.pi)
    n = c["turns"] * c["per_turn"]
    dl = 2 * math.pi / c["per_turn"]
    return HelixScan(n, dl, 0.0, -hp * dl * (n - 1) / 2.0, hp, c["R"], c["SDD"], c["dgamma"],
                     c["drow"], c["nw"], c["nh"])


def _frames(c):
    """Source, position of pixel (0, 0) and the two pixel steps of every view, float64 [nv, 3]:
    the aligned system, then the six misalignment parameters (two shifts along the detector in
    pixels, one along the axis ray, three turns), each turn against the current axes."""
    a = _angles(c)
    z, o = np.zeros_like(a), np.ones_like(a)
    s = np.stack([-np.cos(a) * c["D"], -np.sin(a) * c["D"], c["nz"] / 2.0 - c["nz"] // 2 + z], 1)
    d = np.stack([z, z, s[:, 2]], 1)
    v = np.stack([z, z, c["pw"] * o], 1)
    u = c["pw"] * np.stack([-np.sin(a), np.cos(a), z], 1)
    m = _misalign(c)
    if m is not None:
        m = m.astype(np.float64)
        unit = lambda x: x / np.linalg.norm(x, axis=1, keepdims=True)
        size = lambda x: np.linalg.norm(x, axis=1, keepdims=True)
        d = d + m[0] * u + m[1] * v
        d = d + m[2] * unit(d - s)
        v = size(v) * (math.cos(m[3]) * unit(v) + math.sin(m[3]) * unit(np.cross(u, v)))
        u = size(u) * (math.cos(m[4]) * unit(u) + math.sin(m[4]) * unit(np.cross(u, v)))
        n = np.cross(u, v)
        u, v = (size(u) * (math.cos(m[5]) * unit(u) - math.sin(m[5]) * unit(np.cross(u, n))),
                size(v) * (math.cos(m[5]) * unit(v) + math.sin(m[5]) * unit(np.cross(v, n))))
    return s, d - (c["nw"] // 2) * u - (c["nh"] // 2) * v, u, v


def _helix_frames(c):
    h = _helix(c)
    l = h.lambdas
    z = np.zeros_like(l)
    s = np.stack([c["R"] * np.cos(l), c["R"] * np.sin(l), h.src_z], 1)
    return s, np.stack([-np.cos(l), -np.sin(l), z], 1), np.stack([-np.sin(l), np.cos(l), z], 1)


def _integrals(c, ell, dev, seed, noise=0.02):
    """Line integrals [nv, nh, nw] of ellipsoids along the case's rays, with seeded noise."""
    if c["kind"] == "katsevich":
        s, ev, eu = _helix_frames(c)
        nv = s.shape[0]
        g = (torch.arange(c["nw"], device=dev) - (c["nw"] - 1) / 2.0).double() * c["dgamma"]
        w = (torch.arange(c["nh"], device=dev) - (c["nh"] - 1) / 2.0).double() * c["drow"]
    else:
        s, d0, du, dv = _frames(c)
        nv = c["nv"]
        j = torch.arange(c["nw"], device=dev).double()
        i = torch.arange(c["nh"], device=dev).double()
    out = torch.zeros((nv, c["nh"], c["nw"]), device=dev)
    step = max(1, (1 << 26) // (c["nh"] * c["nw"]))
    for t in range(0, nv, step):
        T = lambda x: torch.as_tensor(x[t:t + step], device=dev)[:, None, None, :]
        if c["kind"] == "katsevich":
            r = c["SDD"] * (torch.cos(g)[None, None, :, None] * T(ev)
                            + torch.sin(g)[None, None, :, None] * T(eu))
            r = r.expand(-1, c["nh"], -1, -1).clone()
            r[..., 2] += w[None, :, None]
        else:
            r = (T(d0) - T(s)) + j[None, None, :, None] * T(du) + i[None, :, None, None] * T(dv)
        r = r.float()
        r /= r.norm(dim=-1, keepdim=True)
        for cen, ax, R, mu in ell:
            M = torch.as_tensor(np.asarray(R).T / np.asarray(ax)[:, None], device=dev)
            q = (T(s) - torch.as_tensor(cen, device=dev)) @ M.T
            e = r @ M.T.float()
            ee = (e * e).sum(-1)
            b = (e * q.float()).sum(-1)
            disc = b * b - ee * ((q * q).sum(-1) - 1.0).float()
            out[t:t + step] += float(2.0 * mu) * disc.clamp_(min=0.0).sqrt_() / ee
    gen = torch.Generator(device=dev).manual_seed(seed + 17)
    return out.add_(torch.randn(out.shape, device=dev, generator=gen), alpha=noise)


def _volume(c, ell, dev, seed):
    return phantom.voxelize(ell, (c["nz"], c["ny"], c["nx"]), 1.0, dev, texture_sigma=0.001,
                            texture_seed=seed)


def _network(c, dev, seed):
    """A network at its initial weights, an FDK-like input and the target it is trained to."""
    gen = torch.Generator(device=dev).manual_seed(seed)
    shape = (c["n"], c["nz"], c["ny"], c["nx"])
    vols = torch.stack([_volume(c, _ellipsoids(c, seed + 100 * k), dev, seed + k)
                        for k in range(c["n"])])
    x = vols + 0.002 * torch.randn(shape, device=dev, generator=gen)
    return UNet3D(seed=seed).to(dev), x, vols


def prepare(case, seed):
    c = case
    dev = torch.device("cuda", torch.cuda.current_device())
    kind = c["kind"]
    s = dict(case=c)
    if kind in ("infer", "train"):
        s["net"], s["x"], s["y"] = _network(c, dev, seed)
        if kind == "infer":
            s["x"] = s["x"][0].contiguous()
        return s
    ell = _ellipsoids(c, seed)
    if kind == "katsevich":
        s["scan"] = _helix(c)
        s["proj"] = _integrals(c, ell, dev, seed).to(DTYPES[c["dtype"]])
        return s
    if kind == "host":
        s["vol"] = _volume(c, ell, dev, seed).cpu().numpy()
        s["angles"] = _angles(c).astype(np.float32)
        s["z0"] = np.full(c["nv"], c["nz"] / 2.0, np.float32)
        return s
    s["geom"] = _geometry(c)
    if kind in ("project", "gradient"):
        s["vol"] = _volume(c, ell, dev, seed).to(DTYPES[c["dtype"]])
    if kind != "project":
        s["proj"] = _integrals(c, ell, dev, seed).to(DTYPES[c["dtype"]])
    if kind == "backproject":
        s["norm"] = torch.full((c["nv"],), 1.0 / c["nv"], device=dev)
    return s


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "project":
        return ops.project(state["vol"], state["geom"], c["step"])
    if kind == "adjoint":
        return ops.adjoint(state["proj"], state["geom"], c["step"])
    if kind == "gradient":
        x = state["vol"].detach().requires_grad_(True)
        r = ops.cone_project(x, state["geom"], c["step"]) - state["proj"]
        loss = 0.5 * (r * r).sum()
        loss.backward()
        return {"residual": r.detach(), "grad": x.grad}
    if kind == "fdk":
        return ops.fdk(state["proj"], state["geom"], c["D"], c["pw"],
                       store_dtype=DTYPES[c["dtype"]])
    if kind == "backproject":
        return ops.backproject(state["proj"], state["geom"], c["mode"], norm=state["norm"])
    if kind == "katsevich":
        return katsevich(state["proj"], state["scan"], (c["nz"], c["ny"], c["nx"]))
    if kind == "infer":
        with torch.no_grad():
            return state["net"](state["x"])
    if kind == "train":
        net = state["net"]
        net.zero_grad(set_to_none=True)
        loss = ((net(state["x"]) - state["y"]) ** 2).mean() * UNet3D.SCALE ** 2
        loss.backward()
        return {k: p.grad for k, p in net.named_parameters()}
    # host arrays, as the drop-in calls take them
    proj = np.zeros((c["nv"], c["nh"], c["nw"]), np.float32)
    rec = np.zeros((c["nz"], c["ny"], c["nx"]), np.float32)
    cone.project(state["vol"], proj, state["angles"], c["D"], state["z0"], pixelWidth=c["pw"])
    cone.backproject(rec, proj, state["angles"], c["D"], state["z0"], pixelWidth=c["pw"])
    return {"proj": proj, "vol": rec}


# ---- what a pass cannot do without ------------------------------------------------------------

SAMPLE = 24.0    # operations of a trilinear sample: positions, seven interpolations, the sum
PIXEL = 16.0     # operations of a bilinear sample with its coordinates and weight

CONVS = [(1, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2),
         (96, 32, 1), (32, 32, 1), (48, 16, 0), (16, 16, 0), (16, 1, 0)]  # in, out, level


def _samples(c):
    """Ray samples of a projection: one per pixel area and step inside every voxel."""
    return c["nz"] * c["ny"] * c["nx"] * c["nv"] / (c["pw"] ** 2 * c["step"])


def work(case):
    c = case
    kind = c["kind"]
    vox = float(c["nz"] * c["ny"] * c["nx"])
    if kind in ("infer", "train"):
        vox *= c["n"]
        mac = sum(27.0 * i * o * vox / 8 ** l for i, o, l in CONVS)
        times = 3.0 if kind == "train" else 1.0      # forward, input and weight gradients
        weights = sum(27 * i * o + o for i, o, _ in CONVS) * 4.0
        return {"bytes": vox * 8.0 + weights * (2.0 if kind == "train" else 1.0),
                "flops": 2.0 * mac * times}
    size = 4.0 if c["dtype"] == "f32" else 2.0
    if kind == "katsevich":
        nv = c["turns"] * c["per_turn"]
        # a voxel sees about half a turn of views through its window
        return {"bytes": nv * c["nh"] * c["nw"] * size + vox * 4.0,
                "flops": vox * 0.55 * c["per_turn"] * PIXEL}
    rays = float(c["nv"] * c["nh"] * c["nw"])
    if kind == "project":
        return {"bytes": vox * size + rays * 4.0, "flops": SAMPLE * _samples(c)}
    if kind == "adjoint":
        return {"bytes": vox * 4.0 + rays * size, "flops": SAMPLE * _samples(c)}
    if kind == "gradient":
        return {"bytes": vox * 8.0 + rays * 8.0, "flops": 2 * SAMPLE * _samples(c)}
    if kind == "host":
        return {"bytes": vox * 8.0 + rays * 4.0,
                "flops": SAMPLE * _samples(c) + PIXEL * vox * c["nv"]}
    return {"bytes": vox * 4.0 + rays * size, "flops": PIXEL * vox * c["nv"]}


# ---- the same in 64 bits ------------------------------------------------------------------------


def _rays64(c, dev):
    """Chunks of rays: (flat ray range, source, unit direction, first and last sample number)."""
    s, d0, du, dv = (torch.as_tensor(x, device=dev) for x in _frames(c))
    n = torch.tensor([c["nx"], c["ny"], c["nz"]], dtype=torch.float64, device=dev)
    org = torch.tensor([-(c["nx"] // 2), -(c["ny"] // 2), -(c["nz"] // 2)], dtype=torch.float64,
                       device=dev)
    per = c["nh"] * c["nw"]
    chunk = max(1, int(4e6 * c["step"] / max(c["nx"], c["ny"], c["nz"]) / c["nw"])) * c["nw"]
    for t in range(c["nv"]):
        for p0 in range(0, per, chunk):
            p = torch.arange(p0, min(per, p0 + chunk), device=dev)
            i = torch.div(p, c["nw"], rounding_mode="floor").double()[:, None]
            j = (p % c["nw"]).double()[:, None]
            u = d0[t] + j * du[t] + i * dv[t] - s[t]
            u = u / u.norm(dim=1, keepdim=True)
            src = s[t] - org                             # in voxel indices
            ta, tb = (-1.0 - src) / u, (n - src) / u
            lo = torch.minimum(ta, tb).amax(1)
            hi = torch.maximum(ta, tb).amin(1)
            k0, k1 = torch.ceil(lo / c["step"]), torch.floor(hi / c["step"])
            k1 = torch.where(hi >= lo, k1, k0 - 1.0)
            yield t * per + p0, src, u, k0, k1


def _corners(c, src, u, k0, k1):
    """The eight (index into a volume with a one-voxel zero border, weight) of a chunk's samples."""
    K = int((k1 - k0).max().item()) + 1
    if K <= 0:
        return
    k = k0[:, None] + torch.arange(K, device=u.device, dtype=torch.float64)
    on = (k <= k1[:, None]).double()
    k = torch.minimum(k, torch.maximum(k0, k1)[:, None])
    f, b = [], []
    for a, n in enumerate((c["nx"], c["ny"], c["nz"])):
        q = (src[a] + k * c["step"] * u[:, a:a + 1]).clamp_(-1.0, n)
        fl = torch.floor(q).clamp_(max=n - 1)
        f.append(q - fl)
        b.append(fl.long() + 1)
    PX, PY = c["nx"] + 2, c["ny"] + 2
    base = (b[2] * PY + b[1]) * PX + b[0]
    for dz in range(2):
        wz = on * (f[2] if dz else 1.0 - f[2])
        for dy in range(2):
            wy = wz * (f[1] if dy else 1.0 - f[1])
            for dx in range(2):
                yield base + (dz * PY + dy) * PX + dx, wy * (f[0] if dx else 1.0 - f[0])


def _project64(c, vol):
    pad = torch.nn.functional.pad(vol.double(), (1, 1) * 3).reshape(-1)
    out = torch.zeros(c["nv"] * c["nh"] * c["nw"], dtype=torch.float64, device=vol.device)
    for r0, src, u, k0, k1 in _rays64(c, vol.device):
        for idx, w in _corners(c, src, u, k0, k1):
            out[r0:r0 + u.shape[0]] += c["step"] * (w * pad[idx]).sum(1)
    return out.view(c["nv"], c["nh"], c["nw"])


def _adjoint64(c, proj):
    y = proj.double().reshape(-1)
    acc = torch.zeros((c["nz"] + 2) * (c["ny"] + 2) * (c["nx"] + 2), dtype=torch.float64,
                      device=proj.device)
    for r0, src, u, k0, k1 in _rays64(c, proj.device):
        yy = c["step"] * y[r0:r0 + u.shape[0], None]
        for idx, w in _corners(c, src, u, k0, k1):
            acc.index_add_(0, idx.reshape(-1), (w * yy).reshape(-1))
    return acc.view(c["nz"] + 2, c["ny"] + 2, c["nx"] + 2)[1:-1, 1:-1, 1:-1].contiguous()


def _bilinear64(img, u, v):
    """Bilinear samples of img [nh, nw], extended by zeros."""
    nh, nw = img.shape
    pad = torch.nn.functional.pad(img, (1, 1, 1, 1)).reshape(-1)
    on = ((u > -1) & (u < nw) & (v > -1) & (v < nh)).double()
    u, v = u.clamp(-1.0, nw), v.clamp(-1.0, nh)
    iu, iv = torch.floor(u).clamp(max=nw - 1), torch.floor(v).clamp(max=nh - 1)
    fu, fv = u - iu, v - iv
    b = ((iv + 1) * (nw + 2) + iu + 1).long()
    lo = pad[b] * (1 - fu) + pad[b + 1] * fu
    hi = pad[b + nw + 2] * (1 - fu) + pad[b + nw + 3] * fu
    return on * (lo * (1 - fv) + hi * fv)


def _backproject64(c, proj, mode):
    dev = proj.device
    ax = [torch.arange(n, device=dev).double() - n // 2 for n in (c["nz"], c["ny"], c["nx"])]
    Z, Y, X = torch.meshgrid(*ax, indexing="ij")
    s, d0, du, dv = (torch.as_tensor(x, device=dev) for x in _frames(c))
    vol = torch.zeros_like(X)
    for t in range(c["nv"]):
        n = torch.linalg.cross(du[t], dv[t])
        # the point at the source plus lam times (voxel - source) lies in the detector plane
        rx, ry, rz = X - s[t, 0], Y - s[t, 1], Z - s[t, 2]
        lam = torch.dot(n, d0[t] - s[t]) / (n[0] * rx + n[1] * ry + n[2] * rz)
        g = torch.linalg.inv(torch.stack([du[t], dv[t], n], 1))      # plane coordinates
        o = g @ (s[t] - d0[t])
        u = o[0] + lam * (g[0, 0] * rx + g[0, 1] * ry + g[0, 2] * rz)
        v = o[1] + lam * (g[1, 0] * rx + g[1, 1] * ry + g[1, 2] * rz)
        vol += lam ** mode * _bilinear64(proj[t].double(), u, v)
    return vol / c["nv"]


def _filter64(c, proj):
    """Cosine of each pixel's ray with the detector normal, then the ramp (rows padded to twice
    their length, pi k / n in bin k of n, an eighth of a bin at zero), over the pixel pitch."""
    dev = proj.device
    s, d0, du, dv = (torch.as_tensor(x, device=dev) for x in _frames(c))
    n = 2 * c["nw"]
    H = math.pi * torch.arange(c["nw"] + 1, device=dev).double() / n
    H[0] = math.pi * 0.125 / n
    j = torch.arange(c["nw"], device=dev).double()[None, :, None]
    i = torch.arange(c["nh"], device=dev).double()[:, None, None]
    out = torch.empty(proj.shape, dtype=torch.float64, device=dev)
    for t in range(c["nv"]):
        nor = torch.linalg.cross(du[t], dv[t])
        p = (d0[t] - s[t]) + j * du[t] + i * dv[t]
        w = (torch.dot(nor, d0[t] - s[t]) / nor.norm()).abs() / p.norm(dim=2)
        f = torch.fft.rfft(proj[t].double() * w, n=n, dim=1) * H
        out[t] = torch.fft.irfft(f, n=n, dim=1)[:, :c["nw"]] / c["pw"]
    return out


def _katsevich64(c, proj):
    """Derivative at a fixed ray direction, cone weight, resampling onto kappa lines, the curved
    detector's Hilbert kernel, resampling back, and the sum over each voxel's window."""
    dev = proj.device
    h = _helix(c)
    nv, nh, nw, npsi = h.nviews, h.nh, h.nw, 2 * h.nh + 1
    A = lambda n: torch.arange(n, device=dev).double()
    p = proj.double()
    gam = (A(nw) - h.col_c) * h.dgamma
    wrow = (A(nh) - h.row_c) * h.drow
    sh = h.dl / h.dgamma

    def shift(x, by):
        pos = A(nw) + by
        f = torch.floor(pos)
        t, j0 = pos - f, f.long()
        x = torch.nn.functional.pad(x, (1, 1))           # one zero column each side
        return (1 - t) * x[..., (j0 + 1).clamp(0, nw + 1)] + t * x[..., (j0 + 2).clamp(0, nw + 1)]

    g2 = torch.zeros_like(p)
    g2[1:-1] = (shift(p[2:], sh) - shift(p[:-2], -sh)) * (0.5 / h.dl)
    g2 *= (h.SDD / torch.sqrt(h.SDD ** 2 + wrow ** 2))[None, :, None]
    am = max(abs(h.col_c), abs(nw - 1 - h.col_c)) * h.dgamma
    pmax = math.pi / 2 + am
    dpsi = 2 * pmax / (npsi - 1)
    psi = -pmax + A(npsi) * dpsi
    pc = torch.where(psi.abs() < 1e-12, torch.ones_like(psi), psi / torch.tan(psi))
    wk = h.SDD * h.hp / h.R * (psi[:, None] * torch.cos(gam) + pc[:, None] * torch.sin(gam))
    row = wk / h.drow + h.row_c                          # [npsi, nw]
    f = torch.floor(row)
    t, i0 = row - f, f.long()
    pad = torch.nn.functional.pad(g2, (0, 0, 1, 1))
    J = torch.arange(nw, device=dev)
    g3 = ((1 - t) * pad[:, (i0 + 1).clamp(0, nh + 1), J]
          + t * pad[:, (i0 + 2).clamp(0, nh + 1), J])    # [nv, npsi, nw]
    d = torch.arange(-(nw - 1), nw, device=dev).double()
    ker = torch.where(d.long() % 2 != 0, 2 * h.dgamma / (math.pi * torch.sin(d * h.dgamma)),
                      torch.zeros_like(d))
    L = 1 << (3 * nw - 2).bit_length()
    fk = torch.fft.rfft(ker, n=L)
    g4 = torch.empty_like(g3)
    for k in range(0, nv, 256):
        g4[k:k + 256] = torch.fft.irfft(torch.fft.rfft(g3[k:k + 256], n=L) * fk,
                                        n=L)[..., nw - 1:2 * nw - 1]
    wt = wk.T.contiguous()                               # increasing in psi for every column
    lo = (torch.searchsorted(wt, wrow.expand(nw, nh).contiguous(), right=True) - 1).T
    inside = (wrow[:, None] >= wk[0]) & (wrow[:, None] <= wk[-1])
    lo = lo.clamp(0, npsi - 2)
    wl, wh = wk.gather(0, lo), wk.gather(0, lo + 1)
    t = (wrow[:, None] - wl) / (wh - wl)
    g5 = inside * ((1 - t) * g4[:, lo, J] + t * g4[:, lo + 1, J])
    del g2, g3, g4, pad
    nz, ny, nx = c["nz"], c["ny"], c["nx"]
    Y, X = torch.meshgrid(A(ny) - ny // 2, A(nx) - nx // 2, indexing="ij")
    Z = (A(nz) - nz // 2)[:, None, None]
    vol = torch.zeros((nz, ny, nx), dtype=torch.float64, device=dev)
    for k in range(nv):
        l, zs = h.l0 + k * h.dl, float(h.src_z[k])
        vs = h.R - X * math.cos(l) - Y * math.sin(l)
        us = -X * math.sin(l) + Y * math.cos(l)
        ga = torch.atan(us / vs)
        sec = 1.0 / torch.cos(ga)
        c0 = h.SDD * h.hp / h.R / h.drow
        top = c0 * (math.pi / 2 - ga) * sec + h.row_c
        bot = -c0 * (math.pi / 2 + ga) * sec + h.row_c
        dr = h.SDD / h.drow / (vs * sec)
        # slices whose rows can lie in the window
        zt = ((top - h.row_c) / dr).max().item() + zs
        zb = ((bot - h.row_c) / dr).min().item() + zs
        a, b = max(0, int(math.floor(zb)) + nz // 2), min(nz, int(math.ceil(zt)) + nz // 2 + 1)
        if a >= b:
            continue
        r = (Z[a:b] - zs) * dr + h.row_c
        u = (ga / h.dgamma + h.col_c).expand_as(r)
        ok = ((r >= bot) & (r <= top)).double()
        vol[a:b] += ok / vs * _bilinear64(g5[k], u, r)
    return vol * (h.dl / (2 * math.pi))


def _net64(net, x):
    P = {k: p.detach().double().requires_grad_(True) for k, p in net.named_parameters()}

    def conv(v, name, relu=True):
        w, b = P["w." + name], P["b." + name]
        pad = torch.nn.functional.pad(v, (0, 0) + (1, 1) * 3)
        _, D, H, W, _ = v.shape
        y = b
        for q in range(27):
            z, r, s = q // 9, q // 3 % 3, q % 3
            y = y + pad[:, z:z + D, r:r + H, s:s + W] @ w[:, q].T
        return torch.relu(y) if relu else y

    def down(v):
        N, D, H, W, C = v.shape
        return v.view(N, D // 2, 2, H // 2, 2, W // 2, 2, C).mean(dim=(2, 4, 6))

    def up(v):
        for a in (1, 2, 3):
            v = v.repeat_interleave(2, dim=a)
        return v

    v = (x.double() * UNet3D.SCALE)[..., None]
    e1 = conv(conv(v, "e1a"), "e1b")
    e2 = conv(conv(down(e1), "e2a"), "e2b")
    bt = conv(conv(down(e2), "b_a"), "b_b")
    d2 = conv(conv(torch.cat([up(bt), e2], -1), "d2a"), "d2b")
    d1 = conv(conv(torch.cat([up(d2), e1], -1), "d1a"), "d1b")
    return x.double() + conv(d1, "out", False)[..., 0] / UNet3D.SCALE, P


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind in ("infer", "train"):
        vox = c["n"] * c["nz"] * c["ny"] * c["nx"]
        if vox > (1 << 24 if kind == "infer" else 1 << 18):
            return None
        s = prepare(c, seed)
        if kind == "infer":
            with torch.no_grad():
                return _net64(s["net"], s["x"][None])[0][0]
        y, P = _net64(s["net"], s["x"])
        (((y - s["y"].double()) ** 2).mean() * UNet3D.SCALE ** 2).backward()
        return {k: p.grad for k, p in P.items()}
    vox = c["nz"] * c["ny"] * c["nx"]
    if kind == "katsevich":
        if vox * c["turns"] * c["per_turn"] > 5e10:
            return None
        return _katsevich64(c, prepare(c, seed)["proj"])
    if kind in ("fdk", "backproject"):
        if vox * c["nv"] > 1e10:
            return None
        p = prepare(c, seed)["proj"]
        if kind == "fdk":
            return _backproject64(c, _filter64(c, p).to(DTYPES[c["dtype"]]), 2)
        return _backproject64(c, p, c["mode"])
    if _samples(c) > (1e10 if kind == "project" else 1.5e9):
        return None
    s = prepare(c, seed)
    if kind == "project":
        return _project64(c, s["vol"])
    if kind == "adjoint":
        return _adjoint64(c, s["proj"])
    if kind == "gradient":
        r = _project64(c, s["vol"]) - s["proj"].double()
        return {"residual": r, "grad": _adjoint64(c, r)}
    # the drop-in projector takes unit steps and zeroes detector column 0
    dev = torch.device("cuda", torch.cuda.current_device())
    proj = _project64(c, torch.from_numpy(s["vol"]).to(dev))
    proj[:, :, 0] = 0.0
    return {"proj": proj, "vol": _backproject64(c, proj, 2)}
