"""GPU parity of the backprojector's view tables, window copies and view splits against the FP64
oracle, at the sizes where they can go wrong: one view, more views than a table holds, view counts
that do not divide into the splits, windows over every edge of the detector, detectors of fewer
columns than a copied unit, partial cubes.

Tolerance: tile coordinates are rounded to FP32 at magnitudes below 128 pixels (about 1e-5 pixel), so
on N(0, 1) data relative L2 < 5e-5, as for every other path; 16-bit storage is compared with the
oracle fed the rounded data.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("nv", [1, 4, 11, 60])
@pytest.mark.parametrize("det", [(26, 30), (9, 3), (5, 1), (40, 70)])
@pytest.mark.parametrize("mode,mis", [(2, None), (1, None),
                                      (0, [0.6, -0.8, 1.5, 0.02, -0.03, 0.01])])
@pytest.mark.parametrize("dt", ["float32", "float16"])
def test_small_volumes(gpu, nv, det, mode, mis, dt):
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    rng = np.random.default_rng(nv + det[1] + mode)
    ang = np.sort(rng.uniform(0, 2 * np.pi, nv))
    vol = (18, 33, 20)
    hmid = rng.uniform(7, 11, nv)
    g = Geometry.circular(ang, 70.0, 0.9, vol, det, hmid=hmid, misalign=mis)
    prob = oracle.Problem(ang, hmid, 70.0, 0.9, vol_dim=vol[::-1], proj_dim=det[::-1], mis=mis)
    y = torch.from_numpy(rng.standard_normal(g.proj_shape).astype(np.float32)).to(
        getattr(torch, dt))
    norm = rng.uniform(0.5, 1.5, nv).astype(np.float32)
    base = torch.from_numpy(rng.standard_normal(vol).astype(np.float32)).to(gpu)
    out = ops.backproject(y.to(gpu), g, mode, norm=norm, out=base.clone())
    ref = oracle.backproject(prob, y.float().numpy(), vol, mode=mode, norm=norm)
    assert rel((out.double() - base.double()).cpu(), ref) < 5e-5


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_several_tables_per_block(gpu, dt):
    # 1331 cubes and 99 views: one block per cube, three tables (48 + 48 + 3 views)
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    rng = np.random.default_rng(5)
    nv, n, det = 99, 176, (150, 220)
    ang = 2 * np.pi * np.arange(nv) / nv
    g = Geometry.circular(ang, 500.0, 0.9, (n, n, n), det)
    y = torch.from_numpy(rng.standard_normal(g.proj_shape).astype(np.float32)).to(
        getattr(torch, dt))
    out = ops.backproject(y.to(gpu), g, 2).cpu().numpy()
    for z0 in (0, 87, 174):
        prob = oracle.Problem(ang, np.full(nv, n / 2), 500.0, 0.9, vol_dim=(n, n, n),
                              vol_start=(0, 0, z0), proj_dim=det[::-1])
        ref = oracle.backproject(prob, y.float().numpy(), (2, n, n), mode=2, norm=np.ones(nv))
        assert rel(out[z0:z0 + 2], ref) < 5e-5


@pytest.mark.parametrize("nv", [1, 50])
@pytest.mark.parametrize("mode,mis", [(2, None), (0, [0.6, -0.8, 1.5, 0.02, -0.03, 0.01])])
@pytest.mark.parametrize("dt", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("pw,det", [(0.33, (40, 110)), (0.15, (100, 200))])
def test_windows_wider_than_the_tile(gpu, nv, mode, mis, dt, pw, det):
    # fine pixels: whole cubes gather all their views from global memory, partial ones some, with taps
    # over every edge of the detector; 50 views are two tables
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    rng = np.random.default_rng(nv + mode + det[0])
    ang = np.sort(rng.uniform(0, 2 * np.pi, nv))
    vol = (18, 33, 20)
    hmid = rng.uniform(7, 11, nv)
    g = Geometry.circular(ang, 70.0, pw, vol, det, hmid=hmid, misalign=mis)
    prob = oracle.Problem(ang, hmid, 70.0, pw, vol_dim=vol[::-1], proj_dim=det[::-1], mis=mis)
    y = torch.from_numpy(rng.standard_normal(g.proj_shape).astype(np.float32)).to(
        getattr(torch, dt))
    base = torch.from_numpy(rng.standard_normal(vol).astype(np.float32)).to(gpu)
    norm = rng.uniform(0.5, 1.5, nv).astype(np.float32)
    out = ops.backproject(y.to(gpu), g, mode, norm=norm, out=base.clone())
    ref = oracle.backproject(prob, y.float().numpy(), vol, mode=mode, norm=norm)
    assert rel((out.double() - base.double()).cpu(), ref) < 5e-5


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_source_inside_the_volume(gpu, mode, dt):
    # the source's plane passes through voxels, whose detector coordinates are infinite there; those a
    # voxel and more from every view's plane are compared
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    rng = np.random.default_rng(mode)
    ang = np.array([0.0, 0.5, 1.0, 1.5, 0.27]) * np.pi
    vol, det, D = (18, 33, 20), (30, 40), 8.0
    hmid = np.full(5, 9.0)
    g = Geometry.circular(ang, D, 0.5, vol, det, hmid=hmid)
    prob = oracle.Problem(ang, hmid, D, 0.5, vol_dim=vol[::-1], proj_dim=det[::-1])
    y = torch.from_numpy(rng.standard_normal(g.proj_shape).astype(np.float32)).to(
        getattr(torch, dt))
    out = ops.backproject(y.to(gpu), g, mode, norm=np.ones(5, np.float32)).cpu().numpy()
    ref = oracle.backproject(prob, y.float().numpy(), vol, mode=mode, norm=np.ones(5))
    yy, xx = np.meshgrid(np.arange(33) - 16, np.arange(20) - 10, indexing="ij")
    c = D + xx[..., None] * np.cos(ang) + yy[..., None] * np.sin(ang)
    far = np.abs(c).min(axis=-1) >= 1.0
    assert (np.abs(c).min(axis=-1) == 0.0).any() and far.sum() > 300
    assert rel(out[:, far], ref[:, far]) < 5e-5


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("angle", [0.3, 2.0, 4.4])
def test_weights_are_rounded_once(gpu, mode, angle):
    # one view of ones: every voxel holds its weight, whose table entry and last operation round it to
    # 2^-24 at most each, 3.5e-8 rms for uniform mantissas: rel. L2 < 2^-24 (the square of a reciprocal
    # in FP32 has 1.1e-7). Whole and partial cubes
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    vol, det, D = (50, 56, 60), (150, 160), 150.0
    g = Geometry.circular([angle], D, 0.9, vol, det)
    out = ops.backproject(torch.ones(g.proj_shape, device=gpu), g, mode,
                          norm=np.ones(1, np.float32)).cpu().numpy()
    yy, xx = np.meshgrid(np.arange(56) - 28.0, np.arange(60) - 30.0, indexing="ij")
    ref = (D / (D + xx * np.cos(angle) + yy * np.sin(angle))) ** mode
    assert rel(out, np.broadcast_to(ref, vol)) < 2.0 ** -24
