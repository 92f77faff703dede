"""Helical cone beam on a cylindrical detector and exact Katsevich reconstruction.

CPU: the oracle's helical projector against closed-form ellipsoid line integrals, and the
oracle's Katsevich reconstruction of analytic projections against the phantom (exactness of the
method inside the reconstructable region pins every filtering stage, its sign and its scale).
GPU: libFastcone's helical projector and fc_katsevich_dev against the oracle on the same data,
then configuration 2 at full size.
"""
import math

import numpy as np
import pytest

import oracle

# a small helix: R = 100, SDD = 200 voxels, 96 x 32 curved detector, pitch 0.8 x detector height
R, SDD, NW, NH, DG, DROW = 100.0, 200.0, 96, 32, 0.0052, 1.0
PITCH = 0.8 * NH * DROW * R / SDD
HP = PITCH / (2 * math.pi)
VPT, TURNS = 360, 3
N = 32
ORIGIN = np.array([-16.0, -16.0, -16.0])
ELL = [(np.array([1.5, -2.0, 0.5]), np.array([12.0, 10.0, 9.0]), np.eye(3), 1.0),
       (np.array([-4.0, 3.0, 1.0]), np.array([3.0, 3.0, 3.0]), np.eye(3), 0.5)]


def small_helix():
    lam = 2 * math.pi * np.arange(VPT * TURNS) / VPT
    zs = HP * (lam - lam.mean())
    return oracle.Helix(lam, zs, R, SDD, DG, DROW, NW, NH, HP)


def analytic_projections(hx):
    proj = np.zeros((hx.n, hx.nh, hx.nw))
    for t in range(hx.n):
        a, pts = hx.ray_points(t)
        proj[t] = oracle.ellipsoid_line_integrals(a, pts, ELL)
    return proj


def phantom_grid():
    zz, yy, xx = np.meshgrid(*(np.arange(N) + o for o in ORIGIN[::-1]), indexing="ij")
    truth = np.zeros((N, N, N))
    inner = np.zeros((N, N, N), bool)
    for c, ax, _, mu in ELL:
        q = ((xx - c[0]) / ax[0]) ** 2 + ((yy - c[1]) / ax[1]) ** 2 + ((zz - c[2]) / ax[2]) ** 2
        truth += mu * (q <= 1)
    # voxels at least ~2 voxels from every ellipsoid surface, inside the reconstructable slab
    d = np.full((N, N, N), np.inf)
    for c, ax, _, mu in ELL:
        q = np.sqrt(((xx - c[0]) / ax[0]) ** 2 + ((yy - c[1]) / ax[1]) ** 2
                    + ((zz - c[2]) / ax[2]) ** 2)
        d = np.minimum(d, np.abs(q - 1) * ax.min())
    inner = (d > 2.0) & (np.abs(zz) < 6) & (np.hypot(xx, yy) < 14)
    return truth, inner


def test_oracle_helical_projector_matches_analytic():
    from fastcone_amd import phantom
    hx = small_helix()
    sub = oracle.Helix(hx.lambdas[::90], hx.zs[::90], R, SDD, DG, DROW, NW, NH, HP)
    ana = analytic_projections(sub)
    vol = phantom.voxelize(ELL, (N, N, N), 1.0).numpy().astype(np.float64)
    p = oracle.project_helical(sub, vol, ORIGIN, h=0.25)
    mask = ana > 0.5 * ana.max()
    assert np.median(np.abs(p[mask] - ana[mask]) / ana[mask]) < 0.02
    assert np.linalg.norm(p - ana) / np.linalg.norm(ana) < 0.06


def test_oracle_katsevich_reconstructs_analytic_phantom():
    hx = small_helix()
    proj = analytic_projections(hx)
    rec = oracle.katsevich(hx, proj, (N, N, N), ORIGIN)
    truth, inner = phantom_grid()
    err = np.abs(rec - truth)[inner]
    print(f"oracle Katsevich: interior max |err| {err.max():.3f}, mean {err.mean():.4f}")
    assert inner.sum() > 2000
    assert err.mean() < 0.01 and err.max() < 0.08


# ---- GPU -------------------------------------------------------------------------------------

def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b))


@pytest.mark.gpu
def test_helical_projector_parity(gpu):
    import torch
    from fastcone_amd import ops
    from fastcone_amd.katsevich import HelixScan
    hx = small_helix()
    scan = HelixScan(hx.n, hx.dl, hx.lambdas[0], hx.zs[0], HP, R, SDD, DG, DROW, NW, NH)
    g = scan.geometry((N, N, N))
    sub = slice(0, hx.n, 37)
    gs = g.subset(sub)
    rng = np.random.default_rng(0)
    x = rng.standard_normal((N, N, N)).astype(np.float32)
    p = ops.project(torch.from_numpy(x).to(gpu), gs, step=0.5).cpu().numpy()
    hs = oracle.Helix(hx.lambdas[sub], hx.zs[sub], R, SDD, DG, DROW, NW, NH, HP)
    ref = oracle.project_helical(hs, x, ORIGIN, h=0.5)
    assert _rel(p, ref) < 5e-5



@pytest.mark.gpu
def test_helical_adjoint_dot_product(gpu):
    # cylindrical records take the adjoint's whole-detector windows; the pair must stay matched
    import torch
    from fastcone_amd import ops
    from fastcone_amd.katsevich import HelixScan
    hx = small_helix()
    scan = HelixScan(hx.n, hx.dl, hx.lambdas[0], hx.zs[0], HP, R, SDD, DG, DROW, NW, NH)
    gs = scan.geometry((N, N, N)).subset(slice(0, hx.n, 53))
    rng = np.random.default_rng(3)
    x = torch.from_numpy(rng.standard_normal((N, N, N)).astype(np.float32)).to(gpu)
    y = torch.from_numpy(rng.standard_normal(gs.proj_shape).astype(np.float32)).to(gpu)
    ax = ops.project(x, gs, step=0.5)
    aty = ops.adjoint(y, gs, step=0.5)
    lhs = float((ax.double() * y.double()).sum())
    rhs = float((x.double() * aty.double()).sum())
    assert abs(lhs - rhs) / abs(lhs) < 1e-5

@pytest.mark.gpu
def test_katsevich_parity(gpu):
    import torch
    from fastcone_amd.katsevich import HelixScan, katsevich
    hx = small_helix()
    scan = HelixScan(hx.n, hx.dl, hx.lambdas[0], hx.zs[0], HP, R, SDD, DG, DROW, NW, NH)
    proj = analytic_projections(hx)
    rec, g5 = katsevich(torch.from_numpy(proj.astype(np.float32)).to(gpu), scan, (N, N, N),
                        origin=tuple(ORIGIN), return_filtered=True)
    ref, g5_ref = oracle.katsevich(hx, proj, (N, N, N), ORIGIN, return_g5=True)
    e_f = _rel(g5.cpu().numpy(), g5_ref)
    e_v = _rel(rec.cpu().numpy(), ref)
    truth, inner = phantom_grid()
    e_p = float(np.abs(rec.cpu().numpy() - truth)[inner].mean())
    print(f"Katsevich GPU vs FP64 oracle: filtered rel L2 {e_f:.2e}, volume rel L2 {e_v:.2e}; "
          f"interior mean |err| vs phantom {e_p:.4f}")
    assert e_f < 1e-4
    assert e_v < 1e-3
    assert e_p < 0.01


@pytest.mark.gpu
@pytest.mark.parametrize("nw,nh,dg,drow,nz,ny,nx,origin,vpt", [
    (96, 32, 0.0052, 1.0, 9, 17, 33, (-16.0, -8.0, -4.0), 90),     # ragged tiles and slabs
    (96, 12, 0.0052, 1.0, 16, 32, 32, (-16.0, -16.0, -8.0), 90),   # detector shorter than the window
    (40, 32, 0.0052, 1.0, 8, 40, 40, (-20.0, -20.0, -4.0), 90),    # columns off the detector
    (480, 160, 0.00104, 0.2, 12, 20, 20, (-10.0, -10.0, -6.0), 60),  # windows too large for the LDS
    (96, 32, 0.0052, 1.0, 20, 16, 16, (74.0, -8.0, -10.0), 90),    # close to the source path
    (64, 24, 0.008, 2.0, 318, 138, 139, (-69.0, -69.0, -159.0), 24),  # four slabs per block
])
def test_katsevich_backprojector_branches(gpu, nw, nh, dg, drow, nz, ny, nx, origin, vpt):
    """Every branch of the backprojector against the oracle, on smooth data (a random field over
    about eight views, rows and columns). A view that a voxel meets exactly at its window's edge (by
    symmetry: voxels on the axis, with a view at a quarter turn) counts or not by rounding, in FP64 as
    in FP32: voxels that differ by more than 1e-4 of the largest value must be such (next to the
    source FP32 coordinates are good to 3 * 2^-24 R, that is 4e-4 of a row or 1e-4 of these data's
    amplitude at one voxel's distance), every other agrees within the filtered data's tolerance of
    test_katsevich_parity."""
    import torch
    from fastcone_amd.katsevich import HelixScan, katsevich
    hp = 0.8 * nh * drow * R / SDD / (2 * math.pi)
    lam = 2 * math.pi * np.arange(2 * vpt) / vpt
    hx = oracle.Helix(lam, hp * (lam - lam.mean()), R, SDD, dg, drow, nw, nh, hp)
    rng = np.random.default_rng(nw + nh)
    k, i, j = np.meshgrid(np.arange(hx.n), np.arange(nh), np.arange(nw), indexing="ij")
    proj = sum(rng.normal() * np.cos(0.1 * rng.normal() * k + 6.0 / nh * rng.normal() * i
                                     + 9.0 / nw * rng.normal() * j) for _ in range(4))
    scan = HelixScan(hx.n, hx.dl, hx.lambdas[0], hx.zs[0], hp, R, SDD, dg, drow, nw, nh)
    rec, g5 = katsevich(torch.from_numpy(proj.astype(np.float32)).to(gpu), scan, (nz, ny, nx),
                        origin=origin, return_filtered=True)
    rec = rec.cpu().numpy().astype(np.float64)
    ref, g5_ref = oracle.katsevich(hx, proj, (nz, ny, nx), np.array(origin), return_g5=True)
    assert _rel(g5.cpu().numpy(), g5_ref) < 1e-4
    off = np.abs(rec - ref) > 1e-4 * np.abs(ref).max()
    assert np.linalg.norm((rec - ref)[~off]) < 1e-4 * np.linalg.norm(ref)
    assert off.sum() < 20
    for z, y, x in np.argwhere(off):
        px, py, pz = x + origin[0], y + origin[1], z + origin[2]
        v = R - px * np.cos(hx.lambdas) - py * np.sin(hx.lambdas)
        u = py * np.cos(hx.lambdas) - px * np.sin(hx.lambdas)
        gam = np.arctan2(u, v)
        dist = np.hypot(u, v)
        row = SDD * (pz - hx.zs) / dist / drow
        edge = SDD * hp / R / drow / np.cos(gam) * np.stack([math.pi / 2 - gam, -math.pi / 2 - gam])
        # FP32 coordinates relative to the source are good to about three roundings of R
        rel = 1e-6 + 3 * 2.0**-24 * R / dist
        tol = rel * (np.abs(row) + np.abs(edge) * (1 + np.abs(np.tan(gam)))
                     + SDD * hp / R / drow / np.cos(gam))
        assert (np.abs(row - edge) < tol).any()


@pytest.mark.gpu
@pytest.mark.parametrize("dg,drow", [(0.0009, 0.5), (0.0016, 1.0)])
def test_katsevich_wide_windows_by_parts(gpu, dg, drow):
    """Views whose windows are wider than the LDS buffers (all, or those near the source), in blocks of
    four slabs, against the same volume in parts of a slab per block: the same samples in the same
    order, so the same bits."""
    import torch
    from fastcone_amd.katsevich import HelixScan, katsevich
    n, nz, nh, vpt = 240, 128, 64, 200
    nw = int(0.72 / dg)
    hp = 0.8 * nh * drow * 500.0 / 900.0 / (2 * math.pi)
    dl = 2 * math.pi / vpt
    views = 3 * vpt
    scan = HelixScan(views, dl, 0.0, -hp * dl * (views - 1) / 2, hp, 500.0, 900.0, dg, drow, nw, nh)
    proj = torch.randn((views, nh, nw), generator=torch.Generator().manual_seed(nw)).to(gpu)
    whole = katsevich(proj, scan, (nz, n, n))
    for z in (0, 64):
        part = katsevich(proj, scan, (64, n, n), origin=(-(n // 2), -(n // 2), z - nz // 2))
        assert torch.equal(whole[z:z + 64], part)
    assert bool(whole.abs().sum() > 0)
