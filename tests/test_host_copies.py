"""Host arrays large enough for the chunked copies (at least 4 MiB) against the same work in parts
small enough for plain ones, bit for bit: sizes of one chunk more or less than a whole number of
chunks, an odd remainder, data that the call accumulates into, and buffers given back in between. A
volume of 64 voxels a side is projected in one layout whatever the number of views, so that parts and
whole run the same arithmetic."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
pytest.importorskip("torch")


@pytest.mark.parametrize("nh,nw,nv", [(64, 128, 128), (64, 129, 128), (61, 131, 133), (96, 96, 114)])
def test_chunked_host_copies(gpu, nh, nw, nv):
    from fastcone_amd import _native
    from fastcone_amd import fastcone as cone
    rng = np.random.default_rng(nh * nw)
    vol = rng.standard_normal((64, 64, 64)).astype(np.float32)
    angles = np.linspace(0.0, 6.0, nv).astype(np.float32)
    z0 = np.full(nv, 32.0, np.float32)
    start = rng.standard_normal((nv, nh, nw)).astype(np.float32)
    assert start.nbytes >= 4 << 20
    whole, parts = start.copy(), start.copy()
    cone.project(vol, whole, angles, 300.0, z0, pixelWidth=0.8)
    for a in range(0, nv, 32):
        b = min(a + 32, nv)
        piece = np.ascontiguousarray(parts[a:b])
        assert piece.nbytes < 4 << 20
        cone.project(vol, piece, angles[a:b], 300.0, z0[a:b], pixelWidth=0.8)
        parts[a:b] = piece
    assert np.array_equal(whole, parts)
    assert _native.lib().fc_release_workspace(gpu.index or 0) == 0
    again = start.copy()
    cone.project(vol, again, angles, 300.0, z0, pixelWidth=0.8)
    assert np.array_equal(whole, again)


def test_chunked_host_volume(gpu):
    # a volume of 5.3 MB, copied in chunks both ways: without views' data it comes back as it was
    from fastcone_amd import fastcone as cone
    rng = np.random.default_rng(3)
    rec = rng.standard_normal((100, 111, 119)).astype(np.float32)
    before = rec.copy()
    proj = np.zeros((3, 40, 50), np.float32)
    cone.backproject(rec, proj, np.array([0.0, 1.0, 2.0], np.float32), 500.0,
                     np.full(3, 50.0, np.float32), pixelWidth=0.8)
    assert np.array_equal(rec, before)


@pytest.mark.parametrize("shape,nv,nh,nw", [((100, 111, 119), 130, 96, 96), ((64, 128, 129), 131, 89, 91)])
def test_chunked_backprojection(gpu, shape, nv, nh, nw):
    # a random volume and projections, both above the size that is copied in chunks, up and down,
    # against slabs and view batches small enough for plain copies: the sums are split otherwise, so
    # equal up to a few FP32 roundings of a voxel's sum of nv terms (sqrt(nv) 2^-24 < 1e-6)
    from fastcone_amd import fastcone as cone
    rng = np.random.default_rng(nv)
    start = rng.standard_normal(shape).astype(np.float32)
    proj = rng.standard_normal((nv, nh, nw)).astype(np.float32)
    assert start.nbytes >= 4 << 20 and proj.nbytes >= 4 << 20
    given = proj.copy()
    out = []
    try:
        for voxels, views in ((0, 0), (16 * shape[1] * shape[2], 40)):
            assert 4 * voxels < 4 << 20 and 4 * views * nh * nw < 4 << 20
            cone.set_tile_limits(voxels, views)
            rec = start.copy()
            cone.backproject(rec, proj, np.linspace(0.0, 6.0, nv).astype(np.float32), 500.0,
                             np.full(nv, shape[0] / 2, np.float32), pixelWidth=0.9,
                             norm=np.ones(nv, np.float32))
            out.append(rec.astype(np.float64))
    finally:
        cone.set_tile_limits(0, 0)
    added = out[1] - start
    assert np.linalg.norm(added) > np.linalg.norm(start)
    assert np.abs(out[0] - out[1]).max() < 1e-5 * np.abs(added).max()
    assert np.array_equal(proj, given)
