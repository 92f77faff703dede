"""Row filter at the edges of its FFT lengths and of its grid: the shortest and longest rows of a
length, an odd number of rows (the last has no partner in its transform), more pairs than the grid
holds at once, and a row whose values must not leak into its partner's result.

Tolerance: FP32 FFT arithmetic of at most 13 radix-2 levels per direction, two roundings of 2^-24
relative RMS each plus tables rounded to FP32: about sqrt(2 * 26 + 4) * 2^-24 / sqrt(3) = 2.6e-7;
1e-6 leaves a factor of four.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nv,nh,nw", [(331, 299, 32), (3, 5, 33), (7, 3, 64), (1, 1, 129),
                                      (5, 5, 256), (103, 61, 257), (103, 31, 600), (1, 3, 1024),
                                      (211, 13, 1025), (1, 1, 2049), (5, 113, 2500)])
def test_rows_at_the_edges(gpu, nv, nh, nw):
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    g = Geometry.circular(np.linspace(0.0, 2.0, nv), 80.0, 1.0, (4, 4, 4), (nh, nw))
    y = np.random.default_rng(nw).standard_normal(g.proj_shape).astype(np.float32)
    t = torch.from_numpy(y).to(gpu)
    q = ops.fdk_filter(t, g, 80.0, 1.0, cosine=False).cpu().numpy().reshape(-1, nw)
    y = y.reshape(-1, nw)
    rows = np.unique(np.r_[0:40, len(y) // 2, len(y) - 40:len(y)].clip(0, len(y) - 1))
    ref = oracle.rampfilter(y[rows].reshape(1, -1, nw).astype(np.float64)).reshape(-1, nw)
    err = np.linalg.norm(q[rows] - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() < 1e-6
    # all rows: against the same rows filtered in another order (other partners, blocks and rounds)
    p = torch.from_numpy(y[::-1].copy().reshape(g.proj_shape)).to(gpu)
    r = ops.fdk_filter(p, g, 80.0, 1.0, cosine=False, out=p).cpu().numpy().reshape(-1, nw)[::-1]
    diff = np.linalg.norm(r - q, axis=1) / np.linalg.norm(q, axis=1)
    assert diff.max() < 2e-6


def test_zero_row_beside_a_large_one(gpu):
    from fastcone_amd import ops
    from fastcone_amd.geometry import Geometry
    g = Geometry.circular(np.array([0.3]), 80.0, 1.0, (4, 4, 4), (2, 300))
    y = np.zeros(g.proj_shape, np.float32)
    y[0, 1] = np.random.default_rng(5).standard_normal(300)
    q = ops.fdk_filter(torch.from_numpy(y).to(gpu), g, 80.0, 1.0).cpu().numpy()
    # the partner's result is the rounding of the common transform
    assert np.abs(q[0, 0]).max() < 1e-6 * np.abs(q[0, 1]).max()
