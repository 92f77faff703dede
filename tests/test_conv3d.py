"""Hand-written conv3d kernels (MFMA) against torch.nn.functional.conv3d in FP32 on the CPU, fed
the same BF16-rounded inputs and weights. Tolerance: FP32 accumulation in a different order, and
BF16 rounding of the outputs (relative 2^-8), so rel. L2 < 1e-2 (outputs and input gradients) and
< 2e-3 (FP32 weight and bias gradients).

The whole network: its forward and backward passes against torch autograd in FP32 on the CPU with
the network's BF16 rounding points reproduced (inputs, weights, every activation and the
gradient at every convolution output), and a short training run that fits a target the network
can represent."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PAIRS = [(16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (96, 32), (48, 16)]


def rel(a, b):
    a = a.double()
    b = b.double()
    return float((a - b).norm() / b.norm())


def _torch_w(w):  # [co][27][ci] -> [co][ci][3][3][3]
    co, _, ci = w.shape
    return w.reshape(co, 3, 3, 3, ci).permute(0, 4, 1, 2, 3).contiguous()


def test_mfma_lane_layout(gpu):
    from fastcone_amd import _native
    import ctypes
    g = torch.Generator().manual_seed(0)
    A32 = torch.randn(16, 32, generator=g).to(torch.bfloat16)
    B32 = torch.randn(32, 16, generator=g).to(torch.bfloat16)
    A4 = torch.randn(16, 4, generator=g)
    B4 = torch.randn(4, 16, generator=g)
    d = {k: v.to(gpu).contiguous() for k, v in dict(A32=A32, B32=B32, A4=A4, B4=B4).items()}
    D32 = torch.zeros(16, 16, device=gpu)
    D4 = torch.zeros(16, 16, device=gpu)
    rc = _native.lib().fc_mfma_layout_probe(0, d["A32"].data_ptr(), d["B32"].data_ptr(),
                                            d["A4"].data_ptr(), d["B4"].data_ptr(),
                                            D32.data_ptr(), D4.data_ptr(),
                                            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _native.check(rc)
    torch.cuda.synchronize()
    assert torch.allclose(D32.cpu(), A32.float() @ B32.float(), rtol=1e-5, atol=1e-4)
    assert torch.allclose(D4.cpu(), A4 @ B4, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("cin,cout", PAIRS + [(1, 16), (16, 1)])
def test_conv_forward_backward(gpu, cin, cout):
    from fastcone_amd.unet import conv3d
    g = torch.Generator().manual_seed(cin * 100 + cout)
    N, D, H, W = 2, 6, 7, 20  # W not a multiple of 16: partial waves
    x = torch.randn((N, D, H, W, cin), generator=g).to(torch.bfloat16)
    w = (torch.randn((cout, 27, cin), generator=g) / np.sqrt(27 * cin))
    b = torch.randn(cout, generator=g) * 0.1
    relu = cout != 1
    xg = x.to(gpu).requires_grad_(cin != 1)
    wg = w.to(gpu).requires_grad_(True)
    bg = b.to(gpu).requires_grad_(True)
    y = conv3d(xg, wg, bg, relu)
    # reference: FP32 CPU with the BF16-rounded weights the kernel reads
    xr = x.float().permute(0, 4, 1, 2, 3).requires_grad_(True)
    wr = _torch_w(w.to(torch.bfloat16).float()).requires_grad_(True)
    br = b.clone().requires_grad_(True)
    yr = torch.nn.functional.conv3d(xr, wr, br, padding=1)
    if relu:
        yr = torch.relu(yr)
    yr_c = yr.permute(0, 2, 3, 4, 1)
    assert rel(y.float().cpu(), yr_c) < 1e-2
    gy = torch.randn(yr_c.shape, generator=g)
    # the kernel's output gradient is taken in BF16 (or FP32 for the 1-channel output)
    gy_k = gy.to(torch.bfloat16).float() if cout != 1 else gy
    (y.float() * gy_k.to(gpu)).sum().backward()
    (yr_c * gy_k).sum().backward()
    # weight and bias gradients from BF16 inputs and output gradients (products exact in FP32,
    # FP32 sums): only the summation order differs from the reference with the same rounding
    e_w = rel(wg.grad.cpu(), wr.grad.permute(0, 2, 3, 4, 1).reshape(cout, 27, cin))
    e_b = rel(bg.grad.cpu(), br.grad)
    print(f"conv {cin}->{cout}: weight gradient {e_w:.1e}, bias gradient {e_b:.1e}")
    assert e_w < 2e-3 and e_b < 2e-3
    if cin != 1:
        # the input gradient is stored in BF16 (relative rounding 2^-9)
        assert rel(xg.grad.float().cpu(), xr.grad.permute(0, 2, 3, 4, 1)) < 1e-2


def test_unet_matches_fp32_reference(gpu):
    from fastcone_amd.unet import UNet3D, LAYERS
    net = UNet3D(seed=1).to(gpu)
    g = torch.Generator().manual_seed(2)
    vol = (torch.rand((2, 16, 16, 16), generator=g) * 0.02).to(gpu)
    out = net(vol)
    # FP32 reference with the same BF16-rounded weights
    W = {k: _torch_w(v.detach().to(torch.bfloat16).float().cpu()) for k, v in net.w.items()}
    B = {k: v.detach().float().cpu() for k, v in net.b.items()}
    F = torch.nn.functional

    def c(x, n, relu=True):
        y = F.conv3d(x, W[n], B[n], padding=1)
        return torch.relu(y) if relu else y

    x = (vol.cpu() * UNet3D.SCALE)[:, None]
    e1 = c(c(x, "e1a"), "e1b")
    e2 = c(c(F.avg_pool3d(e1, 2), "e2a"), "e2b")
    bt = c(c(F.avg_pool3d(e2, 2), "b_a"), "b_b")
    up = lambda t: t.repeat_interleave(2, 2).repeat_interleave(2, 3).repeat_interleave(2, 4)
    d2 = c(c(torch.cat([up(bt), e2], 1), "d2a"), "d2b")
    d1 = c(c(torch.cat([up(d2), e1], 1), "d1a"), "d1b")
    ref = vol.cpu() + c(d1, "out", relu=False)[:, 0] / UNet3D.SCALE
    corr = out.detach().cpu() - vol.cpu()
    corr_ref = ref - vol.cpu()
    assert rel(corr, corr_ref) < 5e-2


@pytest.mark.parametrize("cin,cout", [(16, 16), (32, 64)])
def test_weight_gradient_long_rows(gpu, cin, cout):
    # rows longer than the 256 voxels the weight-gradient kernel stages at once (300 = 256 + 44)
    from fastcone_amd import _native
    g = torch.Generator().manual_seed(7 + cin + cout)
    N, D, H, W = 1, 3, 4, 300
    x = torch.randn((N, D, H, W, cin), generator=g).to(torch.bfloat16)
    gy = torch.randn((N, D, H, W, cout), generator=g).to(torch.bfloat16)
    dw = torch.zeros((cout, 27, cin), dtype=torch.float32, device=gpu)
    xg, gyg = x.to(gpu).contiguous(), gy.to(gpu).contiguous()
    L = _native.lib()
    s = torch.cuda.current_stream(gpu).cuda_stream
    import ctypes
    _native.check(L.fc_conv3d_wgrad_dev(gpu.index, xg.data_ptr(), gyg.data_ptr(), dw.data_ptr(),
                                        N, D, H, W, cin, cout, ctypes.c_void_p(int(s))))
    torch.cuda.synchronize()
    # reference: d/dw of sum(conv3d(x, w) * gy) in FP32 on the CPU
    w0 = torch.zeros((cout, cin, 3, 3, 3), requires_grad=True)
    y = torch.nn.functional.conv3d(x.float().permute(0, 4, 1, 2, 3), w0, padding=1)
    (y * gy.float().permute(0, 4, 1, 2, 3)).sum().backward()
    ref = w0.grad.permute(0, 2, 3, 4, 1).reshape(cout, 27, cin)
    assert rel(dw.cpu(), ref) < 2e-3


class _RoundBF16(torch.autograd.Function):
    """Forward: round to BF16; backward: round the gradient to BF16 (the U-Net's activations and
    the output gradients its convolution kernels read are BF16)."""

    @staticmethod
    def forward(ctx, x):
        return x.to(torch.bfloat16).float()

    @staticmethod
    def backward(ctx, g):
        return g.to(torch.bfloat16).float()


def _reference_unet(net, vol):
    """FP32 CPU autograd restatement of UNet3D.forward with the same BF16 rounding points;
    returns (output, {layer: weight tensor in torch layout}, {layer: bias})."""
    from fastcone_amd.unet import UNet3D, LAYERS
    F = torch.nn.functional
    W = {k: _torch_w(v.detach().to(torch.bfloat16).float().cpu()).requires_grad_(True)
         for k, v in net.w.items()}
    B = {k: v.detach().float().cpu().requires_grad_(True) for k, v in net.b.items()}
    R = _RoundBF16.apply

    def c(x, n):
        relu = next(L[3] for L in LAYERS if L[0] == n)
        y = F.conv3d(x, W[n], B[n], padding=1)
        return R(torch.relu(y)) if relu else y

    x = R(vol.cpu() * UNet3D.SCALE)[:, None]
    e1 = c(c(x, "e1a"), "e1b")
    e2 = c(c(R(F.avg_pool3d(e1, 2)), "e2a"), "e2b")
    bt = c(c(R(F.avg_pool3d(e2, 2)), "b_a"), "b_b")
    up = lambda t: t.repeat_interleave(2, 2).repeat_interleave(2, 3).repeat_interleave(2, 4)
    d2 = c(c(torch.cat([up(bt), e2], 1), "d2a"), "d2b")
    d1 = c(c(torch.cat([up(d2), e1], 1), "d1a"), "d1b")
    out = vol.cpu() + c(d1, "out")[:, 0] / UNet3D.SCALE
    return out, W, B


def test_unet_forward_and_backward_match_fp32_autograd(gpu):
    # whole-network gradients (pooling, upsampling, skip concatenations, the 1/SCALE residual
    # output) for the loss sum(out * G) with a fixed random G, so both sides receive the same
    # output gradient
    from fastcone_amd.unet import UNet3D
    net = UNet3D(seed=3).to(gpu)
    g = torch.Generator().manual_seed(4)
    vol = (torch.rand((2, 16, 16, 16), generator=g) * 0.02).to(gpu)
    G = torch.randn((2, 16, 16, 16), generator=g)
    out = net(vol)
    (out * G.to(gpu)).sum().backward()
    ref, W, B = _reference_unet(net, vol)
    (ref * G).sum().backward()
    e_fwd = rel((out.detach().cpu() - vol.cpu()).double(), (ref.detach() - vol.cpu()).double())
    print(f"U-Net correction vs FP32 autograd: {e_fwd:.1e}")
    assert e_fwd < 1e-2
    for name in net.w:
        gw = net.w[name].grad.cpu()
        gr = W[name].grad.permute(0, 2, 3, 4, 1).reshape(gw.shape)
        e_w = rel(gw, gr)
        e_b = rel(net.b[name].grad.cpu(), B[name].grad)
        print(f"  {name}: weight gradient {e_w:.1e}, bias gradient {e_b:.1e}")
        assert e_w < 3e-2 and e_b < 3e-2, name


def test_unet_training_fits_a_representable_target(gpu):
    # 8 pairs whose target differs from the input by a fixed local linear map (a 3x3x3 blur
    # minus identity): a function the network can represent. Adam at the training settings
    # (lr 1e-3) must bring the training MSE far below the identity start's, which shows that the
    # kernels' gradients drive training; a target that is not a local function of the input
    # (amplified noise) is not fitted by any such network
    from fastcone_amd.unet import UNet3D
    net = UNet3D(seed=5).to(gpu)
    g = torch.Generator(device=gpu).manual_seed(6)
    x = torch.rand((8, 32, 32, 32), device=gpu, generator=g) * 0.02
    k = torch.tensor([0.25, 0.5, 0.25], device=gpu)
    blur = (k[:, None, None] * k[None, :, None] * k[None, None, :])[None, None]
    y = torch.nn.functional.conv3d(x[:, None], blur, padding=1)[:, 0]
    y = x + 0.5 * (y - x)
    opt = torch.optim.Adam(net.parameters(), lr=1e-3)
    mse0 = float(((x - y) ** 2).mean())
    # The weight gradients are summed with float atomics, so runs differ in the last bits and
    # Adam's trajectory with them; single iterates show transient loss spikes (repeats of this
    # run gave 0.015-0.24 of the start's MSE at iteration 300 and 0.005-0.035 at 600), so the
    # check takes the best of three late iterates.
    ratios = []
    for it in range(400):
        idx = torch.arange(4, device=gpu) + 4 * (it % 2)
        loss = ((net(x[idx]) - y[idx]) ** 2).mean() * UNet3D.SCALE ** 2
        opt.zero_grad(set_to_none=True)
        loss.backward()
        opt.step()
        if it + 1 in (300, 350, 400):
            with torch.no_grad():
                ratios.append(float(((net(x) - y) ** 2).mean()) / mse0)
    print("representable target: training MSE at iterations 300, 350, 400: "
          + ", ".join(f"{r:.3f}" for r in ratios) + " of the identity start's")
    assert min(ratios) < 0.2


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 32), (48, 16), (64, 64), (96, 32)])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 5, 8, 32), (2, 9, 17, 33)])
def test_conv_tile_edges(gpu, cin, cout, shape):
    # one voxel, whole tiles, and one voxel past a tile in every direction (tiles of 16 or 32 x 8
    # voxels, chunks of planes). Both results are rounded to BF16 (relative 2^-9
    # each, the sums in FP32): rel. L2 < 2^-8
    from fastcone_amd.unet import conv3d
    g = torch.Generator().manual_seed(cin + cout + sum(shape))
    x = torch.randn(shape + (cin,), generator=g).to(torch.bfloat16)
    w = (torch.randn((cout, 27, cin), generator=g) / np.sqrt(27 * cin)).to(torch.bfloat16).float()
    gy = torch.randn(shape + (cout,), generator=g).to(torch.bfloat16)
    xg = x.to(gpu).requires_grad_(True)
    y = conv3d(xg, w.to(gpu), torch.zeros(cout, device=gpu), False)
    y.backward(gy.to(gpu))
    xr = x.float().permute(0, 4, 1, 2, 3).requires_grad_(True)
    yr = torch.nn.functional.conv3d(xr, _torch_w(w), padding=1)
    yr.backward(gy.float().permute(0, 4, 1, 2, 3))
    assert rel(y.float().cpu(), yr.detach().permute(0, 2, 3, 4, 1)) < 2.0 ** -8
    assert rel(xg.grad.float().cpu(), xr.grad.permute(0, 2, 3, 4, 1)) < 2.0 ** -8


@pytest.mark.parametrize("cin,cout", [(16, 16), (48, 16), (32, 64)])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 2, 8, 32), (2, 9, 17, 33), (1, 3, 26, 65)])
def test_weight_gradient_segment_edges(gpu, cin, cout, shape):
    # rows of one voxel, one whole segment of 32 and one voxel past a segment; one row, and row
    # chunks that leave a remainder. The products are exact in FP32 and the sums differ from the
    # FP64 reference by their FP32 rounding: below sqrt(terms) 2^-24 of the sum of magnitudes, so
    # rel. L2 < 1e-5 for these few thousand terms
    from fastcone_amd.unet import conv3d
    g = torch.Generator().manual_seed(cin + cout + sum(shape))
    x = torch.randn(shape + (cin,), generator=g).to(torch.bfloat16)
    gy = torch.randn(shape + (cout,), generator=g).to(torch.bfloat16)
    w = torch.zeros((cout, 27, cin), device=gpu, requires_grad=True)
    conv3d(x.to(gpu), w, torch.zeros(cout, device=gpu), False).backward(gy.to(gpu))
    wr = torch.zeros((cout, cin, 3, 3, 3), dtype=torch.float64, requires_grad=True)
    yr = torch.nn.functional.conv3d(x.double().permute(0, 4, 1, 2, 3), wr, padding=1)
    yr.backward(gy.double().permute(0, 4, 1, 2, 3))
    ref = wr.grad.permute(0, 2, 3, 4, 1).reshape(cout, 27, cin)
    assert rel(w.grad.cpu(), ref) < 1e-5


@pytest.mark.parametrize("shape", [(1, 2, 2, 2), (2, 4, 6, 10), (1, 6, 2, 130)])
@pytest.mark.parametrize("ca,cb", [(32, 16), (64, 32)])
def test_pool_and_up_cat_match_torch(gpu, shape, ca, cb):
    # rows shorter and longer than a block of 256 units; the layers' results are those of avgpool2,
    # upsample2 and torch.cat, and their gradients those of torch's backward pass up to one BF16
    # rounding of a sum (2^-8 relative)
    from fastcone_amd.unet import _Pool, _UpCat, avgpool2, upsample2
    N, D, H, W = shape
    g = torch.Generator().manual_seed(ca + sum(shape))
    bf = lambda *s: torch.randn(s, generator=g).to(torch.bfloat16).to(gpu)
    e, a = bf(N, D, H, W, cb), bf(N, D // 2, H // 2, W // 2, ca)
    gc, gp = bf(N, D, H, W, ca + cb), bf(N, D // 2, H // 2, W // 2, cb)
    out = []
    for ours in (True, False):
        x, y = e.clone().requires_grad_(True), a.clone().requires_grad_(True)
        skip, pool = _Pool.apply(x) if ours else (x, avgpool2(x))
        c = _UpCat.apply(y, skip) if ours else torch.cat([upsample2(y), skip], dim=-1)
        torch.autograd.backward([c, pool], [gc, gp])
        out.append((c.detach(), pool.detach(), y.grad, x.grad))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert rel(out[0][2].cpu(), out[1][2].cpu()) < 2.0 ** -8
    assert rel(out[0][3].cpu(), out[1][3].cpu()) < 2.0 ** -8


@pytest.mark.parametrize("voxels", [1, 127, 4097, 70001])
@pytest.mark.parametrize("c", [16, 32, 64])
def test_relu_gradient_kernel(gpu, voxels, c):
    # one block and several, with remainders; the masked gradient is exact, a NaN or infinite
    # gradient of a masked value is NaN, and the bias gradient differs from the FP64 sum by FP32
    # rounding: at most sqrt(voxels) 2^-24 of the sum of magnitudes
    import ctypes
    from fastcone_amd import _native
    g = torch.Generator().manual_seed(voxels + c)
    gy = torch.randn((voxels, c), generator=g).to(torch.bfloat16)
    y = torch.randn((voxels, c), generator=g).to(torch.bfloat16)
    ref = gy * (y > 0)
    gd, yd = gy.to(gpu), y.to(gpu)
    gm = torch.empty_like(gd)
    db = torch.zeros(c, device=gpu)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    L = _native.lib()
    _native.check(L.fc_net_relu_grad_dev(gpu.index, gd.data_ptr(), yd.data_ptr(), gm.data_ptr(),
                                         db.data_ptr(), voxels, c, st))
    assert torch.equal(gm.cpu(), ref)
    bound = ref.double().abs().sum(0) * (voxels ** 0.5 + 1.0) * 2.0 ** -24 + 1e-30
    assert bool(((db.double().cpu() - ref.double().sum(0)).abs() <= bound).all())
    gd[0, 0], yd[0, 0] = float("inf"), -1.0
    _native.check(L.fc_net_relu_grad_dev(gpu.index, gd.data_ptr(), yd.data_ptr(), gm.data_ptr(),
                                         db.data_ptr(), voxels, c, st))
    assert bool(gm[0, 0].isnan()) and bool(db[0].isnan())


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (1, 2, 16, 32), (2, 5, 17, 33), (1, 3, 35, 70)])
def test_one_channel_layers(gpu, shape):
    # z chunks, 32-voxel segments and 16-row chunks whole and with remainders. First layer: BF16
    # output (one rounding, 2^-9 each side: rel. L2 < 2^-8); last layer: FP32 sums of 432 exact
    # products (sqrt(432) 2^-24 = 1.2e-6, bound 1e-5), its BF16 input gradient < 2^-8; weight
    # gradients, the last layer's from FP32 output gradients with all 24 bits, < 1e-5 as above
    from fastcone_amd.unet import conv3d
    g = torch.Generator().manual_seed(sum(shape))
    for cin, cout in ((1, 16), (16, 1)):
        x = torch.randn(shape + (cin,), generator=g).to(torch.bfloat16)
        w = (torch.randn((cout, 27, cin), generator=g) / np.sqrt(27 * cin)).to(torch.bfloat16).float()
        b = torch.randn(cout, generator=g)
        gy = torch.randn(shape + (cout,), generator=g)
        gy = gy.to(torch.bfloat16) if cout != 1 else gy
        xg = x.to(gpu).requires_grad_(cin != 1)
        wg = w.to(gpu).requires_grad_(True)
        y = conv3d(xg, wg, b.to(gpu), False)
        y.backward(gy.to(gpu))
        xr = x.double().permute(0, 4, 1, 2, 3).requires_grad_(True)
        wr = _torch_w(w).double().requires_grad_(True)
        yr = torch.nn.functional.conv3d(xr, wr, b.double(), padding=1)
        yr.backward(gy.double().permute(0, 4, 1, 2, 3))
        assert rel(y.cpu(), yr.detach().permute(0, 2, 3, 4, 1)) < (1e-5 if cout == 1 else 2.0 ** -8)
        assert rel(wg.grad.cpu(), wr.grad.permute(0, 2, 3, 4, 1).reshape(cout, 27, cin)) < 1e-5
        if cin != 1:
            assert rel(xg.grad.cpu(), xr.grad.permute(0, 2, 3, 4, 1)) < 2.0 ** -8


@pytest.mark.parametrize("shape,ca,cb,cout", [((1, 2, 2, 2), 32, 16, 16), ((2, 6, 10, 36), 32, 16, 16),
                                              ((1, 34, 18, 16), 32, 16, 16), ((1, 4, 8, 34), 64, 32, 32),
                                              ((3, 2, 22, 14), 64, 32, 32)])
@pytest.mark.parametrize("offset", [0, 1])
def test_up_cat_conv_matches_its_parts(gpu, shape, ca, cb, cout, offset):
    # tiles cut by every side of the volume, several batches and z chunks, operands that start at an
    # odd element: bit for bit the convolution of the concatenation
    from fastcone_amd.unet import _UpCatConv, conv3d, upsample2
    N, D, H, W = shape
    g = torch.Generator().manual_seed(ca + sum(shape))

    def bf(*s):
        n = int(np.prod(s))
        t = torch.randn(n + offset, generator=g).to(torch.bfloat16).to(gpu)
        return t[offset:].view(s)
    a, b = bf(N, D // 2, H // 2, W // 2, ca), bf(N, D, H, W, cb)
    w = torch.randn((cout, 27, ca + cb), generator=g).to(gpu) * 0.05
    bias = torch.randn(cout, generator=g).to(gpu)
    with torch.no_grad():
        for relu in (True, False):
            ref = conv3d(torch.cat([upsample2(a), b], dim=-1).contiguous(), w, bias, relu)
            assert torch.equal(_UpCatConv.apply(a, b, w, bias, relu), ref)


@pytest.mark.parametrize("shape,ca,cb,cout", [((1, 2, 2, 2), 32, 16, 16), ((2, 6, 10, 36), 32, 16, 16),
                                              ((1, 34, 18, 70), 32, 16, 16), ((3, 4, 38, 34), 64, 32, 32)])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("relu", [True, False])
def test_up_cat_conv_gradients_match_their_parts(gpu, shape, ca, cb, cout, offset, relu):
    # rows and x segments cut by the volume, several batches and y chunks. Whole numbers: every
    # sum of the weight and bias gradients is exact in FP32 in any order, so all bits are the same
    from fastcone_amd.unet import _UpCat, _UpCatConv, conv3d
    N, D, H, W = shape
    g = torch.Generator().manual_seed(cb + sum(shape))

    def whole(*s, lim, off=0):
        n = int(np.prod(s))
        t = torch.randint(-lim, lim + 1, (n + off,), generator=g).to(torch.bfloat16).to(gpu)
        return t[off:].view(s)
    a = whole(N, D // 2, H // 2, W // 2, ca, lim=2, off=offset)
    b = whole(N, D, H, W, cb, lim=2, off=offset)
    w = whole(cout, 27, ca + cb, lim=1).float()
    bias = whole(cout, lim=3).float()
    gy = whole(N, D, H, W, cout, lim=1)
    res = []
    for ours in (True, False):
        p = [t.detach().requires_grad_(True) for t in (a, b, w, bias)]
        if ours:
            y = _UpCatConv.apply(*p, relu)
        else:  # the concatenation's operands must start on 16 bytes
            y = conv3d(_UpCat.apply(p[0].clone(), p[1].clone()), p[2], p[3], relu)
        y.backward(gy)
        res.append([y.detach()] + [t.grad for t in p])
    for u, v in zip(*res):
        assert torch.equal(u, v)


def test_bf16_weights_are_rounded_like_torch(gpu):
    # counts around a block and above one grid, special values, tensors that the kernel does not take
    from fastcone_amd.unet import _bf16_weights
    g = torch.Generator().manual_seed(4)
    ws = [torch.randn(n, generator=g).to(gpu) * 10.0 ** e
          for n, e in ((1, 0), (255, -3), (256, 3), (257, -40), (70000, 0), (7, 38))]
    ws[1][:4] = torch.tensor([float("inf"), -float("inf"), 1 + 2.0 ** -8, -0.0])
    for w, b in zip(ws, _bf16_weights(ws, gpu)):
        assert torch.equal(w.to(torch.bfloat16), b)
    assert _bf16_weights([ws[0], ws[2].double()], gpu) == [None, None]
    assert _bf16_weights([ws[0], ws[2][::2]], gpu) == [None, None]


def test_unet_without_gradients_is_the_same_network(gpu):
    from fastcone_amd.unet import UNet3D
    net = UNet3D(3).to(gpu)
    vol = torch.rand((2, 12, 20, 16), generator=torch.Generator().manual_seed(1)).to(gpu) * 0.02
    with torch.no_grad():
        y = net(vol)
    assert torch.equal(y, net(vol).detach())


@pytest.mark.parametrize("cin,cout", [(32, 32), (32, 64), (64, 64), (96, 32), (64, 32)])
@pytest.mark.parametrize("shape", [(1, 32, 64, 129), (2, 67, 33, 50), (1, 130, 20, 36), (3, 3, 120, 340)])
def test_conv_large_layers(gpu, cin, cout, shape):
    # inputs with enough tiles for the plane-by-plane kernel: tiles cut in x and y, chunks of 2 to 32
    # planes with a remainder, several batches. Every output adds its terms in the order of the tiled
    # kernel, which the same volume in pieces of few tiles runs: bit for bit (each piece with the
    # planes around it)
    from fastcone_amd.unet import conv3d
    N, D, H, W = shape
    g = torch.Generator().manual_seed(cin + cout + D)
    x = torch.randn((N, D, H, W, cin), generator=g).to(torch.bfloat16).to(gpu)
    w = torch.randn((cout, 27, cin), generator=g).to(gpu) * 0.05
    b = torch.randn(cout, generator=g).to(gpu)
    with torch.no_grad():
        y = conv3d(x, w, b, True)
        zs = torch.randint(0, D, (4,), generator=g).tolist() + [0, D - 1]
        for n in range(N):
            for z in zs:
                lo, hi = max(z - 1, 0), min(z + 2, D)
                for y0 in range(0, H, 16):
                    ya, yb = max(y0 - 1, 0), min(y0 + 17, H)
                    part = x[n:n + 1, lo:hi, ya:yb].contiguous()
                    ref = conv3d(part, w, b, True)[0, z - lo, y0 - ya:min(y0 + 16, H) - ya]
                    assert torch.equal(y[n, z, y0:y0 + 16], ref)


def test_bias_gradients_are_reproducible(gpu):
    # two passes over the same batch: the ReLU layers' bias gradients bit for bit (many blocks add to
    # each; the weight gradients are float atomics)
    from fastcone_amd.unet import UNet3D
    net = UNet3D(seed=5).to(gpu)
    x = torch.rand((2, 48, 64, 64), generator=torch.Generator().manual_seed(1)).to(gpu) * 0.02
    runs = []
    for _ in range(3):
        net.zero_grad(set_to_none=True)
        ((net(x) - 0.9 * x) ** 2).mean().mul(UNet3D.SCALE ** 2).backward()
        runs.append({k: p.grad.clone() for k, p in net.b.items()})
    for r in runs[1:]:
        assert all(torch.equal(r[k], runs[0][k]) for k in r)


@pytest.mark.parametrize("voxels", [1, 127, 4097, 70001])
@pytest.mark.parametrize("c,rows", [(16, 1024), (32, 3), (64, 65), (64, 5000)])
def test_ordered_bias_gradient(gpu, voxels, c, rows):
    # fewer and more rows of scratch than blocks, rows that are no multiple of a block's 64; bound as
    # in test_relu_gradient_kernel, and nothing written past the rows that were given
    import ctypes
    from fastcone_amd import _native
    g = torch.Generator().manual_seed(voxels + c)
    gy = torch.randn((voxels, c), generator=g).to(torch.bfloat16)
    y = torch.randn((voxels, c), generator=g).to(torch.bfloat16)
    ref = gy * (y > 0)
    gd, yd = gy.to(gpu), y.to(gpu)
    gm, part, db = torch.empty_like(gd), torch.full((rows + 1, c), 7.0, device=gpu), \
        torch.full((c,), 3.0, device=gpu)
    _native.check(_native.lib().fc_net_relu_grad_parts_dev(
        gpu.index, gd.data_ptr(), yd.data_ptr(), gm.data_ptr(), part.data_ptr(), rows,
        db.data_ptr(), voxels, c, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(gm.cpu(), ref)
    bound = ref.double().abs().sum(0) * (voxels ** 0.5 + 1.0) * 2.0 ** -24 + 1e-30
    assert bool(((db.double().cpu() - ref.double().sum(0)).abs() <= bound).all())
    assert bool((part[rows] == 7.0).all())


@pytest.mark.parametrize("cin,cout", [(16, 32), (48, 16), (1, 16), (16, 1)])
def test_output_gradient_at_an_odd_element(gpu, cin, cout):
    # without a ReLU the gradient is read where it lies: one that starts off 16 bytes gives the bits
    # of an aligned copy (whole numbers: every sum is exact)
    from fastcone_amd.unet import _UpCatConv, conv3d
    g = torch.Generator().manual_seed(cin)
    whole = lambda n, lim: torch.randint(-lim, lim + 1, (n,), generator=g).float().to(gpu)
    shape = (2, 4, 6, 34)
    x = whole(int(np.prod(shape)) * cin, 2).to(torch.bfloat16).view(shape + (cin,))
    w, b = whole(cout * 27 * cin, 1).view(cout, 27, cin), whole(cout, 2)
    gy = whole(int(np.prod(shape)) * cout + 1, 1).to(torch.float32 if cout == 1 else torch.bfloat16)
    gy = gy[1:].view(shape + (cout,))
    assert gy.is_contiguous() and gy.data_ptr() % 16
    coarse = whole(int(np.prod(shape)) // 8 * 32, 2).to(torch.bfloat16).view(2, 2, 3, 17, 32)
    res = []
    for grad in (gy, gy.clone()):
        if cin == 48:
            p = [t.detach().requires_grad_(True) for t in (coarse, x[..., 32:].contiguous(), w, b)]
            y = _UpCatConv.apply(*p, False)
        else:
            # the first layer's input has no gradient
            p = [t.detach().requires_grad_(t is not x or cin > 1) for t in (x, w, b)]
            y = conv3d(*p, False)
        y.backward(grad)
        res.append([t.grad for t in p if t.requires_grad])
    for u, v in zip(*res):
        assert torch.equal(u, v)


@pytest.mark.parametrize("skip", ["expanded", "transposed", "none"])
@pytest.mark.parametrize("pooled", ["expanded", "dense"])
def test_pool_gradient_layouts(gpu, skip, pooled):
    # gradients as autograd hands them over: one value per channel for all voxels (the gradient of a
    # sum over voxels), another order of the axes, none at all; against avgpool2 and the tensor itself
    from fastcone_amd.unet import _Pool, avgpool2
    g = torch.Generator().manual_seed(3)
    bf = lambda *s: torch.randn(s, generator=g).to(torch.bfloat16).to(gpu)
    shape, coarse = (2, 4, 6, 8, 16), (2, 2, 3, 4, 16)
    e = bf(*shape)
    gs = {"expanded": bf(16).expand(shape), "none": None,
          "transposed": bf(2, 4, 8, 6, 16).transpose(2, 3)}[skip]
    gp = bf(16).expand(coarse) if pooled == "expanded" else bf(*coarse)
    grads = []
    for ours in (True, False):
        x = e.clone().requires_grad_(True)
        y, p = _Pool.apply(x) if ours else (x * 1.0, avgpool2(x))
        torch.autograd.backward([p] if gs is None else [y, p], [gp] if gs is None else [gs, gp])
        grads.append(x.grad)
    assert rel(grads[0].cpu(), grads[1].cpu()) < 2.0 ** -8


@pytest.mark.parametrize("cin,cout", [(1, 16), (16, 1), (16, 32), (48, 16)])
@pytest.mark.parametrize("where", [(0, 0, 0, 0), (1, 2, 16, 33), (0, 1, 16, 0), (1, 1, 7, 31)])
@pytest.mark.parametrize("operand", ["input", "gradient"])
def test_weight_gradients_of_infinite_values(gpu, cin, cout, where, operand):
    # an infinite value reaches the taps that it is a term of, and not those that lie in the padding
    # there; segments of 32 voxels and one past, volume borders and none. Reference: FP64 sums over
    # the voxels of each tap that lie in the volume; finite ones < 1e-5 as above
    from fastcone_amd.unet import conv3d
    g = torch.Generator().manual_seed(cin + sum(where))
    shape = (2, 3, 17, 34)
    _, D, H, W = shape
    x = torch.randn(shape + (cin,), generator=g).to(torch.bfloat16)
    gy = torch.randn(shape + (cout,), generator=g)
    gy = gy.to(torch.bfloat16) if cout != 1 else gy
    (x if operand == "input" else gy)[where + (0,)] = float("inf")
    w = torch.zeros((cout, 27, cin), device=gpu, requires_grad=True)
    conv3d(x.to(gpu), w, torch.zeros(cout, device=gpu), False).backward(gy.to(gpu))
    dw = w.grad.cpu().double()
    ref = torch.empty_like(dw)
    cut = lambda d, n: (slice(max(0, -d), n - max(0, d)), slice(max(0, d), n + min(0, d)))
    for tap in range(27):
        z, y, xx = (cut(tap // 9 - 1, D), cut(tap // 3 % 3 - 1, H), cut(tap % 3 - 1, W))
        a = gy[:, z[0], y[0], xx[0]].double()
        b = x[:, z[1], y[1], xx[1]].double()
        ref[:, tap] = (a[..., :, None] * b[..., None, :]).sum((0, 1, 2, 3))
    finite = ref.isfinite()
    assert not bool(finite.all())
    assert torch.equal(dw[~finite], ref[~finite])
    if bool(finite.any()):  # not with one input channel and its infinite value inside
        assert rel(dw[finite], ref[finite]) < 1e-5
