"""Small 3D U-Net that gives CGLS a warm start, on libFastcone's hand-written conv3d kernels.

Architecture (3 levels, 16 / 32 / 64 channels, 3x3x3 convolutions, ReLU, BF16 weights and
activations with FP32 accumulation): two convolutions per level, 2x2x2 average pooling down,
nearest-neighbour upsampling up with channel concatenation of the skip connection, a final
3x3x3 convolution to one FP32 channel added to the (scaled) input: the network predicts the
correction from the FDK reconstruction to the CGLS reconstruction.

Convolutions (forward, input gradient, weight gradient) run in fc_conv3d_* (MFMA), the decoder's,
whose concatenated input is not formed, in fc_net_up_cat_conv_dev and fc_net_up_cat_wgrad_dev;
pooling, upsampling, their gradients and the ReLU mask with the bias gradient in fc_net_*; the loss
is torch's. Master weights and
Adam state are FP32; the kernels read BF16 copies.
"""
import ctypes
import math

import numpy as np
import torch

from . import _native

LAYERS = [  # (name, cin, cout, relu)
    ("e1a", 1, 16, True), ("e1b", 16, 16, True),
    ("e2a", 16, 32, True), ("e2b", 32, 32, True),
    ("b_a", 32, 64, True), ("b_b", 64, 64, True),
    ("d2a", 96, 32, True), ("d2b", 32, 32, True),
    ("d1a", 48, 16, True), ("d1b", 16, 16, True),
    ("out", 16, 1, False),
]


def _stream(t):
    return ctypes.c_void_p(int(torch.cuda.current_stream(t.device).cuda_stream))


def _packed(t):
    """t, contiguous and 16-byte aligned (a gradient may come as any view)."""
    t = t.contiguous()
    return t.clone() if t.data_ptr() % 16 else t


def _bf16_weights(ws, device):
    """The BF16 copies the kernels read, by one launch (None each: the convolutions make theirs)."""
    if len(ws) > 16 or any(w.dtype != torch.float32 or w.device != device or
                           not w.is_contiguous() or not w.numel() for w in ws):
        return [None] * len(ws)
    n = [w.numel() for w in ws]
    out = torch.empty(sum(n), dtype=torch.bfloat16, device=device)
    _native.check(_native.lib().fc_net_weights_dev(
        device.index, (ctypes.c_void_p * len(n))(*[w.data_ptr() for w in ws]),
        (ctypes.c_longlong * len(n))(*n), len(n), out.data_ptr(), _stream(out)))
    return [t.view(w.shape) for t, w in zip(out.split(n), ws)]


def _activation(t):
    return t.dim() == 5 and t.dtype == torch.bfloat16 and t.is_contiguous()


def _check_weights(w32, wb):
    assert wb is None or (wb.dtype == torch.bfloat16 and wb.is_contiguous() and
                          wb.shape == w32.shape and wb.device == w32.device)


def _check_up_cat(a, b):
    N, D, H, W, _ = b.shape
    assert _activation(a) and _activation(b) and a.device == b.device
    n, d, h, w, _ = a.shape
    assert n == N and 2 * d == D and 2 * h == H and 2 * w == W


class _Conv(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w32, b32, cin, cout, relu, wb=None):
        N, D, H, W, C = x.shape
        assert C == cin and x.dtype == torch.bfloat16 and x.is_contiguous()
        if wb is None:
            wb = w32.to(torch.bfloat16).contiguous()
        odt = torch.float32 if cout == 1 else torch.bfloat16
        y = torch.empty((N, D, H, W, cout), dtype=odt, device=x.device)
        L = _native.lib()
        rc = L.fc_conv3d_fwd_dev(x.device.index, x.data_ptr(), wb.data_ptr(), b32.data_ptr(),
                                 y.data_ptr(), N, D, H, W, cin, cout, 1 if relu else 0,
                                 _stream(x))
        _native.check(rc)
        ctx.save_for_backward(x, wb, y if relu else torch.empty(0, device=x.device))
        ctx.cfg = (cin, cout, relu)
        return y

    @staticmethod
    def backward(ctx, gy):
        x, wb, y = ctx.saved_tensors
        cin, cout, relu = ctx.cfg
        N, D, H, W, _ = x.shape
        gy, db = _masked(gy, y, cout, relu)
        dw = torch.zeros((cout, 27, cin), dtype=torch.float32, device=x.device)
        rc = _native.lib().fc_conv3d_wgrad_dev(x.device.index, x.data_ptr(), gy.data_ptr(),
                                               dw.data_ptr(), N, D, H, W, cin, cout, _stream(x))
        _native.check(rc)
        if db is None:
            db = gy.float().sum(dim=(0, 1, 2, 3))
        dx = _dgrad(gy, wb, x.shape, cout) if ctx.needs_input_grad[0] else None
        return dx, dw, db, None, None, None, None


def _masked(gy, y, cout, relu):
    """The gradient at the convolution's sum, and the bias gradient (None: not yet summed)."""
    if relu and gy.dtype == torch.bfloat16 and not torch.is_grad_enabled():
        # mask and bias gradient in one pass, the bias's sums in a fixed order
        g0, gy = _packed(gy), torch.empty_like(y)
        part = torch.empty((1024, cout), dtype=torch.float32, device=y.device)
        db = torch.empty(cout, dtype=torch.float32, device=y.device)
        _native.check(_native.lib().fc_net_relu_grad_parts_dev(
            y.device.index, g0.data_ptr(), y.data_ptr(), gy.data_ptr(), part.data_ptr(),
            part.shape[0], db.data_ptr(), y.numel() // cout, cout, _stream(y)))
        return gy, db
    if relu:
        gy = gy * (y > 0)
    return gy.to(torch.float32 if cout == 1 else torch.bfloat16).contiguous(), None


def _dgrad(gy, wb, shape, cout):
    N, D, H, W, cin = shape
    dx = torch.empty(shape, dtype=torch.bfloat16, device=gy.device)
    wt = torch.empty((cin * 27 * cout,), dtype=torch.bfloat16, device=gy.device)
    rc = _native.lib().fc_conv3d_dgrad_dev(gy.device.index, gy.data_ptr(), wb.data_ptr(),
                                           wt.data_ptr(), dx.data_ptr(), N, D, H, W, cin, cout,
                                           _stream(gy))
    _native.check(rc)
    return dx


def conv3d(x, w, b, relu, wb=None):
    """x: [N, D, H, W, Cin] BF16; w: [Cout, 27, Cin] FP32 (wb: its BF16 copy); b: [Cout] FP32."""
    cout, _, cin = w.shape
    _check_weights(w, wb)
    return _Conv.apply(x, w, b, cin, cout, relu, wb)


def avgpool2(x):
    N, D, H, W, C = x.shape
    return x.view(N, D // 2, 2, H // 2, 2, W // 2, 2, C).float().mean(dim=(2, 4, 6)).to(x.dtype)


def upsample2(x):
    N, D, H, W, C = x.shape
    return x[:, :, None, :, None, :, None, :].expand(N, D, 2, H, 2, W, 2, C).reshape(
        N, 2 * D, 2 * H, 2 * W, C)


class _Pool(torch.autograd.Function):
    """A level's output for its skip connection and, average-pooled (avgpool2), for the next level.
    One function for both uses, so that their gradients are added in the pooling's backward pass."""

    @staticmethod
    def forward(ctx, x):
        N, D, H, W, C = x.shape
        assert _activation(x)
        y = torch.empty((N, D // 2, H // 2, W // 2, C), dtype=x.dtype, device=x.device)
        _native.check(_native.lib().fc_net_pool_dev(x.device.index, x.data_ptr(), y.data_ptr(), N,
                                                    D, H, W, C, _stream(x)))
        return x.view_as(x), y

    @staticmethod
    def backward(ctx, gs, gp):
        N, D, H, W, C = gs.shape
        # the skip gradient is a channel slice of the concatenation's: voxels at a fixed pitch
        pitch = gs.stride(3)
        if gs.stride() != (D * H * W * pitch, H * W * pitch, W * pitch, pitch, 1) or pitch % 8 \
                or pitch < C or gs.data_ptr() % 16:
            gs, pitch = _packed(gs), C
        gp = _packed(gp)
        g = torch.empty((N, D, H, W, C), dtype=gs.dtype, device=gs.device)
        _native.check(_native.lib().fc_net_skip_pool_grad_dev(
            gs.device.index, gs.data_ptr(), pitch, gp.data_ptr(), g.data_ptr(), N, D, H, W, C,
            _stream(gs)))
        return g


class _UpCat(torch.autograd.Function):
    """upsample2(a) and b concatenated along the channels."""

    @staticmethod
    def forward(ctx, a, b):
        N, D, H, W, cb = b.shape
        _check_up_cat(a, b)
        ctx.ca = a.shape[4]
        out = torch.empty((N, D, H, W, ctx.ca + cb), dtype=b.dtype, device=b.device)
        _native.check(_native.lib().fc_net_up_cat_dev(b.device.index, a.data_ptr(), b.data_ptr(),
                                                      out.data_ptr(), N, D, H, W, ctx.ca, cb,
                                                      _stream(b)))
        return out

    @staticmethod
    def backward(ctx, g):
        return _up_cat_grad(_packed(g), ctx.ca)


def _up_cat_grad(g, ca):
    N, D, H, W, C = g.shape
    ga = torch.empty((N, D // 2, H // 2, W // 2, ca), dtype=g.dtype, device=g.device)
    _native.check(_native.lib().fc_net_up_cat_grad_dev(g.device.index, g.data_ptr(), ga.data_ptr(),
                                                       N, D, H, W, ca, C - ca, _stream(g)))
    return ga, g[..., ca:]


class _UpCatConv(torch.autograd.Function):
    """conv3d of _UpCat; the concatenation is not formed, the kernels load from both tensors."""

    @staticmethod
    def forward(ctx, a, b, w32, b32, relu, wb=None):
        N, D, H, W, cb = b.shape
        cout, _, cin = w32.shape
        _check_up_cat(a, b)
        assert a.shape[4] + cb == cin
        _check_weights(w32, wb)
        if wb is None:
            wb = w32.to(torch.bfloat16).contiguous()
        y = torch.empty((N, D, H, W, cout), dtype=b.dtype, device=b.device)
        _native.check(_native.lib().fc_net_up_cat_conv_dev(
            b.device.index, a.data_ptr(), b.data_ptr(), wb.data_ptr(), b32.data_ptr(),
            y.data_ptr(), N, D, H, W, cin - cb, cb, cout, 1 if relu else 0, _stream(b)))
        ctx.save_for_backward(a, b, wb, y if relu else torch.empty(0, device=b.device))
        ctx.relu = relu
        return y

    @staticmethod
    def backward(ctx, gy):
        a, b, wb, y = ctx.saved_tensors
        N, D, H, W, cb = b.shape
        cout, _, cin = wb.shape
        gy, db = _masked(gy, y, cout, ctx.relu)
        dw = torch.zeros((cout, 27, cin), dtype=torch.float32, device=b.device)
        _native.check(_native.lib().fc_net_up_cat_wgrad_dev(
            b.device.index, a.data_ptr(), b.data_ptr(), gy.data_ptr(), dw.data_ptr(), N, D, H, W,
            cin - cb, cb, cout, _stream(b)))
        if db is None:
            db = gy.float().sum(dim=(0, 1, 2, 3))
        ga = gb = None
        if ctx.needs_input_grad[0] or ctx.needs_input_grad[1]:
            ga, gb = _up_cat_grad(_dgrad(gy, wb, (N, D, H, W, cin), cout), cin - cb)
        return ga, gb, dw, db, None, None


class UNet3D(torch.nn.Module):
    SCALE = 50.0  # attenuation per voxel ~ 0.02 -> O(1) activations

    def __init__(self, seed=0):
        super().__init__()
        g = torch.Generator().manual_seed(seed)
        self.w = torch.nn.ParameterDict()
        self.b = torch.nn.ParameterDict()
        for name, cin, cout, relu in LAYERS:
            std = math.sqrt(2.0 / (27 * cin)) if relu else 1e-3
            self.w[name] = torch.nn.Parameter(torch.randn((cout, 27, cin), generator=g) * std)
            self.b[name] = torch.nn.Parameter(torch.zeros(cout))

    def _c(self, x, name, wb):
        _, cin, cout, relu = next(L for L in LAYERS if L[0] == name)
        return _Conv.apply(x, self.w[name], self.b[name], cin, cout, relu, wb[name])

    def _up(self, a, b, name, wb):
        relu = next(L for L in LAYERS if L[0] == name)[3]
        # the kernel that forms no concatenation counts a plane's elements in 32 bits
        if b.shape[2] * b.shape[3] * a.shape[4] >= 2 ** 31:
            return self._c(_UpCat.apply(a, b), name, wb)
        return _UpCatConv.apply(a, b, self.w[name], self.b[name], relu, wb[name])

    def forward(self, vol):
        """vol: [N, D, H, W] (or [D, H, W]) FP32 FDK reconstruction -> FP32 prediction of the
        same shape."""
        single = vol.dim() == 3
        if single:
            vol = vol[None]
        for s in vol.shape[1:]:
            if s % 4:
                raise ValueError("volume sides must be multiples of 4")
        x = (vol * self.SCALE).to(torch.bfloat16)[..., None].contiguous()
        names = [L[0] for L in LAYERS]
        wb = dict(zip(names, _bf16_weights([self.w[n] for n in names], x.device)))
        e1, p1 = _Pool.apply(self._c(self._c(x, "e1a", wb), "e1b", wb))
        e2, p2 = _Pool.apply(self._c(self._c(p1, "e2a", wb), "e2b", wb))
        bt = self._c(self._c(p2, "b_a", wb), "b_b", wb)
        d2 = self._c(self._up(bt, e2, "d2a", wb), "d2b", wb)
        d1 = self._c(self._up(d2, e1, "d1a", wb), "d1b", wb)
        out = vol + self._c(d1, "out", wb)[..., 0] / self.SCALE
        return out[0] if single else out

    def save(self, path):
        np.savez(path, **{f"w_{k}": v.detach().cpu().numpy() for k, v in self.w.items()},
                 **{f"b_{k}": v.detach().cpu().numpy() for k, v in self.b.items()})

    def load(self, path):
        z = np.load(path)
        with torch.no_grad():
            for k in self.w:
                self.w[k].copy_(torch.from_numpy(z[f"w_{k}"]))
                self.b[k].copy_(torch.from_numpy(z[f"b_{k}"]))
        return self


def bench(batch=4, train_n=128, infer_n=256, warmup=6, steps=3, log=print):
    """Times a training step (Adam, L2 loss, batch `batch` of train_n^3 random volumes) and one
    inference at infer_n^3 on the current GPU; returns (step ms, inference ms)."""
    import time
    dev = torch.device("cuda", torch.cuda.current_device())
    net = UNet3D(seed=0).to(dev)
    opt = torch.optim.Adam(net.parameters(), lr=1e-3)
    g = torch.Generator(device=dev).manual_seed(0)
    x = torch.rand((batch,) + (train_n,) * 3, device=dev, generator=g) * 0.02
    y = x + 0.001 * torch.randn(x.shape, device=dev, generator=g)

    def train_step():
        loss = ((net(x) - y) ** 2).mean() * UNet3D.SCALE ** 2
        opt.zero_grad(set_to_none=True)
        loss.backward()
        opt.step()

    for _ in range(warmup):
        train_step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        train_step()
    torch.cuda.synchronize()
    step_ms = (time.perf_counter() - t0) / steps * 1e3
    with torch.no_grad():
        v = torch.rand((infer_n,) * 3, device=dev, generator=g) * 0.02
        net(v)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        net(v)
        torch.cuda.synchronize()
    infer_ms = (time.perf_counter() - t0) * 1e3
    log(f"train step (batch {batch}, {train_n}^3): {step_ms:.1f} ms; "
        f"inference ({infer_n}^3): {infer_ms:.1f} ms")
    return step_ms, infer_ms


if __name__ == "__main__":
    import argparse
    ap = argparse.ArgumentParser(description="time the warm-start U-Net on the GPU")
    ap.add_argument("--bench", action="store_true", help="time a training step and an inference")
    ap.add_argument("--batch", type=int, default=4)
    args = ap.parse_args()
    if args.bench:
        bench(batch=args.batch)
