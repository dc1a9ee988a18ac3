"""Denoiser network kernels and the U-Net against PyTorch fp32 references
(computed on the CPU from the same bf16-rounded inputs and weights)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPEC = [(16, 32, 1), (32, 32, 1), (32, 64, 1), (64, 64, 1), (64, 128, 1), (128, 128, 1), (128, 256, 1),
        (384, 128, 1), (192, 64, 1), (96, 32, 1), (32, 32, 1), (32, 16, 0)]


def _bf16(t):
    import torch
    return t.to(torch.bfloat16)


def _layers(p):
    """(weight [Cout, Cin, 3, 3], bias) per layer from the flat parameter vector."""
    import torch
    out, off = [], 0
    for cin, cout, _ in SPEC:
        w = torch.from_numpy(p[off:off + 9 * cin * cout].reshape(3, 3, cout, cin)).permute(2, 3, 0, 1)
        off += 9 * cin * cout
        b = torch.from_numpy(p[off:off + cout])
        off += cout
        out.append((w.contiguous(), b.clone()))
    assert off == p.size
    return out


def _unet_ref(p, x, round_bf16=True):
    """fp32 U-Net on NCHW x (CPU); activations rounded to bf16 like the GPU's."""
    import torch
    import torch.nn.functional as F
    Ls = _layers(p)
    r = (lambda t: t.to(torch.bfloat16).float()) if round_bf16 else (lambda t: t)
    wr = (lambda w: w.to(torch.bfloat16).float()) if round_bf16 else (lambda w: w)

    def conv(i, t):
        w, b = Ls[i]
        y = F.conv2d(t, wr(w), b, padding=1)
        return r(torch.relu(y) if SPEC[i][2] else y)

    pool = lambda t: r(F.avg_pool2d(t, 2))
    up = lambda t: F.interpolate(t, scale_factor=2, mode="nearest")
    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, pool(e0)))
    e2 = conv(5, conv(4, pool(e1)))
    b = conv(6, pool(e2))
    d2 = conv(7, torch.cat([up(b), e2], 1))
    d1 = conv(8, torch.cat([up(d2), e1], 1))
    d0 = conv(10, conv(9, torch.cat([up(d1), e0], 1)))
    o = conv(11, d0)
    return x[:, :4] + o[:, :4]


@pytest.mark.parametrize("Cin,Cout,W,relu,cs_in,co_in,cs_out,co_out", [
    (16, 32, 70, 1, 16, 0, 32, 0),
    (32, 16, 64, 0, 48, 16, 24, 4),
    (96, 64, 40, 1, 96, 0, 96, 32),
    (64, 128, 130, 0, 64, 0, 128, 0),
])
def test_conv3x3_matches_torch(rf, gpu_available, Cin, Cout, W, relu, cs_in, co_in, cs_out, co_out):
    import torch
    import torch.nn.functional as F
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cin * 131 + Cout)
    N, H = 2, 9
    x = _bf16(torch.randn(N, H, W, cs_in, generator=g))
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g))
    b = torch.randn(Cout, generator=g)
    out = torch.zeros(N, H, W, cs_out, dtype=torch.bfloat16)
    xd, wd, bd, od = x.cuda(), w.cuda(), b.cuda(), out.cuda()
    ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, xd.data_ptr(), cs_in, co_in, wd.data_ptr(), bd.data_ptr(), od.data_ptr(),
                                  cs_out, co_out, N, H, W, Cin, Cout, relu))
    got = od.cpu().float()
    ref = F.conv2d(x[..., co_in:co_in + Cin].float().permute(0, 3, 1, 2), w.float().permute(2, 3, 0, 1), b,
                   padding=1)
    if relu:
        ref = torch.relu(ref)
    ref = ref.permute(0, 2, 3, 1)
    g_view = got[..., co_out:co_out + Cout]
    err = (g_view - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-4).all(), float(err.max())
    rest = torch.cat([got[..., :co_out], got[..., co_out + Cout:]], -1)
    assert (rest == 0).all()  # channels outside the output view are untouched


# Channel tiles of the weight gradient: 32x16 (16, 32), 32x32 (96, 32),
# 64x32 (64, 128), 16x32 (32, 16), 16x16 (48, 16); runs of rows that cross
# 64-pixel strips (W 70, 130) and images; (384, 128, 16, 16): 32 rows, 8 runs.
@pytest.mark.parametrize("Cin,Cout,W,H", [(16, 32, 70, 10), (96, 32, 40, 10), (64, 128, 24, 10),
                                          (384, 128, 16, 16), (32, 16, 130, 6), (48, 16, 33, 3)])
def test_conv3x3_gradients_match_torch(rf, gpu_available, Cin, Cout, W, H):
    import torch
    import torch.nn.functional as F
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cin + 7 * Cout)
    N = 2
    x = _bf16(torch.randn(N, H, W, Cin, generator=g))
    dy = _bf16(torch.randn(N, H, W, Cout, generator=g))
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g))
    xr = x.float().permute(0, 3, 1, 2).clone().requires_grad_(True)
    wr = w.float().permute(2, 3, 0, 1).clone().requires_grad_(True)
    br = torch.zeros(Cout, requires_grad=True)
    F.conv2d(xr, wr, br, padding=1).backward(dy.float().permute(0, 3, 1, 2))
    # weight and bias gradients
    dw = torch.zeros(3, 3, Cout, Cin, device="cuda")
    db = torch.zeros(Cout, device="cuda")
    xd, dyd = x.cuda(), dy.cuda()
    ctx.check(ctx.L.rf_nn_conv3x3_wgrad(ctx.h, xd.data_ptr(), Cin, 0, dyd.data_ptr(), Cout, 0, dw.data_ptr(),
                                        db.data_ptr(), N, H, W, Cin, Cout))
    ref_dw = wr.grad.permute(2, 3, 0, 1)
    torch.testing.assert_close(dw.cpu(), ref_dw, rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(db.cpu(), br.grad, rtol=1e-4, atol=1e-3)
    # input gradient: the same convolution kernel on flipped, transposed weights
    wt = torch.zeros(3, 3, Cin, Cout, dtype=torch.bfloat16, device="cuda")
    wd = w.cuda()
    ctx.check(ctx.L.rf_nn_flip_weights(ctx.h, wd.data_ptr(), wt.data_ptr(), Cin, Cout))
    assert torch.equal(wt.cpu(), w.flip(0, 1).permute(0, 1, 3, 2))
    dx = torch.zeros(N, H, W, Cin, dtype=torch.bfloat16, device="cuda")
    ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, dyd.data_ptr(), Cout, 0, wt.data_ptr(), None, dx.data_ptr(), Cin, 0,
                                  N, H, W, Cout, Cin, 0))
    ref_dx = xr.grad.permute(0, 2, 3, 1)
    err = (dx.cpu().float() - ref_dx).abs()
    assert (err <= 2.0 ** -8 * ref_dx.abs() + 1e-4).all(), float(err.max())


# Pixels too far apart for 32-bit offsets (views of a few channels of wide
# pixels): 64 and 32 outputs from whole channel steps of 32, and 16 from one of
# 16 in two parts; a tile at each end of the row.
@pytest.mark.parametrize("Cin,Cout", [(64, 64), (96, 32), (48, 16)])
def test_conv3x3_of_widely_spaced_pixels(rf, gpu_available, Cin, Cout):
    import torch
    import torch.nn.functional as F
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cin)
    W, cs, co = 130, 1 << 20, (1 << 20) - Cin
    near = _bf16(torch.randn(1, 1, W, Cin, generator=g))
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g)).cuda()
    b = torch.randn(Cout, generator=g).cuda()
    far = torch.empty(1, 1, W, cs, dtype=torch.bfloat16, device="cuda")
    far[..., co:] = near.cuda()
    out = []
    for x, xs, xo in ((near.cuda(), Cin, 0), (far, cs, co)):
        o = torch.zeros(1, 1, W, Cout, dtype=torch.bfloat16, device="cuda")
        ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, x.data_ptr(), xs, xo, w.data_ptr(), b.data_ptr(), o.data_ptr(), Cout, 0,
                                      1, 1, W, Cin, Cout, 0))
        out.append(o.cpu())
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
    ref = F.conv2d(near.float().permute(0, 3, 1, 2), w.float().cpu().permute(2, 3, 0, 1), b.cpu(), padding=1)
    # half a bf16 ulp, and fp32 sums of 9 Cin products
    assert ((out[0].float() - ref.permute(0, 2, 3, 1)).abs() <= 2.0 ** -8 * ref.permute(0, 2, 3, 1).abs() + 1e-4).all()


@pytest.mark.parametrize("Cout,cs", [(32, 1 << 29), (16, 1 << 29), (32, (1 << 24) + 8), (32, (1 << 24) - 8)])
def test_conv3x3_into_pixels_gigabytes_apart(rf, gpu_available, Cout, cs):
    """Narrow layers into a row of 16 GiB: its pixels' places exceed 32 bits."""
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cout)
    W, Cin = 16, 32
    x = _bf16(torch.randn(1, 1, W, Cin, generator=g)).cuda()
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g)).cuda()
    b = torch.randn(Cout, generator=g).cuda()
    near = torch.zeros(1, 1, W, Cout, dtype=torch.bfloat16, device="cuda")
    far = torch.empty(1, 1, W, cs, dtype=torch.bfloat16, device="cuda")
    far[..., cs - Cout:] = 0
    for o, os_, oo in ((near, Cout, 0), (far, cs, cs - Cout)):
        ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, x.data_ptr(), Cin, 0, w.data_ptr(), b.data_ptr(), o.data_ptr(), os_, oo,
                                      1, 1, W, Cin, Cout, 1))
    got = far[..., cs - Cout:].cpu()
    del far
    torch.cuda.empty_cache()
    assert torch.equal(near.cpu().view(torch.int16), got.view(torch.int16))


def test_conv3x3_of_pixels_gigabytes_apart(rf, gpu_available):
    """A row of 33 GiB: its pixels' places from the tile's first exceed 32 bits
    of 16-byte units."""
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(1)
    W, cs, Cin, Cout = 66, 1 << 28, 64, 64
    near = _bf16(torch.randn(1, 1, W, Cin, generator=g)).cuda()
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g)).cuda()
    b = torch.randn(Cout, generator=g).cuda()
    far = torch.empty(1, 1, W, cs, dtype=torch.bfloat16, device="cuda")
    far[..., cs - Cin:] = near
    out = []
    for x, xs, xo in ((near, Cin, 0), (far, cs, cs - Cin)):
        o = torch.zeros(1, 1, W, Cout, dtype=torch.bfloat16, device="cuda")
        ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, x.data_ptr(), xs, xo, w.data_ptr(), b.data_ptr(), o.data_ptr(), Cout, 0,
                                      1, 1, W, Cin, Cout, 0))
        out.append(o.cpu())
    del far
    torch.cuda.empty_cache()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("cs,co", [(1 << 24, (1 << 24) - 32), (36, 4), (38, 2), (40, 8)])
def test_conv3x3_wgrad_of_any_channel_stride(rf, gpu_available, cs, co):
    """Pixels too far apart for 32-bit offsets, and views that are no multiples
    of 8 channels, take 64-bit addresses: the same bits."""
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(3)
    N, H, W, Cin, Cout = 1, 5, 3, 32, 32
    x, dy = _bf16(torch.randn(N, H, W, Cin, generator=g)).cuda(), _bf16(torch.randn(N, H, W, Cout, generator=g)).cuda()
    far = torch.empty(N, H, W, cs, dtype=torch.bfloat16, device="cuda")
    far[..., co:co + Cin] = x
    out = []
    for v, xs, xo in ((x, Cin, 0), (far, cs, co)):
        dw, db = torch.zeros(3, 3, Cout, Cin, device="cuda"), torch.zeros(Cout, device="cuda")
        ctx.check(ctx.L.rf_nn_conv3x3_wgrad(ctx.h, v.data_ptr(), xs, xo, dy.data_ptr(), Cout, 0, dw.data_ptr(),
                                            db.data_ptr(), N, H, W, Cin, Cout))
        out.append((dw.cpu(), db.cpu()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


# One pixel, tiles of exactly 8 rows x 64 pixels and one more of each, images
# that end inside a tile, more tiles than workgroups, three channel blocks.
@pytest.mark.parametrize("Cin,Cout,N,H,W", [(16, 32, 1, 1, 1), (32, 32, 1, 8, 64), (32, 16, 2, 9, 65),
                                            (16, 16, 1, 17, 63), (32, 96, 2, 25, 130), (32, 32, 3, 100, 1000),
                                            (16, 32, 5, 50, 900), (32, 16, 5, 70, 1100)])
@pytest.mark.parametrize("relu", [0, 1])
def test_conv3x3_narrow_layers_have_the_general_kernels_bits(rf, gpu_available, Cin, Cout, N, H, W, relu):
    """The persistent kernel of the narrow layers sums in the general kernel's
    order: the same bits.  (An output 8 bytes off a 16-byte run takes the
    general kernel.)"""
    import torch
    import torch.nn.functional as F
    print(f"narrow conv {Cin}->{Cout} {N}x{H}x{W} relu={relu}", flush=True)
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cin + 3 * Cout + H)
    x = _bf16(torch.randn(N, H, W, Cin + 8, generator=g)).cuda()
    w = _bf16(0.1 * torch.randn(3, 3, Cout, Cin, generator=g)).cuda()
    b = torch.randn(Cout, generator=g).cuda()
    out = {}
    for cs, co in ((Cout + 16, 8), (Cout + 8, 4)):
        o = torch.zeros(N, H, W, cs, dtype=torch.bfloat16, device="cuda")
        ctx.check(ctx.L.rf_nn_conv3x3(ctx.h, x.data_ptr(), Cin + 8, 8, w.data_ptr(), b.data_ptr(), o.data_ptr(), cs, co,
                                      N, H, W, Cin, Cout, relu))
        assert not o[..., :co].any() and not o[..., co + Cout:].any()
        out[co] = o[..., co:co + Cout].cpu()
    assert torch.equal(out[8].view(torch.int16), out[4].view(torch.int16))
    ref = F.conv2d(x[..., 8:].float().cpu().permute(0, 3, 1, 2), w.float().cpu().permute(2, 3, 0, 1), b.cpu(), padding=1)
    ref = (torch.relu(ref) if relu else ref).permute(0, 2, 3, 1)
    # half a bf16 ulp, and fp32 sums of 9 Cin products
    assert ((out[8].float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4).all()


# One row, two rows, a strip of exactly 64 pixels and one more, runs that
# start inside a strip, several images: every channel tile.
@pytest.mark.parametrize("Cin,Cout,N,H,W", [(64, 64, 1, 1, 64), (32, 32, 2, 2, 65), (16, 32, 1, 3, 1),
                                            (32, 16, 5, 7, 64), (16, 16, 3, 1, 129), (64, 128, 1, 70, 64),
                                            (32, 64, 2, 37, 200)])
def test_conv3x3_wgrad_at_strip_edges(rf, gpu_available, Cin, Cout, N, H, W):
    import torch
    import torch.nn.functional as F
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(Cin + 7 * Cout + H)
    x = _bf16(torch.randn(N, H, W, Cin, generator=g))
    dy = _bf16(torch.randn(N, H, W, Cout, generator=g))
    wr = torch.zeros(Cout, Cin, 3, 3, requires_grad=True)
    br = torch.zeros(Cout, requires_grad=True)
    F.conv2d(x.float().permute(0, 3, 1, 2), wr, br, padding=1).backward(dy.float().permute(0, 3, 1, 2))
    dw = torch.zeros(3, 3, Cout, Cin, device="cuda")
    db = torch.zeros(Cout, device="cuda")
    xd, dyd = x.cuda(), dy.cuda()
    ctx.check(ctx.L.rf_nn_conv3x3_wgrad(ctx.h, xd.data_ptr(), Cin, 0, dyd.data_ptr(), Cout, 0, dw.data_ptr(),
                                        db.data_ptr(), N, H, W, Cin, Cout))
    # fp32 sums of N H W products of unit variance: their rounding stays far below 1e-3
    torch.testing.assert_close(dw.cpu(), wr.grad.permute(2, 3, 0, 1), rtol=1e-4, atol=1e-3)
    torch.testing.assert_close(db.cpu(), br.grad, rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("npix", [1, 257, 4096 + 3])
def test_log_density_input_matches_formula(rf, gpu_available, npix):
    """bf16(log10(1 + v scale)) in channels 0..3, the noise level
    bf16(log10(1 + scale)) in channel 4, zeros in 5..15; the
    one-pixel-per-thread kernel (16-byte aligned buffers) and the per-value
    kernel (an output 2 bytes off alignment) give the same bits."""
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    g = torch.Generator().manual_seed(npix)
    h = torch.rand(npix, 4, generator=g) * torch.tensor([40.0, 3.0, 0.5, 900.0])
    h[::7] = 0.0
    scale = 0.37
    hd = h.cuda()
    out_a = torch.full((npix * 16,), -1.0, dtype=torch.bfloat16, device="cuda")
    out_b = torch.full((npix * 16 + 1,), -1.0, dtype=torch.bfloat16, device="cuda")
    ctx.log_density_input(hd.data_ptr(), out_a.data_ptr(), npix, scale)
    ctx.log_density_input(hd.data_ptr(), out_b[1:].data_ptr(), npix, scale)
    a = out_a.cpu().view(npix, 16)
    b = out_b[1:].cpu().view(npix, 16)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert (a[:, 5:] == 0).all()
    nl = math.log10(1.0 + float(np.float32(scale)))
    assert (torch.abs(a[:, 4].double() - nl) <= 2.0 ** -8 * nl).all()
    ref = torch.log10(1.0 + h.double() * np.float32(scale))
    err = (a[:, :4].double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-6).all(), float(err.max())
    assert float(out_b[0].float()) == -1.0  # nothing written before the view


def test_adam_matches_formula(rf, gpu_available):
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    rng = np.random.default_rng(1)
    n = 1000
    p0 = rng.standard_normal(n).astype(np.float32)
    tp = torch.from_numpy(p0.copy()).requires_grad_(True)
    opt = torch.optim.Adam([tp], lr=1e-2, betas=(0.9, 0.999), eps=1e-8)
    p, m, v = (torch.from_numpy(p0.copy()).cuda(), torch.zeros(n, device="cuda"), torch.zeros(n, device="cuda"))
    for step in range(1, 6):
        gr = rng.standard_normal(n).astype(np.float32)
        tp.grad = torch.from_numpy(gr)
        opt.step()
        gd = torch.from_numpy(gr).cuda()
        ctx.check(ctx.L.rf_nn_adam(ctx.h, p.data_ptr(), gd.data_ptr(), m.data_ptr(), v.data_ptr(), n, 1e-2, 0.9,
                                   0.999, 1e-8, step))
    torch.testing.assert_close(p.cpu(), tp.detach(), rtol=1e-5, atol=1e-6)


def _inputs(seed, N, H, W):
    import torch
    g = torch.Generator().manual_seed(seed)
    base = torch.rand(N, 4, H // 4, W // 4, generator=g) * 2.0
    base = torch.nn.functional.interpolate(base, scale_factor=4, mode="bilinear", align_corners=False)
    x = torch.zeros(N, 16, H, W)
    x[:, :4] = (base + 0.3 * torch.randn(N, 4, H, W, generator=g)).clamp(min=0)
    t = torch.zeros(N, 16, H, W)
    t[:, :4] = base
    return _bf16(x), _bf16(t)


def test_unet_forward_matches_torch(rf, gpu_available):
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    dn = ctx.denoiser(seed=3)
    assert 1.1e6 < dn.n_params < 1.3e6
    p = dn.params()
    N, H, W = 2, 32, 48
    x, _ = _inputs(5, N, H, W)
    xd = x.permute(0, 2, 3, 1).contiguous().cuda()
    y = torch.zeros(N, H, W, 4, device="cuda")
    dn.infer(xd.data_ptr(), y.data_ptr(), N, H, W)
    ref = _unet_ref(p, x.float()).permute(0, 2, 3, 1)
    got = y.cpu()
    rel = float((got - ref).norm() / ref.norm())
    corr = (got - x.float().permute(0, 2, 3, 1)[..., :4]).flatten()
    refc = (ref - x.float().permute(0, 2, 3, 1)[..., :4]).flatten()
    assert rel < 1e-2, rel
    assert float(torch.nn.functional.cosine_similarity(corr, refc, dim=0)) > 0.99


def test_unet_gradients_match_torch(rf, gpu_available):
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    dn = ctx.denoiser(seed=4)
    p = dn.params()
    p[-(9 * 32 * 16 + 16):] *= 10.0  # a larger output layer gives every layer a sizeable gradient
    dn.set_params(p)
    N, H, W = 1, 32, 32
    x, t = _inputs(6, N, H, W)
    xd = x.permute(0, 2, 3, 1).contiguous().cuda()
    td = t.permute(0, 2, 3, 1).contiguous().cuda()
    g, loss = dn.grads(xd.data_ptr(), td.data_ptr(), N, H, W)
    pt = torch.from_numpy(p.copy()).requires_grad_(True)
    # reference: the same network with autograd through unrounded fp32
    import torch.nn.functional as F
    y = _unet_ref_autograd(pt, x.float())
    ref_loss = ((y - t.float()[:, :4]) ** 2).mean()
    ref_loss.backward()
    assert abs(loss - float(ref_loss)) <= 0.02 * float(ref_loss)
    gr = pt.grad.numpy()
    off = 0
    for i, (cin, cout, _) in enumerate(SPEC):
        n = 9 * cin * cout + cout
        a, b = g[off:off + n], gr[off:off + n]
        off += n
        cos = float(np.dot(a, b) / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
        rel = float(np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-30))
        assert cos > 0.99 and rel < 0.1, (i, cos, rel)


# The smallest image (a bottleneck of one pixel), ragged tiles and strips, a
# batch: pooling, upsampling and ReLU backward run fused in 16-byte pieces.
@pytest.mark.parametrize("N,H,W", [(1, 8, 8), (3, 24, 72), (2, 8, 136)])
def test_unet_gradients_at_tile_edges(rf, gpu_available, N, H, W):
    import torch
    ctx = rf.Context(1 << 12, 1, 16)
    dn = ctx.denoiser(seed=4)
    p = dn.params()
    p[-(9 * 32 * 16 + 16):] *= 10.0
    dn.set_params(p)
    x, t = _inputs(N + W, N, H, W)
    xd = x.permute(0, 2, 3, 1).contiguous().cuda()
    td = t.permute(0, 2, 3, 1).contiguous().cuda()
    g, loss = dn.grads(xd.data_ptr(), td.data_ptr(), N, H, W)
    pt = torch.from_numpy(p.copy()).requires_grad_(True)
    ref_loss = ((_unet_ref_autograd(pt, x.float()) - t.float()[:, :4]) ** 2).mean()
    ref_loss.backward()
    assert abs(loss - float(ref_loss)) <= 0.02 * float(ref_loss)
    gr, off = pt.grad.numpy(), 0
    for i, (cin, cout, _) in enumerate(SPEC):
        n = 9 * cin * cout + cout
        a, b = g[off:off + n], gr[off:off + n]
        off += n
        cos = float(np.dot(a, b) / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
        rel = float(np.linalg.norm(a - b) / (np.linalg.norm(b) + 1e-30))
        assert cos > 0.99 and rel < 0.1, (i, cos, rel)


class _Steps:
    """The training step's gradients in separate steps: whole convolutions and
    weight gradients of tensors that are written out (concatenations and
    upsampled channels among them), and masks, pooling and 2x2 sums in torch."""

    def __init__(self, rf, p):
        import torch
        self.t, self.ctx, off = torch, rf.Context(1 << 12, 1, 16), 0
        self.layers = []
        for cin, cout, relu in SPEC:
            n = 9 * cin * cout
            w = torch.from_numpy(p[off:off + n].copy()).cuda().to(torch.bfloat16).contiguous()
            b = torch.from_numpy(p[off + n:off + n + cout].copy()).cuda()
            wt = torch.empty_like(w)
            self.ctx.check(self.ctx.L.rf_nn_flip_weights(self.ctx.h, w.data_ptr(), wt.data_ptr(), cin, cout))
            self.layers.append((w, b, wt, cin, cout, relu))
            off += n + cout
        self.grads = [None] * len(SPEC)

    def _conv(self, x, w, b, cin, cout, relu):
        t, L = self.t, self.ctx.L
        x = x.contiguous()
        N, H, W, _ = x.shape
        o = t.empty(N, H, W, cout, dtype=t.bfloat16, device="cuda")
        self.ctx.check(L.rf_nn_conv3x3(self.ctx.h, x.data_ptr(), cin, 0, w.data_ptr(), b.data_ptr() if b is not None else None,
                                       o.data_ptr(), cout, 0, N, H, W, cin, cout, relu))
        return o

    def conv(self, i, x):
        w, b, _, cin, cout, relu = self.layers[i]
        return self._conv(x, w, b, cin, cout, relu)

    def dgrad(self, i, dy):
        _, _, wt, cin, cout, _ = self.layers[i]
        return self._conv(dy, wt, None, cout, cin, 0)

    def wgrad(self, i, x, dy):
        t, (_, _, _, cin, cout, _) = self.t, self.layers[i]
        x, dy = x.contiguous(), dy.contiguous()
        N, H, W, _ = x.shape
        dw, db = t.zeros(9 * cin * cout, device="cuda"), t.zeros(cout, device="cuda")
        self.ctx.check(self.ctx.L.rf_nn_conv3x3_wgrad(self.ctx.h, x.data_ptr(), cin, 0, dy.data_ptr(), cout, 0,
                                                      dw.data_ptr(), db.data_ptr(), N, H, W, cin, cout))
        self.grads[i] = t.cat([dw, db])

    def sum4(self, x):
        """2x2 sums in float, left to right and top to bottom."""
        f = x.float()
        return ((f[:, ::2, ::2] + f[:, ::2, 1::2]) + f[:, 1::2, ::2]) + f[:, 1::2, 1::2]

    def run(self, x, target):
        t = self.t
        bf = lambda v: v.to(t.bfloat16)
        keep = lambda v, y: t.where(y > 0, v, t.zeros_like(v))
        up = lambda v: v.repeat_interleave(2, 1).repeat_interleave(2, 2)
        pool = lambda v: bf(0.25 * self.sum4(v))
        e0a = self.conv(0, x)
        e0 = self.conv(1, e0a)
        p0 = pool(e0)
        e1a = self.conv(2, p0)
        e1 = self.conv(3, e1a)
        p1 = pool(e1)
        e2a = self.conv(4, p1)
        e2 = self.conv(5, e2a)
        p2 = pool(e2)
        b = self.conv(6, p2)
        c2 = t.cat([up(b), e2], 3)
        d2 = self.conv(7, c2)
        c1 = t.cat([up(d2), e1], 3)
        d1 = self.conv(8, c1)
        c0 = t.cat([up(d1), e0], 3)
        d0a = self.conv(9, c0)
        d0b = self.conv(10, d0a)
        o = self.conv(11, d0b)
        npix = x.shape[0] * x.shape[1] * x.shape[2]
        inv = float(np.float32(1.0) / (np.float32(4.0) * np.float32(npix)))
        g = t.zeros_like(o)
        g[..., :4] = bf(2.0 * ((x[..., :4].float() + o[..., :4].float()) - target[..., :4].float()) * inv)
        for i, xin, y in ((11, d0b, d0b), (10, d0a, d0a)):
            self.wgrad(i, xin, g)
            g = keep(self.dgrad(i, g), y)
        skips = []
        for i, cat, lo in ((9, c0, d1), (8, c1, d2), (7, c2, b)):
            self.wgrad(i, cat, g)
            d = self.dgrad(i, g)
            skips.append(d[..., lo.shape[3]:])
            g = keep(bf(self.sum4(d[..., :lo.shape[3]])), lo)
        for i, xin, skip, a, y, gs in ((6, p2, e2, 5, e2a, skips[2]), (4, p1, e1, 3, e1a, skips[1]),
                                       (2, p0, e0, 1, e0a, skips[0])):
            self.wgrad(i, xin, g)
            pooled = up(self.dgrad(i, g)).float()
            g = keep(bf(gs.float() + 0.25 * pooled), skip)
            self.wgrad(a, y, g)
            g = keep(self.dgrad(a, g), y)
        self.wgrad(0, x, g)
        return t.cat(self.grads).cpu().numpy()


# Every level one pixel, tiles and strips that end inside an image at each
# level, in each direction, and batches.
@pytest.mark.parametrize("N,H,W", [(1, 8, 8), (2, 24, 72), (1, 16, 136), (1, 16, 528), (1, 264, 16), (3, 40, 200),
                                   (1, 72, 264)])
def test_unet_gradients_have_the_separate_steps_bits(rf, gpu_available, N, H, W):
    """Masks, pooling, 2x2 sums and upsampled reads fused into the convolutions
    and weight gradients change no bit of the gradient."""
    print(f"gradients in separate steps: {N}x{H}x{W}", flush=True)
    ctx = rf.Context(1 << 12, 1, 16)
    dn = ctx.denoiser(seed=4)
    p = dn.params()
    p[-(9 * 32 * 16 + 16):] *= 10.0
    dn.set_params(p)
    x, t = (v.permute(0, 2, 3, 1).contiguous().cuda() for v in _inputs(N + W, N, H, W))
    g, _ = dn.grads(x.data_ptr(), t.data_ptr(), N, H, W)
    ref = _Steps(rf, p).run(x, t)
    off = 0
    for i, (cin, cout, _) in enumerate(SPEC):
        n = 9 * cin * cout + cout
        assert np.abs(ref[off:off + n]).max() > 0
        assert np.array_equal(g[off:off + n], ref[off:off + n]), i
        off += n


def _unet_ref_autograd(pt, x):
    import torch
    import torch.nn.functional as F
    Ls, off = [], 0
    for cin, cout, _ in SPEC:
        w = pt[off:off + 9 * cin * cout].reshape(3, 3, cout, cin).permute(2, 3, 0, 1)
        off += 9 * cin * cout
        b = pt[off:off + cout]
        off += cout
        Ls.append((w, b))

    def conv(i, t):
        y = F.conv2d(t, Ls[i][0], Ls[i][1], padding=1)
        return torch.relu(y) if SPEC[i][2] else y

    up = lambda t: F.interpolate(t, scale_factor=2, mode="nearest")
    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, F.avg_pool2d(e0, 2)))
    e2 = conv(5, conv(4, F.avg_pool2d(e1, 2)))
    b = conv(6, F.avg_pool2d(e2, 2))
    d2 = conv(7, torch.cat([up(b), e2], 1))
    d1 = conv(8, torch.cat([up(d2), e1], 1))
    d0 = conv(10, conv(9, torch.cat([up(d1), e0], 1)))
    o = conv(11, d0)
    return x[:, :4] + o[:, :4]


def test_training_reduces_loss(rf, gpu_available):
    ctx = rf.Context(1 << 12, 1, 16)
    dn = ctx.denoiser(seed=9)
    N, H, W = 2, 64, 64
    x, t = _inputs(7, N, H, W)
    xd = x.permute(0, 2, 3, 1).contiguous().cuda()
    td = t.permute(0, 2, 3, 1).contiguous().cuda()
    losses = [dn.train_step(xd.data_ptr(), td.data_ptr(), N, H, W, 2e-3) for _ in range(60)]
    assert np.isfinite(losses).all()
    assert min(losses[-5:]) < 0.5 * losses[0], (losses[0], losses[-5:])


def test_trained_weights_denoise_held_out_flames(rf, gpu_available):
    """The committed weights bring a 4-spp log-density image of unseen flames
    closer to the same flames' 1024-spp image."""
    import torch
    from refrakt_amd import denoise
    ctx = rf.Context(1 << 12, 1, 16, seed=77)
    dn = ctx.denoiser()
    meta = denoise.load_weights(dn)
    assert meta["n_params"] == dn.n_params
    flames = denoise.training_flames(6, seed=99)  # a seed the training set never used
    S = 512
    X = torch.empty((6, S, S, 16), dtype=torch.bfloat16, device="cuda")
    T = torch.empty_like(X)
    denoise.render_log_density(ctx, flames, S, S, 4.0, X, 64)
    denoise.render_log_density(ctx, flames, S, S, 1024.0, T, 1024)
    y = torch.empty((1, S, S, 4), dtype=torch.float32, device="cuda")
    gain = []
    for i in range(6):
        dn.infer(X[i:i + 1].data_ptr(), y.data_ptr(), 1, S, S)
        t = T[i, :, :, :4].float()
        mse_in = float(((X[i, :, :, :4].float() - t) ** 2).mean())
        mse_out = float(((y[0] - t) ** 2).mean())
        gain.append(10 * np.log10(mse_in / mse_out))
    print("denoiser gain per flame (dB):", [round(g, 2) for g in gain])
    assert np.mean(gain) > 2.0 and min(gain) > 0.0
