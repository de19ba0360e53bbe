"""The U-Net's pooling, output-head and concatenation-gradient passes
(unet.hip), in their vector and element-wise forms, on the C ABI.

  * 2x2 mean and its gradient: bit for bit torch's FP32 evaluation in the same
    order (0.25 * (a + b + c + d), s + 0.25 d: each rounded as written, 0.25 d
    exact), rounded to bf16;
  * head gradient: dy and the masked outer product bit for bit, gw within
    M 2^-24 of the sum of magnitudes (any order of M FP32 additions);
  * gradient of conv([upsample2(low), skip]): the skip part <= 1e-5 relative
    L2 of the FP64 convolution (only the order of the FP32 sums differs), the
    low part's 2x2 sums within one bf16 rounding of it and 1e-5 of its RMS.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _vp(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _lib():
    from sgd_amd import _lib as m
    return m.lib(), m


@pytest.mark.parametrize("B,H,W,C,shift", [(2, 5, 9, 8, 0), (1, 3, 3, 12, 0), (3, 8, 8, 32, 0), (2, 4, 6, 16, 1)])
def test_pool2_and_gradient(cuda, B, H, W, C, shift):
    import torch
    L, m = _lib()
    print("pool2 B %d %dx%d C %d shift %d" % (B, H, W, C, shift), flush=True)
    g = torch.Generator().manual_seed(C + H)
    n, ns = B * H * W * C, 4 * B * H * W * C
    # shift: tensors off the 16-byte alignment
    src = torch.randn(ns + shift, generator=g).to(torch.bfloat16).to(cuda)[shift:]
    dst = torch.zeros(n + shift, dtype=torch.bfloat16, device=cuda)[shift:]
    assert L.sgdct_nn_pool2(_vp(src), _vp(dst), B, H, W, C, None) == 0, m.last_error()
    s = src.float().cpu().view(B, H, 2, W, 2, C)
    ref = (0.25 * (s[:, :, 0, :, 0] + s[:, :, 0, :, 1] + s[:, :, 1, :, 0] + s[:, :, 1, :, 1])).to(torch.bfloat16)
    torch.cuda.synchronize()
    assert torch.equal(dst.cpu().view(B, H, W, C), ref)

    dv = torch.randn(n + shift, generator=g).to(cuda)[shift:]
    gs = torch.randn(ns + shift, generator=g).to(cuda)[shift:]
    out = torch.zeros(ns + shift, dtype=torch.bfloat16, device=cuda)[shift:]
    assert L.sgdct_nn_pool2_back(_vp(dv), _vp(gs), _vp(out), _vp(src), B, H, W, C, None) == 0, m.last_error()
    d = dv.cpu().view(B, H, 1, W, 1, C)
    v = gs.cpu().view(B, H, 2, W, 2, C) + 0.25 * d
    v = torch.where(s > 0, v, torch.zeros(())).to(torch.bfloat16)
    torch.cuda.synchronize()
    assert torch.equal(out.cpu().view(B, H, 2, W, 2, C), v)


@pytest.mark.parametrize("M,C", [(1, 8), (4097, 32), (9000, 128), (777, 24), (1000, 12)])
def test_head_gradient(cuda, M, C):
    import torch
    L, m = _lib()
    print("head_back M %d C %d" % (M, C), flush=True)
    g = torch.Generator().manual_seed(M + C)
    y, t, w = (torch.randn(k, generator=g).to(cuda) for k in (M, M, C))
    act = torch.randn(M * C, generator=g).relu().to(torch.bfloat16).to(cuda)
    other = torch.randn(M * C, generator=g).to(torch.bfloat16).to(cuda)
    n = L.sgdct_nn_head_workspace(M, C)
    ws = torch.empty(n, device=cuda)
    for mask in (act, other):
        dy, gw = torch.empty(M, device=cuda), torch.empty(C + 1, device=cuda)
        out = torch.empty(M * C, dtype=torch.bfloat16, device=cuda)
        assert L.sgdct_nn_head_back(_vp(y), _vp(t), _vp(w), _vp(act), _vp(dy), None, _vp(out), _vp(mask), _vp(gw),
                                    _vp(ws), n, M, C, None) == 0, m.last_error()
        torch.cuda.synchronize()
        d = torch.tensor(np.float32(2.0) / np.float32(M)) * (y.cpu() - t.cpu())
        assert torch.equal(dy.cpu(), d)
        o = torch.where(mask.cpu().view(M, C) > 0, d[:, None] * w.cpu()[None, :], torch.zeros(()))
        assert torch.equal(out.cpu().view(M, C), o.to(torch.bfloat16))
        p = torch.cat([act.cpu().view(M, C).double(), torch.ones(M, 1, dtype=torch.float64)], 1) * d.double()[:, None]
        err = (gw.cpu().double() - p.sum(0)).abs()
        assert bool((err <= M * 2.0 ** -24 * p.abs().sum(0) + 1e-30).all())


# one kernel: 64-, 32- and 16-channel blocks, one-tile and cut images; through a
# workspace: channels off the kernel's multiples, c0 inside a block
@pytest.mark.parametrize("B,H,W,cin,cout,c0", [(2, 18, 30, 32, 96, 64), (1, 34, 18, 64, 192, 128), (1, 2, 2, 8, 96, 32),
                                               (2, 16, 16, 32, 48, 32), (2, 14, 24, 16, 48, 32), (1, 10, 20, 32, 192, 96),
                                               (4, 130, 260, 32, 96, 64), (1, 6, 10, 32, 40, 24), (1, 12, 8, 48, 96, 64)])
def test_concatenation_gradient(cuda, B, H, W, cin, cout, c0):
    import torch
    L, m = _lib()
    print("upback B %d %dx%d cin %d cout %d c0 %d" % (B, H, W, cin, cout, c0), flush=True)
    g = torch.Generator().manual_seed(H * W + cout)
    x = torch.randn((B, H, W, cin), generator=g).to(torch.bfloat16)
    w = (0.1 * torch.randn((cout, 9 * cin), generator=g)).to(torch.bfloat16)
    mask = torch.randn((B, H // 2, W // 2, c0), generator=g).to(torch.bfloat16)
    n = L.sgdct_nn_conv3x3_upback_workspace(B, H, W, cin, cout, c0)
    block = next((k for k in (64, 32, 16) if cout % k == 0), 0)
    assert (n == 0) == ((cin % 32 == 0 or cin in (8, 16)) and block > 0 and c0 % block == 0)
    xd, wd, md = x.to(cuda), w.to(cuda), mask.to(cuda)
    ws = torch.empty(max(n, 1), device=cuda)
    low = torch.empty((B, H // 2, W // 2, c0), dtype=torch.bfloat16, device=cuda)
    skip = torch.empty((B, H, W, cout - c0), device=cuda)
    assert L.sgdct_nn_conv3x3_upback(_vp(xd), _vp(wd), _vp(low), _vp(md), _vp(skip), _vp(ws) if n else None, n, B, H,
                                     W, cin, cout, c0, None) == 0, m.last_error()
    torch.cuda.synchronize()
    wr = w.double().view(cout, 3, 3, cin).permute(0, 3, 1, 2)
    ref = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2), wr, padding=1).permute(0, 2, 3, 1)
    e = float((skip.cpu().double() - ref[..., c0:]).norm() / ref[..., c0:].norm())
    print("  skip rel %.2e" % e)
    assert e <= 1e-5
    s = ref[..., :c0].reshape(B, H // 2, 2, W // 2, 2, c0).sum((2, 4)) * (mask > 0)
    err = (low.cpu().double() - s).abs()
    assert bool((err <= 2.0 ** -8 * s.abs() + 1e-5 * float(s.norm()) / s.numel() ** 0.5).all())
