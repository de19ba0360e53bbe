"""The U-Net's weight and bias gradients (sgdct_nn_wgrad_ex, unet.hip) against
FP64 on the CPU, on bf16-valued operands: the products are exact in FP32 and
only the order of their sums differs, relative L2 error <= 1e-5 over the array.

Tile-staged form (cin, cout multiples of 16, cin 8): 64-, 32- and 16-channel
output tiles, images smaller than a tile, cut tiles, one split and many, the
decoder's concatenation; gathered form: other channel counts, a concatenation
off the channel chunks.
"""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _vp(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


@pytest.mark.parametrize("B,H,W,cin,cout,c0", [
    (1, 3, 5, 32, 32, 0), (2, 37, 50, 32, 64, 0), (3, 64, 80, 64, 32, 0), (1, 18, 34, 96, 32, 64),
    (2, 20, 20, 192, 64, 128), (1, 9, 16, 32, 128, 0), (2, 12, 20, 8, 32, 0), (1, 5, 70, 8, 96, 0), (1, 9, 40, 8, 16, 0),
    (2, 14, 36, 16, 16, 0), (1, 8, 34, 48, 16, 32), (1, 20, 10, 48, 96, 16), (1, 6, 6, 48, 32, 8), (1, 7, 9, 24, 16, 0), (1, 10, 12, 64, 32, 48),
    (1, 11, 13, 32, 40, 0)])
def test_weight_gradient(cuda, B, H, W, cin, cout, c0):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    print("wgrad B %d %dx%d cin %d cout %d concat %d" % (B, H, W, cin, cout, c0), flush=True)
    g = torch.Generator().manual_seed(H * W + cin + cout)
    dy = torch.randn((B, H, W, cout), generator=g).to(torch.bfloat16)
    if c0:
        low = torch.randn((B, H // 2, W // 2, c0), generator=g).to(torch.bfloat16)
        skip = torch.randn((B, H, W, cin - c0), generator=g).to(torch.bfloat16)
        x = torch.cat([low.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], 3)
        src, src2 = low.to(cuda), skip.to(cuda)
    else:
        x = torch.randn((B, H, W, cin), generator=g).to(torch.bfloat16)
        src, src2 = x.to(cuda), None
    n = L.sgdct_nn_wgrad_workspace(B, H, W, cin, cout)
    ws = torch.full((n,), float("nan"), device=cuda)
    dyd = dy.to(cuda)
    xp = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    cols = torch.stack([xp[:, i:i + H, j:j + W] for i in range(3) for j in range(3)], 3)
    ref = dy.double().reshape(-1, cout).T @ cols.reshape(-1, 9 * cin)
    refb = dy.double().sum((0, 1, 2))
    for with_bias in (True, False):
        dw = torch.empty((cout, 9 * cin), device=cuda)
        db = torch.empty(cout, device=cuda) if with_bias else None
        assert L.sgdct_nn_wgrad_ex(_vp(src), _vp(src2), c0, _vp(dyd), _vp(dw), _vp(db), _vp(ws), n, B, H, W, cin,
                                   cout, None) == 0, m.last_error()
        torch.cuda.synchronize()
        e = float((dw.cpu().double() - ref).norm() / ref.norm())
        print("  dw rel %.2e" % e)
        assert e <= 1e-5
        if with_bias:
            assert float((db.cpu().double() - refb).norm() / refb.norm()) <= 1e-5
