"""Convolutions whose output or mask is not 16-byte aligned (a slice of a larger
buffer) equal the aligned ones to one rounding of the sums' order; the split
gradient refuses such outputs with a message."""
import pytest

from test_gpu_unet_conv import _vp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 64), (8, 32)])
@pytest.mark.parametrize("off_out,off_mask", [(1, 0), (0, 3), (5, 1)])
def test_unaligned_output_and_mask(cuda, cin, cout, off_out, off_mask):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    B, H, W = 2, 19, 37
    print("conv %d -> %d, output off %d, mask off %d" % (cin, cout, off_out, off_mask), flush=True)
    g = torch.Generator(device=cuda).manual_seed(cin + cout)
    x = torch.randn((B, H, W, cin), device=cuda, generator=g).to(torch.bfloat16)
    w = (0.1 * torch.randn((cout, 9 * cin), device=cuda, generator=g)).to(torch.bfloat16)
    n = B * H * W * cout
    mask = torch.randn(n, device=cuda, generator=g).to(torch.bfloat16)
    for dtype, f32 in ((torch.float32, 1), (torch.bfloat16, 0)):
        ref, buf = torch.empty(n, dtype=dtype, device=cuda), torch.zeros(n + 16, dtype=dtype, device=cuda)
        mbuf = torch.zeros(n + 16, dtype=torch.bfloat16, device=cuda)
        mbuf[off_mask:off_mask + n] = mask
        for out, mk in ((ref, mask), (buf[off_out:], mbuf[off_mask:])):
            assert L.sgdct_nn_conv3x3_ex(_vp(x), None, 0, _vp(w), None, _vp(out), _vp(mk), B, H, W, cin, cout, 0, f32,
                                         None) == 0, m.last_error()
        torch.cuda.synchronize()
        got = buf[off_out:off_out + n].float()
        assert bool((buf[:off_out] == 0).all()) and bool((buf[off_out + n:] == 0).all())
        tol = 2.0 ** -8 if dtype == torch.bfloat16 else 9 * cin * 2.0 ** -24
        assert bool(((got - ref.float()).abs() <= tol * ref.float().abs().clamp(min=1.0)).all())


def test_unaligned_split_gradient_is_refused(cuda):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    B, H, W, cin, cout, c0 = 1, 16, 16, 32, 96, 64
    x = torch.zeros((B, H, W, cin), dtype=torch.bfloat16, device=cuda)
    w = torch.zeros((cout, 9 * cin), dtype=torch.bfloat16, device=cuda)
    low = torch.zeros(B * H * W // 4 * c0 + 8, dtype=torch.bfloat16, device=cuda)
    skip = torch.zeros(B * H * W * (cout - c0) + 8, device=cuda)
    for lo, mk, sk in ((low[1:], low, skip), (low, low[1:], skip), (low, low, skip[1:])):
        assert L.sgdct_nn_conv3x3_upback(_vp(x), _vp(w), _vp(lo), _vp(mk), _vp(sk), None, 0, B, H, W, cin, cout, c0,
                                         None) == -1
        assert "aligned" in m.last_error()
