"""The halo-tiled 3x3 convolution's block shapes and runs of tiles (unet.hip)
against torch's FP64 conv2d on the CPU: 64-, 32- and 16-channel blocks, 8, 16
and 32 channels per chunk, one and several chunks; images of one tile, of cut
tiles, and of more tiles than blocks (runs of 2 and more, the last one short;
halos kept for all blocks of output channels).
FP32 output <= 1e-5 relative L2 (only the order of the FP32 sums differs), bf16
output with bias, ReLU and mask within one bf16 rounding (2^-8 relative, 1e-6
absolute)."""
import pytest

from test_gpu_unet_conv import _vp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,cin,cout", [
    (1, 1, 1, 16, 16), (2, 33, 18, 8, 16), (1, 17, 40, 16, 32), (1, 9, 20, 16, 64), (2, 20, 20, 64, 16),
    (4, 208, 336, 8, 32), (3, 330, 200, 32, 16), (2, 210, 330, 32, 64), (1, 160, 170, 64, 192),
    (2, 210, 330, 32, 96), (4, 208, 336, 8, 128), (2, 210, 330, 16, 48), (3, 200, 200, 32, 128)])
def test_halo_blocks(cuda, B, H, W, cin, cout):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    print("halo conv B %d %dx%d cin %d cout %d" % (B, H, W, cin, cout), flush=True)
    g = torch.Generator().manual_seed(H + cin + cout)
    x = torch.randn((B, H, W, cin), generator=g).to(torch.bfloat16)
    w = (0.1 * torch.randn((cout, 9 * cin), generator=g)).to(torch.bfloat16)
    bias = torch.randn(cout, generator=g)
    mask = torch.randn((B, H, W, cout), generator=g).to(torch.bfloat16)
    wr = w.double().view(cout, 3, 3, cin).permute(0, 3, 1, 2)
    ref = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2), wr, padding=1).permute(0, 2, 3, 1)
    xd, wd, bd, md = x.to(cuda), w.to(cuda), bias.to(cuda), mask.to(cuda)
    out = torch.empty((B, H, W, cout), device=cuda)
    outb = torch.empty((B, H, W, cout), dtype=torch.bfloat16, device=cuda)
    assert L.sgdct_nn_conv3x3_ex(_vp(xd), None, 0, _vp(wd), None, _vp(out), None, B, H, W, cin, cout, 0, 1, None) == 0
    assert L.sgdct_nn_conv3x3_ex(_vp(xd), None, 0, _vp(wd), _vp(bd), _vp(outb), _vp(md), B, H, W, cin, cout, 1, 0,
                                 None) == 0
    torch.cuda.synchronize()
    e = float((out.cpu().double() - ref).norm() / ref.norm())
    print("  FP32 output rel %.2e" % e)
    assert e <= 1e-5
    rb = (ref + bias.double()).relu() * (mask > 0)
    assert bool(((outb.cpu().double() - rb).abs() <= 2.0 ** -8 * rb.abs() + 1e-6).all())
