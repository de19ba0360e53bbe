"""An infinite activation on the image's edge reaches the weight gradients of the
taps that meet it inside the image and no others: tiles that the edge cuts (4 x
32 pixels) hold zero output gradients beyond it, which must not meet it."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("cin,cout", [(32, 64), (32, 32), (16, 32), (48, 16), (8, 32), (8, 16), (24, 32)])
@pytest.mark.parametrize("H,W", [(9, 40), (10, 33), (11, 63), (8, 65), (12, 64), (5, 7)])
def test_infinite_edge_pixels(cuda, cin, cout, H, W):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    g = torch.Generator().manual_seed(H * W)
    print("wgrad edge %dx%d cin %d cout %d" % (H, W, cin, cout), flush=True)
    dy = torch.randn((2, H, W, cout), generator=g).to(torch.bfloat16)
    x = torch.randn((2, H, W, cin), generator=g).to(torch.bfloat16)
    x[0, H - 1, W - 1, 0] = float("inf")
    x[1, H - 1, 2, 1] = float("inf")
    x[1, 3, W - 1, 2] = float("inf")
    n = L.sgdct_nn_wgrad_workspace(2, H, W, cin, cout)
    ws = torch.full((n,), float("nan"), device=cuda)
    dw = torch.empty((cout, 9, cin), device=cuda)
    xd, dyd = x.to(cuda), dy.to(cuda)
    assert L.sgdct_nn_wgrad(_vp(xd), _vp(dyd), _vp(dw), _vp(ws), n, 2, H, W, cin, cout, None) == 0, m.last_error()
    torch.cuda.synchronize()
    finite = torch.isfinite(dw).all(0).cpu()
    # taps (ky, kx) that meet pixel (y, x): output (y + 1 - ky, x + 1 - kx) inside
    want = torch.ones((9, cin), dtype=torch.bool)
    for y, px, c in ((H - 1, W - 1, 0), (H - 1, 2, 1), (3, W - 1, 2)):
        for t in range(9):
            oy, ox = y + 1 - t // 3, px + 1 - t % 3
            if 0 <= oy < H and 0 <= ox < W:
                want[t, c] = False
    assert torch.equal(finite, want), (finite != want).nonzero().tolist()
