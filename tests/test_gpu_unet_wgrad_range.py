"""An FP32 accumulator of the weight gradient holds at most 8192 pixels' products,
also where the batch is large and the channels leave few pixel ranges: one
output gradient of 2^15 makes its accumulator lose the others of 2^-15 (32 of
them, a matrix step, are a quarter of its last place), so the error is what one
accumulator's 8192 pixels hold, 0.25, and roundings of the partial sums' total
(64 of them, half of 2^-8 each)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("B,H,W,cin,cout", [(8, 256, 256, 256, 256), (8, 256, 250, 96, 192), (4, 512, 512, 48, 80)])
def test_accumulated_pixels(cuda, B, H, W, cin, cout):
    import torch
    from sgd_amd import _lib as m
    L = m.lib()
    print("wgrad B %d %dx%d cin %d cout %d" % (B, H, W, cin, cout), flush=True)
    x = torch.ones((B, H, W, cin), dtype=torch.bfloat16, device=cuda)
    dy = torch.full((B, H, W, cout), 2.0 ** -15, dtype=torch.bfloat16, device=cuda)
    dy[0, 1, 1] = 2.0 ** 15
    n = L.sgdct_nn_wgrad_workspace(B, H, W, cin, cout)
    ws = torch.full((n,), float("nan"), device=cuda)
    dw = torch.empty((cout, 9, cin), device=cuda)
    assert L.sgdct_nn_wgrad(_vp(x), _vp(dy), _vp(dw), _vp(ws), n, B, H, W, cin, cout, None) == 0, m.last_error()
    torch.cuda.synchronize()
    ones = torch.nn.functional.pad(torch.ones((H, W), dtype=torch.float64), (1, 1, 1, 1))
    for t in range(9):
        count = float(ones[t // 3:t // 3 + H, t % 3:t % 3 + W].sum()) * B
        want = 2.0 ** 15 + (count - 1) * 2.0 ** -15
        err = float((dw[:, t].double() - want).abs().max())
        print("  tap %d err %.4f" % (t, err))
        assert err <= 0.25 + 64 * 2.0 ** -9
