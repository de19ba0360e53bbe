"""SF on an image of 4 GiB and a little (32768 x 32776 pixels): A reads the pixels
past 4 GiB.  On an image that is zero before them, <A x, y> = <x, A^T y> (in FP64)
for the transpose, whose pixels are formed from the sinogram alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far_rows", [24, 3])
def test_pixels_past_four_gib(cuda, far_rows):
    import torch
    from sgd_amd.torch_ops import Projector
    nx, ny, nu = 32768, 32776, 700
    ang = np.array([0.3, 1.7])
    P = Projector("SF", nx, ny, ang, nu, 0.01, 0.01, 1.0, 1000.0, 500.0)
    print("SF %d x %d, rows %d.." % (nx, ny, ny - far_rows), flush=True)
    x = torch.zeros(P.img_shape, device=cuda)
    g = torch.Generator(device=cuda).manual_seed(1)
    x[ny - far_rows:] = torch.rand((far_rows, nx), device=cuda, generator=g)
    y = torch.rand(P.sino_shape, device=cuda, generator=g)
    ax = P.forward(x)
    torch.cuda.synchronize()
    tail = x[ny - far_rows:].double()
    del x
    aty = P.backward(y)
    a, b = float((ax.double() * y.double()).sum()), float((tail * aty[ny - far_rows:].double()).sum())
    print("  <A x, y> %.9g  <x, A^T y> %.9g" % (a, b), flush=True)
    assert b > 0 and abs(a - b) <= 1e-5 * abs(b)
