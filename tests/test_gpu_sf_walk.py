"""The SF projector's line walk (FP32 pixel intervals, the weight's line-wise
reciprocal) and bin walk at their extremes, against the FP64 oracle: A and A^T
within 1e-5 relative L2 (as every fan-beam test), the adjoint within 1e-6.
Fans whose waves cross 45 degrees; long thin images, whose interval ends carry
the largest FP32 error; many bins per pixel and many pixels per bin; pixels off
square; views along the axes, whose trapezoids have ramps of (nearly) no width."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nx, ny, dx, dy, nu, du, lso, lsd, first angle
CASES = [
    (64, 64, 1.0, 1.0, 300, 1.0, 60.0, 90.0, 0.2),
    (2048, 3, 0.4, 0.7, 300, 4.0, 1200.0, 1800.0, 0.1),
    (3, 1500, 0.7, 0.4, 200, 4.0, 900.0, 1500.0, 0.0),
    (12, 9, 4.0, 2.5, 700, 0.12, 300.0, 500.0, 0.4),
    (200, 180, 0.3, 0.3, 24, 6.0, 300.0, 500.0, 0.7),
    (65, 33, 1.0, 1.0, 130, 1.0, 1e5, 1.00001e5, 0.0),
]


@pytest.mark.parametrize("nx,ny,dx,dy,nu,du,lso,lsd,a0", CASES)
def test_sf_walk(cuda, oracle_exact, nx, ny, dx, dy, nu, du, lso, lsd, a0):
    import torch
    from pyoracle import Geometry
    from sgd_amd.torch_ops import Projector
    print("SF %dx%d px %.2fx%.2f, %d bins of %.2f, lso %g lsd %g" % (nx, ny, dx, dy, nu, du, lso, lsd), flush=True)
    ang = a0 + np.array([0.0, 0.5 * np.pi, 0.25 * np.pi, 2.3, 4.0])
    P = Projector("SF", nx, ny, ang, nu, dx, dy, du, lsd, lso)
    G = Geometry(oracle_exact, nx, ny, ang, nu, dx, dy, du, lsd, lso)
    rng = np.random.default_rng(nx + nu)
    x = rng.random((ny, nx)).astype(np.float32)
    y = rng.random((len(ang), nu)).astype(np.float32)
    xt, yt = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    ax, aty = P.forward(xt), P.backward(yt)
    torch.cuda.synchronize()
    a, t = ax.double(), aty.double()

    def rel(got, want):
        return float(np.linalg.norm(got.cpu().numpy() - want) / np.linalg.norm(want))

    e1, e2 = rel(a, G.forward("SF", x.astype(np.float64))), rel(t, G.backward("SF", y.astype(np.float64)))
    ea = abs(float((a * yt.double()).sum()) - float((xt.double() * t).sum())) / (float(a.norm()) * float(yt.norm()))
    print("  A %.2e  A^T %.2e  adjoint %.2e" % (e1, e2, ea), flush=True)
    assert e1 <= 1e-5 and e2 <= 1e-5 and ea <= 1e-6
