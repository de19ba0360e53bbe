"""A^T where the image reaches behind the source: the plane through a view's
source and parallel to its detector cuts pixel tiles, whose bins no window of
their corners' projections holds.  Against the FP64 oracle at the parity bar
(1e-5 relative L2) over the pixels more than three pixels off every such plane
(nearer ones have footprints without end; hexagons, six columns)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [  # views, nx, ny, nu, lso, du: windows of up to the whole detector, and below 64 bins
    (3, 64, 64, 300, 40.0, 0.8), (2, 100, 40, 500, 60.0, 0.5), (4, 50, 64, 60, 40.0, 4.0)]


def off_planes(x, y, ang, lso, reach):
    m = np.ones(x.shape, bool)
    for a in ang:
        m &= np.abs(x * np.cos(a) + y * np.sin(a) + lso) > reach
    return m


def check(P, cuda, e, m, y):
    import torch
    r = P.backward(torch.from_numpy(y).to(cuda)).double().cpu().numpy()
    err = float(np.linalg.norm((r - e)[m]) / np.linalg.norm(e[m]))
    print("  A^T %.2e over %d of %d pixels" % (err, m.sum(), m.size), flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("basis", ["B1", "SF"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_backward_behind_the_source(cuda, oracle_exact, basis, case):
    from pyoracle import Geometry
    from sgd_amd.torch_ops import Projector
    n, nx, ny, nu, lso, du = CASES[case]
    ang = 0.3 + 2 * np.pi * np.arange(n) / n
    geo = (nx, ny, ang, nu, 1.7, 1.7, du, 2 * lso, lso)
    print(basis, CASES[case], flush=True)
    y = np.random.default_rng(1).standard_normal((n, nu)).astype(np.float32)
    px, py = np.meshgrid((np.arange(nx) - (nx - 1) / 2) * 1.7, (np.arange(ny) - (ny - 1) / 2) * 1.7)
    check(Projector(basis, *geo), cuda, Geometry(oracle_exact, *geo).backward(basis, y.astype(float)),
          off_planes(px, py, ang, lso, 3 * 1.7), y)


@pytest.mark.parametrize("basis", ["H0", "Hl"])
def test_hex_backward_behind_the_source(cuda, oracle_exact, basis):
    from pyoracle import HexGeometry
    from sgd_amd.torch_ops import Projector
    n, nl, nc, nu, dt, du, lso = 3, 61, 40, 300, 0.8, 1.2, 40.0
    ang = 0.3 + 2 * np.pi * np.arange(n) / n
    geo = (nl, nc, ang, nu, dt, du, 2 * lso, lso)
    print(basis, flush=True)
    y = np.random.default_rng(1).standard_normal((n, nu)).astype(np.float32)
    ic, il = np.meshgrid(np.arange(nc), np.arange(nl))
    px = (ic + 0.5 * (il & 1) - (nc - 1) / 2) * np.sqrt(3) * dt
    py = (il - (nl - 1) / 2) * dt * (1.5 if basis == "H0" else 0.5)
    m = off_planes(px, py, ang, lso, 6 * np.sqrt(3) * dt)
    m[1::2, -1] = False
    check(Projector.hexagonal(basis, *geo), cuda, HexGeometry(oracle_exact, *geo).backward(basis, y.astype(float)), m, y)


@pytest.mark.parametrize("basis", ["B1", "SF", "H0"])
def test_views_by_themselves_behind_the_source(cuda, basis):
    """A of one view is bit for bit the scan's (no other view's footprints)."""
    import torch
    from sgd_amd.torch_ops import Projector
    n = 250 if basis == "H0" else 1024  # hexagons: as many waves per launch as one view takes
    ang = 2 * np.pi * np.arange(n) / n

    def make(a):
        P = (Projector.hexagonal("H0", 301, 300, a, 512, 2.2, 1.7, 1000.0, 500.0) if basis == "H0" else
             Projector(basis, 400, 400, a, 512, 3.2, 3.2, 1.7, 1000.0, 500.0))
        P.set_split(1, 1)
        return P

    P = make(ang)
    x = torch.randn(P.img_shape, device=cuda, generator=torch.Generator(device=cuda).manual_seed(1))
    y = torch.nan_to_num(P.forward(x))
    for k in (0, 5, n // 4 - 1, n // 4, n // 2 + 3, n - 1):
        print(basis, "view", k, flush=True)
        assert torch.equal(torch.nan_to_num(make(ang[k:k + 1]).forward(x))[0], y[k])
