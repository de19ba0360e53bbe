"""The hexagonal projectors' line walks (FP32 point intervals) and H0's chord
form at their extremes, against the FP64 oracle: A and A^T within 1e-5 relative
L2 (as every hexagonal test).  Long lattices, whose interval ends carry the
largest FP32 error; near-parallel rays along and across the lattice's axes,
where a vertex projection vanishes (c = 0) or two coincide (b = c); bins far
smaller and far larger than a point; one to eight values per point."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nl, nc, dt, nu, du, lso, lsd, first angle, images
CASES = [
    (5, 1600, 0.4, 260, 4.0, 1500.0, 2200.0, 0.1, 1),
    (1501, 3, 0.5, 300, 4.0, 1800.0, 2600.0, 0.0, 2),
    (21, 17, 1.0, 41, 0.9, 1e6, 1.00001e6, 0.0, 3),
    (9, 8, 4.0, 500, 0.1, 200.0, 300.0, 0.3, 1),
    (61, 50, 0.4, 20, 6.0, 200.0, 350.0, 0.2, 4),
]


@pytest.mark.parametrize("basis", ["H0", "Hl"])
@pytest.mark.parametrize("nl,nc,dt,nu,du,lso,lsd,a0,batch", CASES)
def test_hex_walk(cuda, oracle_exact, basis, nl, nc, dt, nu, du, lso, lsd, a0, batch):
    import torch
    from pyoracle import HexGeometry
    from sgd_amd.torch_ops import Projector
    print("%s %d x %d points of %.2f, %d bins of %.2f, lso %g lsd %g, batch %d"
          % (basis, nl, nc, dt, nu, du, lso, lsd, batch), flush=True)
    ang = a0 + np.array([0.0, 0.5 * np.pi, np.pi / 6.0, np.pi / 3.0, 2.3, 4.0])
    P = Projector.hexagonal(basis, nl, nc, ang, nu, dt, du, lsd, lso)
    G = HexGeometry(oracle_exact, nl, nc, ang, nu, dt, du, lsd, lso)
    rng = np.random.default_rng(nl + nu)
    x = rng.random((batch, nl, nc)).astype(np.float32)
    x[:, 1::2, -1] = 0.0
    y = rng.random((batch, len(ang), nu)).astype(np.float32)
    ax, aty = P.forward(torch.from_numpy(x).to(cuda)), P.backward(torch.from_numpy(y).to(cuda))
    torch.cuda.synchronize()
    for k in range(batch):
        for got, want in ((ax, G.forward(basis, x[k].astype(np.float64))), (aty, G.backward(basis, y[k].astype(np.float64)))):
            e = float(np.linalg.norm(got[k].double().cpu().numpy() - want) / np.linalg.norm(want))
            print("  image %d rel %.2e" % (k, e), flush=True)
            assert e <= 1e-5
