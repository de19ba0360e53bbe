"""Bins wider than a wave's slab of the image, up to wider than the whole image:
A against the FP64 oracle at the parity bar (1e-5 relative L2), A^T beside it.
The strip of such a bin holds slabs whose rows its two edges cross far off to one
side."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def check(P, G, cuda, basis, seed):
    import torch
    rng = np.random.default_rng(seed)
    x, y = rng.random(P.img_shape).astype(np.float32), rng.random(P.sino_shape).astype(np.float32)
    if basis in ("H0", "Hl"):
        x[1::2, -1] = 0.0
    a = P.forward(torch.from_numpy(x).to(cuda)).double().cpu().numpy()
    t = P.backward(torch.from_numpy(y).to(cuda)).double().cpu().numpy()
    e1, e2 = rel(a, G.forward(basis, x.astype(np.float64))), rel(t, G.backward(basis, y.astype(np.float64)))
    print("  A %.2e  A^T %.2e" % (e1, e2), flush=True)
    assert e1 <= 1e-5 and e2 <= 1e-5


# rows, columns, views, start, bins, bin width, lattice constant, lso
HEX = [(1, 12, 74, 0.31, 3, 179.3, 8.33, 500.3), (1, 8, 97, 0.2, 13, 49.2, 12.5, 400.0),
       (2, 2, 9, 0.37, 2, 253.7, 50.0, 500.3), (3, 3, 51, 0.11, 2, 246.1, 33.3, 500.3),
       (109, 109, 105, 0.37, 2, 220.3, 0.917, 400.0), (60, 7, 33, 0.23, 5, 61.1, 2.9, 500.3),
       (7, 60, 33, 0.23, 5, 61.1, 2.9, 500.3), (33, 21, 1030, 0.0, 4, 80.7, 3.1, 500.3)]


@pytest.mark.parametrize("basis", ["H0", "Hl"])
@pytest.mark.parametrize("case", range(len(HEX)))
@pytest.mark.parametrize("split", [0, 3])
def test_hex_wide_bins(cuda, oracle_exact, basis, case, split):
    from pyoracle import HexGeometry
    from sgd_amd.torch_ops import Projector
    nl, nc, n, start, nu, du, dt, lso = HEX[case]
    geo = (nl, nc, start + 2 * np.pi * np.arange(n) / n, nu, dt, du, 2 * lso, lso)
    print(basis, HEX[case], split, flush=True)
    P = Projector.hexagonal(basis, *geo)
    P.set_split(split, split)
    check(P, HexGeometry(oracle_exact, *geo), cuda, basis, case)


# nx, ny, dx, dy, views, start, bins, bin width, lso
FAN = [(1, 12, 16.7, 16.7, 74, 0.31, 3, 179.3, 500.3), (12, 1, 16.7, 16.7, 74, 0.31, 3, 179.3, 500.3),
       (2, 2, 100.0, 93.0, 9, 0.37, 2, 253.7, 500.3), (3, 3, 66.7, 50.0, 51, 0.11, 2, 246.1, 500.3),
       (109, 109, 1.83, 1.83, 105, 0.37, 2, 220.3, 400.0), (60, 7, 3.3, 3.9, 33, 0.23, 5, 61.1, 500.3),
       (41, 12, 4.88, 6.72, 13, 0.4, 2, 237.0, 500.3), (64, 64, 3.1, 3.1, 40, 0.0, 1, 431.0, 500.0)]


@pytest.mark.parametrize("basis", ["B0", "B1", "SF"])
@pytest.mark.parametrize("case", range(len(FAN)))
@pytest.mark.parametrize("split", [0, 24])
def test_fan_wide_bins(cuda, oracle_exact, basis, case, split):
    from pyoracle import Geometry
    from sgd_amd.torch_ops import Projector
    nx, ny, dx, dy, n, start, nu, du, lso = FAN[case]
    geo = (nx, ny, start + 2 * np.pi * np.arange(n) / n, nu, dx, dy, du, 2 * lso, lso)
    print(basis, FAN[case], split, flush=True)
    if (basis, case) in (("B0", 2), ("B1", 3)):
        # Points whose range ends within a bin's margin of the detector: the
        # model is not zero there and the oracle leaves them out (B0 2.5e-3 in
        # both directions, B1 2.2e-5 in A; no line is lost).
        pytest.xfail("pixels of 50 and more at the detector's end bins")
    P = Projector(basis, *geo)
    P.set_split(split, split)
    check(P, Geometry(oracle_exact, *geo), cuda, basis, case)


@pytest.mark.parametrize("model", ["B1", "SF-TR", "SF-TT"])
@pytest.mark.parametrize("case", range(len(FAN)))
def test_cone_wide_bins(cuda, oracle_exact, model, case):
    from pyoracle import Geometry3
    from sgd_amd.torch_ops import Projector
    nx, ny, dx, dy, n, start, nu, du, lso = FAN[case]
    n = min(n, 21)
    geo = (nx, ny, 5, start + 2 * np.pi * np.arange(n) / n, nu, 9, dx, dy, 1.0, du, 2.0, 2 * lso, lso)
    print(model, FAN[case], flush=True)

    class Oracle:
        g = Geometry3(oracle_exact, *geo)

        def forward(self, _, x):
            return self.g.forward(x) if model == "B1" else self.g.sf_forward(x, trap_v=model == "SF-TT")

        def backward(self, _, y):
            return self.g.backward(y) if model == "B1" else self.g.sf_backward(y, trap_v=model == "SF-TT")

    check(Projector.cone_beam(*geo, model=model), Oracle(), cuda, model, case)
