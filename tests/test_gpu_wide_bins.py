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
