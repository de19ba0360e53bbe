"""Scans whose views coincide (two and three turns) through the grouped
launches, A and A^T against the FP64 oracle at the projectors' parity bar (1e-5
relative L2).  Every output element is written: the outputs start as NaN.  The
fan scans have enough views for their symmetries to be used (256 workgroups of
a view and 64 bins)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def both(P, cuda, x, y):
    import torch
    ax = torch.full(P.sino_shape, float("nan"), device=cuda)
    aty = torch.full(P.img_shape, float("nan"), device=cuda)
    P.forward(torch.from_numpy(x).to(cuda), out=ax)
    P.backward(torch.from_numpy(y).to(cuda), out=aty)
    torch.cuda.synchronize()
    return ax.double().cpu().numpy(), aty.double().cpu().numpy()


FAN = {
    "B1, 2 turns, 8 symmetries": ("B1", 31, 31, 2064, 1032),
    "B1, 3 turns, rectangle": ("B1", 33, 22, 1080, 360),
    "SF, 2 turns, rectangle": ("SF", 24, 37, 1032, 516),
}


@pytest.mark.parametrize("name", list(FAN))
def test_fan_turns_match_oracle(cuda, oracle_exact, name):
    from pyoracle import Geometry
    from sgd_amd.torch_ops import Projector
    basis, nx, ny, n, per = FAN[name]
    geo = (nx, ny, 2 * np.pi * np.arange(n) / per, 60, 1.7, 1.7, 2.9, 1000.0, 500.3)
    P, G = Projector(basis, *geo), Geometry(oracle_exact, *geo)
    print(name, flush=True)
    rng = np.random.default_rng(11)
    x, y = rng.random((ny, nx)).astype(np.float32), rng.standard_normal((n, 60)).astype(np.float32)
    ax, aty = both(P, cuda, x, y)
    e1 = rel(ax, G.forward(basis, x.astype(np.float64)))
    e2 = rel(aty, G.backward(basis, y.astype(np.float64)))
    print("  A %.2e  A^T %.2e" % (e1, e2), flush=True)
    assert e1 <= 1e-5 and e2 <= 1e-5


def test_hex_turns_match_oracle(cuda, oracle_exact):
    from pyoracle import HexGeometry
    from sgd_amd.torch_ops import Projector
    nl, nc, n = 33, 20, 1032
    geo = (nl, nc, 2 * np.pi * np.arange(n) / 516, 70, 1.3, 1.1, 1000.0, 500.3)
    P, G = Projector.hexagonal("H0", *geo), HexGeometry(oracle_exact, *geo)
    print("H0, 2 turns", flush=True)
    rng = np.random.default_rng(12)
    x, y = rng.random((nl, nc)).astype(np.float32), rng.standard_normal((n, 70)).astype(np.float32)
    x[1::2, -1] = 0.0
    ax, aty = both(P, cuda, x, y)
    e1 = rel(ax, G.forward("H0", x.astype(np.float64)))
    e2 = rel(aty, G.backward("H0", y.astype(np.float64)))
    print("  A %.2e  A^T %.2e" % (e1, e2), flush=True)
    assert e1 <= 1e-5 and e2 <= 1e-5


@pytest.mark.parametrize("model", ["B1", "SF-TR", "SF-TT"])
def test_cone_turns_match_oracle(cuda, oracle_exact, model):
    from pyoracle import Geometry3
    from sgd_amd.torch_ops import Projector
    n = 24
    geo = (12, 12, 21, 2 * np.pi * np.arange(n) / 12, 45, 40, 1.1, 1.1, 0.9, 1.3, 1.2, 300.0, 150.3)
    P, G = Projector.cone_beam(*geo, model=model), Geometry3(oracle_exact, *geo)
    print(model, "2 turns", flush=True)
    rng = np.random.default_rng(13)
    x, y = rng.random(P.img_shape).astype(np.float32), rng.random(P.sino_shape).astype(np.float32)
    ax, aty = both(P, cuda, x, y)
    xd, yd, tv = x.astype(np.float64), y.astype(np.float64), model == "SF-TT"
    e1 = rel(ax, G.forward(xd) if model == "B1" else G.sf_forward(xd, trap_v=tv))
    e2 = rel(aty, G.backward(yd) if model == "B1" else G.sf_backward(yd, trap_v=tv))
    print("  A %.2e  A^T %.2e" % (e1, e2), flush=True)
    assert e1 <= 1e-5 and e2 <= 1e-5
