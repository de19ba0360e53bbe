"""Grouped launches: one footprint evaluation serving a scan's symmetric views
and the images of a batch (sgd_amd/csrc/group2d.hpp).

Full-turn scans with 8, 4 and 2 symmetries (view counts 0 and 2 mod 4, odd;
square and rectangular images, odd sizes; other start angles; alternating
source radius) and without any, against the FP64 oracle at the projector's
parity bar (1e-5 relative L2); a batch of 1..9 images is bit for bit the
images by themselves.  The hexagonal lattices likewise.  The view counts are
high enough that the symmetries are used (256 workgroups of a view and 64
bins)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = {
    "8 symmetries": dict(nx=33, ny=33, views=2056, nu=60),
    "8, two bin chunks": dict(nx=40, ny=40, views=1032, nu=70),
    "4, rectangle": dict(nx=37, ny=18, views=1032, nu=64),
    "4, half turns": dict(nx=31, ny=31, views=1034, nu=61),
    "4, turned start": dict(nx=32, ny=32, views=1028, nu=48, start=0.37),
    "4, flying spot": dict(nx=30, ny=30, views=1032, nu=52, focal=0.6),
    "2, odd": dict(nx=21, ny=34, views=521, nu=63),
    "1": dict(nx=29, ny=29, views=300, nu=55, start=0.2),
}


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("basis", ["B0", "B1", "SF"])
@pytest.mark.parametrize("name", list(CASES))
def test_grouped_matches_oracle(cuda, oracle_exact, basis, name):
    import torch
    from pyoracle import Geometry
    from sgd_amd.torch_ops import Projector
    c = CASES[name]
    n = c["views"]
    ang = c.get("start", 0.0) + 2 * np.pi * np.arange(n) / n
    drho = c["focal"] * (-1.0) ** np.arange(n) if "focal" in c else None
    nx, ny, nu = c["nx"], c["ny"], c["nu"]
    geo = (nx, ny, ang, nu, 1.7, 1.7, 2.9, 1000.0, 500.3)
    P = Projector(basis, *geo, drho=drho)
    G = Geometry(oracle_exact, *geo, drho=drho)
    print(basis, name, c, flush=True)
    rng = np.random.default_rng(7)
    x = rng.random((9, ny, nx)).astype(np.float32)
    y = rng.standard_normal((9, n, nu)).astype(np.float32)
    xt, yt = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    ax, aty = P.forward(xt), P.backward(yt)
    torch.cuda.synchronize()
    for k in (0, 8):
        e1 = rel(ax[k].double().cpu().numpy(), G.forward(basis, x[k].astype(np.float64)))
        e2 = rel(aty[k].double().cpu().numpy(), G.backward(basis, y[k].astype(np.float64)))
        print("  image %d: A %.2e  A^T %.2e" % (k, e1, e2), flush=True)
        assert e1 <= 1e-5 and e2 <= 1e-5, (k, e1, e2)
    for b in (1, 2, 3, 4, 5, 8):
        assert torch.equal(P.forward(xt[:b].contiguous()), ax[:b]), b
        assert torch.equal(P.backward(yt[:b].contiguous()), aty[:b]), b


HEX = {
    "4 symmetries, odd rows": dict(nl=33, nc=20, views=1030, nu=70),
    "2, even rows": dict(nl=24, nc=19, views=1028, nu=63),
    "2, odd views": dict(nl=21, nc=18, views=521, nu=75),
    "1": dict(nl=22, nc=17, views=300, nu=60, start=0.2),
    "1, many workgroups": dict(nl=9, nc=8, views=3000, nu=140, start=0.2),
    "2, most workgroups": dict(nl=10, nc=9, views=6200, nu=130),
}


@pytest.mark.parametrize("basis", ["H0", "Hl"])
@pytest.mark.parametrize("name", list(HEX))
def test_grouped_hex_matches_oracle(cuda, oracle_exact, basis, name):
    import torch
    from pyoracle import HexGeometry
    from sgd_amd.torch_ops import Projector
    c = HEX[name]
    n, nl, nc = c["views"], c["nl"], c["nc"]
    ang = c.get("start", 0.0) + 2 * np.pi * np.arange(n) / n
    geo = (nl, nc, ang, c["nu"], 1.3, 1.1, 1000.0, 500.3)
    P = Projector.hexagonal(basis, *geo)
    G = HexGeometry(oracle_exact, *geo)
    print(basis, name, c, flush=True)
    rng = np.random.default_rng(8)
    x = rng.random((9, nl, nc)).astype(np.float32)
    x[:, 1::2, -1] = 0.0
    y = rng.standard_normal((9, n, c["nu"])).astype(np.float32)
    xt, yt = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    ax, aty = P.forward(xt), P.backward(yt)
    torch.cuda.synchronize()
    for k in (0, 8):
        e1 = rel(ax[k].double().cpu().numpy(), G.forward(basis, x[k].astype(np.float64)))
        e2 = rel(aty[k].double().cpu().numpy(), G.backward(basis, y[k].astype(np.float64)))
        print("  image %d: A %.2e  A^T %.2e" % (k, e1, e2), flush=True)
        assert e1 <= 1e-5 and e2 <= 1e-5, (k, e1, e2)
    assert (aty[:, 1::2, -1] == 0).all()
    for b in (1, 2, 3, 5, 8):
        assert torch.equal(P.forward(xt[:b].contiguous()), ax[:b]), b
        assert torch.equal(P.backward(yt[:b].contiguous()), aty[:b]), b


def test_hex_forward_on_two_streams(cuda):
    """One handle's A on two streams at once (each has its own interleaved
    lattice) equals the calls one after the other."""
    import torch
    from sgd_amd.torch_ops import Projector
    ang = 2 * np.pi * np.arange(1024) / 1024
    P = Projector.hexagonal("Hl", 80, 64, ang, 256, 1.0, 1.2, 1000.0, 500.0)
    g = torch.Generator(device=cuda).manual_seed(3)
    xs = [torch.randn((8,) + P.img_shape, device=cuda, generator=g) for _ in range(6)]
    ref = [P.forward(x) for x in xs]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for k, x in enumerate(xs):
        with torch.cuda.stream(streams[k % 2]):
            outs.append(P.forward(x))
    torch.cuda.synchronize()
    for a, b in zip(ref, outs):
        assert torch.equal(a, b)


CONE = {
    "views on the axes": dict(nx=12, ny=12, views=8),
    "3 classes of 4": dict(nx=13, ny=13, views=12, start=np.pi / 12),
    "rectangle": dict(nx=15, ny=10, views=12),
    "half turns": dict(nx=11, ny=11, views=10, start=0.3),
    "quarter turns": dict(nx=10, ny=10, views=12, start=0.3),
    "odd": dict(nx=9, ny=14, views=9),
    "none": dict(nx=9, ny=9, views=7, start=0.2),
    "many rows": dict(nx=6, ny=6, views=8, nz=300, nv=500),
    "most rows": dict(nx=6, ny=6, views=4, nz=20, nv=512),
    "too many rows": dict(nx=6, ny=6, views=4, nz=20, nv=513),
    "too many voxels": dict(nx=5, ny=5, views=4, nz=513, nv=60),
}


@pytest.mark.parametrize("model", ["B1", "SF-TR", "SF-TT"])
@pytest.mark.parametrize("name", list(CONE))
def test_cone_classes_match_oracle(cuda, oracle_exact, model, name):
    """Cone beam: axial trapezoids shared by the views of a class, on either
    side of the sizes the grouped kernels take."""
    import torch
    from pyoracle import Geometry3
    from sgd_amd.torch_ops import Projector
    c = dict(dict(nz=21, nv=40, start=0.0), **CONE[name])
    ang = c["start"] + 2 * np.pi * np.arange(c["views"]) / c["views"]
    geo = (c["nx"], c["ny"], c["nz"], ang, 45, c["nv"], 1.1, 1.1, 0.9, 1.3, 1.2, 300.0, 150.3)
    P = Projector.cone_beam(*geo, model=model)
    G = Geometry3(oracle_exact, *geo)
    print(model, name, c, flush=True)
    rng = np.random.default_rng(9)
    x = rng.random((2,) + P.img_shape).astype(np.float32)
    y = rng.random((2,) + P.sino_shape).astype(np.float32)
    xt, yt = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    ax, aty = P.forward(xt), P.backward(yt)
    torch.cuda.synchronize()
    tv = model == "SF-TT"
    for k in (0, 1):
        xd, yd = x[k].astype(np.float64), y[k].astype(np.float64)
        e1 = rel(ax[k].double().cpu().numpy(), G.forward(xd) if model == "B1" else G.sf_forward(xd, trap_v=tv))
        e2 = rel(aty[k].double().cpu().numpy(), G.backward(yd) if model == "B1" else G.sf_backward(yd, trap_v=tv))
        print("  A %.2e  A^T %.2e" % (e1, e2), flush=True)
        assert e1 <= 1e-5 and e2 <= 1e-5, (k, e1, e2)
