"""An infinite pixel reaches the bins of its corner range and no other: the line
walks of A (SF and the hexagonal lattices) visit a bin's pixels by the FP64 tests
of the corner rule, so that a pixel outside is not multiplied by a zero weight.
Every bin off the pixel's exact range (by 1e-9 of a bin) holds bit for bit what
it holds without the pixel.  Wide fans included, where a strip's edges lean to
both sides and whole lines are tested."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bin_ranges(corners, ang, nu, du, lsd, lso):
    """First and last bin of each view that the corners' box projects into."""
    lo, hi = [], []
    for b in ang:
        c, s = np.cos(b), np.sin(b)
        w = corners - np.array([-lso * c, -lso * s])  # source -> corner
        depth, side = w[:, 0] * c + w[:, 1] * s, -w[:, 0] * s + w[:, 1] * c
        u = side / depth * lsd / du + 0.5 * nu
        lo.append(np.floor(u.min() - 1e-9))
        hi.append(np.floor(u.max() + 1e-9))
    return np.array(lo), np.array(hi)


def check(P, cuda, name, pixels, corners, ang, nu, du, lsd, lso, ends):
    import torch
    rng = np.random.default_rng(4)
    x = torch.from_numpy(rng.random(P.img_shape).astype(np.float32)).to(cuda)
    without = x.repeat(len(pixels), 1, 1)
    for k, (ix, iy) in enumerate(pixels):
        without[k, iy, ix] = 0.0
    with_inf = without.clone()
    for k, (ix, iy) in enumerate(pixels):
        with_inf[k, iy, ix] = float("inf")
    a, b = P.forward(with_inf), P.forward(without)
    u = torch.arange(nu, device=cuda)[None, :]
    wrong = 0
    for k, p in enumerate(pixels):
        lo, hi = (torch.from_numpy(t).to(cuda)[:, None] for t in bin_ranges(corners(*p), ang, nu, du, lsd, lso))
        outside = (u < lo) | (u > hi)
        if not ends:  # ranges are clamped into the detector
            outside[:, [0, nu - 1]] = False
        wrong += int((outside & ~(a[k] == b[k])).sum())
    print(name, "bins changed outside the range:", wrong, flush=True)
    assert wrong == 0


FAN = {
    "full turn": (33, 33, 1.7, 2 * np.pi * np.arange(2056) / 2056, 64, 2.9, 1000.0, 500.3),
    "turned start, rectangle": (41, 30, 1.3, 0.37 + 2 * np.pi * np.arange(501) / 501, 100, 1.6, 1000.0, 500.3),
    "wide fan": (50, 44, 1.0, 0.2 + 2 * np.pi * np.arange(101) / 101, 16, 20.0, 100.0, 60.0),
    "long lines": (700, 40, 0.5, 0.37 + 2 * np.pi * np.arange(201) / 201, 400, 2.0, 1000.0, 500.3),
}


@pytest.mark.parametrize("name", list(FAN))
def test_sf_infinite_pixel(cuda, name):
    from sgd_amd.torch_ops import Projector
    nx, ny, dx, ang, nu, du, lsd, lso = FAN[name]
    P = Projector("SF", nx, ny, ang, nu, dx, dx, du, lsd, lso)
    rng = np.random.default_rng(2)
    pixels = [(int(rng.integers(nx)), int(rng.integers(ny))) for _ in range(24)]

    def corners(ix, iy):
        c = np.array([(ix - 0.5 * (nx - 1)) * dx, (iy - 0.5 * (ny - 1)) * dx])
        return c + 0.5 * dx * np.array([(-1, -1), (-1, 1), (1, -1), (1, 1)])

    check(P, cuda, name, pixels, corners, ang, nu, du, lsd, lso, True)


HEX = {
    "full turn": (33, 20, 1.3, 2 * np.pi * np.arange(1030) / 1030, 70, 1.1, 1000.0, 500.3),
    "turned start": (40, 31, 0.9, 0.2 + 2 * np.pi * np.arange(501) / 501, 90, 1.3, 1000.0, 500.3),
    "wide fan": (44, 30, 0.6, 0.2 + 2 * np.pi * np.arange(101) / 101, 16, 20.0, 100.0, 60.0),
}


@pytest.mark.parametrize("basis", ["H0", "Hl"])
@pytest.mark.parametrize("name", list(HEX))
def test_hex_infinite_point(cuda, basis, name):
    from sgd_amd.torch_ops import Projector
    nl, nc, dt, ang, nu, du, lsd, lso = HEX[name]
    P = Projector.hexagonal(basis, nl, nc, ang, nu, dt, du, lsd, lso)
    rng = np.random.default_rng(2)
    pixels = [(int(rng.integers(nc - 1)), int(rng.integers(nl))) for _ in range(24)]
    dy = dt * (1.5 if basis == "H0" else 0.5)
    turn = np.pi / 2 + np.arange(6) * np.pi / 3

    def corners(ic, il):
        c = np.array([(ic + 0.5 * (il & 1) - 0.5 * (nc - 1)) * np.sqrt(3) * dt, (il - 0.5 * (nl - 1)) * dy])
        return c + dt * np.stack([np.cos(turn), np.sin(turn)], 1)

    check(P, cuda, "%s %s" % (basis, name), pixels, corners, ang, nu, du, lsd, lso, False)
