"""The work that users have this framework do, as cases that can be timed.

Every case is one pass through public entry points on inputs that are resident
where a user's program holds them: projector pairs A / A^T of each basis, from
the smallest image to the largest, one image and batches, the hexagonal
lattices under autograd, the cone beam, a batch of uneven helical slices,
iterative reconstruction, the warm-start network's training step, and the
FP64 host-array operators.

Images are random-ellipse phantoms and fan sinograms their closed-form line
integrals with photon noise, both drawn from the seed.  `exact` evaluates the
same footprints in 64 bits with plain torch: per view a dense matrix D[u, c]
of footprint values, from the definitions (corner rule, box-spline
antiderivatives as sums of truncated powers, trapezoid areas).
"""
import math

import numpy as np
import torch

LSD, LSO = 1000.0, 500.0


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def fan(basis, nx, ny, views, nu, d, du, batch=1, start=0.0, focal=0.0):
    return dict(kind="fan", basis=basis, nx=nx, ny=ny, views=views, nu=nu, d=d, du=du, batch=batch, start=start,
                focal=focal)


def listed():
    return [
        # the smallest call: a test-sized image, where launches and latency count
        dict(fan("B1", 64, 64, 60, 96, 2.4, 3.2), name="fan_b1_64_60v"),
        # the ordinary workload: one 512^2 slice of a full scan
        dict(fan("B1", 512, 512, 720, 768, 0.6, 0.8), name="fan_b1_512_720v"),
        # the same scan with separable footprints
        dict(fan("SF", 512, 512, 720, 768, 0.6, 0.8), name="fan_sf_512_720v"),
        # the largest slice: high-resolution image, long detector
        dict(fan("B1", 2048, 2048, 1440, 3072, 0.15, 0.2), name="fan_b1_2048_1440v"),
        # the warm start's sparse-view data step on a batch of images
        dict(fan("B1", 512, 512, 90, 768, 0.6, 0.8, batch=8), name="fan_b1_512_90v_batch8"),
        # one image on the hexagon-indicator lattice, forward and autograd backward
        dict(kind="hex", basis="H0", nl=296, nc=256, views=1024, nu=1024, dt=0.5, du=0.6, batch=1, name="hex_h0_296"),
        # training with the hexagonal projector as a layer: batch 64
        dict(kind="hex", basis="Hl", nl=296, nc=256, views=1024, nu=1024, dt=0.5, du=0.6, batch=64,
             name="hex_hl_296_batch64"),
        # cone-beam volume
        dict(kind="cone", model="B1", nx=256, ny=256, nz=256, views=360, nu=512, nv=384, d=1.0, du=1.0, dv=1.0,
             name="cone_b1_256_360v"),
        # a helical scan's rebinned slices, uneven in size, views and basis
        dict(kind="slices", count=16, helical=True, set=0, name="slices_16_helical"),
        # SIRT reconstruction from a sparse-view scan (the warm start's input)
        dict(kind="sirt", nx=512, ny=512, views=90, nu=768, d=0.6, du=0.8, batch=4, niter=5, name="sirt_b1_512_90v"),
        # the warm-start network: one training step's gradients
        dict(kind="unet", levels=4, c0=32, batch=8, h=512, w=512, name="unet_grad_512_batch8"),
        # the drop-in operator classes on FP64 host arrays
        dict(kind="host", basis="B0", nx=256, ny=256, views=360, nu=512, d=1.0, du=1.0, name="host_b0_256_360v"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fan_sizes(rng, lo, hi, vlo, vhi):
    n = _log_int(rng, lo, hi)
    nx, ny = (n, n) if rng.random() < 0.7 else (n, max(lo // 2, int(n * rng.uniform(0.5, 1.0))))
    views = _log_int(rng, vlo, vhi)
    d = 307.2 / n
    nu = int(round(1.5 * n)) + rng.randint(0, 7)
    return nx, ny, views, nu, d, 614.4 / nu


def draw(rng):
    kind = rng.choice(["fan"] * 6 + ["hex"] * 2 + ["cone", "slices", "sirt", "unet", "host"])
    if kind == "fan":
        nx, ny, views, nu, d, du = _fan_sizes(rng, 48, 1400, 30, 1400)
        return fan(rng.choice(["B0", "B1", "B1", "SF"]), nx, ny, views, nu, d, du,
                   batch=rng.choice([1, 1, 1, 2, 3, 5, 8]) if nx <= 768 else 1,
                   start=round(rng.uniform(0.0, 6.28), 6) if rng.random() < 0.3 else 0.0,
                   focal=0.6 if rng.random() < 0.2 else 0.0)
    if kind == "hex":
        nc = _log_int(rng, 40, 320)
        nl = int(nc * rng.uniform(0.8, 1.4))
        return dict(kind="hex", basis=rng.choice(["H0", "Hl"]), nl=nl, nc=nc, views=_log_int(rng, 60, 1024),
                    nu=4 * nc + rng.randint(0, 3), dt=0.5 * 256 / nc, du=0.6 * 256 / nc,
                    batch=rng.choice([1, 3, 8, 17, 32]))
    if kind == "cone":
        n = _log_int(rng, 48, 220)
        nz = max(16, int(n * rng.uniform(0.4, 1.1)))
        return dict(kind="cone", model=rng.choice(["B1", "SF-TR", "SF-TT"]), nx=n, ny=n, nz=nz,
                    views=_log_int(rng, 24, 360), nu=2 * n + rng.randint(0, 5), nv=int(1.5 * nz) + rng.randint(0, 5),
                    d=256.0 / n, du=256.0 / n, dv=256.0 / n)
    if kind == "slices":
        return dict(kind="slices", count=rng.randint(2, 16), helical=rng.random() < 0.7, set=rng.randint(1, 10 ** 6))
    if kind == "sirt":
        nx, ny, views, nu, d, du = _fan_sizes(rng, 96, 512, 30, 180)
        return dict(kind="sirt", nx=nx, ny=ny, views=views, nu=nu, d=d, du=du, batch=rng.randint(1, 8),
                    niter=rng.randint(2, 6))
    if kind == "unet":
        return dict(kind="unet", levels=rng.choice([3, 4]), c0=rng.choice([16, 32]), batch=rng.randint(1, 8),
                    h=8 * rng.randint(8, 56), w=8 * rng.randint(8, 56))
    nx, ny, views, nu, d, du = _fan_sizes(rng, 64, 512, 45, 720)
    return dict(kind="host", basis=rng.choice(["B0", "B1"]), nx=nx, ny=ny, views=views, nu=nu, d=d, du=du)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _angles(n, start=0.0):
    return start + 2 * np.pi * np.arange(n) / n


def _focal(case):
    """Flying focal spot: the source radius alternates by the given amount."""
    f = case.get("focal", 0.0)
    return f * np.where(np.arange(case["views"]) % 2 == 0, 1.0, -1.0) if f else None


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed) * 7919 + 13)


def _ellipses(seed, n=10):
    """(cx, cy, a, b, angle, density) in units of the field of view's half-width."""
    rng = np.random.default_rng(int(seed) * 104729 + 5)
    r, phi = 0.8 * np.sqrt(rng.uniform(size=n)), 2 * np.pi * rng.uniform(size=n)
    return np.stack([r * np.cos(phi), r * np.sin(phi), rng.uniform(0.05, 0.4, n), rng.uniform(0.05, 0.4, n),
                     rng.uniform(0, np.pi, n), rng.uniform(0.1, 1.0, n)], 1)


def _raster(seed, X, Y, half):
    out = torch.zeros_like(X)
    for cx, cy, a, b, ang, d in _ellipses(seed):
        c, s = math.cos(ang), math.sin(ang)
        xr, yr = (X / half - cx) * c + (Y / half - cy) * s, -(X / half - cx) * s + (Y / half - cy) * c
        out += d * ((xr / a) ** 2 + (yr / b) ** 2 <= 1.0)
    return out


def _grid(nx, ny, d):
    xs = (torch.arange(nx, device=_dev(), dtype=torch.float64) - 0.5 * (nx - 1)) * d
    ys = (torch.arange(ny, device=_dev(), dtype=torch.float64) - 0.5 * (ny - 1)) * d
    Y, X = torch.meshgrid(ys, xs, indexing="ij")
    return X, Y


def _images(seed, batch, nx, ny, d):
    X, Y = _grid(nx, ny, d)
    return torch.stack([_raster(64 * seed + k, X, Y, 0.5 * min(nx, ny) * d) for k in range(batch)]).float()


def _sinograms(seed, batch, angles, nu, du, half):
    """Line integrals of the phantoms through the bin centres, with the noise
    of 1e5 photons per ray (attenuation 0.02 per unit)."""
    b = torch.as_tensor(np.asarray(angles), device=_dev())[:, None]
    t = ((torch.arange(nu, device=_dev(), dtype=torch.float64) + 0.5 - 0.5 * nu) * du)[None, :]
    px, py = -LSO * torch.cos(b), -LSO * torch.sin(b)
    vx, vy = LSD * torch.cos(b) - t * torch.sin(b), LSD * torch.sin(b) + t * torch.cos(b)
    r = torch.sqrt(vx * vx + vy * vy)
    vx, vy = vx / r, vy / r
    out = []
    for k in range(batch):
        y = torch.zeros_like(r)
        for cx, cy, a, bb, ang, d in _ellipses(64 * seed + k):
            c, s = math.cos(ang), math.sin(ang)
            ox, oy = px - cx * half, py - cy * half
            A, B = a * half, bb * half
            o1, o2 = (ox * c + oy * s) / A, (-ox * s + oy * c) / B
            w1, w2 = (vx * c + vy * s) / A, (-vx * s + vy * c) / B
            qa, qb, qc = w1 * w1 + w2 * w2, o1 * w1 + o2 * w2, o1 * o1 + o2 * o2 - 1.0
            y += d * 2.0 * torch.sqrt(torch.clamp(qb * qb - qa * qc, min=0.0)) / qa
        n = torch.randn(y.shape, generator=_gen(64 * seed + k), device=_dev(), dtype=torch.float64)
        out.append(y + n * torch.exp(0.01 * y) / (0.02 * math.sqrt(1e5)))
    return torch.stack(out).float()


def _slice_specs(case):
    from sgd_amd.batch import uneven_slices
    return uneven_slices(case["count"], seed=case["set"], sizes=(128, 256, 384, 512, 768), views=(180, 1440),
                         helical=case["helical"])


def _hex_points(case):
    dt, nl, nc = case["dt"], case["nl"], case["nc"]
    dx, dy = dt * math.sqrt(3.0), (1.5 if case["basis"] == "H0" else 0.5) * dt
    il = torch.arange(nl, device=_dev(), dtype=torch.float64)
    ic = torch.arange(nc, device=_dev(), dtype=torch.float64)
    Y = ((il - 0.5 * (nl - 1)) * dy)[:, None].expand(nl, nc)
    X = (ic[None, :] + 0.5 * (il % 2)[:, None] - 0.5 * (nc - 1)) * dx
    ok = ~((il % 2 == 1)[:, None] & (ic == nc - 1)[None, :])
    return X.contiguous(), Y.contiguous(), ok, dx, dy


def _unet_target(seed, case):
    X, Y = _grid(case["w"], case["h"], 1.0)
    half = 0.5 * min(case["w"], case["h"])
    clean = torch.stack([_raster(64 * seed + k, X, Y, half) for k in range(case["batch"])])
    g = _gen(seed)
    noise = torch.randn(clean.shape, generator=g, device=_dev(), dtype=torch.float64)
    smooth = torch.nn.functional.avg_pool2d((clean + 0.2 * noise)[:, None], 5, stride=1, padding=2)[:, 0]
    return smooth.float().contiguous(), clean.float().contiguous()


def prepare(case, seed):
    from sgd_amd.torch_ops import Projector
    kind = case["kind"]
    s = dict(case=case)
    if kind == "fan":
        ang = _angles(case["views"], case["start"])
        s["P"] = Projector(case["basis"], case["nx"], case["ny"], ang, case["nu"], case["d"], case["d"], case["du"], LSD,
                           LSO, drho=_focal(case))
        s["x"] = _images(seed, case["batch"], case["nx"], case["ny"], case["d"])
        s["y"] = _sinograms(seed + 1, case["batch"], ang, case["nu"], case["du"],
                            0.5 * min(case["nx"], case["ny"]) * case["d"])
        if case["batch"] == 1:
            s["x"], s["y"] = s["x"][0], s["y"][0]
    elif kind == "hex":
        s["P"] = Projector.hexagonal(case["basis"], case["nl"], case["nc"], _angles(case["views"]), case["nu"],
                                     case["dt"], case["du"], LSD, LSO)
        X, Y, ok, dx, dy = _hex_points(case)
        half = 0.5 * min(case["nc"] * dx, case["nl"] * dy)
        x = torch.stack([_raster(64 * seed + k, X, Y, half) * ok for k in range(case["batch"])]).float()
        s["x"] = x.requires_grad_(True)
        s["y"] = _sinograms(seed + 1, case["batch"], _angles(case["views"]), case["nu"], case["du"], half)
    elif kind == "cone":
        c = case
        s["P"] = Projector.cone_beam(c["nx"], c["ny"], c["nz"], _angles(c["views"]), c["nu"], c["nv"], c["d"], c["d"],
                                     c["d"], c["du"], c["dv"], LSD, LSO, model=c["model"])
        X, Y = _grid(c["nx"], c["ny"], c["d"])
        half = 0.5 * c["nx"] * c["d"]
        z = torch.linspace(-1.0, 1.0, c["nz"], device=_dev(), dtype=torch.float64)[:, None, None]
        a, b = _raster(2 * seed, X, Y, half), _raster(2 * seed + 1, X, Y, half)
        s["x"] = (a * (z.abs() < 0.8) + b * torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))).float().contiguous()
        y = _sinograms(seed + 1, 1, _angles(c["views"]), c["nu"], c["du"], half)[0]
        v = torch.linspace(-1.0, 1.0, c["nv"], device=_dev())[None, :, None]
        n = torch.randn((c["views"], c["nv"], c["nu"]), generator=_gen(seed), device=_dev())
        s["y"] = (y[:, None, :] * (1.0 - 0.5 * v * v) + n).contiguous()
    elif kind == "slices":
        from sgd_amd.batch import SliceBatch, make_projectors
        specs = _slice_specs(case)
        s["B"] = SliceBatch(make_projectors(specs))
        xs, ys = [], []
        for k, p in enumerate(specs):
            xs.append(_images(seed + 31 * k, 1, p["nx"], p["ny"], p["dx"]))
            ys.append(_sinograms(seed + 31 * k + 1, 1, p["angles"], p["nu"], p["du"], 0.5 * p["nx"] * p["dx"]))
        s["x"], s["y"] = s["B"].pack_images(xs), s["B"].pack_sinos(ys)
    elif kind == "sirt":
        from sgd_amd.solvers import SirtWeights
        ang = _angles(case["views"])
        s["P"] = Projector("B1", case["nx"], case["ny"], ang, case["nu"], case["d"], case["d"], case["du"], LSD, LSO)
        s["w"] = SirtWeights(s["P"])
        s["y"] = _sinograms(seed, case["batch"], ang, case["nu"], case["du"],
                            0.5 * min(case["nx"], case["ny"]) * case["d"])
    elif kind == "unet":
        from sgd_amd.unet import UNet
        s["net"] = UNet(case["levels"], case["c0"], seed=3)
        s["x"], s["t"] = _unet_target(seed, case)
    elif kind == "host":
        from sgd_amd import operators
        cls = operators.A_B0_operator if case["basis"] == "B0" else operators.A_B1_operator
        ang = _angles(case["views"])
        s["op"] = cls(case["nx"], case["ny"], case["views"], case["nu"], case["d"], case["d"], case["du"], LSD, LSO, ang)
        x = _images(seed, 1, case["nx"], case["ny"], case["d"])[0]
        y = _sinograms(seed + 1, 1, ang, case["nu"], case["du"], 0.5 * min(case["nx"], case["ny"]) * case["d"])[0]
        s["x"], s["y"] = x.T.contiguous().double().cpu().numpy().ravel(), y.double().cpu().numpy().ravel()
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind in ("fan", "cone"):
        P = state["P"]
        return {"A": P.forward(state["x"]), "At": P.backward(state["y"])}
    if kind == "hex":
        from sgd_amd.torch_ops import project
        x = state["x"]
        x.grad = None
        y = project(x, state["P"])
        y.backward(state["y"])
        return {"A": y.detach(), "grad": x.grad}
    if kind == "slices":
        B = state["B"]
        return {"A": B.forward(state["x"]), "At": B.backward(state["y"])}
    if kind == "sirt":
        from sgd_amd.solvers import sirt_batch
        return {"x": sirt_batch(state["P"], state["y"], state["case"]["niter"], weights=state["w"])}
    if kind == "unet":
        net = state["net"]
        y = net.forward(state["x"])
        net.backward(state["t"])
        out = {"y": y, "head": net.head_g}
        for name, c in net.convs.items():
            out[name + "_w"], out[name + "_b"] = c.gw, c.gb
        return out
    op = state["op"]
    return {"A": op.matvec(state["x"]), "At": op.rmatvec(state["y"])}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(npix, views, reach, d, du):
    """(pixel, bin) pairs of one image and direction: the mean bin range of a
    pixel of half-extent `reach` pixels, over all views."""
    return npix * views * (2.0 * reach * (4.0 / math.pi) * d * (LSD / LSO) / du + 1.0)


def work(case):
    """Each input read and each output written once; one multiply-add for
    every footprint value that is not zero by the corner rule."""
    kind = case["kind"]
    if kind in ("fan", "sirt", "host"):
        npix, nsin = case["nx"] * case["ny"], case["views"] * case["nu"]
        b = case.get("batch", 1)
        reach = 1.0 if case.get("basis", "B1") == "B1" else 0.5
        it = case.get("niter", 1)
        f = 2.0 * 2.0 * _pairs(npix, case["views"], reach, case["d"], case["du"]) * b * it
        if kind == "sirt":
            return {"bytes": 4.0 * b * (npix + nsin), "flops": f}
        return {"bytes": (8.0 if kind == "host" else 4.0) * 2 * b * (npix + nsin), "flops": f}
    if kind == "hex":
        npix, nsin, b = case["nl"] * case["nc"], case["views"] * case["nu"], case["batch"]
        return {"bytes": 4.0 * 2 * b * (npix + nsin),
                "flops": 4.0 * b * _pairs(npix, case["views"], 1.0, case["dt"], case["du"])}
    if kind == "cone":
        ncol, nz = case["nx"] * case["ny"], case["nz"]
        reach = 1.0 if case["model"] == "B1" else 0.5
        mag = LSD / LSO
        rows = nz * (case["d"] * mag / case["dv"] + 1.0)          # (voxel, row) pairs of a column
        pair_uv = _pairs(ncol, case["views"], reach, case["d"], case["du"]) * min(case["nv"], nz * case["d"] * mag)
        return {"bytes": 4.0 * 2 * (ncol * nz + case["views"] * case["nu"] * case["nv"]),
                "flops": 4.0 * (pair_uv + ncol * case["views"] * rows)}
    if kind == "slices":
        by, fl = 0.0, 0.0
        for p in _slice_specs(case):
            npix = p["nx"] * p["ny"]
            by += 8.0 * (npix + p["np"] * p["nu"])
            fl += 4.0 * _pairs(npix, p["np"], 1.0 if p["basis"] == "B1" else 0.5, p["dx"], p["du"])
        return {"bytes": by, "flops": fl}
    from sgd_amd.unet import layer_specs
    by, fl = 3 * 4.0 * case["batch"] * case["h"] * case["w"], 0.0
    for name, ci, co, k in layer_specs(case["levels"], case["c0"]):
        lvl = int(name[3]) if name != "out" else 0
        pix = case["batch"] * (case["h"] >> lvl) * (case["w"] >> lvl)
        fl += 3 * 2.0 * k * k * ci * co * pix       # forward, input gradient, weight gradient
        by += 2 * 2.0 * co * pix                    # activation written, read again in backward
        by += 3 * 4.0 * k * k * ci * co
    return {"bytes": by, "flops": fl}


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------
F64 = torch.float64


def _trunc(x, n):
    return torch.clamp(x, min=0.0) ** n


class _View:
    """One view's geometry: source p, edge rays E_k - p, per-bin tables."""

    def __init__(self, angle, nu, du, drho=0.0, shift=0.0):
        c, s = math.cos(angle), math.sin(angle)
        self.px, self.py = (-LSO + drho) * c, (-LSO + drho) * s
        self.pux, self.puy = -du * s, du * c
        self.e0x = (LSD - LSO) * c - (0.5 * nu + shift) * self.pux - self.px
        self.e0y = (LSD - LSO) * s - (0.5 * nu + shift) * self.puy - self.py
        self.nu = nu
        k = torch.arange(nu, device=_dev(), dtype=F64)
        ax, ay = self.e0x + k * self.pux, self.e0y + k * self.puy
        bx, by = ax + self.pux, ay + self.puy
        self.cx, self.cy = ax + 0.5 * self.pux, ay + 0.5 * self.puy
        ln = torch.sqrt(self.cx ** 2 + self.cy ** 2)
        self.ka, self.kb = -ln / (ax * self.cx + ay * self.cy), -ln / (bx * self.cx + by * self.cy)

    def coord(self, X, Y):
        wx, wy = X - self.px, Y - self.py
        return -(self.e0x * wy - self.e0y * wx) / (self.pux * wy - self.puy * wx)

    def reach(self, X, Y, corners):
        us = [self.coord(X + a, Y + b) for a, b in corners]
        lo, hi = us[0], us[0]
        for u in us[1:]:
            lo, hi = torch.minimum(lo, u), torch.maximum(hi, u)
        return lo, hi

    def offsets(self, X, Y, u):
        """ta, tb of pixel centres at bins u."""
        wx, wy = X - self.px, Y - self.py
        n0, be = self.e0x * wy - self.e0y * wx, self.pux * wy - self.puy * wx
        return self.ka[u] * (n0 + u * be), self.kb[u] * (n0 + (u + 1) * be)


def _spline_cdf(t, nodes, power, scale):
    """Odd antiderivative of a box spline from its truncated powers: the sum
    over (node, weight) of weight (x - node)_+^power / scale at x = -|t|."""
    x = -t.abs()
    s = torch.zeros_like(x)
    for node, w in nodes:
        s = s + w * _trunc(x - node, power)
    return torch.sign(t) * (0.5 - s / scale)


def _box_nodes(widths):
    """Nodes of the convolution of centred boxes of these widths."""
    nodes = [(torch.zeros_like(widths[0]), 1.0)]
    for w in widths:
        nodes = [(n + sg * 0.5 * w, c * (-sg)) for n, c in nodes for sg in (-1.0, 1.0)]
    return nodes


def _mean(cdf, ta, tb):
    return (cdf(tb) - cdf(ta)) / (tb - ta)


def _b0_mean(ta, tb, p, q):
    two = _mean(lambda t: _spline_cdf(t, _box_nodes([p, q]), 2, 2.0 * p * q), ta, tb)
    one = _mean(lambda t: torch.sign(t) * torch.minimum(t.abs() / p, torch.full_like(t, 0.5)), ta, tb)
    return torch.where(q > 1e-6 * p, two, one)


def _b1_mean(ta, tb, a, b):
    four = _mean(lambda t: _spline_cdf(t, _box_nodes([a, a, b, b]), 4, 24.0 * a * a * b * b), ta, tb)
    two = _mean(lambda t: _spline_cdf(t, _box_nodes([a, a]), 2, 2.0 * a * a), ta, tb)
    return torch.where(b > 1e-4 * a, four, two)


def _hl_mean(ta, tb, p, q, r):
    three = _mean(lambda t: _spline_cdf(t, _box_nodes([p, q, r]), 3, 6.0 * p * q * r), ta, tb)
    return torch.where(r > 1e-5 * p, three, _b0_mean(ta, tb, p, q))


def _trap_area(q, lo, hi):
    """Area over [lo, hi] of the unit-height trapezoid with sorted corners q."""
    q0, q1, q2, q3 = q

    def F(s):
        r = torch.clamp(s, q0, q1) - q0
        f = q3 - torch.clamp(s, q2, q3)
        rise = torch.where(q1 > q0, r * r / (2 * (q1 - q0)).clamp_min(1e-300), torch.zeros_like(r))
        full = torch.where(q3 > q2, (q3 - q2) * 0.5, torch.zeros_like(r))
        fall = torch.where(q3 > q2, full - f * f / (2 * (q3 - q2)).clamp_min(1e-300), torch.zeros_like(r))
        return rise + (torch.clamp(s, q1, q2) - q1) + fall

    return F(hi) - F(lo)


def _square(h, d):
    return [(a * h * d, b * h * d) for a in (-1, 1) for b in (-1, 1)]


def _matrix(basis, view, X, Y, d, dt=None, ok=None):
    """Dense D[u, c] of one view: footprint of every pixel c in every bin u."""
    nu = view.nu
    D = torch.zeros((nu, X.numel()), device=X.device, dtype=F64)
    if basis in ("H0", "Hl"):
        corners = [(dt * math.cos(math.pi / 2 + k * math.pi / 3), dt * math.sin(math.pi / 2 + k * math.pi / 3))
                   for k in range(6)]
    else:
        corners = _square(1.0 if basis in ("B1", "C1") else 0.5, d)
    lo, hi = view.reach(X, Y, corners)
    if basis == "CSF":     # cells outside the detector take nothing
        ulo, uhi = torch.floor(lo).long(), torch.floor(hi).long()
    else:
        ulo, uhi = torch.floor(lo).long().clamp(0, nu - 1), torch.floor(hi).long().clamp(0, nu - 1)
    col = torch.arange(X.numel(), device=X.device)
    if basis in ("SF", "CSF"):
        q = torch.sort(torch.stack([view.coord(X + a, Y + b) for a, b in corners]), dim=0).values
        wx, wy = X - view.px, Y - view.py
        amp = d * torch.sqrt(wx ** 2 + wy ** 2) / torch.maximum(wx.abs(), wy.abs())
        if basis == "CSF":
            amp = 2.0 / ((q[3] - q[0]) + (q[2] - q[1]))
    elif basis in ("H0", "Hl"):
        th = torch.atan2(view.cx, view.cy)
        vk = [dt * torch.sin(th + 2 * math.pi * k / 3) for k in range(3)]
    else:
        th = torch.atan2(view.cx.abs(), view.cy.abs())
        vx, vy = (d * torch.cos(th)).abs(), (d * torch.sin(th)).abs()
        big, small = torch.maximum(vx, vy), torch.minimum(vx, vy)
    for j in range(int((uhi - ulo).max()) + 1):
        u = ulo + j
        m = (u <= uhi) & (u >= 0) & (u < nu)
        if ok is not None:
            m = m & ok
        c = col[m]
        u = u[m]
        if basis in ("SF", "CSF"):
            s = u.to(F64)
            g = _trap_area([v[m] for v in q], s, s + 1.0)
            w = torch.where(g > 1e-7, g, torch.zeros_like(g)) * amp[m] if basis == "SF" else g * amp[m]
        else:
            ta, tb = view.offsets(X[m], Y[m], u)
            if basis == "B0":
                w = _b0_mean(ta, tb, big[u], small[u]) * d * d
            elif basis in ("B1", "C1"):
                w = _b1_mean(ta, tb, big[u], small[u]) * (d * d if basis == "B1" else 1.0)
            elif basis == "Hl":
                v = torch.sort(torch.stack([k.abs() for k in vk]), dim=0).values
                w = _hl_mean(ta, tb, v[2][u], v[1][u], v[0][u]).clamp_min(0.0)
            else:
                w = torch.zeros_like(ta)
                for i, k in ((0, 1), (1, 2), (2, 0)):
                    va, vb = vk[i][u], vk[k][u]
                    mid = 0.5 * (va + vb)
                    w = w + _b0_mean(ta - mid, tb - mid, torch.maximum(va.abs(), vb.abs()),
                                     torch.minimum(va.abs(), vb.abs())) / 3.0
                w = w.clamp_min(0.0)
        D[u, c] = w
    return D


def _apply(make, views, nu, x, y):
    """A x and A^T y over all views; x [npix, B], y [views, nu, B]; either may be None."""
    ax = torch.zeros((views, nu, x.shape[1]), device=_dev(), dtype=F64) if x is not None else None
    aty = None
    for v in range(views):
        D = make(v)
        if x is not None:
            ax[v] = D @ x
        if y is not None:
            t = D.T @ y[v]
            aty = t if aty is None else aty + t
        del D
    return ax, aty


def _fan_maker(basis, nx, ny, d, angles, nu, du, drho=None):
    X, Y = _grid(nx, ny, d)
    X, Y = X.reshape(-1), Y.reshape(-1)
    return lambda v: _matrix(basis, _View(angles[v], nu, du, 0.0 if drho is None else drho[v]), X, Y, d)


def _fan_exact(basis, nx, ny, d, angles, nu, du, drho, x, y):
    """x (B, ny, nx), y (B, views, nu) -> the same shapes of A x, A^T y."""
    mk = _fan_maker(basis, nx, ny, d, angles, nu, du, drho)
    b = x.shape[0]
    ax, aty = _apply(mk, len(angles), nu, x.reshape(b, -1).T.to(F64), y.permute(1, 2, 0).to(F64))
    return ax.permute(2, 0, 1).contiguous(), aty.T.reshape(b, ny, nx).contiguous()


def _too_much(npix, views, nu):
    return npix * nu > 1.2e9 or float(npix) * nu * views > 4e11


def _cone_exact(case, x, y):
    """x [nz, ny, nx], y [views, nv, nu] -> A x, A^T y."""
    model, d, dv, nz, nv, nu = case["model"], case["d"], case["dv"], case["nz"], case["nv"], case["nu"]
    X, Y = _grid(case["nx"], case["ny"], d)
    X, Y = X.reshape(-1), Y.reshape(-1)
    ncol = X.numel()
    xt = x.to(F64).reshape(nz, ncol).T.contiguous()
    zc = torch.arange(nz, device=_dev(), dtype=F64) - 0.5 * (nz - 1)
    off = {"B1": 1.0, "SF-TT": 0.5, "SF-TR": 0.0}[model]
    ro = 0.0 if model == "B1" else -0.5
    A = torch.zeros((case["views"], nv, nu), device=_dev(), dtype=F64)
    T = torch.zeros_like(xt)
    ang = _angles(case["views"])
    for p in range(case["views"]):
        view = _View(ang[p], nu, case["du"], shift=0.0 if model == "B1" else 0.5)
        D = _matrix("C1" if model == "B1" else "CSF", view, X, Y, d)

        def slope(ex):  # detector rows per voxel index at the corner X + ex
            depth = (view.puy * (X + ex - view.px) - view.pux * (Y - view.py)) / case["du"]
            return (LSD * d / dv / depth)[:, None]

        ka, kb, vc = slope(-off * d), slope(off * d), 0.5 * nv
        a1, a2, b1, b2 = (vc + ka * (zc - 0.5), vc + ka * (zc + 0.5), vc + kb * (zc - 0.5), vc + kb * (zc + 0.5))
        v0, v3 = torch.minimum(a1, b1), torch.maximum(a2, b2)
        h1, l2 = torch.maximum(a1, b1), torch.minimum(a2, b2)
        v1, v2 = torch.minimum(h1, l2), torch.maximum(h1, l2)
        r2 = ((X - view.px) ** 2 + (Y - view.py) ** 2)[:, None]
        oz = zc * d
        if model == "B1":
            cf = d ** 3 * torch.sqrt(1.0 + oz * oz / r2) * 2.0 / ((v3 - v0) + (v2 - v1))
        else:
            if model == "SF-TR":
                v1, v2 = v0, v3
            area = v3 - v0 if model == "SF-TR" else 0.5 * ((v3 - v0) + (v2 - v1))
            cf = LSD * LSD * d ** 3 / (case["du"] * dv) / ((r2 + oz * oz) * area)
        del a1, a2, b1, b2, h1, l2
        jlo, jhi = torch.floor(v0 - ro).long(), torch.floor(v3 - ro).long()
        Yp = torch.zeros((ncol, nv + 1), device=_dev(), dtype=F64)   # the last entry takes rows off the detector
        Yb = torch.cat([D.T @ y[p].to(F64).T, torch.zeros((ncol, 1), device=_dev(), dtype=F64)], 1)
        xc = xt * cf
        for j in range(int((jhi - jlo).max()) + 1):
            row = jlo + j
            s = row.to(F64) + ro
            g = _trap_area((v0, v1, v2, v3), s, s + 1.0)
            if model == "B1":
                g = torch.where(g > 1e-7, g, torch.zeros_like(g))
            g = torch.where((row <= jhi) & (row >= 0) & (row < nv), g, torch.zeros_like(g))
            at = torch.where((row >= 0) & (row < nv), row, torch.full_like(row, nv))
            Yp.scatter_add_(1, at, xc * g)
            T += cf * g * torch.gather(Yb, 1, at)
        A[p] = (D @ Yp[:, :nv]).T
    return A, T.T.reshape(nz, case["ny"], case["nx"]).contiguous()


def _unet_exact(case, x, t):
    """The network in 64 bits by shifted products; gradients by autograd."""
    from sgd_amd.unet import init_params
    params = {k: (torch.as_tensor(W, device=_dev(), dtype=F64), torch.as_tensor(b, device=_dev(), dtype=F64))
              for k, (W, b) in init_params(case["levels"], case["c0"], 3).items()}
    for W, b in params.values():
        W.requires_grad_(True), b.requires_grad_(True)

    def conv(name, v):                       # NHWC, 3 x 3, zero padding, ReLU
        W, b = params[name]
        p = torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1))
        H, Wd = v.shape[1], v.shape[2]
        out = b
        for ky in range(3):
            for kx in range(3):
                out = out + p[:, ky:ky + H, kx:kx + Wd].reshape(-1, v.shape[3]) @ W[:, ky, kx].T
        return torch.relu(out).reshape(v.shape[0], H, Wd, -1)

    L = case["levels"]
    v = torch.nn.functional.pad(x.to(F64)[..., None], (0, 7))
    enc = []
    for l in range(L):
        if l:
            B, H, W, C = enc[-1].shape
            v = enc[-1].reshape(B, H // 2, 2, W // 2, 2, C).mean(dim=(2, 4))
        enc.append(conv("enc%d_b" % l, conv("enc%d_a" % l, v)))
    d = enc[-1]
    for l in range(L - 2, -1, -1):
        up = d.repeat_interleave(2, 1).repeat_interleave(2, 2)
        d = conv("dec%d_b" % l, conv("dec%d_a" % l, torch.cat([up, enc[l]], 3)))
    W, b = params["out"]
    y = x.to(F64) + (d * W.reshape(-1)).sum(3) + b
    ((y - t.to(F64)) ** 2).mean().backward()
    out = {"y": y.detach(), "head": torch.cat([W.grad.reshape(-1), b.grad])}
    for name, (W, b) in params.items():
        if name != "out":
            out[name + "_w"], out[name + "_b"] = W.grad.reshape(W.shape[0], -1), b.grad
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fan", "sirt", "host"):
        ang = _angles(case["views"], case.get("start", 0.0))
        npix = case["nx"] * case["ny"]
        if _too_much(npix, case["views"] * case.get("niter", 1), case["nu"]):
            return None
        geo = (case["nx"], case["ny"], case["d"], ang, case["nu"], case["du"])
        half = 0.5 * min(case["nx"], case["ny"]) * case["d"]
        b = case.get("batch", 1)
        if kind == "sirt":
            y = _sinograms(seed, b, ang, case["nu"], case["du"], half).permute(1, 2, 0).to(F64)
            mk = _fan_maker("B1", *geo)
            one = torch.ones((npix, 1), device=_dev(), dtype=F64)
            rs, cs = _apply(mk, case["views"], case["nu"], one, torch.ones_like(y[..., :1]))
            W = torch.where(rs > 1e-8, 1.0 / rs.clamp_min(1e-8), torch.zeros_like(rs))
            V = torch.where(cs > 1e-8, 1.0 / cs.clamp_min(1e-8), torch.zeros_like(cs))
            x = torch.zeros((npix, b), device=_dev(), dtype=F64)
            for _ in range(case["niter"]):
                c = torch.zeros_like(x)
                for v in range(case["views"]):
                    D = mk(v)
                    c += D.T @ (W[v] * (y[v] - D @ x))
                x = torch.clamp(x + V * c, min=0.0)
            return {"x": x.T.reshape(b, case["ny"], case["nx"])}
        x = _images(seed, b, case["nx"], case["ny"], case["d"])
        y = _sinograms(seed + 1, b, ang, case["nu"], case["du"], half)
        A, At = _fan_exact(case["basis"], *geo, _focal(case), x, y)
        if kind == "host":
            return {"A": A.reshape(-1), "At": At[0].T.reshape(-1)}
        return {"A": A[0], "At": At[0]} if b == 1 else {"A": A, "At": At}
    if kind == "hex":
        if _too_much(case["nl"] * case["nc"], case["views"], case["nu"]):
            return None
        X, Y, ok, dx, dy = _hex_points(case)
        half = 0.5 * min(case["nc"] * dx, case["nl"] * dy)
        b = case["batch"]
        x = torch.stack([_raster(64 * seed + k, X, Y, half) * ok for k in range(b)]).float()
        ang = _angles(case["views"])
        y = _sinograms(seed + 1, b, ang, case["nu"], case["du"], half)
        X, Y, m = X.reshape(-1), Y.reshape(-1), ok.reshape(-1)
        A, At = _apply(lambda v: _matrix(case["basis"], _View(ang[v], case["nu"], case["du"]), X, Y, dx,
                                         dt=case["dt"], ok=m) * (dx * dy),
                       case["views"], case["nu"], x.reshape(b, -1).T.to(F64), y.permute(1, 2, 0).to(F64))
        return {"A": A.permute(2, 0, 1).contiguous(), "grad": At.T.reshape(b, case["nl"], case["nc"]).contiguous()}
    if kind == "cone":
        if float(case["nx"]) * case["ny"] * case["nz"] * case["views"] > 8e9:
            return None
        s = prepare(case, seed)
        A, At = _cone_exact(case, s["x"], s["y"])
        return {"A": A, "At": At}
    if kind == "slices":
        specs = _slice_specs(case)
        if sum(float(p["nx"] * p["ny"]) * p["np"] * p["nu"] for p in specs) > 3e12:
            return None
        As, Ats = [], []
        for k, p in enumerate(specs):
            x = _images(seed + 31 * k, 1, p["nx"], p["ny"], p["dx"])
            y = _sinograms(seed + 31 * k + 1, 1, p["angles"], p["nu"], p["du"], 0.5 * p["nx"] * p["dx"])
            A, At = _fan_exact(p["basis"], p["nx"], p["ny"], p["dx"], p["angles"], p["nu"], p["du"], p.get("drho"), x, y)
            As.append(A.reshape(-1)), Ats.append(At.reshape(-1))
        return {"A": torch.cat(As), "At": torch.cat(Ats)}
    return _unet_exact(case, *_unet_target(seed, case))
