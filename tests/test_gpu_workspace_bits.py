"""A's values do not depend on the workspace a launch finds: through the 32 MiB
array of sgdct_project_dev_noalloc, which holds the interleaved images of all
the scan's symmetries, of some, or of none (read in place), and under capture,
where an unsplit A reads its images in place, every output is bit for bit that
of sgdct_forward_dev at the same split."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fan(basis, nx, ny, views, nu, fwd, bwd):
    from sgd_amd.torch_ops import Projector
    dx = 400.0 / max(nx, ny)
    P = Projector(basis, nx, ny, 2 * np.pi * np.arange(views) / views, nu, dx, dx, 850.0 / nu, 1000.0, 700.0)
    P.set_split(fwd, bwd)
    return P


def hexagonal(basis, nl, nc, views, nu, fwd, bwd):
    from sgd_amd.torch_ops import Projector
    dt = 200.0 / max(nl, nc)
    P = Projector.hexagonal(basis, nl, nc, 2 * np.pi * np.arange(views) / views, nu, dt, 850.0 / nu, 1000.0, 700.0)
    P.set_split(fwd, bwd)
    return P


NOALLOC = {  # interleaved and transposed copies of one image against 32 MiB
    "B1, 8 symmetries": (fan, "B1", 512, 512, 256, 512, 24, 1, 2),           # 16 MiB
    "B1, 8 as 4": (fan, "B1", 767, 767, 256, 512, 24, 1, 1),                 # 36 MiB
    "SF, 8 as 2": (fan, "SF", 1030, 1030, 256, 512, 0, 1, 1),                # 65 MiB
    "B1, 8 in place": (fan, "B1", 1600, 1600, 256, 512, 24, 1, 1),           # 156 MiB
    "SF, 4 in place, whole": (fan, "SF", 2100, 1500, 256, 512, 1, 1, 1),     # 96 MiB
    "B0, images of a batch": (fan, "B0", 900, 700, 40, 200, 24, 1, 5),       # 5 MiB an image
    "Hl, 4 as 2": (hexagonal, "Hl", 1301, 1300, 512, 500, 0, 1, 2),          # 26 MiB an image at 4
    "H0, 4 in place": (hexagonal, "H0", 2301, 2000, 512, 500, 0, 1, 1),      # 70 MiB
    "H0, 2 in place, segments": (hexagonal, "H0", 2400, 2000, 512, 500, 3, 1, 1),
}


@pytest.mark.parametrize("name", list(NOALLOC))
def test_noalloc_is_bitwise_the_device_call(cuda, name):
    import torch
    from sgd_amd import _lib
    make, basis, a, b, views, nu, fwd, bwd, batch = NOALLOC[name]
    P = make(basis, a, b, views, nu, fwd, bwd)
    print(name, flush=True)
    g = torch.Generator(device=cuda).manual_seed(5)
    x = torch.randn((batch,) + P.img_shape, device=cuda, generator=g)
    y = torch.randn((batch,) + P.sino_shape, device=cuda, generator=g)
    L, s = _lib.lib(), ctypes.c_void_p(torch.cuda.current_stream(cuda).cuda_stream)
    for direction, inp, ref in ((0, x, P.forward(x)), (1, y, P.backward(y))):
        out = torch.full_like(ref, float("nan"))
        rc = L.sgdct_project_dev_noalloc(P.handle, direction, ctypes.c_void_p(inp.data_ptr()),
                                         ctypes.c_void_p(out.data_ptr()), batch, s)
        torch.cuda.synchronize()
        assert rc == 0, _lib.last_error()
        assert torch.equal(out, ref), (direction, float((out - ref).abs().max()))


CAPTURED = {
    "B1": lambda: fan("B1", 128, 128, 1024, 130, 1, 1),
    "SF, rectangle": lambda: fan("SF", 60, 97, 1024, 130, 1, 1),
    "B0": lambda: fan("B0", 110, 97, 300, 150, 1, 1),
    "Hl, 4 symmetries": lambda: hexagonal("Hl", 81, 64, 1032, 256, 0, 1),
    "H0, 2 symmetries": lambda: hexagonal("H0", 60, 41, 1024, 200, 0, 1),
}


@pytest.mark.parametrize("name", list(CAPTURED))
def test_captured_unsplit_forward_is_bitwise_the_eager_one(cuda, name):
    import torch
    P = CAPTURED[name]()
    print(name, flush=True)
    x = torch.randn((2,) + P.img_shape, device=cuda)
    out = torch.empty((2,) + P.sino_shape, device=cuda)
    P.forward(x, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        P.forward(x, out=out)
    for k in range(4):
        x.copy_(torch.randn_like(x))
        ref = P.forward(x)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), k
