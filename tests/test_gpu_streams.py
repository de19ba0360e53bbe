"""One handle's unsplit A on several streams and threads at once: the calls share
the handle's interleaved images, which the device orders, so that every output
is bit for bit the one of calls one after the other."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread: one handle value, a stream for each thread


def handles():
    from sgd_amd.torch_ops import Projector

    def fan(basis, nx, ny, views, nu, split):
        P = Projector(basis, nx, ny, 2 * np.pi * np.arange(views) / views, nu, 1.7, 1.7, 2.9, 1000.0, 500.0)
        P.set_split(split, split)
        return P

    ang = 2 * np.pi * np.arange(1024) / 1024
    return {"Hl": lambda: Projector.hexagonal("Hl", 80, 64, ang, 256, 1.0, 1.2, 1000.0, 500.0),
            "H0": lambda: Projector.hexagonal("H0", 41, 60, ang, 200, 1.0, 1.2, 1000.0, 500.0),
            "B0, split 1": lambda: fan("B0", 110, 97, 300, 150, 1),
            "B1, split 1": lambda: fan("B1", 128, 128, 1024, 130, 1),
            "SF, split 1": lambda: fan("SF", 60, 97, 1024, 130, 1),
            "B1, automatic": lambda: fan("B1", 20, 16, 3200, 4100, 0)}


NAMES = ["Hl", "H0", "B0, split 1", "B1, split 1", "SF, split 1", "B1, automatic"]


def images(P, cuda, n):
    import torch
    g = torch.Generator(device=cuda).manual_seed(3)
    xs = [torch.randn((3,) + P.img_shape, device=cuda, generator=g) for _ in range(n)]
    ref = [P.forward(x) for x in xs]
    torch.cuda.synchronize()
    return xs, ref


@pytest.mark.parametrize("name", NAMES)
def test_unsplit_forward_on_six_streams(cuda, name):
    import torch
    P = handles()[name]()
    xs, ref = images(P, cuda, 12)
    print(name, "6 streams", flush=True)
    streams = [torch.cuda.Stream() for _ in range(6)]
    outs = []
    for k, x in enumerate(xs):
        with torch.cuda.stream(streams[k % 6]):
            outs.append(P.forward(x))
    torch.cuda.synchronize()
    for a, b in zip(ref, outs):
        assert torch.equal(a, b), float((a - b).abs().max())


@pytest.mark.parametrize("name", NAMES)
def test_unsplit_forward_on_per_thread_streams(cuda, name):
    import torch
    from sgd_amd import _lib
    P = handles()[name]()
    xs, ref = images(P, cuda, 12)
    outs = [torch.full_like(r, float("nan")) for r in ref]
    torch.cuda.synchronize()
    print(name, "per-thread streams", flush=True)
    L, rcs = _lib.lib(), []
    gate = threading.Barrier(3)

    def work(first):
        gate.wait()
        for k in range(first, 12, 3):
            rcs.append(L.sgdct_forward_dev(P.handle, ctypes.c_void_p(xs[k].data_ptr()),
                                           ctypes.c_void_p(outs[k].data_ptr()), 3, ctypes.c_void_p(PER_THREAD)))
        torch.cuda.ExternalStream(PER_THREAD).synchronize()  # the thread's stream ends with it

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert rcs == [0] * 12
    for a, b in zip(ref, outs):
        assert torch.equal(a, b), float((a - b).abs().max())
