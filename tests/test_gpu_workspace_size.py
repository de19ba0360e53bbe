"""A handle's workspace follows one image's launch, and a handle that cannot have
it is made all the same: its launches read the images in place, with the same
values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def used(make):
    import torch
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.mem_get_info()[0]
    P = make()
    torch.cuda.synchronize()
    return P, (before - torch.cuda.mem_get_info()[0]) / MIB


def large(views, nu, start):
    from sgd_amd.torch_ops import Projector
    ang = start + 2 * np.pi * np.arange(views) / views
    return Projector("B1", 4096, 4096, ang, nu, 0.1, 0.1, 850.0 / nu, 1000.0, 700.0)


def test_workspace_of_one_image(cuda):
    # 2500 odd views from another start angle: no symmetries; 97 x 2501 pairs of
    # a view and 64 bins: whole launches.  Records 560 MiB, copies 128 MiB.
    P, mib = used(lambda: large(2501, 6144, 0.2))
    print("no symmetries, whole: %.0f MiB" % mib, flush=True)
    assert mib <= 560 + 128 + 128
    del P
    # 8 symmetries: their copies are 1 GiB, the records 89 MiB, 3 partial sums 69
    P, mib = used(lambda: large(720, 4096, 0.0))
    print("8 symmetries: %.0f MiB" % mib, flush=True)
    assert mib <= 89 + 69 + 1024 + 128


def test_creation_without_room_for_the_copies(cuda):
    import torch
    P = large(360, 4200, 0.0)
    x = torch.randn(P.img_shape, device=cuda)
    y = torch.randn(P.sino_shape, device=cuda)
    ax, aty = P.forward(x), P.backward(y)
    torch.cuda.synchronize()
    P.close()
    torch.cuda.empty_cache()
    fill = []
    while torch.cuda.mem_get_info()[0] > 800 * MIB:  # (memory just freed comes back late)
        fill.append(torch.empty((torch.cuda.mem_get_info()[0] - 700 * MIB) // 4, device=cuda))
    print("free %d MiB" % (torch.cuda.mem_get_info()[0] // MIB), flush=True)
    Q, mib = used(lambda: large(360, 4200, 0.0))
    print("made with %.0f MiB" % mib, flush=True)
    bx, bty = torch.empty_like(ax), torch.empty_like(aty)
    Q.forward(x, out=bx)
    Q.backward(y, out=bty)
    torch.cuda.synchronize()
    del fill
    assert mib < 700
    assert torch.equal(ax, bx) and torch.equal(aty, bty)
