"""The FP64 host-array forward projection in line segments added within a
workgroup (capi.cpp run_host_forward), for segment counts below, at, off and
above the workgroup's eight waves: against the FP64 oracle within 1e-5 relative
L2 (as every fan-beam test), and a view's values the same to the last bit
whichever other views the handle holds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis", ["B0", "B1", "SF"])
@pytest.mark.parametrize("split,nx,ny", [(0, 40, 33), (1, 40, 33), (7, 33, 40), (8, 64, 64), (9, 5, 70), (32, 50, 20)])
def test_host_segments(cuda, oracle_exact, basis, split, nx, ny):
    from pyoracle import Geometry
    from sgd_amd import _lib, operators
    print("host %s split %d %dx%d" % (basis, split, nx, ny), flush=True)
    nu, d, du, lsd, lso = 100, 1.1, 1.3, 900.0, 500.0
    ang = np.linspace(0.1, 6.0, 11)
    cls = getattr(operators, "A_%s_operator" % basis)
    x = np.random.default_rng(nx + ny).random(nx * ny)

    def forward(views):
        op = cls(nx, ny, len(views), nu, d, d, du, lsd, lso, views)
        if split:
            assert _lib.lib().sgdct_split_config(op.cpointer, split, 0) == 0, _lib.last_error()
        return op.matvec(x).reshape(len(views), nu)

    a = forward(ang)
    want = Geometry(oracle_exact, nx, ny, ang, nu, d, d, du, lsd, lso).forward(basis, x.reshape(nx, ny).T.copy())
    e = float(np.linalg.norm(a - want) / np.linalg.norm(want))
    print("  rel %.2e" % e, flush=True)
    assert e <= 1e-5
    assert np.array_equal(forward(ang[3:8]), a[3:8])
