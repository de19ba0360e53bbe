"""SliceBatch.config is the launch shape in use: a batch that nobody has
configured runs one launch per slice, or the persistent queue for many small
slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,want", [(3, (0, 0, 0)), (16, (0, 0, 0)), (40, (8, 8, 0))])
def test_unconfigured_shape(cuda, n, want):
    from sgd_amd.batch import SliceBatch
    from sgd_amd.torch_ops import Projector
    ps = [Projector("B1", 16, 16, 2 * np.pi * np.arange(12) / 12, 24, 2.0, 2.0, 3.0, 1000.0, 500.0) for _ in range(n)]
    B = SliceBatch(ps)
    print(n, B.config, flush=True)
    assert B.config == want
    B.set_config(4, 0, 1)
    assert B.config == (4, 0, 1)
