"""RWLS keeps a model's buffers between calls up to a bound; a larger reconstruction gives its device memory back when it
returns, and the next call on the model allocates again."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from petl_amd.petl_server import PETLserver  # noqa: E402

pytestmark = pytest.mark.gpu
GIB = 1 << 30


def test_large_reconstruction_gives_its_memory_back():
    s = PETLserver()
    s.print_warnings = False
    s.add_planogram(0.0, 200.0, 256.0, 256.0, 2.0, 1.0, 1.0)
    s.set_volume(16, 16, 16, 2.0)
    g = [np.ones(tuple(int(x) for x in s.get_planogramSize(0)), np.float32)]
    assert 4 * g[0].nbytes > 4 * GIB  # data, residual, projection and weights
    torch.empty(1, device="cuda:0")
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f = s.RWLS(g, None, 1)
    kept = before - torch.cuda.mem_get_info()[0]
    assert kept < GIB, kept
    assert np.array_equal(f, s.RWLS(g, None, 1))
