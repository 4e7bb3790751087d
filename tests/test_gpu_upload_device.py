"""The reconstructions' C entries copy data from wherever HIP can, a device array or managed memory too: the same images as
from a host array, bit for bit, at sizes on both sides of the chunked upload's."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_upload import data, make  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("i", [0, 1])
def test_device_data(i):
    s = make(i)
    g = data(s, 5)
    ref = s.MLEM(g, None, 2)
    t = torch.from_numpy(g[0]).to("cuda:0")
    torch.cuda.synchronize()
    fp = ctypes.POINTER(ctypes.c_float)
    s.floatstarstar = lambda x: (fp * 1)(ctypes.cast(ctypes.c_void_p(t.data_ptr()), fp))  # the data's addresses
    assert np.array_equal(s.MLEM(g, None, 2), ref)
