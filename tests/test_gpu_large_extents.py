"""The fast kernels at volumes and planogram rows whose byte offsets pass 32 bits: a volume of 2^30 voxels and a v1 row of
2^30 bins, of which the panels see, and the volume meets, only a corner.  The same corner by itself is the reference (covered
against the oracle elsewhere); its positions differ by a float64 rounding, 1e-12 of a bin, so the results by float32
roundings of the weights at most: 1e-6.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from petl_amd.petl_server import PETLserver  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 1.0e-6


def server(psi, D, L, H, T, vm0, vm1, n, offz):
    s = PETLserver()
    s.print_warnings = False
    s.add_planogram(psi, D, L, H, T, vm0, vm1)
    s.set_volume(*n, T, offsetZ=offz)
    assert s.uses_fast_path(0)
    return s


def rel(a, b):
    return float(torch.linalg.norm(a.double() - b.double()) / torch.linalg.norm(b.double()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("psi", [0.0, 90.0])
def test_volume(psi, dtype):
    panel = (psi, 2100.0, 500.0, 16.0, 2.0, 0.01, 0.003)
    plane = (256, 1024) if psi == 0.0 else (1024, 256)
    big, small, off = 4100, 20, -4081.0  # the panels' middle is plane 4090 of the large volume
    sb = server(*panel, (*plane, big), off)
    ss = server(*panel, (*plane, small), off + big - small)
    shape = tuple(int(x) for x in ss.get_planogramSize(0))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1)
    f = torch.rand((small, plane[1], plane[0]), device=DEV, generator=gen).to(dtype)
    fb = torch.zeros((big, plane[1], plane[0]), dtype=dtype, device=DEV)
    fb[big - small:] = f
    g, gb = (torch.full(shape, 7.0, dtype=dtype, device=DEV) for _ in range(2))
    ss.project_gpu([g], f)
    sb.project_gpu([gb], fb)
    assert rel(gb, g) < (TOL if dtype == torch.float32 else 1e-4)  # (a bfloat16 may round the other way, one in hundreds)
    del fb
    y = torch.rand(shape, device=DEV, generator=gen).to(dtype)
    b = torch.empty((small, plane[1], plane[0]), device=DEV)
    bb = torch.full((big, plane[1], plane[0]), 7.0, device=DEV)
    ss.backproject_gpu([y], b)
    sb.backproject_gpu([y], bb)
    assert rel(bb[big - small:], b) < TOL
    assert not bb[:big - small].any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_view_row(dtype):
    n, off = (9, 8, 6), 0.0
    sb = server(0.0, 1020.0, 2.0, 8300.0, 2.0, 1.0, 0.0, n, off)
    ss = server(0.0, 1020.0, 2.0, 16.0, 2.0, 1.0, 0.0, n, off)
    big, small = (tuple(int(x) for x in s.get_planogramSize(0)) for s in (sb, ss))
    assert big[0] == 1 and big[1] * big[2] * big[3] >= 1 << 30 and big[:2] + big[3:] == small[:2] + small[3:]
    a = (big[2] - small[2]) // 2
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1)
    f = torch.rand(n[::-1], device=DEV, generator=gen).to(dtype)
    g = torch.full(small, 7.0, dtype=dtype, device=DEV)
    gb = torch.full(big, 7.0, dtype=dtype, device=DEV)
    ss.project_gpu([g], f)
    sb.project_gpu([gb], f)
    assert rel(gb[:, :, a:a + small[2]], g) < (TOL if dtype == torch.float32 else 1e-4)
    assert not gb[:, :, :a].any() and not gb[:, :, a + small[2]:].any()
    y = torch.rand(small, device=DEV, generator=gen).to(dtype)
    gb.zero_()
    gb[:, :, a:a + small[2]] = y
    b, bb = (torch.full(n[::-1], 7.0, device=DEV) for _ in range(2))
    ss.backproject_gpu([y], b)
    sb.backproject_gpu([gb], bb)
    assert rel(bb, b) < TOL
    if dtype == torch.float32:  # the ratio reads its data there too
        assert rel(*(torch.from_numpy(s.MLEM([x.cpu().numpy()], None, 1)) for s, x in ((sb, gb), (ss, y)))) < TOL
