"""Infinities and NaNs on axis-aligned panels with voxels of another size than the crystals: they reach the bins and
voxels whose footprint meets them, those where the projection of ones in their place is not zero, and no others, so a NaN in
a bin outside the panels (a gradient 1 - y / q where q is zero) leaves a matched back projection as it is.  Values
elsewhere have the tolerance of test_gpu_axis_pitch.py.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_axis_pitch import CASES, DEV, TOL, make, rel  # noqa: E402

pytestmark = pytest.mark.gpu


def forward(s, plan, f):
    g = torch.full(plan.shape, 7.0, dtype=torch.float32, device=DEV)
    s.project_gpu([g], torch.from_numpy(np.ascontiguousarray(f, np.float32)).to(DEV))
    return g.cpu().numpy()


def back(s, vol, g):
    f = torch.full(vol.shape, 7.0, dtype=torch.float32, device=DEV)
    s.backproject_gpu([torch.from_numpy(np.ascontiguousarray(g, np.float32)).to(DEV)], f)
    return f.cpu().numpy()


@pytest.mark.parametrize("i", range(9))
@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_forward(oracle, i, value):
    s, plan, vol = make(oracle, CASES[i])
    f = np.random.default_rng(i).random(vol.shape).astype(np.float32) + np.float32(0.1)
    bad = np.zeros(vol.shape)
    bad[vol.shape[0] // 2, vol.shape[1] // 2, vol.shape[2] // 2] = bad[0, 0, 0] = bad[-1, 1, -1] = 1.0
    ref = oracle.project([plan], vol, np.where(bad > 0, 0.0, f).astype(np.float64), dtype=np.float64)[0]
    g = forward(s, plan, np.where(bad > 0, value, f))
    ok = np.isfinite(g)
    assert np.array_equal(ok, forward(s, plan, bad) == 0)
    assert rel(g[ok], ref[ok]) < TOL


@pytest.mark.parametrize("i", range(9))
@pytest.mark.parametrize("mode", ["petl", "matched"])
def test_back(oracle, i, mode):
    s, plan, vol = make(oracle, CASES[i])
    s.set_backprojector_mode(mode)
    y = np.random.default_rng(i).random(plan.shape).astype(np.float32) + np.float32(0.1)
    c = tuple(n // 2 for n in plan.shape)
    bad = np.zeros(plan.shape)
    bad[c] = bad[c[0], c[1], c[2], 0] = bad[c[0], 0, c[2], -1] = 1.0  # two at the ends of a row
    met = back(s, vol, bad) != 0
    ref = oracle.backproject([plan], vol, [np.where(bad > 0, 0.0, y).astype(np.float64)], mode=mode, dtype=np.float64)
    for value in (np.inf, np.nan):
        b = back(s, vol, np.where(bad > 0, value, y))
        ok = np.isfinite(b)
        assert np.array_equal(ok, ~met)
        if ok.any():
            assert rel(b[ok], ref[ok]) < TOL


@pytest.mark.parametrize("i", range(9))
def test_nan_outside_the_panels(oracle, i):
    s, plan, vol = make(oracle, CASES[i])
    s.set_backprojector_mode("matched")
    y = np.random.default_rng(i).random(plan.shape).astype(np.float32)
    out = np.zeros(plan.shape, bool)
    for iv1, iv0, iu1, iu0 in np.ndindex(*plan.shape):
        if iv1 in (0, plan.shape[0] // 2) and iu1 in (0, plan.shape[2] // 2):
            out[iv1, iv0, iu1, iu0] = oracle.bin_masked(plan, iv1, iv0, iu1, iu0)
    assert out.any()
    b = back(s, vol, np.where(out, np.nan, y))
    assert np.array_equal(b, back(s, vol, np.where(out, 0.0, y)))
