"""The fast projectors' split of values and weights over the whole float32 range: images and planograms whose rows hold
values 2^-36 to 2^-120 apart, and outputs that only a small interpolation weight reaches.

Tolerance.  Beside a hot value the cold outputs are the same products as without it, and an image is the sum of its parts,
so only the order and the rounding of the sums may differ: 2^-24 each, at most 5 per block of 4 inner indices and 3 per v1
row.  ETOL bounds that elementwise for non-negative data: 9 blocks and 13 v1 rows, worst case
(5 * 9 + 3 * 13 + 10) * 2^-24 = 5.6e-6; the planograms' ramps against the float64 oracle carry the weights' 1e-6 as well.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from petl_amd.petl_server import PETLserver  # noqa: E402
from test_gpu_back_tiles import back  # noqa: E402
from test_gpu_forward_tiles import CASES, TOL, forward, make, rel  # noqa: E402

pytestmark = pytest.mark.gpu
ETOL = 7.0e-6


@pytest.mark.parametrize("case", [4, 6, 7])
@pytest.mark.parametrize("k", [36, 44, 60, 75, 100])
def test_cold_bins_beside_a_hot_voxel(oracle, case, k):
    s, plan, vol = make(oracle, CASES[case])
    cold = np.ldexp(np.random.default_rng(k).random(vol.shape) + 0.5, -k).astype(np.float32)
    c = tuple(n // 2 for n in vol.shape)
    cold[c] = 0.0
    hot = np.zeros(vol.shape, np.float32)
    hot[c] = 1.0
    ref = oracle.project([plan], vol, cold.astype(np.float64), dtype=np.float64)[0]
    away = (oracle.project([plan], vol, hot, dtype=np.float64)[0] == 0) & (ref > 0)
    assert away.sum() > 1000
    g, alone = forward(s, plan, cold + hot), forward(s, plan, cold)
    assert rel(g[away] * 2.0 ** k, ref[away] * 2.0 ** k) < TOL
    assert np.all(np.abs(g[away] - alone[away]) <= ETOL * alone[away])


@pytest.mark.parametrize("mode", ["petl", "matched"])
@pytest.mark.parametrize("k", [36, 44, 60, 75, 100])
def test_cold_voxels_beside_a_hot_bin(oracle, k, mode):
    s, plan, vol = make(oracle, CASES[4])
    s.set_backprojector_mode(mode)
    cold = np.ldexp(np.random.default_rng(k).random(plan.shape) + 0.5, -k).astype(np.float32)
    c = tuple(n // 2 for n in plan.shape)
    cold[c] = 0.0
    hot = np.zeros(plan.shape, np.float32)
    hot[c] = 1.0
    ref = oracle.backproject([plan], vol, [cold.astype(np.float64)], mode=mode, dtype=np.float64)
    away = (oracle.backproject([plan], vol, [hot], mode=mode, dtype=np.float64) == 0) & (ref > 0)
    assert away.sum() > 1000
    f, alone = back(s, cold + hot), back(s, cold)
    assert rel(f[away] * 2.0 ** k, ref[away] * 2.0 ** k) < TOL
    assert np.max(np.abs(f[away] / alone[away] - 1.0)) < ETOL


# largest exponent and exponents per voxel or bin: up to 77 and 124 in one row (31 voxels, 64 bins)
@pytest.mark.parametrize("top, step", [(0, -1.5), (0, -2.5), (30, -4.0)])
@pytest.mark.parametrize("flip", [False, True])
def test_ramp_image(oracle, top, step, flip):
    s, plan, vol = make(oracle, CASES[4])
    ramp = np.exp2(top + step * np.arange(vol.shape[2]))
    f = (ramp[::-1] if flip else ramp) * (np.random.default_rng(1).random(vol.shape) + 0.5)
    f = f.astype(np.float32)
    g = forward(s, plan, f).astype(np.float64)
    # the same weights on four columns at a time, whose values take one pass (the oracle's view angles are float64: 1e-6 of a
    # bin beside the planogram's, times the ramp's slope)
    ref = np.zeros(plan.shape)
    for a in range(0, vol.shape[2], 4):
        part = np.zeros_like(f)
        part[:, :, a:a + 4] = f[:, :, a:a + 4]
        ref += forward(s, plan, part)
    on = ref > 0
    assert on.sum() > 10000 and ref[on].min() < 2.0 ** -30 * ref.max()
    assert np.max(np.abs(g[on] / ref[on] - 1.0)) < ETOL


@pytest.mark.parametrize("mode", ["petl", "matched"])
@pytest.mark.parametrize("top, step", [(0, -0.5), (0, -1.2), (30, -1.9)])
def test_ramp_planogram(oracle, top, step, mode):
    s, plan, vol = make(oracle, CASES[4])
    s.set_backprojector_mode(mode)
    g = np.exp2(top + step * np.arange(plan.shape[3])) * (np.random.default_rng(2).random(plan.shape) + 0.5)
    g = g.astype(np.float32)
    ref = oracle.backproject([plan], vol, [g.astype(np.float64)], mode=mode, dtype=np.float64)
    on = ref > 0
    f = back(s, g).astype(np.float64)
    assert np.max(np.abs(f[on] / ref[on] - 1.0)) < ETOL


@pytest.mark.parametrize("k", [12, 16, 20, 24])
def test_small_weights(oracle, k):
    """One voxel up to 2^-k of a bin beside a bin's centre, by another part of it in every view: the bins that get the small
    part hold it to float32 accuracy (fewer than 10 roundings; the smallest weight, 2^-28, is the rest of a float64 position
    near 14 bins, which is good to 2^-50 and so to 2^-22 of it)."""
    s = PETLserver()
    s.print_warnings = False
    args = (0.0, 30.0, 20.0, 8.0, 2.0, 1.0, 0.2)
    s.add_planogram(*args)
    offs = (1.0, float(np.float32(1.3 * 2.0 ** (1 - k))), 0.7)  # bin centres are odd millimetres; y offset x v0 beside them
    s.set_volume(1, 1, 1, 2.0, 0.0, *offs)
    assert s.uses_fast_path(0)
    plan = oracle.planogram(*args)
    vol = oracle.volume(1, 1, 1, 2.0, 0.0, *offs)
    ref = oracle.project([plan], vol, np.full((1, 1, 1), 0.7), dtype=np.float64)[0]
    g = forward(s, plan, np.full((1, 1, 1), 0.7)).astype(np.float64)
    small = (ref > 0) & (ref < 4.0 * 2.0 ** -k)
    small[:, :plan.shape[1] // 2 + 1] = False  # on this side the small weight is one minus a float, no better than 2^-25
    assert small.sum() > 20
    assert np.max(np.abs(g[small] / ref[small] - 1.0)) < 10 * 2.0 ** -24
    iv1, iv0, iu1, iu0 = (int(x[-1]) for x in np.nonzero(small))
    for mode in ("petl", "matched"):
        s.set_backprojector_mode(mode)
        y = np.zeros(plan.shape, np.float32)
        y[iv1, iv0, iu1, iu0] = 0.3
        refb = oracle.backproject([plan], vol, [y.astype(np.float64)], mode=mode, dtype=np.float64)
        assert refb[0, 0, 0] > 0
        assert abs(back(s, y)[0, 0, 0].astype(np.float64) / refb[0, 0, 0] - 1.0) < 10 * 2.0 ** -24
