"""Binning on both sides of the limits between its forms, by view and by bin: 2048 coincidences per view, 3 bins per
coincidence, and a planogram of a single view row (16 coincidences per view is only reached with planograms of 17 GB).
Bit-exact against the oracle: the sums keep the event order in both forms, so the tolerance is zero."""
import numpy as np
import pytest

from petl_amd.petl_server import PETLserver

pytestmark = pytest.mark.gpu

N = (1 << 20) + 1000


@pytest.mark.parametrize("D, L, H, T, vm0, vm1, share, bins", [
    (100.0, 300.0, 100.0, 1.0, 0.5, 0.09, 2286, 15.3),  # too many per view
    (100.0, 300.0, 100.0, 1.0, 0.5, 0.1, 1870, 18.7),
    (100.0, 64.0, 64.0, 2.0, 1.0, 0.3, 1371, 1.91),     # too few bins
    (100.0, 64.0, 64.0, 2.0, 1.0, 0.6, 663, 3.95),
    (200.0, 100.0, 8.0, 0.38, 1.0, 0.0, 1991, 7.9),     # one view row
])
def test_limits_match_oracle(oracle, D, L, H, T, vm0, vm1, share, bins):
    rng = np.random.default_rng(31)
    blue = np.column_stack([rng.uniform(-L / 2, L / 2, N), np.full(N, D / 2), rng.uniform(0, H, N)]).astype(np.float32)
    pink = np.column_stack([rng.uniform(-L / 2, L / 2, N), np.full(N, -D / 2), rng.uniform(0, H, N)]).astype(np.float32)
    if vm1 < 0.2:  # slopes that the few view rows hold
        pink[:, 2] = np.clip(blue[:, 2] + rng.uniform(-1, 1, N) * vm1 * D, 0, H)
    s = PETLserver()
    s.print_warnings = False
    s.add_planogram(0.0, D, L, H, T, vm0, vm1)
    s.set_volume(8, 8, 8, T)
    plan = oracle.planogram(0.0, D, L, H, T, vm0, vm1)
    views = plan.shape[0] * plan.shape[1]
    assert N // views == share and abs(np.prod(plan.shape) / N - bins) < 0.1
    start = [rng.random(plan.shape).astype(np.float32)]
    got, acc = s.bin_events(blue, pink, g=[x.copy() for x in start])
    ref, racc = oracle.bin_events([plan], blue, pink, g=[x.copy() for x in start])
    assert acc == racc and acc[0] > N // 10
    np.testing.assert_array_equal(got[0], ref[0])
