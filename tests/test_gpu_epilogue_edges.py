"""The fast forward's epilogues (MLEM ratio, least-squares residual, with response and weights) at the first u1 row and the
first and last views of its groups of 16, where the tiles' columns begin before the rows read together and end after them:
every datum there counts.

All counts of the data lie in such rows, so that an image holds nothing else.  Tolerance: 1e-5 as for the other one-step
reconstructions, whose images sum ratios of float32 projections (2.4e-7 each).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_forward_tiles import CASES, make, rel  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1.0e-5


def edge_data(plan, view, u1, seed):
    y = np.zeros(plan.shape, np.float32)
    rng = np.random.default_rng(seed)
    y[:, view, u1] = rng.random((plan.shape[0], plan.shape[3])) + 0.5
    return y


@pytest.mark.parametrize("i", [1, 3, 4, 5, 7])
@pytest.mark.parametrize("view, u1", [(0, 0), (1, 0), (16, 0), (-1, -1), (0, -1)])
def test_ratio(oracle, i, view, u1):
    s, plan, vol = make(oracle, CASES[i][:7] + (CASES[i][7][:2] + (plan_rows(oracle, CASES[i]),),))
    y = edge_data(plan, min(view, plan.shape[1] - 1), u1, i)
    ref = oracle.mlem([plan], vol, [y.astype(np.float64)], 1, dtype=np.float64)
    assert (ref > 0).sum() > 10
    assert rel(s.MLEM([y], None, 1), ref) < TOL
    resp = [np.random.default_rng(5).random(plan.shape).astype(np.float32) + np.float32(0.5)]
    s.response = resp
    got = s.MLEM([y], None, 1)
    # one step from ones: f = P^T(R y / (R P 1)) / P^T R
    q = oracle.project([plan], vol, np.ones(vol.shape), dtype=np.float64)[0] * resp[0]
    r = resp[0] * np.divide(y, q, out=np.zeros(q.shape), where=q != 0)
    S = oracle.backproject([plan], vol, [resp[0].astype(np.float64)], dtype=np.float64)
    S[S == 0] = 1.0
    assert rel(got, oracle.backproject([plan], vol, [r], dtype=np.float64) / S) < TOL


def plan_rows(oracle, case):
    """As many heights as the panels have rows: the first and the last row cross the volume."""
    return oracle.planogram(*case[:7]).shape[2]


@pytest.mark.parametrize("i", [3, 4])
@pytest.mark.parametrize("view, u1", [(0, 0), (16, 0), (-1, -1)])
def test_residual(oracle, i, view, u1):
    """One RWLS step from an image of ones with weights in these rows alone: the gradient is P^T W (P 1 - y)."""
    s, plan, vol = make(oracle, CASES[i][:7] + (CASES[i][7][:2] + (plan_rows(oracle, CASES[i]),),))
    view = min(view, plan.shape[1] - 1)
    y, W = edge_data(plan, view, u1, i), edge_data(plan, view, u1, 50 + i)
    ones = np.ones(vol.shape, np.float32)
    ref, _ = oracle.rwls([plan], vol, [y], 1, f=ones.copy(), W=[W])
    assert np.abs(ref - 1.0).max() > 1e-3
    got = s.RWLS([y], ones.copy(), 1, W=[W])
    assert np.linalg.norm(got - ref) < TOL * np.linalg.norm(ref - 1.0) + 2.0 ** -24 * np.linalg.norm(ref)
