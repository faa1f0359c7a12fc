"""Ensembles with more systems than the GPU has lanes for (their wavefronts
hand systems to their lanes in turn) against the same systems in calls small
enough for one system per lane: bitwise the same results and counts.  Ragged
counts, an empty interval, a step limit, and every stage count."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu


def solve(params, y0, te, meth, tol, **kw):
    from rk_amd.ensemble import lv_ensemble
    y, acc, rej = lv_ensemble(params, y0, 0.0, te, meth, tol, **kw)
    return y.cpu().numpy(), acc.cpu().numpy(), rej.cpu().numpy()


@pytest.mark.parametrize("count,te,meth,tol,limit", [
    (1, 4.0, "DOPRI54", 1e-6, 0),
    (65, 4.0, "VERNER65", 1e-6, 0),
    (65537, 3.0, "DOPRI54", 1e-6, 0),
    (140001, 5.0, "VERNER65", 1e-8, 0),
    (70000, 3.0, "RKF23", 1e-4, 40),
    (66000, 2.0, "DOPRI87", 1e-8, 0),
    (66001, 0.5, "RK4", 0.0, 25),
    (65800, 0.5, "HEUN2", 0.0, 10),
    (70001, 0.0, "DOPRI54", 1e-6, 0),
])
def test_refilled_lanes_equal_one_system_per_lane(count, te, meth, tol, limit):
    from rk_amd.ensemble import lv_ensemble_inputs
    params, y0 = lv_ensemble_inputs(count, seed=3)
    kw = dict(step_limit=limit, h0=1e-3)
    Y, A, R = solve(params, y0, te, meth, tol, **kw)
    part = 20000
    for a in range(0, count, part):
        s = slice(a, min(a + part, count))
        y, acc, rej = solve(params[s], y0[s], te, meth, tol, **kw)
        assert np.array_equal(A[s], acc) and np.array_equal(R[s], rej)
        assert np.array_equal(Y[s], y, equal_nan=True)
    if te == 0.0:
        assert np.array_equal(Y, y0) and not A.any() and not R.any()
