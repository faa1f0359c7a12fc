"""Ensembles whose systems all take the same number of attempts, and ones that
fit a wave or two, against the CPU oracle system by system: counts around a
wave, a workgroup and the lanes of the chip, every stage count."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("meth", ["HEUN2", "SSPRK3", "RK4", "RKF23", "DOPRI54", "VERNER65",
                                  "DOPRI87"])
@pytest.mark.parametrize("tol,te,limit", [(0.0, 0.5, 12), (1e-6, 2.0, 60)])
def test_equal_oracle(orc, meth, tol, te, limit):
    from rk_amd.ensemble import lv_ensemble, lv_ensemble_inputs
    params, y0 = lv_ensemble_inputs(66000, seed=11)
    yo, ao, ro = orc.lv_ensemble(params, y0, 0.0, te, meth, tol, 1e-2, step_limit=limit)
    for count in (1, 63, 64, 65, 256, 257, 65536, 65537, 66000):
        Y, acc, rej = lv_ensemble(params[:count], y0[:count], 0.0, te, meth, tol, h0=1e-2,
                                  step_limit=limit)
        assert np.array_equal(acc.cpu().numpy(), ao[:count]), count
        assert np.array_equal(rej.cpu().numpy(), ro[:count]), count
        assert np.array_equal(Y.cpu().numpy().view(np.uint64), yo[:count].view(np.uint64)), count
