"""The tile form of the fused BRUSS2D step (rkx_tile_kernel.hpp) against the
D form, bitwise: every attempted step's (t, h, err), the counts and the final
vector.  The sizes are the edges of the tiles: grids inside one tile, one row
or column around each tile height and strip width, one size per tile shape
that the default rule picks, and the last sizes before the row sweep."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu

METHODS = ["HEUN2", "SSPRK3", "RK4", "RKF23", "DOPRI54", "VERNER65"]
SIZES = [2, 3, 7, 15, 16, 17, 24, 31, 32, 33, 47, 48, 49, 57, 58, 63, 64, 65, 114, 115, 165, 193,
         251, 301, 419, 512, 530, 601, 660]


def run(n, meth, impl, **kw):
    import rk_amd
    p = rk_amd.Bruss2D(n)
    y0 = torch.from_numpy(p.ode_start_seeded(5, n, 0.01)).cuda()
    y = torch.empty_like(y0)
    tol = 1e-6 if rk_amd.method(meth).has_emb else 0.0
    h0 = 1e-3 if tol else 1e-4
    st, tr = rk_amd.solve(p, meth, 0.0, 1.0, y0, y, tol, h0=h0, step_limit=7, impl=impl,
                          trace_cap=16, **kw)
    return (st.steps_acc, st.steps_rej, st.t, st.h), tr, y.cpu().numpy()


@pytest.mark.parametrize("meth", METHODS)
def test_tile_equals_d_form(meth):
    for n in SIZES:
        a, ta, ya = run(n, meth, "D")
        b, tb, yb = run(n, meth, "PipeDls")
        assert a == b, n
        assert np.array_equal(ta, tb), n
        assert np.array_equal(ya, yb), n


def test_tile_host_control_equals_device_control():
    for n in (5, 64, 129):
        a, ta, ya = run(n, "DOPRI54", "PipeDls", ctrl="host")
        b, tb, yb = run(n, "DOPRI54", "PipeDls")
        assert a == b and np.array_equal(ta, tb) and np.array_equal(ya, yb), n


def test_tile_zero_divisor_and_overflow():
    """Zero components raise the error sentinel, and a step far too long
    overflows: the tile form gives the D form's values there too."""
    import rk_amd
    for n in (4, 40, 70, 130):
        for h0, fill in ((1e-3, 0.0), (1e60, 1.0), (1e200, 3.0)):
            p = rk_amd.Bruss2D(n)
            y0 = torch.full((p.n,), fill, dtype=torch.float64, device="cuda")
            res = []
            for impl in ("D", "PipeDls"):
                y = torch.empty_like(y0)
                st, tr = rk_amd.solve(p, "DOPRI54", 0.0, 1e300, y0, y, 0.0, h0=h0, step_limit=2,
                                      impl=impl, trace_cap=4)
                res.append((st.steps_acc, st.steps_rej, tr, y.cpu().numpy()))
            (a0, r0, t0, v0), (a1, r1, t1, v1) = res
            assert (a0, r0) == (a1, r1), (n, h0)
            assert np.array_equal(t0, t1, equal_nan=True), (n, h0)
            assert np.array_equal(v0, v1, equal_nan=True), (n, h0)
