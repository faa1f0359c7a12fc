"""BRUSS2D grids of one workgroup, several attempts to a launch
(rkx_kernels_run.hip), bitwise against the row sweep: every attempt's
(t, h, err), the counts and the final vector.  Sizes at the edges of its blocks
of one and two rows; solves that end within a launch, at the step limit and
past several launches, and that reject steps."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu


def run(n, meth, tol, limit, te=1.0, h0=1e-3, **kw):
    import rk_amd
    p = rk_amd.Bruss2D(n)
    y0 = torch.from_numpy(p.ode_start_seeded(7, n, 0.02)).cuda()
    y = torch.full_like(y0, float("nan"))
    st, tr = rk_amd.solve(p, meth, 0.0, te, y0, y, tol, h0=h0, step_limit=limit, trace_cap=200,
                          **kw)
    return (st.steps_acc, st.steps_rej, st.t, st.h), tr, y.cpu().numpy()


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("meth", ["HEUN2", "SSPRK3", "RKF23", "RK4", "DOPRI54", "VERNER65",
                                  "DOPRI87"])
def test_equal_row_sweep(meth):
    import rk_amd
    emb = rk_amd.method(meth).has_emb
    for n in (2, 3, 15, 16, 17, 31, 32, 33):
        for limit in (1, 31, 32, 33, 100):
            a = run(n, meth, 1e-6 if emb else 0.0, limit, h0=1e-2 if emb else 1e-4)
            b = run(n, meth, 1e-6 if emb else 0.0, limit, h0=1e-2 if emb else 1e-4, tile_rows=8)
            assert same(a, b), (n, limit)


def test_to_the_end_and_untraced():
    """No step limit: the loop ends at te within a launch; without a trace."""
    import rk_amd
    for n in (9, 32):
        a = run(n, "DOPRI54", 1e-9, 0, te=0.7)
        assert same(a, run(n, "DOPRI54", 1e-9, 0, te=0.7, tile_rows=8))
        p = rk_amd.Bruss2D(n)
        y0 = torch.from_numpy(p.ode_start_seeded(7, n, 0.02)).cuda()
        y = torch.empty_like(y0)
        st, _ = rk_amd.solve(p, "DOPRI54", 0.0, 0.7, y0, y, 1e-9, h0=1e-3)
        assert (st.steps_acc, st.steps_rej, st.t, st.h) == a[0]
        assert np.array_equal(y.cpu().numpy(), a[2])
