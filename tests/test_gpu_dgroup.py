"""The D form of BRUSS2D in groups of stages (rkx_kernels_groups.hip) against
the E form's kernels, bitwise: every attempted step's (t, h, err), the counts
and the final vector.  Sizes at the edges of the 64-column, 32-row tiles for
every group size, tables of 2 to 16 stages (one, two, three and four groups),
dense ones and ones with zeros, and the host's step control."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 8, 31, 32, 33, 57, 61, 63, 64, 65, 116, 119, 121, 250]


def custom(s, seed):
    """An explicit table of s stages without a compiled pattern."""
    from rk_amd._lib import Method
    g = np.random.default_rng(seed)
    m = Method()
    m.name = b"CUSTOM"
    m.s, m.ord, m.has_emb = s, 2, 1
    for i in range(s):
        for j in range(i):
            m.A[i][j] = 0.0 if g.random() < 0.2 and j != i - 1 else g.uniform(-0.5, 0.5)
        m.b[i] = g.uniform(0.0, 2.0 / s)
        m.b_hat[i] = m.b[i] + g.uniform(-1e-3, 1e-3)
    return m


def run(n, m, tol, impl, **kw):
    import rk_amd
    p = rk_amd.Bruss2D(n)
    y0 = torch.from_numpy(p.ode_start_seeded(6, n, 0.01)).cuda()
    y = torch.empty_like(y0)
    st, tr = rk_amd.solve(p, m, 0.0, 1.0, y0, y, tol, h0=1e-4, step_limit=5, impl=impl,
                          trace_cap=8, **kw)
    return (st.steps_acc, st.steps_rej, st.t, st.h), tr, y.cpu().numpy()


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("meth", ["HEUN2", "SSPRK3", "RK4", "DOPRI54", "VERNER65", "DOPRI87"])
def test_groups_equal_e_form(meth):
    import rk_amd
    tol = 1e-6 if rk_amd.method(meth).has_emb else 0.0
    for n in SIZES:
        assert same(run(n, meth, tol, "D"), run(n, meth, tol, "E")), n


@pytest.mark.parametrize("s", [2, 3, 4, 5, 6, 9, 16])
def test_custom_tables(s):
    m = custom(s, s)
    for n in (7, 65, 130):
        e = run(n, m, 1e-4, "E")
        assert same(run(n, m, 1e-4, "D"), e), n
        assert same(run(n, m, 1e-4, "PipeDls"), e), n


def test_host_control():
    for n in (9, 100):
        assert same(run(n, "DOPRI54", 1e-6, "D", ctrl="host"), run(n, "DOPRI54", 1e-6, "E")), n
