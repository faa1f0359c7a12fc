"""The LV chain's segment kernel against the D form, bitwise, at the edges of
its segments (64*C - 2s cells for C = 2, 3, 4 cells per lane) and at lengths
for which the default rule takes each C, in one round of waves and in more."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

pytestmark = pytest.mark.gpu


def run(cells, meth, impl):
    import rk_amd
    p = rk_amd.LVChain(cells)
    y0 = torch.from_numpy(p.ode_start_seeded(4, cells, 0.0)).cuda()
    y = torch.empty_like(y0)
    tol = 1e-8 if rk_amd.method(meth).has_emb else 0.0
    st, tr = rk_amd.solve(p, meth, 0.0, 4.0, y0, y, tol, h0=1e-2, step_limit=6, impl=impl,
                          trace_cap=8)
    return (st.steps_acc, st.steps_rej, st.t, st.h), tr, y.cpu().numpy()


@pytest.mark.parametrize("meth", ["HEUN2", "SSPRK3", "RK4", "RKF23", "DOPRI54", "VERNER65"])
def test_chain_equals_d_form(meth):
    import rk_amd
    s = rk_amd.method(meth).s
    edge = [64 * c - 2 * s for c in (2, 3, 4)]
    sizes = [3, 4, 5, 63, 64, 65] + [e + d for e in edge for d in (-1, 0, 1)] + [2 * edge[0] + 1]
    for n in sizes + [120000, 240001, 500000, 700001, 1000000]:
        a, b = run(n, meth, "D"), run(n, meth, "PipeDls")
        assert a[0] == b[0], n
        assert np.array_equal(a[1], b[1]), n
        assert np.array_equal(a[2], b[2]), n
