"""The A, E and F forms of BRUSS2D in groups of stages
(rkx_kernels_groups.hip) bitwise against kernels that share none of that code:
the row sweep for compiled tables, the CPU oracle's seq D for others (tables
with zeros, whose terms A leaves out).  Sizes at the edges of the tiles of
every group size."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

from test_gpu_dgroup import SIZES, custom, run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("impl", ["A", "E", "F"])
@pytest.mark.parametrize("meth", ["HEUN2", "SSPRK3", "RK4", "DOPRI54", "VERNER65", "DOPRI87"])
def test_equal_row_sweep(impl, meth):
    import rk_amd
    tol = 1e-6 if rk_amd.method(meth).has_emb else 0.0
    for n in SIZES:
        ref = run(n, meth, tol, "PipeDls", tile_rows=8)
        assert same(run(n, meth, tol, impl), ref), n


@pytest.mark.parametrize("s", [2, 3, 4, 5, 8, 16])
def test_custom_tables_equal_oracle(orc, s):
    """The host's step control, so that a trace entry is the kernels' alone."""
    import rk_amd
    m = custom(s, 40 + s)
    mo = orc.Method()
    mo.name, mo.s, mo.ord, mo.has_emb = m.name, m.s, m.ord, m.has_emb
    for i in range(s):
        mo.b[i], mo.b_hat[i] = m.b[i], m.b_hat[i]
        for j in range(s):
            mo.A[i][j] = m.A[i][j]
    for n in (7, 65, 130):
        y0 = rk_amd.Bruss2D(n).ode_start_seeded(6, n, 0.01)
        yo, so, tro = orc.solve(orc.make_ode("bruss2d", n), mo, 0.0, 1.0, y0, 1e-4, h0=1e-4,
                                step_limit=5, trace_cap=8)
        for impl in ("A", "E", "F", "D"):
            st, tr, y = run(n, m, 1e-4, impl, ctrl="host")
            assert st[:2] == (so["acc"], so["rej"]), (n, impl)
            assert np.array_equal(tr, tro) and np.array_equal(y, yo), (n, impl)


@pytest.mark.parametrize("meth", ["HEUN2", "RK4", "DOPRI54", "DOPRI87"])
def test_taller_tiles_equal_row_sweep(meth):
    """Grids whose two-row tiles do not all run at once: four rows to a wave."""
    import rk_amd
    tol = 1e-6 if rk_amd.method(meth).has_emb else 0.0
    for n in (530, 641, 713):
        ref = run(n, meth, tol, "PipeDls", tile_rows=32)
        for impl in ("D", "A", "E"):
            assert same(run(n, meth, tol, impl), ref), (n, impl)
