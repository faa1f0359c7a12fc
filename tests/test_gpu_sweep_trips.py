"""Band heights of the whole-trip row sweeps (VERNER65: trips of 9 iterations;
DOPRI87: trips of 14; the last trip may be left early), around the heights
that one more trip or exit makes, bitwise against the D form: every
attempt's (t, h, err) and the final vector.  Grids short enough for the general
ghost rows, with ragged last bands and with paired narrow strips."""
import pytest
import torch  # before the library: both load the HIP runtime

from test_gpu_dgroup import run, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("meth", ["VERNER65", "DOPRI87"])
@pytest.mark.parametrize("n", [5, 24, 47, 131, 300])
def test_band_heights(meth, n):
    ref = run(n, meth, 1e-6, "D")
    for rows in (1, 3, 4, 5, 9, 10, 13, 14, 15, 18, 19, 28, 29):
        for waves in (1, 2):
            got = run(n, meth, 1e-6, "PipeDls", tile_rows=rows, tile_waves=waves)
            assert same(got, ref), (rows, waves)
    assert same(run(n, meth, 1e-6, "PipeDls"), ref)
