"""The tile form on grids of up to 32 x 32, which solves under the host's
control and rkx_solve_noalloc run (device-controlled solves of these sizes make
several attempts to a launch instead): every size, bitwise against the D form
and the one-workgroup form."""
import numpy as np
import pytest
import torch  # before the library: both load the HIP runtime

from test_gpu_tile import METHODS, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("meth", METHODS)
def test_every_size_under_host_control(meth):
    for n in range(2, 34):
        tile = run(n, meth, "PipeDls", ctrl="host")
        for other in (run(n, meth, "PipeDls"), run(n, meth, "D")):
            assert tile[0] == other[0], n
            assert np.array_equal(tile[1], other[1]) and np.array_equal(tile[2], other[2]), n
