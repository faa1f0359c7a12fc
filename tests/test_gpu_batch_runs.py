"""Batches driven by short and uneven runs: after every run each instance's
status and vector are those of a solve of its own with as many attempted
steps, whether it has ended (at any of the run lengths, on an accepted or a
rejected attempt) or goes on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RUNS = {"16+3": (16, 3), "5+2": (5, 2), "6+5": (6, 5), "ones": (1,) * 9, "long+1": (40, 1),
        "mixed": (3, 1, 2, 18, 1, 5, 7)}


def instances(rk):
    """(problem, start, table, h0, step limit, storage); h0 = 1 has its first
    attempts rejected."""
    from rk_amd.workloads import bruss_instance, chain_instance
    b24, y24 = bruss_instance(24, 2e-3, 0, seed=5)
    b90, y90 = bruss_instance(90, 2e-3, 1, seed=5)
    ch, ych = chain_instance(700, 3)
    lv = rk.LV(50)
    ylv = lv.ode_start()
    return [(b24, y24, "DOPRI54", 1e-3, 16, "low"), (b90, y90, "DOPRI54", 1e-3, 5, "low"),
            (b24, y24, "DOPRI54", 1.0, 2, "low"), (b24, y24, "VERNER65", 1e-3, 6, "low"),
            (b90, y90, "DOPRI87", 1e-3, 4, "low"), (ch, ych, "DOPRI54", 1e-3, 6, "low"),
            (lv, ylv, "DOPRI87", 1e-3, 5, "low"), (b24, y24, "DOPRI54", 1e-3, 6, "full"),
            (b90, y90, "DOPRI54", 1e-3, 1000, "low")]


@pytest.mark.parametrize("lengths", RUNS.values(), ids=RUNS.keys())
def test_after_every_run_as_alone(lengths):
    import torch
    assert torch.cuda.is_available()
    import rk_amd as rk
    insts = instances(rk)
    with rk.Batch() as b:
        ids = [b.add(p, m, 0.0, 10.0, y0, 1e-6, h0=h0, step_limit=limit, storage=storage)
               for p, y0, m, h0, limit, storage in insts]
        made = 0
        for n in lengths:
            b.run(n)
            made += n
            for (p, y0, m, h0, limit, storage), i in zip(insts, ids):
                y, alone, _ = rk.solve_host(p, m, 0.0, 10.0, y0, 1e-6, h0=h0,
                                            step_limit=min(made, limit))
                st, done = b.status(i)
                what = (type(p).__name__, m, limit, storage, made)
                assert done == (made >= limit), what
                assert (st.steps_acc, st.steps_rej) == (alone.steps_acc, alone.steps_rej), what
                assert (st.t, st.h) == (alone.t, alone.h), what
                assert np.array_equal(b.result(i), y), what
        assert b.status(ids[2])[0].steps_rej == 2 or made < 2   # ends on a rejected attempt
