"""The library's host side against a recording HIP runtime on the CPU
(tests/hip_record.c): what it orders, keeps and frees.  Each test runs in a
process of its own that loads the recorder ahead of librkx.so; no kernel runs."""
import json
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

CHILD = """
import ctypes, json, os, sys
sys.path.insert(0, %(repo)r)
rec = ctypes.CDLL(%(rec)r, mode=ctypes.RTLD_GLOBAL)
rec.rec_live_bytes.restype = rec.rec_copy_block.restype = ctypes.c_size_t
rec.rec_limit.argtypes = rec.rec_watch_copy.argtypes = [ctypes.c_size_t]
import numpy as np
import rk_amd
out = {}
%(body)s
sys.stdout.write(json.dumps(out))
"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rec") / "libhiprecord.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROCM, "include"), "-o",
                    so, os.path.join(HERE, "hip_record.c")], check=True)

    def run(body):
        src = CHILD % dict(repo=os.path.dirname(HERE), rec=so, body=body)
        r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
        return json.loads(r.stdout)
    return run


def test_new_batch_clears_its_states_in_order(child):
    """rkx_batch_create clears the states before rkx_batch_add writes one: the
    clear must not be left running on a stream the writes do not wait for."""
    out = child("""
p = rk_amd.Bruss2D(24)
with rk_amd.Batch() as b:
    b.add(p, "DOPRI54", 0.0, 1.0, p.ode_start(), 1e-6, h0=1e-3)
    out["unordered"] = rec.rec_unordered_writes()
""")
    assert out["unordered"] == 0


@pytest.mark.parametrize("ends", [200, 333, 400])
def test_step_graph_outlives_its_replays(child, ends):
    """A solve sees its end in pinned memory while the launches behind the last
    attempt are still queued: the graph they come from must not be destroyed
    before they have run."""
    out = child("""
import ctypes as C
p = rk_amd.Bruss2D(64)
y0 = p.ode_start()
rec.rec_next_solve(%d)
y, st, _ = rk_amd.solve_host(p, "DOPRI54", 0.0, 1.0, y0, 1e-6, h0=1e-3)
out["steps"] = st.steps
out["replays"] = rec.rec_graph_replays()
out["early"] = rec.rec_graph_destroyed_early()
""" % ends)
    assert out["replays"] > 0 and out["steps"] == ends
    assert out["early"] == 0


def test_solve_view_is_asked_for_coherent(child):
    """The host reads a solve's progress and end from pinned memory while kernels
    run, so that memory has to be fine-grained by request, not by the
    runtime's default."""
    out = child("""
rec.rec_next_solve(20)
p = rk_amd.Bruss2D(64)
rk_amd.solve_host(p, "DOPRI54", 0.0, 1.0, p.ode_start(), 1e-6, h0=1e-3)
out["flags"] = rec.rec_pinned_flags()
""")
    portable, mapped, coherent = 0x1, 0x2, 0x40000000
    assert out["flags"] == portable | mapped | coherent


@pytest.mark.parametrize("meth,tol,even", [("DOPRI54", 1e-6, False), ("DOPRI87", 1e-8, False),
                                           ("DOPRI54", 0.0, True), ("DOPRI87", 0.0, True),
                                           ("RK4", 0.0, True), ("HEUN2", 1e-6, True)])
def test_even_ensembles_get_a_lane_per_system(child, meth, tol, even):
    """Systems that take their turns on a bounded number of waves lose where all
    of them take the same number of attempts."""
    out = child("""
import ctypes as C
buf, m = (C.c_double * 16)(), rk_amd.method(%r)
p = C.addressof(buf)
out["grid"] = []
for count in (1, 256, 257, 65536, 65537, 262144):
    rc = rk_amd.lib().rkx_lv_ensemble(count, p, p, p, 0.0, 1.0, C.byref(m), %r, 1e-3, 10, p, p, None)
    assert rc == 0
    out["grid"].append(rec.rec_last_grid())
""" % (meth, tol))
    assert out["grid"] == [1, 1, 2, 256] + ([257, 1024] if even else [256, 256])


@pytest.mark.parametrize("problem,impl", [("rk_amd.Bruss2D(64)", "PipeDls"),
                                          ("rk_amd.Bruss2D(64)", "D"), ("rk_amd.LV(100)", "D")])
def test_host_control_waits_once_an_attempt(child, problem, impl):
    """The host's step control waits for each attempt's error and for nothing
    else, and passes its values through pinned memory."""
    out = child("""
p = %s
for limit in (20, 50):
    w, c = rec.rec_waits(), rec.rec_pageable_copies()
    y, st, _ = rk_amd.solve_host(p, "DOPRI54", 0.0, 1e9, p.ode_start(), 0.0, h0=1e-3,
                                 step_limit=limit, impl=%r, ctrl="host")
    assert st.steps == limit
    out[limit] = (rec.rec_waits() - w, rec.rec_pageable_copies() - c)
""" % (problem, impl))
    assert out["50"][0] - out["20"][0] == 30
    assert out["50"][1] == out["20"][1]


def test_kept_blocks_hold_what_is_asked(child):
    """A vector gets no larger block than its own size (to the page): the byte
    counts of a batch and its budget are those of the vectors."""
    out = child("""
big, small = rk_amd.Bruss2D(100), rk_amd.Bruss2D(92)
rec.rec_next_solve(5)
rk_amd.solve_host(big, "DOPRI54", 0.0, 1.0, big.ode_start(), 1e-6, h0=1e-3)
rec.rec_watch_copy(8 * small.n)
with rk_amd.Batch(hbm_budget=rk_amd.Batch.footprint(small, "DOPRI54")) as b:
    b.add(small, "DOPRI54", 0.0, 1.0, small.ode_start(), 1e-6, h0=1e-3)
    out["block"], out["asked"] = rec.rec_copy_block(), 8 * small.n
live = rec.rec_live_bytes()
rec.rec_next_solve(5)
rk_amd.solve_host(big, "DOPRI54", 0.0, 1.0, big.ode_start(), 1e-6, h0=1e-3)
out["again"] = rec.rec_live_bytes() - live
""")
    assert out["asked"] <= out["block"] < out["asked"] + 4096
    assert out["again"] == 0


def test_kept_memory_is_given_back(child):
    """What solves and batches keep goes back on request, and before any of the
    library's own allocations fails for want of it."""
    out = child("""
p = rk_amd.Bruss2D(700)
y0 = p.ode_start()
empty = rec.rec_live_bytes()
def solve():
    rec.rec_next_solve(5)
    rk_amd.solve_host(p, "DOPRI54", 0.0, 1.0, y0, 1e-6, h0=1e-3)
solve()
out["kept"] = rec.rec_live_bytes() - empty
rec.rec_limit(rec.rec_live_bytes() + 1000)
rk_amd.Batch().close()
out["after a batch at the limit"] = rec.rec_live_bytes() - empty
solve()
rec.rec_limit(rec.rec_live_bytes() + 1000)
import ctypes as C
dp = C.POINTER(C.c_double)
q = rk_amd.Bruss2D(280)
big, g = q.ode_start(), np.empty(q.n)
rc = rk_amd.lib().rkx_eval_rng_host(C.byref(q.desc), 0, q.n - 1, 0.0, big.ctypes.data_as(dp),
                                    g.ctypes.data_as(dp))
out["eval at the limit"] = rc
rec.rec_limit(0)
solve()
staged = 2 * 8 * q.n
rk_amd.release_workspaces()
out["released"] = rec.rec_live_bytes() - empty - staged
""")
    assert out["kept"] >= 4 * 8 * 2 * 700 * 700
    assert out["after a batch at the limit"] < out["kept"] / 2     # its own arrays
    assert out["eval at the limit"] == 0
    assert out["released"] == 0


@pytest.mark.parametrize("problem,meth,steps,graph", [
    ("rk_amd.LVChain(100)", "DOPRI87", 60, True), ("rk_amd.LVChain(100)", "DOPRI87", 5, False),
    ("rk_amd.LVChain(100)", "DOPRI54", 60, False), ("rk_amd.LVChain(100)", "DOPRI54", 170, True)])
def test_graph_pays_by_kernels(child, problem, meth, steps, graph):
    """Whether a solve's steps come from a graph depends on the kernels it
    expects to launch: a step of the full-storage forms is many."""
    out = child("""
p = %s
rec.rec_next_solve(%d)
y, st, _ = rk_amd.solve_host(p, %r, 0.0, 1e3, p.ode_start(), 1e-6, h0=1e-3, step_limit=%d)
out["steps"], out["replays"] = st.steps, rec.rec_graph_replays()
out["early"] = rec.rec_graph_destroyed_early()
""" % (problem, steps, meth, steps))
    assert out["early"] == 0 and (out["replays"] > 0) == graph


def test_batches_use_their_arrays_again(child):
    """Another batch after one has ended allocates no device memory, and starts
    with cleared states."""
    out = child("""
with rk_amd.Batch() as b:
    pass
made = rec.rec_allocations()
p = rk_amd.Bruss2D(24)
with rk_amd.Batch() as b:
    out["again"] = rec.rec_allocations() - made
    b.add(p, "DOPRI54", 0.0, 1.0, p.ode_start(), 1e-6, h0=1e-3)
    out["unordered"] = rec.rec_unordered_writes()
""")
    assert out == {"again": 0, "unordered": 0}
