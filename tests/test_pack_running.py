"""The list of running slots of a packed launch, with several queries: each query's slots in consecutive places from a
wave boundary, in admission order, the other places -1, launch after launch while slots run dry, and with query tables
larger than the launch.  The pass runs here on the CPU (tests/native/pack_running.cpp, built with hipcc for the host)."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not HIPCC:
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("pack") / "libpack.so")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "native", "pack_running.cpp")],
                   check=True, capture_output=True)
    return C.CDLL(out)


@pytest.mark.parametrize("queue,n_queries,waves", [
    ([0], 1, 4), ([0, 1], 2, 8), ([5, 2, 7], 64, 65),
    ([3, 1500, 1999], 2000, 8),      # a table of more entries than the launch has threads
    ([699, 4], 700, 4),
])
def test_list_of_running_slots(lib, queue, n_queries, waves):
    rng = np.random.default_rng(len(queue) * 1000 + waves)
    span, launches = 64 * waves, 12
    of_wave = rng.choice(queue, waves)
    state = np.repeat(of_wave, 64)
    alive = np.ones(span, dtype=bool)
    states, runs = [], []
    for _ in range(launches):
        alive = alive & (rng.random(span) < 0.7)
        states.append(np.where(alive.reshape(-1, 64).any(axis=1).repeat(64), state, -1))
        runs.append(alive)
    state = np.ascontiguousarray(states, dtype=np.int32)
    run = np.ascontiguousarray(runs, dtype=np.int32)
    order = np.ascontiguousarray(rng.permutation(waves), dtype=np.int32)
    q = np.ascontiguousarray(queue, dtype=np.int32)
    live = int(run[0].sum())
    list_span = (live + 63) // 64 * 64 + 64 * len(queue)      # Pool::shape's
    at = C.c_int()
    rc = lib.pack_check(launches, C.c_long(span), C.c_long(list_span), n_queries, q.ctypes.data_as(C.c_void_p), len(queue),
                        state.ctypes.data_as(C.c_void_p), run.ctypes.data_as(C.c_void_p), order.ctypes.data_as(C.c_void_p), C.byref(at))
    assert rc == 0, (rc, at.value)
