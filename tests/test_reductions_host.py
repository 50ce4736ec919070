"""The solve kernel's reduction buffers along the step control's own paths (CPU).

A workgroup reduction has one barrier, so a buffer may be written again only if another barrier
lies after its last reads; the control code (bdf_core.h) has paths without one, such as the order
decision right after a corrector that converged in its first iteration at order 1.  red_host.cpp
runs the control code on stiff problems and logs every reduction's buffer and every barrier."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
START = {0: [1.0, 1.0, 1.0], 1: [1.0, 0.0, 0.0], 2: [1.0, 0, 0, 0, 0, 0, 0, 0.0057]}
ENDS = {0: [1e-6, 1e-3, 1.0, 10.0], 1: [1e-4, 0.4, 40.0, 4e5], 2: [1e-3, 1.0, 100.0, 321.8122]}


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("red_host") / "libredhost.so")
    subprocess.check_call([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", out,
                           os.path.join(HERE, "red_host.cpp")])
    lib = ctypes.CDLL(out)
    lib.red_host_run.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_double, ctypes.c_double,
                                 ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
    lib.red_host_cancel.argtypes = [ctypes.c_int] * 4 + [ctypes.c_void_p]
    return lib


@pytest.mark.parametrize("problem", [0, 1, 2])
@pytest.mark.parametrize("rtol", [1e-3, 1e-6, 1e-9])
@pytest.mark.parametrize("mxstep", [10, 10000])
def test_no_buffer_is_reused_without_a_barrier(lib, problem, rtol, mxstep):
    y, ends, out = np.array(START[problem]), np.array(ENDS[problem]), np.zeros(3, dtype=np.int32)
    lib.red_host_run(problem, len(ends), ends.ctypes.data, rtol, rtol * 1e-4, y.ctypes.data, mxstep, out.ctypes.data)
    hazards, reductions, after_correction = out
    assert reductions > 20
    assert after_correction > 0      # the path without a barrier is taken
    assert hazards == 0


@pytest.mark.parametrize("every", [1, 16])
@pytest.mark.parametrize("raised", [1, 2, 3])
def test_every_thread_gets_the_same_answer_to_a_cancel(lib, every, raised):
    """The word is raised between two readings; the threads of a workgroup must agree in every call
    (they meet barriers in what follows), and only one of them reads it."""
    threads, calls = 8, 64
    seen = np.zeros((threads, calls), dtype=np.int32)
    readings = lib.red_host_cancel(threads, calls, every, raised, seen.ctypes.data)
    assert np.all(seen == seen[0])
    assert readings == calls // every
    first = (raised - 1) * every
    want = np.zeros(calls, dtype=np.int32)
    want[first::every] = 1
    assert np.array_equal(seen[0], want)
