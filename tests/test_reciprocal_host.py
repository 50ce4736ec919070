"""Reciprocals of pivots (uclchem_amd/csrc/ucg_recip.h) built for the host (CPU): over the whole
range of doubles a pivot is either refused, and only if its reciprocal is not finite or it is zero or
not finite itself, or its reciprocal is the quotient to half a unit in the last place."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def recip(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("rcp_host") / "librcphost.so")
    subprocess.check_call([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "rcp_host.cpp")])
    f = ctypes.CDLL(out).pivot_reciprocals

    def run(x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        r, bad = np.empty_like(x), np.empty(len(x), dtype=np.int32)
        f(ctypes.c_int(len(x)), *(a.ctypes.data_as(ctypes.c_void_p) for a in (x, r, bad)))
        return r, bad.astype(bool)
    return run


@pytest.mark.parametrize("lo,hi", [(-1074, -1021), (-1022, -990), (-60, 60), (990, 1010), (1010, 1024)])
def test_reciprocal_is_the_quotient(recip, lo, hi):
    rng = np.random.default_rng(1)
    x = np.ldexp(rng.uniform(0.5, 1.0, 20000), rng.integers(lo + 1, hi + 1, 20000)) * rng.choice([-1.0, 1.0], 20000)
    x = x[x != 0]
    r, bad = recip(x)
    with np.errstate(over="ignore"):
        want = 1.0 / x
    assert np.array_equal(bad, ~np.isfinite(want))
    r, want, x = r[~bad], want[~bad], x[~bad]
    # half a unit for the last rounding; the steps before it leave less than 2^-40 of the value
    err = np.abs(r.astype(np.longdouble) * x.astype(np.longdouble) - 1)
    unit = np.spacing(np.abs(want)).astype(np.longdouble) * np.abs(x)
    assert np.all(err <= 0.501 * unit)


def test_pivots_without_a_reciprocal_are_refused(recip):
    _, bad = recip([0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, 2.0 ** -1030, -2.0 ** -1030])
    assert np.all(bad)
