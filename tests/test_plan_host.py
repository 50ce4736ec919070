"""The planner of the device programs (uclchem_amd/csrc/ucg_plan.h) built for the host (CPU)."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("plan_host") / "libplanhost.so")
    subprocess.check_call([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out, os.path.join(HERE, "plan_host.cpp")])
    lib = ctypes.CDLL(out)

    def run(t, change=None):
        from uclchem_amd import gpu
        from uclchem_amd import makerates_hip as mh
        sizes, arrays, ssp, srx = mh.device_descriptor(t)
        if change:
            change(sizes, arrays)
        d = gpu._Desc()
        for k, v in sizes.items():
            if k == "nw_sizes":
                d.nw_sizes[:] = [int(x) for x in v]
            else:
                setattr(d, k, v)
        for k, v in arrays.items():
            setattr(d, k, v.ctypes.data)
        d.special_species[:] = [int(x) for x in ssp]
        d.special_reactions[:] = [int(x) for x in srx]
        res = np.zeros(17, dtype=np.int32)
        assert lib.plan_host(ctypes.byref(d), 8, 128, res.ctypes.data_as(ctypes.c_void_p)) == 0
        return dict(ok=res[0], wide=res[1], presum=res[2], ns=res[3], tail=res[4], slots=res[5],
                    sums=res[6:15].reshape(3, 3), entry_slices=res[15], pivot_slices=res[16])
    return run


def _no_ions(sizes, arrays):
    sizes["nion"] = 0
    arrays["ion_list"] = np.zeros(0, dtype=np.int32)
    arrays["nw_eion"] = np.zeros(0, dtype=np.int32)


@pytest.mark.parametrize("name,tail", [("default", None), ("synthetic_150_1500", None), ("synthetic_150_1500", 0)])
def test_sum_rows_of_a_network_without_positive_ions(plan, name, tail):
    """The solve adds up the replaced rows' right-hand sides, the electron row's among them whenever
    the charge is enforced: with no positive ion its sum is empty, and its row is still one of the
    system's.  Without a tail the sums are formed ahead of the solve, from these rows."""
    import copy
    from uclchem_amd import makerates_hip as mh
    from uclchem_amd import newton_plan
    t = mh.load_network(mh.network_path(name))
    if tail is not None:
        t = copy.copy(t)
        t.arrays = {**t.arrays, **newton_plan.build_plan(t, split=t.neq + 2 - tail)}
    with_ions, without = plan(t), plan(t, _no_ions)
    assert with_ions["ok"] and without["ok"] and bool(without["presum"]) == (tail == 0)
    rows = with_ions["ns"] + with_ions["tail"]
    assert np.all((without["sums"][:, 0] >= 0) & (without["sums"][:, 0] < rows))
    assert np.array_equal(without["sums"][:, 0], with_ions["sums"][:, 0])
    assert without["sums"][2, 1] == without["sums"][2, 2]      # nothing to add


def test_elimination_lists_longer_than_a_wave(plan):
    """A wave holds 64 slice descriptors at a time; the plan that test_gpu_plan_forms runs for longer
    lists has them."""
    import copy
    from uclchem_amd import makerates_hip as mh
    from uclchem_amd import newton_plan
    from uclchem_amd import synthetic as sy
    sp, re = sy.synthetic_species_and_reactions(140, 700)
    t = mh.build_tables(sp, re, "synthetic_140_700")
    t.arrays = {**t.arrays, **newton_plan.build_plan(t, split=t.neq + 2)}
    p = plan(t)
    assert p["ok"] and p["tail"] == 0 and p["pivot_slices"] > 64
