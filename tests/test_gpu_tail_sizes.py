"""Newton solves with the dense tail of the plan at the edges of its 16-row blocks: no tail, one row,
around one block, the sizes the shipped networks use, the largest a workgroup holds in registers as
one block, and past it, where the tail is factored as two blocks (on the large network up to its own
252 rows).  (I - gamma J) x = b against the dense Jacobian
kernel's J; the normwise backward error bounds are those of the same check at the shipped size:
an unpivoted FP64 elimination of a few hundred well-scaled rows stays below 1e-12, FP32 below 1e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base():
    from uclchem_amd import gpu
    from uclchem_amd import makerates_hip as mh
    cache = {}

    def get(name):
        if name not in cache:
            t = mh.load_network(mh.network_path(name))
            cache[name] = t, gpu.Network(t)
        return cache[name]
    return get


@pytest.mark.parametrize("name,tail", [("synthetic_150_1500", n) for n in (0, 1, 15, 16, 17, 77, 112, 113, 127, 128, 129)] +
                         [("synthetic_500_6000", 252)])
def test_newton_solve_at_tail_size(base, name, tail):
    import copy
    from uclchem_amd import gpu, newton_plan, workloads
    from uclchem_amd.params import make_params
    t, net = base(name)
    if int(t.arrays["nw_sizes"][2]) == tail:
        other = net
    else:
        t2 = copy.copy(t)
        plan = newton_plan.build_plan(t, split=t.neq + 2 - tail)
        t2.arrays = {**t.arrays, **plan}
        assert int(plan["nw_sizes"][2]) == tail
        other = gpu.Network(t2)
    rows = net.solve(workloads.static_cloud_point(1e4), max_rec=60)
    rec = rows["rec"][0, :rows["n_rec"][0]]
    rng = np.random.default_rng(tail)
    for enforce in (False, True):
        p = make_params(initialdens=1e4, initialtemp=10.0, finaltime=1e4, enforcechargeconservation=enforce)
        cs = float(np.float32(0.05)) * 3.086e18
        for k in (8, 20):
            y = np.append(rec[k, 4:], rec[k, 1])
            phys = np.array([rec[k, 1], rec[k, 2], rec[k, 2], rec[k, 3], cs, 1e5, 1e-14, 0.0])
            rate, _, _ = net.rates(p[None], phys[None], y[None])
            J = net.jacobian(p[None], phys[None], rate, y[None])[0]
            for gamma in (1e4, 1e9):
                M = np.eye(t.neq) - gamma * J
                b = rng.standard_normal(t.neq)
                for bits, tol in ((64, 1e-12), (32, 1e-5)):
                    x = other.newton_solve(p[None], phys[None], y[None], gamma, b[None], lu_bits=bits)[0]
                    err = np.abs(M @ x - b).max() / (np.abs(M).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max())
                    assert err <= tol, (tail, enforce, k, gamma, bits, err)
