"""Every form a sparse Newton plan runs in: from the workspace (a dense tail beyond 256 rows, or a
working set beyond a CU's LDS), staged, and staged with a partly filled wide tail; program lists
longer than a wave holds at once; reaction terms of more than four factors.  Each case asserts the
form it is there for.

(I - gamma J) x = b against the dense Jacobian kernel's J: normwise backward error below 1e-12 in
FP64 and 1e-5 in FP32, the bounds of the same check on the shipped plans.  Short solves from the
workspace against the dense form: every abundance above 1e-14 within 1%, the bound between the
linear solvers elsewhere."""
import copy

import numpy as np
import pytest

from helpers import phys_of, random_state, term_magnitude

pytestmark = pytest.mark.gpu
W, S, SW = 0, 1, 2   # Network.WORKSPACE, STAGED, STAGED_WIDE


def _network(species, reactions, extra=()):
    """A seeded synthetic network (the shipped one of that size if there is one), with more reactions."""
    from uclchem_amd import makerates_hip as mh
    from uclchem_amd import synthetic as sy
    if not extra and (species, reactions) in ((150, 1500), (500, 6000)):
        return mh.load_network(mh.network_path(f"synthetic_{species}_{reactions}"))
    sp, re = sy.synthetic_species_and_reactions(species, reactions)
    return mh.build_tables(sp, re + list(extra), f"synthetic_{species}_{reactions}")


def _with_tail(t, tail):
    from uclchem_amd import newton_plan
    t2 = copy.copy(t)
    t2.arrays = {**t.arrays, **newton_plan.build_plan(t, split=t.neq + 2 - tail)}
    assert int(t2.arrays["nw_sizes"][2]) == tail
    return t2


def _states(t, net, charge):
    """Two states of a static cloud early and late in its first 1e4 yr."""
    from uclchem_amd import workloads
    from uclchem_amd.params import make_params
    net.set_linear_solver(net.DENSE)
    try:
        rows = net.solve(workloads.static_cloud_point(1e2), max_rec=60)
    finally:
        net.set_linear_solver(net.SPARSE)
    assert rows["status"][0] == 0
    p = make_params(initialdens=1e4, initialtemp=10.0, finaltime=1e4, enforcechargeconservation=charge)
    for k in (4, int(rows["n_rec"][0]) - 1):
        r = rows["rec"][0, k]
        yield p, np.array([r[1], r[2], r[2], r[3], float(np.float32(0.05)) * 3.086e18, 1e5, 1e-14, 0.0]), np.append(r[4:], r[1])


CASES = [((150, 1500), 1, W), ((150, 1500), 16, W), ((150, 1500), 32, S), ((140, 700), 0, S),
         ((300, 6000), 152, SW), ((400, 6000), 202, SW), ((500, 6000), 240, W), ((500, 6000), 257, W),
         ((500, 6000), 300, W)]


@pytest.mark.parametrize("size,tail,form", CASES)
def test_newton_solve_in_every_form(size, tail, form):
    from uclchem_amd import gpu
    t = _with_tail(_network(*size), tail)
    net = gpu.Network(t)
    assert net.plan_form()[0] == form, net.plan_form()
    rng = np.random.default_rng(tail)
    for charge in (False, True):
        for p, phys, y in _states(t, net, charge):
            rate, _, _ = net.rates(p[None], phys[None], y[None])
            J = net.jacobian(p[None], phys[None], rate, y[None])[0]
            for gamma in (1e4, 1e9):
                M = np.eye(t.neq) - gamma * J
                b = rng.standard_normal(t.neq)
                for bits, tol in ((64, 1e-12), (32, 1e-5)):
                    x = net.newton_solve(p[None], phys[None], y[None], gamma, b[None], lu_bits=bits)[0]
                    err = np.abs(M @ x - b).max() / (np.abs(M).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max())
                    assert err <= tol, (size, tail, charge, gamma, bits, err)


@pytest.mark.parametrize("size,tail,years", [((150, 1500), 16, 1e3), ((500, 6000), 300, 10.0)])
@pytest.mark.parametrize("lu_bits", [64, 32])
def test_solves_from_the_workspace(size, tail, years, lu_bits):
    from uclchem_amd import gpu, workloads
    from uclchem_amd.params import INDEX
    t = _with_tail(_network(*size), tail)
    net = gpu.Network(t)
    assert net.plan_form()[0] == W
    params = workloads.collapse_grid(3, final_time=years)
    params[1, INDEX["enforcechargeconservation"]] = 1.0
    out = net.solve(params, lu_bits=lu_bits)
    assert np.all(out["status"] == 0)
    net.set_linear_solver(net.DENSE)
    dense = net.solve(params, lu_bits=64)
    assert np.all(dense["status"] == 0)
    for q in range(len(params)):
        a, b = out["y"][q, :t.nspec], dense["y"][q, :t.nspec]
        m = b > 1e-14
        assert (np.abs(a[m] - b[m]) / b[m]).max() < 0.01, q


def test_lists_longer_than_a_wave():
    """The elimination program of the 140-species plan without a tail has more slices a wave than a
    wave's lanes hold descriptors (test_plan_host), and it runs staged."""
    from uclchem_amd import gpu, workloads
    t = _with_tail(_network(140, 700), 0)
    net = gpu.Network(t)
    assert net.plan_form()[0] == S
    params = workloads.collapse_grid(3, final_time=1e3)
    out = net.solve(params)
    net.set_linear_solver(net.DENSE)
    dense = net.solve(params)
    assert np.all(out["status"] == 0) and np.all(dense["status"] == 0)
    m = dense["y"][:, :t.nspec] > 1e-14
    assert (np.abs(out["y"] - dense["y"])[:, :t.nspec][m] / dense["y"][:, :t.nspec][m]).max() < 0.01


@pytest.fixture(scope="module")
def three_body():
    """A network with three-body reactions (two density powers and three reactants: five factors),
    its handle and its oracle."""
    from oracle import Oracle
    from uclchem_amd import gpu
    from uclchem_amd import makerates_hip as mh
    N = "NAN"
    extra = [mh.Reaction(["H", "H", "H2"], ["H2", "H2", N, N], 1e-28, -0.6, 0.0),
             mh.Reaction(["H", "H", "HE"], ["H2", "HE", N, N], 3e-29, -1.0, 0.0),
             mh.Reaction(["H", "CO", "H2"], ["H", "CO", "H2", N], 1e-26, 0.0, 100.0)]
    t = _network(150, 1500, extra)
    assert int(t.arrays["nfac"].max()) == 5
    return t, gpu.Network(t), Oracle(t)


def _random_states(t, orc, n):
    from uclchem_amd.params import make_params
    rng = np.random.default_rng(11)
    out = []
    for q in range(n):
        p = make_params(initialdens=10 ** rng.uniform(2, 8), initialtemp=rng.uniform(10, 300),
                        zeta=10 ** rng.uniform(0, 2), radfield=10 ** rng.uniform(0, 3), baseav=rng.uniform(0, 10),
                        finaltime=1e6)
        pt, y = random_state(t, orc, rng, p, bare_grains=(q % 3 == 0))
        out.append((p, phys_of(pt), y, pt))
    return out


def test_terms_of_more_than_four_factors(three_body):
    """RHS against the oracle to 1e-12 of each species' term magnitude, as on the other networks."""
    t, net, orc = three_body
    for p, phys, y, pt in _random_states(t, orc, 6):
        ro, yo, _ = orc.rates(pt, y)
        yd, r2 = orc.rhs(pt, ro, yo)
        ydg, _ = net.rhs(p[None], phys[None], ro[None], yo[None])
        assert np.all(np.abs(ydg[0] - yd) <= 1e-12 * term_magnitude(t, r2, yo))


@pytest.mark.parametrize("charge", [False, True])
def test_newton_solve_with_terms_of_more_than_four_factors(three_body, charge):
    t, net, _ = three_body
    assert net.plan_form()[0] == S
    rng = np.random.default_rng(5)
    for p, phys, y in _states(t, net, charge):
        rate, _, _ = net.rates(p[None], phys[None], y[None])
        J = net.jacobian(p[None], phys[None], rate, y[None])[0]
        for gamma in (1e4, 1e9):
            M = np.eye(t.neq) - gamma * J
            b = rng.standard_normal(t.neq)
            for bits, tol in ((64, 1e-12), (32, 1e-5)):
                x = net.newton_solve(p[None], phys[None], y[None], gamma, b[None], lu_bits=bits)[0]
                err = np.abs(M @ x - b).max() / (np.abs(M).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max())
                assert err <= tol, (charge, gamma, bits, err)
