"""Plans at the edge of a CU's LDS.  The dense tail is filled up to whole 16-row blocks where the
working set allows; where it does not, the plan runs staged with the tail it was built with, of 125
rows here, instead of from the workspace.

(I - gamma J) x = b against the dense Jacobian kernel's J: normwise backward error below 1e-12 in
FP64 and 1e-5 in FP32, and a short solve against the dense form within 1%, the bounds of the same
checks on the other plans."""
import numpy as np
import pytest

from test_gpu_plan_forms import S, _network, _states

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def edge():
    from uclchem_amd import gpu
    t = _network(250, 2500)
    assert int(t.arrays["nw_sizes"][2]) == 125
    return t, gpu.Network(t)


def test_plan_that_fits_without_the_filled_block_is_staged(edge):
    form, lds = edge[1].plan_form()
    assert form == S and lds <= 160 * 1024


@pytest.mark.parametrize("charge", [False, True])
def test_newton_solve_with_a_partly_filled_block(edge, charge):
    t, net = edge
    rng = np.random.default_rng(3)
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


@pytest.mark.parametrize("lu_bits", [64, 32])
def test_solves_with_a_partly_filled_block(edge, lu_bits):
    from uclchem_amd import workloads
    t, net = edge
    params = workloads.collapse_grid(3, final_time=1e2)
    out = net.solve(params, lu_bits=lu_bits)
    net.set_linear_solver(net.DENSE)
    try:
        dense = net.solve(params)
    finally:
        net.set_linear_solver(net.SPARSE)
    assert np.all(out["status"] == 0) and np.all(dense["status"] == 0)
    m = dense["y"][:, :t.nspec] > 1e-14
    assert (np.abs(out["y"] - dense["y"])[:, :t.nspec][m] / dense["y"][:, :t.nspec][m]).max() < 0.01


@pytest.mark.parametrize("size,tail", [((150, 1500), 16), ((220, 5000), None), ((500, 6000), 300)])
def test_workspace_form_takes_no_more_lds_than_its_arrays(size, tail):
    """The partials with two scratch vectors, four vectors of the state's length, 40 doubles of
    reduction slots and scalars and the parameters: what a network needs for the device to take it
    (the limit is a CU's LDS) must not grow beyond that."""
    from test_gpu_plan_forms import W, _with_tail
    from uclchem_amd import gpu
    from uclchem_amd.params import NPARAM
    t = _network(*size)
    if tail is not None:
        t = _with_tail(t, tail)
    form, lds = gpu.Network(t).plan_form()
    assert form == W
    pad = lambda n: (n + 7) & ~7
    npart = int(t.arrays["nfac"].sum())
    assert lds <= 8 * (max(t.nreac + 1, pad(npart) + 2 * pad(t.neq)) + 4 * pad(t.neq) + 40 + NPARAM)
