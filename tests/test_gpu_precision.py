"""Rounding errors of the right-hand side's parts against extended precision (numpy's longdouble,
64-bit mantissa), held to what their operations allow: u = 2^-53 for every product, quotient and
sum, 2u for a correctly implemented transcendental function.

* A reaction term with a division by safeMantle: its factors one after another, u each.
* CO photodissociation without dust (Av = 0) at columns on the edges of the shielding table, where
  the splines return table entries exactly: the power of ten and four products."""
import numpy as np
import pytest

from helpers import phys_of, random_state

pytestmark = pytest.mark.gpu
U = 2.0 ** -53
LD = np.longdouble


def _states(t, orc, n, seed):
    from uclchem_amd.params import make_params
    rng = np.random.default_rng(seed)
    P, PH, Y, R = [], [], [], []
    for q in range(n):
        p = make_params(initialdens=10 ** rng.uniform(2, 8), initialtemp=rng.uniform(10, 60), zeta=10 ** rng.uniform(0, 2),
                        radfield=10 ** rng.uniform(0, 3), baseav=rng.uniform(0, 10), finaltime=1e6)
        pt, y = random_state(t, orc, rng, p)
        r, y, _ = orc.rates(pt, y)
        P.append(p)
        PH.append(phys_of(pt))
        Y.append(y)
        R.append(r)
    return np.array(P), np.array(PH), np.array(Y), np.array(R)


@pytest.mark.parametrize("name", ["default", "synthetic_150_1500", "synthetic_500_6000"])
def test_terms_divided_by_the_mantle(name, oracle_of):
    from uclchem_amd import gpu
    from uclchem_amd import makerates_hip as mh
    t = mh.load_network(mh.network_path(name))
    net = gpu.Network(t)
    P, PH, Y, R = _states(t, oracle_of(t), 60, 7)
    _, flux = net.rhs_fluxes(P, PH, R, Y)
    ops, nfac = t.ops, t.arrays["nfac"]
    pick = (ops == mh.OP_DIVSM).any(1) & ~((ops == mh.OP_SWAP) | (ops == mh.OP_BLR)).any(1)
    assert pick.sum() > 50
    checked = 0
    for q in range(len(P)):
        y = Y[q].astype(LD)
        sm = max(LD(1e-30), y[t.nsurface])
        v = R[q].astype(LD) * y[-1] ** t.n_d
        for k in range(ops.shape[1]):
            o = ops[:, k]
            v = np.where(o >= 0, v * y[np.maximum(o, 0)], np.where(o == mh.OP_DIVSM, v / sm, v))
        m = pick & (v > 1e-280)
        err = np.abs(flux[q][m] - v[m]) / v[m]
        assert np.all(err <= nfac[m] * U * (1 + 1e-6)), (q, float((err / (nfac[m] * U)).max()))
        checked += int(m.sum())
    assert checked > 300


def test_co_photodissociation_at_the_table_edges(tables, oracle):
    """kc = 2e-10 (G0 / 1.7) 10^s with s a table entry: the quotient and the products by 2e-10, by the
    shielding and by the dust's 1 (exact) round once each, the power of ten is good to 2u."""
    from uclchem_amd import gpu
    from uclchem_amd.params import INDEX
    t = tables
    net = gpu.Network(t)
    P, PH, Y, R = _states(t, oracle, 200, 9)
    rng = np.random.default_rng(3)
    # shielding table: [log N(CO) 12..18][log N(H2) 18..23], the 42 entries the reference's spline sees
    corner = {(0, 0): 0.0, (1, 0): -2.760, (0, 1): -1.676, (1, 1): -3.888}
    want = np.zeros(len(P), dtype=LD)
    for q in range(len(P)):
        co, h2 = q % 2, (q // 2) % 2
        PH[q, 3] = 0.0                                       # Av: no dust
        PH[q, 4] = 1e19
        Y[q, -1] = 1e4
        Y[q, t.scalars["nh2"]] = 1e-2 if h2 else 1e-8        # N(H2) = 5e20 ... 5e14: set to the edges below
        Y[q, t.scalars["nco"]] = 1e-3 if co else 1e-13
        if h2:
            PH[q, 4] = 1e22                                  # N(H2) = 5e23, beyond the last knot
            Y[q, t.scalars["nco"]] = 1e-6 if co else 1e-16   # N(CO) = 5e19 or 5e9
        P[q, INDEX["radfield"]] = 10 ** rng.uniform(0, 3)
        s = corner[(co, h2)]
        want[q] = LD(2.0e-10) * (LD(P[q, INDEX["radfield"]]) / LD(float(np.float32(1.7)))) * LD(10) ** LD(s)
    _, rate = net.rhs(P, PH, R, Y)
    kc = rate[:, int(t.scalars["nR_CO_hv"])]
    err = (np.abs(kc - want) / want).astype(float)
    print("[photo] CO at the table's corners, worst error in u by corner:",
          [round(float(err[k::4].max() / U), 2) for k in range(4)], flush=True)
    assert np.all(err <= 5 * U * (1 + 1e-6))
