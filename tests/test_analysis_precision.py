"""Rounding of the analysis' geometric swap terms (CPU): they carry the surface's total rate of
change, a sum over reaction terms of both signs.  Against extended precision, relative to the sum of
the terms' magnitudes, it must be no further off than the plain form, each species' rate of change
and then their sum."""
import numpy as np
import pytest


class _Net:
    def __init__(self, t, flux):
        self.t, self.flux = t, flux

    def rhs_fluxes(self, params, phys, rate, y):
        return np.zeros((len(y), self.t.neq)), self.flux


@pytest.mark.parametrize("name", ["default", "synthetic_150_1500", "synthetic_500_6000"])
def test_surface_total_is_as_accurate_as_the_plain_sum(name):
    from uclchem_amd import analysis
    from uclchem_amd import makerates_hip as mh
    t = mh.load_network(mh.network_path(name))
    surf = np.asarray(t.arrays["surface_list"])
    inc = analysis.construct_incidence(t)
    ns = t.scalars
    rows = 200
    rng = np.random.default_rng(17)
    flux = 10 ** rng.uniform(-25, -17, (rows, t.nreac))
    ab = 10 ** rng.uniform(-20, -4, (rows, 1, t.nspec))
    ab[:, 0, ns["nbulk"]], ab[:, 0, ns["nsurface"]] = 1e-4, 1e-5
    physics = np.ones((rows, 1, 8))
    _, out, cols = analysis.rates_to_dy_and_flux(physics, ab, np.ones((rows, 1, t.nreac)), net=_Net(t, flux))
    LD = np.longdouble
    exact = (flux.astype(LD) @ inc.astype(LD)[:, surf]).sum(axis=1)
    # the total back from the terms: the first pair whose term is not zero in the row
    pairs = (out.shape[2] - t.nreac) // 2
    assert pairs > 0
    b, s = analysis._swap_pairs(t)[0]
    yb, ys = (ab[:, 0, int(t.arrays["re"][k][0])].astype(LD) for k in (b, s))
    ybulk, ysurf = ab[:, 0, ns["nbulk"]].astype(LD), ab[:, 0, ns["nsurface"]].astype(LD)
    cover = LD(0.5 * analysis.GAS_DUST_DENSITY_RATIO / analysis.NUM_SITES_PER_GRAIN)
    geo = out[:, 0, t.nreac:]
    want = np.where(exact < 0, exact * np.minimum(LD(1), ybulk / ysurf) * yb / ybulk, exact * cover * ys)
    got = np.where(exact < 0, geo[:, 0], geo[:, pairs])
    plain = (flux @ inc.astype(np.float64))[:, surf].sum(axis=1)
    mag = (flux @ np.abs(inc.astype(np.float64)[:, surf])).sum(axis=1)
    rms = lambda e: float(np.sqrt(np.mean(np.asarray(e, dtype=np.float64) ** 2)))
    error, allowed = rms((got - want) / want * exact / mag), rms((plain - exact) / mag)
    own = 4 * 2.0 ** -53 * rms(exact / mag)      # the terms' own products and quotients round besides
    assert error <= np.hypot(allowed, own), (error, allowed, own)
