"""Muskingum coefficients from the routing parameters (reg_rout,
mo_mrm_mpr.f90:61-119) on the device: per set and domain, for one domain or
all at once, after the network was bound again; the same IEEE operations in
the same order as here, so bit for bit."""
import sys

import numpy as np
import pytest

from mhm_amd import engine, parameters as PM, synth

pytestmark = pytest.mark.gpu


def _reg_rout(dom, p, ts):
    if len(dom.length) == 0:
        return np.zeros(0), np.zeros(0)
    k = p[0] + p[1] * (dom.length * 0.001) + p[2] * dom.slope + p[3] * dom.fFPimp
    xi = np.minimum(p[4] * (1.0 + dom.slope / dom.slope.max()), 0.5)
    xi = np.maximum(xi, 0.005)
    k = np.minimum(k, 0.5 * ts / xi)
    k = np.maximum(k, 0.5 * ts / (1.0 - xi))
    c1 = ts / (k * (1.0 - xi) + 0.5 * ts)
    return c1, 1.0 - c1 * k / ts


@pytest.mark.parametrize("shapes,timestep", [([(1, 1)], 1), ([(1, 2), (16, 17)], 24),
                                             ([(20, 31), (1, 1), (7, 9)], 1), ([(130, 127)], 24)])
def test_reg_rout_matches_numpy(shapes, timestep):
    print(f"case: reg_rout {shapes}, timestep {timestep} h", flush=True)
    sys.stdout.flush()
    doms = [synth.make_domain(r, c, seed=90 + i) for i, (r, c) in enumerate(shapes)]
    model = engine.Model(doms, n_sets=3, timestep=timestep, n_forcing_days=1, route=True)
    rng = np.random.default_rng(91)
    for rebind in range(2):
        if rebind:
            for d in doms:
                d.length = d.length * 1.25
                d.slope = d.slope[::-1].copy()
        model.bind_network()
        gam = PM.draw(rng, 3 * len(doms)).reshape(3, len(doms), -1)
        for s in range(3):
            if s == 1:  # every domain at once
                model.set_routing_params(PM.routing_gamma(gam[s, 0]), s, -1)
            else:
                for i in reversed(range(len(doms))):
                    model.set_routing_params(PM.routing_gamma(gam[s, i]), s, i)
        for s in range(3):
            want = [_reg_rout(d, PM.routing_gamma(gam[s, 0 if s == 1 else i]), float(timestep))
                    for i, d in enumerate(doms)]
            got = model.routing_state(s)
            n = sum(len(d.length) for d in doms)
            assert np.array_equal(got["C1"][:n], np.concatenate([w[0] for w in want]))
            assert np.array_equal(got["C2"][:n], np.concatenate([w[1] for w in want]))
    model.close()
