"""Cells at and beyond the edges of the ranges in which the cell kernels take
the branch-free form of the chain (kernels.hip: ordinary_cell): every second
cell has one parameter or starting state at an edge of its range (where the
branch-free form has to agree with the reference's branches) or outside it
(where the cell takes the branches as written), its neighbours in the wave
are ordinary.  States and fluxes against the oracle to the parity bar of
tests/test_gpu_parity.py (the two forms differ by roundings only), for the
fused and the plain kernel."""
import sys

import numpy as np
import pytest

from mhm_amd import parameters as PM, synth
from pairs import compare_cells, make_pair

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-10, 1e-12
EPS = np.finfo(float).eps

# (field, value): edges first, then values outside the ranges
EDGES = [("FSEALED", 0.0), ("FSEALED", 1.0), ("SEALED_THRESH", 2e-15), ("DEGDAY_INC", 0.0),
         ("DEGDAY_NOPRE", 0.0), ("DEGDAY_MAX", 0.0), ("KARSTLOSS", 0.0), ("ALPHA", -0.5),
         ("ALPHA", 0.0), ("UNSAT_THRESH", 2e-15), ("KBASEFLOW", "one step"), ("KPERCO", 0.02),
         ("KFASTFLOW", 0.01), ("KSLOWFLOW", 0.01), ("SOILMOIST_EXP", 1.0), ("SOILMOIST_EXP", 20.0),
         ("SOILMOIST_SAT", "one"), ("SOILMOIST_FC", "sat"), ("WILTINGPOINT", 0.0),
         ("WILTINGPOINT", "close"), ("FROOTS", 0.0), ("MAXINTER", 0.0), ("MAXINTER", EPS),
         ("MAXINTER", 1e-12), ("TEMP_THRESH", 10.0)]
OUTSIDE = [("SEALED_THRESH", 0.0), ("DEGDAY_INC", -0.4), ("DEGDAY_NOPRE", -0.5),
           ("DEGDAY_MAX", -1.0), ("KBASEFLOW", 0.01), ("ALPHA", -1.5), ("UNSAT_THRESH", 0.0),
           ("SOILMOIST_EXP", 0.3), ("SOILMOIST_SAT", "small"), ("SOILMOIST_FC", "above sat"),
           ("WILTINGPOINT", "fc"), ("WILTINGPOINT", "above fc"), ("FROOTS", -0.1),
           ("KARSTLOSS", -0.2)]


def _special(params, name, value, c, timestep):
    """Puts one field of cell c to a special value."""
    v = params[name]
    sat, fc, wp = (params[k] for k in ("SOILMOIST_SAT", "SOILMOIST_FC", "WILTINGPOINT"))
    if value == "one step":
        v[c] = timestep / 24.0
    elif value in ("one", "small"):
        f = (1.0 if value == "one" else 0.2) / sat[c]
        for a in (sat, fc, wp):
            a[c] = a[c] * f
        sat[c] = 1.0 if value == "one" else 0.2
    elif value == "sat":
        fc[c] = sat[c]
    elif value == "above sat":
        fc[c] = 1.5 * sat[c]
    elif value == "close":
        wp[c] = fc[c] * (1.0 - 1e-9)
    elif value == "fc":
        wp[c] = fc[c]
    elif value == "above fc":
        wp[c] = 1.2 * fc[c]
    else:
        v[c] = value


@pytest.mark.parametrize("nh,soil,timestep", [(1, 1, 1), (3, 1, 1), (3, 3, 1), (3, 1, 24), (6, 2, 6)])
def test_cells_at_and_beyond_the_ranges_match_oracle(nh, soil, timestep):
    depth = {1: [1000.0], 3: [200.0, 500.0, 1000.0],
             6: [50.0, 100.0, 200.0, 400.0, 800.0, 1400.0]}[nh]
    cases = EDGES + OUTSIDE
    # 2 x len(cases) cells and a ragged end, over more than one wave
    dom = synth.make_domain(11, 13, seed=61, horizon_depth=np.array(depth))
    params = synth.cell_params(dom, PM.DEFAULT)
    params = {k: np.array(v, dtype=float) for k, v in params.items()}
    for i, (name, value) in enumerate(cases):
        for c in range(1 + 2 * i, dom.n_cells, 2 * len(cases)):
            _special(params, name, value, c, timestep)
    for mode in (1, 0):
        print(f"case: cell ranges nh={nh} soil={soil} timestep={timestep} mode={mode}", flush=True)
        sys.stdout.flush()
        model, sim, steps, recs = make_pair([dom], n_steps=60, timestep=timestep, soil=soil, seed=62)
        model.set_params(params, 0)
        sim.set_params(params, 0)
        model.run(steps[:36], mode=mode, steps_per_launch=12)
        for r in recs[:36]:
            sim.step(r)
        bad = compare_cells(model, sim, RTOL, ATOL)
        assert bad == [], bad
        # starting states outside their ranges: an overfull horizon, an empty
        # one, an empty and a negative store
        sm = np.array(model.get("SOILMOIST")).reshape(dom.n_cells, nh)
        sm[0::10, 0] = 1.2 * params["SOILMOIST_SAT"][0::10, 0]
        sm[2::10, nh - 1] = 0.0
        un, pack = model.get("UNSATSTW"), model.get("SNOWPACK")
        un[4::10], pack[6::10] = 0.0, -1.0
        satw = model.get("SATSTW")
        satw[8::10] = -0.5
        for name, v in (("SOILMOIST", sm), ("UNSATSTW", un), ("SNOWPACK", pack), ("SATSTW", satw)):
            model.set_var(name, v)
            for d in sim.ds:
                if name == "SOILMOIST":
                    d[0].S[5:5 + nh] = sm.T
                else:
                    d[0].S[{"SNOWPACK": 1, "UNSATSTW": 3, "SATSTW": 4}[name]] = v
        model.run(steps[36:], mode=mode, steps_per_launch=12)
        for r in recs[36:]:
            sim.step(r)
        bad = compare_cells(model, sim, RTOL, ATOL)
        assert bad == [], bad
        model.close()
