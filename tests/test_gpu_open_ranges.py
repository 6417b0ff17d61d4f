"""Values without bound that the reference never reads: the sealed storage and
its threshold in a cell without sealed area.  The branches leave them alone;
the branch-free form (chain.h: sealed_ordinary) weighs them by 0, so a cell
that has them infinite is no ordinary one (ordinary_params, ordinary_states).
Every other state and flux against the oracle, fused and plain."""
import numpy as np
import pytest

from mhm_amd import parameters as PM, synth
from oracle_sim import FLUX_NAMES, STATE_NAMES
from pairs import compare_cells, make_pair

pytestmark = pytest.mark.gpu

INF = np.inf


@pytest.mark.parametrize("store,threshold", [(INF, 2.0), (0.0, -INF), (-INF, 2.0)])
def test_unread_sealed_values_do_not_reach_the_runoff(store, threshold):
    dom = synth.make_domain(9, 11, seed=81)
    params = {k: np.array(v, dtype=float) for k, v in synth.cell_params(dom, PM.DEFAULT).items()}
    odd = np.arange(1, dom.n_cells, 3)
    params["FSEALED"][odd] = 0.0
    params["SEALED_THRESH"][odd] = threshold
    for mode in (1, 0):
        print(f"case: unread sealed values store={store} threshold={threshold} mode={mode}",
              flush=True)
        model, sim, steps, recs = make_pair([dom], n_steps=24, seed=82, route=False)
        model.set_params(params, 0)
        sim.set_params(params, 0)
        seal = model.get("SEALSTW")
        seal[odd] = store
        model.set_var("SEALSTW", seal)
        sim.ds[0][0].S[2] = seal
        model.run(steps, mode=mode, steps_per_launch=8, want_gauges=False)
        for r in recs:
            sim.step(r)
        assert np.array_equal(model.get("SEALSTW")[odd], sim.get("SEALSTW", 0)[odd])
        bad = compare_cells(model, sim, names=[n for n in STATE_NAMES + FLUX_NAMES
                                               if n != "SEALSTW"])
        assert bad == [], bad
        model.close()
