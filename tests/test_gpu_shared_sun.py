"""Daily runs of several parameter sets, whose cells share their days' sun terms
(kernels.hip: sun_kernel), against the plain loop, where every lane evaluates
its own: the same operations, so states, every flux of the last step, output
sums and gauges agree bit for bit.  Sets and calls at and below the sharing's
bounds, a launch length that divides the run and one that does not, a captured
run repeated on other days, a set with latitudes of its own, cells outside the
branch-free ranges, days without PET (tmax <= tmin, cold)."""
import sys

import numpy as np
import pytest

from mhm_amd import _native as N, synth
from pairs import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_sets,n_steps,S,timestep,soil,outputs",
                         [(4, 9, 4, 24, 1, True), (5, 40, 8, 24, 1, True), (3, 20, 8, 24, 1, True),
                          (7, 33, 365, 24, 1, True), (4, 8, 8, 24, 1, True),
                          (6, 30, 12, 12, 1, True), (7, 33, 365, 24, 1, False),
                          (5, 40, 8, 24, 3, False)])
def test_shared_sun_terms_match_the_plain_loop(n_sets, n_steps, S, timestep, soil, outputs):
    print(f"case: {n_sets} sets, {n_steps} steps of {timestep} h, {S} per launch, soil {soil}, "
          f"outputs {outputs}", flush=True)
    sys.stdout.flush()
    dom = synth.make_domain(13, 11, seed=101)
    models = []
    for _ in range(3):
        model, _, steps, _ = make_pair([dom], n_sets=n_sets, n_steps=2 * n_steps, seed=15,
                                       timestep=timestep, soil=soil)
        tmax, tmin = dom.forcing["TMAX"].copy(), dom.forcing["TMIN"]
        tmax[::3, ::5] = tmin[::3, ::5]
        model.set_forcing("TMAX", tmax)
        tavg = dom.forcing["TAVG"].copy()
        tavg[1::4, ::7] = -20.0
        model.set_forcing("TAVG", tavg)
        model.set_var("LATITUDE", dom.lat + 3.0, n_sets - 1)
        odd = np.full(model.n_cells, 0.4)
        odd[::17] = -0.4
        model.set_var("DEGDAY_INC", odd, 1)
        if outputs:
            model.output_accumulate([k != 18 for k in range(1, 22)])
        models.append(model)
    plain, eager, graph = models
    for a, b in ((0, n_steps), (n_steps, 2 * n_steps)):
        want = plain.run(steps[a:b], mode=0)
        for m, g in ((eager, False), (graph, True)):
            got = m.run(steps[a:b], mode=1, steps_per_launch=S, use_graph=g)
            assert np.array_equal(got, want)
            for s in range(n_sets):
                for name in list(N.S) + list(N.X):
                    assert np.array_equal(m.get(name, s), plain.get(name, s)), (name, s)
                if outputs:
                    assert np.array_equal(m.output_sum(11, 1, s)[0], plain.output_sum(11, 1, s)[0])
    for m in models:
        m.close()
