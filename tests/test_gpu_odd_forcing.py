"""Weather for which the branch-free form of the snow (chain.h: snow_meteo) does
not hold: precipitation so far below zero (errors, nodata of -9999) that the
degree-day factor is negative.  A cell that has been given such weather takes the
branches as written, its neighbours in the wave stay as they are.  Every way
the forcing reaches the device, daily and hourly, fused and plain, single sets
and the daily launches that share sun terms, against the oracle to the parity
bar of tests/test_gpu_parity.py."""
import sys

import numpy as np
import pytest

from mhm_amd import calendar, engine, parameters as PM, synth
from oracle_sim import OracleSim
from pairs import START, compare_cells, make_pair

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-10, 1e-12
NODATA = -9999.0


def _domain(n_days):
    """Every second cell has odd days: -0.3 mm (the factor stays positive), -40
    mm and nodata, on days of hard frost, of thaw and as the series has them;
    the snow of the start lies on all cells."""
    dom = synth.make_domain(13, 17, seed=71)
    synth.make_forcing(dom, n_days, 72, doy0=START.timetuple().tm_yday)
    for name, shift in (("TAVG", 0.0), ("TMIN", -5.0), ("TMAX", 5.0)):
        for i, c in enumerate(range(1, dom.n_cells, 2)):
            t = (-15.0, 6.0, None)[i % 3]
            if t is not None:
                dom.forcing[name][:, c] = t + shift
    for i, c in enumerate(range(1, dom.n_cells, 2)):
        day = (i // 9) % n_days
        dom.forcing["PRE"][day, c] = (-0.3, -40.0, NODATA)[(i // 3) % 3]
    return dom


@pytest.mark.parametrize("how,timestep,n_sets", [("set", 1, 1), ("set", 24, 1), ("set", 24, 5),
                                                 ("stream", 1, 2), ("l2", 24, 4), ("l2", 1, 1),
                                                 ("weights", 1, 2)])
def test_odd_weather_matches_oracle(how, timestep, n_sets):
    n_steps, n_days = 96, 4
    for mode in (1, 0):
        print(f"case: odd weather {how} timestep={timestep} sets={n_sets} mode={mode}", flush=True)
        sys.stdout.flush()
        dom = _domain(n_days)
        if how == "weights":
            dom.forcing["PRE"] = np.abs(dom.forcing["PRE"]) % 50.0
        model, sim, steps, recs = make_pair([dom], n_sets=n_sets, timestep=timestep,
                                            n_steps=n_steps, seed=73, route=False,
                                            forcing_columns=n_days if how == "stream" else None,
                                            weights=how == "weights")
        if how == "weights":
            w = [np.array(v, dtype=float) for v in synth.make_meteo_weights(dom.n_cells, 974)]
            w[0].reshape(dom.n_cells, -1)[1::4] *= -3.0
            model.set_meteo_weights(*w)
            sim.set_meteo_weights(*w)
        elif how == "stream":
            model.stream_forcing(dom.forcing, day0=1)
        elif how == "l2":
            model.set_forcing("PRE", np.zeros_like(dom.forcing["PRE"]))
            # cells in Fortran order over a full grid
            grid = dom.forcing["PRE"].reshape(-1, 17, 13).transpose(0, 2, 1)
            ones = np.ones((13, 17), bool)
            model.set_forcing_l2("PRE", 0, grid, ones, 1.0, ones, 1.0)
        for a, b in ((0, n_steps // 2), (n_steps // 2, n_steps)):
            model.run(steps[a:b], mode=mode, steps_per_launch=12, want_gauges=False)
            for r in recs[a:b]:
                sim.step(r)
            bad = compare_cells(model, sim, RTOL, ATOL)
            assert bad == [], bad
        model.close()


def _states(model):
    return {k: model.get(k) for k in ("SNOWPACK", "SOILMOIST", "UNSATSTW", "SATSTW",
                                      "TOTAL_RUNOFF")}


def test_marks_go_with_the_forcing_that_gave_them():
    """Whole-range forcing without odd days leaves no trace of the odd ones
    before it: the states are those of a context that never had them, bit for
    bit (an ordinary cell that took the branches would differ by roundings)."""
    print("case: odd weather replaced", flush=True)
    got = []
    for odd_first in (False, True):
        dom = _domain(4)
        model, _, steps, _ = make_pair([dom], n_steps=96, seed=74, route=False)
        pre = np.abs(dom.forcing["PRE"]) % 40.0
        if odd_first:
            model.run(steps[:24], steps_per_launch=12, want_gauges=False)
            model.set_meteo_weights(*[-v for v in synth.make_meteo_weights(dom.n_cells, 75)])
            model.set_meteo_weights()
            model.default_states()
        model.set_forcing("PRE", pre)
        model.run(steps, steps_per_launch=12, want_gauges=False)
        got.append(_states(model))
        model.close()
    for k in got[0]:
        assert np.array_equal(got[0][k], got[1][k]), k


def test_marks_follow_the_cells_when_the_network_is_bound():
    """Binding a network re-lays the cells; the marks go with them."""
    print("case: odd weather before the network", flush=True)
    got = []
    for late in (False, True):
        dom = _domain(4)
        steps = calendar.step_table(START, 96, 1)
        model = engine.Model([dom], n_forcing_days=4)
        if not late:
            model.bind_network()
        model.set_params(synth.cell_params(dom, PM.DEFAULT), 0)
        model.default_states()
        model.set_domain_forcing()
        if late:
            model.bind_network()
        model.set_routing_params(PM.routing_gamma(PM.DEFAULT), 0)
        model.run(steps, steps_per_launch=12)
        got.append(_states(model))
        model.close()
    for k in got[0]:
        assert np.array_equal(got[0][k], got[1][k]), k


def test_streamed_marks_change_between_launches():
    """Chunks streamed while the loop runs on earlier days: the marks of a chunk
    come when its days are first read, so that two runs agree bit for bit
    however the uploads and the launches fall together."""
    print("case: odd weather streamed ahead", flush=True)
    got = []
    for ahead in (True, True, False):
        dom = _domain(8)
        model, _, steps, _ = make_pair([dom], n_steps=192, seed=77, route=False,
                                       forcing_columns=4)
        chunk = [{v: a[2 * k:2 * k + 2] for v, a in dom.forcing.items()} for k in range(4)]
        model.stream_forcing(chunk[0], day0=1)
        for k in range(4):
            if ahead and k < 3:
                model.stream_forcing(chunk[k + 1], day0=2 * k + 3)
            model.run(steps[48 * k:48 * k + 48], steps_per_launch=12, want_gauges=False)
            if not ahead and k < 3:
                model.sync()
                model.stream_forcing(chunk[k + 1], day0=2 * k + 3)
        got.append(_states(model))
        model.close()
    for other in got[1:]:
        for k in got[0]:
            assert np.array_equal(got[0][k], other[k]), k


def test_a_night_share_above_one_matches_oracle():
    """The day's share is then negative: every cell takes the branches."""
    print("case: odd day and night shares", flush=True)
    share = [1.6] * 12
    dom = _domain(4)
    dom.forcing["PRE"] = 30.0 * np.abs(dom.forcing["PRE"]) % 60.0
    steps, recs = calendar.step_table(START, 96, 1), calendar.step_records(START, 96, 1)
    params = synth.cell_params(dom, PM.DEFAULT)
    for mode in (1, 0):
        model = engine.Model([dom], route=False, n_forcing_days=4, fnight_prec=share)
        sim = OracleSim([dom], n_forcing_days=4, route=False, fnight_prec=share)
        for m in (model, sim):
            m.set_params(params, 0)
            m.default_states()
            m.set_domain_forcing()
        model.run(steps, mode=mode, steps_per_launch=12, want_gauges=False)
        for r in recs:
            sim.step(r)
        bad = compare_cells(model, sim, RTOL, ATOL)
        assert bad == [], bad
        model.close()
