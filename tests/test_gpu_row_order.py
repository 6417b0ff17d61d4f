"""Rows of states, parameters of links and sums come back in the reference's
order, whatever their length (a download of 64k values or more is split into
parts): what was set is what is read, bit for bit, for cells, for nodes of an
equal and of a coarser routing grid, and for links; one cell, a partial wave,
sizes at which the number of parts changes."""
import sys

import numpy as np
import pytest

from mhm_amd import engine, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrows,ncols,refine", [(1, 1, 1), (3, 5, 1), (9, 7, 2), (256, 256, 1),
                                                (131, 1001, 1), (362, 364, 1), (110, 61, 5)])
def test_rows_come_back_in_order(nrows, ncols, refine):
    print(f"case: rows of {nrows}x{ncols} nodes, refinement {refine}", flush=True)
    sys.stdout.flush()
    dom = synth.make_domain(nrows, ncols, seed=81)
    if refine > 1:
        dom = synth.refine_domain(dom, refine, 82)
    rng = np.random.default_rng(83)
    model = engine.Model([dom], n_sets=2, n_forcing_days=1, route=True)
    n, snow, soil = model.n_cells, [], []
    for bound in (False, True):  # the order changes with the network
        if bound:
            model.bind_network()
        for s in range(2):
            snow.append(rng.uniform(size=n))
            soil.append(rng.uniform(size=(n, model.n_horizons)))
            model.set_var("SNOWPACK", snow[-1], s)
            model.set_var("SOILMOIST", soil[-1], s)
        for s in range(2):
            assert np.array_equal(model.get("SNOWPACK", s), snow[-2 + s])
            assert np.array_equal(model.get("SOILMOIST", s), soil[-2 + s])
    nodes, links = model.n_nodes, len(dom.fromN)
    qtin, qtr = rng.uniform(size=(2, nodes))
    c1, c2 = rng.uniform(size=(2, max(links, 1)))
    model.set_routing_state(qtin, qtr, 1, C1=c1, C2=c2)
    got = model.routing_state(1)
    has_link = np.zeros(nodes, bool)
    has_link[dom.fromN - 1] = True
    assert np.array_equal(got["qTIN"], qtin) and np.array_equal(got["Qmod"], qtin)
    assert np.array_equal(got["qTR"][has_link], qtr[has_link])
    if links:
        assert np.array_equal(got["C1"], c1) and np.array_equal(got["C2"], c2)
    assert np.array_equal(model.get("SNOWPACK", 1), snow[-1])
    model.close()


@pytest.mark.parametrize("nrows,ncols,n_sets,nh", [(1, 1, 1, 1), (5, 13, 3, 2), (16, 16, 1, 3),
                                                   (17, 19, 70, 5)])
def test_default_states_fill_every_set(nrows, ncols, n_sets, nh):
    """mo_init_states.f90:273-287: the same value for every cell of every set,
    zero fluxes, whatever was there before."""
    print(f"case: default states {nrows}x{ncols}, {n_sets} sets, {nh} horizons", flush=True)
    sys.stdout.flush()
    dom = synth.make_domain(nrows, ncols, seed=84)
    dom.horizon_depth = np.linspace(100.0, 100.0 * nh, nh)
    model = engine.Model([dom], n_sets=n_sets, n_forcing_days=1, route=False)
    n = model.n_cells
    for s in (0, n_sets - 1):
        for k in ("INTER", "SNOWPACK", "SEALSTW", "UNSATSTW", "SATSTW"):
            model.set_var(k, np.full(n, -3.0), s)
        model.set_var("SOILMOIST", np.full((n, nh), -3.0), s)
    model.default_states()
    hd = dom.horizon_depth
    edge = np.concatenate([[0.0], hd[:-1], [1500.0]])
    want = {"INTER": 0.0, "SNOWPACK": 15.0, "SEALSTW": 0.0, "UNSATSTW": 10.0, "SATSTW": 75.0,
            "TOTAL_RUNOFF": 0.0}
    for s in (0, n_sets // 2, n_sets - 1):
        for k, v in want.items():
            assert np.array_equal(model.get(k, s), np.full(n, v)), (k, s)
        soil = model.get("SOILMOIST", s).reshape(n, nh)
        assert np.array_equal(soil, np.tile((edge[1:] - edge[:-1]) * 0.25, (n, 1))), s
    model.close()
