"""The tiled routing kernel's loops (kernels.hip: tile_sweep) against the
wavefront schedule (one launch per diagonal) and the oracle: windows shorter
than, equal to and no multiple of the fetch distance, a run that ends inside a
window, tiles of 2, 16 and 64 levels, a node with more upstream nodes than the
loop reads together, gauges inside tiles and at their roots, an inflow gauge
that cuts a node's upstream links.  Every schedule does the same operations on
a node's series in the same order, so the schedules agree bit for bit; the
oracle's bar is that of tests/test_gpu_parity.py."""
import sys

import numpy as np
import pytest

from mhm_amd import _native as N, synth
from oracle_sim import rel_close
from pairs import compare_routing, make_pair

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-10, 1e-12


def _domain():
    """A basin in which ten leaves drain into one node of their own instead
    of their neighbours, and seven gauges along the main stem and beside it."""
    dom = synth.make_domain(30, 26, seed=51)
    indeg = np.bincount(dom.toN - 1, minlength=dom.n_cells)
    hub = int(np.argsort(dom.depth)[dom.n_cells // 2])
    leaf = np.flatnonzero(indeg[dom.fromN - 1] == 0)
    far = leaf[dom.toN[leaf] - 1 != hub][:10]
    dom.toN[far] = hub + 1
    dom.rOrder, perm = N.routing_order(dom.fromN, dom.toN, dom.n_cells)
    dom.netPerm = perm[:len(dom.fromN)].copy()
    assert np.bincount(dom.toN - 1).max() >= 10
    stem = np.argsort(dom.depth)[[0, 1, 15, 16, 17, 200, 500]]
    dom.gauge_nodes = (stem + 1).astype(np.int32)
    return dom


def _inflow(dom, n_steps):
    """An inflow gauge that is no headwater, at a node with upstream links."""
    node = int(dom.toN[dom.depth[dom.toN - 1] == 7][0])
    q = 2.0 + np.random.default_rng(5).gamma(2.0, 1.5, size=(n_steps, 1))
    return {"domain": [0], "node": [node], "headwater": [0], "q": q}


@pytest.mark.parametrize("height,window,inflow", [(16, 1, False), (16, 3, True), (16, 4, False),
                                                  (2, 5, True), (64, 8, False), (16, 64, True),
                                                  (64, 21, True)])
def test_tile_loops_match_the_wavefront(height, window, inflow):
    print(f"case: tile height {height}, window {window}, inflow {inflow}, 43 steps", flush=True)
    sys.stdout.flush()
    n, got = 43, []
    for mode, h in ((1, 0), (3, height)):
        dom = _domain()
        kw = {"inflow": _inflow(dom, n)} if inflow else {}
        model, sim, steps, recs = make_pair([dom], n_sets=2, n_steps=n, seed=12, tile_height=h, **kw)
        g = model.run(steps, mode=1, steps_per_launch=6, route_mode=mode,
                      route_window=window if mode == 3 else 0)
        if mode == 3:
            go = np.stack([sim.step(r) for r in recs])
            ok, worst = rel_close(g, go, RTOL, ATOL)
            assert ok, worst
            assert compare_routing(model, sim, RTOL, ATOL) == []
        got.append((g, [model.routing_state(s) for s in range(2)]))
        model.close()
    (g1, r1), (g3, r3) = got
    assert np.array_equal(g1, g3)
    for a, b in zip(r1, r3):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("height,inflow,packed", [(2, True, 0), (16, False, 0), (16, True, 0),
                                                  (64, True, 0), (16, False, 30), (16, False, 530)])
def test_step_by_step_matches_the_windows(height, inflow, packed):
    """mrm_step's one-launch routing (kernels.hip: route_step_kernel), with the
    windowed run in between, gives the windowed run's series bit for bit: the
    same operations per node.  packed: that many basins of a few cells more,
    all in tiles of depth 0 (530: more bins than the one launch is used for)."""
    print(f"case: steps, tile height {height}, inflow {inflow}, {packed} more basins", flush=True)
    sys.stdout.flush()
    n, got = 25, []
    small = [synth.make_domain(2, 3, seed=60 + i) for i in range(packed)]
    for per_step in (False, True):
        doms = ([] if packed > 512 else [_domain()]) + small
        kw = {"inflow": _inflow(doms[0], n)} if inflow else {}
        model, _, steps, _ = make_pair(doms, n_sets=2, n_steps=n, seed=13, tile_height=height, **kw)
        run = dict(mode=1, steps_per_launch=6, route_mode=3, route_window=5)
        if per_step:
            def walk(a, b):
                out = []
                for k in range(a, b):
                    if inflow:
                        model.set_inflow(kw["inflow"]["q"][k:k + 1])
                    model.mhm_step(steps[k])
                    out.append(model.mrm_step(steps[k]))
                return out
            g = walk(0, 9)
            if inflow:
                model.set_inflow(kw["inflow"]["q"][9:16])
            g = np.concatenate([np.stack(g), model.run(steps[9:16], **run), np.stack(walk(16, n))])
        else:
            g = model.run(steps, **run)
        got.append((g, [model.routing_state(s) for s in range(2)]))
        model.close()
    (g1, r1), (g2, r2) = got
    assert np.array_equal(g1, g2)
    for a, b in zip(r1, r2):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("height,window,n,windows", [(16, 64, 320, True), (16, 50, 333, True),
                                                     (24, 64, 330, True), (16, 4, 43, False)])
def test_many_sets_match_the_wavefront(height, window, n, windows):
    """Enough workgroups (bins times sets) to fill the chip: long windows go to
    the windowed launches (kernels.hip: route_tile_kernel), short ones to the
    one launch; with an inflow gauge, in pieces that end inside a window, and
    Qmod sums; bit for bit the wavefront's."""
    print(f"case: 100 sets, tile height {height}, window {window}, {n} steps", flush=True)
    sys.stdout.flush()
    got = []
    for mode, h in ((1, 0), (3, height)):
        dom = synth.make_domain(61, 60, seed=52)
        dom.gauge_nodes = (np.argsort(dom.depth)[[0, 1, 15, 16, 17, 900, 2500]] + 1).astype(np.int32)
        model, _, steps, _ = make_pair([dom], n_sets=100, n_steps=n, seed=14, tile_height=h,
                                       inflow=_inflow(dom, n))
        model.qmod_accumulate()
        model.set_profiling(True, 1)
        g = model.run(steps, mode=1, steps_per_launch=24, route_mode=mode,
                      route_window=window if mode == 3 else 0)
        if mode == 3:
            assert (model.profile()["route_tile"][1] > 3) == windows
        got.append((g, [model.routing_state(s) for s in (0, 77, 99)], model.qmod_sum(77)[0]))
        model.close()
    (g1, r1, q1), (g3, r3, q3) = got
    assert np.array_equal(g1, g3) and np.array_equal(q1, q3)
    for a, b in zip(r1, r3):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
