"""mrm_step's one routing launch (kernels.hip: route_step_kernel) with many bins
that wait for one another: basins of several bins each, packed, so that tickets
count past 512 and tile boundaries lead from bin to bin, in one set and several.
Gauges and states bit for bit those of the wavefront schedule (one launch per
diagonal), which knows no tiles."""
import sys

import numpy as np
import pytest

from mhm_amd import synth
from pairs import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_basins,shape,height,n_sets", [(280, (20, 20), 4, 1),
                                                          (100, (33, 31), 2, 2)])
def test_many_bins_hand_a_step_on(n_basins, shape, height, n_sets):
    print(f"case: step over {n_basins} basins {shape}, height {height}, {n_sets} sets", flush=True)
    sys.stdout.flush()
    kinds = [synth.make_domain(*shape, seed=70 + i) for i in range(4)]
    doms = [kinds[i % 4] for i in range(n_basins)]
    got = []
    for per_step in (False, True):
        model, _, steps, _ = make_pair(doms, n_sets=n_sets, n_steps=6, seed=14,
                                       tile_height=height if per_step else 0)
        if per_step:
            g = []
            for k in range(6):
                model.mhm_step(steps[k])
                g.append(model.mrm_step(steps[k]))
            g = np.stack(g)
        else:
            g = model.run(steps, mode=0, route_mode=1)
        got.append((g, [model.routing_state(s) for s in range(n_sets)]))
        model.close()
    (g1, r1), (g2, r2) = got
    assert np.array_equal(g1, g2)
    for a, b in zip(r1, r2):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
