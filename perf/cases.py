"""The work users of this framework have it do, as measurable cases.

A user runs a basin (or several) through time: in one call of the time loop
(`Model.run`), step by step as a host model or a coupler does
(`Model.mhm_step` + `Model.mrm_step`), for many parameter sets at once, or as
a request of the serving loop (`serve.run_alone`).  The sizes are those of the
benchmark and the tests: basins of a few hundred to 1024 x 1024 cells, hourly
and daily steps, a day to a year, one to 256 parameter sets.

A case is a dict of plain values:

  kind        loop (Model.run), steps (per-step drop-in), request (serving)
  nrows, ncols  cells of the basin; refine > 1: the hydrology grid is that
              much finer than the routing grid (nrows x ncols nodes)
  basins, lo, hi  instead: that many basins of lo..hi cells (log-uniform)
  n_steps, timestep [h], n_sets, nh (soil horizons), soil, pet (process cases)
  weights     meteo weights instead of the day/night factors
  celerity    adaptive routing with this celerity [m/s] (0: Muskingum)
  gauges      discharge gauges per basin, along the rivers
  weather     fronts: rain and temperature that are coherent over a front's
              extent, as gridded daily observations are; local: every cell
              draws its own weather (the synthetic domains' generator)
  mode, S, block, graph, window, tile_height  options of the time loop / context
  restart     the run ends with every state read back, as for a restart file
  outputs     the L1 and L11 output sums are accumulated and read back
  field       L1_total_runoff is read back: after every step (each), after the
              last one (last) or not at all

The inputs come from the seed alone; the terrain and the river network come
from the size (a basin is laid out once and run with many forcings).
"""
import dataclasses
import datetime as dt
import functools
import math

import numpy as np
import torch

from mhm_amd import _native as N
from mhm_amd import calendar, engine, parameters as PM, serve, synth

START = dt.datetime(1990, 1, 1)
HORIZONS = {1: [1000.0], 2: [200.0, 1000.0], 3: [200.0, 500.0, 1000.0],
            4: [100.0, 300.0, 600.0, 1200.0], 5: [50.0, 150.0, 350.0, 700.0, 1300.0],
            6: [50.0, 100.0, 200.0, 400.0, 800.0, 1400.0]}
# outputFlxState switches (index k - 1 for output k) a run commonly writes:
# interception, snowpack, soil moisture per horizon and its mean fraction,
# unsaturated and saturated storage, PET, total aET, total runoff, baseflow,
# percolation, effective precipitation
OUTPUTS = (1, 2, 3, 5, 7, 8, 9, 10, 11, 15, 16, 20)
STATES = ("INTER", "SNOWPACK", "SEALSTW", "UNSATSTW", "SATSTW", "SOILMOIST")
ROUTING = ("qOUT", "qTIN", "qTR", "Qmod")

BASE = {"kind": "loop", "nrows": 64, "ncols": 64, "refine": 1, "basins": 0, "lo": 0, "hi": 0,
        "n_steps": 24, "timestep": 1, "n_sets": 1, "nh": 3, "soil": 1, "pet": 1, "weights": False,
        "celerity": 0.0, "gauges": 1, "weather": "fronts", "mode": N.RUN_FUSED, "S": 0, "block": 0,
        "graph": False, "window": 0, "tile_height": 0, "restart": False, "outputs": False,
        "field": "no"}


def _case(name=None, **kw):
    c = dict(BASE, **kw)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # a small coupled model: one day, a step at a time, the gauge and the
        # runoff field read after every step (the Python surface's loop):
        # launches and latency
        _case("coupled_day_24x30", kind="steps", nrows=24, ncols=30, field="each"),
        # the drop-in for the reference's time loop on a large basin: every
        # state and flux of a step on the device, gauges to the host each step
        _case("coupled_steps_1024", kind="steps", nrows=1024, ncols=1024, n_steps=12, gauges=40,
              tile_height=32, field="last"),
        # a year of one small catchment in one call, then the restart file
        _case("year_64x64", n_steps=8760, S=144, block=64, graph=True, window=64, restart=True,
              gauges=3),
        # the large basin: two months hourly with a gauging network
        _case("season_1024", nrows=1024, ncols=1024, n_steps=1440, S=144, graph=True, window=64,
              gauges=40, field="last"),
        # a calibration ensemble: 256 parameter sets on shared daily forcing
        _case("ensemble_256", n_steps=1095, timestep=24, n_sets=256, S=365, graph=True, window=64,
              weather="local"),
        # many catchments of uneven size packed in one context, a month hourly
        _case("basins_packed", nrows=0, ncols=0, basins=24, lo=500, hi=60000, n_steps=720, S=144,
              graph=True, window=64, field="last"),
        # a ragged basin with the call's defaults and a restart at the end
        _case("defaults_215x301", nrows=215, ncols=301, n_steps=720, restart=True, gauges=5,
              weather="local"),
        # Penman-Monteith on meteo weights with Jarvis stress and five horizons
        _case("penman_jarvis_96x130", nrows=96, ncols=130, n_steps=480, nh=5, soil=3, pet=3,
              weights=True, S=96, graph=True, window=32, restart=True),
        # daily output files from a hydrology grid twice as fine as the routing
        # grid: the sums of an output interval accumulated and read back
        _case("outputs_coarse_110x150", nrows=110, ncols=150, refine=2, n_steps=168, outputs=True,
              gauges=4),
        # every flux of every step on the device in one call (the plain loop)
        _case("plain_fluxes_700x900", nrows=700, ncols=900, n_steps=48, mode=N.RUN_PLAIN,
              gauges=20, field="last"),
        # adaptive routing time step (a constant celerity): several routings a step
        _case("celerity_150x220", nrows=150, ncols=220, n_steps=240, celerity=1.5, gauges=4,
              weather="local", restart=True),
        # a serving request from its arrival to its gauge series: context,
        # network, parameter sets, forcing, the run
        _case("request_141x142", kind="request", nrows=141, ncols=142, n_steps=180, timestep=24,
              n_sets=24, weather="local"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A basin of lo..hi cells, up to 1.6 times as long as wide."""
    n, r = _logint(rng, lo, hi), math.sqrt(rng.uniform(0.6, 1.6))
    nr = max(3, int(round(math.sqrt(n) * r)))
    return {"nrows": nr, "ncols": max(3, int(round(n / nr)))}


def draw(rng):
    weather = rng.choice(["fronts", "local"])
    kind = rng.choice(["steps", "loop", "loop", "graph", "graph", "sets", "packed", "process",
                       "outputs", "plain", "celerity", "request"])
    if kind == "steps":
        g = _grid(rng, 300, 700000)
        n = g["nrows"] * g["ncols"]
        return _case(kind="steps", n_steps=rng.randint(4, 24 if n < 50000 else 8), gauges=rng.randint(1, 30),
                     field="each" if n < 20000 else "last", tile_height=rng.choice([0, 32]), weather=weather, **g)
    if kind == "loop":
        return _case(n_steps=rng.randint(100, 900), gauges=rng.randint(1, 10), weather=weather,
                     restart=True, **_grid(rng, 600, 90000))
    if kind == "graph":
        g = _grid(rng, 2000, 600000)
        n = g["nrows"] * g["ncols"]
        return _case(n_steps=rng.randint(300, 1440) if n > 30000 else rng.randint(1000, 4000),
                     S=rng.choice([24, 72, 144]), block=rng.choice([0, 64, 128]), graph=True,
                     window=rng.choice([16, 32, 64]), gauges=rng.randint(1, 40), weather=weather,
                     restart=n < 60000, field="last", **g)
    if kind == "sets":
        return _case(n_steps=rng.randint(180, 900), timestep=24, n_sets=_logint(rng, 4, 200),
                     S=rng.choice([73, 365]), graph=True, window=64, weather=weather,
                     **_grid(rng, 500, 4200))
    if kind == "packed":
        lo = _logint(rng, 60, 2000)
        return _case(nrows=0, ncols=0, basins=rng.randint(3, 20), lo=lo, hi=lo * rng.randint(2, 25),
                     n_steps=rng.randint(120, 700), S=rng.choice([48, 144]), graph=True,
                     window=rng.choice([8, 64]), weather=weather, field="last")
    if kind == "process":
        return _case(n_steps=rng.randint(100, 480), nh=rng.choice([1, 2, 3, 4, 5, 6]),
                     soil=rng.choice([1, 3]), pet=rng.choice([-1, 0, 1, 2, 3]),
                     weights=rng.random() < 0.5, S=rng.choice([0, 48, 96]), weather=weather,
                     timestep=rng.choice([1, 1, 3, 6]), restart=True, **_grid(rng, 500, 12000))
    if kind == "outputs":
        return _case(refine=rng.choice([1, 2, 3]), n_steps=rng.randint(24, 168), outputs=True,
                     gauges=rng.randint(1, 5), weather=weather, **_grid(rng, 300, 7000))
    if kind == "plain":
        return _case(n_steps=rng.randint(12, 48), mode=N.RUN_PLAIN, gauges=rng.randint(1, 20),
                     weather=weather, field="last", **_grid(rng, 3000, 500000))
    if kind == "celerity":
        return _case(n_steps=rng.randint(48, 240), celerity=rng.uniform(0.3, 2.5),
                     gauges=rng.randint(1, 5), weather=weather, restart=True,
                     **_grid(rng, 400, 33000))
    return _case(kind="request", n_steps=rng.randint(30, 200), timestep=24,
                 n_sets=_logint(rng, 1, 24), weather=weather, **_grid(rng, 1000, 20000))


# ---------------------------------------------------------------------------
# inputs

@functools.lru_cache(maxsize=4)
def _terrain(nrows, ncols, refine, nh, gauges):
    """The basin of a size: terrain, network, soils; gauges at the outlet and
    at the nodes with the largest upstream areas of evenly spread ranks."""
    hd = np.array(HORIZONS[nh])
    dom = synth.make_domain(nrows, ncols, seed=nrows * 7919 + ncols, horizon_depth=hd)
    n = dom.n_cells
    down = np.full(n, -1, np.int64)
    down[dom.fromN - 1] = dom.toN - 1
    acc = np.ones(n)
    for i in np.argsort(-dom.depth, kind="stable")[: n if gauges > 1 else 0]:
        if down[i] >= 0:
            acc[down[i]] += acc[i]
    if gauges > 1:
        ranked = np.argsort(-acc, kind="stable")
        pick = ranked[np.unique(np.geomspace(1, n // 4, gauges).astype(int)) - 1] + 1
        dom.gauge_nodes = np.concatenate([dom.gauge_nodes, np.setdiff1d(pick, dom.gauge_nodes)]).astype(np.int32)
    return dom if refine == 1 else synth.refine_domain(dom, refine, nrows * 31 + ncols)


def _domains(case):
    if not case["basins"]:
        return [dataclasses.replace(_terrain(case["nrows"], case["ncols"], case["refine"], case["nh"],
                                             case["gauges"]))]
    b = case["basins"]
    sizes = np.geomspace(case["lo"], case["hi"], b)[np.argsort(np.sin(np.arange(b) * 12.9898))]
    grids = [(max(2, int(math.sqrt(n) * (0.75 + 0.5 * (k % 5) / 4))), n) for k, n in enumerate(sizes)]
    return [dataclasses.replace(_packed_terrain(nr, max(2, int(n / nr)), case["nh"])) for nr, n in grids]


@functools.lru_cache(maxsize=64)
def _packed_terrain(nrows, ncols, nh):
    return _terrain.__wrapped__(nrows, ncols, 1, nh, 1)


def _days(case):
    return calendar.n_forcing_days_needed(case["n_steps"])


def _smooth(gen, nd, nr, nc, extent):
    """(nd, nr * nc) standard-normal fields, coherent over `extent` cells,
    column-major in the cells."""
    cr, cc = max(2, nr // extent + 2), max(2, nc // extent + 2)
    z = torch.randn(nd, 1, cc, cr, generator=gen, device="cuda", dtype=torch.float64)
    f = torch.nn.functional.interpolate(z, size=(nc, nr), mode="bilinear", align_corners=True)
    return f.reshape(nd, nc * nr)


def _forcing(dom, case, nd, seed):
    """Daily forcing of one basin, {name: (days, cells)} on the host: rain on
    two days in five, annual and day-to-day temperature."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, nr, nc = dom.n_cells, dom.nrows, dom.ncols
    noise = lambda: torch.randn(nd, n, generator=gen, device="cuda", dtype=torch.float64)
    unit = lambda: torch.rand(nd, n, generator=gen, device="cuda", dtype=torch.float64)
    day = torch.arange(nd, device="cuda", dtype=torch.float64)[:, None]
    season = lambda d0: torch.sin(2.0 * math.pi * (day - d0) / 365.0)
    if case["weather"] == "fronts":
        # each day a passing front: its rain and its air mass vary over some
        # 100 cells, amounts and temperatures a little from cell to cell
        front = _smooth(gen, nd, nr, nc, 100)
        wet = front + 0.7 * torch.randn(nd, 1, generator=gen, device="cuda", dtype=torch.float64) > 0.3
        amount = 3.0 * torch.exp(0.8 * front) * torch.exp(0.3 * noise())
        tavg = 10.0 + 12.0 * season(105) + 3.0 * _smooth(gen, nd, nr, nc, 150) + 0.3 * noise()
    else:
        wet = unit() < 0.4
        amount = 4.0 * torch.exp(0.9 * noise() - 0.4)
        tavg = 10.0 + 12.0 * season(105) + 3.0 * noise()
    amount *= wet
    swing = 4.0 + 2.0 * unit()
    out = {"PRE": amount, "TAVG": tavg, "TMIN": tavg - swing, "TMAX": tavg + swing}
    if case["pet"] <= 0:
        out["PET"] = 0.2 + 2.0 * unit() + (1.5 + 1.5 * season(80))
    elif case["pet"] >= 2:
        es = 0.6108 * torch.exp(17.27 * tavg / (tavg + 237.3))
        out["NETRAD"] = 70.0 + 90.0 * season(80) + 25.0 * noise()
        out["ABSVAPPRESS"] = (0.35 + 0.6 * unit()) * 1000.0 * es
        out["WINDSPEED"] = 0.3 - 2.4 * torch.log(1.0 - unit())
    keep = {-1: ("PET",), 0: ("PET",), 1: ("TMIN", "TMAX"), 2: ("NETRAD",),
            3: ("NETRAD", "ABSVAPPRESS", "WINDSPEED")}[case["pet"]]
    return {k: out[k].cpu().numpy() for k in ("PRE", "TAVG") + keep}


def _inputs(case, seed):
    """Everything a run reads, on the host: basins with forcing, a gamma
    vector per (set, basin), meteo weights."""
    doms = _domains(case)
    nd = _days(case)
    rng = np.random.default_rng(seed)
    gam = PM.draw(rng, case["n_sets"] * len(doms)).reshape(case["n_sets"], len(doms), -1)
    for d in doms:
        d.forcing = _forcing(d, case, nd, int(rng.integers(1 << 40)))
        d.n_days = nd
    w = None
    if case["weights"]:
        w = synth.make_meteo_weights(sum(d.n_cells for d in doms), int(rng.integers(1 << 40)))
    return doms, gam, w, nd


def _cell_fields(case, doms, gam_s):
    parts = [synth.cell_params(d, g, pet_case=case["pet"]) for d, g in zip(doms, gam_s)]
    return {k: np.concatenate([p[k] for p in parts], axis=0) for k in parts[0]}


def prepare(case, seed):
    doms, gam, w, nd = _inputs(case, seed)
    if case["kind"] == "request":
        req = serve.Request(0, doms[0], gam[:, 0], case["n_steps"], case["timestep"], START)
        return {"case": case, "request": req}
    m = engine.Model(doms, n_sets=case["n_sets"], timestep=case["timestep"],
                     process_soil=case["soil"], process_pet=case["pet"], n_forcing_days=nd)
    if case["tile_height"]:
        m.set_tile_height(case["tile_height"])
    m.bind_network()
    for s in range(case["n_sets"]):
        m.set_params(_cell_fields(case, doms, gam[s]), s)
        for b in range(len(doms)):
            if case["celerity"]:
                m.set_routing_celerity(case["celerity"], s, b)
            else:
                m.set_routing_params(PM.routing_gamma(gam[s, b]), s, b)
    m.default_states()
    for name in doms[0].forcing:
        m.set_forcing(name, doms[0].forcing[name] if len(doms) == 1 else
                      np.concatenate([d.forcing[name] for d in doms], axis=1))
    if w is not None:
        m.set_meteo_weights(*w)
    for d in doms:
        d.forcing = {}
    m.sync()
    return {"case": case, "model": m, "steps": _steps(case)}


def _steps(case):
    return calendar.step_table(START, case["n_steps"], case["timestep"])


def run(state):
    c = state["case"]
    if c["kind"] == "request":
        return {"gauges": serve.run_alone(state["request"])}
    m, steps = state["model"], state["steps"]
    if c["kind"] == "steps":
        gauges, fields = [], []
        for st in steps:
            m.mhm_step(st)
            gauges.append(m.mrm_step(st))
            if c["field"] == "each":
                fields.append(m.get("TOTAL_RUNOFF"))
        out = {"gauges": np.stack(gauges)}
        if fields:
            out["total_runoff"] = np.stack(fields)
        elif c["field"] == "last":
            out["total_runoff"] = m.get("TOTAL_RUNOFF")
        return out
    if c["outputs"]:
        m.output_accumulate([k in OUTPUTS for k in range(1, 22)])
        m.qmod_accumulate()
    out = {"gauges": m.run(steps, mode=c["mode"], steps_per_launch=c["S"], block=c["block"],
                           use_graph=c["graph"], route_window=c["window"])}
    if c["outputs"]:
        for k in OUTPUTS:
            for h in range(1, (c["nh"] if k == 3 else 1) + 1):
                out[f"output_{k}_{h}"] = m.output_sum(k, h)[0]
        out["qmod"] = m.qmod_sum()[0]
    if c["field"] == "last":
        out["total_runoff"] = m.get("TOTAL_RUNOFF")
    if c["restart"]:
        for k in STATES:
            out[k] = m.get(k)
        rs = m.routing_state()
        out.update({k: rs[k] for k in ROUTING + ("C1", "C2")})
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _cells_nodes(case):
    if case["basins"]:
        n = sum(d.n_cells for d in _domains(case))
        return n, n
    nodes = case["nrows"] * case["ncols"]
    return nodes * case["refine"] ** 2, nodes


def work(case):
    """Bytes: the forcing once, every set's parameters and states in, states
    (and the routing's) out, and, where a pass hands out every step's fluxes
    (plain loop, per-step drop-in), those each step.  Operations: some 290
    floating-point operations per cell and step, 9 per node and routing."""
    n, nodes = _cells_nodes(case)
    s, t, nh = case["n_sets"], case["n_steps"], case["nh"]
    calls = t if case["kind"] == "steps" else 1  # a step's call reads and writes it all
    forcing = {-1: 3, 0: 3, 1: 4, 2: 3, 3: 5}[case["pet"]] * (t if calls > 1 else _days(case))
    states, fluxes = 5 + nh, 17 + 2 * nh
    params = 17 + 5 * nh + (1 if calls > 1 else min(12, 1 + t * case["timestep"] // 730))
    cell = 8 * n * forcing + 8 * n * s * (
        calls * (params + 2 * states) + fluxes * (t if case["mode"] == N.RUN_PLAIN else calls))
    if case["weights"]:
        cell += 3 * 8 * n * 24 * max(1, t * case["timestep"] // 730)
    if case["outputs"]:
        cell += 8 * n * (len(OUTPUTS) + nh - 1)
    route = 8 * nodes * s * 6 * calls
    loops = 1
    if case["celerity"]:
        loops = max(1, round(3600.0 * case["timestep"] / _routing_step(1000.0 / case["celerity"])))
    return {"bytes": float(cell + route), "flops": float(n * s * t * 290 + nodes * s * t * loops * 9)}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch

T_GIVEN = [60.0, 120.0, 180.0, 240.0, 300.0, 360.0, 600.0, 720.0, 900.0, 1200.0, 1800.0, 3600.0,
           7200.0, 10800.0, 14400.0, 21600.0, 28800.0, 43200.0, 86400.0]


def _routing_step(k_min):
    """The routing step [s] for the shortest travel time: the nearest of the
    steps a domain may take, or the one below if that is longer."""
    i = min(range(len(T_GIVEN)), key=lambda j: abs(T_GIVEN[j] - k_min))
    return T_GIVEN[i] if T_GIVEN[i] <= k_min * (1 + 2.3e-16) else T_GIVEN[max(0, i - 1)]


def _gpu(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


class _Rivers:
    """Muskingum routing of all basins and sets, one (step, depth) diagonal at
    a time: nodes deepest first, a node's step t one diagonal after its
    upstream nodes' step t."""

    def __init__(self, case, doms, gam):
        S, ts = case["n_sets"], float(case["timestep"])
        n = sum(d.n_nodes for d in doms)
        self.n, self.S = n, S
        c1, c2 = torch.zeros(S, n, dtype=torch.float64), torch.zeros(S, n, dtype=torch.float64)
        depth, up, own, gauges, links = [], [], np.zeros(n, bool), [], []
        self.loops, off = 1, 0
        for b, d in enumerate(doms):
            down = np.full(d.n_nodes, -1, np.int64)
            down[d.fromN - 1] = d.toN - 1
            dep, todo = np.zeros(d.n_nodes, np.int64), down.copy()
            at = np.nonzero(todo >= 0)[0]
            while at.size:
                dep[at] += 1
                todo[at] = down[todo[at]]
                at = at[todo[at] >= 0]
            depth.append(dep)
            up.append(np.stack([d.fromN - 1, d.toN - 1]) + off)
            own[off + d.fromN - 1] = True
            own[off + (d.toN[d.netPerm[-1] - 1] - 1 if d.n_links else 0)] = True
            gauges.append(d.gauge_nodes - 1 + off)
            links.append(d.fromN - 1 + off)
            for s in range(S):
                if case["celerity"]:
                    K = d.length / case["celerity"]
                    step = _routing_step(K.min())
                    self.loops = max(1, int(math.floor(3600.0 * ts / step + 0.5)))
                    x1 = step / (K + 0.5 * step)
                    x2 = 1.0 - x1 * K / step
                else:
                    p = PM.routing_gamma(gam[s, b])
                    K = p[0] + p[1] * d.length * 0.001 + p[2] * d.slope + p[3] * d.fFPimp
                    xi = np.clip(p[4] * (1.0 + d.slope / d.slope.max()), 0.005, 0.5)
                    K = np.maximum(np.minimum(K, 0.5 * ts / xi), 0.5 * ts / (1.0 - xi))
                    x1 = ts / (K * (1.0 - xi) + 0.5 * ts)
                    x2 = 1.0 - x1 * K / ts
                c1[s, off + d.fromN - 1] = torch.from_numpy(x1)
                c2[s, off + d.fromN - 1] = torch.from_numpy(x2)
            off += d.n_nodes
        depth = np.concatenate(depth)
        order = np.argsort(-depth, kind="stable")  # deepest first
        inv = np.empty(n, np.int64)
        inv[order] = np.arange(n)
        frm, to = np.concatenate(up, axis=1)
        frm, to = inv[frm], inv[to]
        o = np.argsort(to, kind="stable")
        frm, to = frm[o], to[o]
        slot = np.arange(to.size) - np.searchsorted(to, to)
        table = np.full((int(slot.max()) + 1 if to.size else 1, n), n, np.int64)
        table[slot, to] = frm
        self.dmax = int(depth.max())
        lev = depth[order]
        # first node of depth <= k, deepest first
        self.first = np.searchsorted(-lev, -np.arange(self.dmax + 2), side="left")
        self.lev = torch.from_numpy(self.dmax - lev).cuda()
        self.table = torch.from_numpy(table).cuda()
        self.width = [int((t < n).nonzero()[0].max()) + 1 if (t < n).any() else 0 for t in table]
        self.order, self.inv = torch.from_numpy(order).cuda(), torch.from_numpy(inv).cuda()
        self.c1, self.c2 = c1.cuda()[:, self.order], c2.cuda()[:, self.order]
        self.link = torch.zeros(n, dtype=torch.bool, device="cuda")
        self.link[self.inv[torch.from_numpy(np.concatenate(links)).cuda()]] = True
        self.own = torch.from_numpy(own).cuda()[self.order].double()
        self.gauge = self.inv[torch.from_numpy(np.concatenate(gauges).astype(np.int64)).cuda()]
        self.links = [torch.from_numpy(x).cuda() for x in links]

    def route(self, q):
        """q: (steps, sets, nodes) runoff in m3/s.  Gauges (steps, sets,
        gauges), the sum of Qmod over the steps, and the states at the end."""
        T, S, n = q.shape
        L = self.loops
        R = T * L
        q = q[:, :, self.order]
        acc = torch.zeros(S, n, dtype=torch.float64, device="cuda")
        last = torch.zeros_like(acc)
        qtin, qtr = torch.zeros_like(acc), torch.zeros_like(acc)
        pub = torch.zeros(2, S, n + 1, dtype=torch.float64, device="cuda")
        series = torch.zeros(R, S, n if self.gauge.numel() * 8 > n and n < 5000 else self.gauge.numel(),
                             dtype=torch.float64, device="cuda")
        whole = series.shape[2] == n
        flat = q.reshape(T, S * n)
        where = {}
        for g in range(self.gauge.numel()):
            where.setdefault(int(self.dmax - self.lev[self.gauge[g]]), []).append(g)
        where = [(k, torch.tensor(v, device="cuda"), self.gauge[torch.tensor(v, device="cuda")]) for k, v in where.items()]
        col = torch.arange(S, device="cuda")[:, None] * n
        for d in range(R + self.dmax):
            # nodes at depth k handle step d - (dmax - k) of 0 .. R - 1
            k_hi, k_lo = min(self.dmax, self.dmax - d + R - 1), max(0, self.dmax - d)
            a, b = int(self.first[k_hi]), int(self.first[k_lo - 1]) if k_lo > 0 else n
            t = d - self.lev[a:b]
            qo = flat.view(-1)[(torch.div(t, L, rounding_mode="floor") * (S * n) if L > 1 else t * (S * n))
                               + col + torch.arange(a, b, device="cuda")]
            prev, now = pub[(d + 1) & 1], pub[d & 1]
            s = torch.zeros(S, b - a, dtype=torch.float64, device="cuda")
            for j, w in enumerate(self.width):
                e = min(b, w)
                if e > a:
                    s[:, : e - a] += prev[:, self.table[j, a:e]]
            s += qo * self.own[a:b]
            x = qtr[:, a:b] + self.c1[:, a:b] * (qtin[:, a:b] - qtr[:, a:b]) + self.c2[:, a:b] * (s - qtin[:, a:b])
            qtr[:, a:b] = x
            now[:, a:b] = x
            qtin[:, a:b] = s
            if L == 1:
                acc[:, a:b] += s
            else:
                last[:, a:b] += s * (t >= R - L)
            for k, gs, nodes in where:
                tg = d - (self.dmax - k)
                if 0 <= tg < R and not whole:
                    series[tg][:, gs] = qtin[:, nodes]
                elif 0 <= tg < R:
                    series[tg][:, nodes] = qtin[:, nodes]
        g = series if not whole else series[:, :, self.gauge]
        g = g.reshape(T, L, S, -1).mean(dim=1) if L > 1 else g
        back = lambda v: v[0][self.inv].cpu().numpy()
        zero = torch.where(self.link, qtr, torch.zeros_like(qtr))
        state = {"qOUT": back(q[-1]), "qTIN": back(qtin), "qTR": back(zero),
                 "Qmod": back(last / L if L > 1 else qtin)}
        for name, v in (("C1", self.c1), ("C2", self.c2)):
            w = v[0][self.inv]
            state[name] = torch.cat([w[x] for x in self.links]).cpu().numpy()
        return g, back(acc), state


def _pet(case, p, f, day, month, doy):
    """The day's PET before disaggregation, (sets, cells)."""
    pet = case["pet"]
    if pet == -1:
        return p["PETLAICOR"][..., month] * f["PET"][day]
    if pet == 0:
        return p["FASP"] * f["PET"][day]
    tavg = f["TAVG"][day]
    if pet == 1:
        dT = f["TMAX"][day] - f["TMIN"][day]
        dr = 1.0 + 0.0330 * math.cos(2.0 * math.pi * doy / 365.0)
        dl = 0.4090 * math.sin(2.0 * math.pi * doy / 365.0 - 1.3900)
        lat = p["LATITUDE"] * (math.pi / 180.0)
        om = torch.acos(torch.clamp(-torch.tan(lat) * math.tan(dl), -1.0, 1.0))
        ra = 86400.0 / math.pi / 2.45e06 * 1367.0 * dr * (
            om * torch.sin(lat) * math.sin(dl) + torch.cos(lat) * math.cos(dl) * torch.sin(om))
        v = p["HARSAMCOEFF"] * ra * (tavg + 17.8) * torch.sqrt(torch.clamp(dT, min=0.0))
        return p["FASP"] * torch.where((dT <= 0.0) | (tavg <= -17.8), torch.zeros_like(v), v)
    rn = torch.clamp(f["NETRAD"][day], min=0.0)
    es = 0.6108 * torch.exp(17.27 * tavg / (tavg + 237.3))
    slope = 4098.0 * es / (tavg + 237.3) ** 2
    if pet == 2:
        return p["PRIETAYALPHA"][..., month] * slope / (0.0646 + slope) * (rn * 86400.0 / 2.45e06)
    ra = p["AERORESIST"][..., month] / f["WINDSPEED"][day]
    return 86400.0 / 2.45e06 * (slope * rn + 1.225 * 1005.0 * (es - f["ABSVAPPRESS"][day] / 1000.0) / ra) / (
        slope + 0.0646 * (1.0 + p["SURFRESIST"][..., month] / ra))


def _step(case, p, x, pet, prec, temp, month, evap):
    """One step of the cell processes on the states x (changed in place)."""
    nh, eps = case["nh"], 2.220446049250313e-16
    c2 = case["timestep"] / 24.0
    zero = torch.zeros((), dtype=torch.float64, device="cuda")
    # canopy
    cap = p["MAXINTER"][..., month]
    aux = x["INTER"] + prec
    thr = torch.clamp(aux - cap, min=0.0)
    inter = torch.minimum(aux, cap)
    ecan = torch.where(cap > eps, pet * (inter / cap) ** (2.0 / 3.0), zero)
    ecan = torch.minimum(torch.clamp(ecan, min=0.0), inter)
    x["INTER"] = inter - ecan
    # snow
    warm = temp > p["TEMP_THRESH"]
    snow = torch.where(warm, zero, thr)
    dmax, dnp = p["DEGDAY_MAX"] * c2, p["DEGDAY_NOPRE"] * c2
    ddf = torch.where(prec <= (dmax - dnp) / p["DEGDAY_INC"], dnp + p["DEGDAY_INC"] * prec, dmax)
    melt = torch.where(warm, torch.minimum(ddf * (temp - p["TEMP_THRESH"]), x["SNOWPACK"]), zero)
    x["SNOWPACK"] = x["SNOWPACK"] + snow - melt
    peff = melt + (thr - snow)
    # sealed areas
    fs = p["FSEALED"]
    tmp = x["SEALSTW"] + peff
    on = fs > 0.0
    rseal = torch.where(on, torch.clamp(tmp - p["SEALED_THRESH"], min=0.0), zero)
    st = torch.minimum(tmp, p["SEALED_THRESH"])
    es = torch.clamp((pet / evap - ecan) * (st / p["SEALED_THRESH"]), min=0.0)
    es = torch.where(p["SEALED_THRESH"] > eps, torch.minimum(es, st), st)
    aseal = torch.where(on, es, zero)
    x["SEALSTW"] = torch.where(on, st - es, x["SEALSTW"])
    # soil
    pin, used, infil, aet = peff, 0.0, [], []
    sms = []
    for h in range(nh):
        sm, sat = x["SOILMOIST"][h], p["SOILMOIST_SAT"][..., h]
        frac = torch.where(sm > eps, (torch.clamp(sm, min=0.0) / sat) ** p["SOILMOIST_EXP"][..., h], zero)
        tmp = pin * (1.0 - frac)
        full, over = sm > sat, sm + tmp > sat
        inf = torch.where(full, pin, torch.where(over, pin + (sm - sat), pin - tmp))
        sm = torch.where(full, sm, torch.where(over, sat, sm + tmp))
        wp, fr = p["WILTINGPOINT"][..., h], p["FROOTS"][..., h]
        if case["soil"] in (2, 3):
            th = torch.clamp((sm - wp) / (sat - wp), 0.0, 1.0)
            f = torch.where(th >= p["JARVIS_C1"], fr, fr * (th / p["JARVIS_C1"]))
        else:
            fc = p["SOILMOIST_FC"][..., h]
            f = torch.where(sm >= fc, fr, torch.where(sm > wp, fr * (sm - wp) / (fc - wp), zero))
        a = torch.clamp((pet - ecan - used) * f, min=0.0)
        dry = ~(sm > a)
        a = torch.where(dry, sm - eps, a)
        sm = torch.where(dry, zero + eps, sm - a)
        sms.append(torch.clamp(sm, min=eps))
        used = used + torch.clamp(a, min=0.0)
        infil.append(inf)
        aet.append(a)
        pin = inf
    x["SOILMOIST"] = sms
    # unsaturated and saturated zone
    un = x["UNSATSTW"] + pin
    fast = torch.where(un > p["UNSAT_THRESH"], torch.minimum(un - eps, c2 / p["KFASTFLOW"] * (un - p["UNSAT_THRESH"])), zero)
    un = un - fast
    slow = torch.where(un > eps, torch.minimum(un - eps, c2 / p["KSLOWFLOW"] * torch.clamp(un, min=0.0) ** (1.0 + p["ALPHA"])), zero)
    un = un - slow
    perc = c2 / p["KPERCO"] * un
    down = torch.minimum(perc, un)
    x["UNSATSTW"] = un - down
    satw = torch.clamp(x["SATSTW"] + down * p["KARSTLOSS"], min=0.0)
    base = c2 / p["KBASEFLOW"] * satw
    x["SATSTW"] = satw - base
    fns = 1.0 - fs
    total = (base + slow + fast) * fns + rseal * fs
    if not case["outputs"]:
        return total, None
    hsum = lambda v: functools.reduce(torch.add, v)
    out = {1: [x["INTER"]], 2: [x["SNOWPACK"]], 3: sms,
           5: [hsum(sms) / p["SOILMOIST_SAT"].sum(dim=-1)], 7: [x["UNSATSTW"]], 8: [x["SATSTW"]],
           9: [pet], 10: [hsum(aet) * fns + ecan + aseal * fs], 11: [total], 15: [base * fns],
           16: [perc * fns], 20: [peff]}
    return total, out


def exact(case, seed):
    doms, gam, w, nd = _inputs(case, seed)
    S, n = case["n_sets"], sum(d.n_cells for d in doms)
    fields = [_cell_fields(case, doms, gam[s]) for s in range(S)]
    p = {k: torch.stack([_gpu(f[k]) for f in fields]) for k in fields[0]}
    del fields
    f = {k: _gpu(np.concatenate([d.forcing[k] for d in doms], axis=1)) for k in doms[0].forcing}
    if w is not None:
        w = [_gpu(v) for v in w]
    hd, full = HORIZONS[case["nh"]], lambda v: torch.full((S, n), v, dtype=torch.float64, device="cuda")
    top = [0.0] + hd[:-1]
    x = {"INTER": full(0.0), "SNOWPACK": full(15.0), "SEALSTW": full(0.0), "UNSATSTW": full(10.0),
         "SATSTW": full(75.0), "SOILMOIST": [full(0.0) for _ in hd]}
    ts, area = case["timestep"], _gpu(np.concatenate([d.area_km2 for d in doms]))
    nT = 24 // ts
    node, off = [], 0
    for d in doms:
        node.append((np.arange(d.n_cells) if d.l1_l11 is None else d.l1_l11 - 1) + off)
        off += d.n_nodes
    node = None if off == n else torch.from_numpy(np.concatenate(node)).cuda()
    q = torch.zeros(case["n_steps"], S, off, dtype=torch.float64, device="cuda")
    sums, tot_fields, key = {}, [], None
    for k in range(case["n_steps"]):
        now = START + dt.timedelta(hours=k * ts)
        m, day = now.month - 1, k // 24
        doy = now.timetuple().tm_yday
        if (day, doy, m) != key:
            pd = _pet(case, p, f, day, m, doy)
            key = (day, doy, m)
        pet, prec, temp = pd, f["PRE"][day], f["TAVG"][day]
        if w is not None:
            prec, temp, pet = prec * w[0][:, m, now.hour], (temp + 273.15) * w[1][:, m, now.hour] - 273.15, pet * w[2][:, m, now.hour]
        elif nT > 1:
            light = 6 < now.hour <= 18
            pick = lambda v, day_v: day_v if light else v
            prec = 2.0 * prec * pick(synth.FNIGHT_PREC[m], 1.0 - synth.FNIGHT_PREC[m]) / nT
            pet = 2.0 * pet * pick(synth.FNIGHT_PET[m], 1.0 - synth.FNIGHT_PET[m]) / nT
            temp = temp + pick(synth.FNIGHT_TEMP[m], -synth.FNIGHT_TEMP[m])
        if k == 0:
            x["SOILMOIST"] = [0.5 * p["SOILMOIST_FC"][..., h] for h in range(case["nh"])]
        total, out = _step(case, p, x, pet, prec, temp, m, float(synth.EVAP_COEFF[m]))
        r = total * area
        if node is not None:
            r = torch.zeros(S, off, dtype=torch.float64, device="cuda").index_add_(1, node, r)
        q[k] = r * 1000.0 / (3600.0 * ts)
        if out:
            for o, v in out.items():
                sums[o] = [a + b for a, b in zip(sums[o], v)] if o in sums else [1.0 * a for a in v]
        if case["field"] == "each" or case["field"] == "last" and k == case["n_steps"] - 1:
            tot_fields.append(total[0].cpu().numpy())
    gauges, qmod, state = _Rivers(case, doms, gam).route(q)
    res = {"gauges": gauges.cpu().numpy()}
    if tot_fields:
        res["total_runoff"] = np.stack(tot_fields) if case["field"] == "each" else tot_fields[0]
    if case["outputs"]:
        for o in OUTPUTS:
            for h, v in enumerate(sums[o]):
                res[f"output_{o}_{h + 1}"] = v.expand(S, n)[0].cpu().numpy()
        res["qmod"] = qmod
    if case["restart"]:
        for k in STATES:
            v = x[k]
            res[k] = v[0].cpu().numpy() if k != "SOILMOIST" else (
                v[0][0].cpu().numpy() if case["nh"] == 1 else torch.stack([h[0] for h in v], dim=1).cpu().numpy())
        res.update(state)
    return res
