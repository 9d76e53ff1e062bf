"""The calls whose speed counts, through the package's public entry points.

Four kinds of call, as programs make them:

  simulate   GWModel.simulate: one cell, every snapshot copied to the host
  reduced    GWModel.simulate_reduced: one cell, snapshots in the reduced encoding
  ensemble   a Batch of independent cells made, advanced and read out (globals,
             observables, a trace of V, Cai, ICaL and open RyRs), then closed: parameter
             studies, seed ensembles, clamp families
  session    a Batch kept open and advanced a little at a time, its globals and
             post-hoc currents read between the advances (a closed loop on V), the whole
             state of every cell read at the end

Sizes: cells of 64 to 12,500 CRUs (the model's default 1,250 and the full cell among
them), 1 to 1,024 cells, both precisions, all engines, the default launch shape and the
shapes the autotuner picks on large batches. dt is 1e-3 ms throughout. Cells start either
at rest under a stimulus or early in an action potential (a depolarised membrane, activated
INa, channels at rest), where L-type channels open and release starts.
"""
import functools
import importlib
import math

import numpy as np

gwm = importlib.import_module("gw-model_amd")
capi = gwm.capi

DT = 1e-3                       # ms
TRACE_EVERY = 10                # steps between the rows of an ensemble's trace
FLOPS = 331                     # FP64 operations of the SSA iteration that closes a step, one per CRU and step
STATE = {"fp64": 136, "fp32_local": 120}   # bytes of one CRU's state
RECORD = {"simulate": 184, "reduced": 40}  # bytes of one CRU's snapshot
ON_CHIP = 160 << 20             # bytes of registers and LDS of the whole GPU, rounded up
ENGINES = ("xoshiro256**", "xoshiro256++", "xoshiro256+", "xoroshiro128**", "xoroshiro128++", "xoroshiro128+")


def _single(name, kind, crus, steps, every, precision="fp64", engine="xoshiro256++", start="rest"):
    return {"name": name, "kind": kind, "crus": crus, "steps": steps, "record_every": every, "precision": precision,
            "engine": engine, "start": start}


def _batch(name, kind, cells, crus, crus_max, steps, precision, launch="", protocol="pace", engine="xoshiro256**"):
    return {"name": name, "kind": kind, "cells": cells, "crus": crus, "crus_max": crus_max, "steps": steps,
            "precision": precision, "launch": launch, "protocol": protocol, "engine": engine}


def listed():
    return [
        # the smallest call: a toy cell, for a test or a notebook; latency alone counts
        _single("simulate 64", "simulate", 64, 400, 100),
        # the model's default cell with the default engine, a snapshot each 0.1 ms
        _single("simulate 1250", "simulate", 1250, 1000, 100, start="upstroke"),
        # the full cell in FP64, snapshots reduced for storage
        _single("reduced 12500", "reduced", 12500, 1000, 100, start="upstroke"),
        # the full cell in the FP32-local form, a few full snapshots
        _single("simulate 12500 fp32", "simulate", 12500, 1000, 250, "fp32_local", start="upstroke"),
        # a closed loop on a handful of small cells of odd size
        _batch("session 4x1999", "session", 4, 1999, 1999, 400, "fp64"),
        # a voltage-clamp family: 9 potentials x 4 seeds of the full cell, default launch shape
        _batch("clamp 36x12500 fp64", "ensemble", 36, 12500, 12500, 500, "fp64", protocol="clamp"),
        # a seed ensemble of the full cell in the FP32-local form, at its tuned shape
        _batch("seeds 64x12500 fp32", "ensemble", 64, 12500, 12500, 500, "fp32_local", "1x64x4"),
        # a population of uneven cells with scaled conductances, in both forms
        _batch("uneven 256 fp64", "ensemble", 256, 2000, 12500, 250, "fp64", "4x64"),
        _batch("uneven 256 fp32", "ensemble", 256, 2000, 12500, 400, "fp32_local", "1x64x4"),
        # the largest population of full cells, in both forms
        _batch("large 1024x12500 fp64", "ensemble", 1024, 12500, 12500, 150, "fp64", "4x64"),
        _batch("large 1024x12500 fp32", "ensemble", 1024, 12500, 12500, 400, "fp32_local", "1x64x4"),
    ]


def draw(rng):
    """One more case of the ranges above: sizes spread over their logarithm, odd ones among them."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    precision = rng.choice(("fp64", "fp32_local"))
    kind = rng.choice(("simulate", "reduced", "session", "ensemble", "ensemble", "ensemble"))
    if kind in ("simulate", "reduced"):
        steps = spread(200, 1000)
        c = _single("", kind, spread(64, 12500), steps, max(1, steps // rng.randint(2, 10)), precision,
                    rng.choice(ENGINES), rng.choice(("rest", "upstroke")))
    else:
        cells = spread(1, 16) if kind == "session" else spread(2, 1024)
        lo = spread(64, 12500)
        hi = lo if rng.random() < 0.5 else spread(lo, 12500)
        launch = rng.choice(("", "4x64") if precision == "fp64" else ("", "1x64", "1x64x4"))
        most = 4_000_000_000 if launch.startswith("1") else 1_500_000_000   # CRU-steps, below the largest listed cases'
        steps = max(100, min(spread(200, 500), most // (cells * (lo + hi) // 2)))
        c = _batch("", kind, cells, lo, hi, steps, precision, launch, rng.choice(("pace", "pace", "clamp")),
                   "xoshiro256**" if launch else rng.choice(ENGINES))
    del c["name"]
    return c


@functools.lru_cache(maxsize=None)
def _context():
    return capi.Context(0)


def _upstroke(rng):
    """Globals early in an action potential: depolarised, INa activated and inactivating, the rest at rest."""
    return {"V": float(rng.uniform(0.0, 30.0)), "m": float(rng.uniform(0.98, 1.0)), "h": float(rng.uniform(1e-4, 1e-2)),
            "j": float(rng.uniform(0.01, 0.5)), "Cai": float(rng.uniform(1.4e-4, 2.5e-4)),
            "CaNSR": float(rng.uniform(0.85, 0.95))}


def _cells(case, rng):
    """Cell descriptors: CRU counts uniform in the case's range, own seeds, six conductances scaled
    log-uniform in [0.5, 2], paced at 2 Hz, or clamped from -80 mV to one of nine potentials."""
    out = []
    for k in range(case["cells"]):
        p = capi.Params.default()
        if case["protocol"] == "clamp":
            protocol = {"kind": capi.PROTO_CLAMP, "hold": -80.0, "step": -40.0 + 10.0 * (k % 9), "t_on": 0.0, "t_off": 200.0}
        else:
            for field in ("PCaL", "GKr", "GKs", "GK1", "GKv43", "kNaCa"):
                setattr(p, field, getattr(p, field) * float(np.exp(rng.uniform(np.log(0.5), np.log(2.0)))))
            protocol = {"kind": capi.PROTO_PACE, "period": 500.0, "duration": 1.0, "amplitude": 100.0, "start": 0.0}
        n = int(rng.integers(case["crus"], case["crus_max"] + 1))
        out.append(capi.make_cell(n, int(rng.integers(1 << 40)), p, protocol))
    return out


def _open(case, cells, globals_):
    precision = capi.PREC_FP64 if case["precision"] == "fp64" else capi.PREC_FP32_LOCAL
    b = capi.Batch(_context(), cells, precision=precision, prng=capi.PRNG_NAMES.index(case["engine"]), dt=DT,
                   globals_=globals_)
    b.set_mode(frozen=False, digest=False)
    if case["launch"]:
        b.set_launch(*(int(x) for x in (case["launch"] + "x1").split("x")[:3]))
    return b


def prepare(case, seed):
    rng = np.random.default_rng([seed, 2024])
    if case["kind"] in ("simulate", "reduced"):
        n = case["crus"]
        cru_seed, run_seed = (int(x) for x in rng.integers(1 << 40, size=2))
        amplitude = float(rng.uniform(60.0, 140.0))
        g = gwm.gw.GWGlobalState()
        if case["start"] == "upstroke":
            for field, v in _upstroke(rng).items():
                setattr(g, field, v)
        crus = gwm.gw.rest_state(n, cru_seed, case["engine"])
        state = {k: getattr(g, k) for k in ("V", "Nai", "Ki", "Cai", "CaNSR", "CaLTRPN", "CaHTRPN", "m", "h", "j", "xKs",
                                            "XKr", "XKv14", "XKv43")}
        state.update({k: getattr(crus, k) for k in ("CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR", "ClCh")})
        model = gwm.GWModel(state, gwm.GWParameters(NCaRU_sim=n), lambda t: amplitude if t % 1000.0 < 1.0 else 0.0)
        return {"case": case, "model": model, "seed": run_seed}
    g = capi.default_globals()
    for field, v in _upstroke(rng).items():
        setattr(g, field, v)
    state = {"case": case, "cells": _cells(case, rng), "globals": g}
    if case["kind"] == "session":
        state["batch"] = _open(case, state["cells"], g)
        state["batch"].step(500)
    return state


def _globals(b):
    return np.stack([g.as_array() for g in b.get_globals()])


def _observables(b):
    return np.array([list(o.values()) for o in b.obs()])


def run(state):
    case = state["case"]
    if case["kind"] == "simulate":
        s = state["model"].simulate(DT, case["steps"], case["record_every"], PRNG=case["engine"], seed=state["seed"],
                                    precision=case["precision"])
        return {k: getattr(s, k) for k in ("t", "V", "Nai", "Ki", "Cai", "CaNSR", "CaLTRPN", "CaHTRPN", "m", "h", "j", "xKs",
                                           "XKr", "XKv14", "XKv43", "CaSS", "CaJSR", "LCC", "LCC_inactivation", "RyR",
                                           "ClCh")}
    if case["kind"] == "reduced":
        return state["model"].simulate_reduced(DT, case["steps"], case["record_every"], PRNG=case["engine"],
                                               seed=state["seed"], precision=case["precision"])
    if case["kind"] == "ensemble":
        b = _open(case, state["cells"], state["globals"])
        b.enable_trace(TRACE_EVERY, case["steps"] // TRACE_EVERY)
        b.step(case["steps"])
        out = {"globals": _globals(b), "observables": _observables(b), "trace": b.get_trace(), "time": b.time()[0]}
        b.close()
        return out
    b = state["batch"]
    loop = []
    for k in range(4):
        b.step(case["steps"] // 4)
        ical, ito2 = b.currents()
        loop.append({"globals": _globals(b), "ICaL": ical, "Ito2": ito2})
    crus = [b.get_cru_state(c) for c in range(case["cells"])]
    return {"loop": loop, "observables": _observables(b),
            "crus": {k: np.concatenate([c[k] for c in crus]) for k in crus[0]}}


def work(case):
    """One SSA iteration per CRU and step. A step needs the flux sums of the last step but one, over every
    CRU of its cell, so a state larger than the chip crosses memory once each two steps, read and written."""
    steps, state = case["steps"], STATE[case["precision"]]
    if case["kind"] in RECORD:
        n = case["crus"]
        records = -(-steps // case["record_every"])
        return {"bytes": 2 * n * state + records * n * RECORD[case["kind"]], "flops": FLOPS * n * steps}
    n = case["cells"] * (case["crus"] + case["crus_max"]) / 2
    size = n * state
    passes = -(-steps // 2) if size > ON_CHIP else 1
    read_out = n * 216 if case["kind"] == "session" else case["cells"] * 8 * (52 + 4 * (steps // TRACE_EVERY))
    return {"bytes": 2 * size * passes + read_out, "flops": FLOPS * n * steps}


def exact(case, seed):
    """The clock alone: every other output is a path of a seeded random process, which no formula gives in
    64 bits (in FP64 they are the same bits on every run; channel counts are whole numbers in both forms)."""
    t = np.cumsum(np.full(case["steps"], DT))
    if case["kind"] in RECORD:
        return {"t": t[:: case["record_every"]]}
    return {"time": float(t[-1])} if case["kind"] == "ensemble" else None
