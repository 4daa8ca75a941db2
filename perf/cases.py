"""The workloads this framework is timed on: what its users have it do, through its public entry points.

A case is a dict of plain values. `listed()` names the fixed ones, `draw(rng)` makes more of the same ranges, `prepare`
builds what a program holds before the call (inputs from the seed alone), `run` is one pass, `work` the bytes and
operations of a pass, `exact` the floating-point outputs in 64 bits.

Five kinds of pass, each starting from the same start states so that a pass can be repeated:

  step      the decision loop of a policy that sees every state: the batch reset, then one launch per decision
  run       controls known ahead (replays, scripted opponents): all decisions in one launch, static or queued
  host      a policy on the host: states uploaded, then per decision controls up, step, result words and states down
  regroup   the learned cost model's ordering of a batch: features, prediction, order, states gathered
  gradients one training batch of the cost model: row losses and the parameter gradient
"""
import concurrent.futures
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rocketsim-cuda_amd"))
import rsim  # noqa: E402
import rsim.cost as cost  # noqa: E402
from rsim import layout  # noqa: E402

SCENARIOS = {"kickoff": rsim.SCEN_KICKOFF, "open": rsim.SCEN_OPEN, "pinch": rsim.SCEN_PINCH, "headon": rsim.SCEN_HEADON,
             "goalframe": rsim.SCEN_GOALFRAME, "contact": rsim.SCEN_CONTACT, "mixed": rsim.SCEN_MIXED,
             "open_contact": rsim.SCEN_OPEN_CONTACT}


def _step(n, scenario, worlds=1, decisions=4, trace=False, **name):
    return dict(name, kind="step", n=n, scenario=scenario, worlds=worlds, decisions=decisions, trace=trace)


def _run(n, scenario, worlds=1, decisions=25, queued=False, **name):
    return dict(name, kind="run", n=n, scenario=scenario, worlds=worlds, decisions=decisions, queued=queued)


def listed():
    return [
        # the smallest batch anyone steps: a debugging session or one evaluation match on each lane of a wave
        _step(64, "mixed", name="step_64"),
        # the first thing a new user runs: every arena at a kickoff
        _step(1024, "kickoff", name="step_kickoff_1024"),
        # an evaluation pool of odd size, half of it in contact
        _step(5003, "open_contact", name="step_ragged_5003"),
        # open play over the seven hitbox presets, each arena in its own pairing's world
        _step(16384, "open", worlds=7, name="step_open_16384"),
        # the headline batch: contact-heavy training, one launch per decision
        _step(65536, "contact", name="step_contact_65536"),
        # every tick's state kept, for offline analysis of goal-mouth play
        _step(3000, "goalframe", decisions=1, trace=True, name="trace_3000"),
        # the headline batch with the controls known ahead: 25 decisions in one launch
        _run(65536, "contact", name="run_contact_65536"),
        # the largest batch: a mix over presets and mutators, on the block queue
        _run(131072, "mixed", worlds=28, decisions=10, queued=True, name="queue_mixed_131072"),
        # a scripted batch of middling size
        _run(4096, "open_contact", decisions=8, name="run_4096"),
        # a policy on the host, which reads every state back
        dict(name="host_2048", kind="host", n=2048, scenario="open_contact", decisions=2),
        # the cost model orders the headline batch
        dict(name="regroup_65536", kind="regroup", n=65536, scenario="open_contact"),
        # one training batch of the cost model
        dict(name="gradients_4096", kind="gradients", batch=4096),
    ]


def _size(rng, lo, hi):
    """Log-uniform over lo..hi, odd sizes as likely as even ones."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "run", "run", "host", "regroup", "gradients"])
    scenario = rng.choice(sorted(SCENARIOS))
    if kind == "step":
        trace = rng.random() < 0.2
        n = _size(rng, 1, 4096 if trace else 65536)
        return _step(n, scenario, worlds=rng.choice([1, 1, 7]), decisions=rng.randint(1, 1 if trace else 4), trace=trace)
    if kind == "run":
        n = _size(rng, 64, 131072)
        most = max(2, min(25, 1200000 // n))
        return _run(n, scenario, worlds=rng.choice([1, 1, 7, 28]), decisions=rng.randint(2, most), queued=rng.random() < 0.5)
    if kind == "host":
        return dict(kind="host", n=_size(rng, 1, 4096), scenario=scenario, decisions=rng.randint(1, 3))
    if kind == "regroup":
        return dict(kind="regroup", n=_size(rng, 64, 131072), scenario=scenario)
    return dict(kind="gradients", batch=_size(rng, 64, 16384))


# ---- inputs -----------------------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _device():
    return rsim.SimDevice(0)


@functools.lru_cache(maxsize=None)
def _worlds(count):
    """The world table: the seven hitbox presets in turn, with Soccar's mutators first and drawn ones after."""
    rng = np.random.default_rng(7)
    out = []
    for i in range(count):
        p = i % rsim.NUM_PRESETS
        mut = () if i < rsim.NUM_PRESETS else (float(rng.uniform(-800, -500)), float(rng.uniform(0.8, 1.2)),
                                               float(rng.uniform(91.25, 100)))
        out.append(rsim.build_world(p, p, *mut))
    return np.stack(out)


def _variant(case, seed):
    count = case.get("worlds", 1)
    return None if count == 1 else np.random.default_rng(seed).integers(0, count, case["n"]).astype(np.uint32)


def _start_states(case, seed):
    """The batch's start states on the host: sampled in chunks by a few threads (arena i depends only on the seed and i)."""
    n, scen = case["n"], SCENARIOS[case["scenario"]]
    worlds, variant = _worlds(case.get("worlds", 1)), _variant(case, seed)
    out = np.empty((n, rsim.ARENA_WORDS), np.uint32)

    def fill(lo):
        hi = min(n, lo + 4096)
        if variant is None:
            out[lo:hi] = rsim.sample_arenas(worlds[0], scen, seed, hi - lo, first=lo)
        else:
            out[lo:hi] = rsim.sample_arenas_in(worlds, variant[lo:hi], scen, seed, first=lo)

    with concurrent.futures.ThreadPoolExecutor(8) as pool:
        list(pool.map(fill, range(0, n, 4096)))
    return out


def _controls(case, seed):
    return np.concatenate([rsim.sample_controls(seed + 1, d, case["n"]) for d in range(case["decisions"])])


def _train_batch(case, seed):
    """Normalised features, log-cost targets and contact flags as the labelling pass yields them."""
    rng, b = np.random.default_rng(seed), case["batch"]
    feat = np.clip(rng.standard_normal((b, cost.FEATURES)), -4, 4).astype(np.float32)
    return feat, rng.standard_normal(b).astype(np.float32), (rng.random(b) < 0.4).astype(np.float32)


class _Memory:
    """A device buffer of the framework as the array interface torch reads (no copy; keeps the buffer)."""

    def __init__(self, buf, words, typestr, shape):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (buf.ptr, False), "version": 2}
        assert math.prod(shape) == words


def _tensor(buf, typestr="<i4", shape=None, words=None):
    words = words or (rsim.aosoa_words(buf.n) if isinstance(buf, rsim.DeviceStates) else buf.n)
    return torch.as_tensor(_Memory(buf, words, typestr, shape or (words,)), device="cuda")


def prepare(case, seed):
    dev, kind = _device(), case["kind"]
    s = {"case": case, "dev": dev}
    if kind == "gradients":
        b = case["batch"]
        s["model"] = cost.CostModel(dev, seed=seed)
        s["batch"] = [dev.upload_words(np.ascontiguousarray(x).reshape(-1).view(np.uint32)) for x in _train_batch(case, seed)]
        s["scratch"], s["loss"] = dev.alloc_words(b * cost.ACT_WORDS), dev.alloc_words(b)
        s["out"] = {"loss": _tensor(s["loss"], "<f4"), "grad": _tensor(s["model"].grad, "<f4")}
        return s
    n, start = case["n"], _start_states(case, seed)
    if kind == "regroup":
        s["start"] = dev.upload_states(start)
        s["group"] = cost.Regrouper(dev, cost.CostModel(dev, seed=seed), None, dev.alloc_states(n))
        g = s["group"]
        s["out"] = {"features": _tensor(g.feat, "<f4", (n, cost.FEATURES)), "prediction": _tensor(g.pred, "<f4", (n, 2)),
                    "order": _tensor(g.where), "states": _tensor(g.cur)}
        return s
    controls, variant, decisions = _controls(case, seed), _variant(case, seed), case["decisions"]
    s["worlds"] = dev.upload_worlds(_worlds(case.get("worlds", 1)))
    s["variant"] = None if variant is None else dev.upload_words(variant)
    if kind == "host":
        s["states"], s["start"] = dev.alloc_states(n), start
        s["control"], s["result"] = dev.alloc_words(n * rsim.CONTROL_WORDS), dev.alloc_words(n)
        s["controls"] = np.ascontiguousarray(controls).reshape(decisions, n * rsim.CONTROL_WORDS)
        return s
    s["start"], s["states"] = dev.upload_states(start), dev.alloc_states(n)
    s["controls"], s["results"] = dev.upload_words(controls), dev.alloc_words(decisions * n)
    w = n * rsim.CONTROL_WORDS
    s["each"] = [(s["controls"].view(d * w, w), s["results"].view(d * n, n)) for d in range(decisions)]
    s["trace"] = dev.alloc_words(rsim.TICKS_PER_DECISION * rsim.aosoa_words(n)) if case.get("trace") else None
    s["out"] = {"states": _tensor(s["states"]), "results": _tensor(s["results"])}
    if s["trace"] is not None:
        s["out"]["trace"] = _tensor(s["trace"])
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------------------
def run(s):
    case, dev, kind = s["case"], s["dev"], s["case"]["kind"]
    if kind == "gradients":
        s["model"].gradients(*s["batch"], case["batch"], s["scratch"], s["loss"])
        return s["out"]
    if kind == "regroup":
        s["group"].reset(s["start"])
        s["group"].regroup()
        return s["out"]
    if kind == "host":
        dev.write_states(s["states"], s["start"])
        results = []
        for c in s["controls"]:
            dev.write_words(s["control"], c)
            dev.sim8(s["states"], s["worlds"], s["control"], s["result"])
            results.append(dev.read_words(s["result"]).view(np.int32))
            states = dev.download_states(s["states"])
        return {"states": states.view(np.int32), "results": results}
    dev.copy_states(s["states"], s["start"])
    if kind == "run":
        go = dev.run_queued if case["queued"] else dev.run
        go(s["states"], s["worlds"], s["controls"], s["results"], case["decisions"], variant=s["variant"])
    else:
        for c, r in s["each"]:
            if s["variant"] is None:
                dev.sim8(s["states"], s["worlds"], c, r, trace=s["trace"])
            else:
                dev.sim8_variants(s["states"], s["worlds"], s["variant"], c, r, trace=s["trace"])
    return s["out"]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
# Floating-point operations of one arena's tick, of the order of what the CPU build executes: the physics is branching
# scalar arithmetic, a few thousand operations between rays, contacts and constraint rows.
TICK_FLOPS = 6000


def work(case):
    kind = case["kind"]
    if kind == "gradients":  # three products of the two hidden layers and the head; the batch in, losses and gradient out
        b, macs = case["batch"], 48 * 64 + 64 * 64 + 64 * 2
        return {"bytes": 4 * (b * (cost.FEATURES + 2) + b + 2 * cost.PARAMS), "flops": b * (6 * macs - 2 * 48 * 64)}
    n = case["n"]
    state = 4 * rsim.ARENA_WORDS * n
    if kind == "regroup":  # states read and written in the new order, the features and the prediction in between
        return {"bytes": 2 * state + 4 * n * (cost.FEATURES + 2 + 1),
                "flops": n * 2 * (48 * 64 + 64 * 64 + 64 * 2)}
    d = case["decisions"]
    each = n * (4 * rsim.CONTROL_WORDS + 4)
    out = {"bytes": 2 * state + d * each + case.get("worlds", 1) * 4 * rsim.STATIC_WORDS,
           "flops": d * rsim.TICKS_PER_DECISION * n * TICK_FLOPS}
    if case.get("trace"):
        out["bytes"] += rsim.TICKS_PER_DECISION * n * 4 * rsim.TICK_WORDS
    if kind == "host":  # every decision's states go back to the host
        out["bytes"] += (d - 1) * state
    return out


# ---- the floating-point outputs in 64 bits ----------------------------------------------------------------------------------
def _features64(states):
    a = layout.arena_view(states)

    def vec(v):
        return np.stack([v["x"], v["y"], v["z"]], 1).astype(np.float64)

    field = np.array([4096.0, 5120.0, 2044.0])
    ball, f = a["ball"], np.zeros((len(states), 48))
    bp = vec(ball["pos"])
    f[:, 0:3], f[:, 3:6], f[:, 6:9] = bp / field, vec(ball["vel"]) / 6000, vec(ball["ang_vel"]) / 6
    cp = []
    for c in range(2):
        car, o = a["cars"][:, c], 9 + 13 * c
        p = vec(car["pos"])
        f[:, o:o + 3], f[:, o + 3:o + 6], f[:, o + 6:o + 9] = p / field, vec(car["vel"]) / 2300, vec(car["ang_vel"]) / 5.5
        f[:, o + 9], f[:, o + 10] = car["boost"] / 100.0, car["is_on_ground"] != 0
        f[:, o + 11], f[:, o + 12] = car["rot_mat"]["z_axis"]["z"], car["is_demoed"] != 0
        cp.append(p)
    f[:, 35:37], f[:, 37] = (field[:2] - np.abs(bp[:, :2])) / field[:2], (field[2] - bp[:, 2]) / field[2]
    f[:, 38:40] = (field[:2] - np.abs(cp[0][:, :2])) / field[:2]
    f[:, 40:42] = (field[:2] - np.abs(cp[1][:, :2])) / field[:2]
    for i, d in enumerate((cp[0] - cp[1], cp[0] - bp, cp[1] - bp)):
        f[:, 42 + i] = np.sqrt((d * d).sum(1)) / 1000
    f[:, 45], f[:, 46], f[:, 47] = a["n_pairs"] / 16, a["n_manifolds"] / 16, a["n_dyn_cells"] / 64
    return np.clip(f, -4, 4)


def _layers(seed):
    p = cost.init_params(seed).astype(np.float64)
    return (p[cost.W1:cost.B1].reshape(48, 64), p[cost.B1:cost.W2], p[cost.W2:cost.B2].reshape(64, 64), p[cost.B2:cost.W3],
            p[cost.W3:cost.B3].reshape(64, 2), p[cost.B3:])


def _forward(x, layers):
    w1, b1, w2, b2, w3, b3 = layers
    h1 = np.maximum(x @ w1 + b1, 0)
    h2 = np.maximum(h1 @ w2 + b2, 0)
    return h1, h2, h2 @ w3 + b3


def exact(case, seed):
    if case["kind"] == "regroup":
        x = _features64(_start_states(case, seed))
        return {"features": x, "prediction": _forward(x, _layers(seed))[2], "order": None, "states": None}
    if case["kind"] != "gradients":
        return None  # words and bytes: compared as they are
    feat, target, contact = (v.astype(np.float64) for v in _train_batch(case, seed))
    layers = _layers(seed)
    h1, h2, y = _forward(feat, layers)
    e, z, b = y[:, 0] - target, y[:, 1], case["batch"]
    loss = e * e + np.logaddexp(0, z) - contact * z
    dy = np.stack([2 * e, 1 / (1 + np.exp(-z)) - contact], 1) / b
    dh2 = (dy @ layers[4].T) * (h2 > 0)
    dh1 = (dh2 @ layers[2].T) * (h1 > 0)
    grad = [feat.T @ dh1, dh1.sum(0), h1.T @ dh2, dh2.sum(0), h2.T @ dy, dy.sum(0)]
    return {"loss": loss, "grad": np.concatenate([g.ravel() for g in grad])}
