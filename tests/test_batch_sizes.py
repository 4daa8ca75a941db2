"""The launch shapes of the production block by batch size, each against the oracle word for word: one and three arenas per
wave with the states in LDS (small_kernels.hip), waves of 32 lanes, and full waves. The sizes are the edges of those
ranges and their remainders; each shape also with a world table, a trace, several decisions per launch, the queue's
entry point, goals, overflows and a world index past the table."""
import numpy as np
import pytest

import forced_cases as fc
from conftest import first_diff
from helpers import TICK_WORDS
from rsim import layout

pytestmark = pytest.mark.gpu

EDGES = [1, 63, 511, 512, 513, 514, 515, 3071, 3072, 3073, 32767, 32768, 32769]


def same(got, want, what):
    fd = first_diff(got[:, :TICK_WORDS], want[:, :TICK_WORDS])
    assert fd is None, "%s: arena %d word %d differs" % (what, fd[0], fd[1])


@pytest.mark.parametrize("n", EDGES)
def test_sim8_at_the_edges(rsim, oracle, world, device, dev_world, n):
    print("[case] sim8, %d contact arenas, 2 decisions" % n, flush=True)
    states = rsim.sample_arenas(world, rsim.SCEN_CONTACT, 900, n)
    d, r, cpu = device.upload_states(states), device.alloc_words(n), states.copy()
    for k in range(2):
        ctl = rsim.sample_controls(901, k, n)
        device.sim8(d, dev_world, device.upload_controls(ctl), r)
        assert np.array_equal(device.read_words(r), oracle.sim8(cpu, world, ctl, threads=8)), k
    same(device.download_states(d), cpu, "sim8 %d" % n)


@pytest.mark.parametrize("entry", ["run", "run_queued"])
@pytest.mark.parametrize("n", [2, 512, 514, 3072, 3075, 4100])
def test_worlds_and_decisions(rsim, oracle, device, n, entry):
    print("[case] %s, %d arenas in 5 worlds, 3 decisions" % (entry, n), flush=True)
    worlds = np.stack([rsim.build_world(p, p) for p in range(5)])
    variant = np.random.default_rng(n).integers(0, 5, n).astype(np.uint32)
    states = rsim.sample_arenas_in(worlds, variant, rsim.SCEN_OPEN_CONTACT, 902)
    ctl = np.stack([rsim.sample_controls(903, k, n) for k in range(3)])
    d, dw = device.upload_states(states), device.upload_worlds(worlds)
    c, r, v = device.upload_words(ctl), device.alloc_words(3 * n), device.upload_words(variant)
    getattr(device, entry)(d, dw, c, r, 3, variant=v)
    got, cpu = device.read_words(r).reshape(3, n), states.copy()
    for k in range(3):
        assert np.array_equal(got[k], oracle.sim8_in(cpu, worlds, variant, ctl[k], threads=8)), k
    same(device.download_states(d), cpu, "%s %d" % (entry, n))
    bad = variant.copy()
    bad[n // 2] = 5  # past the table: flagged, and the arena left as it was
    d2 = device.upload_states(states)
    device.sim8_variants(d2, dw, device.upload_words(bad), device.upload_controls(ctl[0]), r)
    one, after = device.read_words(r, n), device.download_states(d2)
    assert one[n // 2] == rsim.SIM8_BAD_VARIANT and np.array_equal(after[n // 2], states[n // 2])
    assert np.array_equal(np.delete(one, n // 2), np.delete(got[0], n // 2))


@pytest.mark.parametrize("variants", [False, True])
@pytest.mark.parametrize("n", [128, 700, 3200])
def test_trace_goals_and_overflow(rsim, oracle, world, device, dev_world, n, variants):
    print("[case] traced sim8, %d arenas with goals on every tick and overflows, variants %d" % (n, variants), flush=True)
    goals, over = fc.goal_states(rsim, world, 7)[0][::2], fc.overflow_states(rsim, world, 64, 17)
    some = np.concatenate([goals, over])[:n]
    states = np.concatenate([some, rsim.sample_arenas(world, rsim.SCEN_GOALFRAME, 904, n)])[:n]
    states = np.ascontiguousarray(states[np.random.default_rng(3).permutation(n)])
    ctl = np.zeros((n, 16), np.uint32)
    d, r = device.upload_states(states), device.alloc_words(n)
    trace = device.alloc_words(8 * rsim.aosoa_words(n))
    if variants:
        device.sim8_variants(d, dev_world, device.upload_words(np.zeros(n, np.uint32)), device.upload_controls(ctl), r, trace=trace)
    else:
        device.sim8(d, dev_world, device.upload_controls(ctl), r, trace=trace)
    word = device.read_words(r)
    slabs = device.read_words(trace).reshape(8, -1)
    cpu, ticks = states.copy(), states.copy()
    assert np.array_equal(word, oracle.sim8(cpu, world, ctl, threads=8))
    assert ((word & 0xFF) > 0).any() and (word & rsim.SIM8_OVERFLOW).any()
    same(device.download_states(d), cpu, "traced %d" % n)
    scored = word & 0xFF
    for t in range(1, 9):
        live = (scored == 0) | (scored >= t)
        idx = np.nonzero(live[:100])[0]
        for a in idx:
            oracle.set_controls(ticks[a], ctl[a])
            oracle.step_tick(ticks[a], world)
        got = rsim.aosoa_unpack(slabs[t - 1], n)
        same(got[idx], ticks[idx], "trace tick %d" % t)
        assert not got[~live].any(), "ticks after a goal are not written"


@pytest.mark.parametrize("n", [1, 63, 64, 65, 6143, 6144, 6145, 12289])
def test_states_to_the_device_and_back(rsim, device, n):
    """The device's packing against the host's (rsim_aosoa_pack / unpack), at the edges of a block and of the staging
    buffer; the padding lanes come out zero whatever the buffer held."""
    print("[case] states up and down, %d arenas" % n, flush=True)
    rng = np.random.default_rng(n)
    states, before = (rng.integers(0, 2**32, (n, rsim.ARENA_WORDS), dtype=np.uint32) for _ in range(2))
    d = device.upload_states(before)
    device.write_states(d, states)
    words = device.download_words(d)
    assert np.array_equal(words, rsim.aosoa_pack(states))
    assert np.array_equal(device.download_states(d), rsim.aosoa_unpack(words, n))


@pytest.mark.parametrize("block", [64, 128, 256])
def test_full_waves_of_one_arena(rsim, oracle, world, device, dev_world, block):
    """256 contact arenas, each in all 64 lanes of a wave of its own: every lane brings the same walks, so some waves fill the
    pooled walk's queues to their last slots and some past them (a wave of 15 leaves a lane has 960)."""
    print("[case] waves of one arena, block %d" % block, flush=True)
    k, copies = 256, 256 if block == 64 else 64  # at block 64, enough arenas for full waves
    states = rsim.sample_arenas(world, rsim.SCEN_CONTACT, 5, k)
    d, r = device.upload_states(np.repeat(states, copies, axis=0)), device.alloc_words(copies * k)
    for decision in range(4):
        ctl = rsim.sample_controls(9, decision, k)
        device.sim8(d, dev_world, device.upload_controls(np.repeat(ctl, copies, axis=0)), r, block=block)
        assert np.array_equal(device.read_words(r), np.repeat(oracle.sim8(states, world, ctl, threads=8), copies)), decision
    same(device.download_states(d), np.repeat(states, copies, axis=0), "waves of one arena, block %d" % block)


@pytest.mark.parametrize("n", [3, 64, 700])
def test_cars_tied_to_each_other(rsim, oracle, world, device, dev_world, n):
    """A small batch gives each car a lane of its own; cars whose updates touch shared state take turns. Arena by arena:
    both cars demoed and due in the same tick (they draw from one random state), the second car standing on the first
    (its wheels push it), the first car standing on the ball, and a plain kickoff beside them in the same wave."""
    print("[case] tied cars, %d arenas" % n, flush=True)
    states = rsim.sample_arenas(world, rsim.SCEN_KICKOFF, 77, n)
    a = layout.arena_view(states)
    for i in range(n):
        kind, cars, bodies = i % 4, a["cars"][i], a["bodies"][i]
        if kind == 0:
            cars["is_demoed"][:] = 1
            cars["demo_respawn_timer"][:] = np.float32((1 + i % 7) / 120.0)
            continue
        if kind == 3:
            continue
        below = {f: float(cars[0]["pos"][f]) for f in "xyz"}  # kind 1: the second car over the first
        if kind == 2:  # the first car over the ball
            fc.place_ball(a, i, (below["x"], below["y"], 93.0), (0, 0, 0))
            below["z"] = 93.0 + 91.0
        top = 1 if kind == 1 else 0
        for f in "xyz":
            x = np.float32(below[f] + (40.0 if f == "z" else 0.0))
            cars[top]["pos"][f] = x
            for t in ("world_trans", "interp_world_trans"):
                bodies[1 + top][t]["translation"][f] = x * fc.UU_TO_BT
    d, r = device.upload_states(states), device.alloc_words(n)
    stood = np.zeros(n, bool)
    for k in range(3):
        ctl = rsim.sample_controls(78, k, n)
        device.sim8(d, dev_world, device.upload_controls(ctl), r)
        assert np.array_equal(device.read_words(r), oracle.sim8(states, world, ctl, threads=8)), k
        ray = a["cars"]["wheels"]["raycast_info"]
        stood |= ((ray["some"] != 0) & (ray["v"]["ground_stick"]["some"] != 0)).any((1, 2))
    assert stood[1::4].any() and (n < 4 or stood[2::4].any()), "some wheels stood on a car, some on the ball"
    same(device.download_states(d), states, "tied cars %d" % n)


@pytest.mark.parametrize("per_wave", [1, 3])
def test_small_batches_past_the_pooled_queues(rsim, oracle, device, per_wave):
    """A ball of 800 uu, whose box takes in up to some hundred mesh leaves: the pooled walk of a small batch's wave holds 232
    leaves, and the arenas are chosen so that waves end below that, on its last slot and past it (each lane then walks its
    own meshes)."""
    slots, n = 232, 300 if per_wave == 1 else 900
    print("[case] %d arenas, %d a wave, around %d leaves a wave" % (n, per_wave, slots), flush=True)
    world = rsim.build_world(0, 0, ball_radius=800.0)
    many = rsim.sample_arenas(world, rsim.SCEN_PINCH, 905, 3000)
    leaves = np.array([oracle.mesh_leaves(s, world) for s in many])
    waves = np.random.default_rng(906).integers(0, len(many), (20000, per_wave))
    total = leaves[waves].sum(1)
    near = np.argsort(np.abs(total - slots), kind="stable")[:n // per_wave * 9 // 10]
    waves, total = np.concatenate([waves[near], waves[:n // per_wave - len(near)]]), total[near]
    assert (total < slots).any() and (total == slots).any() and (total > slots).any()
    states = np.ascontiguousarray(many[waves.ravel()])
    d, dw, r = device.upload_states(states), device.upload_static(world), device.alloc_words(n)
    for k in range(3):
        ctl = rsim.sample_controls(907, k, n)
        device.sim8(d, dw, device.upload_controls(ctl), r)
        assert np.array_equal(device.read_words(r), oracle.sim8(states, world, ctl, threads=8)), k
    same(device.download_states(d), states, "past the pooled queues, %d a wave" % per_wave)
