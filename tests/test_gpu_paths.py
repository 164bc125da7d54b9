"""The device's launch paths against the C oracle at the sizes where a path begins or ends.

A world is a container of bodies whose shapes are a fixture's, so that their geometry
records are the reference's own; every step is compared as tests/test_gpu_oracle.py
compares it, bit for bit, with the oracle stepping the device's previous state.
"""
import ctypes
import os
import time

import numpy as np
import pytest

import forge2d_amd as F
from forge2d_amd import scenes
from forge2d_amd import snapshot as S
from oracle import pyoracle as O
from tests.conftest import GOLDEN, load_fixture
from tests.flat_util import FlatWorld
from tests.test_gpu_oracle import compare

pytestmark = pytest.mark.gpu
GEOM_BYTES = 148


def container(bodies: int, seed: int, bullets: float = 0.0, sleep: bool = False, speed: float = 0.0,
              columns: int = 0, asleep: int = 0, shapeless: int = 0) -> tuple[bytes, bytes]:
    """(spec, geometry records) of a world of `bodies` dynamic bodies in rows in a
    container, their shapes drawn from the "mixed" fixture's dynamic ones; the first
    `asleep` are created asleep, and `shapeless` bodies without shapes follow them. One
    static body, the container's, comes before."""
    src, _, _ = load_fixture("mixed")
    (_, fb, fs, _), = scenes.parse(src)
    fg = np.load(os.path.join(GOLDEN, "mixed.npz"))["geoms"].reshape(-1, GEOM_BYTES)
    dynamic = np.flatnonzero((fb["type"][fs["body"]] == scenes.DYNAMIC) & (fs["kind"] != scenes.K_SEGMENT))
    walls = np.flatnonzero(fs["kind"] == scenes.K_SEGMENT)
    hw = np.abs(fs["data"][walls][:, [0, 2]]).max()
    rng = np.random.default_rng(seed)
    pick = rng.choice(dynamic, bodies)
    columns = columns or int((2.0 * hw - 2.0) / 1.7)
    at = np.arange(bodies)
    b = np.zeros(bodies + 1, scenes.BODY_DT)
    b["qc"], b["gravity_scale"], b["sleep_threshold"] = 1.0, 1.0, 0.05
    b["flags"] = scenes.BF_ENABLE_SLEEP | scenes.BF_AWAKE
    b["type"][1:] = scenes.DYNAMIC
    b["px"][1:] = 1.7 * (at % columns - (columns - 1) / 2.0) + rng.uniform(-0.1, 0.1, bodies)
    b["py"][1:] = 1.0 + 1.3 * (at // columns) + rng.uniform(-0.1, 0.1, bodies)
    b["vx"][1:], b["vy"][1:] = speed * rng.uniform(-1, 1, bodies), -speed * rng.random(bodies)
    b["flags"][1:] |= np.where(rng.random(bodies) < bullets, scenes.BF_BULLET, 0).astype(np.int32)
    s = np.concatenate([fs[walls], fs[pick]])
    s["body"][:len(walls)], s["body"][len(walls):] = 0, 1 + at
    b["flags"][1:1 + asleep] &= ~scenes.BF_AWAKE
    extra = np.zeros(shapeless, scenes.BODY_DT)
    extra["qc"], extra["flags"], extra["type"] = 1.0, scenes.BF_ENABLE_SLEEP | scenes.BF_AWAKE, scenes.DYNAMIC
    extra["px"], extra["vx"], extra["w"], extra["lin_damp"] = np.arange(shapeless), 0.5, 1.0, 0.25
    b = np.concatenate([b, extra])
    h = scenes.world_header(sleep=sleep)
    h["body_count"], h["shape_count"] = len(b), len(s)
    spec = scenes.MAGIC + np.array([1, 0], "<i4").tobytes() + h.tobytes() + b.tobytes() + s.tobytes()
    return spec, np.concatenate([fg[walls], fg[pick]]).tobytes()


def follow(spec: bytes, geoms: bytes, steps: int, b: F.Batch | None = None):
    b = b or F.Batch(spec)
    raw = b.export(0)
    prev = S.parse_one(raw)
    for k in range(1, steps + 1):
        b.step(steps=1)
        assert b.sync() == 0
        mine_raw = b.export(0)
        mine = S.parse_one(mine_raw)
        compare(mine, S.parse_one(O.step(spec, geoms, raw, prev).export()))
        raw, prev = mine_raw, mine


# bullets sweep against the proxies in query order from LDS up to 2,048 shapes a world and
# from HBM above: one bullet, a few, more than a workgroup's 64 lanes, and either side of
# the limit (the fixture's container has four walls)
@pytest.mark.parametrize("bodies,bullets,sleep,steps", [(9, 1.0, False, 40), (70, 0.1, True, 40), (200, 0.6, False, 40),
                                                        (2044, 0.05, False, 6), (2045, 0.05, False, 6)])
def test_bullets(gpu, bodies, bullets, sleep, steps):
    spec, geoms = container(bodies, 11 + bodies, bullets=bullets, sleep=sleep, speed=25.0)
    follow(spec, geoms, steps)


# the solver stages: contacts in registers (up to three a lane), or streamed with the bodies
# in LDS (more contacts than that, or worlds above 1,024 bodies, as 1,024 here are with their
# container), or a launch a stage (above 4,096 bodies: 4,095 are the most that is not); lanes
# a power of two from 64, worlds on both sides of what they hold
@pytest.mark.parametrize("bodies,block,steps", [(1, 64, 30), (2, 1024, 30), (63, 64, 40), (64, 64, 40), (130, 64, 60),
                                                (130, 128, 60), (500, 64, 40), (500, 256, 40), (500, 512, 40),
                                                (1000, 1024, 30), (1023, 512, 20), (1024, 1024, 20), (3000, 1024, 12),
                                                (4095, 1024, 6), (4096, 256, 6), (4097, 1024, 6)])
def test_solver_stages(gpu, bodies, block, steps):
    spec, geoms = container(bodies, 23 + bodies, speed=4.0)
    b = F.Batch(spec)
    b.set_block(block)
    follow(spec, geoms, steps, b)


# the solver stages streamed with nothing in LDS, as in worlds whose states do not fit: the size
# set to 0, or so many more bodies than shapes that the scratch region has no room for the
# per-step body terms. Stepped one by one, a batch's worlds take the size of its largest
@pytest.mark.parametrize("bodies,shapeless,solve_lds,block,steps", [
    (1, 0, 0, 64, 30), (130, 0, 0, 64, 60), (500, 0, 0, 512, 30), (1500, 0, 0, 1024, 12), (40, 1100, None, 256, 40),
    (300, 3000, None, 1024, 20)])
def test_solver_stages_without_lds(gpu, bodies, shapeless, solve_lds, block, steps):
    spec, geoms = container(bodies, 29 + bodies, speed=4.0, shapeless=shapeless)
    b = F.Batch(spec)
    b.upload()
    b.set_block(block)
    if solve_lds is not None:
        b.set_class_solve_lds(0, solve_lds)
    follow(spec, geoms, steps, b)


def test_worlds_stepped_one_by_one_without_lds(gpu):
    specs = [container(n, 31 + n, speed=4.0)[0] for n in (200, 1500, 5000)]  # 160 KB of states in the last
    spec = scenes.MAGIC + np.array([len(specs), 0], "<i4").tobytes() + b"".join(s[16:] for s in specs)
    one, all_ = F.Batch(spec), F.Batch(spec)
    one.step_each(steps=8)
    all_.step(steps=8)
    assert one.sync() == 0 and all_.sync() == 0
    for w in range(len(specs)):
        assert one.export(w) == all_.export(w), w


# the reported solve LDS of every class can be given back, as can what the sizes between the
# solver's forms are; less than the body states cannot
def test_solve_lds_given_back(gpu):
    specs = [container(n, 3 + n)[0] for n in (40, 200, 500, 900, 1100, 3000, 6000)]
    b = F.Batch(scenes.MAGIC + np.array([len(specs), 0], "<i4").tobytes() + b"".join(s[16:] for s in specs))
    b.upload()
    classes = b.size_classes()
    assert len(classes) == 7
    for k, c in enumerate(classes):
        for size in (c["solve_lds"], 0, 32 * c["max_bodies"], 64 * (c["max_bodies"] + 1)):
            if size <= 159744:
                b.set_class_solve_lds(k, size)
                assert b.size_classes()[k]["solve_lds"] == size
        for size in (32 * c["max_bodies"] - 1, 163841, -1):
            with pytest.raises(RuntimeError):
                b.set_class_solve_lds(k, size)
        b.set_class_solve_lds(k, c["solve_lds"])
    assert b.size_classes() == classes


# a frame's body events come from records written behind the step, or, once the mirror was
# read back, from the mirror: the same, for worlds around the record kernel's 256 lanes
@pytest.mark.parametrize("bodies,sleep,steps", [(1, True, 90), (255, False, 4), (256, True, 4), (700, False, 4)])
def test_frame_records(gpu, bodies, sleep, steps):
    L = F.lib()
    spec, _ = container(bodies, 41 + bodies, sleep=sleep, speed=1.0)
    w = FlatWorld(spec)
    a, b = np.zeros((bodies + 1, 7)), np.zeros((bodies + 1, 7))
    pos = (ctypes.c_float * 2)()
    asleep = 0
    for k in range(steps):
        w.step()
        n = L.f2d_world_get_body_event_count(w.w)
        assert L.f2d_world_get_body_events(w.w, a.ctypes.data_as(F._PD)) == n
        L.f2d_body_get_position(*w.bodies[1], pos)  # reads the mirror back
        assert L.f2d_world_get_body_events(w.w, b.ctypes.data_as(F._PD)) == n
        assert np.array_equal(a[:n], b[:n])
        asleep += int(a[:n, 6].sum())
    assert asleep > 0 or not (sleep and bodies == 1)
    # an edit between the step and the read shows, as it always did
    w.step()
    L.f2d_body_set_transform(*w.bodies[1], 3.0, 4.0, 1.0, 0.0)
    n = L.f2d_world_get_body_events(w.w, a.ctypes.data_as(F._PD))
    assert n == 0 or a[:n][a[:n, 0] == w.bodies[1][0]][0, 2:4].tolist() == [3.0, 4.0]
    w.close()


# islands split on all lanes, their edges in LDS or (above 1,024 bodies) in the scratch region
@pytest.mark.parametrize("bodies,steps", [(40, 200), (300, 150), (1500, 100)])
def test_islands_sleep_and_split(gpu, bodies, steps):
    spec, geoms = container(bodies, 7 + bodies, sleep=True, speed=1.0)
    follow(spec, geoms, steps)


# every sleeping body is a set of its own, and a body falls on each: hundreds of sets wake in
# one state loop, among contacts that begin without one
@pytest.mark.parametrize("sets,steps", [(30, 30), (400, 16)])
def test_sets_woken_together(gpu, sets, steps):
    spec, geoms = container(2 * sets, 61 + sets, sleep=True, speed=2.0, columns=sets, asleep=sets)
    follow(spec, geoms, steps)


# four times the sleeping boxes, each woken in the first step, take about four times as long
# (16 times if a wake cost what the world is large); the larger world of the two is the one
# whose loop the cost would rule
def test_waking_a_set_costs_the_set(gpu):
    def first_step(sets: int) -> float:
        w = scenes.World(scenes.world_header(sleep=True))
        for i in range(sets):
            w.add_box(w.add_body(scenes.DYNAMIC, 2.0 * i, 0.5, flags=scenes.BF_ENABLE_SLEEP), 0.5, 0.5)
        for i in range(sets):
            w.add_box(w.add_body(scenes.DYNAMIC, 2.0 * i, 1.51), 0.5, 0.5)
        b = F.Batch([w])
        b.upload()
        b.synchronize()
        t = time.perf_counter()
        b.step(steps=1)
        b.synchronize()
        t = time.perf_counter() - t
        assert b.sync() == 0 and b.counters(0)["touching"] == sets
        return t

    first_step(10)  # the library's code objects are loaded
    small, large = first_step(500), first_step(2000)
    assert large < 8 * small, (small, large)


# a plank made last touches every box in one step, and each contact links the islands so far
# below the next box's: four times the boxes take about four times as long (16 times if each
# link walked the links before it)
def test_links_of_one_island_with_many(gpu):
    def state_loop(boxes: int) -> float:
        w = scenes.World(scenes.world_header())
        for i in range(boxes):
            w.add_box(w.add_body(scenes.DYNAMIC, 1.2 * i, 0.5), 0.5, 0.5)
        w.add_box(w.add_body(scenes.DYNAMIC, 0.6 * boxes, 1.25), 0.6 * boxes + 1.0, 0.25)
        b = F.Batch([w])
        b.upload()
        b.synchronize()
        t = time.perf_counter()
        b.step(steps=1, phases=F.PH_PAIRS | F.PH_COLLIDE | F.PH_STATE)
        b.synchronize()
        t = time.perf_counter() - t
        assert b.sync() == 0 and b.counters(0)["touching"] == boxes
        return t

    state_loop(10)  # the library's code objects are loaded
    small, large = state_loop(4000), state_loop(16000)
    assert large < 8 * small, (small, large)


# trees of more than 1,024 proxies are rebuilt beside the contacts and the solve: steps
# queued one behind the other give what steps with a wait between them give
@pytest.mark.parametrize("bodies,steps", [(1024, 8), (1025, 8), (2400, 8), (4200, 6)])
def test_tree_rebuild_beside_the_solve(gpu, bodies, steps):
    spec, geoms = container(bodies, 5 + bodies, bullets=0.02, speed=20.0)
    follow(spec, geoms, 2)
    queued, waited = F.Batch(spec), F.Batch(spec)
    queued.step(steps=steps)
    for _ in range(steps):
        waited.step(steps=1)
        assert waited.sync() == 0
    assert queued.sync() == 0 and queued.error_bits() == 0
    assert queued.export(0) == waited.export(0)
