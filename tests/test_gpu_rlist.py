"""Rings step! on Verlet lists (one kernel per step, mavi_rlist.hip) against
the chunk gather (MAVI_OPT_NLIST 0): the lists add a particle's pairs in the
gather's order, so positions, polarisations, forces, areas, centres of mass and
continuous positions are the same bits, whatever the box, the ring sizes, the
length of the lists, the rebuild times and the split into calls.  The gather
itself is checked against the oracle in test_gpu_rings.py."""
import sys

import numpy as np
import pytest

from test_gpu_rings import normal_case, types_case

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def mixture(**kw):
    from mavi_hip import workloads as wl

    return wl.rings_mixture(**kw)


def squeezed(case, factor, dt):
    """The case shrunk: many pairs in range of a particle, long lists."""
    import mavi_hip as mv
    from mavi_hip import rings

    state, space, cfg, ic = case
    g = space.geometry_cfg
    L, H = g.length * factor, g.height * factor
    state = rings.RingsState(rings_pos=state.rings_pos * factor, pol=state.pol, num_particles=state.num_particles,
                             types=state.types)
    reach = 1.2
    space = mv.SpaceCfg(geometry_cfg=mv.RectangleCfg(length=L, height=H), wall_type=mv.PeriodicWalls())
    ic = mv.IntCfg(dt=dt, chunks_cfg=mv.ChunksCfg(int(L // reach - 1e-9), int(H // reach - 1e-9)), device=mv.GPU())
    return state, space, cfg, ic


OFF_LISTS = ("tiny_box", "rings_of_two")  # no 3 x 3 cells of range + skin; more sums in a wave than lanes
CASES = {
    "normal": lambda: normal_case(True),
    "normal_ragged": lambda: normal_case(True, n=21, cols=7, rows=5, seed=3),
    "smallest_rings": lambda: normal_case(True, n=4, cols=6, rows=7, seed=4),
    "rings_of_two": lambda: normal_case(True, n=2, cols=12, rows=11, seed=13),
    "rings_of_three": lambda: normal_case(True, n=3, cols=11, rows=9, seed=14),
    "largest_rings": lambda: normal_case(True, n=32, cols=5, rows=3, seed=5),
    "few_cells": lambda: normal_case(True, n=9, cols=2, rows=2, seed=6),
    "tiny_box": lambda: normal_case(True, n=3, cols=2, rows=2, seed=15),
    "types": lambda: types_case(True),
    "mixture": lambda: mixture(nrings=120, seed=8),
    "dense": lambda: squeezed(normal_case(True, n=10, cols=9, rows=8), 0.62, 1e-4),
    "dense_types": lambda: squeezed(types_case(True), 0.7, 1e-4),
    "touching": lambda: squeezed(normal_case(True, n=10, cols=9, rows=8), 0.66, 1e-4),
}


def make(case, lists, seed=11, dt=None):
    import mavi_hip as mv
    from mavi_hip import _lib, rings

    state, space, cfg, ic = CASES[case]()
    if dt is not None:
        ic = mv.IntCfg(dt=dt, chunks_cfg=ic.chunks_cfg, device=mv.GPU())
    s = rings.RingsSystem(state=state, space_cfg=space, dynamic_cfg=cfg, int_cfg=ic, seed=seed)
    if not lists:
        s.dev.set_option(_lib.MAVI_OPT_NLIST, 0)
    return s


def same(tag, a, b):
    for s in (a, b):
        s.download()
    for what, x, y in (("pos", a.state.pos, b.state.pos), ("pol", a.state.pol, b.state.pol),
                       ("forces", a.forces, b.forces), ("areas", a.areas, b.areas), ("cms", a.cms, b.cms),
                       ("continuos_pos", a.continuos_pos, b.continuos_pos)):
        assert np.array_equal(x, y), (tag, what, float(np.abs(np.asarray(x) - np.asarray(y)).max()))


@pytest.mark.parametrize("case", list(CASES))
def test_same_bits_as_the_gather(gpu_ctx, case):
    a, b = make(case, True), make(case, False)
    info = a.dev.nlist_info()
    say(f"[rings lists] {case} {info}")
    assert info["eligible"] == (case != "rings_of_two") and not b.dev.nlist_info()["active"]
    for k in (8, 61, 1, 30):
        a.advance(k)
        b.advance(k)
        same((case, k), a, b)
    say(f"[rings lists] {case} {a.dev.nlist_info()}")
    assert (a.dev.nlist_info()["rebuilds"] >= 1) == (case not in OFF_LISTS)


def partners(s, reach):
    """Particles within `reach` of each particle, bonded neighbours left out."""
    pos = s.state.pos.reshape(-1, 2)
    g = s.space_cfg.geometry_cfg
    n = s.state.rings_pos.shape[1]
    d = pos[:, None, :] - pos[None, :, :]
    box = np.array([g.length, g.height])
    d -= box * np.round(d / box)
    near = (d ** 2).sum(axis=2) <= reach ** 2
    ring, k = np.arange(len(pos)) // n, np.arange(len(pos)) % n
    gap = np.abs(k[:, None] - k[None, :])
    near &= ~((ring[:, None] == ring[None, :]) & ((gap <= 1) | (gap == n - 1)))
    return near.sum(axis=1)


@pytest.mark.parametrize("case", [c for c in CASES if c not in OFF_LISTS])
def test_same_bits_with_every_step_on_lists(gpu_ctx, case):
    """At a time step short enough for the lists not one step goes to the
    gather: a third system with the launch counters on says so."""
    from mavi_hip import _lib

    dt = min(1e-3, CASES[case]()[3].dt)
    a, b, c = make(case, True, dt=dt), make(case, False, dt=dt), make(case, True, dt=dt)
    if case == "dense":  # more pairs in range than the first four entries hold
        assert partners(a, 1.2).max() > 4
    if case == "touching":  # three or four pairs in range, all among the first entries: put in order there
        assert partners(a, 1.2).max() >= 3 and partners(a, 1.2 * 1.02).max() <= 4
        for s in (a, c):
            s.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, 20)
    c.dev.prof_enable(True)
    for k in (8, 61, 31):
        for s in (a, b, c):
            s.advance(k)
        same((case, k), a, b)
        same((case, k, "direct launches"), c, b)
    gathers, steps = c.dev.prof_get(_lib.MAVI_PROF_FORCE)[1], c.dev.prof_get(_lib.MAVI_PROF_RINGS)[1]
    say(f"[rings lists] {case} gathers {gathers} list steps {steps} {a.dev.nlist_info()} {c.dev.nlist_info()}")
    assert gathers == 0 and steps >= 100 and a.dev.nlist_info()["active"]


@pytest.mark.parametrize("skin,block,graphs", [(0, 0, 0), (50, 64, 1), (100, 7, 1), (600, 0, 1), (1000, 1, 1)])
def test_skins_blocks_and_rollbacks(gpu_ctx, skin, block, graphs):
    """Rebuild times, rolled-back blocks (a skin too thin for its fixed
    block) and direct launches change nothing."""
    from mavi_hip import _lib

    a, b = make("normal", True), make("normal", False)
    a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, skin)
    a.dev.set_option(_lib.MAVI_OPT_NLIST_BLOCK, block)
    a.dev.set_option(_lib.MAVI_OPT_GRAPHS, graphs)
    a.advance(100)
    b.advance(100)
    info = a.dev.nlist_info()
    say(f"[rings lists] skin {skin} block {block} graphs {graphs} {info}")
    if block == 64:
        assert info["rollbacks"] >= 1
    same((skin, block), a, b)


def test_long_lists_hand_over(gpu_ctx):
    """Lists of more than 16 partners switch off; the gather runs the steps."""
    from mavi_hip import _lib

    a, b = make("dense", True), make("dense", False)
    a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, 2000)
    a.advance(40)
    b.advance(40)
    info = a.dev.nlist_info()
    say(f"[rings lists overflow] {info}")
    assert not info["active"]
    same("overflow", a, b)


def test_state_changes_between_runs(gpu_ctx):
    """Between list runs: a new state, forces!, a binning, the noise stream
    moved and reseeded, an invasion schedule, contact neighbours on and off."""
    from mavi_hip import rings

    a, b = make("mixture", True), make("mixture", False)
    rng = np.random.default_rng(5)
    for s in (a, b):
        s.advance(40)
    pos = np.mod(a.state.pos + rng.uniform(-0.01, 0.01, size=a.state.pos.shape), a.space_cfg.geometry_cfg.length)
    for s in (a, b):
        s.state.pos[...] = pos
        s.upload()
        s.advance(20)
    same("new state", a, b)
    for s in (a, b):
        s.dev.forces()
        s.advance(12)
        s.dev.bin()
        s.advance(12)
        s.dev.set_noise_state(77, 1000)
        s.advance(16)
    same("forces, bin, noise", a, b)
    assert a.dev.noise_state() == b.dev.noise_state()
    grid = rings.ring_chunks_grid(a.state, a.space_cfg, a.dynamic_cfg, type(a.int_cfg.chunks_cfg)(8, 8))
    for s in (a, b):
        s.dev.rings_invasions_cfg(True, 7, *grid)
        s.advance(45)
    assert np.array_equal(a.dev.rings_invasions(), b.dev.rings_invasions())
    same("invasions", a, b)
    for s in (a, b):
        s.dev.rings_neighbors_cfg(True, 1.1, False)
        s.advance(10)
    for x, y in zip(a.dev.rings_neighbors(), b.dev.rings_neighbors()):
        assert np.array_equal(x, y)
    for s in (a, b):
        s.dev.rings_neighbors_cfg(False)
        s.advance(9)
    same("neighbours", a, b)


def test_errors_are_the_gathers(gpu_ctx):
    """A chunk over its capacity and a non-finite position fail the same way."""
    import mavi_hip as mv
    from mavi_hip import _lib, rings

    state, space, cfg, ic = CASES["normal"]()
    d, chunks, keep = rings.describe(state, space, cfg, ic, 1)
    d.nc = 1
    for lists in (1, 0):
        dev = _lib.DeviceSystem(gpu_ctx, d, keep=keep)
        dev.set_option(_lib.MAVI_OPT_NLIST, lists)
        dev.upload(state.pos, None, state.pol)
        with pytest.raises(mv.CellOverflowError):
            dev.step(20)
    d.nc = chunks.nc
    bad = state.pos.copy()
    bad[17] = np.nan
    for lists in (1, 0):
        dev = _lib.DeviceSystem(gpu_ctx, d, keep=keep)
        dev.set_option(_lib.MAVI_OPT_NLIST, lists)
        dev.upload(bad, None, state.pol)
        with pytest.raises(mv.MaviError):
            dev.step(20)
        dev.upload(state.pos, None, state.pol)  # a good state runs again
        dev.step(20)


def test_skin_changes_on_a_grid_of_several_scan_tiles(gpu_ctx):
    """A list grid of several scan tiles whose number changes with the skin:
    each grid's scan starts afresh."""
    from mavi_hip import _lib, rings

    def one():
        state, space, cfg, ic = normal_case(True, n=10, cols=64, rows=60, seed=12)
        return rings.RingsSystem(state=state, space_cfg=space, dynamic_cfg=cfg, int_cfg=ic, seed=3)

    a, b = one(), one()
    b.dev.set_option(_lib.MAVI_OPT_NLIST, 0)
    for skin in (0, 100, 350, 0):
        a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, skin)
        a.advance(20)
        b.advance(20)
        assert a.dev.nlist_info()["active"]
        same(skin, a, b)


def test_lists_come_back_after_a_full_chunk(gpu_ctx):
    """Chunks over their capacity fail the call; a good state uploaded after it
    runs on lists again, and so does a thinner skin after lists that were too
    long."""
    import mavi_hip as mv
    from mavi_hip import _lib, rings

    state, space, cfg, ic = CASES["normal"]()
    ic = mv.IntCfg(dt=1e-3, chunks_cfg=ic.chunks_cfg, device=mv.GPU())
    d, _, keep = rings.describe(state, space, cfg, ic, 1)
    d.nc = 6
    crowd = state.pos.copy().reshape(-1, 10, 2)
    box, num = space.geometry_cfg, ic.chunks_cfg
    ang = np.arange(10) * 2 * np.pi / 10
    for k in range(4):  # four rings drawn together about the corner of four chunks
        at = np.array([box.length / num.num_cols, box.height / num.num_rows]) * 4
        crowd[k] = at + (0.35 * (2 * (k % 2) - 1), 0.35 * (2 * (k // 2) - 1)) + \
            0.3 * np.stack([np.cos(ang), np.sin(ang)], axis=1)
    out = []
    for lists in (1, 0):
        dev = _lib.DeviceSystem(gpu_ctx, d, keep=keep)
        dev.set_option(_lib.MAVI_OPT_NLIST, lists)
        dev.upload(crowd.reshape(-1, 2), None, state.pol)
        with pytest.raises(mv.CellOverflowError):
            dev.step(30)
        dev.set_noise_state(1, 0)
        dev.upload(state.pos, None, state.pol)
        dev.step(40)
        say(f"[rings lists] after a full chunk: {dev.nlist_info()}")
        assert dev.nlist_info()["active"] == bool(lists)
        pos, pol = np.zeros_like(state.pos), np.zeros_like(state.pol)
        dev.download(pos, None, pol)
        out.append((pos, pol))
    for x, y in zip(*out):
        assert np.array_equal(x, y)

    a, b = make("dense", True), make("dense", False)
    a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, 2000)
    for s in (a, b):
        s.dev.step(20)
    assert not a.dev.nlist_info()["active"]
    a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, 0)
    for s in (a, b):
        s.dev.step(20)
    assert a.dev.nlist_info()["active"]
    same("after long lists", a, b)


def test_steps_too_long_for_lists_go_to_the_gather(gpu_ctx):
    """Runs whose particles cross half the skin in a step or two: the lists are
    tried now and then, not once or twice in every call."""
    from mavi_hip import _lib

    a, b = make("normal", True, dt=0.02), make("normal", False, dt=0.02)
    a.dev.set_option(_lib.MAVI_OPT_NLIST_SKIN, 100)
    start = a.state.pos.copy()
    for s in (a, b):
        for _ in range(30):
            s.state.pos[...] = start
            s.upload()
            s.dev.step(10)
    info = a.dev.nlist_info()
    say(f"[rings lists] long steps {info}")
    assert info["active"] and info["rebuilds"] <= 8
    same("long steps", a, b)
