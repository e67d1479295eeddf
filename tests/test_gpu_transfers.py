"""Host transfers: small ones go through a pinned buffer and one kernel, larger
ones by a copy each.  Both give back what was handed in, bit for bit, on either
side of the line (6451 particles) and for one particle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 777, 6451, 6452, 9000])
@pytest.mark.parametrize("kind", ["gas", "active"])
def test_round_trip(gpu_ctx, n, kind):
    import mavi_hip as mv

    rng = np.random.default_rng(n)
    side = int(np.ceil(np.sqrt(n))) + 3
    L = 2.0 * side
    ix = np.arange(n)
    pos = np.stack([(ix % side + 0.5) * 2.0, (ix // side + 0.5) * 2.0], axis=1) + rng.uniform(-0.2, 0.2, (n, 2))
    space = mv.SpaceCfg(wall_type=mv.PeriodicWalls(), geometry_cfg=mv.RectangleCfg(length=L, height=L))
    ic = mv.IntCfg(dt=1e-3, chunks_cfg=mv.ChunksCfg(num_cols=side // 2 + 1, num_rows=side // 2 + 1), device=mv.GPU())
    if kind == "gas":
        extra = rng.normal(size=(n, 2))
        dyn = mv.HarmTruncCfg(k_rep=10.0, k_atr=1.0, dist_eq=1.0, dist_max=1.2)
        s = mv.System(state=mv.SecondLawState(pos=pos.copy(), vel=extra.copy()), space_cfg=space, dynamic_cfg=dyn,
                      int_cfg=ic)
    else:
        extra = rng.uniform(-3.0, 3.0, n)
        dyn = mv.SzaboCfg(vo=1.0, mobility=1.0, relax_time=1.0, k_rep=10.0, k_adh=0.75, r_eq=0.9, r_max=1.1,
                          rot_diff=0.1)
        s = mv.System(state=mv.SelfPropelledState(pos=pos.copy(), pol_angle=extra.copy()), space_cfg=space,
                      dynamic_cfg=dyn, int_cfg=ic)
    for k in range(2):  # the buffer again
        s.upload()
        s.state.pos[...] = 0.0
        (s.state.vel if kind == "gas" else s.state.pol_angle)[...] = 0.0
        s.download()
        assert np.array_equal(s.state.pos, pos)
        assert np.array_equal(s.state.vel if kind == "gas" else s.state.pol_angle, extra)
    f = s.calc_forces().copy()
    s.forces[...] = 7.0
    s.download()
    assert np.array_equal(s.forces, f)
    # an array the device cannot write into directly
    odd = np.zeros((n, 4), dtype=np.float64)[:, ::2]
    s.dev.get_forces(odd)
    assert np.array_equal(odd, f) and np.array_equal(s.dev.get_forces(), f)


def test_buffers_change_hands(gpu_ctx):
    """Systems and batches of several sizes made and dropped in turn, in two
    threads with a context each: every one reads back what it was given, in
    buffers that others had before it."""
    import threading

    import mavi_hip as mv
    from mavi_hip import _lib
    from mavi_hip import batch as mb

    def case(n, rng):
        side = int(np.ceil(np.sqrt(n))) + 3
        ix = np.arange(n)
        pos = np.stack([(ix % side + 0.5) * 2.0, (ix // side + 0.5) * 2.0], axis=1) + rng.uniform(-0.2, 0.2, (n, 2))
        space = mv.SpaceCfg(wall_type=mv.PeriodicWalls(),
                            geometry_cfg=mv.RectangleCfg(length=2.0 * side, height=2.0 * side))
        ic = mv.IntCfg(dt=1e-3, chunks_cfg=mv.ChunksCfg(num_cols=side // 2 + 1, num_rows=side // 2 + 1), device=mv.GPU())
        dyn = mv.HarmTruncCfg(k_rep=10.0, k_atr=1.0, dist_eq=1.0, dist_max=1.2)
        return mv.SecondLawState(pos=pos, vel=rng.normal(size=(n, 2))), space, dyn, ic

    failed = []

    def work(seed):
        try:
            ctx = _lib.Context(0)
            rng = np.random.default_rng(seed)
            held = []
            for k in range(40):
                n = int(rng.choice([5, 300, 301, 1500, 6451, 7000]))
                st, space, dyn, ic = case(n, rng)
                s = mv.System(state=st, space_cfg=space, dynamic_cfg=dyn, int_cfg=ic, ctx=ctx)
                held.append((s, st.pos.copy(), st.vel.copy()))
                if k % 5 == 4:
                    b = mb.Batch(ctx=ctx)
                    b.add(st, space, dyn, ic)
                    b.finalize()
                    b.upload(0, st.pos, st.vel)
                    pos, vel, _ = b.download(0)
                    assert np.array_equal(pos, st.pos) and np.array_equal(vel, st.vel)
                    del b
                for s, pos, vel in held:
                    s.state.pos[...] = 0.0
                    s.state.vel[...] = 0.0
                    s.download()
                    assert np.array_equal(s.state.pos, pos) and np.array_equal(s.state.vel, vel)
                del s
                while len(held) > 4:
                    held.pop(int(rng.integers(len(held))))
        except Exception as e:  # noqa: BLE001 (handed to the test's thread)
            failed.append(e)

    threads = [threading.Thread(target=work, args=(seed,)) for seed in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed, failed
