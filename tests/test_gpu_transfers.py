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
