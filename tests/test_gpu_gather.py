"""The chunk gather with eight candidates in flight (systems up to 300k
particles) against the two-candidate loops, which the two-phase option still
takes: the same candidates in the same order, and a candidate out of range adds
an exact zero, so the same bits."""
import numpy as np
import pytest

from test_gpu_parity import FORCE_RTOL, force_rel_err, make_plain, say

pytestmark = pytest.mark.gpu

# particles, columns, rows: fewer than a wave, a whole wave, one over; grids of
# one row or column (rigid), the smallest periodic grid (every column at an
# edge), chunks of 0 to ~20 particles (remainders of a batch of eight)
SIZES = [(1, 3, 3), (63, 3, 3), (64, 4, 3), (65, 3, 5), (130, 1, 1), (200, 1, 7), (200, 6, 1), (700, 17, 5),
         (5000, 33, 29)]


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("kind", ["lj", "ht"])
@pytest.mark.parametrize("n,cols,rows", SIZES)
def test_deep_gather_bitexact(gpu_ctx, oracle_mod, n, cols, rows, kind, periodic):
    import mavi_hip as mv
    from mavi_hip import _lib

    if periodic and (cols < 3 or rows < 3):
        pytest.skip("periodic grids have at least three chunks a side")
    rng = np.random.default_rng(n + 31 * cols + rows)
    # chunks 3 sigma wide; particles jittered on a square lattice over the box,
    # so that no pair is closer than 0.55 of the lattice step
    L, H = 3.0 * cols, 3.0 * rows
    nx = int(np.ceil(np.sqrt(n * L / H)))
    ny = int(np.ceil(n / nx))
    ix = np.arange(n)
    jit = 0.2 * rng.uniform(-1.0, 1.0, (n, 2))
    pos = np.stack([(ix % nx + 0.5 + jit[:, 0]) * L / nx, (ix // nx + 0.5 + jit[:, 1]) * H / ny], axis=1)
    vel = rng.normal(size=(n, 2))
    sigma = min(1.0, L / nx, H / ny)
    if kind == "lj":
        dyn = mv.LenJonesCfg(sigma=sigma, epsilon=1.0, cutoff=2.5 * sigma)
    else:
        dyn = mv.HarmTruncCfg(k_rep=10.0, k_atr=1.0, dist_eq=sigma, dist_max=1.5 * sigma)
    wall = mv.PeriodicWalls() if periodic else mv.RigidWalls()
    space = mv.SpaceCfg(wall_type=wall, geometry_cfg=mv.RectangleCfg(length=L, height=H))
    ic = mv.IntCfg(dt=1e-4 * sigma, chunks_cfg=mv.ChunksCfg(num_cols=cols, num_rows=rows), device=mv.GPU())
    say(f"[deep gather] {kind} n={n} {cols}x{rows} periodic={periodic}")
    out = []
    for two_phase in (0, 1):
        s = make_plain(pos.copy(), vel.copy(), space, dyn, ic)
        s.dev.set_option(_lib.MAVI_OPT_NLIST, 0)
        s.dev.set_option(_lib.MAVI_OPT_TWO_PHASE, two_phase)
        f = s.calc_forces().copy()
        s.advance(20)
        s.download()
        out.append((f, s.state.pos.copy(), s.state.vel.copy(), s.forces.copy()))
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    if min(cols, rows) == 1:
        return  # the oracle's stencil needs two chunks a side
    o = oracle_mod.from_system(n, space, dyn, ic)
    f_ref, ab = o.forces(pos, with_absum=True)
    assert force_rel_err(out[0][0], f_ref, ab) <= FORCE_RTOL
