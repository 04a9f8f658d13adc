"""The small-box routes (a fused stage of 4x4x4 tiles; one thread per face)
against the marching tiles, bit for bit, on both sides of every rule that
chooses between them (GPU)."""
import numpy as np
import pytest

from nmhd_amd import capi, problems as P

pytestmark = pytest.mark.gpu


def rough(cfg, seed):
    """Independent random rho, v, p, B per cell, B = 0 on 1/16 of the faces."""
    n = cfg["n"]
    idx = np.arange(n[0] * n[1] * n[2], dtype=np.uint64)
    u = [P.uniform01(seed, idx, c).reshape(n[2], n[1], n[0]) for c in range(8)]
    W = np.stack([0.2 + u[0], u[1] - 0.5, u[2] - 0.5, u[3] - 0.5, 0.2 + u[4],
                  u[5] - 0.5, u[6] - 0.5, u[7] - 0.5]).astype(np.float32)
    for f in (5, 6, 7):
        W[f][(idx.reshape(W[f].shape) * np.uint64(2654435761) >> np.uint64(7)) % np.uint64(16)
             == f] = 0.0
    return W


def run(cfg, W, tiles):
    """Two frozen-size steps' worth of state: a step, then a goal-clipped one."""
    ctx = capi.Context(cfg)
    if tiles:
        ctx.set_tiles(*tiles)
    ctx.set_state(W)
    ctx.set_time(0.3)
    dt, _ = ctx.step()
    out = [ctx.get_state()]
    goal = float(np.float32(ctx.get_time()[0] + 0.25 * dt))
    assert ctx.run(goal, 3) == (1, True)  # two inactive steps follow
    out.append(ctx.get_state())
    t = ctx.get_time()
    ctx.close()
    return dt, t, out


# one cell, one row, one column, one plane; remainders of the 4x4x4 tiles; the
# largest fused box (1024 tiles) and one more, sizes around a wave and a
# workgroup; the last below and above the limit of 400,000 cells
SIZES = [(1, 1, 1), (3, 1, 1), (1, 1, 5), (64, 1, 1), (1, 67, 1), (1, 1, 70), (17, 15, 1),
         (2, 2, 2), (4, 4, 4), (5, 6, 7), (7, 9, 4), (33, 9, 3), (16, 16, 1), (31, 33, 35),
         (64, 32, 32), (61, 30, 33), (65, 32, 32), (4100, 1, 1), (64, 72, 33), (100, 80, 50),
         (101, 80, 50)]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("recon,integrator", [(0, 0), (1, 0), (0, 1)])
def test_direct_equals_tiles(gpu_ready, n, recon, integrator):
    cfg = P.make_config(n, cfl=0.1, recon=recon, integrator=integrator)
    W = rough(cfg, 11)
    ref = run(cfg, W, (capi.TILE_32x8, capi.TILE_64x4))
    got = run(cfg, W, None)
    assert got[:2] == ref[:2]
    for a, b in zip(got[2], ref[2]):
        assert np.isfinite(b).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [(5, 4, 1), (24, 12, 9), (64, 64, 30), (90, 70, 50), (70, 70, 80)])
@pytest.mark.parametrize("fixes", [0, 7])
def test_direct_equals_tiles_shearing(gpu_ready, n, fixes):
    cfg = dict(P.config_c2(n, cfl=0.1), fixes=fixes)
    W = rough(cfg, 12)
    ref = run(cfg, W, (capi.TILE_32x8, capi.TILE_64x4))
    got = run(cfg, W, None)
    assert got[:2] == ref[:2]
    for a, b in zip(got[2], ref[2]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("recon", [0, 1])
@pytest.mark.parametrize("integrator", [0, 1])
def test_large_box_equals_its_periodic_cell(gpu_ready, recon, integrator):
    """3.51M cells, just past the size from which the tiles store past the
    caches: 4x4x4 copies of a 38^3 box do what the box does, bit for bit."""
    print("\n[case] 152^3 of 4x4x4 copies, recon %d, integrator %d" % (recon, integrator),
          flush=True)
    kw = dict(cfl=0.3, recon=recon, integrator=integrator)
    small = P.make_config((38, 38, 38), global_extent=(38 / 64,) * 3, **kw)
    large = P.make_config((152, 152, 152), global_extent=(152 / 64,) * 3, **kw)
    W = rough(small, 5)
    dt, t, out = run(small, W, None)
    dt4, t4, out4 = run(large, np.tile(W, (1, 4, 4, 4)), None)
    assert (dt, t) == (dt4, t4)
    for a, b in zip(out, out4):
        assert np.array_equal(np.tile(a, (1, 4, 4, 4)).view(np.uint32), b.view(np.uint32))


AUTO = capi.TILE_AUTO
T328, T644 = capi.TILE_32x8, capi.TILE_64x4


def test_automatic_tiles_can_be_set_again(gpu_ready):
    """get_tiles returns what set_tiles takes: setting it back changes nothing,
    and the small-box kernels, left by naming a shape, can be had again."""
    cfg = P.make_config((16, 16, 16), cfl=0.1)
    ctx = capi.Context(cfg)
    ctx.set_state(rough(cfg, 3))
    ctx.timing_enable()

    def fused():
        ctx.timing_reset()
        ctx.run(1e30, 2)
        t = ctx.timing()
        assert t["update_s2"][1] == 2
        return t["faces_s2"][1] == 0

    assert ctx.get_tiles() == (AUTO, AUTO) and fused()
    ctx.set_tiles(*ctx.get_tiles())
    assert fused()
    for tiles in ((T328, T644), (AUTO, T644), (T328, AUTO)):
        ctx.set_tiles(*tiles)
        assert ctx.get_tiles() == tiles and not fused()
    ctx.set_tiles(AUTO, AUTO)
    assert fused()
    for bad in ((-2, 0), (0, -2), (3, 0), (AUTO, 3)):
        with pytest.raises(capi.NmhdError):
            ctx.set_tiles(*bad)
    assert ctx.get_tiles() == (AUTO, AUTO)
    ctx.close()


@pytest.mark.parametrize("n", [(16, 16, 16), (65, 32, 32), (101, 80, 50)])
@pytest.mark.parametrize("tiles", [(AUTO, T644), (T328, AUTO), (AUTO, capi.TILE_16x16)])
def test_one_automatic_tile(gpu_ready, n, tiles):
    """A shape for one kernel alone: the other takes a tile too."""
    cfg = P.make_config(n, cfl=0.1)
    W = rough(cfg, 11)
    ref, got = run(cfg, W, (T328, T644)), run(cfg, W, tiles)
    assert got[:2] == ref[:2]
    for a, b in zip(got[2], ref[2]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# 850,000 cells is the last size that takes a thread per face; the frozen step
# without allocation has room for its fluxes to 687,000
@pytest.mark.parametrize("n", [(85, 100, 100), (100, 85, 101)])
@pytest.mark.parametrize("recon,integrator", [(0, 0), (1, 1)])
def test_direct_equals_tiles_at_its_limit(gpu_ready, n, recon, integrator):
    cfg = P.make_config(n, cfl=0.1, recon=recon, integrator=integrator)
    W = rough(cfg, 11)
    ref, got = run(cfg, W, (T328, T644)), run(cfg, W, None)
    assert got[:2] == ref[:2]
    for a, b in zip(got[2], ref[2]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [(100, 67, 102), (100, 67, 103), (85, 100, 100), (100, 85, 101)])
@pytest.mark.parametrize("integrator", [0, 1])
def test_noalloc_step_at_the_limits_of_direct_faces(gpu_ready, n, integrator):
    import torch
    from nmhd_amd import adjoint as A
    cfg = P.make_config(n, cfl=0.1, integrator=integrator)
    W = torch.tensor(rough(cfg, 4), device="cuda")
    S = A.Stepper(cfg)
    dt = S.cfl_dt(W)
    ref = S.forward(W, dt)
    got = A.forward_noalloc(cfg, W, dt, torch.full_like(W, float("nan")))
    assert np.array_equal(got.cpu().numpy().view(np.uint32), ref.cpu().numpy().view(np.uint32))
    S.close()


@pytest.mark.parametrize("n", [(75, 75, 75), (90, 90, 90), (100, 100, 80)])
def test_boxes_below_the_limit_are_faster_than_on_tiles(gpu_ready, n):
    """The limit lies where the faces' threads stop to pay (75^3 70 us a step
    against 80 on tiles, 90^3 103 against 116)."""
    import time
    cfg = P.make_config(n, cfl=0.1)
    W = P.orszag_tang(cfg)
    W[4] += 1.0
    ctx = [capi.Context(cfg) for _ in range(3)]
    ctx[1].set_tiles(T328, T644)
    ctx[2].set_tiles(T328, T328)
    best = [1e9] * 3
    for c in ctx:
        c.set_state(W)
        c.run(1e30, 32)
    for rep in range(6):
        for i, c in enumerate(ctx):
            t = time.perf_counter()
            c.run(1e30, 64)
            best[i] = min(best[i], time.perf_counter() - t)
    print("\n[case] %s us a step: default %.1f, tiles %.1f, %.1f" % ((n,) + tuple(
        b / 64 * 1e6 for b in best)), flush=True)
    assert best[0] < 0.97 * min(best[1:])
    for c in ctx:
        c.close()


@pytest.mark.parametrize("n", [(90, 90, 90), (84, 100, 100)])
def test_steps_past_the_goal_are_cheap(gpu_ready, n):
    """A step enqueued past the goal solves no faces (90^3: 37 us, 54 when its
    first launch did; a taken one 103).  Sizes at which the GPU, not the host's
    enqueueing, sets the time."""
    import time
    cfg = P.make_config(n, cfl=0.1)
    W = P.orszag_tang(cfg)
    W[4] += 1.0
    ctx = capi.Context(cfg)
    ctx.set_state(W)
    ctx.run(1e30, 32)

    def best(goal):
        out = []
        for rep in range(8):
            ctx.reset_run()
            t = time.perf_counter()
            ctx.enqueue_steps(goal, 32)
            k, reached = ctx.synchronize()
            out.append(time.perf_counter() - t)
        assert (k, reached) == ((32, False) if goal > 1e29 else (1, True))
        return min(out)

    taken = best(1e30)
    state = ctx.get_state()
    past = best(ctx.get_time()[0])
    print("\n[case] %s: 32 steps taken %.0f us, past the goal %.0f" % (n, taken * 1e6, past * 1e6),
          flush=True)
    assert past < 0.45 * taken
    # the one taken is of size zero, or what t lacks to the goal in float
    assert np.allclose(ctx.get_state(), state, rtol=1e-3, atol=1e-4)
    ctx.close()
