"""Batched boxes (nmhd_batch_*): many boxes of uneven sizes (periodic or
shearing) in per-tile-shape or persistent launches over a work table,
per-box dt and ghost fills, HIP-graph replay and the autotuner.

The batched kernels run the single-box tile functions, and a cell's
arithmetic does not depend on the tiling, so the invariant checked here is
bit-identity: a box advanced in a batch (eager or graph, any tile shape, z
chunk, launch mode or workgroup count, tuned or not) equals the same box advanced alone
by a Context on the tiled path, state and time, bit for bit.  The tiled path
itself is checked against the oracle in test_gpu_parity.py; one batched box
is compared with the oracle here as well.
"""
import os

import numpy as np
import pytest

import pyoracle as po
from mhd_checks import bitwise_equal, div_b, group_rel_err, perturb_ulps
from nmhd_amd import capi, problems as P

pytestmark = pytest.mark.gpu

SMALL = [(16, 24, 8), (32, 16, 16), (24, 24, 24), (48, 16, 8), (16, 16, 32), (64, 8, 12)]


def announce(msg):
    print("\n[case] " + msg, flush=True)


def small_boxes(seed=11):
    out = []
    for b, shape in enumerate(SMALL):
        cfg = P.make_config(shape, cfl=0.4)
        if b % 2 == 0:
            W = P.orszag_tang_noisy(cfg, seed=seed + b, b0=0.3 + 0.05 * b)
        else:
            u = P.uniform01(seed, b, 0)
            W = P.blast(cfg, (float(np.cos(6.0 * u)), float(np.sin(6.0 * u)), 0.3))
        out.append((cfg, W))
    return out


def make_batch(boxes):
    B = capi.Batch([c for c, _ in boxes])
    for i, (_, W) in enumerate(boxes):
        B.set_state(i, W)
    return B


def single_runs(boxes, goal, nsteps):
    out = []
    for cfg, W in boxes:
        g = capi.Context(cfg, path=capi.PATH_TILED)
        g.set_state(W)
        k, _ = g.run(goal, nsteps)
        out.append((g.get_state(), g.get_time(), k))
        g.close()
    return out


def assert_batch_equals(B, ref):
    for i, (W, (t, gen), k) in enumerate(ref):
        got = B.get_state(i)
        assert bitwise_equal(got, W), "box %d state differs" % i
        tb, gb = B.get_time(i)
        assert tb == t and gb == gen, (i, tb, t, gb, gen)


def test_batch_eager_equals_single_boxes(gpu_ready):
    announce("batch eager 6 boxes x 5 steps vs single contexts")
    boxes = small_boxes()
    ref = single_runs(boxes, 1e30, 5)
    B = make_batch(boxes)
    k, reached = B.run(1e30, 5, use_graph=False)
    assert k == 5 and not reached
    assert_batch_equals(B, ref)
    # the boxes took different dt
    dts = {B.status(i)[2] for i in range(B.nbox)}
    assert len(dts) > 1


def shearing_mix():
    """Shearing boxes of uneven sizes (one with vertical ghost planes too,
    one with all three quirk corrections, one with first-order
    reconstruction) mixed with periodic boxes (one first-order)."""
    out = []
    for k, shape in enumerate([(16, 16, 8), (24, 16, 16), (32, 24, 8)]):
        cfg = P.config_c2(shape)
        if k == 2:
            cfg = dict(cfg, fixes=capi.FIX_ALL)
        out.append((cfg, P.shearing_box_mri(cfg, seed=40 + k)))
    cfg = P.make_config((16, 24, 8), margin=(0, 4, 2), cfl=0.4, source=1, shear_y=1)
    out.append((cfg, P.shearing_box_mri(cfg, seed=44)))
    # first-order reconstruction in one shearing and one periodic box
    cfg = dict(P.config_c2((16, 16, 16)), recon=1)
    out.append((cfg, P.shearing_box_mri(cfg, seed=45)))
    per = small_boxes(seed=31)[:3]
    per[1] = (dict(per[1][0], recon=1), per[1][1])
    return out + per


def test_batch_shearing_boxes_equal_single_boxes(gpu_ready):
    """Shearing boxes in a batch (per-box shear remap of the radial ghost
    rows at each box's own time, periodic vertical ghost planes, the ghost
    cells' CFL added to each box's minimum), mixed with periodic boxes:
    every box equals its single-box tiled context bit for bit, eagerly and
    replayed from the graph, and across a goal that some boxes reach."""
    announce("batch of shearing and periodic boxes vs single contexts")
    boxes = shearing_mix()
    ref = single_runs(boxes, 1e30, 6)
    B = make_batch(boxes)
    k, _ = B.run(1e30, 3, use_graph=False)
    assert k == 3
    k, _ = B.run(1e30, 3, use_graph=True)
    assert k == 3
    assert_batch_equals(B, ref)
    # a goal ahead of every box's time: each box clips its own last step
    # and stops there
    goal = max(t for _, (t, _), _ in ref) + 0.02
    ref2 = []
    for (cfg, W), (Wr, (t, gen), _) in zip(boxes, ref):
        g = capi.Context(cfg, path=capi.PATH_TILED)
        g.set_state(Wr)
        g.set_time(t, gen)
        g.run(goal, 5)
        ref2.append((g.get_state(), g.get_time(), 0))
        g.close()
    B.run(goal, 5)
    assert_batch_equals(B, ref2)
    reached = [B.status(i)[1] for i in range(B.nbox)]
    assert any(reached), reached
    B.close()


def test_batch_with_cfl_speed_fix_equals_single_boxes(gpu_ready):
    """Boxes with NMHD_FIX_CFL_SPEED (|v| + c) in a batch, mixed with boxes
    without it: each equals its single-box tiled context bit for bit, and the
    fixed boxes take their own, shorter steps (each box record carries its
    own corrections; a bulk flow of -0.3 along x makes |v| + c exceed
    |v + c| in the fastest cells)."""
    announce("batch with per-box CFL-speed fix")
    boxes = []
    for i, (cfg, W) in enumerate(small_boxes(seed=23)):
        if i % 2:
            W = W.copy()
            W[1] -= np.float32(0.3)
            cfg = dict(cfg, fixes=capi.FIX_CFL_SPEED)
        boxes.append((cfg, W))
    ref = single_runs(boxes, 1e30, 4)
    B = make_batch(boxes)
    k, _ = B.run(1e30, 4)
    assert k == 4
    assert_batch_equals(B, ref)
    plain = single_runs([(dict(c, fixes=0), W) for c, W in boxes], 1e30, 4)
    for i in range(1, len(boxes), 2):
        assert ref[i][1][0] < plain[i][1][0], i


def test_batch_graph_equals_eager(gpu_ready):
    announce("batch graph vs eager, 7 + 4 steps (every rotation phase, replays)")
    boxes = small_boxes(seed=3)
    A = make_batch(boxes)
    G = make_batch(boxes)
    A.run(1e30, 7, use_graph=False)
    G.run(1e30, 7, use_graph=True)
    for i in range(A.nbox):
        assert bitwise_equal(A.get_state(i), G.get_state(i)), i
    A.run(1e30, 4, use_graph=False)
    G.run(1e30, 4, use_graph=True)
    ref = single_runs(boxes, 1e30, 11)
    assert_batch_equals(G, ref)
    assert_batch_equals(A, ref)


@pytest.mark.parametrize("ft,ut,fz,uz,fw,uw", [
    (capi.TILE_64x4, capi.TILE_64x4, 8, 32, 1, 4),
    (capi.TILE_32x8, capi.TILE_16x16, 5, 7, 3, 1),
    (capi.TILE_16x16, capi.TILE_32x8, 32, 3, 2, 2),
    (capi.TILE_32x8, capi.TILE_64x4, 8, 16, 0, 0),
    (capi.TILE_64x4, capi.TILE_16x16, 3, 8, 0, 3),
    (capi.TILE_16x16, capi.TILE_32x8, 16, 5, 2, 0),
    (capi.TILE_32x8, capi.TILE_64x4, 1, 2, 0, 0),
    (capi.TILE_16x16, capi.TILE_32x8, 2, 1, 2, 2),
])
def test_batch_tilings_bit_identical(gpu_ready, ft, ut, fz, uz, fw, uw):
    announce("batch tiling faces %d update %d zc %d/%d wg %d/%d" % (ft, ut, fz, uz, fw, uw))
    boxes = small_boxes(seed=5)
    ref = single_runs(boxes, 1e30, 3)
    B = make_batch(boxes)
    B.set_tiles(ft, ut)
    B.set_launch(fz, uz, fw, uw)
    B.run(1e30, 3, use_graph=True)
    assert_batch_equals(B, ref)


@pytest.mark.parametrize("fw,uw", [(0, 0), (2, 2)])
def test_batch_mixed_tile_shapes_bit_identical(gpu_ready, fw, uw):
    announce("batch with a different tile shape per box, wg %d/%d" % (fw, uw))
    boxes = small_boxes(seed=9)
    ref = single_runs(boxes, 1e30, 3)
    B = make_batch(boxes)
    for i in range(B.nbox):
        B.set_tiles(i % 3, (i + 1) % 3, box=i)
    B.set_launch(8, 16, fw, uw)
    B.run(1e30, 3, use_graph=True)
    assert_batch_equals(B, ref)


def test_batch_per_box_goal_clipping(gpu_ready):
    announce("batch goal clipping: boxes reach the goal at different steps")
    boxes = small_boxes(seed=8)
    # a goal that some boxes reach within 6 steps and others do not
    probe = make_batch(boxes)
    probe.run(1e30, 1, use_graph=False)
    dts = sorted(probe.status(i)[2] for i in range(probe.nbox))
    goal = float(np.float32(3.5 * dts[len(dts) // 2]))
    ref = single_runs(boxes, goal, 6)
    B = make_batch(boxes)
    kmin, all_reached = B.run(goal, 6, use_graph=True)
    assert_batch_equals(B, ref)
    reached = [B.status(i)[1] for i in range(B.nbox)]
    assert any(reached) and not all(reached)
    for i, r in enumerate(reached):
        t, _ = B.get_time(i)
        if r:
            assert t == pytest.approx(goal, rel=0, abs=1e-6)
    assert kmin == min(k for _, _, k in ref)


def test_batch_autotune_cached_and_identical(gpu_ready, tmp_path):
    announce("batch autotune (cache in tmp) and results after tuning")
    boxes = small_boxes(seed=9)
    ref = single_runs(boxes, 1e30, 3)
    B = make_batch(boxes)
    cache = str(tmp_path / "tune.txt")
    n1 = B.autotune(cache)
    assert n1 == len(set(SMALL))
    assert os.path.exists(cache)
    text = open(cache).read()
    assert text.count("\nshape ") == len(set(SMALL)) and "\nlaunch " in text
    B2 = make_batch(boxes)
    assert B2.autotune(cache) == 0  # every shape from the cache
    assert B2.get_launch() == B.get_launch()
    B.run(1e30, 3, use_graph=True)
    assert_batch_equals(B, ref)


def test_batch_box_against_oracle(gpu_ready):
    announce("batched box vs oracle, 3 steps")
    cfg = P.make_config((16, 24, 8), cfl=0.4)
    W = P.orszag_tang_noisy(cfg, seed=21)
    other_cfg = P.make_config((32, 16, 16), cfl=0.4)
    B = capi.Batch([other_cfg, cfg])
    B.set_state(0, P.orszag_tang(other_cfg))
    B.set_state(1, W)
    B.run(1e30, 3, use_graph=True)
    o = po.Oracle(cfg, W)
    o.run(1e30, 3)
    got, want = B.get_state(1), o.get_state()
    errs = group_rel_err(got, want)
    assert errs.max() < 1e-3, errs
    assert B.get_time(1)[0] == pytest.approx(o.time, rel=1e-6)
    bmax = np.abs(got[5:8]).max()
    assert np.abs(div_b(got, cfg["d"])).max() * max(cfg["d"]) < 1e-6 * bmax



def test_batch_thin_boxes_equal_single_boxes(gpu_ready):
    """Boxes one cell thick (the reference's shock-tube demo along x, y and
    z, 128 cells long, one with first-order reconstruction) next to a 3D box:
    tiles far wider than the box, periodic wrap onto the same cell."""
    announce("batch of thin shock-tube boxes + a 3D box vs single contexts")
    boxes = [P.shock_tube(0, 128), P.shock_tube(1, 128), P.shock_tube(2, 128, recon=1)]
    cfg, W = P.shock_tube(1, 64)
    boxes.append((cfg, W))
    boxes.append(small_boxes()[2])
    ref = single_runs(boxes, 0.05, 20)
    B = make_batch(boxes)
    B.run(0.05, 20, use_graph=True)
    assert_batch_equals(B, ref)


def test_c4_workload_autotuned_graph_steps(gpu_ready, tmp_path):
    """The multi-box workload itself: 64 boxes of edges from {16, ..., 96}
    (seed 1004; Orszag-Tang and blast boxes), autotuned, then 5 steps
    replayed from the captured graph.  Every box equals a single-box tiled
    context bit for bit (state and time), and two Orszag-Tang and two blast
    boxes stay within three times the oracle's own one-ulp sensitivity of
    the oracle (both states are mirror symmetric, so CT upwind sums are
    exactly zero on whole rows of edges and their choice is a round-off
    tie)."""
    announce("C4: 64 boxes, autotune, 5 graph steps vs single contexts and oracle")
    boxes = P.batch_boxes(seed=1004, nbox=64)
    B = make_batch(boxes)
    B.autotune(str(tmp_path / "tune.txt"))
    print("launch (faces zchunk, update zchunk, faces wg/CU, update wg/CU):", B.get_launch(),
          flush=True)
    k, reached = B.run(1e30, 5, use_graph=True)
    assert k == 5 and not reached
    ref = single_runs(boxes, 1e30, 5)
    assert_batch_equals(B, ref)
    checked = {0: [], 1: []}
    for i, (cfg, W) in enumerate(boxes):
        kind = i % 2
        if len(checked[kind]) == 2:
            continue
        o = po.Oracle(cfg, W)
        o2 = po.Oracle(cfg, perturb_ulps(W))
        o.run(1e30, 5)
        o2.run(1e30, 5)
        want = o.get_state()
        env = group_rel_err(o2.get_state(), want)
        err = group_rel_err(B.get_state(i), want)
        print("box %d %s %s: err %s, oracle 1-ulp envelope %s"
              % (i, "OT" if kind == 0 else "blast", cfg["global_size"],
                 np.array2string(err, precision=2), np.array2string(env, precision=2)))
        assert np.all(err <= 3.0 * env + 1e-6), (i, err, env)
        # the dt sequence follows the state's round-off ties: 1e-5 per step
        assert B.get_time(i)[0] == pytest.approx(o.time, rel=1e-5)
        checked[kind].append(i)
    assert len(checked[0]) == len(checked[1]) == 2


def test_batch_second_run_after_goal(gpu_ready):
    """Boxes that reached the goal keep the CFL minimum of their last active
    step through the trailing inactive steps, so a second run to a later goal
    takes the same steps as single contexts whose second run recomputes the
    CFL over the whole box."""
    announce("batch run(g1) then run(g2) vs single contexts")
    boxes = small_boxes(seed=8)
    probe = make_batch(boxes)
    probe.run(1e30, 1, use_graph=False)
    dts = sorted(probe.status(i)[2] for i in range(probe.nbox))
    g1 = float(np.float32(3.5 * dts[len(dts) // 2]))
    g2 = float(np.float32(2.0 * g1))
    ref = []
    for cfg, W in boxes:
        g = capi.Context(cfg, path=capi.PATH_TILED)
        g.set_state(W)
        g.run(g1, 40)
        g.set_path(capi.PATH_TILED)  # the second run starts from a full CFL pass
        k, _ = g.run(g2, 40)
        ref.append((g.get_state(), g.get_time(), k))
        g.close()
    B = make_batch(boxes)
    B.run(g1, 40, use_graph=True)
    assert all(B.status(i)[1] for i in range(B.nbox))
    B.run(g2, 40, use_graph=True)
    assert_batch_equals(B, ref)
    for i in range(B.nbox):
        assert B.status(i)[0] == ref[i][2], i


@pytest.mark.parametrize("integrator", [0, 1])
@pytest.mark.parametrize("ft,launch", [(None, None), (capi.TILE_64x4, (1, 1, 0, 0)),
                                       (capi.TILE_16x16, (5, 3, 0, 0)), (None, (2, 3, 1, 1))])
def test_batch_opened_steps_and_carried_boxes(gpu_ready, integrator, ft, launch):
    """Steps opened inside the first face launch, boxes that stop at the goal
    carried by the last update, at tile edges and chunk remainders, both
    reconstructions in one table; eager and graph steps alternate over the
    three rotation phases, and a second run goes on."""
    announce("batch steps, integrator %d, tiles %s, launch %s" % (integrator, ft, launch))
    shapes = [(17, 9, 1), (33, 8, 5), (16, 16, 16), (64, 4, 3), (1, 40, 7)]
    boxes = []
    for i, n in enumerate(shapes):
        cfg = P.make_config(n, cfl=0.4, integrator=integrator, recon=i % 2)
        boxes.append((cfg, P.orszag_tang_noisy(cfg, seed=40 + i, b0=0.3)))
    probe = make_batch(boxes)
    probe.run(1e30, 1, use_graph=False)
    dts = sorted(probe.status(i)[2] for i in range(probe.nbox))
    g1 = float(np.float32(2.5 * dts[len(dts) // 2]))
    ref = []
    for cfg, W in boxes:
        g = capi.Context(cfg, path=capi.PATH_TILED)
        g.set_state(W)
        g.run(g1, 5)
        k, _ = g.run(2 * g1, 6)
        ref.append((g.get_state(), g.get_time(), k))
        g.close()
    B = make_batch(boxes)
    if ft is not None:
        B.set_tiles(ft, ft)
    if launch is not None:
        B.set_launch(*launch)
        assert B.get_launch() == launch
    B.run(g1, 5, use_graph=True)
    reached = [B.status(i)[1] for i in range(B.nbox)]
    assert any(reached)
    B.run(2 * g1, 6, use_graph=False)
    assert_batch_equals(B, ref)
    assert [B.status(i)[0] for i in range(B.nbox)] == [k for _, _, k in ref]


@pytest.mark.parametrize("n", [(5, 3, 2), (64, 64, 31), (64, 64, 32), (64, 64, 33)])
def test_batch_state_into_any_memory(gpu_ready, n):
    """Fields fetched into pageable, pinned or device arrays, and into some of
    each, on both sides of the size from which pinned ones are copied to
    directly."""
    import ctypes
    import torch
    announce("batch get_state of %s into pageable, pinned and device memory" % (n,))
    cfg = P.make_config(n)
    W = np.random.default_rng(3).random((8, n[2], n[1], n[0]), np.float32)
    B = make_batch([(cfg, W)])
    kinds = [lambda: torch.zeros(W[0].size), lambda: torch.zeros(W[0].size, pin_memory=True),
             lambda: torch.zeros(W[0].size, device="cuda")]
    for case in ([0] * 8, [1] * 8, [2] * 8, [0, 1, 2, 0, 1, 2, 0, 1], [1, 1, 1, 0, 1, 1, 1, 1]):
        out = [kinds[k]() for k in case]
        torch.cuda.synchronize()
        ptrs = capi._ptrs([t.data_ptr() for t in out])
        assert capi.load().nmhd_batch_get_state(B.h, 0, ptrs) == 0
        for f in range(8):
            assert bitwise_equal(out[f].cpu().numpy().reshape(W[f].shape), W[f]), (case, f)
    B.close()


def test_batch_state_into_pinned_memory_is_one_copy(gpu_ready):
    """A large box fetched into pinned arrays goes there directly (1.3 ms for
    128^3; 2.3 through the buffer that pageable arrays need, which takes 2.4)."""
    import time
    import torch
    announce("batch get_state of 128^3, pinned against pageable")
    B = capi.Batch([P.make_config((128, 128, 128))])
    best = []
    for pin in (False, True):
        out = torch.ones((8, 128 ** 3), pin_memory=pin)
        ptrs = capi._ptrs([out[f].data_ptr() for f in range(8)])
        times = []
        for _ in range(8):
            t = time.perf_counter()
            assert capi.load().nmhd_batch_get_state(B.h, 0, ptrs) == 0
            times.append(time.perf_counter() - t)
        best.append(min(times))
    print("pageable %.0f us, pinned %.0f us" % (best[0] * 1e6, best[1] * 1e6), flush=True)
    assert best[1] < 0.8 * best[0]
    B.close()


def test_batch_default_tiling_can_be_set_again(gpu_ready):
    """Chunks of 0 and automatic tiles give back the tiling of a new batch."""
    announce("batch tiling set and set back")
    boxes = small_boxes(seed=17)
    ref = single_runs(boxes, 1e30, 4)
    B = make_batch(boxes)
    fresh = B.get_launch()
    B.set_tiles(capi.TILE_64x4, capi.TILE_16x16)
    B.set_launch(29, 31, 1, 0)
    assert B.get_launch() == (29, 31, 1, 0)
    B.run(1e30, 2)
    B.set_launch(0, 7, 0, 0)
    assert B.get_launch()[1:] == (7, 0, 0)
    B.set_launch(0, 0, 0, 0)
    B.set_tiles(capi.TILE_AUTO, capi.TILE_AUTO)
    assert B.get_launch() == fresh
    B.run(1e30, 2)
    assert_batch_equals(B, ref)
    for bad in ((-1, 1, 0, 0), (1, -1, 0, 0)):
        with pytest.raises(capi.NmhdError):
            B.set_launch(*bad)
    with pytest.raises(capi.NmhdError):
        B.set_tiles(-2, 0)
    B.close()


@pytest.fixture(scope="module")
def large_mix():
    """3.61M cells, just past the 3.5M from which the batch kernels store past
    the caches: a periodic, a shearing and a small first-order box, with their
    single-box results after 3 steps."""
    boxes = []
    cfg = P.make_config((128, 128, 128), cfl=0.4)
    boxes.append((cfg, P.orszag_tang_noisy(cfg, seed=51)))
    cfg = P.config_c2((112, 112, 112))
    boxes.append((cfg, P.shearing_box_mri(cfg, seed=52)))
    cfg = P.make_config((33, 20, 17), cfl=0.4, recon=1)
    boxes.append((cfg, P.orszag_tang_noisy(cfg, seed=53)))
    assert sum(P.ncell(c) for c, _ in boxes) > 3500000
    return boxes, single_runs(boxes, 1e30, 3)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("launch", [(0, 0, 0, 0), (16, 7, 2, 3), (5, 16, 0, 3), (16, 16, 4, 0)])
def test_batch_past_the_caches(gpu_ready, large_mix, launch, wide):
    """A workgroup per item and walking workgroups, with and without 64x4 face
    tiles, in a batch past the size from which results go past the caches
    (small_boxes' tests run the same launches through them)."""
    announce("large batch, launch %s, 64x4 face tiles %s" % (launch, wide))
    boxes, ref = large_mix
    B = make_batch(boxes)
    B.set_tiles(capi.TILE_16x16, capi.TILE_64x4, box=1)
    B.set_tiles(capi.TILE_64x4 if wide else capi.TILE_32x8, capi.TILE_32x8, box=2)
    B.set_launch(*launch)
    B.run(1e30, 1, use_graph=False)
    B.run(1e30, 2, use_graph=True)
    assert_batch_equals(B, ref)
    B.close()


def test_batch_chunks_fill_the_rounds_of_64x4_tiles(gpu_ready):
    """Three workgroups of 64x4 face tiles share a CU, four of the other
    shapes: 768 are resident, and a chunk that makes 1000 of them waits for a
    second round (64x4x2000 cells: the faces take 35 us, 30 with 667)."""
    announce("face chunk of 64x4 tiles")
    B = capi.Batch([P.make_config((64, 4, 2000))])
    B.set_tiles(capi.TILE_64x4, capi.TILE_64x4)
    assert 512 < -(-2000 // B.get_launch()[0]) <= 768
    B.set_tiles(capi.TILE_32x8, capi.TILE_64x4)
    assert 768 < 2 * -(-2000 // B.get_launch()[0]) <= 1024
    B.close()


def test_batch_autotune_drops_other_kernels_entries(gpu_ready, tmp_path):
    """A cache file whose entries carry no version of the kernels, or values
    that name no tiling, is tuned anew."""
    import torch
    announce("autotune with entries of other kernels in the cache")
    boxes = small_boxes(seed=9)
    arch = torch.cuda.get_device_properties(0).gcnArchName.split(":")[0]
    cache = tmp_path / "tune.txt"
    cache.write_text("".join("shape %s %d %d %d 0 0 : 0 2\n" % ((arch,) + n) for n in SMALL))
    B = make_batch(boxes)
    assert B.autotune(str(cache)) == len(set(SMALL))
    lines = cache.read_text().splitlines()
    assert B.autotune(str(cache)) == 0
    cache.write_text("\n".join(l.split(" : ")[0] + " : 7 1" if l.startswith("shape") else l
                               for l in lines))
    assert B.autotune(str(cache)) == len(set(SMALL))
    B.close()


@pytest.mark.parametrize("nbox", [14, 64])
def test_batch_autotune_is_not_slower_than_the_default(gpu_ready, tmp_path, nbox):
    """The default tiling is one of the tuner's candidates, timed as a step
    runs it (64 boxes: 797 us a step tuned, 757 by default, when it was not)."""
    import time
    announce("autotuned against default, %d boxes" % nbox)
    boxes = P.batch_boxes(seed=1004, nbox=nbox)
    batches = [make_batch(boxes) for _ in range(2)]
    batches[1].autotune(str(tmp_path / "tune.txt"))
    best = [1e9, 1e9]
    for rep in range(6):
        for i, B in enumerate(batches):
            t = time.perf_counter()
            B.run(1e30, 40)
            best[i] = min(best[i], time.perf_counter() - t)
    print("default %.0f us a step, tuned %.0f, %s" % (best[0] / 40 * 1e6, best[1] / 40 * 1e6,
                                                      batches[1].get_launch()), flush=True)
    assert best[1] < 1.03 * best[0]
    for B in batches:
        B.close()
