"""Step bookkeeping between enqueued steps and device state transfers (GPU).

The first kernel of a step commits the previous one and decides dt; a run
must not depend on how its steps were enqueued, nor on steps enqueued after
it reached its goal.
"""
import numpy as np
import pytest

from nmhd_amd import capi, problems as P

pytestmark = pytest.mark.gpu


def boxes():
    shear = P.config_c2((24, 12, 9))
    ghosts_z = P.make_config((20, 12, 10), margin=(0, 2, 3), cfl=0.4)
    euler = P.make_config((17, 9, 5), cfl=0.4, recon=1, integrator=1)
    return [("shear", shear, P.shearing_box_mri(shear)),
            ("periodic", P.config_c1(16), P.orszag_tang_noisy(P.config_c1(16))),
            ("ghost_z", ghosts_z, P.orszag_tang_noisy(ghosts_z)),
            ("euler", euler, P.orszag_tang_noisy(euler))]


@pytest.mark.parametrize("path", [capi.PATH_TILED, capi.PATH_STRICT])
@pytest.mark.parametrize("box", range(4))
def test_enqueueing_does_not_matter(gpu_ready, box, path):
    name, cfg, W = boxes()[box]
    whole, single, split = (capi.Context(cfg, path=path) for _ in range(3))
    for c in (whole, single, split):
        c.set_state(W)
        c.set_time(0.2)
    k, reached = whole.run(1e30, 7)
    assert (k, reached) == (7, False)
    for _ in range(7):
        single.step()
    split.reset_run()
    split.enqueue_steps(1e30, 3)
    split.enqueue_steps(1e30, 0)
    split.enqueue_steps(1e30, 4)
    assert split.synchronize() == (7, False)
    t, g = whole.get_time()
    assert g == 7 and single.get_time() == (t, g) and split.get_time() == (t, g)
    ref = whole.get_state()
    for c in (single, split):
        assert np.array_equal(ref.view(np.uint32), c.get_state().view(np.uint32)), name
    # a goal reached inside an enqueued group: the rest of it (an even or an
    # odd number of steps) changes nothing, and the next run goes on from there
    dt, _ = single.step()
    goal = float(np.float32(single.get_time()[0] + 1.5 * dt))
    steps = []
    for c, extra in ((whole, 8), (split, 9)):
        c.run(1e30, 1)
        c.reset_run()
        c.enqueue_steps(goal, extra)
        k, reached = c.synchronize()
        assert reached
        steps.append(k)
    n = 0
    while True:
        n += 1
        if single.step(goal)[1]:
            break
    assert steps == [n, n]
    for c in (whole, single, split):
        assert c.get_time()[0] == pytest.approx(goal, abs=1e-12 + abs(goal) * 2 ** -23)
        assert c.run(1e30, 3) == (3, False)
    ref = whole.get_state()
    for c in (single, split):
        assert whole.get_time() == c.get_time()
        assert np.array_equal(ref.view(np.uint32), c.get_state().view(np.uint32)), name
        assert np.isfinite(ref).all()
    for c in (whole, single, split):
        c.close()


@pytest.mark.parametrize("path", [capi.PATH_TILED, capi.PATH_STRICT])
@pytest.mark.parametrize("box", range(4))
def test_state_loaded_after_the_goal(gpu_ready, box, path):
    """Steps enqueued without a new run after the goal was reached do nothing,
    also where a state was loaded in between: the next run's dt is that of the
    loaded state alone, not of the one before it, of the ghost rows it came
    with, of those steps' goal, nor (after the strict path) none at all."""
    name, cfg, W = boxes()[box]
    a, b = capi.Context(cfg, path=path), capi.Context(cfg, path=capi.PATH_TILED)
    a.set_state(W)
    dt, _ = a.step()
    assert a.run(float(np.float32(a.get_time()[0] + 0.5 * dt)), 1) == (1, True)
    a.set_path(capi.PATH_TILED)
    X = W.copy()
    X[4] *= 2.0
    m = cfg["m"]
    ny, nz = cfg["n"][1], cfg["n"][2]
    X[4][nz // 2, ny // 2] *= 4.0  # rows that no ghost row copies
    X[4][:, [y for y in range(ny) if y < m[1] or y >= ny - m[1]], :] *= 100.0
    X[4][[z for z in range(nz) if z < m[2] or z >= nz - m[2]]] *= 100.0
    a.set_state(X)
    a.enqueue_steps(1e-6, 3)
    a.synchronize()
    assert np.array_equal(a.get_state().view(np.uint32), X.view(np.uint32)), name
    b.set_state(X)
    b.set_time(*a.get_time())
    for _ in range(2):
        assert a.step()[0] == b.step()[0], name
    assert np.array_equal(a.get_state().view(np.uint32), b.get_state().view(np.uint32)), name
    a.close()
    b.close()


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (5, 3, 1), (17, 9, 7), (64, 32, 16)])
@pytest.mark.parametrize("offset", [0, 1, 2, 4])
def test_device_state_transfer(gpu_ready, n, offset):
    """set_state_device / get_state_device at every alignment of the fields,
    with nothing written outside them."""
    import torch
    ctx = capi.Context(P.make_config(n))
    nc = ctx.ncell
    stride = nc + 5
    src = torch.rand(8 * stride + 8, device="cuda")
    dst = torch.full_like(src, -1.0)
    torch.cuda.synchronize()
    start = [offset + f * stride for f in range(8)]
    ctx.set_state_device([src.data_ptr() + 4 * s for s in start])
    ctx.get_state_device([dst.data_ptr() + 4 * s for s in start])
    host = ctx.get_state().reshape(8, nc)
    a, d = src.cpu().numpy(), dst.cpu().numpy()
    inside = np.zeros(d.size, bool)
    for f, s in enumerate(start):
        assert np.array_equal(host[f], a[s:s + nc]) and np.array_equal(d[s:s + nc], a[s:s + nc])
        inside[s:s + nc] = True
    assert (d[~inside] == -1.0).all()
    ctx.close()


def test_device_state_transfer_after_another_call_failed(gpu_ready):
    """An error that an earlier HIP call of the program left behind is not that
    of a transfer or of set_time."""
    ctx = capi.Context(P.make_config((4, 2, 2)))
    import torch
    W = torch.rand(8, 16, device="cuda")
    torch.cuda.synchronize()
    ptrs = [W[f].data_ptr() for f in range(8)]
    for call in (lambda: ctx.set_state_device(ptrs), lambda: ctx.get_state_device(ptrs),
                 lambda: ctx.set_time(0.5, 3)):
        assert capi.load().hipSetDevice(10000) != 0
        call()
    assert np.array_equal(ctx.get_state().reshape(8, 16), W.cpu().numpy())
    assert ctx.get_time() == (0.5, 3)
    ctx.close()


def test_device_state_transfer_outside_an_allocation(gpu_ready):
    """A field that runs past the end of its allocation is refused, as a copy
    refuses it: here by half its 64 bytes, which still lie in the page."""
    import ctypes
    ctx = capi.Context(P.make_config((4, 2, 2)))
    W = np.arange(8 * 16, dtype=np.float32).reshape(8, 2, 2, 4) + 1.0
    ctx.set_state(W)
    L = capi.load()
    buf = ctypes.c_void_p()
    size = 3584
    assert L.hipMalloc(ctypes.byref(buf), ctypes.c_size_t(size)) == 0
    whole = [buf.value + 64 * f for f in range(8)]
    ctx.get_state_device(whole)
    for f in (0, 7):
        ptrs = list(whole)
        ptrs[f] = buf.value + size - 32
        with pytest.raises(capi.NmhdError):
            ctx.set_state_device(ptrs)
        ctx.set_state(W)
        with pytest.raises(capi.NmhdError):
            ctx.get_state_device(ptrs)
    # the last place where it fits
    ptrs = whole[:7] + [buf.value + size - 64]
    ctx.get_state_device(ptrs)
    ctx.set_state(W + 1.0)
    ctx.set_state_device(ptrs)
    assert np.array_equal(ctx.get_state(), W)
    ctx.close()
    assert L.hipFree(buf) == 0


@pytest.mark.parametrize("shift", [0, 3, 15, 16])
def test_device_state_fields_that_overlap(gpu_ready, shift):
    """Fields fetched into arrays that overlap: the later field's values stay,
    as after a copy per field in turn."""
    import torch
    ctx = capi.Context(P.make_config((4, 2, 2)))
    W = np.arange(8 * 16, dtype=np.float32).reshape(8, 2, 2, 4) + 1.0
    ctx.set_state(W)
    dst = torch.full((8 * 16,), -1.0, device="cuda")
    torch.cuda.synchronize()
    ctx.get_state_device([dst.data_ptr() + 4 * shift * f for f in range(8)])
    want = np.full(8 * 16, -1.0, np.float32)
    for f in range(8):
        want[shift * f:shift * f + 16] = W[f].reshape(-1)
    assert np.array_equal(dst.cpu().numpy(), want)
    # the same arrays may all be read
    ctx.set_state_device([dst.data_ptr() + 4 * shift * f for f in range(8)])
    got = ctx.get_state().reshape(8, 16)
    for f in range(8):
        assert np.array_equal(got[f], want[shift * f:shift * f + 16])
    ctx.close()


@pytest.mark.parametrize("n,margin", [((24, 12, 9), 4), ((1, 3, 1), 1), ((5, 2, 2), 2),
                                      ((70, 4, 3), 4), ((33, 9, 17), 3)])
@pytest.mark.parametrize("fixes,shear_y", [(0, 1), (7, 1), (2, 1), (1, 0)])
def test_ghost_fill_reduces_the_cfl_minimum(gpu_ready, n, margin, fixes, shear_y):
    """The fill adds the ghost cells' CFL times as it writes them: every dt
    equals that of a full pass over the same state, bit for bit, with the
    shortest CFL time in the ghost rows (their interior sources are fast
    where the shear makes them faster still)."""
    cfg = P.make_config(n, margin=(0, margin, 0), cfl=0.1, source=1, shear_y=shear_y)
    cfg["fixes"] = fixes
    W = P.shearing_box_mri(cfg, amp=0.2)
    a, b = capi.Context(cfg), capi.Context(cfg)
    a.set_state(W)
    a.set_time(0.7)
    for _ in range(4):
        b.set_state(a.get_state())
        b.set_time(*a.get_time())
        dt_full, _ = b.step()  # after set_state: a full pass
        assert a.step()[0] == dt_full
        assert np.array_equal(a.get_state().view(np.uint32), b.get_state().view(np.uint32))
    a.close()
    b.close()
