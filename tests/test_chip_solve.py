"""The SOR solve held on the chip (one launch, les_sor_res.hip) against the colour sweeps, bit for
bit: cuts with one and several workgroups along j and k, partial top level blocks and last rows,
colour rows with padding, odd jp (the periodic seam joins cells of one colour), every number of
levels per thread with one and with several level blocks; the queue form that serves it when its workgroups cannot all be
resident; two handles taking turns on one device; and the residual with the early exit."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

FIELDS = ("p", "u", "v", "w", "rhs")


def _handle(dims, nmaxp, sweeps, dx=4.0, pjuge=0.0):
    from les_halo_amd import LES, inputs
    L = LES(*dims, **common.REF_PHYS, omega=1.5, pjuge=pjuge, nmaxp=nmaxp)
    L.load_case(inputs.make_case(*dims, seed=5, hmax=20.0, dx=dx))
    L.ifdata()
    if sweeps:
        L.set_sor_tile(0)
    return L


def _same(a, b, names=FIELDS):
    for nm in names:
        x, y = a.download(nm), b.download(nm)
        assert common.bits_equal(x, y), common.mismatch_report(x, y, nm)
    assert np.abs(a.download("p")).max() > 0


def _ran(h, solves, queued=0):
    """The solves that were to run on the chip did, and in the form that was to be tested."""
    i = h.solve_info()
    assert (i["solves"], i["queued"], i["on_chip"], i["given_up"]) == (solves, queued, 1, 0), i


# 1 workgroup; level blocks in one workgroup, the last partial; several along k; along j and k
# with a partial top block; odd jp in one tile and in several; ip > 320; 9 levels a thread
GRIDS = [(16, 12, 10), (31, 18, 17), (48, 48, 32), (150, 44, 61), (35, 27, 19), (20, 5, 7),
         (147, 133, 61), (512, 100, 20), (300, 300, 90)]


@pytest.mark.parametrize("dims", GRIDS)
@pytest.mark.parametrize("dx", [4.0, 5.0])
def test_chip_solve_equals_colour_sweeps(dims, dx):
    print(dims, dx, flush=True)
    a, b = _handle(dims, 7, False, dx), _handle(dims, 7, True, dx)
    a.run(1, 4)   # eager first step, then graph replays that carry the split copy
    b.run(1, 4)
    _same(a, b)
    a.press_sor_solve()  # scatter, solve, gather
    b.press_sor_solve()
    _same(a, b, ("p",))
    _ran(a, 5)
    assert b.solve_info()["solves"] == 0 and not b.solve_info()["on_chip"]
    a.close()
    b.close()


@pytest.mark.parametrize("dims", [(32, 24, 16), (96, 96, 20), (35, 27, 19)])
def test_queue_form_equals_colour_sweeps(dims):
    from les_halo_amd._lib import lib
    print(dims, flush=True)
    a, b = _handle(dims, 6, False), _handle(dims, 6, True)
    assert lib().les_internal_sor_wait(a.h, ctypes.c_long(-1)) == 0
    a.run(1, 4)
    b.run(1, 4)
    _same(a, b)
    _ran(a, 4, 4)
    assert lib().les_internal_sor_wait(a.h, ctypes.c_long(30000)) == 0
    a.run(5, 2)   # back to the resident form on the same buffers
    b.run(5, 2)
    _same(a, b)
    _ran(a, 6, 4)
    a.close()
    b.close()


def test_two_handles_take_turns():
    dims = (150, 150, 30)
    hs = [_handle(dims, 10, False) for _ in range(2)] + [_handle(dims, 10, True)]
    for n in range(1, 9, 2):  # enqueued without waiting in between
        for h in hs[:2]:
            h.run(n, 2)
    hs[2].run(1, 8)
    for h in hs[:2]:
        _same(h, hs[2])
        _ran(h, 8)
    for h in hs:
        h.close()


# pjuge: never met; just above the residual of iteration 4 of the first step
@pytest.mark.parametrize("queue", [False, True])
@pytest.mark.parametrize("dims", [(16, 12, 10), (48, 48, 32), (35, 27, 19), (150, 44, 61),
                                  (147, 133, 61), (300, 300, 90)])
def test_early_exit_equals_colour_sweeps(dims, queue):
    from les_halo_amd._lib import lib
    if queue and dims[0] > 100:
        pytest.skip("the queue form is covered on the small grids")
    probe = _handle(dims, 4, True, pjuge=1e-30)
    probe.run(1, 1)
    s4 = probe.scalars()["sor"]
    probe.close()
    for pjuge in (1e-30, float(np.float32(s4) * np.float32(1.0001))):
        print(dims, queue, pjuge, flush=True)
        a, b = _handle(dims, 9, False, pjuge=pjuge), _handle(dims, 9, True, pjuge=pjuge)
        if queue:
            assert lib().les_internal_sor_wait(a.h, ctypes.c_long(-1)) == 0
        for n, m in ((1, 1), (2, 3)):  # eager, then graph replays
            a.run(n, m)
            b.run(n, m)
            sa, sb = a.scalars(), b.scalars()
            if n == 1:
                assert sb["sor_iters"] == (9 if pjuge == 1e-30 else 4), sb
            assert sa == sb
            _same(a, b)
        a.press_sor_solve()
        b.press_sor_solve()
        assert a.scalars() == b.scalars()
        _same(a, b, ("p",))
        r = a.download("rhs")
        for scale in (1e9, 1e-9):  # terms above and below what the FP64 accumulators hold
            for h in (a, b):
                h.upload("rhs", (r * np.float32(scale)).astype(np.float32))
                h.press_sor_solve()
            assert a.scalars() == b.scalars()
            _same(a, b, ("p",))
        _ran(a, 7, 7 if queue else 0)
        a.close()
        b.close()


def test_queue_form_ends_with_the_exit():
    """Many tasks a sweep, the exit in the middle of the solve, again and again on one handle: no
    task of a sweep past the exit may run."""
    from les_halo_amd._lib import lib
    dims = (96, 96, 60)
    probe = _handle(dims, 3, True, pjuge=1e-30)
    probe.run(1, 1)
    pjuge = float(np.float32(probe.scalars()["sor"]) * np.float32(1.0001))
    probe.close()
    a, b = _handle(dims, 40, False, pjuge=pjuge), _handle(dims, 40, True, pjuge=pjuge)
    assert lib().les_internal_sor_wait(a.h, ctypes.c_long(-1)) == 0
    for n in range(1, 9):
        a.run(n, 1)
        b.run(n, 1)
        assert a.scalars() == b.scalars()
        assert n > 1 or a.scalars()["sor_iters"] == 3
        _same(a, b)
    _ran(a, 8, 8)
    a.close()
    b.close()


@pytest.mark.parametrize("pjuge", [0.0, 1e-30])
@pytest.mark.parametrize("dims", [(48, 48, 32), (147, 133, 61)])
def test_solve_that_gives_up_is_an_error(dims, pjuge):
    """Waits that end unanswered (bounded to no second look here): the missing words are NaN, the next
    call that waits for the device fails, and the handle goes on with the other forms, the sums'
    scratch memory as clean as before."""
    from les_halo_amd._lib import lib
    from les_halo_amd.les import LESError
    print(dims, pjuge, flush=True)
    a, b = _handle(dims, 5, False, pjuge=pjuge), _handle(dims, 5, True, pjuge=pjuge)
    for h in (a, b):
        h.run(1, 3)
    p, rhs = a.download("p"), a.download("rhs")
    assert lib().les_internal_sor_polls(a.h, 0) == 0
    a.press_sor_solve()
    with pytest.raises(LESError, match="SOR solve"):
        a.sync()
    assert np.isnan(a.download("p")).any()
    assert lib().les_internal_sor_polls(a.h, 1 << 22) == 0
    for h in (a, b):
        h.upload("p", p)
        h.press_boundp()
        h.upload("rhs", rhs)
        h.press_sor_solve()
        h.run(4, 2)
    assert a.scalars() == b.scalars()
    _same(a, b)
    a.close()
    b.close()


def test_polls_are_counted_per_sweep():
    """The bound of the waits is one sweep's: a solve of thousands of sweeps, whose unanswered polls
    together pass it many times over, ends like the sweeps' one."""
    from les_halo_amd._lib import lib
    dims = (48, 48, 32)
    a, b = _handle(dims, 40000, False), _handle(dims, 40000, True)
    # a sweep takes 2 us, a poll some tenths, and every sweep leaves some unanswered
    assert lib().les_internal_sor_polls(a.h, 1 << 15) == 0
    for h in (a, b):
        h.step(1)
    a.sync()
    _same(a, b)
    a.close()
    b.close()


def test_first_solves_while_another_thread_captures():
    """Handles whose first solves on the chip fall into another thread's captures of its step:
    neither may get into the other's capture, nor miss its turn."""
    import threading

    from les_halo_amd._lib import lib
    dims, small = (96, 96, 20), (64, 64, 24)
    a, b = _handle(dims, 4, False), _handle(dims, 4, True)
    cs, c0 = [_handle(small, 4, False) for _ in range(12)], _handle(small, 4, True)
    a.run(1, 3)
    b.run(1, 3)
    errs, done = [], threading.Event()

    def first_solves():
        try:
            for c in cs:
                c.run(1, 8)
                c.sync()
        except Exception as e:  # noqa: BLE001
            errs.append(e)
        finally:
            done.set()

    t = threading.Thread(target=first_solves)
    t.start()
    n = 4
    try:
        while not done.is_set() and n < 4000:
            assert lib().les_internal_sor_polls(a.h, 1 << 22) == 0  # its graph is captured anew
            a.run(n, 1)
            n += 1
    finally:
        t.join()
    assert not errs, errs
    b.run(4, n - 4)
    c0.run(1, 8)
    _same(a, b)
    for c in cs:
        _same(c, c0)
    for h in [a, b, c0] + cs:
        h.close()


def test_handle_leaves_the_queue_form():
    """16 solves in a row that find no room: the other forms from then on, the same values; one
    resident solve in between starts the count anew."""
    from les_halo_amd._lib import lib
    dims = (48, 48, 32)
    a, b = _handle(dims, 4, False), _handle(dims, 4, True)

    def steps(first, last, wait):
        assert lib().les_internal_sor_wait(a.h, ctypes.c_long(wait)) == 0
        for n in range(first, last + 1):
            a.run(n, 1)
            a.sync()

    steps(1, 10, -1)
    steps(11, 11, 30000)
    steps(12, 26, -1)
    _ran(a, 26, 25)
    steps(27, 32, -1)
    i = a.solve_info()
    assert (i["solves"], i["queued"], i["on_chip"], i["given_up"]) == (27, 26, 0, 1), i
    b.run(1, 32)
    _same(a, b)
    a.close()
    b.close()


def test_no_memory_for_a_solve_that_is_not_used():
    """A handle whose form was set by hand, or whose horizontal grid is not uniform, holds no face
    slots, also after a captured step."""
    from les_halo_amd import LES, inputs
    dims = (48, 48, 32)
    a = _handle(dims, 4, True)
    b = LES(*dims, **common.REF_PHYS, omega=1.5, pjuge=0.0, nmaxp=4)
    case = inputs.make_case(*dims, seed=5, hmax=20.0)
    case["dx1"] = (case["dx1"] * np.linspace(1.0, 1.5, case["dx1"].size)).astype(np.float32)
    d = case["dx1"]
    case["dxs"] = (d[1:dims[0] + 2] / np.float32(2) + d[2:dims[0] + 3] / np.float32(2)).astype(np.float32)
    b.load_case(case)
    b.ifdata()
    c = _handle(dims, 4, False)
    for h, held in ((a, False), (b, False), (c, True)):
        h.run(1, 4)
        i = h.solve_info()
        assert (i["face_bytes"] > 0, i["on_chip"] == 1, i["solves"] == 4) == (held,) * 3, i
        h.close()


def test_autotune_gives_the_form_back():
    """After les_set_sor_tile, and after a row of solves in the queue form."""
    from les_halo_amd._lib import lib
    dims = (48, 48, 32)
    a, b = _handle(dims, 4, False), _handle(dims, 4, True)
    a.run(1, 2)
    a.set_sor_tile(4, 5)
    a.run(3, 2)
    assert a.solve_info()["solves"] == 2 and not a.solve_info()["on_chip"]
    a.autotune(2)
    a.run(5, 2)
    _ran(a, 4)
    assert lib().les_internal_sor_wait(a.h, ctypes.c_long(-1)) == 0
    a.run(7, 16)
    assert a.solve_info()["given_up"]
    a.autotune(2)
    a.run(23, 3)
    _ran(a, 23, 19)
    assert lib().les_internal_sor_wait(a.h, ctypes.c_long(30000)) == 0
    a.run(26, 2)
    _ran(a, 25, 19)
    b.run(1, 27)
    _same(a, b)
    a.close()
    b.close()


SHARED = [(96, 96, 20), (48, 48, 32), (147, 133, 61), (35, 27, 19), (150, 150, 90), (300, 300, 90)]


@pytest.mark.parametrize("pjuge", [0.0, 1e-30])
def test_handles_share_the_device(pjuge):
    """Handles launched in alternation: solves on a half or a quarter of the CUs beside each other (the
    grid of 8.1 M cells on all of them), the same values; then one of them alone again."""
    from les_halo_amd import Ensemble
    for dims in (SHARED[:2], SHARED):
        print(dims, pjuge, flush=True)
        hs = [_handle(d, 5, False, pjuge=pjuge) for d in dims]
        refs = [_handle(d, 5, True, pjuge=pjuge) for d in dims]
        E = Ensemble(hs, batched=False)
        E.run(1, 2)
        E.run(3, 12)
        for h in hs:
            h.press_sor_solve()
        for h, r in zip(hs, refs):
            r.run(1, 14)
            r.press_sor_solve()
            _same(h, r)
            assert pjuge == 0.0 or h.scalars() == r.scalars()
            i = h.solve_info()
            assert i["solves"] == 15 and not i["given_up"], i
        shared = [h.solve_info()["shared"] for h in hs]
        assert all((n > 0) == (d != (300, 300, 90)) for d, n in zip(dims, shared)), shared
        for h, r in ((hs[0], refs[0]), (hs[-1], refs[-1])):
            h.run(15, 3)
            h.sync()
            r.run(15, 3)
            _same(h, r)
        assert [h.solve_info()["shared"] for h in hs] == shared
        E.close()
        for h in hs + refs:
            h.close()


# (levels per thread, several level blocks), grid, CUs to cut it for: every instance of the kernel, with
# even and odd jp, several workgroups along j and k and a remainder along both
CUTS = [((1, 0), (96, 20, 12), 96), ((1, 0), (61, 27, 12), 96), ((1, 1), (24, 44, 20), 48),
        ((1, 1), (24, 27, 20), 24), ((2, 0), (391, 20, 33), 64), ((2, 0), (391, 27, 33), 96),
        ((2, 1), (130, 20, 20), 12), ((2, 1), (35, 27, 33), 8), ((3, 0), (300, 44, 20), 64),
        ((3, 0), (300, 61, 20), 64), ((3, 1), (48, 64, 33), 12), ((3, 1), (35, 27, 33), 4),
        ((4, 0), (391, 20, 61), 48), ((4, 0), (391, 27, 33), 48), ((4, 1), (150, 44, 20), 12),
        ((4, 1), (24, 27, 90), 4), ((5, 0), (391, 44, 33), 64), ((5, 0), (391, 61, 33), 96),
        ((5, 1), (48, 64, 61), 12), ((5, 1), (61, 27, 33), 4), ((6, 0), (300, 64, 33), 32),
        ((6, 0), (300, 61, 33), 32), ((6, 1), (96, 64, 33), 12), ((6, 1), (48, 27, 61), 4),
        ((7, 0), (391, 44, 12), 12), ((7, 0), (391, 27, 12), 8), ((7, 1), (200, 44, 33), 16),
        ((7, 1), (35, 27, 90), 4), ((8, 0), (200, 44, 61), 24), ((8, 0), (150, 61, 61), 24),
        ((9, 0), (130, 64, 33), 12), ((9, 0), (150, 27, 33), 8), ((10, 0), (130, 64, 48), 16),
        ((10, 0), (130, 61, 48), 16)]


@pytest.mark.parametrize("kind, dims, ncu", CUTS)
def test_every_cut_equals_colour_sweeps(kind, dims, ncu):
    from les_halo_amd._lib import lib
    for pjuge in (0.0, 1e-30):
        print(kind, dims, ncu, pjuge, flush=True)
        a, b = _handle(dims, 7, False, pjuge=pjuge), _handle(dims, 7, True, pjuge=pjuge)
        assert lib().les_internal_sor_cut(a.h, ncu) == 0
        a.run(1, 3)
        b.run(1, 3)
        _same(a, b)
        assert pjuge == 0.0 or a.scalars() == b.scalars()
        _ran(a, 3)
        i = a.solve_info()
        assert (i["levels"], int(i["level_blocks"] > 1)) == kind, i
        a.close()
        b.close()


# grids near the largest that fit: 5 to 10 levels a thread on the whole device
@pytest.mark.parametrize("dims, levels", [((166, 343, 68), 5), ((157, 525, 52), 6), ((194, 509, 66), 7),
                                          ((283, 306, 78), 8), ((296, 328, 90), 10),
                                          ((391, 224, 95), 10)])
def test_large_grids_equal_colour_sweeps(dims, levels):
    print(dims, flush=True)
    a, b = _handle(dims, 3, False), _handle(dims, 3, True)
    a.run(1, 2)
    b.run(1, 2)
    _same(a, b, ("p", "u", "rhs"))
    _ran(a, 2)
    assert a.solve_info()["levels"] == levels, a.solve_info()
    a.close()
    b.close()
