"""The chip-resident solve's host arithmetic (les_sor_res.h), on the CPU."""
import ctypes
import random

import pytest

from les_halo_amd._lib import lib


@pytest.mark.parametrize("dims", [(300, 300, 90), (147, 133, 61), (32, 24, 16)])
@pytest.mark.parametrize("nwg", [1, 3, 240])
@pytest.mark.parametrize("nmaxp", [0, 1, 50, 500000, 2 ** 31 - 1])
def test_queue_tasks_of_any_number_of_iterations(dims, nwg, nmaxp):
    ip, jp, kp = dims
    f = lib().les_internal_sor_tasks
    f.restype = ctypes.c_int64
    groups = ((ip + 1) // 2 + 3) // 4 * jp * kp
    assert f(ip, jp, kp, nwg, nmaxp) == min(nwg, -(-groups // 512)) * (1 + 2 * nmaxp * (2 if jp % 2 else 1))


def _plan(dims, ncu):
    out = (ctypes.c_int * 5)()
    assert lib().les_internal_sor_plan(*dims, ncu, out) == 0
    return tuple(out)


def _grids():
    r = random.Random(5)
    some = [tuple(r.randint(1, m) for m in (520, 600, 128)) for _ in range(120)]
    return some + [(1, 1, 1), (2, 3, 1), (8, 1, 5), (512, 40, 90), (300, 300, 90), (296, 328, 90), (16, 12, 10)]


def test_cuts_cover_the_grid_within_the_kernel():
    """Every cut: its workgroups on the CUs given, its threads on a workgroup, its rows and levels
    over the whole grid with none empty, its j faces in the words a thread takes, the level blocks
    only where the kernel has them."""
    found = 0
    for dims in _grids():
        ip, jp, kp = dims
        ng = ((ip + 1) // 2 + 3) // 4
        for ncu in (1, 4, 37, 64, 128, 256, 304):
            tk, ks, rj, njt, nkt = _plan(dims, ncu)
            if tk == 0:
                continue
            found += 1
            assert 1 <= tk <= 10 and ks >= 1 and njt * nkt <= ncu, (dims, ncu)
            assert ks == 1 or (tk <= 7 and ks * tk <= 128)
            assert ks * rj * ng <= (448 if tk == 10 else 512)
            assert 4 * ng * ks * tk <= (tk * 160 + 511) // 512 * 512
            rows = [jp * (q + 1) // njt - jp * q // njt for q in range(njt)]
            assert sum(rows) == jp and max(rows) <= rj and min(rows) >= 1
            assert (nkt - 1) * ks * tk < kp <= nkt * ks * tk
    assert found > 200


def test_grids_that_fit_256_cus():
    """The limits that the documents give: rows of up to 512 cells; about 9 M cells of rows up to
    408 (8 M at 400), 4 M of rows of 440 to 512."""
    def most(ip):
        return max((jp * ip * kp for kp in (16, 32, 48, 64, 90) for jp in range(20, 1200, 4)
                    if _plan((ip, jp, kp), 256)[0]), default=0)
    assert most(300) > 8.5e6 and most(320) > 8.5e6 and most(400) > 8e6
    assert 3.5e6 < most(440) < 4.5e6 and 3.5e6 < most(512) < 4.5e6
    assert most(513) == 0
