"""The chip-resident solve's host arithmetic (les_sor_res.h), on the CPU."""
import ctypes

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
