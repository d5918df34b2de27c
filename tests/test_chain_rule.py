"""The rules that choose chain kernels and their workgroups, on the CPU."""
import ctypes

import pytest

from nutrlan_amd import trlan as T


def rule(n, kind, cus, nb=None, nnz=1000, jnd=20, mixed=0, active=1):
    wgs = ctypes.c_int()
    rw = T.lib().trlhip_chain_rule(n, kind, mixed, -(-n // 256) if nb is None else nb, nnz, jnd, cus, active,
                                   ctypes.byref(wgs))
    return rw, wgs.value


def batch_rule(rows, maxn, cus):
    f = T.lib().trlhip_batch_chain_rule
    f.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    maxg = ctypes.c_int()
    return f(rows, maxn, cus, ctypes.byref(maxg)), maxg.value


@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("kind", [-3, -2, -1, 0])
@pytest.mark.parametrize("cus", [1, 2, 16, 32, 38, 64, 80, 128, 228, 256, 304])
def test_workgroups_fit_the_device(kind, cus, mixed):
    """All workgroups of a chain wait for each other, so there is at most one
    per CU, and never more than the flags a context holds."""
    taken = 0
    for n in [10, 256, 257, 512, 1024, 1025, 4096, 10000, 20000, 32768, 32769, 50000, 65536, 65537, 98304, 131072,
              131073, 200000, 262144, 262145, 500000]:
        rw, wgs = rule(n, kind, cus, mixed=mixed)
        if rw:
            taken += 1
            assert wgs * 256 * rw >= n and wgs <= min(cus, 256)
            assert rule(n, kind, cus, mixed=mixed, active=1) == (rw, wgs)
        else:
            assert -(-n // (512 if kind > -2 else 1024)) > min(cus, 256)
    assert taken


def test_row_waves():
    for kind in (-2, -3):
        assert rule(131072, kind, 256) == (2, 256) and rule(131073, kind, 256) == (4, 129)
        assert rule(65536, kind, 256, mixed=1) == (2, 128) and rule(65537, kind, 256, mixed=1) == (4, 65)
        assert rule(20000, kind, 32) == (4, 20) and rule(32769, kind, 32)[0] == 0
    assert rule(131072, 0, 256, mixed=1) == (2, 256)


@pytest.mark.parametrize("mixed", [0, 1])
def test_share_beside_others(mixed):
    """Beside others a chain takes its share of the CUs, 4 row waves if it
    needs them, or up to a quarter of the CUs."""
    assert rule(62500, -2, 256, mixed=mixed) == (2, 123)
    assert rule(62500, -2, 256, mixed=mixed, active=2) == (2, 123)
    assert rule(62500, -2, 256, mixed=mixed, active=3) == (4, 62)
    assert rule(62500, -2, 256, mixed=mixed, active=16) == (4, 62)
    assert rule(65537, -2, 256, mixed=mixed, active=16)[0] == 0
    assert rule(122500, -2, 256, mixed=mixed, active=2) == (4, 120)
    assert rule(122500, -2, 256, mixed=mixed, active=3)[0] == 0
    assert rule(10000, -2, 256, mixed=mixed, active=8) == (2, 20)
    assert rule(10000, -2, 256, mixed=mixed, active=16) == (4, 10)
    assert rule(32768, 0, 256, mixed=mixed, active=16) == (2, 64)
    assert rule(32769, 0, 256, mixed=mixed, active=4)[0] == 0
    for cus in (8, 32, 256):
        for active in (2, 3, 5, 9, 100):
            for n in (300, 5000, 20000, 40000, 100000, 200000):
                rw, wgs = rule(n, -2, cus, mixed=mixed, active=active)
                assert wgs <= max(cus // active, cus // 4)


def test_batch_chains_scale_with_the_device():
    """A chain takes a quarter of the CUs at most, and workgroups of two row
    waves while the launch's rows fit 512 a CU."""
    assert batch_rule(131072, 20000, 256) == (2, 64)
    assert batch_rule(131073, 20000, 256) == (4, 64)
    assert batch_rule(131072, 32769, 256) == (4, 64)
    assert batch_rule(20000, 4096, 64) == (2, 16)
    assert batch_rule(32769, 4096, 64) == (4, 16)
    assert batch_rule(20000, 8193, 64) == (4, 16)
    assert batch_rule(1000, 500, 3)[1] == 0


def test_shapes_that_keep_the_ordinary_kernels():
    assert rule(10000, -2, 256, jnd=192)[0] and not rule(10000, -2, 256, jnd=193)[0]
    assert not rule(262145, -2, 256)[0] and not rule(131073, 0, 256)[0]
    assert rule(10000, 0, 256, nnz=2048)[0] and not rule(10000, 0, 256, nnz=2049)[0]
    assert rule(10000, 0, 256, nb=160)[0] and not rule(10000, 0, 256, nb=161)[0]
