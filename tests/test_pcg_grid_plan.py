"""The host's rules for the PCG in one launch (grid_plan, GridLease), without a GPU: the launch never has more
workgroups than the device has CUs, one solve at a time holds a device, and a wait that ran out keeps the next
solves away from it. The library's C++ functions are called by their symbols."""
import ctypes as C

import pytest

from luisacomputesimulator_amd import load_library, pcg_form_counts


def plan(most, n_rb, width, wgs):
    fn = load_library()._ZN4lcsx9grid_planEjjjj
    fn.restype, fn.argtypes = C.c_uint64, [C.c_uint32] * 4
    v = fn(most, n_rb, width, wgs)
    return v & 0xFFFFFFFF, v >> 32  # row groups and blocks per thread; (0, 0): the launches


@pytest.mark.parametrize("wgs", [0, 1, 32, 64, 80, 256])
def test_plan_fits_the_device(wgs):
    for n_rb in {1, 2, wgs - 1, wgs, wgs + 1, 2 * wgs, 2 * wgs + 1, 256, 257, 512, 513} - {-1, 0}:
        for width in (6, 12, 13, 16, 17, 32, 33):
            U, K = plan(n_rb, n_rb, width, wgs)
            if U:
                per = U * 512 // 1024
                assert (n_rb + per - 1) // per <= wgs and 4 * K >= width
            assert bool(U) == (width <= 32 and n_rb <= (2 * wgs if width <= 12 else wgs))


def test_lease_and_waits():
    lib = load_library()
    take, outcome, drop = (lib._ZN4lcsx9GridLease4takeEi, lib._ZN4lcsx9GridLease7outcomeEjb, lib._ZN4lcsx9GridLeaseD1Ev)
    take.restype, take.argtypes = C.c_bool, [C.c_void_p, C.c_int]
    outcome.restype, outcome.argtypes = None, [C.c_void_p, C.c_uint32, C.c_bool]
    drop.restype, drop.argtypes = None, [C.c_void_p]
    dev = 63  # of which no machine here has one

    class Lease:
        def __init__(self):
            self.dev = C.c_int(-1)
            self.got = take(C.byref(self.dev), dev)

        def end(self, fail=None, remember=True):
            if fail is not None:
                outcome(C.byref(self.dev), fail, remember)
            drop(C.byref(self.dev))

    def counts():
        return list(pcg_form_counts(dev).values())

    a, b = Lease(), Lease()
    assert a.got and not b.got and counts() == [0, 0, 0, 1]
    b.end()
    c = Lease()
    assert not c.got  # b never held it, so its end gives nothing back
    c.end()
    a.end(0)
    a = Lease()
    assert a.got
    a.end(1)  # rows that do not fit say nothing about the device
    a = Lease()
    assert a.got and counts() == [1, 1, 0, 2]
    a.end(2, False)  # nor does a wait that the caller bounded
    for away in (1024, 2048):
        a = Lease()
        assert a.got
        a.end(2)
        for _ in range(away):
            x = Lease()
            assert not x.got
            x.end()
    a = Lease()
    assert a.got and counts() == [1, 1, 3, 2 + 1024 + 2048]
    a.end(0)
    for bad in (-1, 64):
        x = C.c_int(-1)
        assert not take(C.byref(x), bad)
