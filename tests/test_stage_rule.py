"""How much pinned memory a simulator keeps for the host arrays of its batched calls (bps_nav_amd/csrc/stage_rule.h), on the CPU."""
import ctypes as C
import os

import numpy as np
import pytest

CHECKS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "libbpsx_checks.so")
MOST, AT_ONCE, PAYS = 16 << 20, 256 << 10, 8


def stage(calls, refuse=0):
    """(allocations, bytes held at each call)"""
    L = C.CDLL(CHECKS)
    L.bpsx_check_stage.argtypes = [C.c_void_p, C.c_uint32, C.c_uint32, C.c_void_p]
    calls = np.ascontiguousarray(calls, np.uint64)
    held = np.zeros(len(calls), np.uint64)
    made = L.bpsx_check_stage(calls.ctypes.data, len(calls), refuse, held.ctypes.data)
    return made, held.astype(np.int64)


@pytest.mark.parametrize("bytes_", [1, AT_ONCE, AT_ONCE + 1, 2 << 20, MOST - 1, MOST])
def test_calls_of_one_size(bytes_):
    made, held = stage([bytes_] * 20)
    copies = 0 if bytes_ <= AT_ONCE else PAYS
    assert made == 1 and not held[:copies].any() and (held[copies:] >= bytes_).all() and held.max() <= MOST


def test_calls_beyond_the_limit_copy_and_count_for_nothing():
    assert stage([MOST + 1] * 50)[0] == 0
    made, held = stage([MOST + 1] * 50 + [1 << 20] * PAYS + [1 << 20])
    assert made == 1 and not held[:-1].any() and held[-1] >= 1 << 20


@pytest.mark.parametrize("each", [(28, 44, 28), (44, 28, 28), (28, 28, 44, 36), (6, 44, 1)])
@pytest.mark.parametrize("n", [50000, 9000])
def test_one_allocation_serves_calls_of_several_sizes(each, n):
    """50000 samples, moves and snaps: memory is taken once, for the largest of them, when the calls have copied
    eight times as much as that."""
    calls = [n * e for e in each] * 40
    made, held = stage(calls)
    large = [b for b in calls if b > AT_ONCE]
    assert held[-1] >= max(calls) and made <= 1 + (min(calls) <= AT_ONCE)
    copied = sum(b for b, h in zip(calls, held) if b > h)
    assert PAYS * max(large) <= copied < (PAYS + 1) * max(large)


def test_small_calls_between_large_ones_do_not_put_them_off():
    calls = [1 << 20, 100] * 20
    made, held = stage(calls)
    assert made == 2 and (held[2 * PAYS:] >= 1 << 20).all() and (held[1:2 * PAYS] == AT_ONCE).all()


def test_larger_calls_later_grow_it():
    calls = [1 << 20] * 20 + [4 << 20] * 20
    made, held = stage(calls)
    assert made == 2 and held[19] < 4 << 20 and (held[20 + PAYS:] >= 4 << 20).all()
    assert (np.diff(held) >= 0).all()


def test_memory_that_is_refused():
    """What is held stays, and the next attempt comes after as much copying again, at once for small calls."""
    made, held = stage([1000, *[1 << 20] * 40], refuse=2)
    assert made == 2 and (held[:2 * PAYS + 2] == AT_ONCE).all() and (held[2 * PAYS + 2:] >= 1 << 20).all()
    made, held = stage([1000] * 3, refuse=1)
    assert made == 0 and not held.any()
