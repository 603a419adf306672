"""How the host waits for a launch that tells of its end (bps_nav_amd/csrc/wait_rule.h), on the CPU."""
import ctypes as C
import os

import numpy as np

CHECKS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "libbpsx_checks.so")
BUSY, IDLE, GONE, FAILED = range(4)
TOLD, NEVER, ERROR = range(3)


def wait(comes, answers, drained=0, patience=1000):
    """(outcome, looks, questions, waits for the device); drained: 1 the word is there then, 0 it is not, -1 the wait fails"""
    L = C.CDLL(CHECKS)
    L.bpsx_check_wait.argtypes = [C.c_uint32, C.c_int, C.c_uint32, C.c_void_p, C.c_uint32, C.c_void_p]
    a, out = np.array(answers, np.int32), np.zeros(3, np.uint32)
    return (L.bpsx_check_wait(comes, drained, patience, a.ctypes.data, len(a), out.ctypes.data), *out.tolist())


def test_a_word_that_comes_ends_the_wait():
    assert wait(1, [FAILED]) == (TOLD, 1, 0, 0)
    assert wait(900, [FAILED]) == (TOLD, 900, 0, 0)     # the stream is not asked before
    r, looks, asked, drains = wait(5000, [BUSY])         # a long launch: it is asked now and then
    assert (r, looks, drains) == (TOLD, 5000, 0) and 10 < asked < 20


def test_a_launch_that_has_failed():
    assert wait(0, [BUSY, BUSY, FAILED])[::2] == (ERROR, 3)
    assert wait(0, [GONE], drained=-1)[::3] == (ERROR, 1)


def test_a_stream_that_is_gone():
    assert wait(0, [BUSY, GONE], drained=1)[::3] == (TOLD, 1)
    assert wait(0, [GONE], drained=0)[::3] == (NEVER, 1)


def test_an_idle_stream():
    first = wait(0, [IDLE])[1]
    # the word came between the last look and the question: nothing more is waited for
    assert wait(first - 1, [IDLE])[::3] == (TOLD, 0)
    assert wait(0, [IDLE], drained=1)[::3] == (TOLD, 1)
    # nothing is left to run and nobody has told: the launch has not run, which is no success
    assert wait(0, [IDLE], drained=0)[::3] == (NEVER, 1)
    assert wait(0, [BUSY, BUSY, IDLE], drained=0)[::3] == (NEVER, 1)
