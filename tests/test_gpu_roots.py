"""The path search's square roots are the correctly rounded ones for every float: costs, totals and their ties are the
reference's only if they are."""
import ctypes as C
import os

import pytest

pytestmark = pytest.mark.gpu

CHECKS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "libbpsx_checks.so")
LOW, INF = 0x0f800000, 0x7f800000   # 2^-96, from where on the short form is taken


# the whole range of the short form; below it a wavefront takes the library's routine
@pytest.mark.parametrize("first, end", [(LOW, INF), (1, LOW)])
def test_roots_are_correctly_rounded(first, end):
    import torch
    L = C.CDLL(CHECKS)
    L.bpsx_check_roots.argtypes = [C.c_uint32, C.c_uint32, C.c_void_p, C.c_void_p, C.c_void_p]
    chunk = 1 << 26
    a, b = torch.empty(chunk, device="cuda"), torch.empty(chunk, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    steps = torch.arange(chunk, dtype=torch.int32, device="cuda")
    print(f"case: roots of the floats with bits {first:#x} to {end:#x}", flush=True)
    for at in range(first, end, chunk):
        n = min(chunk, end - at)
        a.fill_(-1.0), b.fill_(-1.0)
        assert L.bpsx_check_roots(at, n, a.data_ptr(), b.data_ptr(), stream) == 0
        x, r = (steps[:n] + at).view(torch.float32).double(), a[:n]
        assert torch.equal(r.view(torch.int32), b[:n].view(torch.int32))
        # The middles between a root and its two neighbours have 25 bits and their squares 50, which 64-bit floats hold:
        # a root is correctly rounded where its argument lies between those squares (and never is one of them).
        mid = [((r.double() + (r.view(torch.int32) + k).view(torch.float32).double()) * 0.5) for k in (-1, 1)]
        wrong = ~((mid[0] * mid[0] < x) & (x < mid[1] * mid[1]))
        assert not bool(wrong.any()), [hex(at + int(i)) for i in torch.nonzero(wrong)[:5]]


def test_roots_of_the_ends():
    """Zero, infinity, and both sides of the two lines, where one argument of a wavefront decides for both roots."""
    import torch
    L = C.CDLL(CHECKS)
    L.bpsx_check_roots.argtypes = [C.c_uint32, C.c_uint32, C.c_void_p, C.c_void_p, C.c_void_p]
    for first, n in ((0, 1), (0, 64), (INF, 1), (LOW - 64, 128), (INF - 63, 64), (LOW, 63), (0x3f800000, 1)):
        a, b = torch.full((n,), -1.0, device="cuda"), torch.full((n,), -1.0, device="cuda")
        assert L.bpsx_check_roots(first, n, a.data_ptr(), b.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
        x = (torch.arange(n, dtype=torch.int32) + first).view(torch.float32)
        want = x.double().sqrt().float()   # twice rounded is once rounded for roots of floats
        assert torch.equal(a.cpu(), want) and torch.equal(b.cpu(), want), (hex(first), n)
