"""The reference's heap as a search's log of its open list's operations rebuilds it (bps_nav_amd/csrc/geodesic_device.h, replay_log),
against the heap itself (dtNodeQueue, DetourNode.cpp:150-200) entry by entry, at the sizes up to which an operation takes one
round or another, with totals that differ and with many equal ones."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHECKS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "libbpsx_checks.so")
HEADER, UNORDERED, POLY = 1 << 31, 1 << 30, 7 << 11


class Heap:
    """dtNodeQueue: [total, node], the root first"""
    def __init__(self):
        self.h = []

    def up(self, i, e):
        while i > 0 and self.h[(i - 1) // 2][0] > e[0]:
            self.h[i] = self.h[(i - 1) // 2]
            i = (i - 1) // 2
        self.h[i] = e

    def push(self, e):
        self.h.append(e)
        self.up(len(self.h) - 1, e)

    def pop(self):
        root, e = self.h[0], self.h.pop()
        if self.h:
            i, c = 0, 1
            while c < len(self.h):
                if c + 1 < len(self.h) and self.h[c][0] > self.h[c + 1][0]:
                    c += 1
                self.h[i] = self.h[c]
                i, c = c, 2 * c + 1
            self.up(i, e)
        return root


@pytest.mark.parametrize("apart", [100000, 6])   # totals that differ as a rule, and few of them
@pytest.mark.parametrize("size", [1, 2, 3, 31, 32, 33, 62, 63, 64, 65, 66, 100, 126, 127, 128, 129, 130, 190, 254, 255, 256, 257, 300, 370])
def test_replayed_heap_is_the_reference_heap(size, apart):
    import torch   # its HIP runtime is the one that the library then uses
    assert torch.cuda.is_available()
    L = C.CDLL(CHECKS)
    rng = np.random.default_rng(1000 * size + apart)
    H, nodes, log = Heap(), 1, []
    for _ in range(size):
        H.push((1000000 + int(rng.integers(apart)), nodes | POLY))
        nodes += 1
    entries = np.zeros((384, 2), np.uint32)
    entries[1:size + 1] = H.h
    start = nodes
    while len(log) < 2500 and nodes < 1990 and H.h:
        # a pass of up to eight nodes, each with up to six updates (0: of a node that had been there before the pass, else a new one's
        # index, in the order of the rows); the first two may be taken in either order
        before, rows = nodes, min(int(rng.integers(1, 9)), len(H.h))
        plan = []
        for _ in range(rows):
            few = len(H.h) > min(size + 2, 320)
            k = int(rng.random() < 0.9) if few else int(rng.integers(0, 7 if rng.random() < 0.3 else 3))
            plan.append([])
            for _ in range(k):
                known = rng.random() < 0.15
                plan[-1].append(0 if known else nodes)
                nodes += not known
        unordered = rows > 1 and rng.random() < 0.3
        swapped = unordered and rng.random() < 0.5
        first = 0x3ffffff if swapped else H.h[0][1]   # the node that the log says row 0 expanded
        recs = [[] for _ in range(rows)]
        for r in [1, 0][:2 * swapped] + list(range(2 * swapped, rows)):
            t0 = H.pop()[0]
            for node in plan[r]:
                e = (t0 + int(rng.integers(3 * apart)), node | POLY)
                if node:
                    H.push(e)
                else:
                    # an open node takes a smaller total, or one that has been closed is open again
                    i = [i for i, old in enumerate(H.h) if (old[1] & 0x7ff) < before and old[0] > e[0]]
                    gone = sorted(set(range(1, before)) - {old[1] & 0x7ff for old in H.h})
                    if i and rng.random() < 0.7:
                        i = int(rng.choice(i))
                        e = (e[0], H.h[i][1])
                        H.up(i, e)
                    elif gone:
                        e = (e[0], int(rng.choice(gone)) | POLY)
                        H.push(e)
                    else:
                        continue
                recs[r].append((e[0], e[1] | r << 26))
        flat = [x for u in recs for x in u]
        log += flat + [(rows | len(flat) << 8, HEADER | (UNORDERED | first if unordered else 0))]
    log = np.array(log, np.uint32)
    got = np.ascontiguousarray(entries)
    print(f"case: {size} entries, {len(log)} records", flush=True)
    n = L.bpsx_check_replay(got.ctypes.data_as(C.c_void_p), size, start, log.ctypes.data_as(C.c_void_p), len(log))
    assert n == len(H.h)
    assert np.array_equal(got[1:n + 1], np.array(H.h, np.uint32).reshape(-1, 2))
