"""The wavefront that keeps a search's heap (bps_nav_amd/csrc/geodesic_device.h, follow) raises its priority while the search waits
for its answer, and only then.  Its loop as it stands in the source, compiled for the host with one lane, a heap that counts
passes, and a search that moves on whenever the loop comes by."""
import os
import re
import shutil
import subprocess

import pytest

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "csrc", "geodesic_device.h")

HOST = r"""
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#define BPSX_DEV static
struct uint2 { uint32_t x, y; };
struct OpRec { uint32_t key, word; };
struct GeoSlot { alignas(8) OpRec oplog[64]; };
struct GeoLds {
  uint2 ref_heap[4], start;
  uint32_t published, applied, heap_size;
  uint16_t arrived;
  uint2* heap() { return ref_heap; }
} lds;
constexpr uint32_t kFollowEnd = 0xffffu, kFollowQuit = 0xffffffffu, kOpHeader = 1u << 29;
static int priority, at, applied_waiting, applied_ahead;
static bool waits() { return (lds.published & 0xffffu) && lds.published != lds.applied; }
static void check(const char* where) {
  if (priority && !waits()) { printf("step %d: priority %d %s, and no search waits\n", at, priority, where); exit(1); }
}
static int lane_here(int lane) { return lane; }
static int uniform_i(int v) { return v; }
static void wave_sync() {}
static unsigned long long lanes_where(bool b) { return b; }
static uint32_t lds_word(const uint32_t* p) { return *p; }
static uint32_t* lds_address(uint32_t* p) { return p; }
static void lds_store_where(unsigned long long, uint32_t* p, uint32_t v) { *p = v; }
static void lds_store_where(unsigned long long, uint2* p, uint32_t x, uint32_t y) { *p = {x, y}; }
template <bool> struct RefHeap { uint2* h; int size; RefHeap(uint2* e, int n, int) : h(e), size(n) {} };
static int apply_pass(RefHeap<true>&, uint32_t, uint32_t, unsigned long long, int, int&) {
  check("for a pass");
  if (waits()) { applied_waiting++; if (priority != 3) { printf("step %d: the search waits, priority %d\n", at, priority); exit(1); } }
  else applied_ahead++;
  return 1;
}
// the search: the next step when what it asked for last is done
struct { uint32_t published; int arrived; } const steps[] = {
    {0x10000u, 0}, {0x10000u, 3},      // a search, and three passes ahead of any question
    {0x10005u, 5},                     // a tie: the two behind them, and the answer
    {0x10005u, 9}, {0x10005u, 12},     // the passes behind it
    {0x1000du, 13}, {0x1000du, 15},    // another
    {0x1ffffu, 15},                    // the end of a search that had asked
    {0x20000u, 0}, {0x20000u, 4},      // one that does not
    {0x2ffffu, 4}, {0x30000u, 0}, {0x30002u, 2}, {0x3ffffu, 2}, {kFollowQuit, 2}};
static void polled() {
  check("between passes");
  if (lds.published != lds.applied && (lds.published & 0xffffu)) return;
  lds.published = steps[at].published;
  lds.arrived = (uint16_t)steps[at].arrived;
  at++;
}
#define __builtin_amdgcn_s_sleep(n) polled()
#define __builtin_amdgcn_s_setprio(p) (void)(priority = (p))
#define __hip_atomic_load(p, order, scope) (*(p))
@LOOP@
int main() {
  static GeoSlot slot;
  for (OpRec& r : slot.oplog) r.word = kOpHeader;
  lds.published = lds.applied = kFollowEnd;
  follow(&lds, &slot, 0);
  printf("%d %d %d\n", applied_waiting, applied_ahead, priority);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs the compiler")
def test_raised_only_while_the_search_waits(tmp_path):
    with open(SOURCE) as f:
        loop = re.search(r"^BPSX_DEV void follow\(.*?^}\n", f.read(), re.S | re.M).group(0)
    (tmp_path / "follow.cpp").write_text(HOST.replace("@LOOP@", loop))
    subprocess.run(["g++", "-std=c++17", "-o", "follow", "follow.cpp"], cwd=tmp_path, check=True)
    run = subprocess.run(["./follow"], cwd=tmp_path, capture_output=True, text=True, timeout=20)
    assert run.returncode == 0, run.stdout
    # passes applied for a search that waits, and ahead of its questions; the priority at the end
    assert run.stdout.split() == ["5", "16", "0"]
