// Geodesic distance on the GPU: Detour's A* over the polygon graph followed by the funnel
// (string pulling) and the summed segment length, with the exact buffer limits and failure
// conventions of the reference, so that the value equals PathFinder::findPath's.
//
// Execution model: one wavefront (64 lanes) owns one query at a time and pulls the next from
// a shared queue when done.  The search touches almost only nodes it created recently (the
// frontier of A* is narrow), so LDS holds what is hot and small and HBM holds the rest:
//   - the open list in registers: its smallest entries sorted by total (OpenList), which lets a
//     pass expand up to kRows nodes at once (astar_fast); when totals tie, the reference's binary
//     heap is rebuilt from a log of the list's operations (RefHeap, replay_log) or has been kept from it all
//     along by a second wavefront (follow), and a search whose
//     list outgrows what this form holds, or has more equal totals in front than registers, goes on with that heap,
//   - the hash heads of the node pool,
//   - for the first kLinksLds nodes one word with the polygon id and the hash chain link,
//   - the position and cost of the kWindow most recently created nodes (slot = index
//     modulo kWindow); every write of those also goes to the wavefront's slot in HBM, so an older
//     node is simply read from there.
// Links beyond kLinksLds spill to the same slot.  A query runs the instantiation of the loop without
// spill code until one more pass could outgrow the links in LDS, then carries on in a spilling one.
// Per expanded node the regular HBM traffic is the polygon's six 16-byte edge records (lane j
// of the wavefront handles edge j: node lookup, cost, heuristic) plus the write-through of
// updated nodes; heap updates are applied in edge order, which is what makes the result
// identical to the sequential algorithm, ties included.  A wavefront spends its time in one
// chain of dependent steps, so the code is written for few of them: heap pops and pushes are
// done by all lanes at once, what is the same for all lanes lives in scalar registers, and
// LDS and HBM accesses stay separate instructions.
//
// Reference semantics followed: DetourNavMeshQuery.cpp:945-1178 (findPath, getPathToNode),
// :1661-1696, 1765-1994 (appendVertex, findStraightPath), :2279-2381 (getPortalPoints,
// getEdgeMidPoint); DetourNode.cpp:50-200 (node pool, heap order); PathFinder.cpp:473-541.
//
// The sizes of the LDS structures are build parameters (BPSX_LINKS_LDS,
// BPSX_WINDOW, BPSX_HASH, BPSX_TAG_SLOTS; BPSX_FOLLOWER: a second wavefront keeps the reference's heap),
// and everything that depends on them lives in namespace
// bpsx::BPSX_GEO_NS (default geo): the file can be included again with other values and
// another namespace name to get a second instantiation of the same search.
#include "nav_device.h"

#ifndef BPSX_GEODESIC_COMMON_H
#define BPSX_GEODESIC_COMMON_H
namespace bpsx {

#ifdef BPSX_PHASE_TIMING
// diagnostic build: cycles per phase of the sorted-list loop -> counters: 0 front of the list, 1 fetch, 2 lookup,
// 3 costs, 4 rows that stand, 5 new nodes and stores, 6 log and list; 7 counts the passes
// (the comment that the asm statement leaves in the compiler's assembly output names the loop's
// instantiation and the mark, for tests/measure_astar_loop_phases.py)
#define FM(k) do { constexpr int slot_[11] = {7, 0, 1, 2, 3, 4, 5, 5, 5, 6, 6}; const unsigned long long now_ = __builtin_readcyclecounter(); \
    asm volatile("; astar_fast spill=%0 mark=%1" :: "i"((int)S), "i"(k)); \
    if ((k) == 0) g.phase[7]++; else g.phase[slot_[k]] += now_ - g.phase_t0; g.phase_t0 = now_; } while (0)
#else
#define FM(k) do { } while (0)
#endif

BPSX_DEV void wave_sync() {
  // All lanes belong to one wavefront: LDS and memory operations issue in program order, so
  // only the compiler has to be kept from reordering across this point.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// Keeps the compiler from folding an LDS access and an HBM access of two branches into one
// generic-address access (which would wait on both memory counters and on pending stores).
#define BPSX_KEEP_APART() asm volatile("")
// s_setprio takes an immediate
BPSX_DEV void set_wave_priority(int p) {
  if (p >= 3) __builtin_amdgcn_s_setprio(3);
  else if (p == 2) __builtin_amdgcn_s_setprio(2);
  else if (p == 1) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
}
// mask of the lanes where b holds (takes the condition as such, not widened to an integer and compared again)
BPSX_DEV unsigned long long lanes_where(bool b) { return __builtin_amdgcn_ballot_w64(b); }
// a lane mask held in scalar registers as a condition: sets algebra of conditions on the scalar unit,
// instead of conditions that are widened to integers and compared again for the next mask
BPSX_DEV bool in_mask(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
BPSX_DEV int uniform_i(int v) { return __builtin_amdgcn_readfirstlane(v); }
BPSX_DEV float lane_f(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }
BPSX_DEV uint32_t rlane(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lane); }

// The lane, for a part of the search that is entered once in a while: what is computed from it there is not worth
// keeping in registers all the time, which the compiler would do.
BPSX_DEV int lane_here(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}
// lanes from .. from + n - 1 (n < 64)
BPSX_DEV unsigned long long lane_range(int n, int from) {
  unsigned long long r;
  asm("s_bfm_b64 %0, %1, %2" : "=s"(r) : "s"(n), "s"(from));
  return r;
}
// index of the lowest set bit, -1 for an empty mask (the instruction's own convention)
BPSX_DEV int first_lane(unsigned long long mask) {
  int r;
  asm("s_ff1_i32_b64 %0, %1" : "=s"(r) : "s"(mask));
  return r;
}
// `Bits` bits of v from bit From on, as an instruction that the compiler cannot join to the scaling of an index: an LDS
// address is then two instructions instead of three
template <int From, int Bits> BPSX_DEV uint32_t field(uint32_t v) {
  uint32_t r;
  asm("v_bfe_u32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "n"(From), "n"(Bits));
  return r;
}
// Stores in the lanes of a mask, called by whole wavefronts (all lanes active before and after).  A store under
// a condition would get a branch around it, which costs a wavefront more than the store, and a loop
// with such a branch in it is rebuilt by the compiler as if all its branches were the lanes' own: every
// early way out then goes through copies of the loop's state and tests of flags.
typedef float Float4 __attribute__((ext_vector_type(4)));
BPSX_DEV uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; }
BPSX_DEV uint32_t lds_word(const uint32_t* p) {   // as another wavefront of the block may have written it
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
BPSX_DEV void lds_store_where(unsigned long long mask, uint2* p, uint32_t x, uint32_t y) {
  const unsigned long long v = ((unsigned long long)y << 32) | x;
  asm volatile("s_mov_b64 exec, %0\n\tds_write_b64 %1, %2\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(lds_address(p)), "v"(v) : "memory");
}
BPSX_DEV void lds_store_where(unsigned long long mask, uint32_t address, float4 f) {
  const Float4 v = {f.x, f.y, f.z, f.w};
  asm volatile("s_mov_b64 exec, %0\n\tds_write_b128 %1, %2\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(address), "v"(v) : "memory");
}
BPSX_DEV void lds_store_where(unsigned long long mask, uint32_t address, uint32_t x) {
  asm volatile("s_mov_b64 exec, %0\n\tds_write_b32 %1, %2\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(address), "v"(x) : "memory");
}
BPSX_DEV void lds_store_half_where(unsigned long long mask, uint32_t address, uint32_t x) {
  asm volatile("s_mov_b64 exec, %0\n\tds_write_b16 %1, %2\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(address), "v"(x) : "memory");
}
BPSX_DEV uint32_t lds_half(uint32_t address) { return *(__attribute__((address_space(3))) const uint16_t*)(uintptr_t)address; }
// (Offset: bytes behind p)
template <int Offset> BPSX_DEV void lds_min_where(unsigned long long mask, const uint32_t* p, uint32_t x) {
  asm volatile("s_mov_b64 exec, %0\n\tds_min_u32 %1, %2 offset:%3\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(lds_address(p)), "v"(x), "n"(Offset) : "memory");
}
// base[offset bytes] = v, base the same for all lanes
BPSX_DEV void store_where(unsigned long long mask, void* base, uint32_t offset, uint32_t v) {
  asm volatile("s_mov_b64 exec, %0\n\tglobal_store_dword %1, %2, %3\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(offset), "v"(v), "s"(base) : "memory");
}
BPSX_DEV void store_where(unsigned long long mask, void* base, uint32_t offset, uint32_t x, uint32_t y) {
  const unsigned long long v = ((unsigned long long)y << 32) | x;
  asm volatile("s_mov_b64 exec, %0\n\tglobal_store_dwordx2 %1, %2, %3\n\ts_mov_b64 exec, -1" :: "s"(mask), "v"(offset), "v"(v), "s"(base) : "memory");
}
// old with lane Lane replaced by v (uniform)
template <int Lane> BPSX_DEV uint32_t wlane_at(uint32_t old, uint32_t v) {
  asm("v_writelane_b32 %0, %1, %2" : "+v"(old) : "s"(__builtin_amdgcn_readfirstlane((int)v)), "n"(Lane));
  return old;
}
// index of the lowest bit that is not set, -1 if all are
BPSX_DEV int first_other_lane(unsigned long long mask) {
  int r;
  asm("s_ff0_i32_b64 %0, %1" : "=s"(r) : "s"(mask));
  return r;
}
BPSX_DEV unsigned long long with_lane(unsigned long long mask, int lane) {
  asm("s_bitset1_b64 %0, %1" : "+s"(mask) : "s"(lane));
  return mask;
}
BPSX_DEV unsigned long long without_lane(unsigned long long mask, int lane) {
  asm("s_bitset0_b64 %0, %1" : "+s"(mask) : "s"(lane));
  return mask;
}

// min(v, v of the lane that the DPP control names); lanes without such a lane, or outside the
// row mask (one bit per 16 lanes), keep v.  (The other lane's value defaults to the identity of
// the minimum, which lets the compiler fold the lane move into the v_min itself.)
template <int Ctrl, int RowMask> BPSX_DEV uint32_t umin_dpp(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, Ctrl, RowMask, 0xf, false);
  return o < v ? o : v;
}
// One word per node holds what the search loop reads of it besides the window.  The parent index is
// needed for the final path only and lives in HBM.  What the reference keeps besides is not needed:
//   - whether a node is open or closed only decides between a push and a modify, which the list
//     tells by whether it holds the node;
//   - the polygon that a node was reached from need not be left out of its neighbours: the way back
//     costs no less than the parent's own cost (costs only ever fall, both ways have the same
//     length, and rounding is monotonic), so its total is no better and it is left alone anyway.
//     (With a NaN two nodes would update each other for ever: there is none, see AEdge.)
// Without both a pass is some 25 of 630 instructions and three LDS accesses shorter: 1.286 -> 1.229 ms
// of k_geodesic at 16384 agents over mazes, 5 % off the longest of 64 searches alone on the GPU.
// A chain is linked by the byte offsets of the nodes' words (GeoWave::offset_of), so that a step along it is
// one access to LDS and three instructions.
constexpr uint32_t kNoPoly = 0xffffu;   // what the word at a chain's end has for a polygon
BPSX_DEV uint32_t link_id(uint32_t l) { return l & 0xffffu; }
BPSX_DEV uint32_t link_next(uint32_t l) { return l >> 16; }
BPSX_DEV uint32_t make_link(uint32_t id, uint32_t next) { return id | (next << 16); }

// Open-list entries: the total as a bit pattern, compared as an unsigned integer (totals are sums of
// distances between finite points, never negative and never NaN, and for such floats the integer
// order of the bits is the float order), and the node's index (bits 0-10) with its polygon index above
// it, so that the entry at the front names the edge records to fetch without a detour through LDS.
static_assert(kMaxNodes <= 2048, "open-list entries keep the node index in 11 bits");
constexpr uint32_t kEmptyKey = 0x7fefffffu;   // above +inf, and below the totals' bits that would make an entry of the list a NaN (OpenList)

// The open list as a sorted array in registers.  dtNodeQueue::pop returns the entry with the
// smallest total; while that smallest total is held by one entry only, which entry that is
// does not depend on how the reference's binary heap happens to be arranged.  So a search can
// keep its open list in any form that yields the minimum, as long as it notices when two
// entries share the smallest total (a tie, about one pop in ten thousand) and then asks the
// exact heap.
// An entry is 64 bits, the total over the packed node: as bits of a double, which for such numbers are in the
// order of the integers (denormal ones among them, which this target's double arithmetic keeps), so that one
// minimum and one maximum put an entry in its place.  Sorted, one per lane, the smallest in lane `base`, the greatest
// in the last but one; zeros below (node kNone), which are smaller than every entry, and a total above all in the last lane.  The
// list grows downwards: an entry that enters moves those below it down a lane, and what a pass
// expands leaves by a move of the base.
// Entries with totals from `bound` on are kept apart, in no order, in the wavefront's slot (GeoWave::far_list): they cost one store
// now, and a search comes back to half of them at most.  Where fewer than kRefill are left in registers, those up to a new
// bound come from there (refill); where more than kSplit are, the greater ones go there (split).  An entry whose node is
// updated meanwhile stays there, and is known by its total when it is looked at.
// (With up to 256 sorted entries in four register pairs, counted into place together and moved through LDS from the second
// pair on, and with totals and nodes selected apart and a lane permute that closed the gap of those that left: 600 to 860
// cycles of a pass instead of 500 to 600, 1500 instead of 600 over cluttered plans, whose lists have 73 entries on average and up to
// 300.  Steps of 64 agents 148 -> 136 us, of 1024 over room plans 589 -> 500, of 510 in two groups 1112 -> 968, of 4096 over
// cluttered plans 1280 -> 1190, of 16384 over mazes 805 -> 796, of 65536 over mixed scenes 2810 -> 2676, a reset of 2048 over mazes
// 476 -> 447, 300 queries over room plans 265 -> 242, 1000 pairs over a maze 949 -> 931.)
struct OpenList {
  static constexpr int kEnd = 63;       // the lane behind the last entry
  static constexpr int kMost = 62;      // entries in registers at most: there is always a zero below them
  static constexpr int kSplit = 54, kRefill = 9;   // a pass looks at nine entries
  // As much as the reference's heap has LDS for where a second wavefront keeps it.  (With 48 and 244, and 40 entries brought back at
  // most instead of 46, one search over cluttered plans in a few thousand outgrew the list, and a step of 4096 agents, as long as its
  // longest search, took 1154 us instead of 1060; 1024 agents over room plans 474 and 467, 65536 over mixed scenes 2518 and 2480.)
  static constexpr int kFarMost = 268;  // entries apart before a pass at most ...
  static constexpr int kFarKeep = 260;  // ... and, once those of updated nodes are gone, for the search to go on in this form
  static constexpr int kFarCap = 378;
  static_assert(kFarMost + kMost <= kFarCap, "a pass adds up to 48, and what a split adds was in registers");
  static constexpr int kMostOfAll = kSplit + kFarMost + 48;   // entries, behind a pass
  static constexpr uint32_t kEmpty = kEmptyKey;
  static constexpr uint32_t kNone = 0;   // the start node, which never enters the list again: what is read by it is there
  unsigned long long e;
  int base;
  uint32_t bound;
  int far;
  int low;         // a pass may go on while base - low, without a sign, is no more than
  uint32_t span;
  BPSX_DEV uint32_t total() const { return (uint32_t)(e >> 32); }
  BPSX_DEV uint32_t node() const { return (uint32_t)e; }
  static BPSX_DEV unsigned long long entry(uint32_t total, uint32_t node) { return ((unsigned long long)total << 32) | node; }
  BPSX_DEV int size() const { return kEnd - base; }
  BPSX_DEV void init(int lane, uint32_t first, uint32_t node) {
    e = lane == kEnd ? entry(kEmpty, kNone) : lane == kEnd - 1 ? entry(first, node) : 0ull;
    base = kEnd - 1;
    bound = kEmpty;
    far = 0;
    set_limits();
  }
  BPSX_DEV void set_limits() {
    low = far > kFarMost ? 2 * kEnd : kEnd - kSplit;
    span = (uint32_t)((far ? kEnd - kRefill : kEnd) - (kEnd - kSplit));
  }
  BPSX_DEV bool needs_care() const { return (uint32_t)(base - low) > span; }
  // lane L takes v of lane L + 1, lane 63 zero
  static BPSX_DEV uint32_t down1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
  }
  // lane L takes v of lane L - 1, lane 0 zero
  static BPSX_DEV uint32_t up1(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138 /* wave_shr:1 */, 0xf, 0xf, true);
  }
  // The entries of lanes `rest` (totals tb, nodes `packed`) enter, one after the other: every lane takes the smaller of the
  // entry above its own and the greater of its own and the new one.  As one piece, two entries a round, nine instructions each, of
  // which none waits for the scalar unit, in an order that keeps the distances that this hardware asks for and does
  // not watch over, two instructions between a vector instruction that writes a scalar register (a
  // lane read) and the vector instruction that reads it, and between one that writes
  // a register and the lane move that reads it.  With an odd number the last round's second is lane 63 (the first of an
  // empty mask, taken modulo 64), where tb is all ones: a NaN, which minima and maxima leave out.
  BPSX_DEV void enter(unsigned long long rest, uint32_t tb, uint32_t packed) {
    unsigned long long above, greater;
    int at;
    const unsigned long long end = entry(kEmpty, kNone);   // what lane 63, which has no lane above it, has there
    asm volatile("s_cmp_eq_u64 %[rest], 0\n\t"
                 "s_cbranch_scc1 2f\n"
                 "1:\n\t"
                 "s_ff1_i32_b64 %[at], %[rest]\n\t"
                 "s_bitset0_b64 %[rest], %[at]\n\t"
                 "v_readlane_b32 vcc_lo, %[packed], %[at]\n\t"
                 "v_readlane_b32 vcc_hi, %[tb], %[at]\n\t"
                 "v_mov_b32_dpp v42, v40 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_mov_b32_dpp v43, v41 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f64 v[44:45], vcc, v[40:41]\n\t"
                 "s_ff1_i32_b64 %[at], %[rest]\n\t"
                 "s_bitset0_b64 %[rest], %[at]\n\t"
                 "v_min_f64 v[40:41], v[42:43], v[44:45]\n\t"
                 "v_readlane_b32 vcc_lo, %[packed], %[at]\n\t"
                 "v_readlane_b32 vcc_hi, %[tb], %[at]\n\t"
                 "v_mov_b32_dpp v42, v40 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_mov_b32_dpp v43, v41 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"
                 "v_max_f64 v[44:45], vcc, v[40:41]\n\t"
                 "s_cmp_lg_u64 %[rest], 0\n\t"
                 "v_min_f64 v[40:41], v[42:43], v[44:45]\n\t"
                 "s_cbranch_scc1 1b\n\t"
                 "s_nop 1\n"
                 "2:"
                 : [rest] "+s"(rest), "+{v[40:41]}"(e), "={v[42:43]}"(above), "=&{v[44:45]}"(greater), [at] "=&s"(at)
                 : [tb] "v"(tb), [packed] "v"(packed), "2"(end)
                 : "vcc", "scc");
  }
  // The list with as many entries in the lanes from 0 on, in any order, as it has zeros at least: all of them in order, five
  // instructions for each of the 21 steps of a bitonic sort, where `enter` has nine for each entry.  A step leaves the smaller
  // of two entries in the lower one of two lanes and the greater one in the other.  For that the upper one of them has its
  // negative, and takes the smaller of that and the negative of what the other has.  Distances as in `enter`; the sign of
  // the next step is made between the last one's and the lane moves.
#define BPSX_SORT_STEP(get, next) "v_bfi_b32 v41, %[keep], v41, v44\n\tv_lshlrev_b32 v44, " next ", %[lane]\n\t" get "v_min_f64 v[40:41], v[40:41], -v[42:43]\n\t"
#define BPSX_SORT_DPP(ctrl) "v_mov_b32_dpp v42, v40 " ctrl " row_mask:0xf bank_mask:0xf\n\tv_mov_b32_dpp v43, v41 " ctrl " row_mask:0xf bank_mask:0xf\n\t"
#define BPSX_SORT_SHIFT4 "v_mov_b32_dpp v42, v40 row_shl:4 row_mask:0xf bank_mask:0x5\n\tv_mov_b32_dpp v43, v41 row_shl:4 row_mask:0xf bank_mask:0x5\n\t" \
                         "v_mov_b32_dpp v42, v40 row_shr:4 row_mask:0xf bank_mask:0xa\n\tv_mov_b32_dpp v43, v41 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
#define BPSX_SORT_LDS(op, which) op " v42, v40 " which "\n\t" op " v43, v41 " which "\n\ts_waitcnt lgkmcnt(0)\n\t"
#define BPSX_SORT_FAR "ds_bpermute_b32 v42, %[far], v40\n\tds_bpermute_b32 v43, %[far], v41\n\ts_waitcnt lgkmcnt(0)\n\t"
  BPSX_DEV void sort(int lane) {
    unsigned long long other, sign;
    const int far_lane = (63 - lane) * 4;
    asm volatile("v_lshlrev_b32 v44, 31, %[lane]\n\t"
                 // blocks of 2, 4, 8 lanes and so on: with the mirror image in the block, then with what is half a block away, a quarter ...
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "30")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[3,2,1,0]"), "31")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "29")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("row_half_mirror"), "30")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[2,3,0,1]"), "31")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "28")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("row_mirror"), "29")
                 BPSX_SORT_STEP(BPSX_SORT_SHIFT4, "30")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[2,3,0,1]"), "31")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "27")
                 BPSX_SORT_STEP(BPSX_SORT_LDS("ds_swizzle_b32", "offset:0x7c1f"), "28")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("row_ror:8"), "29")
                 BPSX_SORT_STEP(BPSX_SORT_SHIFT4, "30")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[2,3,0,1]"), "31")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "26")
                 BPSX_SORT_STEP(BPSX_SORT_FAR, "27")
                 BPSX_SORT_STEP(BPSX_SORT_LDS("ds_swizzle_b32", "offset:0x401f"), "28")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("row_ror:8"), "29")
                 BPSX_SORT_STEP(BPSX_SORT_SHIFT4, "30")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[2,3,0,1]"), "31")
                 BPSX_SORT_STEP(BPSX_SORT_DPP("quad_perm:[1,0,3,2]"), "31")
                 "v_and_b32 v41, %[keep], v41\n\t"
                 "s_nop 1"
                 : "+{v[40:41]}"(e), "=&{v[42:43]}"(other), "=&{v[44:45]}"(sign)
                 : [lane] "v"(lane), [far] "v"(far_lane), [keep] "s"(0x7fffffff)
                 : "memory");
  }
#undef BPSX_SORT_STEP
#undef BPSX_SORT_DPP
#undef BPSX_SORT_SHIFT4
#undef BPSX_SORT_LDS
#undef BPSX_SORT_FAR
  // v as a select operand under a lane mask that a scalar instruction has written (the compiler does not know the
  // select for a vector instruction, which has to keep two instructions' distance from a comparison: a mask that a
  // comparison alone has made takes a plain select on in_mask.  tests/test_inline_asm_distances.py reads the assembly.)
  static BPSX_DEV uint32_t pick(unsigned long long mask, uint32_t yes, uint32_t no) {
    uint32_t r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(no), "v"(yes), "s"(mask));
    return r;
  }
  // A pass's changes: the first c entries leave, and so does the entry of every node in lanes
  // `known` that has one here (a modify; a node without an entry is pushed); the nodes in lanes `upd`,
  // packed and with total bits tb, enter.
  // Returns the node of entry `row` of the new list and the total of the one behind it (of kNone and kEmpty
  // where there is none).
  BPSX_DEV uint2 merge(int c, unsigned long long upd, unsigned long long known, uint32_t tb, uint32_t packed, int row) {
    base += c;
    const unsigned long long left = lane_range(base, 0);
    e = in_mask(left) ? 0ull : e;
    const int n = __popcll(upd);
    while (known) {
      const int src = first_lane(known);
      known = without_lane(known, src);
      const unsigned long long old = lanes_where(node() == rlane(packed, src));   // (kNone is no node that is updated)
      if (!old) continue;
      // those below it move up a lane
      const unsigned long long upTo = old ^ (old - 1ull);
      const uint32_t t = up1(total()), nd = up1(node());
      e = in_mask(upTo) ? entry(t, nd) : e;
      base++;
    }
    base -= n;
    int from = (base + row) * 4;
    asm volatile("" : "+v"(from));   // (before the entries enter, for which it does not wait)
    enter(upd, tb, packed);
    return front_from(from);
  }
  BPSX_DEV uint2 front(int row) const { return front_from((base + row) * 4); }
  BPSX_DEV uint2 front_from(int from) const {
    return make_uint2((uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)node()), (uint32_t)__builtin_amdgcn_ds_bpermute(from + 4, (int)total()));
  }
};

struct AstarState {
  int lastBest;      // the goal's node once it has been popped
  bool outOfNodes;
  OpenList ol;
  int logEnd;        // records in the slot's operation log
  int synced;        // records already applied to the replay's heap
  int replaySize;    // entries of that heap, which the slot keeps between replays
  int replayNodes;       // nodes created by the records already applied
  uint32_t replayRoot;   // packed node of the entry at its root after a replay
};

constexpr uint32_t kFollowEnd = 0xffffu, kFollowQuit = 0xffffffffu;   // see follow

enum AstarExit { kAstarOn = -1, kAstarEmpty = 0, kAstarGoal = 1, kAstarGrowLinks = 2, kAstarGrowHeap = 3, kAstarTie = 4, kAstarLogFull = 5, kAstarCare = 6 };

// Two correctly rounded square roots, the values sqrtf returns on the host, of arguments that are zero or
// at least 2^-96 and finite, as squared distances between points of a mesh are; a wavefront that meets
// another (or zero, which this form would make NaN) takes the library routine.  One test of the
// arguments' range for both.  One step from the reciprocal root's estimate, with the residual exact
// through a fused multiply-add.  That by itself is not enough (an estimate a unit in the last place off can give the
// neighbouring float); with this hardware's estimates it is right for every float from 2^-96 up, all of which
// tests/test_gpu_roots.py compares.  (The estimate of the root and the residuals of its two
// neighbours, which of the three it is, are nine instructions instead of five.)
BPSX_DEV void sqrt_exact2(float x, float y, float* rx, float* ry) {
  const uint32_t lo = 0x0f800000u, span = 0x7f800000u - lo;
  const uint32_t xr = __float_as_uint(x) - lo, yr = __float_as_uint(y) - lo;
  const unsigned long long others = lanes_where((xr > yr ? xr : yr) >= span);
  const float px = __builtin_amdgcn_rsqf(x), py = __builtin_amdgcn_rsqf(y);
  const float gx = x * px, gy = y * py;
  float sx = fmaf(fmaf(-gx, gx, x), 0.5f * px, gx), sy = fmaf(fmaf(-gy, gy, y), 0.5f * py, gy);
  asm volatile("" : "+v"(sx), "+v"(sy));   // the branch comes behind them, when the test has long been made
  if (__builtin_expect(others != 0, 0)) { sx = sqrtf(x); sy = sqrtf(y); }
  *rx = sx; *ry = sy;
}

BPSX_DEV float tri_area2d(const float* a, const float* b, const float* c) {
  const float abx = b[0] - a[0], abz = b[2] - a[2];
  const float acx = c[0] - a[0], acz = c[2] - a[2];
  return acx * abz - abx * acz;
}
BPSX_DEV bool vequal(const float* a, const float* b) {
  const float thr = (1.0f / 16384.0f) * (1.0f / 16384.0f);
  const float dx = b[0] - a[0], dy = b[1] - a[1], dz = b[2] - a[2];
  return dx * dx + dy * dy + dz * dz < thr;
}

}  // namespace bpsx
#endif  // BPSX_GEODESIC_COMMON_H

#ifndef BPSX_GEO_NS
#define BPSX_GEO_NS geo
#endif
namespace bpsx {
namespace BPSX_GEO_NS {

// As many links as let ten blocks of two wavefronts share a CU's 160 KB, which are given out in units of
// 1280 bytes: 12 units a block, 20 wavefronts a CU, which is also what 96 vector registers allow.
// (With 1215 links, 14 units and nine blocks: 4.43 instead of 3.80 ms at 65536 agents over mixed
// scenes, within the noise at 16384 over mazes.)
#ifndef BPSX_LINKS_LDS
#define BPSX_LINKS_LDS 896
#endif
#ifndef BPSX_WINDOW
#define BPSX_WINDOW 128
#endif
constexpr int kLinksLds = BPSX_LINKS_LDS;   // nodes whose link word is kept in LDS
constexpr int kWindow = BPSX_WINDOW;        // most recent nodes whose position and cost are kept in LDS
#ifndef BPSX_HASH
#define BPSX_HASH 512
#endif
constexpr int kHashSize = BPSX_HASH;        // buckets of the node pool's hash table
// Where all chains end: the word behind the links in LDS, which names no polygon and itself as the next.
constexpr uint32_t kChainEnd = 4u * (uint32_t)kLinksLds;
constexpr uint32_t kEndWord = kNoPoly | (kChainEnd << 16);
static_assert(4 * (kMaxNodes + 1) <= 0xffff, "offsets of links have 16 bits");
constexpr bool kAllLds = kWindow >= kMaxNodes;   // every node is kept in LDS, and none in HBM
#ifndef BPSX_FOLLOWER
#define BPSX_FOLLOWER 0
#endif
constexpr bool kFollower = BPSX_FOLLOWER;   // a second wavefront keeps the reference's heap up to date (follow)
static_assert(!kAllLds || kLinksLds >= kMaxNodes, "a pool in LDS has its links there too");
#ifndef BPSX_TAG_SLOTS
#define BPSX_TAG_SLOTS 256
#endif
constexpr int kTagSlots = BPSX_TAG_SLOTS;
constexpr int kRows = 8;                    // nodes expanded per pass of astar_fast, one per row of 64 / kRows lanes
constexpr int kRowLanes = 64 / kRows;
constexpr int kRowShift = 3;
static_assert(kRowLanes == (1 << kRowShift) && kRowLanes > kNvp, "a row needs a lane per edge and one for the node itself");
// lanes of the rows below j
constexpr unsigned long long rows_below(int j) { return j * kRowLanes >= 64 ? ~0ull : (1ull << (j * kRowLanes)) - 1ull; }
static_assert((kWindow & (kWindow - 1)) == 0 && kWindow >= 2 * kNvp, "window must be a power of two");

// LDS of one wavefront.
struct GeoLds {
  alignas(16) uint16_t first[kHashSize];
  // Node links: polygon index | offset of the next node's link in the hash chain << 16.  Behind them the
  // marks of which lane of a pass updates a polygon first (see astar_fast), all kEndWord between passes
  // and while chains are walked: the first of them is the word that ends every chain.
  alignas(16) uint32_t n_link[kLinksLds + kTagSlots];
  alignas(16) float4 w_node[kWindow];   // position, cost
  BPSX_DEV uint32_t* marks() { return n_link + kLinksLds; }
#if BPSX_FOLLOWER
  // What the two wavefronts of a search share (see follow): how far the log has arrived, the heap and its size,
  // the search's state, how far the log has been read, and the entry that a search begins with.
#if BPSX_WINDOW >= 2048
  // Next to every node, the parent indices; where a lane without a node would store its own, `arrived`.
  uint16_t parents[kMaxNodes];
  uint16_t arrived, unused;
#endif
  alignas(16) uint2 ref_heap[380];
  uint2 start;
  uint32_t published, applied, heap_size;
#if BPSX_WINDOW < 2048
  uint16_t arrived, unused;
#endif
  BPSX_DEV uint2* heap() { return ref_heap; }
#else
  BPSX_DEV uint2* heap() { return reinterpret_cast<uint2*>(n_link + kLinksLds); }
#endif
};
// After A* its LDS is dead; the funnel reuses it for the corridor and its portals.  The
// corridor is written while the nodes' links are still being read: it lies over the hash
// heads, which are no longer needed by then.
struct FunnelLds {
  uint16_t corridor[kMaxPath];
  uint16_t pad[kHashSize - kMaxPath];
  float portals[kMaxPath][6];
};
static_assert(offsetof(FunnelLds, portals) == offsetof(GeoLds, n_link), "corridor must overlay the hash heads only");
static_assert(!kFollower || sizeof(FunnelLds) <= offsetof(GeoLds, w_node) + kWindow * sizeof(float4),
              "the portals must end before what the two wavefronts share: the follower may still be at work when they are written");
union GeoShared {
  GeoLds a;
  FunnelLds f;
};

// Accessors take the instantiation's spill switch S: with S false, or with room in LDS for the links
// of all nodes, every node index is below kLinksLds and no address-space branch is generated.
struct GeoWave {
  using Shared = GeoShared;
  static constexpr bool kFollowed = kFollower;
  GeoLds* L;
  GeoSlot* ws;
  int lane;
  int nodeCount;
  uint32_t linkSpills, heapSpills;   // queries that left the LDS links / whose heap, once they went on with it, left LDS
#ifdef BPSX_PHASE_TIMING
  unsigned long long phase[8], phase_t0;
#endif
  uint32_t exactRuns;                // queries that went on with the reference's heap
  uint32_t tieReplays;               // ties resolved by replaying the operation log through the exact heap
  uint32_t pairTies;                 // passes that took two nodes of equal total in one go
#if BPSX_FOLLOWER
  uint32_t epoch;                    // of the search, in the upper 16 bits (see follow)
  BPSX_DEV void publish(uint32_t word) const { lds_store_where(1ull, lds_address(&L->published), word); }
  // until the follower has done all that the word asks for
  BPSX_DEV void settle(uint32_t word) const {
    while ((uint32_t)uniform_i((int)lds_word(&L->applied)) != word) __builtin_amdgcn_s_sleep(1);
    wave_sync();
  }
#endif

  // ---------------------------------------------------------------- node pool
  // A node's index is handled as four times itself, the offset of its word among the links.  Offset of its link
  // within the chains: that of the links in LDS, beyond them that of the slot's shifted past kChainEnd.
  template <bool S> static BPSX_DEV uint32_t offset_of(uint32_t i4) {
    return !S || kLinksLds >= kMaxNodes ? i4 : i4 + (i4 >= kChainEnd ? 4u : 0u);
  }
  template <bool S> static BPSX_DEV uint32_t node4_at(uint32_t offset) {
    return !S || kLinksLds >= kMaxNodes ? offset : offset - (offset > kChainEnd ? 4u : 0u);
  }
  // where node i's link lies
  template <bool S> BPSX_DEV uint32_t link(int i) const {
    if (!S || kLinksLds >= kMaxNodes || i < kLinksLds) return L->n_link[i];
    BPSX_KEEP_APART();
    const uint32_t v = ws->links[i];
    BPSX_KEEP_APART();
    return v;
  }
  // and that of the node as its chain's first
  template <bool S> BPSX_DEV void set_links(unsigned long long mask, uint32_t i4, uint32_t v, uint32_t first, uint32_t own) const {
    if (!S || kLinksLds >= kMaxNodes) {
      asm volatile("s_mov_b64 exec, %0\n\tds_write_b32 %1, %2\n\tds_write_b16 %3, %4\n\ts_mov_b64 exec, -1"
                   :: "s"(mask), "v"(lds_address(L->n_link) + i4), "v"(v), "v"(first), "v"(own) : "memory");
    } else {
      const unsigned long long near = lanes_where(i4 < kChainEnd);
      lds_store_where(mask & near, lds_address(L->n_link) + i4, v);
      store_where(mask & ~near, ws->links, i4, v);
      lds_store_half_where(mask, first, own);
    }
  }
  // The entries that the open list keeps apart, over the links that LDS has places for
  BPSX_DEV void* far_list() const {
    static_assert(OpenList::kFarCap * sizeof(uint2) <= kLinksLds * sizeof(uint32_t) && offsetof(GeoSlot, links) % 8 == 0, "the slot's links begin behind them");
    return ws->links;
  }
  // node i, whose position and cost are not looked for in the window; and a node and its parent index stored outside of it
  BPSX_DEV float4 node(int i) const {
#if BPSX_WINDOW >= 2048
    return L->w_node[i];
#else
    return ws->nodes[i];
#endif
  }
  // the node and its parent index, in the lanes of mask; offsets of both by shifts of i4, which the caller keeps the
  // compiler from knowing as a multiple of the index (it would multiply)
  // (With all nodes in LDS: the parent index only.)
  BPSX_DEV void keep_node(unsigned long long mask, uint32_t i4, float4 n, uint32_t parent) const {
#if BPSX_WINDOW >= 2048
    asm volatile("s_mov_b64 exec, %0\n\tds_write_b16 %1, %2\n\ts_mov_b64 exec, -1"
                 :: "s"(mask), "v"(lds_address(L->parents) + (i4 >> 1)), "v"(parent) : "memory");
#else
    const Float4 v = {n.x, n.y, n.z, n.w};
    asm volatile("s_mov_b64 exec, %0\n\tglobal_store_dwordx4 %1, %2, %3\n\tglobal_store_short %4, %5, %6\n\ts_mov_b64 exec, -1"
                 :: "s"(mask), "v"(i4 << 2), "v"(v), "s"(ws->nodes), "v"(i4 >> 1), "v"(parent), "s"(ws->parents) : "memory");
#endif
  }
#if BPSX_FOLLOWER
  // A pass's updated nodes and its records of the log, at `offset` bytes, and as `arrived` the number of records before
  // the pass: those were stored before it asked for its edge records, for which it has waited, so they
  // are in the L2.  All lanes that store a record store that number, or only the header's, which
  // has no node, where its parent index would go.
  BPSX_DEV void keep_pass(unsigned long long mask, unsigned long long header, uint32_t i4, float4 n, uint32_t parent, uint32_t before, uint32_t offset,
                          uint32_t key, uint32_t word) const {
    const unsigned long long r = ((unsigned long long)word << 32) | key;
#if BPSX_WINDOW >= 2048
    (void)n;
    static_assert(kLinksLds == kMaxNodes && offsetof(GeoLds, arrived) == offsetof(GeoLds, parents) + kChainEnd / 2, "the header's lane has kChainEnd for a node");
    const uint32_t p = wlane_at<62>(parent, before);
    asm volatile("s_mov_b64 exec, %0\n\tglobal_store_dwordx2 %1, %2, %3\n\tds_write_b16 %4, %5\n\ts_mov_b64 exec, -1"
                 :: "s"(mask | header), "v"(offset), "v"(r), "s"(ws->oplog), "v"(lds_address(L->parents) + (i4 >> 1)), "v"(p) : "memory");
#else
    const Float4 v = {n.x, n.y, n.z, n.w};
    asm volatile("s_mov_b64 exec, %0\n\tglobal_store_dwordx4 %1, %2, %3\n\tglobal_store_short %4, %5, %6\n\t"
                 "s_mov_b64 exec, %7\n\tglobal_store_dwordx2 %8, %9, %10\n\tds_write_b16 %11, %12\n\ts_mov_b64 exec, -1"
                 :: "s"(mask), "v"(i4 << 2), "v"(v), "s"(ws->nodes), "v"(i4 >> 1), "v"(parent), "s"(ws->parents),
                    "s"(mask | header), "v"(offset), "v"(r), "s"(ws->oplog), "v"(lds_address(&L->arrived)), "v"(before) : "memory");
#endif
  }
#endif
  // the multiply as the full-rate 24-bit instruction (polygon indices have 15 bits)
  static BPSX_DEV uint32_t hash_product(uint32_t ip) {
    uint32_t m;
    asm("v_mul_u32_u24 %0, %1, %2" : "=v"(m) : "v"(ip), "s"(0x9e3779u));
    return m;
  }
  // the bucket, of `size` ones
  template <int size> static BPSX_DEV uint32_t bucket_of(uint32_t product) {
    static_assert((size & (size - 1)) == 0);
    return field<9, __builtin_ctz(size)>(product);
  }
  static BPSX_DEV uint32_t hash(uint32_t ip) { return bucket_of<kHashSize>(hash_product(ip)); }
  // where in the window node i4 lies (any place for one that has left it)
  static BPSX_DEV uint32_t window_slot(uint32_t i4) { return kAllLds ? (i4 >> 2) & (kWindow - 1) : field<2, __builtin_ctz(kWindow)>(i4); }
  BPSX_DEV void clear_marks() {
    static_assert(kTagSlots == 256, "one 16-byte store per lane");
    reinterpret_cast<uint4*>(L->marks())[lane] = make_uint4(kEndWord, kEndWord, kEndWord, kEndWord);
  }
  BPSX_DEV void clear() {
    constexpr uint32_t two = kChainEnd | (kChainEnd << 16);
    static_assert(kHashSize % 512 == 0, "16 bytes a lane");
    static_for<0, kHashSize / 512>([&](auto K) BPSX_INLINE_LAMBDA {
      reinterpret_cast<uint4*>(L->first)[64 * decltype(K)::value + lane] = make_uint4(two, two, two, two);
    });
    clear_marks();
    nodeCount = 0;
    wave_sync();
  }
  // Offset of polygon ip's node (offset_of), whose chain's first has address `chain`, kChainEnd if it has none; *head receives that of the bucket's first
  // node (what a new node of this bucket links to).  Called by all lanes (those without a polygon with
  // valid == false): the chains are walked in step, one LDS access per lane and round, until every lane
  // has hit or run out, which reads the word at the chains' end again.
  template <bool S> BPSX_DEV uint32_t find(unsigned long long valid, uint32_t ip, uint32_t chain, uint32_t* head) const {
    uint32_t cur = lds_half(chain);
    cur = in_mask(valid) ? cur : kChainEnd;
    *head = cur;
    uint32_t found = kChainEnd;
    const char* links = reinterpret_cast<const char*>(L->n_link);
    do {
      uint32_t l;
      if (!S || kLinksLds >= kMaxNodes) {
        l = *reinterpret_cast<const uint32_t*>(links + cur);
      } else {
        l = *reinterpret_cast<const uint32_t*>(links + (cur < kChainEnd ? cur : kChainEnd));
        const unsigned long long far = lanes_where(cur > kChainEnd);
        if (far) {
          BPSX_KEEP_APART();
          const uint32_t f = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(ws->links) + (in_mask(far) ? cur - 4u : 0u));
          BPSX_KEEP_APART();
          l = in_mask(far) ? f : l;
        }
      }
      const bool hit = link_id(l) == ip;
      found = hit ? cur : found;
      cur = hit ? kChainEnd : link_next(l);
    } while (lanes_where(cur != kChainEnd));
    return found;
  }
};

// The reference's heap (dtNodeQueue, DetourNode.cpp:150-200), needed when the sorted list cannot say
// what comes first (a tie) or cannot hold what is open: position q (root = 1) in entry q of an array
// in LDS, over the conflict marks (but the first two) and the window, or in the wavefront's slot.  All lanes
// work on one operation: a push takes one round of accesses, a pop one up to 128 entries (searches
// over mazes keep 23 on average, over cluttered plans 73), beyond that two, in the slot one per five levels.  Bound by
// those rounds and by a lone wavefront's instructions between them, five cycles each and twenty where a result goes
// from the vector to the scalar unit and back; a replay is a chain of them.  In cycles, a pop of 63, 100, 200, 300 entries
// takes 200, 250, 510, 590, a push 190, a pass of the log some 230 besides.
// (With a lane for every entry, which looked at its sibling and was on the route if none of its ancestors was the
// greater of a pair, two masked stores per 64 entries, a pop took 300, 510, 820, 1070 cycles; with every row of a pass
// looking for its records among the lanes, a pass 500 besides.  Steps of 4096 agents over cluttered plans, of which the longest
// search waits for this at a tie, 1069 -> 965 us, of 16384 over mazes 769 -> 734, of 65536 over mixed scenes 2505 -> 2469,
// 1000 pairs over a maze 813 -> 732.)
// (In the slot, heaps of up to 256 entries had a form of their own with one round, and geo_long's stayed in LDS up to 639 entries.
// Searches of equal totals over a room, all of whose heaps come to leave LDS, and some back to a few entries: 400 of them 2.67 ms with
// those and the pops above, now 2.58; 4000 4.86 and 4.60.)
// (In registers, entry q in lane q mod 64, with the entries that move exchanged between lanes instead of through
// LDS, the levels from the seventh on one after the other on the scalar unit: 300, 465, 800, 1025 cycles a pop, 250 to 670
// a push, 804 us for 1000 pairs.)
constexpr int kHeapLds = kFollower ? 379 : kWindow == 128 ? 383 : 511;   // entries that it holds; a pop looks at 511 at most
static_assert(kHeapLds <= 511);
static_assert(kFollower || (kTagSlots * 4 + kWindow * 16) / (int)sizeof(uint2) > kHeapLds, "an entry 0, which is none, and those");
static_assert(kLinksLds % 4 == 0 && offsetof(GeoLds, w_node) == offsetof(GeoLds, n_link) + 4 * (kLinksLds + kTagSlots),
              "the marks are accessed as 16 bytes, and the heap lies over the marks and the window");
static_assert(kRows * kNvp <= 48 && kHeapLds >= OpenList::kMostOfAll + kRows, "a heap with as many entries as the sorted list must fit");
template <bool Lds> struct RefHeap {
  uint2* h;    // total bits, packed node
  int size, lane;
  uint32_t ways, way;   // as bits, the positions above position `lane`, and those of them that it lies to the right below
  BPSX_DEV RefHeap(uint2* entries, int n, int lane_) : h(entries), size(uniform_i(n)), lane(lane_) {
    ways = 0; way = lane == 0;   // lane 0 is no position
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      if ((lane >> k) < 2) continue;
      ways |= 1u << (lane >> (k + 1));
      way |= (uint32_t)((lane >> k) & 1) << (lane >> (k + 1));
    }
  }
  // h[at] = e in the lanes of mask (in LDS without a branch around it)
  BPSX_DEV void put(unsigned long long mask, uint32_t at, uint32_t x, uint32_t y) const {
    if constexpr (Lds) {
      lds_store_where(mask, &h[at], x, y);
    } else {
      if (in_mask(mask)) h[at] = make_uint2(x, y);
    }
  }
  // The entry (t, n), on its way up from position q: lane k has position q >> k and looks at the entry
  // above.  Those with a greater total, a run from q upwards, move down one level each.
  BPSX_DEV void bubble_up(int q, uint32_t t, uint32_t n) {
    const uint32_t at = (uint32_t)q >> (lane & 31);
    const uint2 above = h[at >> 1];
    wave_sync();
    const unsigned long long falls = lanes_where(above.x > t) & lanes_where(at > 1u);
    put(falls ^ (falls + 1ull), at, in_mask(falls) ? above.x : t, in_mask(falls) ? above.y : n);   // and the next lane
    wave_sync();
  }
  // where node n's entry is, 0 if it has none
  template <int K> BPSX_DEV int position(uint32_t n) const {
    unsigned long long m[K];
#pragma unroll
    for (int k = 0; k < K; ++k) m[k] = lanes_where(h[64 * k + lane].y == n);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      m[k] &= upto(size - 64 * k) & (k ? ~0ull : ~1ull);
      if (m[k]) return 64 * k + first_lane(m[k]);
    }
    return 0;
  }
  BPSX_DEV int position(uint32_t n) const {
    if (size < 64) return position<1>(n);
    if (size < 128) return position<2>(n);
    if (size < 256) return position<4>(n);
    for (int base = 1; base <= size; base += 64) {
      const int i = base + lane;
      const unsigned long long m = lanes_where(h[i <= size ? i : size].y == n);
      if (m) { const int q = base + first_lane(m); return q <= size ? q : size; }
    }
    return 0;
  }
  // lanes 0 .. i, none below 0
  static BPSX_DEV unsigned long long upto(int i) { return i < 0 ? 0ull : i >= 63 ? ~0ull : (2ull << i) - 1ull; }
  BPSX_DEV void push(uint32_t t, uint32_t n) { bubble_up(++size, t, n); }
  // a node that has an entry takes a smaller total (dtNodeQueue::modify), one without gets one (push)
  BPSX_DEV void update(bool mayHaveEntry, uint32_t t, uint32_t n) {
    if (mayHaveEntry) {
      const int q = position(n);
      if (q) return bubble_up(q, t, n);
    }
    bubble_up(++size, t, n);
  }
  // The root leaves: the hole moves to a leaf along the smaller children (the left one of two
  // equal), then the former last entry rises from there.  Totals never decrease along that route,
  // so the entry lands above the first route element greater than it and nothing below moves.
  //
  // Lane p looks after position p and has both entries below it.  It is on the route when the smaller entries of all the
  // positions above it lie towards it, which is one comparison of bits; there it takes the smaller of its two, or the
  // last entry if that is smaller still.  So a pop of up to 64 entries is one round of reads and one masked store, and of up to 128
  // another store of one entry; what is below the seventh level is looked at in a second round.
  BPSX_DEV void pop_at_once() {
    const int s = size;
    const uint2 last = h[s];
    const uint4 below = reinterpret_cast<const uint4*>(h)[lane];
    wave_sync();
    size = s - 1;
    // the left, and the right entry below is there (before the last)
    const unsigned long long lefts = lanes_where(2 * lane < s), rights = lanes_where(2 * lane < size);
    const unsigned long long right = lanes_where(below.z < below.x) & rights;
    const uint32_t x = in_mask(right) ? below.z : below.x, y = in_mask(right) ? below.w : below.y;
    const unsigned long long route = lanes_where((ways & (uint32_t)right) == way);
    const unsigned long long takes = route & lefts & lanes_where(x <= last.x);
    const unsigned long long rest = route & ~takes;
    if (__builtin_expect(rest != 0, 1)) {
      put(with_lane(takes, first_lane(rest)), (uint32_t)lane, in_mask(takes) ? x : last.x, in_mask(takes) ? y : last.y);
      wave_sync();
      return;
    }
    put(takes, (uint32_t)lane, x, y);
    const int bottom = 63 - __builtin_clzll(takes);
    uint32_t hole = 2u * (uint32_t)bottom + (uint32_t)((right >> bottom) & 1ull);
    if (2 * (int)hole < s) {
      // lane 1 has the hole, lanes 2 and 3 the positions below it
      const uint32_t at = lane < 2 ? hole : 2u * hole + (uint32_t)(lane & 1);
      const uint32_t from = 2u * at < (uint32_t)s ? at : hole;
      const uint4 two = reinterpret_cast<const uint4*>(h)[from];
      wave_sync();
      const uint32_t r2 = (uint32_t)lanes_where(two.z < two.x && 2u * at + 1u < (uint32_t)s);
      const uint32_t tx = in_mask(r2) ? two.z : two.x, ty = in_mask(r2) ? two.w : two.y;
      const uint32_t t2 = (uint32_t)lanes_where(tx <= last.x && 2u * at < (uint32_t)s);
      if (t2 & 2u) {
        const uint32_t next = 2u + ((r2 >> 1) & 1u);
        const bool deeper = (t2 >> next) & 1u;
        put(2u | (deeper ? 1u << next : 0u), at, tx, ty);
        hole = 2u * hole + ((r2 >> 1) & 1u);
        if (deeper) hole = 2u * hole + ((r2 >> next) & 1u);
      }
    }
    put(1ull, hole, last.x, last.y);
    wave_sync();
  }
  BPSX_DEV void pop() {
    if constexpr (Lds) return pop_at_once();
    uint32_t anc0, anc1;   // as bits, the entries of 64 at and above entry `lane`, but for the root
    {
      unsigned long long a = 0;
#pragma unroll
      for (int k = 0; k < 5; ++k)
        if ((lane >> k) >= 2) a |= 1ull << (lane >> k);
      anc0 = (uint32_t)a; anc1 = (uint32_t)(a >> 32);
    }
    const int depth = 31 - __clz(lane | (lane == 0));
    uint32_t lt = 0, ln = 0;
    int root = 1, at = 1;
    for (;;) {
      // lane l >= 1: node l of the subtree under `root`, six levels of it; lane 0: the last entry
      const int pos = lane == 0 ? size : (root << depth) | (lane & ((1 << depth) - 1));
      const bool there = pos < size;
      uint2 e = h[pos <= size ? pos : 1];
      if (root == 1) { lt = rlane(e.x, 0); ln = rlane(e.y, 0); }
      if (!there) e.x = kEmptyKey;
      // one comparison with the neighbouring lane says which of two siblings the hole moves to
      const uint32_t sibling = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e.x, 0xb1 /* quad_perm:[1,0,3,2] */, 0xf, 0xf, false);
      constexpr unsigned long long kOdd = 0xaaaaaaaaaaaaaaaaull;
      const unsigned long long less = lanes_where(e.x < sibling);
      const unsigned long long greater = ~((less & kOdd) | (~(less >> 1) & ~kOdd));
      // the hole comes by where neither the node nor one of its ancestors is the greater of its pair
      const bool take = there && e.x <= lt && ((anc0 & (uint32_t)greater) | (anc1 & (uint32_t)(greater >> 32))) == 0;
      const int q = 63 - __builtin_clzll(lanes_where(take && lane > 1) | 2ull);   // the deepest that moves up
      wave_sync();
      put(lanes_where(take && lane > 1), (uint32_t)pos >> 1, e.x, e.y);
      wave_sync();
      const int m = 31 - __builtin_clz((uint32_t)q);
      at = (root << m) | (q & ((1 << m) - 1));
      if (m < 5 || 2 * at >= size) break;
      root = at;
    }
    put(1ull, (uint32_t)at, lt, ln);   // of a heap of one entry: that entry once more, beyond the end
    size--;
    wave_sync();
  }
};

// Applies one pass of the log to the reference's heap.  The lanes hold records; the pass's begin in lane h and
// end with the first of `headers` from there.  seen: nodes created by the passes before.  Returns the number of
// records, header included.
BPSX_DEV int apply_pass(RefHeap<true>& rh, uint32_t rk, uint32_t rw, unsigned long long headers, int h, int& seen) {
  const int end = h + __builtin_ctzll(headers >> h);
  const uint32_t hk = rlane(rk, end), hw = rlane(rw, end);
  const int c = (int)(hk & 0xffu), nrec = (int)(hk >> 8);
  // rows in the reference's order: the first two swap when the heap has row 1's node on top
  if ((hw & kOpUnordered) && (uint32_t)uniform_i((int)rh.h[1].y) != (hw & 0x3ffffffu)) {
    const unsigned long long mine = lane_range(nrec, h);
    const uint32_t myRow = (rw >> 26) & 7u;
    const int n0 = __popcll(lanes_where(myRow == 0u) & mine), n1 = __popcll(lanes_where(myRow == 1u) & mine);
    const int at = rh.lane - h;
    const int from = 4 * (at < 0 || at >= n0 + n1 ? rh.lane : at < n1 ? rh.lane + n0 : rh.lane - n1);
    rk = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)rk);
    rw = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)rw);
    rw ^= in_mask(lane_range(n0 + n1, h)) ? 1u << 26 : 0u;
    asm("" : "+v"(rk), "+v"(rw));   // they have come: else every record waits as if they might not
  }
  // the pass's new nodes are those whose index had not been given out before it
  const int before = uniform_i(seen);
  int row = -1, news = 0;
  uint32_t word = rlane(rw, h), key = rlane(rk, h);
  for (int i = h; i < end;) {
    for (const int to = (int)((word >> 26) & 7u); row < to; ++row) rh.pop();
    const uint32_t total = key, node = word & 0x3ffffffu;
    i++;
    word = rlane(rw, i); key = rlane(rk, i);
    if ((int)(node & 0x7ffu) >= before) {
      news++;
      rh.push(total, node);
    } else {
      rh.update(true, total, node);   // (a known node without an entry, closed or of a row before, is pushed)
    }
  }
  for (; row < c - 1; ++row) rh.pop();
  seen = before + news;
  return 1 + nrec;
}

#if BPSX_FOLLOWER
// Where a search has a second wavefront to itself, that one applies the log to the reference's heap while the search
// goes on, and a tie costs the search a question instead of a replay of all that came before.  Both are of
// one block, so both are there until the block ends, and each wait of one is for something that the other does
// in any case.
//   published   written by the search: its epoch << 16 | 0 when it begins, the records of the log when it asks for the
//               heap, kFollowEnd when it is over; kFollowQuit when there will be no more searches.
//   arrived     written by every pass: the records of the log that may be read (GeoWave::keep_pass).
//   applied     written by the follower: the last word of `published` that it has done all for.  The heap is the
//               search's from then on, until it goes on with another pass.
// A new search begins, and writes over the log and the heap, only when the follower has answered the end of the one
// before (astar waits for that).  The end of all searches it does not answer: what it has fetched by then is not applied.
// Bound by the heap's operations (RefHeap), which take a little longer than the search's passes where lists are long.  For the
// search it is one or two instructions a pass, and two fewer around its stores.  (With `arrived` stored apart, five
// instructions a pass, it cost the searches without ties 2.5 %: steps of 64 agents 161 -> 165 us, a reset of 2048 over
// mazes 471 -> 483.)
static_assert(kOpLogCap < (int)kFollowEnd, "a count of records is told from the marks");
BPSX_DEV void follow_init(GeoLds* L) { L->published = L->applied = kFollowEnd; }   // of a search before the first
BPSX_DEV void follow(GeoLds* L, const GeoSlot* ws, int lane) {
  lane = lane_here(lane);
  RefHeap<true> rh(L->heap(), 0, lane);
  const unsigned long long* log = reinterpret_cast<const unsigned long long*>(ws->oplog);
  static_assert(sizeof(OpRec) == 8 && offsetof(GeoSlot, oplog) % 8 == 0, "a record is one access");
  uint32_t done = kFollowEnd;
  int pos = 0, seen = 1;   // of the search of done's epoch: records applied, nodes created by them
  auto answer = [&](uint32_t word) {
    lds_store_where(1ull, lds_address(&L->heap_size), (uint32_t)rh.size);
    lds_store_where(1ull, lds_address(&L->applied), word);
    done = word;
  };
  for (;;) {
    const uint32_t word = (uint32_t)uniform_i((int)lds_word(&L->published));
    if (word == kFollowQuit) return;
    const int asked = (int)(word & 0xffffu);
    if (asked == (int)kFollowEnd) {
      if (word != done) answer(word);
      __builtin_amdgcn_s_sleep(2);
      continue;
    }
    if ((word ^ done) >> 16) {   // a search begins
      wave_sync();
      const uint2 e = L->start;
      lds_store_where(1ull, &rh.h[1], e.x, e.y);
      wave_sync();
      rh.size = 1;
      pos = 0; seen = 1;
      done = word & 0xffff0000u;
    }
    wave_sync();
    const int arrived = uniform_i((int)__hip_atomic_load(&L->arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    const int end = arrived > asked ? arrived : asked;
    // The search waits for a word that is not done: at the highest priority until the answer, and not for the passes behind it, which
    // would issue before other blocks' searches.
    if (word != done) __builtin_amdgcn_s_setprio(3);
    if (pos < end) {
      const unsigned long long r = __hip_atomic_load(log + (pos + lane < end ? pos + lane : pos), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t rk = (uint32_t)r, rw = (uint32_t)(r >> 32);
      const unsigned long long headers = lanes_where((rw & kOpHeader) != 0) & lanes_where(pos + lane < end);
      wave_sync();
      if (((uint32_t)uniform_i((int)lds_word(&L->published)) ^ word) >> 16) continue;   // there are no more searches
      int h = 0;
      while (h < 64 && (headers >> h)) h += apply_pass(rh, rk, rw, headers, h, seen);
      pos += h;
    }
    if (pos != end) continue;
    if (word != done) { answer(word); __builtin_amdgcn_s_setprio(0); }
    else __builtin_amdgcn_s_sleep(2);
  }
}
#endif

// Applies log records [st.synced, st.logEnd) to the reference's heap, pass by pass.  Records are
// fetched 64 at a time, one per lane, and again when the next pass is not among them in full (a
// pass has at most 1 + 8 * 6 records).  Between replays the slot keeps the heap; during one it lies
// over the window, which the caller has restored if it goes on with the sorted list.
BPSX_DEV void replay_log(GeoWave& g, AstarState& st) {
  const int lane = lane_here(g.lane);
  const OpRec* log = g.ws->oplog;
  uint2* kept = reinterpret_cast<uint2*>(g.ws->heap_spill);
  RefHeap<true> rh(g.L->heap(), st.replaySize, lane);
  // the pass that ended here has left its marks: the first of them, which ends the hash chains, lies
  // under the heap's unused entry 0 and has to stand while a search goes on with the heap
  g.clear_marks();
  wave_sync();
  for (int i = lane + 1; i <= rh.size; i += 64) rh.h[i] = kept[i];
  wave_sync();
  int base = st.synced;        // record held by lane 0
  int seen = st.replayNodes;   // nodes created so far
  uint32_t rk = 0, rw = 0;
  unsigned long long headers = 0;
  auto fetch = [&](int from) {
    base = from;
    const OpRec r = log[base + lane < st.logEnd ? base + lane : base];   // what lies behind the end is not looked at
    rk = r.key; rw = r.word;
    headers = lanes_where((rw & kOpHeader) != 0);
  };
  if (base < st.logEnd) fetch(base);
  for (int pos = st.synced; pos < st.logEnd;) {
    // the pass ends with the next header; a fetch is a round trip to HBM: one only when the pass at hand is
    // not all there
    if (pos >= base + 64 || !(headers >> (pos - base))) fetch(pos);
    pos += apply_pass(rh, rk, rw, headers, pos - base, seen);
  }
  st.synced = st.logEnd;
  st.replayNodes = seen;
  st.replaySize = rh.size;
  st.replayRoot = (uint32_t)uniform_i((int)rh.h[1].y);
  for (int i = lane + 1; i <= rh.size; i += 64) kept[i] = rh.h[i];
  wave_sync();
}
// The window and the marks after something else has used their LDS.
BPSX_DEV void restore_window(GeoWave& g) {
  if (kFollower) return;   // nothing else has
  const int from = g.nodeCount > kWindow ? g.nodeCount - kWindow : 0;
  for (int i = from + g.lane; i < g.nodeCount; i += 64) {
    BPSX_KEEP_APART();
    const float4 node = g.ws->nodes[i];
    BPSX_KEEP_APART();
    g.L->w_node[i & (kWindow - 1)] = node;
  }
  g.clear_marks();
  wave_sync();
}

// One node per round with the reference's heap as it is: what a search goes on with when its open
// list outgrows the sorted form or its log is full.  The nodes' bodies are read from
// the slot (the heap lies over the window).  Lds: the heap is in LDS, and the loop ends with
// kAstarGrowHeap before it outgrows it; otherwise it is in the slot, which holds any heap.
template <bool Lds>
BPSX_DEV AstarExit astar_exact(GeoWave& g, AstarState& st, const AEdge* edges, uint32_t endIp, const float* endPos, uint32_t* pops) {
  const int lane = lane_here(g.lane);
  GeoLds* L = g.L;
  const float H_SCALE = 0.999f;
  RefHeap<Lds> rh(Lds ? L->heap() : reinterpret_cast<uint2*>(g.ws->heap_spill), st.replaySize, lane);
  for (;;) {
    st.replaySize = rh.size;
    if (rh.size <= 0) return kAstarEmpty;
    if (Lds && rh.size > kHeapLds - kNvp) return kAstarGrowHeap;
    const uint32_t front = (uint32_t)uniform_i((int)rh.h[1].y);
    const int bi = (int)(front & 0x7ffu);
    const uint32_t bestIp = front >> 11;
    if (bestIp == endIp) { st.lastBest = bi; return kAstarGoal; }
    // what the expansion needs from HBM is asked for before the heap is set in order
    const AEdge edge = edges[bestIp * kEdgeStride + (uint32_t)(lane & (kRowLanes - 1))];
    const float4 b = g.node(bi);
    rh.pop();
    (*pops)++;
    const uint32_t nb = edge.nb;
    float m0 = edge.mid[0], m1 = edge.mid[1], m2 = edge.mid[2];
    const uint32_t bucket = GeoWave::hash(nb);
    uint32_t chainHead;
    const unsigned long long valid = lanes_where(nb != kNoNb) & ((1ull << kNvp) - 1ull);
    const uint32_t at = g.find<true>(valid, nb, lds_address(&L->first[bucket]), &chainHead);
    const unsigned long long known = lanes_where(at != kChainEnd);
    uint32_t ni4 = GeoWave::node4_at<true>(at);
    const float4 pc = g.node((int)(in_mask(known) ? ni4 >> 2 : 0u));   // (no pick: the mask is a comparison's)
    m0 = in_mask(known) ? pc.x : m0; m1 = in_mask(known) ? pc.y : m1; m2 = in_mask(known) ? pc.z : m2;
    const float cx = m0 - b.x, cy = m1 - b.y, cz = m2 - b.z;
    const float ex = endPos[0] - m0, ey = endPos[1] - m1, ez = endPos[2] - m2;
    float curCost, toEnd;
    sqrt_exact2(cx * cx + cy * cy + cz * cz, ex * ex + ey * ey + ez * ez, &curCost, &toEnd);
    const bool last = nb == endIp;
    const float cost = last ? b.w + curCost * 1.0f + toEnd * 1.0f : b.w + curCost * 1.0f;
    const float heuristic = last ? 0.0f : toEnd * H_SCALE;
    const float total = cost + heuristic;
    const unsigned long long update = valid & ~(known & lanes_where(total >= pc.w + heuristic));
    // new nodes take consecutive indices in edge order; those that share a bucket are chained one after the other
    const unsigned long long fresh = update & ~known;
    const int want = g.nodeCount + __popcll(fresh);
    if (want > kMaxNodes) { st.outOfNodes = true; return kAstarEmpty; }   // reported as failure whatever follows
    ni4 = OpenList::pick(fresh, 4u * ((uint32_t)g.nodeCount + __builtin_amdgcn_mbcnt_lo((uint32_t)fresh, 0u)), ni4);
    g.nodeCount = want;
    const uint32_t own = GeoWave::offset_of<true>(ni4);
    for (unsigned long long rest = fresh; rest;) {
      g.set_links<true>(rest, ni4, make_link(nb, chainHead), lds_address(&L->first[bucket]), own);
      wave_sync();
      chainHead = L->first[bucket];
      rest &= lanes_where(chainHead != own);   // another of the bucket has overwritten it at the chain's head: behind that
      wave_sync();
    }
    g.keep_node(update, ni4, make_float4(m0, m1, m2, cost), (uint32_t)bi + 1u);
    if (kAllLds) lds_store_where(update, lds_address(L->w_node) + (ni4 << 2), make_float4(m0, m1, m2, cost));
    wave_sync();
    const uint32_t packed = (ni4 >> 2) | (nb << 11);
    for (unsigned long long upd = update; upd;) {
      const int src = first_lane(upd);
      upd = without_lane(upd, src);
      rh.update(((known >> src) & 1ull) != 0, __float_as_uint(lane_f(total, src)), rlane(packed, src));
    }
  }
}

// The entries that the list keeps apart, looked through: those of nodes that have been updated since are dropped, and the
// smallest, if the list has room for them, enter it: kPull of them at most, and kPullLeast at least, if there is a bound that
// parts so few from the others.  False if the search cannot go on in this form.  (A bound is found in five or six guesses.  With
// 30 at least there was one guess less, but the entries lasted for fewer passes: 4096 agents over cluttered plans 902 and 892 us,
// 65536 over mixed scenes 2408 and 2399.  With 38 at most and 26 at least 918 and 2430.)
// Bound by two round trips to HBM, for the entries and their nodes, the search for the bound and the sort; once in ten
// to fifty passes.  (With those that enter taken one after the other, nine instructions each for some forty: steps of 510 agents
// in two groups 898 -> 881 us, of 1024 over room plans 462 -> 449, of 4096 over cluttered plans 953 -> 936, of 65536 over mixed
// scenes 2441 -> 2414, 300 queries over room plans 267 -> 265.5.)
BPSX_DEV bool refill(const GeoWave& g, OpenList& ol, uint32_t endIp, const float* endPos) {
  // 63 entries at a time: none in lane 63 (enter)
  constexpr int kAtOnce = 63, K = OpenList::kFarCap / kAtOnce, kPull = 46, kPullLeast = 42;
  static_assert(OpenList::kFarCap % kAtOnce == 0, "whole rounds");
  const int lane = lane_here(g.lane);
  uint2* apart = reinterpret_cast<uint2*>(g.far_list());
  uint32_t t[K], n[K];
  unsigned long long live[K];
  static_for<0, K>([&](auto J) BPSX_INLINE_LAMBDA {
    constexpr int k = decltype(J)::value;
    t[k] = n[k] = 0;
    if (ol.far > kAtOnce * k) {
      const uint2 v = apart[kAtOnce * k + lane < ol.far ? kAtOnce * k + lane : 0];
      t[k] = v.x; n[k] = v.y;
    }
  });
  int count = 0;
  uint32_t most = 0;
  static_for<0, K>([&](auto J) BPSX_INLINE_LAMBDA {
    constexpr int k = decltype(J)::value;
    live[k] = 0;
    if (ol.far > kAtOnce * k) {
      // an entry is its node's if its total is what the node's would be now
      const float4 p = g.node((int)(n[k] & 0x7ffu));
      const float ex = endPos[0] - p.x, ey = endPos[1] - p.y, ez = endPos[2] - p.z;
      const float ee = ex * ex + ey * ey + ez * ez;
      float toEnd, same;
      sqrt_exact2(ee, ee, &toEnd, &same);
      const float heuristic = (n[k] >> 11) == endIp ? 0.0f : toEnd * 0.999f;
      live[k] = lanes_where(__float_as_uint(p.w + heuristic) == t[k]) & lanes_where(kAtOnce * k + lane < ol.far) & ~(1ull << kAtOnce);
      count += __popcll(live[k]);
      const uint32_t mine = in_mask(live[k]) ? t[k] : 0u;
      most = mine > most ? mine : most;
    }
  });
  const auto below = [&](uint32_t bound) BPSX_INLINE_LAMBDA {
    int c = 0;
    static_for<0, K>([&](auto J) BPSX_INLINE_LAMBDA { constexpr int k = decltype(J)::value; c += __popcll(lanes_where(t[k] < bound) & live[k]); });
    return c;
  };
  uint32_t bound = ol.bound;   // below it there is none
  if (ol.size() < OpenList::kRefill) {
    bound = OpenList::kEmpty;
    if (count > kPull) {
      // the greatest of all lanes, in the last one
      most = umin_dpp<0x118, 0xf>(umin_dpp<0x114, 0xf>(umin_dpp<0x112, 0xf>(umin_dpp<0x111, 0xf>(~most))));
      most = ~umin_dpp<0x143, 0xc>(umin_dpp<0x142, 0xa>(most));
      uint32_t lo = ol.bound, hi = rlane(most, 63) + 1u;   // too few below the one, too many below the other
      int at_lo = 0, at_hi = count;
      while (hi - lo > 1u) {
        const uint32_t mid = lo + (hi - lo) / 2u;
        const int c = below(mid);
        if (c > kPull) { hi = mid; at_hi = c; }
        else { lo = mid; at_lo = c; if (c >= kPullLeast) break; }
      }
      // (entries of one total stay together)
      bound = at_lo >= kPullLeast || at_hi + ol.size() > OpenList::kSplit ? lo : hi;
    }
  }
  int kept = 0, entered = 0;
  static_for<0, K>([&](auto J) BPSX_INLINE_LAMBDA {
    constexpr int k = decltype(J)::value;
    if (live[k]) {
      const unsigned long long in = lanes_where(t[k] < bound) & live[k], out = live[k] & ~in;
      // those that enter go to the lanes from `entered` on; the others to the last one, where nobody looks
      const int c = __popcll(in);
      const uint32_t place = __builtin_amdgcn_mbcnt_hi((uint32_t)(in >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)in, (uint32_t)entered));
      const int to = (int)(in_mask(in) ? place : 63u) * 4;
      const uint32_t pt = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)t[k]), pn = (uint32_t)__builtin_amdgcn_ds_permute(to, (int)n[k]);
      ol.e = in_mask(lane_range(c, entered)) ? OpenList::entry(pt, pn) : ol.e;
      entered += c;
      store_where(out, apart, 8u * (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(out >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)out, (uint32_t)kept)), t[k], n[k]);
      kept += __popcll(out);
    }
  });
  ol.base -= entered;
  if (entered) ol.sort(lane);
  ol.far = kept;
  ol.bound = kept ? bound : OpenList::kEmpty;
  return kept <= OpenList::kFarKeep && (!kept || ol.size() >= OpenList::kRefill);
}
// The list put in order between two passes, as its limits ask for; full: the next pass has no room for what it adds.
// (Equal totals that a replay has put in another order leave the list before anything enters it: one that is full is
// only split.)
BPSX_DEV bool care_for_list(const GeoWave& g, OpenList& ol, uint32_t endIp, const float* endPos, bool full) {
  const int lane = lane_here(g.lane);
  if (!full && (ol.far > OpenList::kFarMost || ol.size() < OpenList::kRefill) && !refill(g, ol, endIp, endPos)) return false;
  if (full || ol.size() > OpenList::kSplit) {
    // the greater ones, from the first of their total on
    const int keep = ol.size() > OpenList::kSplit ? 42 : ol.size() >> 1;
    const uint32_t bound = rlane(ol.total(), ol.base + keep);
    if (bound == rlane(ol.total(), ol.base)) return false;
    const unsigned long long away = lanes_where(ol.total() >= bound) & ~(1ull << OpenList::kEnd);
    const int n = __popcll(away);
    store_where(away, g.far_list(), 8u * (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(away >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)away, (uint32_t)ol.far)), ol.total(), ol.node());
    const int from = (lane - n) * 4;   // of the lanes from n on; zeros come before
    const uint32_t t = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)ol.total()), nd = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)ol.node());
    ol.e = lane == OpenList::kEnd ? ol.e : lane < n ? 0ull : OpenList::entry(t, nd);
    ol.far += n;
    ol.base += n;
    ol.bound = bound;
  }
  ol.set_limits();
  return true;
}

// The expansion loop with the open list as a sorted array (OpenList), up to kRows nodes per
// pass.  Row r of kRowLanes lanes works on entry r of the list (lane kRowLanes r + j on edge j
// of its polygon, the lane after the last edge on the node itself): the edge records of all of them arrive in one load, and node lookup, costs, node
// creation and stores are done by the same instructions for all rows.  Every row computes
// from the state before the pass.  Rows 0 .. c-1 are what the reference does next, in that
// order, when for every row j below c
//   - entry j's total is below entry j + 1's, and every total that an earlier row puts on the
//     open list is above it: entry j is then the only entry with the smallest total when its
//     turn comes, whatever the arrangement of the reference's heap,
//   - no earlier row creates or updates row j's own node or a node that row j updates too (a
//     neighbour of both).  A neighbour that row j reads and leaves alone, because the way
//     through row j is no better than the node's total, may be updated by an earlier row: its
//     total only gets lower.  This is found with one LDS word per polygon hash: every lane that
//     updates notes itself there (the first lane wins, one of the earliest row), then these lanes and
//     the rows' own lanes look for a note of an earlier row.  Two polygons with the same hash
//     only make c smaller.  A row's update falls away, and the row stands, where its way to the
//     place that the earlier row gives the node is no better than the earlier row's.
//   - entry j is not the goal (the goal ends the search when it is first in line).
// The pass commits c >= 1 rows: their new nodes take consecutive indices in row and edge
// order, their entries leave the list, their updates enter it.  A later row may improve the
// node of an earlier one (it sees it as open, the reference as closed): both views lead to
// the same node state and the same list, because a modify that finds no entry is a push.
// Returns kAstarTie when the first two entries share the smallest total.
template <bool S>
BPSX_DEV AstarExit astar_fast(GeoWave& g, AstarState& st, const AEdge* edges, uint32_t endIp, const float* endPos, uint32_t* pops,
                             int frontResolved) {
  const int lane = lane_here(g.lane);
  GeoLds* L = g.L;
  const float H_SCALE = 0.999f;
  const float e0 = endPos[0], e1 = endPos[1], e2 = endPos[2];
  endIp = (uint32_t)uniform_i((int)endIp);
  OpenList& ol = st.ol;
  const int row = lane >> kRowShift, el = lane & (kRowLanes - 1);
  // the lanes of every row that look after the row's own node in the conflict test
  constexpr unsigned long long kOwnLanes = 0x4040404040404040ull;
  static_assert(kNvp == 6 && kRowLanes == 8, "the lane masks of a row");
  constexpr unsigned long long kRows1 = rows_below(1), kRows2 = rows_below(2);   // lanes of the first rows
  constexpr int kHeaderLane = 62;   // no edge's lane, and all that a pass updates lies before it
  const char* edges_of = reinterpret_cast<const char*>(edges);
  int resolved = uniform_i(frontResolved);   // (a truth value would be a mask of lanes, and the branches around it the lanes' own)
  // of every row: its entry of the list, and the total of the entry behind that
  const uint2 first = ol.front(row);
  uint32_t cand = first.x, nextTotal = first.y;
  // Written for few instructions and few waits on the common path: what is rare sits behind one branch
  // each; conditions are lane masks on the scalar unit; LDS reads whose results are needed later go out
  // early (the marks' before the scan over the rows, the chain heads' before the stores); the next
  // pass's nodes and totals come back with the merged list instead of through lane permutes; stores take
  // 32-bit offsets from uniform bases.  No branch depends on the lanes: loads of lanes that have nothing
  // to load go to an address that exists, stores go out under a mask.  A wavefront issues an
  // instruction of any kind every five cycles at best, a branch costs it fifteen and a result that goes
  // from the vector to the scalar unit and back twenty, so a search alone on a SIMD lasts as long as its
  // instructions, and many of them are bound by the units' issue.  (With branches around loads and
  // stores, and the loop rebuilt around them with some sixty instructions more per pass: steps of 64
  // agents 216 us, now 184, of 1024 over room plans 836 and 697, of 16384 over mazes 1026 and 902, of
  // 65536 over mixed scenes 3740 and 3233; a reset of 2048 over mazes 655 and 525.)
  // The next pass's edge records are asked for as soon as its nodes are known, before it is known how many of them
  // can be taken.  What a pass stores in HBM goes out while the list's entries come back from LDS: the wait
  // for the records is one for all that was asked for before.  What a pass stores in LDS goes out behind that
  // request, for whose time a lone search has it for nothing.  (Steps of 1024 agents over room plans 693 -> 656 us,
  // of 510 in two groups 1327 -> 1230, of 16384 over mazes 902 -> 883 and, with the stores in LDS so late, 845 -> 829,
  // of 65536 over mixed scenes 3222 -> 3150 and 2992 -> 2913, a reset of 2048 over mazes 525 -> 495.)
  struct {
    unsigned long long updated, fresh;   // lanes of updated nodes, of new ones among them
    uint32_t node4, link;                // the node, its link
    uint32_t chain;                      // address of its chain's first among L->first
    float4 node;
  } late;
  late.updated = late.fresh = 0;
  late.node4 = late.link = 0;
  late.chain = lds_address(L->first);
  late.node = make_float4(0, 0, 0, 0);
  const auto insert = [&]() BPSX_INLINE_LAMBDA {
    // The new nodes insert all at once in front of the chain head their lookup saw.  Of several
    // that share a bucket one store wins; the others see that when the head that is read back has come
    // (looked at below, after the stores that need not wait for it).
    g.clear_marks();
    const uint32_t own = GeoWave::offset_of<S>(late.node4);
    g.set_links<S>(late.fresh, late.node4, late.link, late.chain, own);
    wave_sync();
    uint32_t head = lds_half(late.chain);
    if (kAllLds) lds_store_where(late.updated, lds_address(L->w_node) + (late.node4 << 2), late.node);
    else lds_store_where(late.updated & lanes_where((int)late.node4 >= 4 * (g.nodeCount - kWindow)),
                         lds_address(L->w_node) + 16u * GeoWave::window_slot(late.node4), late.node);
    // new nodes that another of their bucket has overwritten at the chain's head go in behind it
    for (unsigned long long lost = late.fresh & lanes_where(head != own); __builtin_expect(lost != 0, 0);) {
      g.set_links<S>(lost, late.node4, make_link(link_id(late.link), head), late.chain, own);
      wave_sync();
      head = lds_half(late.chain);
      lost &= lanes_where(head != own);
      wave_sync();
    }
  };
  // What is late on a way out of the loop is no more than a name: else the compiler keeps it for that way, and copies it at every
  // pass's end.  (Not where links may spill, whose two instantiations it then gives loops of several ends: 65536 agents over
  // mixed scenes 2465 -> 2604 us.)  With it, the branch of the roots behind them, and the stores that share a mask in one
  // statement, a pass is 332 -> 322 instructions in k_geodesic_few: steps of 64 agents 124.7 -> 122.6 us, of 1024 over room plans
  // 478 -> 468, 3007 fleeing ones 487 -> 463, of 65536 over mixed scenes 2469 -> 2430, of 16384 over mazes 722 -> 710, 300 queries
  // over room plans 246 -> 240.
  const auto leave = [&](AstarExit way) BPSX_INLINE_LAMBDA -> AstarExit {
    if constexpr (kLinksLds >= kMaxNodes) {
      asm("" : "=s"(late.updated), "=s"(late.fresh), "=v"(late.node4), "=v"(late.link), "=v"(late.chain));
      asm("" : "=v"(late.node.x), "=v"(late.node.y), "=v"(late.node.z), "=v"(late.node.w));
    }
    return way;
  };
  const auto pass = [&]() BPSX_INLINE_LAMBDA -> AstarExit {
    FM(0);
    // ---- the edge records of the first entries' polygons (of polygon 0 where there is no entry)
    const uint32_t ip = cand >> 11;
    static_assert(kEdgeStride * sizeof(AEdge) == 128, "a polygon's records");
    const AEdge edge = *reinterpret_cast<const AEdge*>(edges_of + ((ip << 7) | (uint32_t)(el << 4)));
    insert();
    FM(1);
    if (st.logEnd > kOpLogCap - (1 + kRows * kNvp)) return leave(kAstarLogFull);
    if (ol.needs_care()) return leave(kAstarCare);
    // ---- how many entries at the front are each the only one with their total, and not the goal
    const unsigned long long uniq = lanes_where(ol.total() < OpenList::down1(ol.total())) >> ol.base;
    const unsigned long long goal = lanes_where((ol.node() >> 11) == endIp) >> ol.base;
    uint32_t lim = (uint32_t)first_other_lane(uniq & ~goal);
    lim = lim < (uint32_t)kRows ? lim : (uint32_t)kRows;
    const int bi = (int)(cand & 0x7ffu);
    int pairTie = 0;   // 2: with the goal as one of the two
    uint32_t headerWord = kOpHeader;
    if (__builtin_expect(lim == 0, 0)) {
      if (ol.base >= OpenList::kEnd) return leave(kAstarEmpty);
      if (uniq & 1ull) lim = (uint32_t)kRows;   // the goal
      else if (resolved) { lim = 1; resolved = 0; }   // the caller has put the reference's next node first
      else {
        // The first two entries share the smallest total.  When they are alone in that and their
        // expansions are independent of each other (neither updates what the other reads, and
        // whatever they put on the list lies above their total), the reference expands them one
        // after the other, in the order its heap has them in, and ends in the same state either
        // way: the pass takes both and notes in the log that their order is open.
        if (!(uniq & 2ull)) return leave(kAstarTie);
        pairTie = 1;
        g.pairTies++;   // counts the attempts: one that fails comes back through the log
        lim = (uint32_t)__builtin_ctzll(~(uniq | 3ull) | (1ull << kRows));
      }
      if ((goal & 1ull) && !pairTie) {
        st.lastBest = uniform_i(bi);
        return leave(kAstarGoal);
      }
      // the goal as one of a tied pair: both rows are looked at
      if (pairTie && (goal & 3ull)) { pairTie = 2; lim = 2; }
      else if (pairTie && goal) { const uint32_t jg = (uint32_t)__builtin_ctzll(goal); lim = jg < lim ? jg : lim; }
    }
    const unsigned long long rowOn = lanes_where(row < (int)lim);
    float4 b = L->w_node[bi & (kWindow - 1)];
    if (!kAllLds) {
      const unsigned long long left = lanes_where(bi < g.nodeCount - kWindow) & rowOn;
      if (__builtin_expect(left != 0, 0)) {   // a node has left the window: rare
        BPSX_KEEP_APART();
        const float4 kept = g.ws->nodes[bi];
        BPSX_KEEP_APART();
        b.x = in_mask(left) ? kept.x : b.x; b.y = in_mask(left) ? kept.y : b.y; b.z = in_mask(left) ? kept.z : b.z; b.w = in_mask(left) ? kept.w : b.w;
      }
    }
    FM(2);
    // ---- node lookup; the row's own lane hashes its own polygon for the conflict test
    const uint32_t nb = edge.nb;
    const unsigned long long valid = lanes_where(nb != kNoNb) & rowOn;
    const uint32_t hashed = GeoWave::hash_product(in_mask(kOwnLanes) ? ip : nb), bucket = GeoWave::bucket_of<kHashSize>(hashed);
    const uint32_t chain = lds_address(&L->first[bucket]);
    uint32_t chainHead;
    const uint32_t at = g.find<S>(valid, nb, chain, &chainHead);
    FM(3);
    // ---- costs.  A lane without a node to read (idle, or its node is new) reads one of the window's slots.
    const unsigned long long known = lanes_where(at != kChainEnd);
    uint32_t ni4 = GeoWave::node4_at<S>(at);
    float4 p = L->w_node[GeoWave::window_slot(ni4)];
    if (!kAllLds) {
      const unsigned long long left = lanes_where((int)ni4 < 4 * (g.nodeCount - kWindow)) & known;
      if (__builtin_expect(left != 0, 0)) {   // a node has left the window: rare
        BPSX_KEEP_APART();
        const float4 kept = g.ws->nodes[OpenList::pick(left, ni4 >> 2, 0u)];
        BPSX_KEEP_APART();
        p.x = in_mask(left) ? kept.x : p.x; p.y = in_mask(left) ? kept.y : p.y; p.z = in_mask(left) ? kept.z : p.z; p.w = in_mask(left) ? kept.w : p.w;
      }
    }
    const float p0 = in_mask(known) ? p.x : edge.mid[0], p1 = in_mask(known) ? p.y : edge.mid[1], p2 = in_mask(known) ? p.z : edge.mid[2];   // a new node lies on the portal's midpoint
    const float cx = p0 - b.x, cy = p1 - b.y, cz = p2 - b.z;
    const float ex = e0 - p0, ey = e1 - p1, ez = e2 - p2;
    const float cc = cx * cx + cy * cy + cz * cz, ee = ex * ex + ey * ey + ez * ez;
    float curCost, toEnd;
    sqrt_exact2(cc, ee, &curCost, &toEnd);
    curCost = curCost * 1.0f;
    const bool last = nb == endIp;
    const float cost = last ? b.w + curCost + toEnd * 1.0f : b.w + curCost;
    const float heuristic = last ? 0.0f : toEnd * H_SCALE;
    const float total = cost + heuristic;
    // the lanes that update their node, and the total as bits there, all ones elsewhere.  (A node's
    // total so far is the sum it was computed as, of its cost and the same heuristic.)
    unsigned long long upd = valid & ~(known & lanes_where(total >= p.w + heuristic));
    uint32_t tb = in_mask(upd) ? __float_as_uint(total) : 0xffffffffu;
    FM(4);
    // ---- how many rows stand
    // conflicts: the first lane that updates a polygon leaves its mark at the polygon's hash, lanes of later rows
    // look for it (no marks stand when a pass begins)
    const uint32_t* mark = reinterpret_cast<const uint32_t*>(L) + GeoWave::bucket_of<kTagSlots>(hashed);
    constexpr int marksAt = (int)offsetof(GeoLds, n_link) + 4 * kLinksLds;
    lds_min_where<marksAt>(upd, mark, (uint32_t)lane);
    wave_sync();
    const uint32_t seen = mark[marksAt / 4];   // the marking lane, or above all lanes
    // the first entry that an update of a row before it reaches or undercuts: the smallest updated total of
    // every row, then of all rows up to it (a scan over the rows), and each row compares that with the
    // total of the entry behind its own
    uint32_t low = tb;   // all ones where the lane updates nothing
    low = umin_dpp<0xb1, 0xf>(low);    // quad_perm [1,0,3,2]
    low = umin_dpp<0x4e, 0xf>(low);    // quad_perm [2,3,0,1]
    low = umin_dpp<0x141, 0xf>(low);   // row_half_mirror: every lane has its row's smallest
    low = umin_dpp<0x118, 0xf>(low);   // row_shr:8: odd rows, with the row before
    low = umin_dpp<0x142, 0xa>(low);   // row_bcast:15 into the second and fourth 16 lanes
    low = umin_dpp<0x143, 0xc>(low);   // row_bcast:31 into the upper 32 lanes
    const unsigned long long reached = lanes_where(low <= nextTotal) << kRowLanes;   // in the lanes of the row behind
    // an earlier row's update matters to a row only at its own node and at the polygons it
    // updates itself: where it reads and leaves alone (a total no better than the node's), a
    // total lowered further changes nothing
    const unsigned long long cares = upd | (rowOn & kOwnLanes);
    unsigned long long clash = lanes_where(seen < (uint32_t)(lane - el)) & cares;
    uint32_t c = (uint32_t)first_lane(reached | ~rowOn), clashAt = (uint32_t)first_lane(clash);   // in the first row that does not stand
    c = c < 64u ? c : 64u;
    if (clashAt < (c & ~(uint32_t)(kRowLanes - 1))) {
      // A later row that updates what an earlier one does stands all the same when its update falls away: behind the
      // earlier one the node lies where that one has put it, and the way through the later row costs no less.
      // (The heuristic of both is the node's, so the totals are in the costs' order.)  A third of the passes ended at such
      // a pair of rows, nine in ten of them at one of this kind: 10 to 14 % fewer passes, for some thirty
      // instructions and a round of lane permutes in a third of them.  (Steps of 64 agents 155 -> 148 us, of 1024 over
      // room plans 619 -> 589, of 65536 over mixed scenes 2919 -> 2810, of 16384 over mazes 820 -> 805, a reset of 2048 over
      // mazes 482 -> 476.  With the later cost itself, its root included, 150, 601, 2820, 801 and 475.)
      const int from = (int)(seen * 4u);
      const uint32_t theirs = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)nb);
      const float q0 = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(p0)));
      const float q1 = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(p1)));
      const float q2 = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(p2)));
      const float theirCost = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(cost)));
      // its way costs no less if its step is as long as the costs' difference, with room for the rounding of both
      // (cost = b.w + the step's length never falls when the length grows).  The square of a difference below 2^-63 has fewer
      // bits than that room needs, or none, and where there is no difference any step is long enough: there one of 2^-63 has to be.
      const float mx = q0 - b.x, my = q1 - b.y, mz = q2 - b.z, less = fmaxf(theirCost - b.w, 0x1p-63f);
      const unsigned long long far = lanes_where(mx * mx + my * my + mz * mz >= less * less * 1.00001f);
      const unsigned long long falls = pairTie ? 0ull : far & lanes_where(theirs == nb) & clash & upd;
      upd &= ~falls;
      clash &= ~falls;
      clashAt = (uint32_t)first_lane(clash);
      c = clashAt < c ? clashAt : c;
    }
    c >>= kRowShift;
    if (__builtin_expect(pairTie != 0, 0)) {
      asm("" : "+s"(pairTie));   // (or both tests of it come first)
      if (pairTie == 2) {
        // The goal shares the smallest total with one other node.  If the reference takes the goal
        // first the search ends here; if it takes the other node first, it expands it and ends
        // then.  The path is the goal's node and its ancestors: it is the same both ways when
        // that expansion only creates nodes (none of them can be on the path) and the node pool
        // holds them (an exhausted pool is reported as failure).  Otherwise the heap must say.
        const unsigned long long other = upd & ~lanes_where(ip == endIp);
        if ((other & known) || g.nodeCount + __popcll(other) > kMaxNodes) return leave(kAstarTie);
        st.lastBest = (int)rlane((uint32_t)bi, first_lane(goal & 3ull) << kRowShift);
        return leave(kAstarGoal);
      }
      // a tied pair: both its rows must lie above entry 1's total, ...
      const bool above = rlane(low, kRowLanes) > rlane(nextTotal, 0);
      if (!above) c = 1;
      // ... and in either order: row 0 must not read what row 1 updates either
      bool fails = c < 2 || (lanes_where((seen >> kRowShift) == 1u) & cares & kRows1) != 0;
      if (fails && above && !(reached & kRows2)) {
        // The marks are kept per polygon hash, and a pair that fails costs a replay of the log:
        // the polygons that either row updates are compared with those the other row reads,
        // and a clash that was two polygons with one hash lets the pair (and only it) stand.
        const uint32_t readPoly = OpenList::pick(cares & kOwnLanes, ip, OpenList::pick(upd, nb, 0xffffffffu));
        unsigned long long w = upd & kRows2;
        bool real = false;
        while (w) {
          const int src = first_lane(w);
          w = without_lane(w, src);
          const unsigned long long others = src < kRowLanes ? (kRows2 & ~kRows1) : kRows1;
          if (lanes_where(readPoly == rlane(nb, src)) & others) real = true;
        }
        if (!real) { fails = false; c = 2; }
      }
      if (fails) return leave(kAstarTie);
      headerWord = kOpHeader | kOpUnordered | rlane(cand, 0);
    }
    FM(5);
    upd &= lanes_where(row < (int)c);
    const int nrec = __popcll(upd);
    const unsigned long long fresh = upd & ~known;
    const int want = g.nodeCount + __popcll(fresh);
    const unsigned long long nearby = upd & lanes_where(tb < ol.bound);
    // Nothing has changed yet: a list that would outgrow its registers is split first,
    // links that would outgrow LDS go on in the instantiation that spills.
    if (__builtin_expect(ol.base + (int)c - __popcll(nearby) < OpenList::kEnd - OpenList::kMost, 0)) return leave(kAstarGrowHeap);
    if (!S && __builtin_expect(want > kLinksLds, 0)) return leave(kAstarGrowLinks);
    (*pops) += c;
    // the reference carries on without the nodes that do not fit, but reports anything found
    // after that as failure (only plain DT_SUCCESS counts, PathFinder.cpp:506): stop
    if (S && __builtin_expect(want > kMaxNodes, 0)) {
      st.outOfNodes = true;
      return leave(kAstarEmpty);
    }
    FM(6);
    // ---- new nodes (always taken) get consecutive indices in row and edge order
    const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(fresh >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)fresh, 0u));
    ni4 = OpenList::pick(fresh, 4u * (uint32_t)(g.nodeCount + rank), ni4);   // (opaque, as keep_node wants it)
    late.fresh = fresh;
    late.updated = upd;
    late.node4 = ni4;
    late.link = make_link(nb, chainHead);
    late.chain = chain;
    late.node = make_float4(p0, p1, p2, cost);
    g.nodeCount = want;
    FM(7);
    // the pass in the operation log: the updates in lane order, then the header
    const uint32_t packed = (ni4 >> 2) | (nb << 11);
    tb = wlane_at<kHeaderLane>(tb, c | ((uint32_t)nrec << 8));
    const uint32_t word = wlane_at<kHeaderLane>(packed | ((uint32_t)row << 26), headerWord);
    const auto store = [&]() BPSX_INLINE_LAMBDA {
      const uint32_t rec = __builtin_amdgcn_mbcnt_hi((uint32_t)(upd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)upd, (uint32_t)st.logEnd));
#if BPSX_FOLLOWER
      static_assert(kHeaderLane == 62);
      g.keep_pass(upd, 1ull << kHeaderLane, ni4, late.node, (uint32_t)bi + 1u, (uint32_t)st.logEnd, rec * (uint32_t)sizeof(OpRec), tb, word);
#else
      store_where(upd | (1ull << kHeaderLane), g.ws->oplog, rec * (uint32_t)sizeof(OpRec), tb, word);
      g.keep_node(upd, ni4, late.node, (uint32_t)bi + 1u);
#endif
      st.logEnd += 1 + nrec;
    };
    FM(8);
    store();
    if (upd & ~nearby) {
      const unsigned long long away = upd & ~nearby;
      store_where(away, g.far_list(), 8u * (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(away >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)away, (uint32_t)ol.far)), tb, packed);
      ol.far += __popcll(away);
      ol.set_limits();
    }
    FM(9);
    // ---- the open list: the committed entries leave, the updates enter
    const uint2 front = ol.merge((int)c, nearby, nearby & known, tb, packed, row);
    cand = front.x;
    nextTotal = front.y;
    FM(10);
    return kAstarOn;
  };
  // All ways out of a pass meet here, and the loop has one end: with several the compiler keeps a flag for each,
  // and copies of the loop's state.  (The empty statement keeps it from joining a way out to what follows it.)
  int way;
  // Else the compiler has every pass wait for loads that came before the loop.  (Not where a search has a SIMD nearly to itself, where
  // the wait is none and the other order of instructions costs 0.7 %.)
  if constexpr (!kFollower) __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
  do {
    way = (int)pass();
    asm volatile("" : "+s"(way));
  } while (way == (int)kAstarOn);
  asm volatile("" : "+s"(way));   // (what is asked about it behind the loop is not joined to what the loop asks)
  return (AstarExit)way;
}

// Runs A* for one query. Returns the corridor length (corridor written to F->corridor), or 0
// when the reference would report anything but plain DT_SUCCESS.
BPSX_DEV int astar(GeoWave& g, FunnelLds* F, const NavData& nav, const SceneDev& s, uint32_t startIp, uint32_t endIp,
                   const float* startPos, const float* endPos, uint32_t* pops) {
  const int lane = lane_here(g.lane);
  if (startIp == endIp) {
    if (lane == 0) F->corridor[0] = (uint16_t)startIp;
    wave_sync();
    return 1;
  }
  AstarState st;
  const AEdge* edges = nav.aedges + (size_t)(uint32_t)uniform_i((int)s.poly_base) * kEdgeStride;
  g.clear();
  const float dx = endPos[0] - startPos[0], dy = endPos[1] - startPos[1], dz = endPos[2] - startPos[2];
  const float total = sqrtf(dx * dx + dy * dy + dz * dz) * 0.999f;
  g.nodeCount = 1;
  if (lane == 0) {
    GeoLds* L = g.L;
    L->w_node[0] = make_float4(startPos[0], startPos[1], startPos[2], 0.0f);
    L->n_link[0] = make_link(startIp, kChainEnd);
    L->first[GeoWave::hash(startIp)] = 0;
    reinterpret_cast<uint2*>(g.ws->heap_spill)[1] = make_uint2(__float_as_uint(total), startIp << 11);
  }
  g.keep_node(1ull, 0, make_float4(startPos[0], startPos[1], startPos[2], 0.0f), 0u);
  wave_sync();
#if BPSX_FOLLOWER
  g.settle(g.epoch | kFollowEnd);   // the search before is over for the follower too
  g.epoch = (g.epoch + 0x10000u) & 0x7fff0000u;
  if (lane == 0) { g.L->start = make_uint2(__float_as_uint(total), startIp << 11); g.L->arrived = 0; }
  wave_sync();
  g.publish(g.epoch);
#endif
  st.lastBest = 0;
  st.outOfNodes = false;
  st.logEnd = st.synced = 0;
  st.replaySize = st.replayNodes = 1;
#ifdef BPSX_PHASE_TIMING
  g.phase_t0 = __builtin_readcyclecounter();
#endif
  st.ol.init(lane, __float_as_uint(total), startIp << 11);
  // the loop is instantiated for links in LDS only or spilling (one instantiation where the LDS
  // holds all links); a search moves on when one more pass could outgrow what it runs in
  AstarExit ex;
  int resolved = 0;
  int spill = kLinksLds >= kMaxNodes;
  int cared = -1, times = 0;   // where the log was when the list was last put in order, and how often it was there
  for (;;) {
    if constexpr (kLinksLds >= kMaxNodes) ex = astar_fast<true>(g, st, edges, endIp, endPos, pops, resolved);
    else ex = uniform_i(spill) ? astar_fast<true>(g, st, edges, endIp, endPos, pops, resolved) : astar_fast<false>(g, st, edges, endIp, endPos, pops, resolved);
    resolved = 0;
    if (ex == kAstarGrowLinks) { g.clear_marks(); g.linkSpills++; spill = 1; continue; }   // the pass that did not fit has left its marks
    if (ex == kAstarCare || ex == kAstarGrowHeap) {
      g.clear_marks();
      // (a list that is not in order after a few rounds, of equal totals, does not come to be)
      times = cared == st.logEnd ? times + 1 : 0;
      cared = st.logEnd;
      if (times < 4 && care_for_list(g, st.ol, endIp, endPos, ex == kAstarGrowHeap)) continue;
    }
    if (ex == kAstarEmpty || ex == kAstarGoal) break;
    __builtin_amdgcn_s_setprio(3);   // a search that pays for a replay is late from here on
#if BPSX_FOLLOWER
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    g.publish(g.epoch | (uint32_t)st.logEnd);
    g.clear_marks();   // the pass that ended here has left its own
    g.settle(g.epoch | (uint32_t)st.logEnd);
    st.replaySize = uniform_i((int)g.L->heap_size);
    st.replayRoot = (uint32_t)uniform_i((int)g.L->heap()[1].y);
#else
    replay_log(g, st);
#endif
    // The reference pops what its heap has at the root: that entry goes first, and what was before it moves up a lane,
    // in the order that it has.
    const unsigned long long root = lanes_where(st.ol.node() == st.replayRoot && st.ol.total() == rlane(st.ol.total(), st.ol.base));
    if (ex == kAstarTie && root) {
      restore_window(g);
      g.tieReplays++;
      const uint32_t before = OpenList::up1(st.ol.node());
      const uint32_t node = in_mask(root | (root - 1ull)) ? (lane == st.ol.base ? st.replayRoot : before) : st.ol.node();
      st.ol.e = lane < st.ol.base ? 0ull : OpenList::entry(st.ol.total(), node);
      resolved = 1;
      continue;
    }
    // such a tie, a list beyond the registers or a full log: on with the reference's heap
    g.exactRuns++;
    ex = astar_exact<true>(g, st, edges, endIp, endPos, pops);
    if (ex == kAstarGrowHeap) {
      g.heapSpills++;
      uint2* kept = reinterpret_cast<uint2*>(g.ws->heap_spill);
      const uint2* h = g.L->heap();
      for (int i = lane + 1; i <= st.replaySize; i += 64) kept[i] = h[i];
      wave_sync();
      ex = astar_exact<false>(g, st, edges, endIp, endPos, pops);
    }
    break;
  }
#if BPSX_FOLLOWER
  g.publish(g.epoch | kFollowEnd);
#endif
  // an open list that ran empty, or a pool that ran out, is DT_PARTIAL_RESULT or
  // DT_OUT_OF_NODES in the reference: no path to build, the result is a failure
  if (ex != kAstarGoal || st.outOfNodes) return 0;
  const int lastBest = st.lastBest;
  // getPathToNode: a walk up the parents notes the node indices, then all lanes fill the corridor,
  // which overlays the hash heads; the links stay readable while it is written.  The walk is a
  // chain of dependent reads, 70 of them on average: the parent indices, which HBM also holds
  // side by side, are first copied into the window's arrays (no longer needed), so that the
  // chain runs in LDS; a node beyond what fits there is read from HBM.  The i-th node is noted in lane i mod 64 of a
  // register: a step is the read and six instructions.  (Through a scalar
  // register, with the nodes noted in LDS and copies of two parents a lane: steps of 64 agents 134 us, now 130, of 1024 over room
  // plans 483 and 473, of 16384 over mazes 757 and 750, a reset of 2048 over mazes 417 and 407.)
  wave_sync();
#if BPSX_WINDOW >= 2048
  const uint16_t* lparent = g.L->parents;
  constexpr int inLds = kMaxNodes;
#else
  // (of 256 nodes it holds them all.  The follower may still be at work on its heap: waiting for it cost a search 8 us)
  constexpr int kParentsLds = (int)(kWindow * sizeof(float4) / sizeof(uint16_t));
  uint16_t* lparent = reinterpret_cast<uint16_t*>(g.L->w_node);
  const int inLds = kParentsLds >= kMaxNodes ? kMaxNodes : kParentsLds;
  {
    static_assert(offsetof(GeoSlot, parents) % 16 == 0 && kParentsLds % 512 == 0, "eight parents a lane");
    const uint4* src = reinterpret_cast<const uint4*>(g.ws->parents);
    uint4* dst = reinterpret_cast<uint4*>(lparent);
    static_for<0, kParentsLds / 512>([&](auto K) BPSX_INLINE_LAMBDA {
      constexpr int k = decltype(K)::value;
      if (g.nodeCount > 512 * k) dst[64 * k + lane] = src[64 * k + lane];
    });
  }
  wave_sync();
#endif
  constexpr int kWalk = kMaxPath / 64;
  static_assert(kMaxPath % 64 == 0);
  uint32_t walk[kWalk];
  int length = 0;
  uint32_t up = (uint32_t)lastBest + 1u;   // the same in all lanes
  static_for<0, kWalk>([&](auto K) BPSX_INLINE_LAMBDA {
    constexpr int k = decltype(K)::value;
    walk[k] = 1u;
    for (int m = 0; m < 64 && lanes_where(up != 0); ++m) {
      walk[k] = lane == m ? up : walk[k];
      length++;
      if (inLds == kMaxNodes || !lanes_where(up > (uint32_t)inLds)) {
        up = lparent[up - 1u];
      } else {
        BPSX_KEEP_APART();
        up = g.ws->parents[up - 1u];
        BPSX_KEEP_APART();
      }
    }
  });
  wave_sync();
  const bool ok = !lanes_where(up != 0) && link_id(g.link<true>(lastBest)) == endIp && !st.outOfNodes;
  if (!ok) return 0;
  static_for<0, kWalk>([&](auto K) BPSX_INLINE_LAMBDA {
    constexpr int k = decltype(K)::value;
    const int i = 64 * k + lane;
    if (i < length) F->corridor[length - 1 - i] = (uint16_t)link_id(g.link<true>((int)walk[k] - 1));
  });
  wave_sync();
  return length;
}

// String pulling over F->corridor[0..n) and the summed length; +inf for every outcome the
// reference maps to "no path" (straight path of 256 points or more, missing portal).
// Bound by its instructions: a round of sixteen portals is some 130 of them and ends with a move of the apex as a rule, after
// five or six portals on average.  The corridor's edges are compared in registers, and its two end points projected next to each
// other, a lane per edge.  (One portal after the other, its five areas a lane each, took 600 to 750 cycles a portal: 23 us of
// the 176 of a search over mazes when each has a wavefront to itself, 29 of 241 among 20 wavefronts per CU.  Steps of 64
// agents 141 -> 135 us, of 1024 over room plans 492 -> 484, of 16384 over mazes 779 -> 757, of 65536 over mixed scenes 2655 ->
// 2541, a reset of 2048 over mazes 433 -> 421, 300 queries over room plans 264 -> 254.)
BPSX_DEV float funnel_length(int lane, FunnelLds* F, const NavData& nav, const SceneDev& s, int n, const float* startPos,
                             const float* endPos) {
  const float INF = __int_as_float(0x7f800000);
  lane = lane_here(lane);
  // gather the portals of the corridor, 64 at a time
  bool missing = false;
  for (int i = lane; i + 1 < n; i += 64) {
    const PolyRec& r = nav.polys[s.poly_base + F->corridor[i]];
    const uint32_t* w = reinterpret_cast<const uint32_t*>(&r);
    static_assert(offsetof(PolyRec, nei) == 72 && offsetof(PolyRec, nv) == 98, "words of a record");
    const uint32_t codes[3] = {w[18], w[19], w[20]};
    const int nv = (int)((w[24] >> 16) & 0xffu);
    const uint32_t want = (uint32_t)F->corridor[i + 1] + 1u;   // below 0x8000: neither a wall nor a tile border
    int e = -1;
    static_for<0, kNvp>([&](auto K) BPSX_INLINE_LAMBDA {
      constexpr int k = kNvp - 1 - decltype(K)::value;   // the first that fits
      e = k < nv && ((codes[k >> 1] >> (16 * (k & 1))) & 0xffffu) == want ? k : e;
    });
    missing |= e < 0;
    const float* l = r.v[e < 0 ? 0 : e];
    const float* rr = r.v[e + 1 < nv ? e + 1 : 0];
    float* p = F->portals[i];
    p[0] = l[0]; p[1] = l[1]; p[2] = l[2]; p[3] = rr[0]; p[4] = rr[1]; p[5] = rr[2];
  }
  // closestPointOnPolyBoundary of the start point in the first polygon (lanes 0 to 7 of sixteen) and of the end point
  // in the last one (lanes 8 to 15): the point itself when inside (xz), else its projection onto the first of
  // the nearest edges; lane j has the edge from vertex j.
  float cs[3], ce[3];
  {
    const bool atEnd = (lane & 8) != 0;
    const int j = lane & 7;
    const float pos[3] = {atEnd ? endPos[0] : startPos[0], atEnd ? endPos[1] : startPos[1], atEnd ? endPos[2] : startPos[2]};
    const PolyRec& r = nav.polys[s.poly_base + F->corridor[atEnd ? n - 1 : 0]];
    const int nv = r.nv;
    const float* va = r.v[j < nv ? j : 0];
    const float* vb = r.v[j + 1 < nv ? j + 1 : 0];
    const float a[3] = {va[0], va[1], va[2]}, b[3] = {vb[0], vb[1], vb[2]};
    const bool crosses = j < nv && ((b[2] > pos[2]) != (a[2] > pos[2])) && (pos[0] < (a[0] - b[0]) * (pos[2] - b[2]) / (a[2] - b[2]) + b[0]);
    float t;
    const float d = dist_pt_seg_sqr2d(pos[0], pos[2], a, b, t);
    // the smallest by their bits, which order distances; a NaN is never smaller than what came before, so it
    // only counts as the first
    uint32_t key = d == d ? __float_as_uint(d) : j == 0 ? 0u : 0xfffffffeu;
    key = j < nv ? key : 0xffffffffu;
    const uint32_t nearest = Row::umin(key);
    const unsigned long long inside = lanes_where(crosses), first = lanes_where(key == nearest);
    const float on[3] = {a[0] + (b[0] - a[0]) * t, a[1] + (b[1] - a[1]) * t, a[2] + (b[2] - a[2]) * t};
    const int ls = first_lane(first & 0xffull), le = first_lane(first & 0xff00ull);
    const bool sIn = __popcll(inside & 0xffull) & 1, eIn = __popcll(inside & 0xff00ull) & 1;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      cs[k] = sIn ? startPos[k] : lane_f(on[k], ls);
      ce[k] = eIn ? endPos[k] : lane_f(on[k], le);
    }
  }
  if (lane < 6) F->portals[n - 1][lane] = lane == 0 || lane == 3 ? ce[0] : lane == 1 || lane == 4 ? ce[1] : ce[2];   // where the walk ends
  wave_sync();
  if (lanes_where(missing)) return INF;
  // straight-path points are only needed pairwise: keep the last one and the running length.
  // Every lane computes the same values; the conditions are taken through a ballot so that the
  // control flow is the scalar unit's (no lane masks, no copies at the joins).
  auto all = [](bool b) { return lanes_where(b) != 0; };
  float last[3] = {cs[0], cs[1], cs[2]};
  int npts = 1;
  float length = 0.0f;
  bool finished = false, overflow = false;
  int merged = 0;
  auto append = [&](const float* p, bool isEnd) {
    if (all(vequal(last, p))) {
      // Merged with the previous point.  Between finite portals the apex then moves on to a later one, but
      // for once at the first.  At a side that is not finite all may stay as it was, and the reference walks
      // for ever: no path.
      if (++merged > 2 * kMaxPath) { overflow = true; finished = true; }
      return;
    }
    const float dx = last[0] - p[0], dy = last[1] - p[1], dz = last[2] - p[2];
    length += sqrtf(dx * dx + (dy * dy + dz * dz));
    last[0] = p[0]; last[1] = p[1]; last[2] = p[2];
    npts++;
    if (npts >= kMaxPath) { overflow = true; finished = true; return; }
    if (isEnd) finished = true;
  };
  if (n > 1) {
    // Sixteen portals at a time: the first sixteen lanes have their right points, the next their left ones, relative to the
    // apex and, the left ones, mirrored, so that one rule serves both: a point that does not lie outside its side becomes
    // the side.  What the sides are behind each portal is a scan, of the narrower of two points; the comparisons of rounded
    // areas need not be transitive, so every portal's own test, against the side that the scan has put before it,
    // is made too, and where one of them says otherwise than the scan the round ends before that portal.  The first portal at
    // which a point crosses to the other side moves the apex.  A point's third word: its portal's index + 1 (0: the apex), and
    // whether it lies at the apex (vequal).
    const bool isLeft = (lane & 16) != 0;
    const uint32_t mirror = isLeft ? 0x80000000u : 0u, kAtApex = 0x10000u;
    const int j = lane & 15;
    const float* mine = &F->portals[0][isLeft ? 0 : 3];
    const float thr = (1.0f / 16384.0f) * (1.0f / 16384.0f);
    float ax = cs[0], ay = cs[1], az = cs[2];
    struct Side { float x, z; uint32_t at; } side;
    auto narrow = [&]() BPSX_INLINE_LAMBDA {   // both sides at the apex (0, or NaN for an apex that is not finite, as the difference is)
      const float x = ax - ax, y = ay - ay, z = az - az;
      side = {x, z, x * x + y * y + z * z < thr ? kAtApex : 0u};
    };
    narrow();
    auto area = [](float sx, float sz, float px, float pz) BPSX_INLINE_LAMBDA { return px * sz - sx * pz; };   // tri_area2d(apex, side, point)
    int apexIndex = 0;
    int leftLast = -1, rightLast = -1;       // the portal whose point the side was last: the last one is "poly ref == 0" of the reference
    int i = 0;
    {
      const float* p = F->portals[0];
      float t;
      const float l[3] = {p[0], p[1], p[2]}, r[3] = {p[3], p[4], p[5]};
      if (all(dist_pt_seg_sqr2d(ax, az, l, r, t) < 0.001f * 0.001f)) i = 1;
    }
    while (i < n) {
      const int k = i + j;
      const float* p = mine + 6 * (k < n ? k : n - 1);
      Side own, in, ex;
      const float px = p[0] - ax, py = p[1] - ay;
      own.z = p[2] - az;
      own.at = (uint32_t)(k + 1) | (px * px + py * py + own.z * own.z < thr ? kAtApex : 0u);
      own.x = __uint_as_float(__float_as_uint(px) ^ mirror);
      in = own;
      if (j == 0 && !(area(side.x, side.z, own.x, own.z) <= 0.0f)) in = side;
      static_for<0, 4>([&](auto K) BPSX_INLINE_LAMBDA {
        constexpr int up = 0x110 + (1 << decltype(K)::value);   // row_shr: that many lanes up
        const float ox = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(in.x), __float_as_int(in.x), up, 0xf, 0xf, false));
        const float oz = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(in.z), __float_as_int(in.z), up, 0xf, 0xf, false));
        const uint32_t oat = (uint32_t)__builtin_amdgcn_update_dpp((int)in.at, (int)in.at, up, 0xf, 0xf, false);
        const bool narrower = area(ox, oz, in.x, in.z) <= 0.0f;
        in.x = narrower ? in.x : ox;
        in.z = narrower ? in.z : oz;
        in.at = narrower ? in.at : oat;
      });
      // the sides before each portal
      ex.x = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(side.x), __float_as_int(in.x), 0x111, 0xf, 0xf, false));
      ex.z = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(side.z), __float_as_int(in.z), 0x111, 0xf, 0xf, false));
      ex.at = (uint32_t)__builtin_amdgcn_update_dpp((int)side.at, (int)in.at, 0x111, 0xf, 0xf, false);
      const bool moves = area(ex.x, ex.z, own.x, own.z) <= 0.0f;
      const bool differs = in.at != (moves ? own.at : ex.at);
      // the other side: for a right point the left one before the portal, for a left point the right one behind it
      const uint32_t sx = __float_as_uint(isLeft ? ex.x : in.x), sz = __float_as_uint(isLeft ? ex.z : in.z);
      const auto tx = __builtin_amdgcn_permlane16_swap(sx, sx, false, false), tz = __builtin_amdgcn_permlane16_swap(sz, sz, false, false);
      const float ox = -__uint_as_float(isLeft ? tx[0] : tx[1]), oz = __uint_as_float(isLeft ? tz[0] : tz[1]);   // mirrored as this lane's points
      const bool within = area(ox, oz, own.x, own.z) > 0.0f;
      const uint32_t valid = (n - i >= 16 ? 0xffffu : (1u << (n - i)) - 1u) * 0x10001u;
      const uint32_t bad = (uint32_t)lanes_where(differs) & valid;
      const uint32_t stops = (uint32_t)(lanes_where(moves) & ~(lanes_where((ex.at & kAtApex) != 0) | lanes_where(within))) & valid;
      // the first portals of either kind, 16 or more for none
      const int badAt = __builtin_ctz(((bad | (bad >> 16)) & 0xffffu) | 0x10000u);
      const int rightStop = __builtin_ctz((stops & 0xffffu) | 0x10000u), leftStop = __builtin_ctz((stops >> 16) | 0x10000u);
      const int stop = rightStop < leftStop ? rightStop : leftStop;
      if (stop >= badAt || stop == 16) {
        int m = n - i < 16 ? n - i : 16;
        m = badAt < m ? badAt : m;
        const uint32_t ra = rlane(in.at, m - 1), la = rlane(in.at, m + 15);
        side.x = isLeft ? lane_f(in.x, m + 15) : lane_f(in.x, m - 1);
        side.z = isLeft ? lane_f(in.z, m + 15) : lane_f(in.z, m - 1);
        side.at = isLeft ? la : ra;
        if (ra & 0xffffu) rightLast = (int)(ra & 0xffffu) - 1;
        if (la & 0xffffu) leftLast = (int)(la & 0xffffu) - 1;
        i += m;
        continue;
      }
      const bool atRight = rightStop <= leftStop;   // of one portal the right point comes first
      const int ra = (int)(rlane(atRight ? ex.at : in.at, stop) & 0xffffu), la = (int)(rlane(ex.at, stop + 16) & 0xffffu);
      if (ra) rightLast = ra - 1;
      if (la) leftLast = la - 1;
      const int to = atRight ? la : ra;
      if (to) {
        apexIndex = to - 1;
        const float* q = F->portals[apexIndex] + (atRight ? 0 : 3);
        ax = q[0]; ay = q[1]; az = q[2];
      }
      const float apex[3] = {ax, ay, az};
      append(apex, (atRight ? leftLast : rightLast) + 1 == n);
      if (finished) break;
      narrow();
      i = apexIndex + 1;
    }
  }
  if (!finished) {
    append(ce, true);
    if (npts >= kMaxPath) overflow = true;
  }
  return overflow ? INF : length;
}

// Full PathFinder::findPath distance for one query, executed by a wavefront.
BPSX_DEV float geodesic_query(GeoWave& g, const NavData& nav, const GeoQuery& q, uint32_t* pops, uint32_t* corridor) {
  const float INF = __int_as_float(0x7f800000);
  {
    // Eigen isApprox with default precision; sums of three reduce as a0 + (a1 + a2)
    const float d0 = q.a[0] - q.b[0], d1 = q.a[1] - q.b[1], d2 = q.a[2] - q.b[2];
    const float dd = d0 * d0 + (d1 * d1 + d2 * d2);
    const float aa = q.a[0] * q.a[0] + (q.a[1] * q.a[1] + q.a[2] * q.a[2]);
    const float bb = q.b[0] * q.b[0] + (q.b[1] * q.b[1] + q.b[2] * q.b[2]);
    const float mn = bb < aa ? bb : aa;
    const float prec = 1e-5f;
    if (dd <= prec * prec * mn) return 0.0f;
  }
  const SceneDev& s = nav.scenes[q.scene];
  const uint32_t sIp = decode_ref(s, q.a_ref), eIp = decode_ref(s, q.b_ref);
  if (sIp == kInvalidPoly || eIp == kInvalidPoly) return INF;
  if (nav.polys[s.poly_base + sIp].island != nav.polys[s.poly_base + eIp].island) return INF;
  if (!finite3(q.a[0], q.a[1], q.a[2]) || !finite3(q.b[0], q.b[1], q.b[2])) return INF;
  FunnelLds* F = &reinterpret_cast<GeoShared*>(g.L)->f;
  const int n = astar(g, F, nav, s, sIp, eIp, q.a, q.b, pops);
  if (n <= 0) return INF;
  *corridor += (uint32_t)n;
  const float len = funnel_length(g.lane, F, nav, s, n, q.a, q.b);
  return len;
}

}  // namespace BPSX_GEO_NS
}  // namespace bpsx
