// HIP kernels of the batch environment step (gfx950) and their launch wrappers.
//
// One step of a group of n point-goal or fleeing agents is three launches:
//   step_move      row of eight lanes per agent: action, turn / forward move with wall sliding, polar
//                  observation, and a geodesic query (goal -> agent) when the agent moved or
//                  the episode ended; an agent whose episode ended also picks its next episode
//                  here and is queued for reset (simulator.cpp:620-632, 651-710, 601-610)
//   geodesic       wavefront per query, both kinds in one launch: A* + funnel; blocks of two
//                  wavefronts so that the longest searches can take a block's whole LDS, or in launches of
//                  fewer queries a block per query
//                                                        (PathFinder.cpp:485-541)
//   step_finish    lane per agent: info, reward, mask from the terminal transition, then the
//                  new episode's distance bookkeeping    (simulator.cpp:634-641, 758-822, 749-755)
// In blocks of their own in one of the last two (geodesic where its searches leave room) a wavefront per snap: start
// and goal of the new episode, polar, and the new episode's first query (agent -> goal) (simulator.cpp:611-614, 744-751).
// The first query of an episode that begins in step t is answered by step t + 1's geodesic launch, and
// its result enters the bookkeeping at the start of step t + 1's step_finish.  No output of step t
// depends on it (the reference computes it inside the reset and uses it from the next step on).  A reset
// of a whole group (bpsx_reset) draws the episodes and snaps their points before geodesic, first queries
// included: by one launch (k_reset_begin) while the device holds a wavefront for each point, by two beyond
// (k_reset_all, k_reset_snap).  A step whose launches are timed has k_reset_snap for the snaps, too.
// The Flee task (simulator.cpp:830-869) runs through the same launches:
// Flee keeps the episode's start point where PointNav keeps the snapped goal, so its
// "distance from start" is the same start-point -> agent query.  Exploration makes no queries and
// keeps its visited cells per agent in HBM; a step is one launch of its own (k_step_explore).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "../../include/bpsx.h"
#include "geodesic_device.h"
// A second instantiation of the same search for the few longest queries of a step: all 2048
// link words, twice the window and twice the hash heads in LDS.  Such a query takes the LDS of a
// whole two-wavefront block (see k_geodesic).
#undef BPSX_GEO_NS
#undef BPSX_LINKS_LDS
#undef BPSX_WINDOW
#undef BPSX_HASH
#define BPSX_GEO_NS geo_long
#define BPSX_LINKS_LDS 2048
#define BPSX_WINDOW 256
#define BPSX_HASH 1024
#include "geodesic_device.h"
// A third, for launches that have a block for each query or nearly so: 2048 hash heads, and a second
// wavefront that keeps the reference's heap, 20 KB for both (see k_geodesic_mid).
#undef BPSX_GEO_NS
#undef BPSX_HASH
#undef BPSX_FOLLOWER
#define BPSX_GEO_NS geo_mid
#define BPSX_HASH 2048
#define BPSX_FOLLOWER 1
#include "geodesic_device.h"
// And a fourth, for launches of few queries: the whole node pool in LDS as well, 52 KB (see k_geodesic_few).
#undef BPSX_GEO_NS
#undef BPSX_WINDOW
#define BPSX_GEO_NS geo_few
#define BPSX_WINDOW 2048
#include "geodesic_device.h"
#include "kernels.h"

namespace bpsx {

namespace {

// ---- counter-based reset stream (identical integer arithmetic on host and device)
BPSX_DEV uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
BPSX_DEV uint64_t reset_key(uint64_t seed, uint32_t env, uint32_t count) {
  return mix64(seed + 0x9E3779B97F4A7C15ull * ((uint64_t)env + 1) + 0xD1B54A32D192ED03ull * ((uint64_t)count + 1));
}
BPSX_DEV uint32_t reset_draw(uint64_t key, uint32_t k) {
  return (uint32_t)(mix64(key + 0x9E3779B97F4A7C15ull * ((uint64_t)k + 1)) >> 32);
}
BPSX_DEV uint32_t draw_index(uint32_t r, uint32_t n) { return (uint32_t)(((uint64_t)r * (uint64_t)n) >> 32); }
BPSX_DEV float draw_unit(uint32_t r) { return (float)(r >> 8) * (1.0f / 16777216.0f); }

// ---- glm closed forms, quaternions stored x,y,z,w
BPSX_DEV void quat_mul(const float* p, const float* q, float* o) {
  const float w = p[3] * q[3] - p[0] * q[0] - p[1] * q[1] - p[2] * q[2];
  const float x = p[3] * q[0] + p[0] * q[3] + p[1] * q[2] - p[2] * q[1];
  const float y = p[3] * q[1] + p[1] * q[3] + p[2] * q[0] - p[0] * q[2];
  const float z = p[3] * q[2] + p[2] * q[3] + p[0] * q[1] - p[1] * q[0];
  o[0] = x; o[1] = y; o[2] = z; o[3] = w;
}
BPSX_DEV void cross3(const float* a, const float* b, float* o) {
  o[0] = a[1] * b[2] - b[1] * a[2];
  o[1] = a[2] * b[0] - b[2] * a[0];
  o[2] = a[0] * b[1] - b[0] * a[1];
}
BPSX_DEV void quat_rotate(const float* q, const float* v, float* o) {
  float uv[3], uuv[3];
  cross3(q, v, uv);
  cross3(q, uv, uuv);
  for (int k = 0; k < 3; ++k) o[k] = v[k] + ((uv[k] * q[3]) + uuv[k]) * 2.0f;
}
// polar observation (rho, -phi) of the goal in the agent's frame (simulator.cpp:666-676)
BPSX_DEV void write_polar(const AgentArrays& A, uint32_t gi, const float* pos, const float* q, const float* goal) {
  const float v[3] = {goal[0] - pos[0], goal[1] - pos[1], goal[2] - pos[2]};
  const float qxx = q[0] * q[0], qyy = q[1] * q[1], qzz = q[2] * q[2];
  const float qxz = q[0] * q[2], qxy = q[0] * q[1], qyz = q[1] * q[2];
  const float qwx = q[3] * q[0], qwy = q[3] * q[1], qwz = q[3] * q[2];
  const float m00 = 1.0f - 2.0f * (qyy + qzz), m01 = 2.0f * (qxy + qwz), m02 = 2.0f * (qxz - qwy);
  const float m20 = 2.0f * (qxz + qwy), m21 = 2.0f * (qyz - qwx), m22 = 1.0f - 2.0f * (qxx + qyy);
  const float vx = m00 * v[0] + m01 * v[1] + m02 * v[2];
  const float vz = m20 * v[0] + m21 * v[1] + m22 * v[2];
  const float x = -vz, y = vx;
  A.polars[(size_t)gi * 2 + 0] = sqrtf(x * x + y * y);
  A.polars[(size_t)gi * 2 + 1] = -atan2f(y, x);
}

// the copy of the counters that this block adds to
BPSX_DEV uint64_t* counter_shard(uint64_t* counters) { return counters + (blockIdx.x % kCounterShards) * kCounterStride; }

BPSX_DEV void load3(const float* p, size_t i, float* o) { o[0] = p[i * 3]; o[1] = p[i * 3 + 1]; o[2] = p[i * 3 + 2]; }
BPSX_DEV void store3(float* p, size_t i, const float* v) { p[i * 3] = v[0]; p[i * 3 + 1] = v[1]; p[i * 3 + 2] = v[2]; }

// Exploration::InfoFunctor::update (simulator.cpp:897-904): the cell of the agent in the frame
// of the episode's start pose (position ip, inverse rotation iq) ...
BPSX_DEV void cell_of(const float* ip, const float* iq, const float* pos, int32_t* c) {
  const float d[3] = {pos[0] - ip[0], pos[1] - ip[1], pos[2] - ip[2]};
  float g[3];
  quat_rotate(iq, d, g);
  // int(x) of the reference; for a value no int32 holds (or NaN) the x86 conversion the
  // reference compiles to gives INT32_MIN, the GPU's would saturate: made explicit
  for (int k = 0; k < 3; ++k) {
    const float x = g[k] / 1.0f;
    c[k] = (x > -2147483648.0f && x < 2147483648.0f) ? (int32_t)x : (int32_t)0x80000000;
  }
}
// ... joins the episode's set of n cells.  Returns the set's size.  By a row of eight lanes, eight cells
// at a time (an agent that wanders for hundreds of steps has entered up to a hundred).
BPSX_DEV uint32_t visit_cell(const Row& row, const AgentArrays& A, uint32_t gi, uint32_t n, const float* ip, const float* iq, const float* pos) {
  int32_t c[3];
  cell_of(ip, iq, pos, c);
  int32_t* cells = A.exp_cells + (size_t)gi * A.cell_cap * 3;
  for (uint32_t i = 0; i < n; i += 8) {
    const uint32_t k = i + (uint32_t)row.el;
    const int32_t* o = &cells[(size_t)(k < n ? k : i) * 3];
    if (row.mask(o[0] == c[0] && o[1] == c[1] && o[2] == c[2])) return n;
  }
  if (n >= A.cell_cap) return n;   // cannot happen: one update per step and per reset
  if (row.el == 0) {
    for (int k = 0; k < 3; ++k) cells[(size_t)n * 3 + k] = c[k];
    A.exp_count[gi] = n + 1;
  }
  return n + 1;
}

// The end of a block of a step's last launch, for all its threads.  Its last block of `blocks` tells a host that waits that all
// that the launch has written can be seen: a host that waits for an event behind the launch hears of it later (a step of 64
// agents in a room 121.4 -> 117.1 us, of 1024 that explore 27.4 -> 23.4).  One write-back for a block, once its
// wavefronts' stores have arrived: one for each wavefront costs the half of the gain.
BPSX_DEV void tell_host(const StepParams& P, uint32_t blocks) {
  if (!P.done_flag) return;
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x != 0) return;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
  const uint32_t before = atomicInc(P.done_blocks, blocks - 1u);   // 0 again after the last
  if (before == blocks - 1u) __hip_atomic_store(P.done_flag, P.done_value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// makes scene-table entry `target` what the envs of `slot` move to when their episodes end
__global__ void k_set_swap(uint32_t* swap_target, uint32_t* swap_remaining, uint32_t slot, uint32_t target, uint32_t envs) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    swap_remaining[slot] = envs;
    swap_target[slot] = target;
  }
}

// The next episode of agent gi in scene-table entry sc, its pose (position, rotation) and goal; returns its index.  By a
// row of eight lanes; count: the agent's resets so far.
BPSX_DEV uint32_t draw_episode(const Row& row, const NavData& nav, const StepParams& P, uint32_t gi, uint32_t sc, uint32_t count, float* ep) {
  const SceneDev& s = nav.scenes[sc];
  const uint64_t key = reset_key(P.seed, gi, count);
  uint32_t e = 0;
  if (P.reset_mode == 0) {
    e = draw_index(reset_draw(key, 0), s.ep_count);
    for (int k = 0; k < 10; ++k) ep[k] = nav.episodes[(size_t)(s.ep_base + e) * 10 + k];
  } else {
    float a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
    uint32_t ip;
    sample_point_row(row, nav, s, draw_unit(reset_draw(key, 0)), draw_unit(reset_draw(key, 1)), draw_unit(reset_draw(key, 2)), a, &ip);
    sample_point_row(row, nav, s, draw_unit(reset_draw(key, 3)), draw_unit(reset_draw(key, 4)), draw_unit(reset_draw(key, 5)), b, &ip);
    const uint32_t turns = draw_index(reset_draw(key, 6), 36);
    float q[4] = {0, 0, 0, 1};
    for (uint32_t t = 0; t < turns; ++t) quat_mul(q, P.turn_left, q);
    ep[0] = a[0]; ep[1] = a[1]; ep[2] = a[2];
    ep[3] = q[0]; ep[4] = q[1]; ep[5] = q[2]; ep[6] = q[3];
    ep[7] = b[0]; ep[8] = b[1]; ep[9] = b[2];
  }
  return e;
}
// and by one lane, the episode as the agent's
BPSX_DEV void store_episode(const AgentArrays& A, uint32_t gi, uint32_t count, uint32_t e, const float* ep) {
  A.nresets[gi] = count + 1;
  A.step[gi] = 1;
  A.last_cost[gi] = kCostUnknown;
  A.episode[gi] = e;
  store3(A.pos, gi, ep);
  for (int k = 0; k < 4; ++k) A.rot[(size_t)gi * 4 + k] = ep[3 + k];
  store3(A.goal, gi, ep + 7);
}
// Picks the next episode of agent gi and writes its pose; the snaps follow in reset_snap.
BPSX_DEV void begin_reset(const Row& row, const NavData& nav, const AgentArrays& A, const StepParams& P, uint32_t gi, uint32_t sc,
                          uint32_t count) {
  float ep[10];
  const uint32_t e = draw_episode(row, nav, P, gi, sc, count, ep);
  if (row.el == 0) store_episode(A, gi, count, e, ep);
}
// Where the agent's next episode takes place: if a new scene waits for this env's slot, there (simulator.cpp:1636-1642).
// By one lane.
BPSX_DEV uint32_t next_scene(const AgentArrays& A, const StepParams& P, uint32_t gi, uint32_t scene) {
  const uint32_t tgt = P.swap_target[scene % P.num_slots];
  if (tgt == kNoSwap || tgt == scene) return scene;
  A.scene[gi] = tgt;
  atomicSub(&P.swap_remaining[scene % P.num_slots], 1u);
  return tgt;
}

// A row of eight lanes per agent, kMoveItems agents per block: all lanes of a row read the agent's state
// and decide alike, the first one writes it.  Bound by latency, a chain of dependent loads (state,
// scene, polygon, its neighbours, height mesh), which is why the loads of one link go out together.
// (With a lane per agent: 33 us for 64 agents in a room, now 12; 1017 agents 41 -> 13; 16384 agents over
// mazes 35 -> 22; 4096 over cluttered plans with sampled resets, whose two searches for a polygon were
// thirty dependent reads, 79 -> 30; 65536 over mixed scenes 65, as before.)
struct MoveQueueLds {
  uint32_t count[kGeoClasses + 1], base[kGeoClasses + 1];   // of the block's queries per class, and of its resets
  uint32_t forward, polys;
};
__global__ __launch_bounds__(kMoveItems * 8) void k_step_move(NavData nav, AgentArrays A, StepQueues Q, StepParams P,
                                                   const int64_t* __restrict__ actions) {
  __shared__ MoveLds move_lds;
  __shared__ __attribute__((aligned(16))) uint16_t entered[kMoveItems][kTinyNodes];
  __shared__ MoveQueueLds queue;
  static_assert(kGeoClasses + 1 <= kMoveItems * 8, "a thread per class");
  if (threadIdx.x <= (uint32_t)kGeoClasses) queue.count[threadIdx.x] = 0;
  if (threadIdx.x == 0) queue.forward = queue.polys = 0;
  __syncthreads();
  const Row row;
  const uint32_t item = threadIdx.x >> 3, i = blockIdx.x * kMoveItems + item;
  const bool lead = row.el == 0;
  bool want = false, reset = false;
  uint32_t cls = 0;
  GeoQuery q{};
  uint32_t movePolys = 0, gi = 0;
  if (i < P.n) {
    gi = P.base + i;
    const int64_t action = actions[i];
    if (action < 0 || action > 3) {
      // the reference aborts here (simulator.cpp:704-708); flag it and leave the agent alone
      if (lead) {
        atomicOr(P.error_flag, 1u);
        A.flags[gi] = kAgentSkip;
      }
    } else {
      // Everything the step may need of the agent is read here, before the first store: the
      // loads then go out together instead of one dependent round trip after the other.
      const uint32_t step = A.step[gi] + 1;
      const uint32_t scene0 = A.scene[gi];
      float pos[3], rot[4], goal[3], navNow[3], goalNav[3];
      load3(A.pos, gi, pos);
      load3(A.goal, gi, goal);
      for (int k = 0; k < 4; ++k) rot[k] = A.rot[(size_t)gi * 4 + k];
      load3(A.nav_xyz, gi, navNow);
      uint32_t navRefNow = A.nav_ref[gi];
      load3(A.goal_xyz, gi, goalNav);
      const uint32_t goalRef = A.goal_ref[gi];
      const bool distOk = A.dist_ok[gi] == 1;
      const uint32_t expected = A.last_cost[gi];
      const uint32_t resets = A.nresets[gi];
      if (lead) A.step[gi] = step;
      bool done = (float)step >= P.max_steps;
      bool moved = false;
      // The goal->agent distance is a deterministic function of the two navmesh points. When
      // the agent's point is bit-identical to the one the last step query of this episode was
      // made for (blocked forward move, turn, stop), that query's result is the answer again.
      bool samePoint = true;
      if (action == 0) {
        done = true;
      } else {
        if (action == 1) {
          const float fwd[3] = {0.f * 0.25f, 0.f * 0.25f, -1.f * 0.25f};
          float delta[3];
          quat_rotate(rot, fwd, delta);
          const SceneDev& s = nav.scenes[scene0];
          const NavPt st{navNow[0], navNow[1], navNow[2], navRefNow};
          const NavPt r = try_step_row(row, nav, s, st, pos[0] + delta[0], pos[1] + delta[1], pos[2] + delta[2], &movePolys,
                                       entered[item], move_lds, (int)item);
          samePoint = __float_as_uint(r.x) == __float_as_uint(st.x) && __float_as_uint(r.y) == __float_as_uint(st.y) &&
                      __float_as_uint(r.z) == __float_as_uint(st.z) && r.ref == st.ref;
          pos[0] = r.x; pos[1] = r.y; pos[2] = r.z;
          navNow[0] = r.x; navNow[1] = r.y; navNow[2] = r.z;
          navRefNow = r.ref;
          if (lead) {
            store3(A.nav_xyz, gi, pos);
            A.nav_ref[gi] = r.ref;
            store3(A.pos, gi, pos);
          }
          moved = true;
        } else {
          quat_mul(rot, action == 2 ? P.turn_left : P.turn_right, rot);
          if (lead) for (int k = 0; k < 4; ++k) A.rot[(size_t)gi * 4 + k] = rot[k];
        }
        if (lead) write_polar(A, gi, pos, rot, goal);
      }
      // PointNav measures the distance on every move and at the end of the episode, Flee on
      // moves only (simulator.cpp:758-790, 845-856)
      const bool measure = moved || (done && P.task == BPSX_TASK_POINTNAV);
      const bool reuse = measure && samePoint && distOk;
      if (lead) A.flags[gi] = (done ? kAgentDone : 0u) | (moved ? kAgentMoved : 0u) | (reuse ? kAgentReuse : 0u);
      if (measure && !reuse) {
        want = true;
        for (int k = 0; k < 3; ++k) { q.a[k] = goalNav[k]; q.b[k] = navNow[k]; }
        q.a_ref = goalRef;
        q.b_ref = navRefNow;
        q.scene = scene0;
        q.out = gi;
        q.cost_slot = done ? kNoCostSlot : gi;   // a finished episode's search predicts nothing
        q.pad = 0;
        cls = expected == kCostUnknown ? kGeoClassUnknown : geo_class(expected);
      }
      if (done) {
        // the terminal query above holds copies of the old episode's points: the pose arrays can
        // take the next episode now; distance bookkeeping waits for step_finish.
        uint32_t scene = scene0;
        if (lead) scene = next_scene(A, P, gi, scene0);
        scene = row.get(scene, 0);
        begin_reset(row, nav, A, P, gi, scene, resets);
        reset = true;
      }
    }
  }
  // Queue the queries and the resets: places within the block from counters in LDS, then one atomic per
  // block and class present in it, all of them in flight together.
  want = want && lead;
  reset = reset && lead;
  uint32_t place = 0, rplace = 0;
  if (want) place = atomicAdd(&queue.count[cls], 1u);
  if (reset) rplace = atomicAdd(&queue.count[kGeoClasses], 1u);
  if (lead && movePolys) {
    atomicAdd(&queue.forward, 1u);
    atomicAdd(&queue.polys, movePolys);
  }
  __syncthreads();
  if (threadIdx.x <= (uint32_t)kGeoClasses && queue.count[threadIdx.x])
    queue.base[threadIdx.x] = atomicAdd(&Q.counts[threadIdx.x < (uint32_t)kGeoClasses ? kQGeo + threadIdx.x : (uint32_t)kQReset], queue.count[threadIdx.x]);
  if (threadIdx.x == 0 && queue.forward) {
    atomicAdd((unsigned long long*)&counter_shard(P.counters)[kCntForward], (unsigned long long)queue.forward);
    atomicAdd((unsigned long long*)&counter_shard(P.counters)[kCntMovePolys], (unsigned long long)queue.polys);
  }
  __syncthreads();
  if (want) Q.queries[(size_t)cls * Q.stride + queue.base[cls] + place] = q;
  if (reset) Q.reset_list[queue.base[kGeoClasses] + rplace] = gi;
  if (i == 0 && lead) atomicAdd((unsigned long long*)&counter_shard(P.counters)[kCntSteps], (unsigned long long)P.n);
}

// The state that hangs on an episode's start point, p snapped to r, and the polar observation.  By one lane.
BPSX_DEV void start_state(const AgentArrays& A, uint32_t task, uint32_t gi, const float* p, const float* rot, const float* goal, const NavPt& r) {
  const float xyz[3] = {r.x, r.y, r.z};
  store3(A.nav_xyz, gi, xyz);
  A.nav_ref[gi] = r.ref;
  write_polar(A, gi, p, rot, goal);
  if (task == BPSX_TASK_POINTNAV) return;
  const float zero[3] = {0, 0, 0};
  const bool flee = task == BPSX_TASK_FLEE;
  store3(A.goal_xyz, gi, flee ? xyz : zero);   // Flee: navmeshStart_
  A.goal_ref[gi] = flee ? r.ref : 0u;
  if (!flee) {
    // glm::inverse(q) = conjugate(q) / dot(q, q)
    const float d = (rot[3] * rot[3] + rot[0] * rot[0]) + (rot[1] * rot[1] + rot[2] * rot[2]);
    const float inv[4] = {-rot[0] / d, -rot[1] / d, -rot[2] / d, rot[3] / d};
    for (int k = 0; k < 4; ++k) A.exp_inv[(size_t)gi * 4 + k] = inv[k];
    store3(A.exp_init, gi, p);
    cell_of(p, inv, p, A.exp_cells + (size_t)gi * A.cell_cap * 3);   // the set's first
    A.exp_count[gi] = 1;
  }
}

// by one lane: the snapped goal, and it and the snapped start in the episode's first query
BPSX_DEV void goal_state(const AgentArrays& A, uint32_t gi, const NavPt& r, GeoQuery* q) {
  const float xyz[3] = {r.x, r.y, r.z};
  store3(A.goal_xyz, gi, xyz);
  A.goal_ref[gi] = r.ref;
  q->b[0] = r.x; q->b[1] = r.y; q->b[2] = r.z; q->b_ref = r.ref;
}
BPSX_DEV void start_of_query(const StepParams& P, uint32_t gi, uint32_t scene, const NavPt& r, GeoQuery* q) {
  q->a[0] = r.x; q->a[1] = r.y; q->a[2] = r.z; q->a_ref = r.ref;
  q->scene = scene;
  q->out = P.total + gi;
  q->cost_slot = kNoCostSlot;   // searched agent -> goal: says little about the searches to come
  q->pad = 0;
}
// The snaps of the episodes that begin, a wavefront for each start and, in PointNav, each goal (the
// other tasks snap no goal, simulator.cpp:838-843, 906-916): wavefront w of nw takes every nw-th.  The
// wavefront of the start writes the state that hangs on it and the polar observation; each writes its
// half of the episode's first query (agent -> goal) to Qout, in the order of the reset list: the class
// of unknown length is empty when this begins (the queues of the next step, or cleared ones) and
// nothing else fills it meanwhile.
BPSX_DEV void snap_new_episodes(const NavData& nav, const AgentArrays& A, const StepQueues& Q, const StepQueues& Qout, const StepParams& P,
                                uint32_t w, uint32_t nw, SnapLds& lds) {
  const uint32_t n = Q.counts[kQReset];
  const bool pointnav = P.task == BPSX_TASK_POINTNAV;
  const bool first = (threadIdx.x & 63u) == 0;
  uint32_t cands = 0;
  for (uint32_t it = w; it < (pointnav ? 2u * n : n); it += nw) {
    const uint32_t i = pointnav ? it >> 1 : it;
    const bool ofGoal = pointnav && (it & 1u);
    const uint32_t gi = Q.reset_list[i], scene = A.scene[gi];
    float p[3];
    load3(ofGoal ? A.goal : A.pos, gi, p);
    const NavPt r = snap_point_wave(nav, nav.scenes[scene], p[0], p[1], p[2], lds, &cands);
    if (!first) continue;
    GeoQuery* q = &Qout.queries[(size_t)kGeoClassUnknown * Qout.stride + i];   // a new episode: no history
    if (ofGoal) {
      goal_state(A, gi, r, q);
      continue;
    }
    float goal[3], rot[4];
    load3(A.goal, gi, goal);
    for (int k = 0; k < 4; ++k) rot[k] = A.rot[(size_t)gi * 4 + k];
    start_state(A, P.task, gi, p, rot, goal, r);
    if (pointnav) start_of_query(P, gi, scene, r, q);
  }
  if (w == 0 && first && n) {
    atomicAdd((unsigned long long*)&counter_shard(P.counters)[kCntResets], (unsigned long long)n);
    if (pointnav) Qout.counts[kQGeo + kGeoClassUnknown] = n;
  }
  if (first && cands) atomicAdd((unsigned long long*)&counter_shard(P.counters)[kCntSnapCands], (unsigned long long)cands);
}
constexpr uint32_t kSnapWaves = 4;   // per block
// 128 of the 133 registers that the compiler would take, without scratch: a whole-group reset of 2048 agents
// has 4096 snaps, which then all run at once.
__global__ __launch_bounds__(kSnapWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_reset_snap(NavData nav, AgentArrays A, StepQueues Q, StepQueues Qout, StepParams P) {
  __shared__ SnapLds lds[kSnapWaves];
  const uint32_t half = threadIdx.x >> 6;
  snap_new_episodes(nav, A, Q, Qout, P, blockIdx.x * kSnapWaves + half, gridDim.x * kSnapWaves, lds[half]);
}

// The bookkeeping of a step's agent.
BPSX_DEV void finish_agent(const AgentArrays& A, const StepParams& P, uint32_t gi) {
  const uint32_t f = A.flags[gi];
  if (f & kAgentSkip) return;
  const bool done = f & kAgentDone, moved = f & kAgentMoved;
  if (P.task != BPSX_TASK_POINTNAV) {
    if (!(f & kAgentResetOnly)) {
      // Flee (an exploring agent comes here for its reset only)
      float v = A.info_prev[gi];
      if (moved) {
        if (!(f & kAgentReuse)) v = A.geo[gi];
        A.info_prev[gi] = v;
        A.dist_ok[gi] = 1;
      }
      A.rewards[gi] = v - A.rew_prev[gi];
      A.rew_prev[gi] = v;
      A.masks[gi] = done ? 0 : 1;
      A.infos[gi] = v;
    }
    if (done || (f & kAgentResetOnly)) {
      // Flee: distance 0 at the start; Exploration: the start cell is in the set (count 1)
      A.info_prev[gi] = 0.0f;
      A.rew_prev[gi] = 0.0f;
      A.dist_ok[gi] = 0;
    }
    return;
  }
  if (A.dist_ok[gi] == 2) {
    // the episode began in the previous step: its first distance has been measured in this one
    const float d = A.geo[(size_t)P.total + gi];
    A.init[gi] = d;
    A.info_prev[gi] = d;   // agent->goal: not a goal->agent result, so not reusable
    A.rew_prev[gi] = d;
    A.dist_ok[gi] = 0;
  }
  if (!(f & kAgentResetOnly)) {
    float dist, success = 0, spl = 0;
    const float fresh = (f & kAgentReuse) ? A.info_prev[gi] : A.geo[gi];
    if (done) {
      dist = fresh;
      success = dist < 0.2f ? 1.0f : 0.0f;
      const float init = A.init[gi], cum = A.cum[gi];
      const float mx = init < cum ? cum : init;
      spl = success * init / mx;
    } else if (moved) {
      dist = fresh;
      A.dist_ok[gi] = 1;
      float pos[3], pp[3];
      load3(A.pos, gi, pos);
      load3(A.prev_pos, gi, pp);
      const float dx = pos[0] - pp[0], dy = pos[1] - pp[1], dz = pos[2] - pp[2];
      A.cum[gi] = A.cum[gi] + sqrtf(dx * dx + dy * dy + dz * dz);
      A.info_prev[gi] = dist;
      store3(A.prev_pos, gi, pos);
    } else {
      dist = A.info_prev[gi];
    }
    float reward = -1e-2f;
    if (done) reward += 2.5f * spl;
    else reward += A.rew_prev[gi] - dist;
    A.rew_prev[gi] = dist;
    A.rewards[gi] = reward;
    A.masks[gi] = done ? 0 : 1;
    A.infos[(size_t)gi * 3 + 0] = success;
    A.infos[(size_t)gi * 3 + 1] = spl;
    A.infos[(size_t)gi * 3 + 2] = dist;
  }
  if (done || (f & kAgentResetOnly)) {
    // InfoFunctor::reset / RewardFunctor::reset with the new episode's first distance, which a
    // step leaves to the next step's launch (no output of this step depends on it)
    A.cum[gi] = 0;
    if (P.defer_first_distance && !(f & kAgentResetOnly)) {
      A.dist_ok[gi] = 2;
    } else {
      const float d = A.geo[(size_t)P.total + gi];
      A.init[gi] = d;
      A.info_prev[gi] = d;   // agent->goal: not a goal->agent result, so not reusable
      A.dist_ok[gi] = 0;
      A.rew_prev[gi] = d;
    }
    float pos[3];
    load3(A.pos, gi, pos);
    store3(A.prev_pos, gi, pos);
  }
}

// A step of exploring agents, which ask for no distance: one launch.  A block has kRowWaves wavefronts of eight agents each, a row
// of eight lanes for an agent as in k_step_move, with the bookkeeping by the row itself, and kSnaps wavefronts that begin the episodes
// of those that end while the rows move: whether an episode ends hangs on the action and on the step's number alone.  Their
// rows draw all of the block's episodes, one each, and each wavefront snaps the start of one.  What that writes is in the rows'
// place only when those are done; if more episodes end than there are such wavefronts, all of the block's take the rest.  With no
// such wavefront the others draw when they have moved.
// Bound by latency, as moves and snaps are, 12 us each.  No list of queries or resets is filled, so the counters of both sets of queues
// stay as they are, empty.
// (As k_step_move and k_step_finish, with the snaps in the second, one after the other: 1017 agents over room plans 41.4 us a
// step, now 24.)
template <uint32_t kRowWaves, uint32_t kSnaps>
__global__ __launch_bounds__((kRowWaves + kSnaps) * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_step_explore(
    NavData nav, AgentArrays A, StepParams P, const int64_t* __restrict__ actions) {
  constexpr uint32_t kWaves = kRowWaves + kSnaps, kItems = kRowWaves * 8;
  static_assert(kItems <= kMoveItems);
  __shared__ MoveLds move_lds;
  __shared__ __attribute__((aligned(16))) uint16_t entered[kItems][kTinyNodes];
  __shared__ SnapLds snap_lds[kWaves];
  __shared__ struct {
    uint32_t count, forward, polys, cands;
    uint32_t gi[kItems], scene[kItems], resets[kItems];
    float pose[kItems][10];   // of the episodes that begin, and their indices
    uint32_t episode[kItems];
  } ends;   // the episodes that end in the block
  if (threadIdx.x == 0) ends.count = ends.forward = ends.polys = ends.cands = 0;
  __syncthreads();
  const Row row;
  const uint32_t wave = (uint32_t)uniform_i((int)(threadIdx.x >> 6));
  const bool lead = row.el == 0, of_rows = wave < kRowWaves;
  const uint32_t item = threadIdx.x >> 3, i = blockIdx.x * kItems + item;
  uint32_t gi = 0, scene0 = 0, navRef = 0, cnt = 0;
  int64_t action = -1;
  bool done = false;
  float pos[3], rot[4], goal[3], navNow[3], ip[3], iq[4], rewPrev = 0;
  if (of_rows && i < P.n) {
    gi = P.base + i;
    action = actions[i];
    if (action < 0 || action > 3) {
      // the reference aborts here (simulator.cpp:704-708); flag it and leave the agent alone
      if (lead) atomicOr(P.error_flag, 1u);
      action = -1;
    } else {
      // all that the step needs of the agent, asked for together
      const uint32_t step = A.step[gi] + 1, resets = A.nresets[gi];
      scene0 = A.scene[gi];
      load3(A.pos, gi, pos);
      load3(A.goal, gi, goal);
      for (int k = 0; k < 4; ++k) rot[k] = A.rot[(size_t)gi * 4 + k];
      load3(A.nav_xyz, gi, navNow);
      navRef = A.nav_ref[gi];
      cnt = A.exp_count[gi];
      load3(A.exp_init, gi, ip);
      for (int k = 0; k < 4; ++k) iq[k] = A.exp_inv[(size_t)gi * 4 + k];
      rewPrev = A.rew_prev[gi];
      done = action == 0 || (float)step >= P.max_steps;
      if (lead) {
        A.step[gi] = step;
        if (done) {
          const uint32_t k = atomicAdd(&ends.count, 1u);
          ends.gi[k] = gi; ends.scene[k] = next_scene(A, P, gi, scene0); ends.resets[k] = resets;
        }
      }
    }
  }
  __syncthreads();
  const uint32_t nends = (uint32_t)uniform_i((int)ends.count);
  uint32_t cands = 0;
  NavPt start{};
  auto snap = [&](uint32_t k) {
    const float* ep = ends.pose[k];
    const uint32_t scene = (uint32_t)uniform_i((int)ends.scene[k]);
    start = snap_point_wave(nav, nav.scenes[scene], lane_f(ep[0], 0), lane_f(ep[1], 0), lane_f(ep[2], 0), snap_lds[wave], &cands);
  };
  auto store = [&](uint32_t k) {
    if ((threadIdx.x & 63u) != 0) return;
    const float* ep = ends.pose[k];
    store_episode(A, ends.gi[k], ends.resets[k], ends.episode[k], ep);
    start_state(A, BPSX_TASK_EXPLORATION, ends.gi[k], ep, ep + 3, ep + 7, start);
  };
  // a wavefront's share of all that end, eight at a time
  constexpr uint32_t kDrawers = kSnaps ? kSnaps : kWaves;
  const uint32_t mine = kSnaps ? wave - kRowWaves : wave;
  auto draw = [&]() {
    for (uint32_t k0 = mine; k0 < nends; k0 += kDrawers * 8u) {
      const uint32_t k = k0 + kDrawers * ((threadIdx.x & 63u) >> 3);
      if (k < nends) {
        float ep[10];
        const uint32_t e = draw_episode(row, nav, P, ends.gi[k], ends.scene[k], ends.resets[k], ep);
        if (lead) {
          for (int j = 0; j < 10; ++j) ends.pose[k][j] = ep[j];
          ends.episode[k] = e;
        }
      }
    }
    wave_sync();
  };
  const bool snaps = !of_rows && mine < nends;
  if (!of_rows) {
    draw();
    if (snaps) snap(mine);
  } else if (action >= 0) {
    bool moved = false;
    if (action == 1) {
      const float fwd[3] = {0.f * 0.25f, 0.f * 0.25f, -1.f * 0.25f};
      float delta[3];
      quat_rotate(rot, fwd, delta);
      const NavPt st{navNow[0], navNow[1], navNow[2], navRef};
      uint32_t polys = 0;
      const NavPt r = try_step_row(row, nav, nav.scenes[scene0], st, pos[0] + delta[0], pos[1] + delta[1], pos[2] + delta[2], &polys,
                                   entered[item], move_lds, (int)item);
      pos[0] = r.x; pos[1] = r.y; pos[2] = r.z;
      if (lead) {
        store3(A.nav_xyz, gi, pos);
        A.nav_ref[gi] = r.ref;
        store3(A.pos, gi, pos);
        if (polys) { atomicAdd(&ends.forward, 1u); atomicAdd(&ends.polys, polys); }
      }
      moved = true;
    } else if (action > 1) {
      quat_mul(rot, action == 2 ? P.turn_left : P.turn_right, rot);
      if (lead) for (int k = 0; k < 4; ++k) A.rot[(size_t)gi * 4 + k] = rot[k];
    }
    if (moved) cnt = visit_cell(row, A, gi, cnt, ip, iq, pos);
    if (lead) {
      if (action != 0) write_polar(A, gi, pos, rot, goal);
      // (simulator.cpp:918-940)
      const float v = (float)(cnt - 1);
      A.rewards[gi] = (float)(0.25 * (double)(v - rewPrev));
      A.masks[gi] = done ? 0 : 1;
      A.infos[gi] = v;
      A.rew_prev[gi] = done ? 0.0f : v;
      if (done) { A.info_prev[gi] = 0.0f; A.dist_ok[gi] = 0; }
    }
  }
  if constexpr (kSnaps == 0) draw();
  __syncthreads();
  if (snaps) store(mine);
  for (uint32_t k = kSnaps + wave; k < nends; k += kWaves) {
    snap(k);
    store(k);
  }
  if ((threadIdx.x & 63u) == 0 && cands) atomicAdd(&ends.cands, cands);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t* counters = counter_shard(P.counters);
    auto count = [&](int c, uint32_t n) { if (n) atomicAdd((unsigned long long*)&counters[c], (unsigned long long)n); };
    count(kCntForward, ends.forward);
    count(kCntMovePolys, ends.polys);
    count(kCntResets, nends);
    count(kCntSnapCands, ends.cands);
    if (blockIdx.x == 0) count(kCntSteps, P.n);
  }
  tell_host(P, gridDim.x);
}

// The bookkeeping of a step's agents, and in its first snap_blocks blocks, unless the searches' launch has taken
// them, the snaps of the episodes that began in it, which touch nothing that the bookkeeping touches: no output of this step depends on an
// episode's first distance (the reference computes it inside the reset and uses it from the next step
// on), so its query goes to the next step's queues.
// (On a second stream next to the searches they cost the step two waits between streams, 6 to 17 us before
// the searches begin and 6 at its end, for the 9 us by which they outlast the bookkeeping of a small
// group: a step of 64 agents 232 us, now 219.  At 16384 agents, whose 655
// new episodes take 22 us here, it makes no difference: 1193 us both ways without the copies of the counters.)
// Q: the lists of queries that this step's searches have just served; Qnext: the other set.  The
// counters of both are left as the next step expects them, so that a step needs no launch of its own
// for it: the served lists and their ticket counter empty, and the reset list of the step before.
__global__ __launch_bounds__(256) void k_step_finish(NavData nav, AgentArrays A, StepParams P, StepQueues Q, StepQueues Qnext, uint32_t snap_blocks) {
  __shared__ SnapLds lds[kSnapWaves];
  static_assert(kSnapWaves * 64 == 256, "a wavefront each");
  if (blockIdx.x < snap_blocks) {
    const uint32_t wave = threadIdx.x >> 6;
    snap_new_episodes(nav, A, Q, Qnext, P, blockIdx.x * kSnapWaves + wave, snap_blocks * kSnapWaves, lds[wave]);
  } else {
    const uint32_t block = blockIdx.x - snap_blocks;
    if (block == 0) {
      static_assert(kQGeoHead == kQGeo + kGeoClasses && kGeoClasses + 1 < 256, "one thread per counter");
      if (threadIdx.x <= (uint32_t)kGeoClasses) Q.counts[kQGeo + threadIdx.x] = 0;
      else if (threadIdx.x == (uint32_t)kGeoClasses + 1u) Qnext.counts[kQReset] = 0;
    }
    const uint32_t i = block * 256u + threadIdx.x;
    if (i < P.n) finish_agent(A, P, P.base + i);
  }
  tell_host(P, gridDim.x);
}

// A reset of all agents of a group: their episodes drawn, for k_reset_snap.
__global__ __launch_bounds__(256) void k_reset_all(NavData nav, AgentArrays A, StepQueues Q, StepQueues Qother, StepParams P) {
  // both sets of queues are empty but for the list of resets
  if (blockIdx.x == 0 && threadIdx.x < kQCounters) {
    Q.counts[threadIdx.x] = threadIdx.x == kQReset ? P.n : 0u;
    Qother.counts[threadIdx.x] = 0u;
  }
  const uint32_t i = blockIdx.x * 32u + (threadIdx.x >> 3);   // a row of eight lanes per agent
  if (i >= P.n) return;
  const Row row;
  const uint32_t gi = P.base + i;
  begin_reset(row, nav, A, P, gi, A.scene[gi], A.nresets[gi]);
  if (row.el != 0) return;
  A.flags[gi] = kAgentResetOnly;
  Q.reset_list[i] = gi;
}

// Both by one launch: the wavefront of a start draws its agent's episode, for that of the goal too.  Both sets of queues are empty but
// for the episodes' first queries.  Bound by latency, the chain of the draw and of the snap.  (As two launches, and as one: 64
// point-goal agents 127 and 123 us, 2048 over mazes 383 and 380, 1024 fleeing ones 33.7 and 29.5, 4096 exploring ones 52.3 and 49.8.)
__global__ __launch_bounds__(kSnapWaves * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_reset_begin(NavData nav, AgentArrays A, StepQueues Q, StepQueues Qother, StepParams P) {
  __shared__ SnapLds lds[kSnapWaves];
  __shared__ float pose[kSnapWaves][10];   // of the episode that a wavefront has drawn
  const bool pointnav = P.task == BPSX_TASK_POINTNAV;
  const uint32_t wave = (uint32_t)uniform_i((int)(threadIdx.x >> 6)), items = pointnav ? 2u * P.n : P.n;
  const bool first = (threadIdx.x & 63u) == 0;
  static_assert(kQCounters <= kSnapWaves * 64, "one thread per counter");
  if (blockIdx.x == 0 && threadIdx.x < kQCounters) {
    Q.counts[threadIdx.x] = pointnav && threadIdx.x == kQGeo + kGeoClassUnknown ? P.n : 0u;
    Qother.counts[threadIdx.x] = 0u;
  }
  const Row row;
  const uint32_t it = blockIdx.x * kSnapWaves + wave, i = pointnav ? it >> 1 : it, gi = P.base + i;
  const bool ofGoal = pointnav && (wave & 1u);
  uint32_t scene = 0;
  if (it < items) {
    scene = (uint32_t)uniform_i((int)A.scene[gi]);
    if (!ofGoal) {
      const uint32_t count = (uint32_t)uniform_i((int)A.nresets[gi]);
      float ep[10];
      const uint32_t e = draw_episode(row, nav, P, gi, scene, count, ep);
      if (first) {
        store_episode(A, gi, count, e, ep);
        for (int k = 0; k < 10; ++k) pose[wave][k] = ep[k];
      }
    }
  }
  __syncthreads();
  if (it >= items) return;
  uint32_t cands = 0;
  const float* ep = pose[ofGoal ? wave - 1u : wave];
  const float* p = ofGoal ? ep + 7 : ep;
  const NavPt r = snap_point_wave(nav, nav.scenes[scene], lane_f(p[0], 0), lane_f(p[1], 0), lane_f(p[2], 0), lds[wave], &cands);
  if (!first) return;
  uint64_t* shard = counter_shard(P.counters);
  if (it == 0) atomicAdd((unsigned long long*)&shard[kCntResets], (unsigned long long)P.n);
  if (cands) atomicAdd((unsigned long long*)&shard[kCntSnapCands], (unsigned long long)cands);
  GeoQuery* q = &Q.queries[(size_t)kGeoClassUnknown * Q.stride + i];   // a new episode: no history
  if (ofGoal) {
    goal_state(A, gi, r, q);
    return;
  }
  start_state(A, P.task, gi, ep, ep + 3, ep + 7, r);
  if (pointnav) start_of_query(P, gi, scene, r, q);
  A.flags[gi] = kAgentResetOnly;
}

#ifdef BPSX_QUERY_TRACE
#include "diag_trace.h"   // diagnostic build only: per-query trace buffer
#endif
// Work of one wavefront on one query, whichever instantiation g belongs to: the search, the
// result and the agent's cost estimate.
struct GeoTotals {
  uint32_t pops = 0, corridor = 0, done = 0;
  uint32_t linkSpills = 0, heapSpills = 0, exactRuns = 0, tieReplays = 0, pairTies = 0;
  template <class Wave> BPSX_DEV void add(const Wave& g, int lane, uint64_t* counters) {
    linkSpills += g.linkSpills; heapSpills += g.heapSpills; exactRuns += g.exactRuns; tieReplays += g.tieReplays; pairTies += g.pairTies;
#ifdef BPSX_PHASE_TIMING
    if (lane == 0) for (int k = 0; k < 8; ++k) atomicAdd((unsigned long long*)&counters[8 + k], g.phase[k]);
#endif
  }
  BPSX_DEV void count(int lane, uint64_t* counters) const {
    if (lane != 0 || !done) return;
    atomicAdd((unsigned long long*)&counters[kCntGeoQueries], (unsigned long long)done);
    atomicAdd((unsigned long long*)&counters[kCntAstarPops], (unsigned long long)pops);
    atomicAdd((unsigned long long*)&counters[kCntCorridor], (unsigned long long)corridor);
    if (linkSpills) atomicAdd((unsigned long long*)&counters[kCntLinkSpills], (unsigned long long)linkSpills);
    if (heapSpills) atomicAdd((unsigned long long*)&counters[kCntHeapSpills], (unsigned long long)heapSpills);
    if (exactRuns) atomicAdd((unsigned long long*)&counters[kCntExactRuns], (unsigned long long)exactRuns);
    if (tieReplays) atomicAdd((unsigned long long*)&counters[kCntTieReplays], (unsigned long long)tieReplays);
    if (pairTies) atomicAdd((unsigned long long*)&counters[kCntPairTies], (unsigned long long)pairTies);
  }
};
template <class Wave>
BPSX_DEV void serve_query(Wave& g, const NavData& nav, const GeoQuery& q, int cls, float* out, uint32_t* last_cost, GeoTotals& T) {
  const uint32_t pops0 = T.pops;
#ifdef BPSX_QUERY_TRACE
  const unsigned long long trace_t0 = wall_clock64();
  const uint32_t trace_replays0 = g.tieReplays, trace_spills0 = g.linkSpills, trace_bridges0 = g.exactRuns;
  const unsigned long long trace_pred = (last_cost && q.cost_slot != kNoCostSlot) ? last_cost[q.cost_slot] : 0xffffu;
#endif
  // the longer the expected search, the sooner its instructions issue; a search of unknown
  // length may be among the longest, but most are not: they run just below those known to be long
  const int priority = cls == (int)kGeoClassUnknown ? 2 : (int)(((uint32_t)(kGeoClasses - 1 - cls) * kGeoClassWidth) / 400u);
  set_wave_priority(Wave::kFollowed && priority < 1 ? 1 : priority);   // above the wavefronts that keep the heaps
  const float d = geodesic_query(g, nav, q, &T.pops, &T.corridor);
  if (g.lane == 0) {
#ifdef BPSX_QUERY_TRACE
    const unsigned int ti = atomicAdd(&g_trace_n, 1u);
    if (ti < (1u << 17)) {
      g_trace[ti][0] = trace_t0; g_trace[ti][1] = wall_clock64(); g_trace[ti][2] = T.pops - pops0;
      // class, predicted length, ties resolved from the log, link spills, bridges to the exact loops
      g_trace[ti][3] = (unsigned long long)cls | ((trace_pred & 0xffffu) << 8) | ((unsigned long long)((g.tieReplays - trace_replays0) & 0xfffu) << 24) |
                        ((unsigned long long)((g.linkSpills - trace_spills0) & 0xfffu) << 36) | ((unsigned long long)((g.exactRuns - trace_bridges0) & 0xffu) << 48);
    }
#endif
    out[q.out] = d;
    // estimate for the agent's next search: this one's length, decaying from earlier peaks
    if (last_cost && q.cost_slot != kNoCostSlot) {
      const uint32_t prev = last_cost[q.cost_slot], now = T.pops - pops0;
      const uint32_t faded = prev == kCostUnknown ? 0u : prev - (prev >> 2);
      last_cost[q.cost_slot] = now > faded ? now : faded;
    }
  }
  T.done++;
  wave_sync();
}

// Blocks of two wavefronts, each wavefront persistent and serving queries from the shared
// queue on its half of the block's LDS.  The launch ends with its longest search, so the
// queries of the kLongClasses longest classes are treated apart: block b takes the b-th of
// them, if there is one, and gives it the whole block's LDS (the larger instantiation: no link
// spills, half the window misses, shorter hash chains; 7 % faster on such searches) while its
// second wavefront leaves.  Every other wavefront's first query is fixed by its index too;
// from the second query on a wavefront draws from the queue's counter.
constexpr int kLongClasses = (int)geo_class(1400);   // the classes of an expected cost of 1400 nodes and more
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(5, 5))) void k_geodesic(NavData nav, const GeoQuery* __restrict__ queries, uint32_t stride,
                                                  const uint32_t* __restrict__ counts, uint32_t* head,
                                                  float* out, uint32_t* last_cost, GeoSlot* slots, uint64_t* counters) {
  constexpr size_t kHalf = sizeof(geo::GeoShared);
  static_assert(kHalf % 16 == 0 && sizeof(geo_long::GeoShared) <= 2 * kHalf, "the long search must fit the LDS of one block");
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kHalf];
  const int lane = (int)(threadIdx.x & 63), half = uniform_i((int)(threadIdx.x >> 6));   // the same in all lanes, and known to be: addresses derived from it stay in scalar registers
  GeoSlot* slot = &slots[blockIdx.x * 2 + half];
  // Classes are served in order: class c owns the ticket numbers from the sum of the counts
  // before it.  A wavefront's tickets only go up, so it keeps the class it is in and that
  // class's range of tickets, and moves on through the counts as its tickets pass the range.
  uint32_t nq = 0, nlong = 0;
  for (int c = 0; c < kGeoClasses; ++c) {
    nq += (uint32_t)uniform_i((int)counts[c]);
    if (c + 1 == kLongClasses) nlong = nq;
  }
  // With a block for every query all of them are run that way (560 queries over room plans: 0.90 -> 0.87 ms).
  if (nq <= gridDim.x) nlong = nq;
  int curCls = 0;
  uint32_t curLo = 0, curHi = (uint32_t)uniform_i((int)counts[0]);
  auto class_of = [&](uint32_t ticket) {   // ticket < nq, not below an earlier one
    while (ticket >= curHi) {
      curCls++;
      curLo = curHi;
      curHi += (uint32_t)uniform_i((int)counts[curCls]);
    }
    return curCls;
  };
  GeoTotals T;
  counters = counter_shard(counters);
  // The first query of every wavefront needs no ticket counter: the grid is what the device
  // holds at once, so block b takes long query b if there is one, and the wavefronts of the
  // other blocks take the queries after the long ones in the order of their index.  (Some
  // thousand atomics on one counter at the start of a launch are served one after the other.)
  const uint32_t lt = blockIdx.x;
  if (lt < nlong) {
    if (half == 1) return;
    geo_long::GeoWave gl;
    gl.lane = lane;
    gl.L = &reinterpret_cast<geo_long::GeoShared*>(lds)->a;
    gl.ws = slot;
    gl.nodeCount = 0;
    gl.linkSpills = gl.heapSpills = gl.exactRuns = gl.tieReplays = gl.pairTies = 0;
#ifdef BPSX_PHASE_TIMING
    for (int k = 0; k < 8; ++k) gl.phase[k] = 0;
#endif
    const int cls = class_of(lt);
    const GeoQuery q = queries[(size_t)cls * stride + (lt - curLo)];
    serve_query(gl, nav, q, cls, out, last_cost, T);
    T.add(gl, lane, counters);
    if (lane == 0) atomicAdd((unsigned long long*)&counters[kCntLongPath], 1ull);
  }
  geo::GeoWave g;
  g.lane = lane;
  g.L = &reinterpret_cast<geo::GeoShared*>(lds + (size_t)half * kHalf)->a;
  g.ws = slot;
  g.nodeCount = 0;
  g.linkSpills = g.heapSpills = g.exactRuns = g.tieReplays = g.pairTies = 0;
#ifdef BPSX_PHASE_TIMING
  for (int k = 0; k < 8; ++k) g.phase[k] = 0;
#endif
  // tickets below `taken` went to the blocks' first wavefronts above
  const uint32_t taken = nlong < gridDim.x ? nlong : gridDim.x;
  const uint32_t nstatic = (gridDim.x - taken) * 2u;   // wavefronts that start on the general queries
  bool firstQuery = blockIdx.x >= taken;
  for (;;) {
    uint32_t qi = 0;
    if (firstQuery) {
      qi = taken + (blockIdx.x - taken) * 2u + (uint32_t)half;
      firstQuery = false;
    } else {
      if (lane == 0) qi = atomicAdd(head, 1u);
      qi = taken + nstatic + (uint32_t)uniform_i((int)qi);
    }
    if (qi >= nq) break;
    const int cls = class_of(qi);
    const GeoQuery q = queries[(size_t)cls * stride + (qi - curLo)];
    serve_query(g, nav, q, cls, out, last_cost, T);
  }
  T.add(g, lane, counters);
  T.count(lane, counters);
}

// Launches with a block for each query, or nearly so, last as long as their longest searches, chains of dependent
// steps.  A block has one search at a time, more LDS for it, and a second wavefront that keeps the
// reference's heap next to it, so that a tie costs no replay (follow).  Replays were a fifth of such launches:
// 1000 pairs over a maze 1368 -> 990 us, steps of 4096 agents over cluttered plans 1825 -> 1360.  The second
// wavefronts take issue slots from the searches, 2 to 3 % where no search ties (a reset of 2048 over mazes 471 ->
// 483).
// The last blocks of a step's launch take the snaps of the episodes that begin in it, which touch nothing
// that the searches touch: the step's last launch would last 9 us longer with them, here they end long before the
// searches do.  (Steps of 64 agents 161 -> 154 us, of 510 in two groups 1199 -> 1186, of 1024 over room plans 625 ->
// 618, of 4096 over cluttered plans 1350 -> 1320.  In k_geodesic, whose searches fill the device, they would cost
// its loop registers.)
struct SnapWork {
  AgentArrays A;
  StepQueues Q, Qnext;
  StepParams P;
  uint32_t blocks;
};
struct NoSnaps {};   // a launch without them, whose kernel is spared their code (it costs the searches 1.6 %)
template <class Wave, class Snaps>
BPSX_DEV void one_search_per_block(typename Wave::Shared* lds, const NavData& nav, const GeoQuery* __restrict__ queries, uint32_t stride,
                                   const uint32_t* __restrict__ counts, uint32_t* head, float* out, uint32_t* last_cost, GeoSlot* slots,
                                   uint64_t* counters, const Snaps& snaps) {
  const int lane = (int)(threadIdx.x & 63), half = uniform_i((int)(threadIdx.x >> 6));
  uint32_t blocks = gridDim.x;   // for searches
  if constexpr (std::is_same_v<Snaps, SnapWork>) {
    blocks -= snaps.blocks;
    if (blockIdx.x >= blocks) {
      static_assert(2 * sizeof(SnapLds) <= sizeof(*lds) && sizeof(SnapLds) % 16 == 0, "one for each wavefront");
      return snap_new_episodes(nav, snaps.A, snaps.Q, snaps.Qnext, snaps.P, (blockIdx.x - blocks) * 2u + (uint32_t)half, snaps.blocks * 2u,
                               reinterpret_cast<SnapLds*>(lds)[half]);
    }
  }
  uint32_t nq = 0;
  for (int c = 0; c < kGeoClasses; ++c) nq += (uint32_t)uniform_i((int)counts[c]);
  if (blockIdx.x >= nq) return;
  if (threadIdx.x == 0) follow_init(&lds->a);
  __syncthreads();
  if (half == 1) return follow(&lds->a, &slots[blockIdx.x], lane);
  Wave g;
  g.lane = lane;
  g.L = &lds->a;
  g.ws = &slots[blockIdx.x];
  g.nodeCount = 0;
  g.epoch = 0;
  g.linkSpills = g.heapSpills = g.exactRuns = g.tieReplays = g.pairTies = 0;
#ifdef BPSX_PHASE_TIMING
  for (int k = 0; k < 8; ++k) g.phase[k] = 0;
#endif
  int cls = 0;
  uint32_t lo = 0, hi = (uint32_t)uniform_i((int)counts[0]);
  GeoTotals T;
  counters = counter_shard(counters);
  // the first query by the block's index, further ones from the counter, the longest classes first
  for (uint32_t qi = blockIdx.x; qi < nq;) {
    while (qi >= hi) {
      cls++;
      lo = hi;
      hi += (uint32_t)uniform_i((int)counts[cls]);
    }
    const GeoQuery q = queries[(size_t)cls * stride + (qi - lo)];
    serve_query(g, nav, q, cls, out, last_cost, T);
    if (lane == 0) qi = atomicAdd(head, 1u);
    qi = blocks + (uint32_t)uniform_i((int)qi);
  }
  g.publish(kFollowQuit);
  T.add(g, lane, counters);
  T.count(lane, counters);
  if (lane == 0 && T.done) atomicAdd((unsigned long long*)&counters[kCntLongPath], (unsigned long long)T.done);
}
// Three blocks per CU.  With every node in LDS no step waits for a node that has left a window, and only the log
// is written.  (1024 agents over room plans, 560 queries: 0.87 ms with a block's 15 KB for each, 0.82 here; 510
// agents in two groups: 0.75 and 0.71 each.)
template <class Snaps>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_geodesic_few(NavData nav, const GeoQuery* __restrict__ queries, uint32_t stride,
                                                  const uint32_t* __restrict__ counts, uint32_t* head,
                                                  float* out, uint32_t* last_cost, GeoSlot* slots, uint64_t* counters, Snaps snaps) {
  __shared__ __attribute__((aligned(16))) geo_few::GeoShared lds;
  static_assert(sizeof(lds) <= 42 * 1280, "three blocks per CU");
  one_search_per_block<geo_few::GeoWave>(&lds, nav, queries, stride, counts, head, out, last_cost, slots, counters, snaps);
}
// Eight blocks per CU.  (With 1024 hash heads and a window of 128, and the parent indices in their place: a reset of
// 2048 over mazes 498 us instead of 483, 1000 pairs 987 instead of 925.)
template <class Snaps>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_geodesic_mid(NavData nav, const GeoQuery* __restrict__ queries, uint32_t stride,
                                                  const uint32_t* __restrict__ counts, uint32_t* head,
                                                  float* out, uint32_t* last_cost, GeoSlot* slots, uint64_t* counters, Snaps snaps) {
  __shared__ __attribute__((aligned(16))) geo_mid::GeoShared lds;
  static_assert(sizeof(lds) <= 16 * 1280, "eight blocks per CU");
  one_search_per_block<geo_mid::GeoWave>(&lds, nav, queries, stride, counts, head, out, last_cost, slots, counters, snaps);
}

// ---- batched PathFinder-level kernels (one lane per item, or one group per item)
__global__ __launch_bounds__(64) void k_snap_batch(NavData nav, uint32_t scene, const float* pts, uint32_t n, float* oxyz,
                                                   uint32_t* oref) {
  __shared__ SnapLds lds;
  const uint32_t i = blockIdx.x;
  if (i >= n) return;
  uint32_t c = 0;
  const NavPt r = snap_point_wave(nav, nav.scenes[scene], pts[(size_t)i * 3], pts[(size_t)i * 3 + 1], pts[(size_t)i * 3 + 2], lds, &c);
  if (threadIdx.x == 0) {
    oxyz[(size_t)i * 3] = r.x; oxyz[(size_t)i * 3 + 1] = r.y; oxyz[(size_t)i * 3 + 2] = r.z;
    oref[i] = r.ref;
  }
}
// per: points of a wavefront, up to kSnapBatch
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_snap_points(NavData nav, uint32_t scene, const float* pts,
                                                                                         uint32_t n, uint32_t per, float* oxyz, uint32_t* oref) {
  __shared__ SnapBatchLds lds;
  const uint32_t i = blockIdx.x * per + threadIdx.x;
  const bool mine = threadIdx.x < per && i < n;
  float p[3] = {0, 0, 0};
  if (mine) load3(pts, i, p);
  const NavPt r = snap_points_batch(nav, nav.scenes[scene], mine, p[0], p[1], p[2], lds);
  if (!mine) return;
  oxyz[(size_t)i * 3] = r.x; oxyz[(size_t)i * 3 + 1] = r.y; oxyz[(size_t)i * 3 + 2] = r.z;
  oref[i] = r.ref;
}
__global__ __launch_bounds__(kMoveItems * 8) void k_try_step_batch(NavData nav, uint32_t scene, const float* sxyz, const uint32_t* sref,
                                                                   const float* exyz, uint32_t n, float* oxyz, uint32_t* oref) {
  __shared__ MoveLds move_lds;
  __shared__ __attribute__((aligned(16))) uint16_t entered[kMoveItems][kTinyNodes];
  const Row row;
  const uint32_t item = threadIdx.x >> 3, i = blockIdx.x * kMoveItems + item;
  if (i >= n) return;
  uint32_t c = 0;
  NavPt st{sxyz[(size_t)i * 3], sxyz[(size_t)i * 3 + 1], sxyz[(size_t)i * 3 + 2], sref[i]};
  const NavPt r = try_step_row(row, nav, nav.scenes[scene], st, exyz[(size_t)i * 3], exyz[(size_t)i * 3 + 1], exyz[(size_t)i * 3 + 2], &c,
                               entered[item], move_lds, (int)item);
  if (row.el != 0) return;
  oxyz[(size_t)i * 3] = r.x; oxyz[(size_t)i * 3 + 1] = r.y; oxyz[(size_t)i * 3 + 2] = r.z;
  oref[i] = r.ref;
}
// and the counts and the ticket counter of a batch of n queries, all in class cls
__global__ __launch_bounds__(256) void k_make_queries(uint32_t scene, const float* sxyz, const uint32_t* sref, const float* exyz,
                               const uint32_t* eref, uint32_t n, GeoQuery* q, uint32_t* counts, uint32_t cls) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= (uint32_t)kGeoClasses) counts[i] = i == cls ? n : 0u;
  if (i >= n) return;
  GeoQuery o;
  for (int k = 0; k < 3; ++k) { o.a[k] = sxyz[(size_t)i * 3 + k]; o.b[k] = exyz[(size_t)i * 3 + k]; }
  o.a_ref = sref[i]; o.b_ref = eref[i]; o.scene = scene; o.out = i;
  o.cost_slot = kNoCostSlot; o.pad = 0;
  q[i] = o;
}
__global__ __launch_bounds__(256) void k_random_points(NavData nav, uint32_t scene, const float* u, uint32_t n, float* oxyz, uint32_t* oref) {
  const uint32_t i = blockIdx.x * 32u + (threadIdx.x >> 3);   // a row of eight lanes per point
  if (i >= n) return;
  const Row row;
  const SceneDev& s = nav.scenes[scene];
  float p[3] = {0, 0, 0};
  uint32_t ip = 0;
  const bool ok = sample_point_row(row, nav, s, u[(size_t)i * 3], u[(size_t)i * 3 + 1], u[(size_t)i * 3 + 2], p, &ip);
  if (row.el != 0) return;
  oxyz[(size_t)i * 3] = p[0]; oxyz[(size_t)i * 3 + 1] = p[1]; oxyz[(size_t)i * 3 + 2] = p[2];
  oref[i] = ok ? (s.ref_base | ip) : 0;
}

}  // namespace

// ------------------------------------------------------------------ launch wrappers
static inline dim3 grid_for(uint32_t n, uint32_t block) { return dim3((n + block - 1) / block); }

uint32_t geodesic_blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_geodesic, 128, 0) != hipSuccess || n < 1) n = 1;
  return (uint32_t)n;
}
uint32_t geodesic_few_blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_geodesic_few<SnapWork>, 128, 0) != hipSuccess || n < 1) n = 1;
  return (uint32_t)n;
}

uint32_t geodesic_mid_blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_geodesic_mid<SnapWork>, 128, 0) != hipSuccess || n < 1) n = 1;
  return (uint32_t)n;
}

// Where the number of queries to expect is no more than the blocks that k_geodesic_few keeps on the device at once
// (768) it serves them.  Up to a multiple of its own blocks (2048) k_geodesic_mid does, which has fewer searches under
// way than k_geodesic (5120), but each is shorter.  In a step the longest begin first, and it is ahead up to 9/4
// of its blocks, 6144 agents.  Of a reset's or a batch's searches nothing is known, and a long one that begins late
// costs more: up to 5/4 of them.  All in us over room plans, cluttered plans, mazes:
//   k_geodesic_few, _mid    resets of 768: 582, 622; 926, 997; 436, 454; 1024: 586, 630; 946, 1011; 499, 458
//                           pairs, 768: 312, 335; 1154, 1301; 817, 825; 1000: 326, 323; 1272, 1209; 1149, 814
//   k_geodesic_mid, k_geodesic
//                           steps of 3072: 648, 694; 1044, 1372; 527, 576; 6144: 665, 822; 1117, 1541; 555, 638;
//                           12288: 717, 877; 1687, 1730; 883, 692
//                           resets of 2048: 641, 633; 1039, 1049; 480, 468; 3072: 664, 785; 1136, 1283; 601, 572;
//                           4096: 693, 812; 1326, 1369; 686, 622
//                           pairs, 2000: 326, 312; 1362, 1874; 947, 1341; 2560: 382, 366; 1527, 1704; 1239, 1373;
//                           4000: 444, 489; 2000, 2183; 1538, 1850; 6000: 493, 465; 2525, 2678; 2067, 2107
// The line at 5/4 is not the best one everywhere: k_geodesic_mid is ahead for pairs up to 4000 at least, behind for resets
// over mazes at 2048 already (2 %) and ahead for resets over plans beyond the line.
// k_geodesic takes no snaps.
static uint32_t snap_blocks_of(const SnapWork& s) { return s.blocks; }
static uint32_t snap_blocks_of(NoSnaps) { return 0; }
template <class Snaps> static SearchKernel launch_geodesic(const NavData& nav, const GeoQuery* queries, uint32_t stride, const uint32_t* counts, uint32_t* head,
                            float* out, uint32_t* last_cost, const GeoPool& G, uint32_t expected, uint32_t mid_most,
                            uint64_t* counters, const Snaps& snaps, hipStream_t st) {
  if (expected <= G.few_blocks) {
    hipLaunchKernelGGL(k_geodesic_few<Snaps>, dim3(G.few_blocks + snap_blocks_of(snaps)), dim3(128), 0, st, nav, queries, stride, counts, head, out,
                       last_cost, G.slots, counters, snaps);
    return kSearchFew;
  }
  if (expected <= mid_most) {
    hipLaunchKernelGGL(k_geodesic_mid<Snaps>, dim3(G.mid_blocks + snap_blocks_of(snaps)), dim3(128), 0, st, nav, queries, stride, counts, head, out,
                       last_cost, G.slots, counters, snaps);
    return kSearchMid;
  }
  hipLaunchKernelGGL(k_geodesic, dim3(G.blocks), dim3(128), 0, st, nav, queries, stride, counts, head, out,
                     last_cost, G.slots, counters);
  return kSearchMany;
}

// Blocks of as few agents as leave one block for each compute unit, and as many wavefronts to begin episodes as have one for each of
// eight agents, or half as many; of 32 agents and four such wavefronts while two blocks on each compute unit hold all agents; and
// beyond that without them, since blocks that wait for a place cost more than a draw and a snap behind the moves.  Us a step
// if none of the agents ends its episode, one in 25, one in four, all; over cluttered plans with sampled episodes:
//   agents   as two launches      <1, 8>               <2, 4>               <4, 4>               <4, 0>
//       64   28  49  54   44      22  32  36   39      22  33  44   55      23  33  46   71      23  42   63   98
//     2048   30  54  73  113      24  34  37   40      24  34  46   61      24  36  52   75      24  47   70  103
//     4096   30  54  70  114      36  53  60   67      25  35  47   61      24  39  53   76      24  48   71  103
//     8192   30  55  70  117      57  82 105  122      28  38  52   71      25  40  54   79      25  49   72  106
//    16384   31  59  76  132      88 132 183  211      45  65  99  154      29  47  63   93      29  56   82  120
//    32768   42  80 122  230     160 241 339  391      67 103 157  247      47  72 110  163      32  62   91  145
// (In one form, <4, 4> with a wavefront for each draw, 64 agents 23 33 57 105, 32768 48 80 134 248.)
template <uint32_t kRowWaves, uint32_t kSnaps>
static void launch_explore_as(const NavData& nav, const AgentArrays& A, const StepParams& P, const int64_t* actions_dev, hipStream_t st) {
  hipLaunchKernelGGL((k_step_explore<kRowWaves, kSnaps>), grid_for(P.n, kRowWaves * 8), dim3((kRowWaves + kSnaps) * 64), 0, st, nav, A, P, actions_dev);
}
static void launch_explore(const NavData& nav, const AgentArrays& A, const StepParams& P, const int64_t* actions_dev, uint32_t compute_units,
                           hipStream_t st) {
  if (P.n <= 8u * compute_units) launch_explore_as<1, 8>(nav, A, P, actions_dev, st);
  else if (P.n <= 16u * compute_units) launch_explore_as<2, 4>(nav, A, P, actions_dev, st);
  else if (P.n <= 64u * compute_units) launch_explore_as<4, 4>(nav, A, P, actions_dev, st);
  else launch_explore_as<4, 0>(nav, A, P, actions_dev, st);
}

SearchKernel launch_step(const NavData& nav, const AgentArrays& A, const StepQueues& Q, const StepQueues& Qnext, const StepParams& P,
                 const int64_t* actions_dev, const GeoPool& G, uint32_t snap_blocks, hipStream_t st, hipEvent_t* ev) {
  int e = 0;
  auto mark = [&]() { if (ev) (void)hipEventRecord(ev[e++], st); };
  mark();
  if (P.task == BPSX_TASK_EXPLORATION) {
    launch_explore(nav, A, P, actions_dev, snap_blocks / 8u, st);
    for (int k = 1; k < kStepEvents; ++k) mark();
    return kSearchNone;
  }
  // Q's lists of queries were emptied two steps ago and have since taken the first queries of
  // the episodes that began in the previous step; its reset list and ticket counter, and the
  // lists of Qnext, were emptied by the previous step's last launch
  hipLaunchKernelGGL(k_step_move, grid_for(P.n, kMoveItems), dim3(kMoveItems * 8), 0, st, nav, A, Q, P, actions_dev);
  mark();
  // a grid for one agent in sixteen ending its episode; more take further rounds
  const uint32_t step_snap_blocks = std::min(snap_blocks, std::max(16u, P.n / 32u));
  // (the snaps are a launch of their own when the launches are being timed one by one)
  if (ev) hipLaunchKernelGGL(k_reset_snap, dim3(step_snap_blocks), dim3(kSnapWaves * 64), 0, st, nav, A, Q, Qnext, P);
  mark();
  // Three agents in five ask for a distance in a step; a group's queries are taken for three in four, with
  // room for one that asks more, so k_geodesic_few serves groups of up to 1024 agents.  (The line could lie
  // higher: a step over room plans, cluttered plans, mazes takes 450, 718, 414 us by k_geodesic_few and 493, 775, 433 by
  // k_geodesic_mid at 1200 agents, 472, 747, 482 and 516, 788, 507 at 2048, 479, 839, 499 and 518, 835, 471 at 3072.)
  const SearchKernel searches = launch_geodesic(nav, Q.queries, Q.stride, &Q.counts[kQGeo], &Q.counts[kQGeoHead], A.geo,
                               A.last_cost, G, P.n - P.n / 4u, G.mid_steps, P.counters,
                               SnapWork{A, Q, Qnext, P, ev ? 0u : step_snap_blocks * (kSnapWaves / 2u)}, st);
  mark();
  const bool snapped = ev || searches == kSearchFew || searches == kSearchMid;
  const uint32_t with_snaps = snapped ? 0u : step_snap_blocks;
  hipLaunchKernelGGL(k_step_finish, dim3(with_snaps + grid_for(P.n, 256).x), dim3(256), 0, st, nav, A, P, Q, Qnext, with_snaps);
  mark();
  return searches;
}

SearchKernel launch_reset(const NavData& nav, const AgentArrays& A, const StepQueues& Q, const StepQueues& Qother, const StepParams& P,
                  const GeoPool& G, uint32_t snap_blocks, hipStream_t st) {
  const uint32_t snaps = P.task == BPSX_TASK_POINTNAV ? 2u * P.n : P.n, blocks = (snaps + kSnapWaves - 1u) / kSnapWaves;
  // In one launch as long as the device holds all blocks at once, four on each compute unit (half of snap_blocks): a draw by a
  // wavefront of its own takes the place of a snap.  (Two launches, and one: 8192 exploring agents of sampled episodes 68.5 and 78 us,
  // 4096 point-goal agents of sampled episodes 789 and 793, over mazes 527 and 525.)
  if (2u * blocks <= snap_blocks) {
    hipLaunchKernelGGL(k_reset_begin, dim3(blocks), dim3(kSnapWaves * 64), 0, st, nav, A, Q, Qother, P);
  } else {
    hipLaunchKernelGGL(k_reset_all, grid_for(P.n, 32), dim3(256), 0, st, nav, A, Q, Qother, P);
    hipLaunchKernelGGL(k_reset_snap, dim3(snap_blocks), dim3(kSnapWaves * 64), 0, st, nav, A, Q, Q, P);
  }
  SearchKernel searches = kSearchNone;
  if (P.task != BPSX_TASK_EXPLORATION)
    searches = launch_geodesic(nav, Q.queries, Q.stride, &Q.counts[kQGeo], &Q.counts[kQGeoHead], A.geo,
                               A.last_cost, G, P.n, G.mid_batch, P.counters, NoSnaps{}, st);
  // and, as the next step expects them, all lists of Q empty; Qother's have been from the start
  // (by a launch of its own a reset of 2048 agents over mazes took 393.1 us, now 391.4)
  hipLaunchKernelGGL(k_step_finish, grid_for(P.n, 256), dim3(256), 0, st, nav, A, P, Q, Q, 0u);
  return searches;
}
void launch_snap_batch(const NavData& nav, uint32_t scene, const float* pts, uint32_t n, float* oxyz, uint32_t* oref,
                       uint32_t waves, hipStream_t st) {
  // With more points than wavefronts the device holds at once, each wavefront takes several, so that all of them
  // are under way from the start.  (4096 waves; 4200 points over a cluttered plan, a maze: 43, 36 us by a wavefront
  // for each, 43, 38 by two points a wavefront; 6000: 52, 44 and 44, 39; 16384: 105, 87 and 72, 51.  Up to 4096,
  // a wavefront for each is a shorter chain.)
  if (n <= waves) {
    hipLaunchKernelGGL(k_snap_batch, dim3(n), dim3(64), 0, st, nav, scene, pts, n, oxyz, oref);
    return;
  }
  const uint32_t per = std::min((uint32_t)kSnapBatch, (n - 1u) / waves + 1u);
  hipLaunchKernelGGL(k_snap_points, grid_for(n, per), dim3(64), 0, st, nav, scene, pts, n, per, oxyz, oref);
}
void launch_try_step_batch(const NavData& nav, uint32_t scene, const float* sxyz, const uint32_t* sref, const float* exyz,
                           uint32_t n, float* oxyz, uint32_t* oref, hipStream_t st) {
  hipLaunchKernelGGL(k_try_step_batch, grid_for(n, kMoveItems), dim3(kMoveItems * 8), 0, st, nav, scene, sxyz, sref, exyz, n, oxyz, oref);
}
SearchKernel launch_geodesic_batch(const NavData& nav, uint32_t scene, const float* sxyz, const uint32_t* sref, const float* exyz,
                                   const uint32_t* eref, uint32_t n, GeoQuery* qbuf, uint32_t* count_head /* [kGeoClasses + 1] */, float* out,
                                   const GeoPool& G, uint64_t* counters, hipStream_t st) {
  // one class only, that of the shortest
  static_assert(kGeoClasses < 256, "the first block writes the counts");
  hipLaunchKernelGGL(k_make_queries, grid_for(n, 256), dim3(256), 0, st, scene, sxyz, sref, exyz, eref, n, qbuf, count_head, (uint32_t)kGeoClasses - 1u);
  // stride 0 puts the class's queries at the start of the buffer
  return launch_geodesic(nav, qbuf, 0, &count_head[0], &count_head[kGeoClasses], out, nullptr, G, n,
                         G.mid_batch, counters, NoSnaps{}, st);
}
void launch_set_swap(uint32_t* swap_target, uint32_t* swap_remaining, uint32_t slot, uint32_t target, uint32_t envs,
                     hipStream_t st) {
  hipLaunchKernelGGL(k_set_swap, dim3(1), dim3(64), 0, st, swap_target, swap_remaining, slot, target, envs);
}
void launch_random_points(const NavData& nav, uint32_t scene, const float* u, uint32_t n, float* oxyz, uint32_t* oref,
                          hipStream_t st) {
  hipLaunchKernelGGL(k_random_points, grid_for(n, 32), dim3(256), 0, st, nav, scene, u, n, oxyz, oref);
}

#ifdef BPSX_QUERY_TRACE
#define BPSX_DIAG_TRACE_HOST
#include "diag_trace.h"
#endif
}  // namespace bpsx
