// Launch interface between the engine (host) and the kernels.
#pragma once
#include <hip/hip_runtime.h>

#include "device_types.h"

namespace bpsx {

// Node pools of the path searches and the launches they allow: one pool per wavefront.
struct GeoPool {
  GeoSlot* slots;
  uint32_t blocks;       // blocks of two wavefronts of k_geodesic
  uint32_t few_blocks;   // blocks of k_geodesic_few, one pool each; 0: never
  uint32_t mid_blocks;   // blocks of k_geodesic_mid, one pool each
  uint32_t mid_steps, mid_batch;   // most queries that it serves, in order of their expected cost and without such an order
};

// The kernels that serve path searches; kSearchNone: no launch of them.
enum SearchKernel { kSearchFew, kSearchMid, kSearchMany, kSearchNone };

enum QueueCounter { kQGeo = 0 /* one per cost class */, kQGeoHead = kGeoClasses, kQReset, kQCounters };

// Work queues of one step, all in HBM, sized for every agent of a group.
struct StepQueues {
  uint32_t* counts;          // [kQCounters], see QueueCounter
  GeoQuery* queries;         // [kGeoClasses][stride]: one per moved/finished agent plus one per reset
  uint32_t stride;           // 2n
  uint32_t* reset_list;      // [n] agent indices being reset
};

struct StepParams {
  uint32_t n;          // agents in the group
  uint32_t base;       // index of the group's first agent
  uint32_t total;      // agents in the simulator (reset results live at geo[total + i])
  float max_steps;
  uint32_t reset_mode;
  uint32_t task;       // BPSX_TASK_*
  uint32_t info_width; // floats per agent in the infos output
  uint64_t seed;
  float turn_left[4], turn_right[4];  // glm::angleAxis(+-radians(10), up), x,y,z,w
  uint32_t* error_flag;
  uint64_t* counters;
  // scene rotation: per scene slot the scene-table entry its envs move to when their episode
  // ends (kNoSwap: none) and how many envs have yet to move
  uint32_t num_slots;
  const uint32_t* swap_target;
  uint32_t* swap_remaining;
  // 1: the first distance of an episode that begins in this step is measured in the next step's
  // launch (see launch_step); 0: in this one
  uint32_t defer_first_distance;
  // what the launch's last block tells a waiting host (tell_host): done_value at done_flag, in pinned memory, null if nobody waits;
  // done_blocks counts the blocks that have ended, and is 0 between launches
  uint32_t* done_flag;
  uint32_t* done_blocks;
  uint32_t done_value;
};
constexpr uint32_t kNoSwap = 0xffffffffu;

constexpr int kStepEvents = 5;  // timestamps recorded by launch_step when asked to

// One step of a group.  Q holds the step's queries, among them the first queries of the episodes
// that began in the previous step; the episodes that begin in this one are snapped in its last
// launch, and their first queries go to Qnext, the next step's queues.  snap_blocks: most blocks for
// the snaps.  These return what the searches went to.
SearchKernel launch_step(const NavData& nav, const AgentArrays& A, const StepQueues& Q, const StepQueues& Qnext, const StepParams& P,
                 const int64_t* actions_dev, const GeoPool& G, uint32_t snap_blocks, hipStream_t st, hipEvent_t* ev);
// Reset of a whole group, all on st; Qother (the group's other set of queues) is emptied.
SearchKernel launch_reset(const NavData& nav, const AgentArrays& A, const StepQueues& Q, const StepQueues& Qother, const StepParams& P,
                  const GeoPool& G, uint32_t snap_blocks, hipStream_t st);
void launch_snap_batch(const NavData& nav, uint32_t scene, const float* pts, uint32_t n, float* oxyz, uint32_t* oref,
                       uint32_t waves, hipStream_t st);
void launch_try_step_batch(const NavData& nav, uint32_t scene, const float* sxyz, const uint32_t* sref, const float* exyz,
                           uint32_t n, float* oxyz, uint32_t* oref, hipStream_t st);
SearchKernel launch_geodesic_batch(const NavData& nav, uint32_t scene, const float* sxyz, const uint32_t* sref, const float* exyz,
                                   const uint32_t* eref, uint32_t n, GeoQuery* qbuf, uint32_t* count_head /* [kGeoClasses + 1] */,
                                   float* out, const GeoPool& G, uint64_t* counters, hipStream_t st);
void launch_random_points(const NavData& nav, uint32_t scene, const float* u, uint32_t n, float* oxyz, uint32_t* oref,
                          hipStream_t st);

void launch_set_swap(uint32_t* swap_target, uint32_t* swap_remaining, uint32_t slot, uint32_t target, uint32_t envs,
                     hipStream_t st);

// Blocks of the A* kernels that one compute unit holds at once (bounded by their LDS).
uint32_t geodesic_blocks_per_cu();
uint32_t geodesic_few_blocks_per_cu();
uint32_t geodesic_mid_blocks_per_cu();

}  // namespace bpsx
