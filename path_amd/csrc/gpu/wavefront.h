// Wavefront ("Streaming") integrator: parameter block and launchers.
#pragma once

#include "kernels.h"

namespace pt {
namespace gpu {

// Counter words of one pipeline (device memory, zero at a render's start).
enum WfCounter : uint32_t {
  kExtTotal = 0,      // 64-bit: extension rays queued so far (words 0, 1)
  kShadowTotal = 2,   // 64-bit: shadow rays queued so far (words 2, 3)
  kBusyIters = 4,     // iterations that queued at least one ray
  kIterations = 5,    // iterations traced
  kNumCounters = 8,
};

// What the host learns of an iteration, in pinned memory: the traversal
// launch writes it when it starts, so the next iteration is enqueued while it
// runs.
struct WfReport {
  uint32_t ext, shadow; // rays queued
  uint32_t samples_left; // 0: every sample of this pipeline has been started
  uint32_t iteration;   // number of the iteration, from 1: written last
};

// Queue groups. Shade block b belongs to group b % n_groups (n_groups =
// min(kQueueGroups, shade blocks)): it appends its rays to the group's queue
// segment and starts new samples from the group's share of the sample range
// (shares proportional to the group's blocks). Each group's counters sit in
// their own 4 KB: device-scope atomics on one address serialise (about 12 ns
// each measured on MI355X, i.e. ~200 us per shade step for one counter hit by
// all 16k blocks), so one counter per group spreads them over 16 addresses.
constexpr uint32_t kQueueGroups = 16;
constexpr uint32_t kGroupStride = 1024; // uint32 words between group counters
// Odd and even iterations count in sets of their own: while one set is read by
// its traversal launch, that launch zeroes the other for the next shade step.
enum GroupCounter : uint32_t {
  kGroupExt = 0,    // entries in the group's extension-ray segment (set 0; set 1: + 2)
  kGroupShadow = 1, // entries in the group's shadow-ray segment (set 0; set 1: + 2)
  kGroupSample = 4, // 64-bit: samples the group has started
  kGroupKinds = 5,
};
constexpr size_t kGroupCounterWords = size_t(kGroupKinds) * kQueueGroups * kGroupStride;

__host__ __device__ inline uint32_t *group_counter(uint32_t *base, uint32_t kind,
                                                   uint32_t g) {
  return base + (size_t(kind) * kQueueGroups + g) * kGroupStride;
}

// Three packed floats (12 bytes: one dwordx3 access per lane).
struct F3 {
  float x, y, z;
};

// Per-slot path state, structure of arrays (one 16- or 12-byte record per
// slot and array, so a wave's accesses are contiguous).
struct WfState {
  uint4 *meta;       // location, sample, rng counter, flags
  float4 *mult;      // ray multiplier xyz, light target distance
  F3 *light;         // light-sample multiplier
  F3 *total;         // accumulated radiance
  F3 *origin;        // origin of the pending rays (last vertex / camera)
  F3 *dir;           // direction of the pending continuation ray
  float4 *light_dir; // direction of the pending light ray, target distance
  uint2 *hit_ext;    // packed closest hit of the continuation ray
  uint2 *hit_light;  // packed closest hit of the light ray
  uint32_t *scene;   // scene of the slot (batched renders only)
};

// Ray queues hold slot indices; the rays themselves are read from the state.
// Group g's entries start at g * group_cap; the traversal kernels read the
// group counts and concatenate the segments.
struct WfQueues {
  uint32_t *ext;
  uint32_t *shadow;
  uint32_t group_cap;
};

// One scene of a batched render. Offsets index the concatenated arrays of all
// scenes (nodes in GpuNode units, triangles in GpuTri units, etc.).
struct SceneDesc {
  uint32_t node_off, tri_off, shade_off, mat_off;
  uint32_t light_off, n_lights, x_dim, y_dim;
  uint32_t pixel_off, has_nodes, pad0, pad1;
  float film_to_world[12];
};

// What a wavefront render's samples are.
enum WfKind : int {
  kWfImage, // pixels of one scene's image
  kWfBatch, // pixels of many scenes' images (WfBatch)
  kWfRays,  // given rays of many scenes (WfBatch: scene i has x_dim rays)
};

struct WfBatch {
  const SceneDesc *scenes;
  const unsigned long long *sample_begin; // n_scenes + 1 prefix of pixels*spp
  uint32_t n_scenes;
  const float4 *nodes, *tris;             // concatenated BVHs
  const ShadeTri<float> *shade;
  const Material<float> *materials;
  const TriGeom<float> *light_tris;
  const float *light_cdf;
  // kWfRays: 6 floats per ray; triangle each ray hits first at distance 1
  // (InitialIdxAndDir), or null; per-step outputs (0: one value per sample)
  const float *rays;
  const uint32_t *initial_idx;
  uint32_t n_steps;
};

struct WfParams {
  DeviceScene scene; // single-scene renders
  WfBatch batch;     // batched renders
  IntegratorSettings settings;
  RngParams rng;
  float film_to_world[12];
  uint32_t x_dim, y_dim;
  unsigned long long total_samples;
  uint32_t n_slots;
  WfState st;
  WfQueues q;
  uint32_t *counters;       // WfCounter words
  WfReport *report;         // pinned host memory
  uint32_t set;             // set of queue counters of this iteration: 0 / 1
  uint32_t fresh;           // first iteration: every slot is empty, whatever it holds
  uint32_t *group_counters; // GroupCounter words per group (group_counter())
  uint32_t n_groups;        // min(kQueueGroups, shade blocks)
  uint32_t n_shade_blocks;
  // Samples are dealt over the groups of every pipeline of a render (the
  // path pool can be split into independent pipelines on separate streams):
  // this launch's group g is group group_base + g of n_groups_total.
  uint32_t group_base, n_groups_total;
  // [pixel * spp + sample] * 3; with n_steps one such array per step, zero
  // where a path ends before the step
  float *out_samples;
  float *gbuffer; // first hit of sample 0 per pixel: position, normal,
                  // albedo, emission (12 floats) or null
  int *stack_overflow;                // traversal stack spill area
  uint32_t overflow_stride;           // threads of a traversal launch
};

hipError_t launch_wf_shade(const WfParams &p, WfKind kind, hipStream_t s);
// Closest hits of the iteration's extension rays and occlusion of its shadow
// rays, both queues in one launch; also adds the iteration's queue counts to
// the totals, reports them to the host and zeroes the other set of counters.
hipError_t launch_wf_trace(const WfParams &p, WfKind kind, uint32_t grid_blocks,
                           hipStream_t s);
// Takes the paths of the iteration's queues to their ends, each lane tracing
// its own rays, instead of launch_wf_trace: for an iteration after which few
// paths and no samples are left.
constexpr uint32_t kFinishBlockPaths = 64; // queue entries per block and round
hipError_t launch_wf_finish(const WfParams &p, WfKind kind, uint32_t grid_blocks,
                            hipStream_t s);
// Per-pixel sum of the per-sample radiance in the mega-kernel's order
// (sequential per thread range, then the lane tree), divided by spp.
hipError_t launch_wf_reduce(const float *samples, const WorkDivision &wd,
                            uint32_t samples_per, float *out_rgb,
                            hipStream_t s);
// The same for many images whose samples and pixels are concatenated, one
// launch: each item has a work division of one sample block, all of block_size.
struct WfReduceItem {
  WorkDivision wd;
  uint32_t block_begin; // first block of the item's total_num_blocks()
  uint32_t pixel_off;
};
hipError_t launch_wf_reduce_batch(const float *samples, const WfReduceItem *items, uint32_t n,
                                  uint32_t block_size, uint32_t total_blocks,
                                  uint32_t samples_per, float *out_rgb, hipStream_t s);
// out[pixel] = (sum over the pixel's samples, sequential in FP64) / spp
hipError_t launch_sum_samples_f64(const float *samples, uint32_t n_pixels,
                                  uint32_t samples_per, double *out, hipStream_t s);

} // namespace gpu
} // namespace pt
