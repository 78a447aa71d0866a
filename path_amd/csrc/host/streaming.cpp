// Host loop of the wavefront integrator: shade -> trace (extension, shadow)
// until every sample has finished, then the per-pixel reduction.
#include "renderer.h"
#include "settings.h"

#include "../gpu/trace.h"
#include "../gpu/wavefront.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <string>
#include <system_error>
#include <thread>

using namespace pt;
using namespace pt::host;

#define HIP_TRY(expr)                                                          \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess)                                                      \
      return set_error(PT_ERR_HIP, std::string(#expr) + ": " +                 \
                                       hipGetErrorString(e_));                 \
  } while (0)

namespace pt {
namespace host {

// Paths that make a pipeline of their own worth its host thread, stream and
// launches: 16,384 samples of a 20,516-triangle scene 1,193 -> 799 us and of
// the 36-triangle box 452 -> 265 with one pipeline, 1.0 M samples of a
// 5,156-triangle scene 1,152 with three and 1,657 with one (2^16 / 2^18 / 2^19
// paths per pipeline, 0.25 M samples of that scene: 1,769 / 1,808 / 1,808).
constexpr uint32_t kMinPipeSlots = 1u << 18;

// Rays queued by an iteration after which the remaining paths are finished by
// one launch (k_wf_finish). 988,317 samples of the 36-triangle box with
// roulette (28 iterations), never / 2,048 / 8,192 / 32,768 / 131,072 rays: 1,197 /
// 1,051 / 999 / 928 / 959 us; 82k triangles, 16.8 M samples: no difference. The
// limit keeps a small render's first vertices (16,384 paths, 20,516 triangles:
// 771 us, 895 when finished from there) in the shared queues.
constexpr uint32_t kFinishRays = 12288;

// Counters of the first n pipelines: every pipeline's WfCounter words (padded
// to a group counter's 4 KB), then the group counters, in one buffer that one
// fill clears.
static size_t counter_words(int n) {
  static_assert(kMaxPipes * gpu::kNumCounters <= gpu::kGroupStride);
  return gpu::kGroupStride + size_t(n) * gpu::kGroupCounterWords;
}

// Pipelines of a pool of n_slots paths: a given number is kept to one shade
// block each.
static uint32_t pipelines(const pt_renderer &r, uint32_t n_slots) {
  const uint32_t n = r.n_pipes ? std::min(r.n_pipes, n_slots / 256)
                               : std::min(3u, n_slots / kMinPipeSlots);
  return std::max(1u, std::min(n, uint32_t(kMaxPipes)));
}

int HandOver::does_not_fit(pt_renderer &r) {
  (void)hipGetLastError();
  no_memory = true;
  r.ray_samples.release();
  r.wf_meta.release();
  r.wf_hit_ext.release();
  r.wf_hit_light.release();
  r.wf_mult.release();
  r.wf_light_dir.release();
  r.wf_light.release();
  r.wf_total.release();
  r.wf_origin.release();
  r.wf_dir.release();
  r.wf_q_ext.release();
  r.wf_q_shadow.release();
  r.wf_stack_overflow.release();
  r.wf_counters.release();
  r.wf_scene.release();
  return PT_OK;
}

void HandOver::trim(pt_renderer &r) {
  if (r.ray_samples.count * sizeof(float) > kKept)
    r.ray_samples.release();
}

uint64_t hand_over_paths(const pt_renderer &r, uint64_t samples, bool batched,
                         uint32_t max_blocks) {
  uint64_t paths = std::min<uint64_t>(samples, 1u << 22);
  if (max_blocks == 0)
    return paths;
  if (max_blocks < uint32_t(r.n_cus) * r.trace_blocks_for(batched))
    return 0; // (the traversal's grid, whatever the pool)
  // 256 paths per shade block; a smaller pool may have fewer pipelines
  for (;;) {
    const uint64_t most = uint64_t(max_blocks) * 256 * pipelines(r, uint32_t(paths));
    if (paths <= most)
      return paths;
    paths = most;
  }
}

int wavefront_alloc(pt_renderer &r, WfPipes &w, const gpu::WfParams &base,
                    uint32_t n_slots, uint64_t total_samples, gpu::WfKind kind,
                    uint32_t trace_blocks) {
  HIP_TRY(r.wf_meta.ensure(n_slots));
  HIP_TRY(r.wf_hit_ext.ensure(n_slots));
  HIP_TRY(r.wf_hit_light.ensure(n_slots));
  HIP_TRY(r.wf_mult.ensure(n_slots));
  HIP_TRY(r.wf_light.ensure(n_slots));
  HIP_TRY(r.wf_total.ensure(n_slots));
  HIP_TRY(r.wf_origin.ensure(n_slots));
  HIP_TRY(r.wf_dir.ensure(n_slots));
  HIP_TRY(r.wf_light_dir.ensure(n_slots));
  const bool batched = kind != gpu::kWfImage;
  if (batched)
    HIP_TRY(r.wf_scene.ensure(n_slots));
  if (!base.out_samples)
    HIP_TRY(r.wf_samples.ensure(size_t(total_samples) * 3));
  // Pipelines have an equal share of the slots each, their own stream, queues
  // and counters: the memory-bound shade step of one overlaps the ALU-bound
  // traversal of another.
  w.n = int(pipelines(r, n_slots));
  uint32_t first[kMaxPipes + 1] = {0};
  for (int h = 0; h < w.n; ++h) {
    const uint32_t left = n_slots - first[h], pipes_left = uint32_t(w.n - h);
    uint32_t take = (left + pipes_left - 1) / pipes_left;
    take = std::min(left, (take + 255) / 256 * 256);
    first[h + 1] = first[h] + take;
  }
  uint32_t groups[kMaxPipes], caps[kMaxPipes], groups_total = 0;
  size_t queue_total = 0;
  for (int h = 0; h < w.n; ++h) {
    const uint32_t blocks = (first[h + 1] - first[h] + 255) / 256;
    groups[h] = std::min(gpu::kQueueGroups, blocks);
    caps[h] = (blocks + groups[h] - 1) / groups[h] * 256;
    groups_total += groups[h];
    queue_total += size_t(caps[h]) * groups[h];
  }
  HIP_TRY(r.wf_q_ext.ensure(queue_total));
  HIP_TRY(r.wf_q_shadow.ensure(queue_total));
  HIP_TRY(r.wf_counters.ensure(counter_words(kMaxPipes)));
  const uint32_t trace_threads = trace_blocks * 256;
  HIP_TRY(r.wf_stack_overflow.ensure(size_t(kMaxPipes) * gpu::kOverflowDepth * trace_threads));
  size_t queue_off = 0;
  uint32_t group_base = 0;
  for (int h = 0; h < w.n; ++h) {
    gpu::WfParams &p = w.p[h];
    const uint32_t f = first[h];
    p = base;
    p.total_samples = total_samples;
    p.n_slots = first[h + 1] - f;
    p.st = {r.wf_meta.ptr + f,      r.wf_mult.ptr + f,    r.wf_light.ptr + f,
            r.wf_total.ptr + f,     r.wf_origin.ptr + f,  r.wf_dir.ptr + f,
            r.wf_light_dir.ptr + f, r.wf_hit_ext.ptr + f, r.wf_hit_light.ptr + f,
            batched ? r.wf_scene.ptr + f : nullptr};
    p.q = {r.wf_q_ext.ptr + queue_off, r.wf_q_shadow.ptr + queue_off, caps[h]};
    queue_off += size_t(caps[h]) * groups[h];
    p.counters = r.wf_counters.ptr + size_t(h) * gpu::kNumCounters;
    p.group_counters = r.wf_counters.ptr + counter_words(0) + size_t(h) * gpu::kGroupCounterWords;
    p.n_groups = groups[h];
    p.n_shade_blocks = (p.n_slots + 255) / 256;
    p.group_base = group_base;
    p.n_groups_total = groups_total;
    group_base += groups[h];
    if (!base.out_samples)
      p.out_samples = r.wf_samples.ptr;
    p.stack_overflow = r.wf_stack_overflow.ptr + size_t(h) * gpu::kOverflowDepth * trace_threads;
    p.overflow_stride = trace_threads;
  }
  return PT_OK;
}

// Enqueue iteration number `iter` (from 0) of one pipeline: shade, then trace
// the extension and shadow rays (one launch, which also reports the queues'
// sizes to the host), or, with finish_blocks, take its paths to their ends.
static hipError_t enqueue_iteration(pt_renderer &r, gpu::WfParams &p, int pipe, uint64_t iter,
                                    gpu::WfKind kind, uint32_t trace_blocks, bool graph,
                                    bool profile_events, uint32_t finish_blocks = 0) {
  hipStream_t s = r.pipe_stream(pipe);
  hipEvent_t *ev = r.ev_prof[pipe];
  hipError_t e;
  p.set = uint32_t(iter & 1);
  p.fresh = iter == 0 && !graph;
  if ((e = gpu::launch_wf_shade(p, kind, s)) != hipSuccess)
    return e;
  if (profile_events && (e = hipEventRecord(ev[0], s)) != hipSuccess)
    return e;
  e = finish_blocks ? gpu::launch_wf_finish(p, kind, finish_blocks, s)
                    : gpu::launch_wf_trace(p, kind, trace_blocks, s);
  if (e != hipSuccess)
    return e;
  if (profile_events && (e = hipEventRecord(ev[1], s)) != hipSuccess)
    return e;
  return hipSuccess;
}

// Wait until the pipeline has reported iteration `iteration` (numbered from
// 1): its traversal has started. The stream is asked now and then, so that a
// failed launch ends the wait. The cores may be wanted (a program's scene
// generation): after the first moments the thread yields, and where an iteration
// takes long it sleeps, since the traversal that reports then runs on for longer
// than a sleep. (From 0.1 ms on, a batch of 1.15 M ray samples and three steps took
// 1,690 us, and 1,600 from 0.25 ms on, as without sleeps. Cores busy during 64
// generated scenes at 128 samples: 3.1 without, 1.1 with.)
static hipError_t wait_report(const volatile gpu::WfReport *rep, uint32_t iteration,
                              hipStream_t s) {
  auto there = [&] {
    return int32_t(__atomic_load_n(&rep->iteration, __ATOMIC_ACQUIRE) - iteration) >= 0;
  };
  using clock = std::chrono::steady_clock;
  const clock::time_point sleep_from = clock::now() + std::chrono::microseconds(250);
  bool sleeping = false;
  for (uint32_t turn = 1; !there(); ++turn) {
    if (sleeping) {
      std::this_thread::sleep_for(std::chrono::microseconds(50));
    } else if (turn % 64 != 0) {
      __builtin_ia32_pause();
    } else {
      std::this_thread::yield();
      sleeping = clock::now() >= sleep_from;
    }
    if (turn % (sleeping ? 16 : 8192) != 0)
      continue;
    const hipError_t e = hipStreamQuery(s);
    if (e == hipErrorNotReady)
      continue;
    if (e != hipSuccess)
      return e;
    return there() ? hipSuccess : hipErrorUnknown; // drained: it has been written, or never will
  }
  return hipSuccess;
}

int wavefront_run(pt_renderer &r, WfPipes &w, gpu::WfKind kind, uint32_t trace_blocks,
                  uint32_t iters_per_sync) {
  hipStream_t s0 = r.stream;
  const bool prof = r.profiling;
  const bool use_graph = r.use_graphs && !prof;
  HIP_TRY(hipMemsetAsync(r.wf_counters.ptr, 0, sizeof(uint32_t) * counter_words(w.n), s0));
  if (use_graph) // its iterations are all alike, so empty slots have to say so
    for (int h = 0; h < w.n; ++h)
      HIP_TRY(hipMemsetAsync(w.p[h].st.meta, 0, size_t(w.p[h].n_slots) * sizeof(uint4), s0));
  if (!r.wf_reports)
    HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&r.wf_reports),
                          sizeof(gpu::WfReport) * kMaxPipes, hipHostMallocDefault));
  for (int h = 0; h < w.n; ++h) {
    r.wf_reports[h] = gpu::WfReport{};
    w.p[h].report = r.wf_reports + h;
  }
  // the other pipelines start after everything enqueued so far on stream 0
  // (scene upload, state clears)
  HIP_TRY(hipEventRecord(r.ev_fork, s0));
  for (int h = 1; h < w.n; ++h)
    HIP_TRY(hipStreamWaitEvent(r.pipe_stream(h), r.ev_fork, 0));
  if (iters_per_sync == 0)
    iters_per_sync = 1;
  // Profiling needs per-iteration event reads, so it syncs every iteration.
  if (prof)
    iters_per_sync = 1;
  // a graph holds whole pairs of iterations (the two sets of queue counters)
  if (use_graph)
    iters_per_sync += iters_per_sync & 1u;
  // Each pipeline runs its own host loop (pipelines 1.. on host threads of
  // their own), so the pipelines drift apart and one's shade step overlaps
  // another's traversal instead of running in lockstep.
  struct PipeResult {
    hipError_t err = hipSuccess;
    std::string what;
    uint64_t launches = 0;
    double trace_ms = 0.0;
  };
  PipeResult res[kMaxPipes];
  auto run_pipe = [&](int h) {
    PipeResult &out = res[h];
    hipStream_t s = r.pipe_stream(h);
    if ((out.err = hipSetDevice(r.device)) != hipSuccess) {
      out.what = "hipSetDevice";
      return;
    }
    hipGraphExec_t exec = nullptr;
    if (use_graph) {
      hipGraph_t graph = nullptr;
      hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
      for (uint32_t k = 0; k < iters_per_sync && e == hipSuccess; ++k)
        e = enqueue_iteration(r, w.p[h], h, k, kind, trace_blocks, true, false);
      hipError_t e2 = hipStreamEndCapture(s, &graph);
      if (e == hipSuccess && e2 == hipSuccess)
        e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      if (graph)
        (void)hipGraphDestroy(graph);
      if (e != hipSuccess || e2 != hipSuccess) {
        out.err = e != hipSuccess ? e : e2;
        out.what = "graph capture";
        if (exec)
          (void)hipGraphExecDestroy(exec);
        return;
      }
    }
    for (;;) {
      if (use_graph) {
        out.err = hipGraphLaunch(exec, s);
        out.launches += iters_per_sync;
      } else {
        for (uint32_t k = 0; k < iters_per_sync && out.err == hipSuccess; ++k) {
          out.err = enqueue_iteration(r, w.p[h], h, out.launches, kind, trace_blocks, false,
                                      prof);
          out.launches += 1;
        }
      }
      // The sizes of the last iteration's queues, as its traversal starts: the
      // next iteration is enqueued while it runs. (Profiling reads that
      // traversal's events, so it waits for its end.)
      const volatile gpu::WfReport *rep = r.wf_reports + h;
      if (out.err == hipSuccess)
        out.err = prof ? hipStreamSynchronize(s)
                       : wait_report(rep, uint32_t(out.launches), s);
      if (out.err != hipSuccess) {
        (void)hipStreamSynchronize(s); // nothing of this render is left running
        out.what = "launch / sync";
        break;
      }
      const uint32_t ne = rep->ext, ns = rep->shadow;
      if (prof && ne + ns) {
        float a = 0.f;
        (void)hipEventElapsedTime(&a, r.ev_prof[h][0], r.ev_prof[h][1]);
        out.trace_ms += a;
      }
      // a slot holds a path iff it queued at least one ray
      if (ne + ns == 0)
        break;
      // Few paths are left and no sample is waiting for a slot: one launch
      // takes them to their ends. A path has at most two queue entries.
      if (!use_graph && !prof && rep->samples_left == 0 && ne + ns <= kFinishRays) {
        const uint32_t entries = 2 * (ne + ns);
        const uint32_t blocks =
            std::min(trace_blocks, (entries + gpu::kFinishBlockPaths - 1) / gpu::kFinishBlockPaths);
        out.err = enqueue_iteration(r, w.p[h], h, out.launches, kind, trace_blocks, false,
                                    false, blocks);
        out.launches += 1;
        if (out.err != hipSuccess)
          out.what = "launch";
        break;
      }
    }
    // the last iteration's launches (they found empty queues) and the graph's
    // last use
    if (out.err == hipSuccess && (out.err = hipStreamSynchronize(s)) != hipSuccess)
      out.what = "sync";
    if (exec)
      (void)hipGraphExecDestroy(exec);
  };
  {
    // A pipeline whose thread cannot be started runs on this thread after
    // pipeline 0 (the pipelines are independent, only slower that way).
    std::thread others[kMaxPipes - 1];
    int started = 1;
    try {
      for (; started < w.n; ++started)
        others[started - 1] = std::thread(run_pipe, started);
    } catch (const std::system_error &) {
    }
    run_pipe(0);
    for (int h = started; h < w.n; ++h)
      run_pipe(h);
    for (int h = 1; h < started; ++h)
      others[h - 1].join();
  }
  uint64_t launches = 0;
  for (int h = 0; h < w.n; ++h) {
    if (res[h].err != hipSuccess)
      return set_error(PT_ERR_HIP, "wavefront pipeline " + std::to_string(h) + " " +
                                       res[h].what + ": " + hipGetErrorString(res[h].err));
    launches += res[h].launches;
    r.stats.trace_ms += res[h].trace_ms;
  }
  // every pipeline's last iteration queued nothing, so the totals are complete
  uint32_t c[kMaxPipes * gpu::kNumCounters];
  HIP_TRY(hipMemcpyAsync(c, r.wf_counters.ptr, sizeof(uint32_t) * w.n * gpu::kNumCounters,
                         hipMemcpyDeviceToHost, s0));
  HIP_TRY(hipStreamSynchronize(s0));
  uint64_t ext = 0, shadow = 0;
  uint32_t busy_iters = 0;
  for (int h = 0; h < w.n; ++h) {
    const uint32_t *ch = c + size_t(h) * gpu::kNumCounters;
    ext += uint64_t(ch[gpu::kExtTotal]) | (uint64_t(ch[gpu::kExtTotal + 1]) << 32);
    shadow += uint64_t(ch[gpu::kShadowTotal]) | (uint64_t(ch[gpu::kShadowTotal + 1]) << 32);
    busy_iters += ch[gpu::kBusyIters];
  }
  r.stats.ext_rays = ext;
  r.stats.shadow_rays = shadow;
  // traversal launches over all pipelines (each traces both queues)
  r.stats.busy_trace_launches = busy_iters;
  r.stats.trace_launches = launches;
  r.stats.pipelines = uint32_t(w.n);
  return PT_OK;
}

int render_streaming(pt_renderer &r, const pt_sample_spec &spec,
                     const gpu::DeviceScene &scene, uint32_t samples_per,
                     const pt_settings &settings, const gpu::RngParams &rng,
                     uint32_t x_dim, uint32_t y_dim, const float **final_rgb,
                     uint64_t *rays_out, HandOver *hand_over) {
  if (spec.type != PT_SAMPLE_SQUARE_IMAGE)
    return set_error(PT_ERR_UNSUPPORTED,
                     "the Streaming integrator takes SquareImage sample specs");
  WorkDivision wd;
  if (!WorkDivision::make(work_division_settings(settings.render_work_division),
                          samples_per, x_dim, y_dim, &wd) ||
      wd.block_size > 1024)
    return set_error(PT_ERR_INVALID, "invalid render work division settings");
  const uint64_t n_pixels = uint64_t(x_dim) * y_dim;
  const uint64_t total = n_pixels * samples_per;
  uint64_t slots64 = hand_over ? hand_over->max_paths : settings.max_num_samples_per_launch;
  if (slots64 == 0)
    return set_error(PT_ERR_INVALID, "max_num_samples_per_launch must be positive");
  if (slots64 > total)
    slots64 = total;
  const uint32_t trace_blocks = uint32_t(r.n_cus) * r.trace_blocks_for(false);
  gpu::WfParams p{};
  p.scene = scene;
  p.settings = integrator_settings(settings);
  p.rng = rng;
  std::memcpy(p.film_to_world, spec.film_to_world, sizeof(p.film_to_world));
  p.x_dim = x_dim;
  p.y_dim = y_dim;
  if (hand_over) {
    if (r.ray_samples.ensure(size_t(total) * 3) != hipSuccess)
      return hand_over->does_not_fit(r);
    p.out_samples = r.ray_samples.ptr;
  }
  WfPipes w;
  int rc = wavefront_alloc(r, w, p, uint32_t(slots64), total, gpu::kWfImage, trace_blocks);
  if (rc != PT_OK)
    return hand_over ? hand_over->does_not_fit(r) : rc;
  hipError_t e = r.rgb.ensure(size_t(wd.num_sample_blocks) * n_pixels * 3);
  if (e == hipSuccess && wd.num_sample_blocks != 1)
    e = r.rgb2.ensure(size_t(n_pixels) * 3);
  if (e != hipSuccess && hand_over)
    return hand_over->does_not_fit(r);
  HIP_TRY(e);
  rc = wavefront_run(r, w, gpu::kWfImage, trace_blocks, r.iters_per_sync);
  if (rc != PT_OK)
    return rc;
  hipStream_t s = r.stream;
  HIP_TRY(gpu::launch_wf_reduce(w.p[0].out_samples, wd, samples_per, r.rgb.ptr, s));
  const float *out = r.rgb.ptr;
  if (wd.num_sample_blocks != 1) {
    HIP_TRY(gpu::launch_reduce_sample_blocks(r.rgb.ptr, wd.num_sample_blocks,
                                             uint32_t(n_pixels), samples_per,
                                             r.rgb2.ptr, s));
    out = r.rgb2.ptr;
  }
  *final_rgb = out;
  *rays_out = r.stats.ext_rays + r.stats.shadow_rays;
  if (!hand_over) {
    r.last_wf_x = x_dim;
    r.last_wf_y = y_dim;
    r.last_wf_spp = samples_per;
  }
  return PT_OK;
}

} // namespace host
} // namespace pt
