// A HIP runtime and kernel launchers that run nothing, to link the library's
// host sources against on a machine without a GPU. Device memory is host
// memory under a limit, launches are counted by name and can be made to fail,
// a traversal launch reports empty queues (at once or after a delay), and
// copies out of pinned memory count as in flight until their stream is waited
// for.
#include "../../path_amd/csrc/gpu/radix_sort.h"
#include "../../path_amd/csrc/host/renderer.h"
#include "../../path_amd/csrc/mlp/mlp_kernels.h"

#include <rocrand/rocrand.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>

namespace {
struct Fake {
  std::mutex m;
  std::map<const char *, size_t> device, pinned;
  std::map<std::string, uint64_t> launches;
  std::map<hipStream_t, int> reads;               // copies out of pinned memory
  std::string failing;
  size_t limit = size_t(1) << 60, live = 0, largest = 0;
  uint64_t pool = 0;   // paths of the wavefront renders begun
  uint64_t blocks = 0; // largest grid of a wavefront launch
  uint32_t report_delay_ms = 0;
  std::atomic<int> late{0}; // reports still to come
} f;

bool inside(const std::map<const char *, size_t> &blocks, const void *p) {
  auto it = blocks.upper_bound(static_cast<const char *>(p));
  return it != blocks.begin() && static_cast<const char *>(p) < (--it)->first + it->second;
}

hipError_t launch(const char *name, uint64_t pool = 0, uint64_t blocks = 0) {
  std::lock_guard<std::mutex> l(f.m);
  f.launches[name] += 1;
  f.pool += pool;
  f.blocks = std::max(f.blocks, blocks);
  return f.failing == name ? hipErrorLaunchFailure : hipSuccess;
}
} // namespace

extern "C" {
void fake_reset() {
  std::lock_guard<std::mutex> l(f.m);
  f.launches.clear(), f.reads.clear(), f.failing.clear();
  f.limit = size_t(1) << 60, f.largest = 0, f.pool = f.blocks = 0, f.report_delay_ms = 0;
}
void fake_limit(uint64_t bytes) { f.limit = bytes; }
void fake_fail(const char *name) { f.failing = name; }
void fake_report_delay(uint32_t ms) { f.report_delay_ms = ms; }
uint64_t fake_live() { return f.live; }
uint64_t fake_largest() { return f.largest; }
uint64_t fake_launches(const char *name) { return f.launches[name]; }
uint64_t fake_pool() { return f.pool; }
uint64_t fake_blocks() { return f.blocks; }
uint64_t fake_in_flight() {
  uint64_t n = 0;
  for (auto &s : f.reads)
    n += s.second;
  return n;
}

hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> l(f.m);
  f.largest = std::max(f.largest, n);
  if (f.live + n > f.limit)
    return hipErrorOutOfMemory;
  *p = std::calloc(n, 1);
  f.device[static_cast<char *>(*p)] = n;
  f.live += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> l(f.m);
  auto it = f.device.find(static_cast<char *>(p));
  if (it != f.device.end()) {
    f.live -= it->second;
    f.device.erase(it);
    std::free(p);
  }
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> l(f.m);
  *p = std::calloc(n, 1);
  f.pinned[static_cast<char *>(*p)] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> l(f.m);
  f.pinned.erase(static_cast<char *>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  std::lock_guard<std::mutex> l(f.m);
  std::memcpy(d, s, n);
  if (inside(f.pinned, s))
    f.reads[st] += 1;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  if (n < (size_t(1) << 24)) // large arrays are fresh, zero already
    std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return f.late ? hipErrorNotReady : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) {
  while (f.late)
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
  std::lock_guard<std::mutex> l(f.m);
  f.reads[st] = 0;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  static std::atomic<uintptr_t> next{1};
  *s = reinterpret_cast<hipStream_t>(next++);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  std::lock_guard<std::mutex> l(f.m);
  if (!inside(f.device, p))
    return hipErrorInvalidValue;
  a->type = hipMemoryTypeDevice;
  a->device = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake error"; }
// captured iterations are not part of these tests
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
rocrand_status rocrand_get_direction_vectors32(const unsigned int **,
                                               rocrand_direction_vector_set) {
  return ROCRAND_STATUS_INTERNAL_ERROR;
}
}

namespace pt {
namespace host {
int noalloc_init(int, std::string *) { return PT_OK; }
} // namespace host

namespace gpu {
hipError_t launch_wf_shade(const WfParams &p, WfKind, hipStream_t) {
  return launch("wf_shade", p.fresh ? p.n_slots : 0, p.n_shade_blocks);
}
hipError_t launch_wf_trace(const WfParams &p, WfKind, uint32_t blocks, hipStream_t) {
  WfReport *rep = p.report;
  const uint32_t it = ++p.counters[kIterations];
  auto tell = [rep, it] {
    rep->ext = rep->shadow = rep->samples_left = 0;
    __atomic_store_n(&rep->iteration, it, __ATOMIC_RELEASE);
  };
  if (f.report_delay_ms) {
    ++f.late;
    std::thread([tell, ms = f.report_delay_ms] {
      std::this_thread::sleep_for(std::chrono::milliseconds(ms));
      tell();
      --f.late;
    }).detach();
  } else {
    tell();
  }
  return launch("wf_trace", 0, blocks);
}
hipError_t launch_wf_finish(const WfParams &, WfKind, uint32_t, hipStream_t) {
  return launch("wf_finish");
}
hipError_t launch_wf_reduce(const float *, const WorkDivision &, uint32_t, float *, hipStream_t) {
  return launch("wf_reduce");
}
hipError_t launch_wf_reduce_batch(const float *, const WfReduceItem *, uint32_t, uint32_t,
                                  uint32_t, uint32_t, float *, hipStream_t) {
  return launch("wf_reduce_batch");
}
hipError_t launch_megakernel(const MegaParams &, uint32_t, uint32_t, bool, hipStream_t) {
  return launch("mega");
}
hipError_t launch_megakernel_batch(const MegaBatchParams &, uint32_t, uint32_t, uint32_t,
                                   hipStream_t) {
  return launch("mega_batch");
}
hipError_t launch_reduce_sample_blocks(const float *, uint32_t, uint32_t, uint32_t, float *,
                                       hipStream_t) {
  return launch("reduce_sample_blocks");
}
hipError_t launch_to_bgra(const float *, uint32_t, uint32_t *, hipStream_t) { return launch("bgra"); }

#define UNUSED(decl)                                                           \
  hipError_t decl { return hipErrorNotSupported; }
UNUSED(launch_intersect(const DeviceScene &, const float *, uint32_t, float *, uint32_t *,
                        uint32_t *, hipStream_t))
UNUSED(launch_sobol_table(const uint32_t *, uint32_t, uint32_t, float *, hipStream_t))
UNUSED(launch_reduce_samples(const WorkDivision &, const float *, uint32_t, float *, hipStream_t))
UNUSED(launch_sum_samples_f64(const float *, uint32_t, uint32_t, double *, hipStream_t))
UNUSED(launch_adjoint(const AdjointParams &, hipStream_t))
UNUSED(launch_adjoint_finalize(const float *, uint32_t, uint32_t, double, double *, float *,
                               hipStream_t))
UNUSED(launch_l2_gradient(const float *, const float *, uint64_t, float *, hipStream_t))
UNUSED(launch_nrc_paths(const NrcParams &, hipStream_t))
UNUSED(launch_nrc_first_vertex(const NrcParams &, hipStream_t))
UNUSED(launch_nrc_combine(const float *, const float *, const float *, uint32_t, uint32_t, float *,
                          hipStream_t))
UNUSED(build_lbvh(const LbvhBuffers &, const LbvhRoot *, uint32_t, LbvhBuilder, hipStream_t,
                  uint32_t *))
UNUSED(lbvh_sort_temp_bytes(uint32_t, uint32_t, size_t *))
UNUSED(radix_sort_pairs(unsigned long long *, uint32_t *, unsigned long long *, uint32_t *,
                        uint32_t, uint32_t, void *, size_t, hipStream_t))
size_t radix_sort_temp_bytes(uint32_t) { return 0; }
uint32_t adjoint_finalize_groups(uint32_t) { return 1; }
} // namespace gpu

namespace mlp {
hipError_t launch_mlp_tile(const MlpTileArgs &, uint32_t, bool, hipStream_t) { return launch("tile"); }
hipError_t launch_mlp_wgrad(const MlpWgradArgs &, hipStream_t) { return launch("wgrad"); }
hipError_t launch_mlp_update(const MlpUpdateArgs &, int, hipStream_t) { return launch("update"); }
uint32_t mlp_tile_rows(uint32_t) { return 32; }
uint32_t mlp_wgrad_splits(uint32_t) { return 42; }
UNUSED(launch_gemm(const GemmArgs &, int, hipStream_t))
UNUSED(launch_encode(const float *, uint32_t, uint32_t, bf16 *, hipStream_t))
UNUSED(launch_compact_pred(const float *, uint32_t, float *, hipStream_t))
} // namespace mlp
} // namespace pt
