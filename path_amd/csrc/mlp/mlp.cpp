// Radiance MLP host side: parameters, forward / backward schedules, Adam,
// resident training set, C ABI.
#include "mlp.h"

#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

using namespace pt;
using namespace pt::host;
using namespace pt::mlp;

#define HIP_TRY(expr)                                                          \
  do {                                                                         \
    hipError_t e_ = (expr);                                                    \
    if (e_ != hipSuccess)                                                      \
      return set_error(PT_ERR_HIP, std::string(#expr) + ": " +                 \
                                       hipGetErrorString(e_));                 \
  } while (0)

pt_mlp::~pt_mlp() {
  if (ev0)
    (void)hipEventDestroy(ev0);
  if (ev1)
    (void)hipEventDestroy(ev1);
  if (stream)
    (void)hipStreamDestroy(stream);
}

// He-uniform initialisation with a seeded SplitMix64; padded input columns of
// layer 0 and padded output rows of the last layer are zero.
static std::vector<float> init_weights(uint64_t seed) {
  std::vector<float> w(param_count(), 0.f);
  uint64_t s = seed * 0x2545f4914f6cdd1dull + 0x51ed27ull;
  auto next = [&]() {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return double(z >> 11) * 0x1p-53;
  };
  for (uint32_t l = 0; l < kLayers; ++l) {
    const uint32_t in = layer_in(l), out = layer_out(l);
    const uint32_t in_valid = l == 0 ? kEncoded : in;
    const uint32_t out_valid = l + 1 == kLayers ? kOut : out;
    const double bound = std::sqrt(6.0 / in_valid) * (l + 1 == kLayers ? 0.1 : 1.0);
    float *wl = w.data() + layer_offset(l);
    for (uint32_t o = 0; o < out_valid; ++o)
      for (uint32_t i = 0; i < in_valid; ++i)
        wl[size_t(o) * in + i] = float((2.0 * next() - 1.0) * bound);
  }
  return w;
}

bool pt_mlp::init(int dev, uint64_t seed, std::string *err) {
  device = dev;
  hipError_t e = hipSetDevice(dev);
  if (e == hipSuccess)
    e = hipStreamCreateWithFlags(&stream, hipStreamNonBlocking);
  if (e == hipSuccess)
    e = hipEventCreate(&ev0);
  if (e == hipSuccess)
    e = hipEventCreate(&ev1);
  const uint64_t P = param_count();
  std::vector<float> w = init_weights(seed);
  if (e == hipSuccess)
    e = w32.upload(w.data(), P, stream);
  if (e == hipSuccess)
    e = wbf.ensure(P);
  if (e == hipSuccess)
    e = w_frag.ensure(kWFragElems);
  if (e == hipSuccess)
    e = wt_frag.ensure(kWtFragElems);
  if (e == hipSuccess)
    e = adam_m.ensure(P);
  if (e == hipSuccess)
    e = adam_v.ensure(P);
  if (e == hipSuccess)
    e = grad.ensure(P);
  if (e == hipSuccess)
    e = out_grad.ensure(size_t(kOut) * kWidth);
  // outputs 16 .. 31 of the output layer's fragments stay zero
  if (e == hipSuccess)
    e = hipMemsetAsync(w_frag.ptr, 0, kWFragElems * sizeof(bf16), stream);
  if (e == hipSuccess)
    e = hipMemsetAsync(adam_m.ptr, 0, P * 4, stream);
  if (e == hipSuccess)
    e = hipMemsetAsync(adam_v.ptr, 0, P * 4, stream);
  if (e == hipSuccess && update(kUpdatePack, 0) != PT_OK)
    e = hipErrorUnknown;
  if (e == hipSuccess)
    e = hipStreamSynchronize(stream);
  if (e != hipSuccess) {
    *err = std::string("MLP init: ") + hipGetErrorString(e);
    return false;
  }
  return true;
}

int pt_mlp::ensure_training(uint32_t rows_pad, uint32_t steps) {
  const uint32_t tiles = rows_pad / mlp_tile_rows(rows_pad);
  HIP_TRY(a_frag.ensure(size_t(kHidden) * rows_pad * kWidth));
  HIP_TRY(g_frag.ensure(size_t(kHidden) * rows_pad * kWidth));
  HIP_TRY(masks.ensure(size_t(rows_pad) * (kHidden * kWidth / 32)));
  HIP_TRY(out_part.ensure(size_t(tiles) * kOut * kWidth));
  HIP_TRY(loss_part.ensure(tiles));
  HIP_TRY(split_part.ensure(size_t(kHidden) * mlp_wgrad_splits(rows_pad) * kWidth * kWidth));
  HIP_TRY(step_losses.ensure(std::max<uint32_t>(steps, 1)));
  return PT_OK;
}

static GemmArgs gemm_args(const bf16 *A, uint32_t lda, const bf16 *B, uint32_t ldb,
                          uint32_t M, uint32_t N, uint32_t K, void *C, uint32_t ldc) {
  GemmArgs g{};
  g.A = A;
  g.B = B;
  g.lda = lda;
  g.ldb = ldb;
  g.M = M;
  g.N = N;
  g.K = K;
  g.C = C;
  g.ldc = ldc;
  return g;
}

int pt_mlp::forward_device(const float *d_feat, uint32_t n, uint32_t rows_pad, hipStream_t on) {
  hipStream_t stream = on ? on : this->stream;
  HIP_TRY(pred.ensure(size_t(rows_pad) * kOut));
  if (fused_forward) {
    MlpTileArgs t{};
    t.feat = d_feat;
    t.n = n;
    t.w_frag = reinterpret_cast<const uint16_t *>(w_frag.ptr);
    t.pred = pred.ptr;
    HIP_TRY(launch_mlp_tile(t, rows_pad, false, stream));
    return PT_OK;
  }
  HIP_TRY(pred_pad.ensure(size_t(rows_pad) * kOutPad));
  HIP_TRY(x0.ensure(size_t(rows_pad) * kInPad));
  for (auto &a : act)
    HIP_TRY(a.ensure(size_t(rows_pad) * kWidth));
  HIP_TRY(launch_encode(d_feat, n, rows_pad, x0.ptr, stream));
  const bf16 *in = x0.ptr;
  for (uint32_t l = 0; l < kLayers; ++l) {
    const bf16 *w = wbf.ptr + layer_offset(l);
    if (l + 1 < kLayers) {
      bf16 *out = act[l & 1].ptr;
      HIP_TRY(launch_gemm(gemm_args(in, layer_in(l), w, layer_in(l), rows_pad, kWidth,
                                    layer_in(l), out, kWidth),
                          kEpiReluBf16, stream));
      in = out;
    } else {
      HIP_TRY(launch_gemm(gemm_args(in, kWidth, w, kWidth, rows_pad, kOutPad, kWidth,
                                    pred_pad.ptr, kOutPad),
                          kEpiF32, stream));
      HIP_TRY(launch_compact_pred(pred_pad.ptr, rows_pad, pred.ptr, stream));
    }
  }
  return PT_OK;
}

int pt_mlp::gradients(const float *d_feat, const float *d_targ, uint64_t set_rows,
                      uint64_t seed, uint32_t n, uint32_t rows_pad, float *loss_dev) {
  MlpTileArgs t{};
  t.feat = d_feat;
  t.targ = d_targ;
  t.set_rows = set_rows;
  t.seed = seed;
  t.n = n;
  t.w_frag = reinterpret_cast<const uint16_t *>(w_frag.ptr);
  t.wt_frag = reinterpret_cast<const uint16_t *>(wt_frag.ptr);
  t.a_frag = a_frag.ptr;
  t.g_frag = g_frag.ptr;
  t.layer_stride = size_t(rows_pad) * kWidth;
  t.masks = masks.ptr;
  t.out_part = out_part.ptr;
  t.loss_part = loss_part.ptr;
  HIP_TRY(launch_mlp_tile(t, rows_pad, true, stream));
  MlpWgradArgs g{};
  g.a_frag = a_frag.ptr;
  g.g_frag = g_frag.ptr;
  g.layer_stride = t.layer_stride;
  g.rows_pad = rows_pad;
  g.splits = mlp_wgrad_splits(rows_pad);
  g.tiles = rows_pad / mlp_tile_rows(rows_pad);
  g.part = split_part.ptr;
  g.out_part = out_part.ptr;
  g.loss_part = loss_part.ptr;
  g.out_grad = out_grad.ptr;
  g.loss = loss_dev;
  HIP_TRY(launch_mlp_wgrad(g, stream));
  return PT_OK;
}

int pt_mlp::update(int mode, uint32_t rows_pad, float lr) {
  MlpUpdateArgs u{};
  u.part = split_part.ptr;
  u.out_grad = out_grad.ptr;
  u.splits = mlp_wgrad_splits(rows_pad);
  u.grad = grad.ptr;
  u.w = w32.ptr;
  u.m = adam_m.ptr;
  u.v = adam_v.ptr;
  u.w_rows = reinterpret_cast<uint16_t *>(wbf.ptr);
  u.w_frag = reinterpret_cast<uint16_t *>(w_frag.ptr);
  u.wt_frag = reinterpret_cast<uint16_t *>(wt_frag.ptr);
  u.lr = lr;
  u.beta1 = 0.9f;
  u.beta2 = 0.99f;
  u.eps = 1e-8f;
  if (mode == kUpdateAdam) {
    ++step;
    u.c1 = 1.f - powf(u.beta1, float(step));
    u.c2 = 1.f - powf(u.beta2, float(step));
  }
  HIP_TRY(launch_mlp_update(u, mode, stream));
  return PT_OK;
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int pt_mlp_create(int device, uint64_t seed, pt_mlp **out) {
  if (!out)
    return set_error(PT_ERR_INVALID, "null output pointer");
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0)
    return set_error(PT_ERR_NO_DEVICE, "no HIP device");
  if (device < 0 || device >= count)
    return set_error(PT_ERR_INVALID, "device index out of range");
  auto m = new (std::nothrow) pt_mlp();
  if (!m)
    return set_error(PT_ERR_INVALID, "out of host memory");
  std::string err;
  if (!m->init(device, seed, &err)) {
    delete m;
    return set_error(PT_ERR_HIP, err);
  }
  *out = m;
  return PT_OK;
}

void pt_mlp_destroy(pt_mlp *m) { delete m; }

int pt_mlp_param_count(uint64_t *count) {
  if (!count)
    return set_error(PT_ERR_INVALID, "null argument");
  *count = param_count();
  return PT_OK;
}

int pt_mlp_get_weights(pt_mlp *m, float *w) {
  if (!m || !w)
    return set_error(PT_ERR_INVALID, "null argument");
  HIP_TRY(hipSetDevice(m->device));
  HIP_TRY(hipMemcpyAsync(w, m->w32.ptr, param_count() * 4, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return PT_OK;
}

int pt_mlp_set_weights(pt_mlp *m, const float *w) {
  if (!m || !w)
    return set_error(PT_ERR_INVALID, "null argument");
  HIP_TRY(hipSetDevice(m->device));
  HIP_TRY(m->w32.upload(w, param_count(), m->stream));
  int rc = m->update(kUpdatePack, 0);
  if (rc != PT_OK)
    return rc;
  HIP_TRY(hipMemsetAsync(m->adam_m.ptr, 0, param_count() * 4, m->stream));
  HIP_TRY(hipMemsetAsync(m->adam_v.ptr, 0, param_count() * 4, m->stream));
  m->step = 0;
  HIP_TRY(hipStreamSynchronize(m->stream));
  return PT_OK;
}

int pt_mlp_set_forward_kernel(pt_mlp *m, int fused) {
  if (!m)
    return set_error(PT_ERR_INVALID, "null argument");
  m->fused_forward = fused != 0;
  return PT_OK;
}

int pt_mlp_forward(pt_mlp *m, const float *features, uint32_t n, float *out) {
  if (!m || (n && (!features || !out)))
    return set_error(PT_ERR_INVALID, "null argument");
  if (n == 0)
    return PT_OK;
  HIP_TRY(hipSetDevice(m->device));
  const uint32_t rp = mlp_pad_rows(n);
  HIP_TRY(m->feat.upload(features, size_t(n) * kFeatures, m->stream));
  int rc = m->forward_device(m->feat.ptr, n, rp);
  if (rc != PT_OK)
    return rc;
  HIP_TRY(hipMemcpyAsync(out, m->pred.ptr, size_t(n) * kOut * 4, hipMemcpyDeviceToHost,
                         m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return PT_OK;
}

// Upload a host batch and queue its forward, loss and backward.
static int batch_gradients(pt_mlp *m, const float *features, const float *targets, uint32_t n,
                           uint32_t *rp_out) {
  const uint32_t rp = mlp_pad_rows(n);
  int rc = m->ensure_training(rp, 1);
  if (rc != PT_OK)
    return rc;
  HIP_TRY(m->feat.upload(features, size_t(n) * kFeatures, m->stream));
  HIP_TRY(m->targ.upload(targets, size_t(n) * kOut, m->stream));
  *rp_out = rp;
  return m->gradients(m->feat.ptr, m->targ.ptr, 0, 0, n, rp, m->step_losses.ptr);
}

int pt_mlp_gradient(pt_mlp *m, const float *features, const float *targets, uint32_t n,
                    float *grad, float *loss) {
  if (!m || !features || !targets || !grad || n == 0)
    return set_error(PT_ERR_INVALID, "null argument or empty batch");
  HIP_TRY(hipSetDevice(m->device));
  uint32_t rp;
  int rc = batch_gradients(m, features, targets, n, &rp);
  if (rc == PT_OK)
    rc = m->update(kUpdateGradient, rp);
  if (rc != PT_OK)
    return rc;
  HIP_TRY(hipMemcpyAsync(grad, m->grad.ptr, param_count() * 4, hipMemcpyDeviceToHost,
                         m->stream));
  if (loss)
    HIP_TRY(hipMemcpyAsync(loss, m->step_losses.ptr, 4, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return PT_OK;
}

int pt_mlp_train_step(pt_mlp *m, const float *features, const float *targets, uint32_t n,
                      float lr, float *loss) {
  if (!m || !features || !targets || n == 0)
    return set_error(PT_ERR_INVALID, "null argument or empty batch");
  HIP_TRY(hipSetDevice(m->device));
  uint32_t rp;
  int rc = batch_gradients(m, features, targets, n, &rp);
  if (rc == PT_OK)
    rc = m->update(kUpdateAdam, rp, lr);
  if (rc != PT_OK)
    return rc;
  if (loss)
    HIP_TRY(hipMemcpyAsync(loss, m->step_losses.ptr, 4, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return PT_OK;
}

// Times `iters` inference passes over `rows` device-resident rows (features
// all 0.25): the average duration of one hidden 256x256 layer GEMM (layer 1)
// and of the whole forward pass, both with HIP events on the MLP's stream.
int pt_mlp_time_forward(pt_mlp *m, uint32_t rows, uint32_t iters, float *gemm_ms,
                        float *forward_ms) {
  if (!m || rows == 0 || iters == 0)
    return set_error(PT_ERR_INVALID, "null argument or empty workload");
  HIP_TRY(hipSetDevice(m->device));
  const uint32_t rp = mlp_pad_rows(rows);
  for (auto &a : m->act)
    HIP_TRY(a.ensure(size_t(rp) * kWidth));
  std::vector<float> f(size_t(rp) * kFeatures, 0.25f);
  HIP_TRY(m->feat.upload(f.data(), f.size(), m->stream));
  int rc = m->forward_device(m->feat.ptr, rp, rp);
  if (rc != PT_OK)
    return rc;
  GemmArgs g = gemm_args(m->act[0].ptr, kWidth, m->wbf.ptr + layer_offset(1), kWidth, rp,
                         kWidth, kWidth, m->act[1].ptr, kWidth);
  HIP_TRY(hipEventRecord(m->ev0, m->stream));
  for (uint32_t i = 0; i < iters; ++i)
    HIP_TRY(launch_gemm(g, kEpiReluBf16, m->stream));
  HIP_TRY(hipEventRecord(m->ev1, m->stream));
  HIP_TRY(hipEventSynchronize(m->ev1));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
  if (gemm_ms)
    *gemm_ms = ms / float(iters);
  HIP_TRY(hipEventRecord(m->ev0, m->stream));
  for (uint32_t i = 0; i < iters && rc == PT_OK; ++i)
    rc = m->forward_device(m->feat.ptr, rp, rp);
  if (rc != PT_OK)
    return rc;
  HIP_TRY(hipEventRecord(m->ev1, m->stream));
  HIP_TRY(hipEventSynchronize(m->ev1));
  HIP_TRY(hipEventElapsedTime(&ms, m->ev0, m->ev1));
  if (forward_ms)
    *forward_ms = ms / float(iters);
  return PT_OK;
}

int pt_mlp_set_dataset(pt_mlp *m, const float *features, const float *targets, uint64_t rows) {
  if (!m || (rows && (!features || !targets)))
    return set_error(PT_ERR_INVALID, "null argument");
  if (rows >= (1ull << 32))
    return set_error(PT_ERR_INVALID, "at most 2^32 - 1 training rows");
  HIP_TRY(hipSetDevice(m->device));
  HIP_TRY(m->ds_feat.upload(features, rows * kFeatures, m->stream));
  HIP_TRY(m->ds_targ.upload(targets, rows * kOut, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  m->ds_rows = rows;
  return PT_OK;
}

int pt_mlp_train(pt_mlp *m, uint32_t steps, uint32_t batch, float lr, uint64_t seed,
                 float *losses, double *seconds) {
  if (!m || batch == 0)
    return set_error(PT_ERR_INVALID, "null argument or empty batch");
  if (m->ds_rows == 0)
    return set_error(PT_ERR_INVALID, "no training set (pt_mlp_set_dataset)");
  HIP_TRY(hipSetDevice(m->device));
  const uint32_t rp = mlp_pad_rows(batch);
  int rc = m->ensure_training(rp, losses ? steps : 1);
  if (rc != PT_OK)
    return rc;
  auto t0 = std::chrono::steady_clock::now();
  for (uint32_t it = 0; it < steps; ++it) {
    rc = m->gradients(m->ds_feat.ptr, m->ds_targ.ptr, m->ds_rows,
                      seed + it * 0x632be59bd9b4e019ull, batch, rp,
                      m->step_losses.ptr + (losses ? it : 0));
    if (rc == PT_OK)
      rc = m->update(kUpdateAdam, rp, lr);
    if (rc != PT_OK)
      return rc;
  }
  // the per-step losses stay on the device until the end: no step waits
  // for the host
  if (losses && steps)
    HIP_TRY(hipMemcpyAsync(losses, m->step_losses.ptr, size_t(steps) * sizeof(float),
                           hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  if (seconds)
    *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  return PT_OK;
}

} // extern "C"
