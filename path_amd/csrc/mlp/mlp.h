// Radiance MLP state behind the C ABI.
#pragma once

#include "../host/renderer.h"
#include "mlp_kernels.h"

struct pt_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  uint32_t step = 0; // Adam steps taken
  bool fused_forward = true; // inference through k_mlp_tile

  pt::host::DeviceBuf<float> w32, adam_m, adam_v, grad;
  // bf16 weights: row-major (the kernels' column order in layer 0) and in the
  // fused kernels' forward and backward fragment orders
  pt::host::DeviceBuf<pt::mlp::bf16> wbf, w_frag, wt_frag;

  // per-batch buffers (grow-only, rows padded to kRowAlign)
  pt::host::DeviceBuf<float> feat, targ, pred;
  pt::host::DeviceBuf<pt::mlp::bf16> x0, act[2]; // layer-by-layer forward
  pt::host::DeviceBuf<float> pred_pad;           // and its padded output
  // training: layer inputs and output gradients in fragment order, activation
  // bits, per-tile and per-split partial sums
  pt::host::DeviceBuf<uint16_t> a_frag, g_frag;
  pt::host::DeviceBuf<uint32_t> masks;
  pt::host::DeviceBuf<float> out_part, out_grad, loss_part, split_part;
  pt::host::DeviceBuf<float> step_losses; // one mean loss per step

  // resident training set
  pt::host::DeviceBuf<float> ds_feat, ds_targ;
  uint64_t ds_rows = 0;

  ~pt_mlp();
  bool init(int dev, uint64_t seed, std::string *err);
  int ensure_training(uint32_t rows_pad, uint32_t steps);
  // Forward on device features (n rows; rows up to rows_pad count as zero
  // features): pred[rows_pad x 3] fp32, by the fused kernel unless disabled.
  int forward_device(const float *d_feat, uint32_t n, uint32_t rows_pad,
                     hipStream_t on = nullptr);
  // Forward, loss, backward of a batch of n rows: per-split gradients in
  // split_part / out_grad, the mean loss in *loss_dev (device). With set_rows,
  // row i is row random(seed, i) of the set_rows rows at d_feat / d_targ.
  int gradients(const float *d_feat, const float *d_targ, uint64_t set_rows, uint64_t seed,
                uint32_t n, uint32_t rows_pad, float *loss_dev);
  // Sum the splits: into `grad`, or into one Adam step; or refresh the bf16
  // copies of w32 (mlp::MlpUpdate).
  int update(int mode, uint32_t rows_pad, float lr = 0.f);
};

namespace pt {
namespace host {
inline uint32_t mlp_pad_rows(uint64_t n) {
  return uint32_t((n + mlp::kRowAlign - 1) / mlp::kRowAlign * mlp::kRowAlign);
}
} // namespace host
} // namespace pt
