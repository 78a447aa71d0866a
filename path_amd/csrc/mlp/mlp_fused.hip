// The radiance MLP's fused kernels: the forward pass of a row tile with its
// activations in LDS (inference), the same with loss and data gradients
// (training), the weight gradients, and the update (split sums, Adam, BF16
// copies).
//
// Everything the matrix cores read from memory is stored in fragment order:
// 64 lanes x 8 bf16 = 1 KB that a wave loads with one 16-byte load per lane.
//   forward weights   [layer][32 outputs][16 inputs][lane]: lane l holds
//                     W[out = l % 32][in = 8 (l / 32) ..+8] of the block
//   backward weights  [layer][32 inputs][16 outputs][lane]: lane l holds
//                     W[out = 8 (l / 32) ..+8][in = l % 32]
//   A_l, G_l          [16 rows][32 columns][lane]: lane l holds
//                     rows 8 (l / 32) ..+8 of column l % 32 (the operands of
//                     the weight gradient, whose K is the batch)
// Row-major weights made a wave's load touch 32 cache lines for 32 of their
// 128 bytes each, four times the useful L2 traffic (2^20 queries: 0.94 ms).
#include "mlp_encode.h"

namespace pt {
namespace mlp {

namespace {

typedef short s16x2_t __attribute__((ext_vector_type(2)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

static_assert(kInPad == kWidth, "hidden weight matrices are all kWidth x kWidth");
constexpr uint32_t kXStride = kWidth + 8; // LDS row of the tile's activations
constexpr uint32_t kDStride = 40;         // LDS row of d(loss)/d(pred): 32 columns
constexpr uint32_t kFrag = 512;           // bf16 per fragment
constexpr uint32_t kKSteps = kWidth / 16;
constexpr uint32_t kColBlocks = kWidth / 32;
constexpr uint32_t kLayerFrags = kColBlocks * kKSteps; // fragments of a hidden layer
// weight fragments in flight ahead of their MFMAs (2 / 3 / 4: 611 / 613 / 606
// us per 2^20 queries, 270 / 267 / 266 us per training step of 65,536 rows with
// cached stores)
constexpr uint32_t kWAhead = 3;

// Row of the training set that row i of a step draws (SplitMix64).
__device__ __forceinline__ uint32_t random_row(uint32_t i, uint64_t n_rows, uint64_t seed) {
  uint64_t z = seed + 0x9e3779b97f4a7c15ull * (uint64_t(i) + 1);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  z ^= z >> 31;
  return uint32_t(z % n_rows);
}

// Operand fragment whose K is the row, from a row-major LDS tile: lane l gets
// rows 16 rb + 8 (l / 32) ..+8 of column 32 cb + l % 32. A transposing read
// takes four rows x 16 columns per 16 lanes: lane j of the 16 supplies the
// address of row j / 4, columns 4 (j % 4) ..+4, and receives column j.
__device__ __forceinline__ bf16x8_t column_frag(const uint16_t *tile, uint32_t stride,
                                                uint32_t rb, uint32_t cb) {
  const uint32_t lane = threadIdx.x & 63u, j = lane & 15u, g = lane >> 4;
  const uint16_t *p = tile + (rb * 16u + (g >> 1) * 8u + (j >> 2)) * stride + cb * 32u +
                      (g & 1u) * 16u + (j & 3u) * 4u;
  typedef __attribute__((address_space(3))) s16x4_t *lds_ptr;
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * stride));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Batches of at least kStreamRows rows write A and G past the caches and read
// them back the same way: what one kernel writes (0.15 GB there, 0.4 GB at
// 65,536 rows) is evicted before the next reads it, and takes the weights with
// it. Training step, us, cached / stores streamed / loads too: 16,384 rows 91 /
// 94 / 94; 24,576: 111 / 116 / 115; 32,768: 139 / 139 / 129; 65,536: 258 / 242 /
// 216; 131,072: 497 / 440 / 395.
constexpr uint32_t kStreamRows = 24576;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// The tile's fragments for the weight gradient: wave w writes the column
// blocks 2 w and 2 w + 1. (Tiles of more than 32 rows are those of batches of
// at least kStreamRows.)
template <uint32_t kI>
__device__ __forceinline__ void store_column_frags(const uint16_t *X, uint16_t *__restrict__ dst,
                                                   uint32_t wave) {
  const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
  for (uint32_t rb = 0; rb < 2 * kI; ++rb)
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      const uint32_t cb = 2 * wave + j;
      auto *at = reinterpret_cast<bf16x8_t *>(dst + (size_t(rb) * kColBlocks + cb) * kFrag +
                                              lane * 8u);
      const bf16x8_t v = column_frag(X, kXStride, rb, cb);
      if constexpr (kI > 1)
        __builtin_nontemporal_store(v, at);
      else
        *at = v;
    }
}

// One 256 x 256 layer on the tile: acc[i][j] = 32 outputs x 32 rows, wave w
// computes outputs 64 w + 32 j, rows 32 i. `wf`: the layer's fragments.
// Weights are the MFMA's A operand, so register r of lane l is output
// 8 (r / 4) + 4 (l / 32) + r % 4 of row l % 32 and a lane's four adjacent
// outputs are one 8-byte LDS store. Weight fragments are loaded kWAhead K
// steps before their MFMAs (a ring of registers); scheduling barriers keep
// the compiler from sinking the loads next to their use.
template <uint32_t kI>
__device__ __forceinline__ void layer_products(const uint16_t *__restrict__ wf,
                                               const uint16_t *X, uint32_t wave,
                                               f32x16_t (&acc)[kI][2]) {
  const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, khalf = (lane >> 5) * 8u;
#pragma unroll
  for (uint32_t i = 0; i < kI; ++i)
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.f;
  const uint16_t *wp = wf + size_t(2 * wave) * kKSteps * kFrag + lane * 8u;
  bf16x8_t wq[kWAhead + 1][2];
#pragma unroll
  for (uint32_t s = 0; s < kWAhead; ++s)
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j)
      wq[s][j] = *reinterpret_cast<const bf16x8_t *>(wp + (j * kKSteps + s) * kFrag);
#pragma unroll
  for (uint32_t ks = 0; ks < kKSteps; ++ks) {
    if (ks + kWAhead < kKSteps) {
#pragma unroll
      for (uint32_t j = 0; j < 2; ++j)
        wq[(ks + kWAhead) % (kWAhead + 1)][j] =
            *reinterpret_cast<const bf16x8_t *>(wp + (j * kKSteps + ks + kWAhead) * kFrag);
    }
    __builtin_amdgcn_sched_barrier(0);
    bf16x8_t x[kI];
#pragma unroll
    for (uint32_t i = 0; i < kI; ++i)
      x[i] = *reinterpret_cast<const bf16x8_t *>(X + (i * 32u + l32) * kXStride + ks * 16u +
                                                 khalf);
#pragma unroll
    for (uint32_t i = 0; i < kI; ++i)
#pragma unroll
      for (uint32_t j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wq[ks % (kWAhead + 1)][j], x[i],
                                                            acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Where lane l's four outputs q of acc[i][j] go in the tile.
__device__ __forceinline__ uint2 *tile_slot(uint16_t *X, uint32_t wave, uint32_t i, uint32_t j,
                                            uint32_t q) {
  const uint32_t lane = threadIdx.x & 63u;
  return reinterpret_cast<uint2 *>(X + (i * 32u + (lane & 31u)) * kXStride + wave * 64u +
                                   j * 32u + q * 8u + (lane >> 5) * 4u);
}

// ReLU, rounding, store. With kMask, mask[i] collects which of the lane's 32
// outputs of row block i are positive: pair p's bits end up at p and 16 + p
// (0 - v has its sign bit set exactly where the bf16 v >= 0 is not zero).
template <uint32_t kI, bool kMask>
__device__ __forceinline__ void store_relu(const f32x16_t (&acc)[kI][2], uint16_t *X,
                                           uint32_t wave, uint32_t *mask) {
#pragma unroll
  for (uint32_t i = 0; i < kI; ++i) {
    uint32_t m = 0;
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        uint32_t v[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
          const float a = acc[i][j][4 * q + 2 * h], b = acc[i][j][4 * q + 2 * h + 1];
          v[h] = f2bf2(a > 0.f ? a : 0.f, b > 0.f ? b : 0.f);
          if constexpr (kMask) {
            const s16x2_t neg = s16x2_t{0, 0} - __builtin_bit_cast(s16x2_t, v[h]);
            m = (m >> 1) | (__builtin_bit_cast(uint32_t, neg) & 0x80008000u);
          }
        }
        *tile_slot(X, wave, i, j, q) = make_uint2(v[0], v[1]);
      }
    if constexpr (kMask)
      mask[i] = m;
  }
}

// Rounding, the mask of the layer's forward outputs, store.
template <uint32_t kI>
__device__ __forceinline__ void store_masked(const f32x16_t (&acc)[kI][2], uint16_t *X,
                                             uint32_t wave, const uint32_t *mask) {
#pragma unroll
  for (uint32_t i = 0; i < kI; ++i)
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q) {
        uint32_t v[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
          const uint32_t pair = j * 8u + q * 2u + h;
          const s16x2_t keep = __builtin_bit_cast(s16x2_t, mask[i] << (15u - pair)) >> 15;
          v[h] = f2bf2(acc[i][j][4 * q + 2 * h], acc[i][j][4 * q + 2 * h + 1]) &
                 __builtin_bit_cast(uint32_t, keep);
        }
        *tile_slot(X, wave, i, j, q) = make_uint2(v[0], v[1]);
      }
}

template <uint32_t kI> constexpr size_t tile_lds(bool train) {
  return size_t(32) * kI * kXStride * 2 + (train ? size_t(32) * kI * (kDStride * 2 + 4) + 16 : 0);
}

} // namespace

// One workgroup of 4 waves per tile of 32 kI rows: encoding, six hidden
// layers and the output layer with the activations in LDS. Inference writes
// pred. Training goes on in the same workgroup: the loss, d(loss)/d(pred), the
// output layer's weight gradient (its operands are in LDS) and the data
// gradients back to layer 0; per layer it writes only A_l and G_l in fragment
// order for k_mlp_wgrad and one bit per activation (a tile's threads read
// their own bits back). Rows from n on count as zero features and add nothing
// to the gradient. The MFMAs of every output element run in the K order of
// k_gemm's and round the same way, so the forward results equal the
// layer-by-layer GEMMs' bit for bit (GPU test).
// Inference is bound by the matrix cores: 2^20 queries 0.60 ms, 1.34 PFLOP/s
// (0.94 ms with row-major weights and two-byte stores of the encoding); a
// large bf16 library product reaches 1.23 on the same card. Training at
// 65,536 rows: 130 us for 75 us of matrix work and 0.4 GB written (one GEMM
// launch per layer and direction with row-major and transposed copies took
// 420 us and moved 2.2 GB).
template <uint32_t kI, bool kTrain>
__global__ __launch_bounds__(256, 2) void k_mlp_tile(MlpTileArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t X[];
  constexpr uint32_t kRows = 32 * kI;
  uint16_t *D = X + kRows * kXStride;                                   // training only
  uint32_t *row_of = reinterpret_cast<uint32_t *>(D + kRows * kDStride); // [kRows]
  float *wave_loss = reinterpret_cast<float *>(row_of + kRows);          // [4]
  const uint32_t row0 = blockIdx.x * kRows;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t l32 = lane & 31u, khalf = (lane >> 5) * 8u;
  if constexpr (kTrain) {
    for (uint32_t r = threadIdx.x; r < kRows; r += 256u)
      row_of[r] = a.set_rows ? random_row(row0 + r, a.set_rows, a.seed) : row0 + r;
    __syncthreads();
  }
  for (uint32_t k = threadIdx.x; k < kRows * kFeatures; k += 256u) {
    const uint32_t r = k / kFeatures, d = k % kFeatures;
    float x = 0.f;
    if (row0 + r < a.n) {
      const size_t src = kTrain ? row_of[r] : row0 + r;
      x = a.feat[src * kFeatures + d];
    }
    encode_feature(x, d, X + r * kXStride);
  }
  for (uint32_t k = threadIdx.x; k < kRows * (kInPad - kEncoded); k += 256u)
    X[(k / (kInPad - kEncoded)) * kXStride + kEncoded + k % (kInPad - kEncoded)] = 0;
  __syncthreads();
  f32x16_t acc[kI][2];
  const size_t frag0 = size_t(row0) * kWidth; // this tile's fragments within a layer's
  const size_t mask0 = (size_t(blockIdx.x) * kHidden * 256u + threadIdx.x) * kI;
#pragma unroll 1
  for (uint32_t l = 0; l < kHidden; ++l) {
    if constexpr (kTrain)
      store_column_frags<kI>(X, a.a_frag + l * a.layer_stride + frag0, wave);
    layer_products<kI>(a.w_frag + size_t(l) * kLayerFrags * kFrag, X, wave, acc);
    __syncthreads(); // every wave has read this layer's input
    uint32_t mask[kI];
    store_relu<kI, kTrain>(acc, X, wave, mask);
    if constexpr (kTrain)
#pragma unroll
      for (uint32_t i = 0; i < kI; ++i)
        a.masks[mask0 + size_t(l) * 256u * kI + i] = mask[i];
    __syncthreads();
  }
  // output layer, wave w on rows 32 w: rows are the A operand, columns 16..31
  // of the weight fragments are zero
  if (wave < kI) {
    const uint16_t *wp = a.w_frag + size_t(kHidden) * kLayerFrags * kFrag + lane * 8u;
    f32x16_t o;
#pragma unroll
    for (int r = 0; r < 16; ++r)
      o[r] = 0.f;
    bf16x8_t wq[kKSteps];
#pragma unroll
    for (uint32_t ks = 0; ks < kKSteps; ++ks)
      wq[ks] = *reinterpret_cast<const bf16x8_t *>(wp + ks * kFrag);
#pragma unroll
    for (uint32_t ks = 0; ks < kKSteps; ++ks) {
      const bf16x8_t x = *reinterpret_cast<const bf16x8_t *>(
          X + (wave * 32u + l32) * kXStride + ks * 16u + khalf);
      o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, wq[ks], o, 0, 0, 0);
    }
    float loss = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const uint32_t row = wave * 32u + (r / 4) * 8u + (lane >> 5) * 4u + (r % 4);
      if constexpr (kTrain) {
        // relative L2 on three outputs, the prediction held constant in the
        // denominator; lane l32 is output l32
        uint16_t d = 0;
        if (l32 < kOut && row0 + row < a.n) {
          const float inv = 1.f / (3.f * float(a.n));
          const float p = o[r], t = a.targ[size_t(row_of[row]) * kOut + l32];
          const float den = p * p + 0.01f, e = p - t;
          loss += e * e / den * inv;
          d = f2bf(2.f * e / den * inv);
        }
        D[row * kDStride + l32] = d;
      } else if (l32 < kOut) {
        a.pred[size_t(row0 + row) * kOut + l32] = o[r];
      }
    }
    if constexpr (kTrain) {
      for (int off = 32; off >= 1; off >>= 1)
        loss += __shfl_xor(loss, off, 64);
      if (lane == 0)
        wave_loss[wave] = loss;
    }
  }
  if constexpr (kTrain) {
    __syncthreads();
    if (threadIdx.x == 0) {
      float s = wave_loss[0];
      for (uint32_t i = 1; i < kI; ++i)
        s += wave_loss[i];
      a.loss_part[blockIdx.x] = s;
    }
    // output layer's weight gradient of this tile: acc is 32 inputs x 32
    // outputs, lanes 0..2 of each half hold outputs 0..2 (the others are zero)
#pragma unroll
    for (uint32_t j = 0; j < 2; ++j) {
      f32x16_t o;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[r] = 0.f;
#pragma unroll
      for (uint32_t rb = 0; rb < 2 * kI; ++rb)
        o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(column_frag(X, kXStride, rb, 2 * wave + j),
                                                    column_frag(D, kDStride, rb, 0), o, 0, 0, 0);
      if (l32 < kOut) {
        float *dst = a.out_part + (size_t(blockIdx.x) * kOut + l32) * kWidth + wave * 64u +
                     j * 32u + (lane >> 5) * 4u;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4 *>(dst + 8 * q) =
              make_float4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
      }
    }
    // gradient of the last hidden layer's outputs: K = 16 outputs, one step
    {
      const uint16_t *wp =
          a.wt_frag + size_t(kHidden - 1) * kLayerFrags * kFrag + 2 * wave * kFrag + lane * 8u;
#pragma unroll
      for (uint32_t i = 0; i < kI; ++i) {
        const bf16x8_t d =
            *reinterpret_cast<const bf16x8_t *>(D + (i * 32u + l32) * kDStride + khalf);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) {
          f32x16_t z;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            z[r] = 0.f;
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              *reinterpret_cast<const bf16x8_t *>(wp + j * kFrag), d, z, 0, 0, 0);
        }
      }
    }
#pragma unroll 1
    for (uint32_t l = kHidden; l-- > 0;) {
      // acc: gradient of layer l's outputs before its ReLU's mask
      uint32_t mask[kI];
#pragma unroll
      for (uint32_t i = 0; i < kI; ++i)
        mask[i] = a.masks[mask0 + size_t(l) * 256u * kI + i];
      __syncthreads(); // every wave has read the previous tile contents
      store_masked<kI>(acc, X, wave, mask);
      __syncthreads();
      store_column_frags<kI>(X, a.g_frag + l * a.layer_stride + frag0, wave);
      if (l)
        layer_products<kI>(a.wt_frag + size_t(l - 1) * kLayerFrags * kFrag, X, wave, acc);
    }
  }
}

// A tile's fixed costs (weights from L2, 12 barriers' latencies) favour many
// rows, the chip's 256 CUs many tiles. Training step, us, tiles of 32 / 64 /
// 128 rows: 3,001 rows 60 / 69 / 93; 16,384: 93 / 95 / 117; 24,576: 113 / 113 /
// 131; 32,768: 151 / 142 / 157; 49,152: 210+ / 203 / 210; 65,536: 313 / 276 /
// 267 (all with cached stores and loads). Inference: 4,096 rows 12 / 17 / 26; 16,384: 20 / 18 / 27; 65,536: 66 /
// 52 / 45; 2^20: 879 / 677 / 607.
uint32_t mlp_tile_rows(uint32_t rows_pad) {
  return rows_pad < kStreamRows ? 32u : rows_pad < 57344u ? 64u : 128u;
}

template <uint32_t kI> static hipError_t launch_tile(const MlpTileArgs &a, uint32_t rows_pad,
                                                     bool train, hipStream_t s) {
  const dim3 grid(rows_pad / (32 * kI));
  if (train)
    hipLaunchKernelGGL((k_mlp_tile<kI, true>), grid, dim3(256), tile_lds<kI>(true), s, a);
  else
    hipLaunchKernelGGL((k_mlp_tile<kI, false>), grid, dim3(256), tile_lds<kI>(false), s, a);
  return hipGetLastError();
}

hipError_t launch_mlp_tile(const MlpTileArgs &a, uint32_t rows_pad, bool train, hipStream_t s) {
  if (rows_pad % kRowAlign || a.n > rows_pad)
    return hipErrorInvalidValue;
  if (rows_pad == 0)
    return hipSuccess;
  const uint32_t rows = mlp_tile_rows(rows_pad);
  return rows == 32   ? launch_tile<1>(a, rows_pad, train, s)
         : rows == 64 ? launch_tile<2>(a, rows_pad, train, s)
                      : launch_tile<4>(a, rows_pad, train, s);
}

// ---------------------------------------------------------------------------
// Weight gradients of the hidden layers: dW_l[out][in] = sum over rows of
// G_l[row][out] A_l[row][in], split over the rows. One workgroup of 8 waves
// computes a whole 256 x 256 partial (wave: 128 outputs x 64 inputs), so both
// operands are read from memory exactly once. Stages of 32 rows (32 KB, both
// operands contiguous in memory) go through registers two stages ahead into a
// double-buffered LDS tile. Bound by HBM: 65,536 rows read 0.40 GB and write
// 66 MB of partials in 82 us, 5.7 TB/s where a large copy reaches 4.7 (108 us
// with cached loads; 128 x 128 tiles and 128 splits took 140 us, and 43 us to
// sum).
// The first blocks of the grid do the small sums: the output layer's partial
// gradients (one block per output) and the loss.
// ---------------------------------------------------------------------------
constexpr uint32_t kWgExtra = kOut + 1;

__device__ __forceinline__ void sum_tiles(const MlpWgradArgs &a) {
  __shared__ double red[512];
  const uint32_t t = threadIdx.x;
  double s = 0.0;
  if (blockIdx.x < kOut) {
    // two halves of the tiles per column
    const uint32_t col = t & 255u;
#pragma unroll 8
    for (uint32_t i = t >> 8; i < a.tiles; i += 2)
      s += double(a.out_part[(size_t(i) * kOut + blockIdx.x) * kWidth + col]);
    red[t] = s;
    __syncthreads();
    if (t < 256)
      a.out_grad[blockIdx.x * kWidth + t] = float(red[t] + red[t + 256]);
  } else {
    for (uint32_t i = t; i < a.tiles; i += 512)
      s += double(a.loss_part[i]);
    red[t] = s;
    __syncthreads();
    for (uint32_t off = 256; off >= 1; off >>= 1) {
      if (t < off)
        red[t] += red[t + off];
      __syncthreads();
    }
    if (t == 0)
      *a.loss = float(red[0]);
  }
}

template <bool kStream>
__global__ __launch_bounds__(512, 2) void k_mlp_wgrad(MlpWgradArgs a) {
  if (blockIdx.x < kWgExtra) { // whole block
    sum_tiles(a);
    return;
  }
  constexpr uint32_t kStage = 2 * kColBlocks * kFrag; // bf16 of one operand's stage
  __shared__ __attribute__((aligned(16))) uint16_t buf[2][2 * kStage];
  const uint32_t b = blockIdx.x - kWgExtra;
  const uint32_t l = b / a.splits, z = b % a.splits;
  const uint32_t stages = a.rows_pad / 32u;
  const uint32_t s0 = uint32_t(uint64_t(stages) * z / a.splits);
  const uint32_t s1 = uint32_t(uint64_t(stages) * (z + 1) / a.splits);
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint32_t wm = wave >> 2, wn = wave & 3u;
  const uint4 *g = reinterpret_cast<const uint4 *>(a.g_frag + l * a.layer_stride);
  const uint4 *x = reinterpret_cast<const uint4 *>(a.a_frag + l * a.layer_stride);
  f32x16_t acc[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0.f;
  // a stage past the last is clamped to it (loaded, not used), so
  // that the loads stay unconditional
  struct Regs {
    uint4 g0, g1, x0, x1;
  };
  auto fetch = [&](uint32_t s) __attribute__((always_inline)) {
    const size_t o = size_t(min(s, stages - 1)) * (kStage / 8) + t;
    if constexpr (kStream) {
      auto load = [](const uint4 *p) __attribute__((always_inline)) {
        return __builtin_bit_cast(
            uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p)));
      };
      return Regs{load(g + o), load(g + o + 512), load(x + o), load(x + o + 512)};
    } else {
      return Regs{g[o], g[o + 512], x[o], x[o + 512]};
    }
  };
  Regs v0 = fetch(s0), v1 = fetch(s0 + 1);
  auto step = [&](uint32_t s, Regs &r, uint16_t *tile) __attribute__((always_inline)) {
    uint4 *d = reinterpret_cast<uint4 *>(tile);
    d[t] = r.g0;
    d[t + 512] = r.g1;
    d[t + 1024] = r.x0;
    d[t + 1536] = r.x1;
    __syncthreads();
    r = fetch(s + 2);
#pragma unroll
    for (uint32_t rb = 0; rb < 2; ++rb) {
      const uint16_t *gp = tile + (rb * kColBlocks + 4 * wm) * kFrag + lane * 8u;
      const uint16_t *xp = tile + kStage + (rb * kColBlocks + 2 * wn) * kFrag + lane * 8u;
      bf16x8_t ga[4], xb[2];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ga[i] = *reinterpret_cast<const bf16x8_t *>(gp + i * kFrag);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        xb[j] = *reinterpret_cast<const bf16x8_t *>(xp + j * kFrag);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ga[i], xb[j], acc[i][j], 0, 0, 0);
    }
  };
  // A wave that passes stage s's barrier has read stage s - 2 from the same
  // buffer before stage s - 1's, so one barrier per stage is enough.
  for (uint32_t s = s0; s < s1; s += 2) {
    step(s, v0, buf[0]);
    if (s + 1 < s1)
      step(s + 1, v1, buf[1]);
  }
  float *dst = a.part + (size_t(l) * a.splits + z) * kWidth * kWidth;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t out = wm * 128u + i * 32u + (r / 4) * 8u + (lane >> 5) * 4u + (r % 4);
        dst[size_t(out) * kWidth + wn * 64u + j * 32u + (lane & 31u)] = acc[i][j][r];
      }
}

// One workgroup per CU for the six layers together on a 256-CU chip, at least
// 128 rows (4 stages) each.
uint32_t mlp_wgrad_splits(uint32_t rows_pad) {
  const uint32_t most = (256u - kWgExtra) / kHidden, s = (rows_pad + 127u) / 128u;
  return s < 1u ? 1u : s < most ? s : most;
}

hipError_t launch_mlp_wgrad(const MlpWgradArgs &a, hipStream_t s) {
  if (a.rows_pad % kRowAlign || a.splits == 0)
    return hipErrorInvalidValue;
  const dim3 grid(kWgExtra + kHidden * a.splits);
  if (a.rows_pad >= kStreamRows)
    hipLaunchKernelGGL(k_mlp_wgrad<true>, grid, dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL(k_mlp_wgrad<false>, grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Update: one block per 8 outputs x 64 inputs of a layer sums the splits
// (wave w takes splits w, w + 4, ..; then the waves' sums in order), applies
// Adam and writes the BF16 copies: row-major (inputs in the kernels' column
// order) and both fragment orders, one 16-byte store per 8 values.
// ---------------------------------------------------------------------------
template <int kMode>
__global__ __launch_bounds__(256) void k_mlp_update(MlpUpdateArgs a) {
  __shared__ float red[4][8][64];
  __shared__ __attribute__((aligned(16))) uint16_t wb[8][64];
  constexpr uint32_t kBlocks = (kWidth / 8) * (kWidth / 64); // per hidden layer
  const uint32_t l = min(blockIdx.x / kBlocks, kHidden);
  const uint32_t b = blockIdx.x - l * kBlocks;
  const uint32_t o0 = b / 4 * 8, c0 = b % 4 * 64;
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  if constexpr (kMode != kUpdatePack) {
    float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (l < kHidden) {
      const float *p = a.part + size_t(l) * a.splits * kWidth * kWidth + size_t(o0) * kWidth +
                       c0 + lane;
#pragma unroll 2
      for (uint32_t z = wave; z < a.splits; z += 4)
#pragma unroll
        for (uint32_t r = 0; r < 8; ++r)
          sum[r] += p[(size_t(z) * kWidth + r) * kWidth];
    } else if (wave == 0 && o0 == 0) {
#pragma unroll
      for (uint32_t r = 0; r < kOut; ++r)
        sum[r] = a.out_grad[r * kWidth + c0 + lane];
    }
#pragma unroll
    for (uint32_t r = 0; r < 8; ++r)
      red[wave][r][lane] = sum[r];
    __syncthreads();
  }
  const uint32_t r = t / 32u;
#pragma unroll
  for (uint32_t k = 0; k < 2; ++k) {
    const uint32_t c = (t % 32u) + 32u * k;
    const uint32_t col = l == 0 ? outer_column(c0 + c) : c0 + c;
    const size_t i = size_t(l) * kWidth * kWidth + size_t(o0 + r) * kWidth + col;
    float gi = 0.f;
    if constexpr (kMode != kUpdatePack)
      gi = ((red[0][r][c] + red[1][r][c]) + red[2][r][c]) + red[3][r][c];
    if constexpr (kMode == kUpdateGradient) {
      a.grad[i] = gi;
    } else if constexpr (kMode == kUpdateAdam) {
      const float mi = a.beta1 * a.m[i] + (1.f - a.beta1) * gi;
      const float vi = a.beta2 * a.v[i] + (1.f - a.beta2) * gi * gi;
      a.m[i] = mi;
      a.v[i] = vi;
      const float wi = a.w[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
      a.w[i] = wi;
      wb[r][c] = f2bf(wi);
    } else {
      wb[r][c] = f2bf(a.w[i]);
    }
  }
  if constexpr (kMode != kUpdateGradient) {
    __syncthreads();
    if (t < 64) {
      const uint32_t o = o0 + t / 8, c = c0 + 8 * (t % 8);
      const uint4 v = *reinterpret_cast<const uint4 *>(&wb[t / 8][8 * (t % 8)]);
      *reinterpret_cast<uint4 *>(a.w_rows + size_t(l) * kWidth * kWidth + size_t(o) * kWidth +
                                 c) = v;
      const size_t f = size_t(l) * kLayerFrags + (l < kHidden ? (o / 32) * kKSteps : 0) + c / 16;
      *reinterpret_cast<uint4 *>(a.w_frag + f * kFrag + (o % 32 + 32 * (c / 8 % 2)) * 8) = v;
    } else if (t < 128 && l >= 1) {
      const uint32_t c = c0 + lane;
      uint32_t v[4];
#pragma unroll
      for (uint32_t k = 0; k < 4; ++k)
        v[k] = uint32_t(wb[2 * k][lane]) | (uint32_t(wb[2 * k + 1][lane]) << 16);
      const size_t f = size_t(l - 1) * kLayerFrags +
                       (l < kHidden ? (c / 32) * kKSteps + o0 / 16 : c / 32);
      *reinterpret_cast<uint4 *>(a.wt_frag + f * kFrag + (c % 32 + 32 * (o0 / 8 % 2)) * 8) =
          make_uint4(v[0], v[1], v[2], v[3]);
    }
  }
}

hipError_t launch_mlp_update(const MlpUpdateArgs &a, int mode, hipStream_t s) {
  const dim3 grid(kHidden * (kWidth / 8) * (kWidth / 64) + (kOutPad / 8) * (kWidth / 64));
  if (mode == kUpdateGradient)
    hipLaunchKernelGGL((k_mlp_update<kUpdateGradient>), grid, dim3(256), 0, s, a);
  else if (mode == kUpdateAdam)
    hipLaunchKernelGGL((k_mlp_update<kUpdateAdam>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_mlp_update<kUpdatePack>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

} // namespace mlp
} // namespace pt
