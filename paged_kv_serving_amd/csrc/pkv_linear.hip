// The matrix products of a small decoder with the row-wise steps around them in one launch each:
// RMSNorm of the input rows before the product, and after it the residual add, RoPE with the
// slot-mapped append, or the SwiGLU gate. At the sizes this serves (up to 512 rows, d_model up
// to 256) every launch is latency: a library product takes 4.5-6.7 us, a norm 3.2, RoPE + append
// 3.8, a gate 2.7, whatever they compute, and a layer had eight of them beside attention's passes.
//
// Products are float32 (v_mfma_f32_16x16x4f32). One workgroup computes 16 rows x 64 columns, a
// wavefront 16 of the columns, so that even 128 rows of 384 columns are 48 workgroups. The 16 input
// rows are staged whole in LDS (padded by 4 floats: the operand reads of 16 rows hit every bank
// once); the weights are read once per workgroup straight into registers, 128 of the depth at a
// time, the first of them before the rows are staged. Measured, one iteration of a 4-layer decoder
// (d_model 128, 128 rows), logits back on the host: 286 us with the library's products and the
// separate steps, 207 us with these (6 launches a layer with both attention passes, in place of 10).
#include <math.h>

#include "pkv_common.h"

namespace pkv {
namespace {

constexpr int kRows = 16;      // rows per workgroup
constexpr int kCols = 64;      // columns per workgroup
constexpr int kLinearThreads = 256;
constexpr int kDepthStep = 16;   // depth of one operand read (four products)
constexpr int kAheadSteps = 8;   // steps whose weights are in registers at a time

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename PoolT>
__device__ __forceinline__ void store_pool(PoolT* p, float x);
template <>
__device__ __forceinline__ void store_pool<float>(float* p, float x) {
  *p = x;
}
template <>
__device__ __forceinline__ void store_pool<uint16_t>(uint16_t* p, float x) {
  *p = static_cast<uint16_t>(f32_to_bf16_bits(x));
}

// Column of the weights that column j (0..63) of workgroup column tile `tile` is. The gate form
// takes 32 gate columns and the 32 up columns they multiply.
template <int kKind>
__device__ __forceinline__ int weight_column(const pkv_linear& a, int tile, int j) {
  if constexpr (kKind == PKV_LINEAR_SWIGLU) {
    const int col = tile * (kCols / 2) + (j & (kCols / 2 - 1));
    return col < a.cols ? (j < kCols / 2 ? col : a.cols + col) : -1;
  } else {
    const int col = tile * kCols + j;
    return col < a.cols ? col : -1;
  }
}

template <int kKind, typename PoolT>
__global__ __launch_bounds__(kLinearThreads) void linear_kernel(const pkv_linear a) {
  constexpr bool kNorm = kKind != PKV_LINEAR_ADD;
  constexpr bool kTransposed = kKind == PKV_LINEAR_LOGITS;  // weights [cols, depth]
  extern __shared__ __align__(16) float s_rows[];           // [kRows][depth + 4]
  __shared__ float s_out[kRows][kCols + 4];
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int c = lane >> 4;
  const int n = lane & 15;
  const int tile = blockIdx.x;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * kRows;
  const int stride = a.depth + 4;
  const int steps = a.depth / kDepthStep;

  // Lane (c, n)'s weights of depth 16 s + 4 c + [0, 4) in column n of the wavefront's sixteen.
  const int col = weight_column<kKind>(a, tile, 16 * wave + n);
  const float* w = a.weights + (kTransposed ? static_cast<int64_t>(col < 0 ? 0 : col) * a.weight_stride + 4 * c
                                            : static_cast<int64_t>(4 * c) * a.weight_stride + (col < 0 ? 0 : col));
  f32x4 b[kAheadSteps];
  auto load_weights = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kAheadSteps; ++u) {
      const int s = min(s0 + u, steps - 1);
      if constexpr (kTransposed) {
        b[u] = *reinterpret_cast<const f32x4*>(w + s * kDepthStep);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) b[u][e] = w[static_cast<int64_t>(s * kDepthStep + e) * a.weight_stride];
      }
    }
  };
  load_weights(0);

  // Sixteen threads per input row stage it, and normalise their own elements in place.
  {
    const int64_t row = row0 + tid / 16;
    const int t = tid % 16;
    int64_t source = -1;  // -1: a row of zeros
    if (row < a.rows) {
      source = row;
      if constexpr (kKind == PKV_LINEAR_LOGITS) {
        source = a.row_index[row];
        if (source < 0 || source >= a.input_rows) source = -1;
      }
    }
    const float* in = a.input + (source < 0 ? 0 : source) * a.input_stride;
    float* s = s_rows + (tid / 16) * stride;
    float squares = 0.f;
    for (int k = 4 * t; k < a.depth; k += 64) {
      const f32x4 x = source >= 0 ? *reinterpret_cast<const f32x4*>(in + k) : f32x4{0.f, 0.f, 0.f, 0.f};
      *reinterpret_cast<f32x4*>(s + k) = x;
#pragma unroll
      for (int e = 0; e < 4; ++e) squares += x[e] * x[e];
    }
    if constexpr (kNorm) {
#pragma unroll
      for (int mask = 8; mask > 0; mask >>= 1) squares += __shfl_xor(squares, mask);
      // A row of zeros stays one, also with eps 0.
      const float scale = source >= 0 ? sqrtf(squares / static_cast<float>(a.depth) + a.eps) : 1.f;
      for (int k = 4 * t; k < a.depth; k += 64) {
        f32x4 x = *reinterpret_cast<const f32x4*>(s + k);
        const f32x4 g = *reinterpret_cast<const f32x4*>(a.norm_weight + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (x[e] / scale) * g[e];
        *reinterpret_cast<f32x4*>(s + k) = x;
      }
    }
  }
  __syncthreads();

  // Two chains of products, so that one does not wait for the other's result.
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  const float* rows = s_rows + n * stride + 4 * c;
  for (int s0 = 0; s0 < steps; s0 += kAheadSteps) {
    f32x4 held[kAheadSteps];
#pragma unroll
    for (int u = 0; u < kAheadSteps; ++u) held[u] = b[u];
    if (s0 + kAheadSteps < steps) load_weights(s0 + kAheadSteps);
#pragma unroll
    for (int u = 0; u < kAheadSteps; ++u) {
      if (s0 + u >= steps) break;  // uniform
      const f32x4 x = *reinterpret_cast<const f32x4*>(rows + (s0 + u) * kDepthStep);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[u & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], held[u][e], acc[u & 1], 0, 0, 0);
      }
    }
  }
  const f32x4 sum = acc[0] + acc[1];  // register r: row 4 c + r, column n of the wavefront's

  if constexpr (kKind == PKV_LINEAR_ADD || kKind == PKV_LINEAR_LOGITS) {
    if (col < 0) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t row = row0 + 4 * c + r;
      if (row >= a.rows) continue;
      float* o = a.output + row * a.output_stride + col;
      *o = kKind == PKV_LINEAR_ADD ? *o + sum[r] : sum[r];
    }
    return;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) s_out[4 * c + r][16 * wave + n] = sum[r];
  __syncthreads();
  const int64_t row = row0 + tid / 16;
  if (row >= a.rows) return;
  const float* out = s_out[tid / 16];
  if constexpr (kKind == PKV_LINEAR_SWIGLU) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = tid % 16 + 16 * i;
      const int column = tile * (kCols / 2) + j;
      if (column < a.cols) {
        const float g = out[j], u = out[j + kCols / 2];
        const float sigmoid = 1.f / (1.f + expf(-fminf(fmaxf(g, -60.f), 60.f)));
        a.output[row * a.output_stride + column] = (g * sigmoid) * u;
      }
    }
  }
  if constexpr (kKind == PKV_LINEAR_ROPE_APPEND) {
#pragma clang fp contract(off)
    // The tile holds whole heads (32 or 64 dimensions) of q, k and v; a thread takes two rotation
    // pairs of its row, each product and sum rounded on its own (as pkv_rope_append).
    const int64_t pos = a.positions[row];
    if (pos < 0 || pos >= a.table_rows) return;
    const int64_t slot = a.slots[row];
    const bool stored = slot >= 0 && slot < a.num_slots;
    const int half = a.head_dim / 2;
    const int model = a.num_heads * a.head_dim;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int pair = tid % 16 + 16 * i;
      const int lo = pair / half * a.head_dim + pair % half;  // column of the tile
      const int column = tile * kCols + lo;
      if (column >= a.cols) continue;
      const int part = column / model;  // 0: q, 1: k, 2: v
      const int within = column - part * model;
      float x = out[lo], y = out[lo + half];
      if (part < 2) {
        const float cs = a.cos_table[pos * half + pair % half], sn = a.sin_table[pos * half + pair % half];
        const float xc = x * cs, ys = y * sn, yc = y * cs, xs = x * sn;
        x = xc - ys;
        y = yc + xs;
      }
      if (part == 0) {
        a.output[row * a.output_stride + within] = x;
        a.output[row * a.output_stride + within + half] = y;
      } else if (stored) {
        PoolT* pool = static_cast<PoolT*>(part == 1 ? a.key_pool : a.value_pool) + slot * model + within;
        store_pool(pool, x);
        store_pool(pool + half, y);
      }
    }
  }
}

template <int kKind, typename PoolT>
int launch_linear(const pkv_linear& a, hipStream_t stream) {
  const int tile = kKind == PKV_LINEAR_SWIGLU ? kCols / 2 : kCols;
  const dim3 grid(static_cast<uint32_t>((a.cols + tile - 1) / tile), static_cast<uint32_t>((a.rows + kRows - 1) / kRows));
  const size_t bytes = static_cast<size_t>(kRows) * (a.depth + 4) * sizeof(float);
  hipLaunchKernelGGL((linear_kernel<kKind, PoolT>), grid, dim3(kLinearThreads), bytes, stream, a);
  return check_launch();
}

}  // namespace
}  // namespace pkv

extern "C" int pkv_linear_forward(const pkv_linear* args, int device, void* stream) {
  using namespace pkv;
  if (!args) return PKV_EINVAL;
  const pkv_linear& a = *args;
  if (a.rows < 0 || a.cols < 1 || a.depth < 1 || a.input_stride < a.depth || a.weight_stride < 1) return PKV_EINVAL;
  if (a.depth % kDepthStep != 0 || a.depth > PKV_LINEAR_MAX_DEPTH || a.rows > 65535LL * kRows) return PKV_EUNSUPPORTED;
  if (a.rows == 0) return PKV_OK;
  if (!a.input || !a.weights || !a.output) return PKV_EINVAL;
  if (!aligned16(a.input) || a.input_stride % 4 != 0) return PKV_EUNSUPPORTED;
  if (a.kind != PKV_LINEAR_ADD && (!a.norm_weight || !(a.eps >= 0.f))) return PKV_EINVAL;
  if (a.kind != PKV_LINEAR_ADD && !aligned16(a.norm_weight)) return PKV_EUNSUPPORTED;
  if (a.kind == PKV_LINEAR_LOGITS) {
    if (!a.row_index || a.input_rows < 0 || a.weight_stride < a.depth) return PKV_EINVAL;
    if (!aligned16(a.weights) || a.weight_stride % 4 != 0) return PKV_EUNSUPPORTED;
  } else if (a.weight_stride < (a.kind == PKV_LINEAR_SWIGLU ? 2LL * a.cols : a.cols)) {
    return PKV_EINVAL;
  }
  if (a.kind == PKV_LINEAR_ROPE_APPEND) {
    if (a.head_dim != 32 && a.head_dim != 64) return PKV_EUNSUPPORTED;
    if (a.num_heads < 1 || a.cols != 3 * static_cast<int64_t>(a.num_heads) * a.head_dim || !a.positions || !a.slots ||
        !a.cos_table || !a.sin_table || !a.key_pool || !a.value_pool || a.num_slots < 0 || a.table_rows < 0 ||
        a.output_stride < static_cast<int64_t>(a.num_heads) * a.head_dim) {
      return PKV_EINVAL;
    }
  } else if (a.output_stride < a.cols) {
    return PKV_EINVAL;
  }
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  (void)hipGetLastError();
  auto s = static_cast<hipStream_t>(stream);
  switch (a.kind) {
    case PKV_LINEAR_ADD:
      return launch_linear<PKV_LINEAR_ADD, float>(a, s);
    case PKV_LINEAR_SWIGLU:
      return launch_linear<PKV_LINEAR_SWIGLU, float>(a, s);
    case PKV_LINEAR_LOGITS:
      return launch_linear<PKV_LINEAR_LOGITS, float>(a, s);
    case PKV_LINEAR_ROPE_APPEND:
      if (a.pool_dtype == PKV_F32) return launch_linear<PKV_LINEAR_ROPE_APPEND, float>(a, s);
      if (a.pool_dtype == PKV_BF16) return launch_linear<PKV_LINEAR_ROPE_APPEND, uint16_t>(a, s);
      return PKV_EINVAL;
    default:
      return PKV_EINVAL;
  }
}
