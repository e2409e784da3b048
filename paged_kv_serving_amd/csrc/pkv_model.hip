// The elementwise and row-wise steps of the decoder's forward pass around the KV data path, each
// one launch instead of a chain of framework kernels: RMSNorm, optionally fused with the residual
// add that precedes it, the SwiGLU gate product, and the row gather of the embedding lookup and
// of the logits rows. The matrix products are rocBLAS/hipBLASLt GEMMs.
//
// Both follow the float32 expressions of the reference model (src/paged_kv_serving/engine/
// model.py:43-51) operation by operation. Products, quotients and square roots are IEEE float32
// operations on both sides (hipcc keeps float32 division and sqrtf correctly rounded by default),
// and the sum of squares is summed in another order (a wavefront tree here, pairwise blocks in
// NumPy). The exponential is the device's expf, which, like NumPy's float32 exp, is not correctly
// rounded, so silu agrees with the reference to a few units in the last place rather than bit for
// bit; the tests hold silu_mul to a relative 1e-6 (about 8 float32 ulp) of the reference's silu
// and rms_norm to 2e-6.
#include <math.h>

#include "pkv_common.h"

namespace pkv {
namespace {

constexpr int kNormThreads = 256;
constexpr int kNormRows = kNormThreads / kWave;  // one wavefront per row
constexpr int kGateThreads = 256;

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int mask = 32; mask > 0; mask >>= 1) x += __shfl_xor(x, mask);
  return x;
}

// Row r: h = hidden[r] (+ delta[r], written back to hidden[r] when delta is given), then
// out[r] = h / sqrt(mean(h * h) + eps) * weight. Lane l handles columns l, l + 64, ... and
// writes output column j only after the whole row's sum is known, so out may be hidden itself.
__global__ __launch_bounds__(kNormThreads) void rms_norm_kernel(
    float* out, int64_t out_stride, float* hidden, int64_t hidden_stride,
    const float* __restrict__ delta, int64_t delta_stride, const float* __restrict__ weight,
    int64_t num_rows, int32_t dim, float eps) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kNormRows + threadIdx.x / kWave;
  if (row >= num_rows) return;
  const int lane = threadIdx.x & (kWave - 1);
  float* h = hidden + row * hidden_stride;
  float squares = 0.f;
  if (delta != nullptr) {
    const float* d = delta + row * delta_stride;
    for (int j = lane; j < dim; j += kWave) {
      const float v = h[j] + d[j];
      h[j] = v;
      squares += v * v;
    }
  } else {
    for (int j = lane; j < dim; j += kWave) {
      const float v = h[j];
      squares += v * v;
    }
  }
  const float mean = wave_sum(squares) / static_cast<float>(dim);
  const float scale = sqrtf(mean + eps);
  float* o = out + row * out_stride;
  for (int j = lane; j < dim; j += kWave) o[j] = (h[j] / scale) * weight[j];
}

// The same with the row held in registers between the two passes over it: kRowThreads threads per
// row, each with up to kCache 16-byte vectors of it (vector i * kRowThreads + t), so the row is
// read and written once. Needs 16-byte aligned rows and dim <= 16 * kCache * kRowThreads / 4 floats.
//
// Bound: HBM (hidden and delta read, hidden and out written). A wavefront per row with 4-byte
// accesses kept too few bytes in flight and read the row twice. 1024 rows of 4096 with the residual
// add (67 MB) over buffers that rotate through 1 GB: 52.1 us, 256 threads a row 16.7 (4.0 TB/s).
// Over one set of buffers, which the 256 MB Infinity Cache holds between passes: 38-40 and 10-11.5.
template <int kRowThreads, int kCache>
__global__ __launch_bounds__(kRowThreads < kNormThreads ? kNormThreads : kRowThreads) void rms_norm_vec_kernel(
    float* out, int64_t out_stride, float* hidden, int64_t hidden_stride, const float* __restrict__ delta,
    int64_t delta_stride, const float* __restrict__ weight, int64_t num_rows, int32_t dim, float eps) {
  constexpr int kRows = kRowThreads < kNormThreads ? kNormThreads / kRowThreads : 1;
  constexpr int kRowWaves = kRowThreads / kWave;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + threadIdx.x / kRowThreads;
  if (row >= num_rows) return;  // whole wavefronts; with several wavefronts per row, whole workgroups
  const int t = threadIdx.x % kRowThreads;
  const int vectors = dim / 4;
  f32x4* h = reinterpret_cast<f32x4*>(hidden + row * hidden_stride);
  f32x4 x[kCache];
#pragma unroll
  for (int i = 0; i < kCache; ++i) {
    const int v = i * kRowThreads + t;
    x[i] = v < vectors ? h[v] : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (delta != nullptr) {
    const f32x4* d = reinterpret_cast<const f32x4*>(delta + row * delta_stride);
#pragma unroll
    for (int i = 0; i < kCache; ++i) {
      const int v = i * kRowThreads + t;
      if (v < vectors) {
        x[i] += d[v];
        h[v] = x[i];
      }
    }
  }
  float squares = 0.f;
#pragma unroll
  for (int i = 0; i < kCache; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) squares += x[i][e] * x[i][e];
  }
  squares = wave_sum(squares);
  if constexpr (kRowWaves > 1) {
    __shared__ float s_sum[kRowWaves];
    if (threadIdx.x % kWave == 0) s_sum[threadIdx.x / kWave] = squares;
    __syncthreads();
    squares = 0.f;
#pragma unroll
    for (int w = 0; w < kRowWaves; ++w) squares += s_sum[w];
  }
  const float scale = sqrtf(squares / static_cast<float>(dim) + eps);
  f32x4* o = reinterpret_cast<f32x4*>(out + row * out_stride);
  const f32x4* w4 = reinterpret_cast<const f32x4*>(weight);
#pragma unroll
  for (int i = 0; i < kCache; ++i) {
    const int v = i * kRowThreads + t;
    if (v < vectors) {
      const f32x4 w = w4[v];
      o[v] = f32x4{(x[i].x / scale) * w.x, (x[i].y / scale) * w.y, (x[i].z / scale) * w.z, (x[i].w / scale) * w.w};
    }
  }
}

__device__ __forceinline__ float silu_product(float g, float u) {
  const float sigmoid = 1.f / (1.f + expf(-fminf(fmaxf(g, -60.f), 60.f)));
  return (g * sigmoid) * u;
}

// out[r, j] = silu(gate[r, j]) * up[r, j], silu(x) = x * (1 / (1 + exp(-clip(x, -60, 60)))), four
// adjacent elements per thread. 2^lane_bits threads (all 256, or as many as a narrower row has
// vectors, rounded up) per row or chunk of a row. Grid: (chunks of a row, groups of rows), the rows
// beyond the grid's strided.
//
// Bound: HBM (gate and up read, out written). 1024 rows of 11008 (135 MB) over buffers that rotate
// through 1.6 GB: 35.6 us with one element per thread and a 64-bit division for its row, 26.2 with
// this (5.2 TB/s). Over one set of buffers, which the Infinity Cache mostly holds: 27.4 and 24.5.
// Narrow rows by the workgroups: 4096 rows of 64 took 3.93 us with a workgroup each, 2.54 with one
// element per thread.
__global__ __launch_bounds__(kGateThreads) void silu_mul_vec_kernel(float* __restrict__ out, int64_t out_stride,
                                                                    const float* __restrict__ gate,
                                                                    const float* __restrict__ up, int64_t in_stride,
                                                                    int64_t num_rows, int32_t vectors,
                                                                    int lane_bits) {
  const int lanes = 1 << lane_bits;
  const int64_t v = static_cast<int64_t>(blockIdx.x) * lanes + (threadIdx.x & (lanes - 1));
  if (v >= vectors) return;
  const int group = kGateThreads >> lane_bits;  // rows at a time
  for (int64_t r = static_cast<int64_t>(blockIdx.y) * group + (threadIdx.x >> lane_bits); r < num_rows;
       r += static_cast<int64_t>(gridDim.y) * group) {
    const f32x4 g = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(gate + r * in_stride) + v);
    const f32x4 u = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(up + r * in_stride) + v);
    reinterpret_cast<f32x4*>(out + r * out_stride)[v] =
        f32x4{silu_product(g.x, u.x), silu_product(g.y, u.y), silu_product(g.z, u.z), silu_product(g.w, u.w)};
  }
}

// The same one element at a time, for rows that are not 16-byte aligned and up to kGateSmall elements.
__global__ __launch_bounds__(kGateThreads) void silu_mul_kernel(float* __restrict__ out,
                                                                int64_t out_stride,
                                                                const float* __restrict__ gate,
                                                                const float* __restrict__ up,
                                                                int64_t in_stride, int64_t num_rows,
                                                                int32_t width) {
  const int64_t total = num_rows * width;
  for (int64_t e = static_cast<int64_t>(blockIdx.x) * kGateThreads + threadIdx.x; e < total;
       e += static_cast<int64_t>(gridDim.x) * kGateThreads) {
    const int64_t r = e / width;
    const int64_t j = e - r * width;
    const float g = gate[r * in_stride + j];
    const float u = up[r * in_stride + j];
    out[r * out_stride + j] = silu_product(g, u);
  }
}

// out[r] = src[index[r]] (float32 rows of `width`), or zeros when index[r] lies outside
// [0, src_rows). One wavefront per row; kVec: 16-byte accesses (both row starts aligned).
template <bool kVec>
__global__ __launch_bounds__(kNormThreads) void gather_rows_kernel(float* __restrict__ out, int64_t out_stride,
                                                                    const float* __restrict__ src,
                                                                    int64_t src_stride,
                                                                    const int64_t* __restrict__ index,
                                                                    int64_t num_rows, int32_t width,
                                                                    int64_t src_rows) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kNormRows + threadIdx.x / kWave;
  if (row >= num_rows) return;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t at = index[row];
  const bool ok = at >= 0 && at < src_rows;
  float* o = out + row * out_stride;
  const float* s = src + (ok ? at : 0) * src_stride;
  if constexpr (kVec) {
    for (int j = 4 * lane; j < width; j += 4 * kWave) {
      const float4 v = ok ? *reinterpret_cast<const float4*>(s + j) : make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<float4*>(o + j) = v;
    }
  } else {
    for (int j = lane; j < width; j += kWave) o[j] = ok ? s[j] : 0.f;
  }
}

// The int32 metadata of a call over one sequence: out = positions, one zero per query (its sequence
// index), the table and the context length. One launch of a few hundred bytes in place of four
// framework kernels (two casts, two fills): the 1 x 256-key call 36.5 -> 23.7 us, which the host's
// launches bound.
template <typename PositionT, typename BlockT>
__global__ __launch_bounds__(kNormThreads) void sequence_metadata_kernel(int32_t* __restrict__ out,
                                                                         const PositionT* __restrict__ positions,
                                                                         int64_t num_queries,
                                                                         const BlockT* __restrict__ table,
                                                                         int64_t num_blocks, int32_t context_len) {
  const int64_t total = 2 * num_queries + num_blocks + 1;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * kNormThreads + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * kNormThreads) {
    int32_t v = 0;
    if (i < num_queries) {
      v = static_cast<int32_t>(positions[i]);
    } else if (i >= 2 * num_queries) {
      const int64_t b = i - 2 * num_queries;
      v = b < num_blocks ? static_cast<int32_t>(table[b]) : context_len;
    }
    out[i] = v;
  }
}

}  // namespace
}  // namespace pkv

extern "C" int pkv_sequence_metadata(int32_t* out, const void* positions, int32_t position_bytes,
                                     int64_t num_queries, const void* block_table, int32_t table_bytes,
                                     int64_t num_blocks, int32_t context_len, int device, void* stream) {
  using namespace pkv;
  if (num_queries < 0 || num_blocks < 0 || (position_bytes != 4 && position_bytes != 8) ||
      (table_bytes != 4 && table_bytes != 8) || !out || (num_queries > 0 && !positions) ||
      (num_blocks > 0 && !block_table)) {
    return PKV_EINVAL;
  }
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  (void)hipGetLastError();
  const int64_t wanted = (2 * num_queries + num_blocks + 1 + kNormThreads - 1) / kNormThreads;
  const dim3 grid(static_cast<uint32_t>(wanted < 1024 ? wanted : 1024));
  auto launch = [&](auto position, auto block) {
    using P = decltype(position);
    using B = decltype(block);
    hipLaunchKernelGGL((sequence_metadata_kernel<P, B>), grid, dim3(kNormThreads), 0,
                       static_cast<hipStream_t>(stream), out, static_cast<const P*>(positions), num_queries,
                       static_cast<const B*>(block_table), num_blocks, context_len);
    return check_launch();
  };
  if (position_bytes == 8) return table_bytes == 8 ? launch(int64_t{}, int64_t{}) : launch(int64_t{}, int32_t{});
  return table_bytes == 8 ? launch(int32_t{}, int64_t{}) : launch(int32_t{}, int32_t{});
}

extern "C" int pkv_gather_rows(float* out, int64_t out_stride, const float* src, int64_t src_stride,
                               int64_t src_rows, const int64_t* index, int64_t num_rows, int32_t width,
                               int device, void* stream) {
  using namespace pkv;
  if (num_rows < 0 || width < 1 || src_rows < 0 || out_stride < width || src_stride < width) return PKV_EINVAL;
  if (num_rows == 0) return PKV_OK;
  if (!out || !src || !index) return PKV_EINVAL;
  const int64_t blocks = (num_rows + kNormRows - 1) / kNormRows;
  if (blocks > 0x7fffffff) return PKV_EUNSUPPORTED;
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  (void)hipGetLastError();
  const bool vec = width % 4 == 0 && out_stride % 4 == 0 && src_stride % 4 == 0 && aligned16(out) && aligned16(src);
  auto s = static_cast<hipStream_t>(stream);
  if (vec) {
    hipLaunchKernelGGL(gather_rows_kernel<true>, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, s, out,
                       out_stride, src, src_stride, index, num_rows, width, src_rows);
  } else {
    hipLaunchKernelGGL(gather_rows_kernel<false>, dim3(static_cast<uint32_t>(blocks)), dim3(kNormThreads), 0, s, out,
                       out_stride, src, src_stride, index, num_rows, width, src_rows);
  }
  return check_launch();
}

extern "C" int pkv_rms_norm(float* out, int64_t out_stride, float* hidden, int64_t hidden_stride,
                            const float* delta, int64_t delta_stride, const float* weight,
                            int64_t num_rows, int32_t dim, float eps, int device, void* stream) {
  using namespace pkv;
  if (num_rows < 0 || dim < 1 || out_stride < dim || hidden_stride < dim ||
      (delta != nullptr && delta_stride < dim) || !(eps >= 0.f)) {
    return PKV_EINVAL;
  }
  if (num_rows == 0) return PKV_OK;
  if (!out || !hidden || !weight) return PKV_EINVAL;
  const int64_t blocks = (num_rows + kNormRows - 1) / kNormRows;
  if (blocks > 0x7fffffff) return PKV_EUNSUPPORTED;
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  (void)hipGetLastError();
  auto s = static_cast<hipStream_t>(stream);
  // 16-byte accesses where every row allows them. A wavefront per row holds 1024 floats in four
  // vectors a lane, 256 threads 4096, 1024 threads 16384; longer rows take the two-pass kernel, and
  // so do rows of at most 64, one element a lane (1024 rows of 64 with the residual add 2.56 us
  // against 2.68, of 32 2.56 against 2.97; of 100 3.13 against 2.94).
  const bool vec = dim > 64 && dim % 4 == 0 && out_stride % 4 == 0 && hidden_stride % 4 == 0 && aligned16(out) &&
                   aligned16(hidden) && aligned16(weight) &&
                   (delta == nullptr || (delta_stride % 4 == 0 && aligned16(delta)));
  auto launch = [&](auto kernel, int64_t groups, int threads) {
    if (groups > 0x7fffffff) return static_cast<int>(PKV_EUNSUPPORTED);
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(groups)), dim3(threads), 0, s, out, out_stride, hidden,
                       hidden_stride, delta, delta_stride, weight, num_rows, dim, eps);
    return check_launch();
  };
  if (vec && dim <= 256) return launch(rms_norm_vec_kernel<64, 1>, blocks, kNormThreads);
  if (vec && dim <= 1024) return launch(rms_norm_vec_kernel<64, 4>, blocks, kNormThreads);
  if (vec && dim <= 4096) return launch(rms_norm_vec_kernel<256, 4>, num_rows, 256);
  if (vec && dim <= 16384) return launch(rms_norm_vec_kernel<1024, 4>, num_rows, 1024);
  return launch(rms_norm_kernel, blocks, kNormThreads);
}

extern "C" int pkv_silu_mul(float* out, int64_t out_stride, const float* gate, const float* up,
                            int64_t in_stride, int64_t num_rows, int32_t width, int device,
                            void* stream) {
  using namespace pkv;
  if (num_rows < 0 || width < 1 || out_stride < width || in_stride < width) return PKV_EINVAL;
  if (num_rows == 0) return PKV_OK;
  if (!out || !gate || !up) return PKV_EINVAL;
  auto s = static_cast<hipStream_t>(stream);
  // Up to 2^17 elements a call is latency: one per thread measures 2.27-2.36 us where four measure
  // 2.33-2.41 (16 rows of 1000, 256 of 512); 256 rows of 1000 2.5 both.
  constexpr int64_t kGateSmall = 1 << 17;
  const bool vec = width % 4 == 0 && out_stride % 4 == 0 && in_stride % 4 == 0 && aligned16(out) && aligned16(gate) &&
                   aligned16(up) && num_rows * width > kGateSmall;
  if (vec) {
    DeviceGuard guard(device);
    if (!guard.ok()) return PKV_EHIP;
    (void)hipGetLastError();
    const int32_t vectors = width / 4;
    int lane_bits = 0;
    while ((1 << lane_bits) < kGateThreads && (1 << lane_bits) < vectors) ++lane_bits;
    const int64_t groups = (num_rows + (kGateThreads >> lane_bits) - 1) / (kGateThreads >> lane_bits);
    const dim3 grid(static_cast<uint32_t>((vectors + kGateThreads - 1) / kGateThreads),
                    static_cast<uint32_t>(groups < 65535 ? groups : 65535));
    hipLaunchKernelGGL(silu_mul_vec_kernel, grid, dim3(kGateThreads), 0, s, out, out_stride, gate, up, in_stride,
                       num_rows, vectors, lane_bits);
    return check_launch();
  }
  const int64_t total = num_rows * width;
  const int64_t wanted = (total + kGateThreads - 1) / kGateThreads;
  const uint32_t blocks = static_cast<uint32_t>(wanted < 65536 ? wanted : 65536);
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  (void)hipGetLastError();
  hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(kGateThreads), 0, s, out, out_stride, gate, up, in_stride, num_rows, width);
  return check_launch();
}
