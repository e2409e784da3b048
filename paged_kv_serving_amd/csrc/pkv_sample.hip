// Greedy sampling on the device: the index of each logits row's maximum, with NumPy's argmax
// rules (ties resolve to the lowest index; a NaN beats every number and the first NaN wins), so
// only one int32 per row crosses PCIe instead of the whole vocabulary row.
#include <math.h>

#include "pkv_common.h"

namespace pkv {
namespace {

constexpr int kArgmaxLoads = 4;  // 16-byte loads in flight per thread

typedef float f32x4 __attribute__((ext_vector_type(4)));

// A candidate (value, index); index -1 marks "nothing above -inf seen".
struct Best {
  float value;
  int32_t index;
};

// True when candidate a is argmax-preferred over candidate b.
__device__ __forceinline__ bool beats(const Best& a, const Best& b) {
  if (a.index < 0) return false;
  if (b.index < 0) return true;
  const bool an = isnan(a.value);
  const bool bn = isnan(b.value);
  if (an != bn) return an;
  if (!an && a.value != b.value) return a.value > b.value;
  return a.index < b.index;  // equal values (or both NaN): the lower index
}

__device__ __forceinline__ Best shfl_xor_best(const Best& b, int mask) {
  Best o;
  o.value = __shfl_xor(b.value, mask);
  o.index = __shfl_xor(b.index, mask);
  return o;
}

// One workgroup per row. The row's 16-byte aligned body is read kArgmaxLoads vectors per thread at
// a time (each thread scans increasing indices, so a later element only wins by being strictly
// greater, or by being the first NaN); the up to three elements before and after it are merged.
// A row without any element above -inf is its first element's.
//
// Bound: short rows by the launch and the merge of the wavefronts, long ones by one CU's read rate
// (a row is one workgroup's), many rows by HBM. Measured, rows of an odd vocabulary starting off a
// 16-byte boundary: 64 rows of 50257 32.7 us with 256 threads and one 4-byte load in flight each,
// 9.2 with 1024 threads and four vectors, 5.8 with the scan's checks out of the full steps; 512 rows
// 69.5 -> 18.6 us.
template <int kThreads>
__global__ __launch_bounds__(kThreads) void greedy_kernel(int32_t* __restrict__ out, const float* __restrict__ logits,
                                                          int64_t row_stride, int32_t vocab) {
  constexpr int kWaves = kThreads / kWave;
  const int64_t row = blockIdx.x;
  const float* x = logits + row * row_stride;
  Best best{-INFINITY, -1};
  auto consider = [&](float v, int32_t i) {
    if (!(v <= best.value) && !isnan(best.value)) best = Best{v, i};
  };
  auto consider_vector = [&](const f32x4& v, int32_t i) {
    consider(v.x, i);
    consider(v.y, i + 1);
    consider(v.z, i + 2);
    consider(v.w, i + 3);
  };
  const int32_t to_line = static_cast<int32_t>((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / 4;
  const int32_t head = to_line < vocab ? to_line : vocab;  // elements before the aligned body
  const f32x4* body = reinterpret_cast<const f32x4*>(x + head);
  const int32_t quads = (vocab - head) / 4;
  int32_t q = threadIdx.x;
  for (; q + (kArgmaxLoads - 1) * kThreads < quads; q += kArgmaxLoads * kThreads) {
    f32x4 v[kArgmaxLoads];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) v[u] = body[q + u * kThreads];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) consider_vector(v[u], head + 4 * (q + u * kThreads));
  }
  if (q < quads) {  // the thread's last vectors, fewer than kArgmaxLoads
    f32x4 v[kArgmaxLoads - 1];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads - 1; ++u) v[u] = body[min(q + u * kThreads, quads - 1)];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads - 1; ++u) {
      if (q + u * kThreads < quads) consider_vector(v[u], head + 4 * (q + u * kThreads));
    }
  }
  // The elements outside the body, one thread each: merged, as they are not in scan order.
  const int32_t tail = head + 4 * quads;
  const int32_t outside = head + (vocab - tail);
  if (static_cast<int32_t>(threadIdx.x) < outside) {
    const int32_t t = static_cast<int32_t>(threadIdx.x);
    const int32_t i = t < head ? t : tail + (t - head);
    const Best other{x[i], x[i] == -INFINITY ? -1 : i};
    if (beats(other, best)) best = other;
  }
  // Merge within the wavefront, then across the wavefronts through LDS.
#pragma unroll
  for (int mask = kWave / 2; mask > 0; mask >>= 1) {
    const Best other = shfl_xor_best(best, mask);
    if (beats(other, best)) best = other;
  }
  __shared__ float s_value[kWaves];
  __shared__ int32_t s_index[kWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  if (lane == 0) {
    s_value[wave] = best.value;
    s_index[wave] = best.index;
  }
  __syncthreads();
  if (wave == 0) {
    Best total = lane < kWaves ? Best{s_value[lane], s_index[lane]} : Best{-INFINITY, -1};
#pragma unroll
    for (int mask = kWaves / 2; mask > 0; mask >>= 1) {
      const Best other = shfl_xor_best(total, mask);
      if (beats(other, total)) total = other;
    }
    if (lane == 0) out[row] = max(total.index, 0);
  }
}

}  // namespace
}  // namespace pkv

extern "C" int pkv_greedy_tokens(int32_t* token_ids, const float* logits, int64_t row_stride,
                                 int64_t num_rows, int64_t vocab_size, int device,
                                 void* stream) {
  using namespace pkv;
  if (num_rows < 0 || vocab_size < 1 || vocab_size > 0x7fffffff || row_stride < vocab_size) {
    return PKV_EINVAL;
  }
  if (num_rows == 0) return PKV_OK;
  if (!token_ids || !logits) return PKV_EINVAL;
  if (num_rows > 0x7fffffff) return PKV_EUNSUPPORTED;
  DeviceGuard guard(device);
  if (!guard.ok()) return PKV_EHIP;
  // Few wavefronts where a row has little to scan: each one more adds to the merge and, over many
  // rows, to the launch. Measured (us; 64 / 128 / 512 / 1024 threads): 16 rows of 512 2.98 / 3.01 /
  // - / 3.46, of 4099 4.14 / 3.66 / 3.78 / 4.17, of 8192 5.4 / 4.26 / 3.77 / 4.32, of 50257 20.3 /
  // 12.0 / 5.97 / 5.69; 2048 rows of 512 3.7 / 4.1 / - / 10.6, of 4099 7.1 / 6.8 / 10.8 / 17.3; 64
  // rows of 128256 56 / 32 / 13.3 / 10.3, 256 rows 67 / 38 / 21.7 / 22.6.
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(num_rows)), dim3(threads), 0,
                       static_cast<hipStream_t>(stream), token_ids, logits, row_stride, static_cast<int32_t>(vocab_size));
    return check_launch();
  };
  if (vocab_size <= 512) return launch(greedy_kernel<64>, 64);
  if (vocab_size <= 4096) return launch(greedy_kernel<128>, 128);
  if (vocab_size <= 32768 || num_rows > 128) return launch(greedy_kernel<512>, 512);
  return launch(greedy_kernel<1024>, 1024);
}
