// Greedy sampling on the device: the index of each logits row's maximum, with NumPy's argmax
// rules (ties resolve to the lowest index; a NaN beats every number and the first NaN wins), so
// only one int32 per row crosses PCIe instead of the whole vocabulary row.
#include <math.h>

#include "pkv_common.h"

namespace pkv {
namespace {

constexpr int kArgmaxThreads = 1024;
constexpr int kArgmaxWaves = kArgmaxThreads / kWave;
constexpr int kArgmaxLoads = 4;  // 16-byte loads in flight per thread

typedef float f32x4 __attribute__((ext_vector_type(4)));

// A candidate (value, index); index -1 marks "no element seen".
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
//
// Bound: latency and one CU's read rate, as a row is one workgroup's. With 256 threads, one 4-byte
// load in flight each (rows of an odd vocabulary start off a 16-byte boundary), 64 rows of 50257
// took 60.5 us a call; 1024 threads with four vectors in flight take 9.6 us.
__global__ __launch_bounds__(kArgmaxThreads) void greedy_kernel(int32_t* __restrict__ out,
                                                                const float* __restrict__ logits,
                                                                int64_t row_stride, int32_t vocab) {
  const int64_t row = blockIdx.x;
  const float* x = logits + row * row_stride;
  Best best{0.f, -1};
  auto consider = [&](float v, int32_t i) {
    if (best.index < 0 || (isnan(v) && !isnan(best.value)) || v > best.value) best = Best{v, i};
  };
  const int32_t to_line = static_cast<int32_t>((16 - (reinterpret_cast<uintptr_t>(x) & 15)) & 15) / 4;
  const int32_t head = to_line < vocab ? to_line : vocab;  // elements before the aligned body
  const f32x4* body = reinterpret_cast<const f32x4*>(x + head);
  const int32_t quads = (vocab - head) / 4;
  for (int32_t q0 = threadIdx.x; q0 < quads; q0 += kArgmaxLoads * kArgmaxThreads) {
    f32x4 v[kArgmaxLoads];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) v[u] = body[min(q0 + u * kArgmaxThreads, quads - 1)];
#pragma unroll
    for (int u = 0; u < kArgmaxLoads; ++u) {
      const int32_t q = q0 + u * kArgmaxThreads;
      if (q >= quads) break;
      const int32_t i = head + 4 * q;
      consider(v[u].x, i);
      consider(v[u].y, i + 1);
      consider(v[u].z, i + 2);
      consider(v[u].w, i + 3);
    }
  }
  // The elements outside the body, one thread each: merged, as they are not in scan order.
  const int32_t tail = head + 4 * quads;
  const int32_t outside = head + (vocab - tail);
  if (static_cast<int32_t>(threadIdx.x) < outside) {
    const int32_t t = static_cast<int32_t>(threadIdx.x);
    const int32_t i = t < head ? t : tail + (t - head);
    const Best other{x[i], i};
    if (beats(other, best)) best = other;
  }
  // Merge within the wavefront, then across the wavefronts through LDS.
#pragma unroll
  for (int mask = kWave / 2; mask > 0; mask >>= 1) {
    const Best other = shfl_xor_best(best, mask);
    if (beats(other, best)) best = other;
  }
  __shared__ float s_value[kArgmaxWaves];
  __shared__ int32_t s_index[kArgmaxWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  if (lane == 0) {
    s_value[wave] = best.value;
    s_index[wave] = best.index;
  }
  __syncthreads();
  if (wave == 0) {
    Best total = lane < kArgmaxWaves ? Best{s_value[lane], s_index[lane]} : Best{0.f, -1};
#pragma unroll
    for (int mask = kArgmaxWaves / 2; mask > 0; mask >>= 1) {
      const Best other = shfl_xor_best(total, mask);
      if (beats(other, total)) total = other;
    }
    if (lane == 0) out[row] = total.index;
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
  hipLaunchKernelGGL(greedy_kernel, dim3(static_cast<uint32_t>(num_rows)), dim3(kArgmaxThreads), 0,
                     static_cast<hipStream_t>(stream), token_ids, logits, row_stride, static_cast<int32_t>(vocab_size));
  return check_launch();
}
