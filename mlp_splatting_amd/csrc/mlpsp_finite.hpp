// A look through f32 arrays for what is not finite: a launch of its own, or a share of it done by another kernel's wavefronts.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"

namespace mlpsp {

typedef float scan_f32x4 __attribute__((ext_vector_type(4)));

// One read-only pass over up to 16 f32 arrays; flag[0] |= 1 if any element is NaN or infinite
// (training_wmma.cuh:24-60: one fused scan and one read-back instead of a reduction per tensor).
struct FiniteScanInputs {
  const float* pointers[16];
  long long lengths[16];
  int count;
};

// Bound by memory: 2.86 GB of inputs at 200,000 primitives 481 -> 411 us, 6.95 TB/s, against a load at a time in 8,192 blocks that
// come and go.  Eight loads on their way per thread and blocks that all run at once (512 blocks 419 us, 1,024 483, 2,048 455),
// past the caches (471 us with 512 blocks through them).
constexpr int kScanAhead = 8, kScanBlocks = 768;
// One thread's share: 16 bytes at first, first + stride, ...; with the whole wavefront.
__device__ __forceinline__ void finite_scan(const FiniteScanInputs& in, long long first, long long stride,
                                            int32_t* __restrict__ flag) {
  uint32_t most = 0u;                // the largest of the magnitudes, as bits: 0x7f800000 and more are not finite
  const auto look = [&](float v) { most = max(most, __float_as_uint(v) & 0x7fffffffu); };
  for (int t = 0; t < in.count; ++t) {
    const float* __restrict__ src = in.pointers[t];
    const long long n = in.lengths[t];
    // 16-byte loads over the aligned middle, scalar loads for the ragged ends
    const long long head = min(n, (long long)(((16 - (reinterpret_cast<uintptr_t>(src) & 15)) & 15) / 4));
    const long long quads = (n - head) / 4;
    const scan_f32x4* __restrict__ mid = reinterpret_cast<const scan_f32x4*>(src + head);
    long long i = first;
    for (; i + (kScanAhead - 1) * stride < quads; i += kScanAhead * stride) {
      scan_f32x4 v[kScanAhead];
#pragma unroll
      for (int k = 0; k < kScanAhead; ++k) v[k] = __builtin_nontemporal_load(mid + i + k * stride);
#pragma unroll
      for (int k = 0; k < kScanAhead; ++k) {
#pragma unroll
        for (int q = 0; q < 4; ++q) look(v[k][q]);
      }
    }
    for (; i < quads; i += stride) {
      const scan_f32x4 v = mid[i];
#pragma unroll
      for (int q = 0; q < 4; ++q) look(v[q]);
    }
    for (long long i = first; i < head; i += stride) look(src[i]);
    for (long long i = head + 4 * quads + first; i < n; i += stride) look(src[i]);
  }
  if (__ballot(most >= 0x7f800000u) != 0ull && (threadIdx.x & 63) == 0) atomicOr(flag, 1);
}
static __global__ __launch_bounds__(256) void finite_scan_kernel(FiniteScanInputs in, int32_t* __restrict__ flag) {
  finite_scan(in, (long long)blockIdx.x * blockDim.x + threadIdx.x, (long long)blockDim.x * gridDim.x, flag);
}
inline void launch_finite_scan(const FiniteScanInputs& in, int32_t* flag, hipStream_t s) {
  long long largest = 0;
  for (int t = 0; t < in.count; ++t) largest = in.lengths[t] > largest ? in.lengths[t] : largest;
  const long long want = (largest / 4 + 255) / 256;
  const unsigned blocks = (unsigned)(want < 1 ? 1 : (want > kScanBlocks ? kScanBlocks : want));
  hipLaunchKernelGGL(finite_scan_kernel, dim3(blocks), dim3(256), 0, s, in, flag);
}
inline int64_t finite_scan_bytes(const FiniteScanInputs& in) {
  int64_t floats = 0;
  for (int t = 0; t < in.count; ++t) floats += in.lengths[t];
  return 4 * floats;
}
// The arrays that are not empty; false: not to be read.
inline bool finite_scan_inputs(const float* const* arrays, const int64_t* lengths, int num_arrays, FiniteScanInputs& in) {
  if (num_arrays < 0 || num_arrays > 16 || (num_arrays > 0 && (!arrays || !lengths))) return false;
  for (int t = 0; t < num_arrays; ++t) {
    if (lengths[t] < 0) return false;
    if (lengths[t] == 0) continue;
    if (!arrays[t] || (reinterpret_cast<uintptr_t>(arrays[t]) & 3) != 0) return false;
    in.pointers[in.count] = arrays[t];
    in.lengths[in.count++] = lengths[t];
  }
  return true;
}

}  // namespace mlpsp
