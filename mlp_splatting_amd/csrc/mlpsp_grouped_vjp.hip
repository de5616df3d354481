// libmlpsp_hip: weight gradients of the per-primitive 72->32->32->4 MLP over a primitive-major CSR of hit
// records (counterpart of the reference's Triton kernels _grouped_vjp and _reduce_partials,
// scannet/primitive_gemm.py:101-183).
//
// One wavefront owns one segment (at most `segment` consecutive records of one primitive) and walks it in
// blocks of 32 records.  Per block it re-computes the forward pass (encoding, two hidden layers), pushes the
// output adjoints back through the layers and accumulates the three weight gradients, all as 32x32 MFMA
// tiles with f32 accumulation over the whole segment:
//     H1 = relu(ENC W1^T + b1)      H2 = relu(H1 W2^T + b2)
//     D2 = (D3 W3) * act2           D1 = (D2 W2) * act1
//     gW1 += D1^T ENC     gW2 += D2^T H1     gW3 += D3^T H2     gb_l += column sums of D_l
// Operand type T: float (v_mfma_f32_32x32x2_f32, an exact IEEE f32 fma chain: the reference's "ieee" path),
// _Float16 or __bf16 (v_mfma_f32_32x32x16).  As in the reference, operands are rounded to T, the adjoint d3 is
// scaled by `scale` before rounding and the result divided by it, and the bias gradients sum the ROUNDED
// adjoints so that biases and matrices see the same values (:168-171).  act_l comes from the saved ReLU masks
// if given, else from the recomputed pre-activations (:148-155).
//
// The 16-bit kernels keep every tile in registers (mlpsp_vjp16.hpp); the f32 kernel stages its tiles in LDS (further below).
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_segment_reduce.hpp"
#include "mlpsp_vjp16.hpp"

namespace mlpsp {

template <typename T, bool SAVED>
__global__ __launch_bounds__(64) void grouped_vjp16_kernel(
    const float* __restrict__ x6, const float* __restrict__ grad4, const int32_t* __restrict__ masks,
    const long long* __restrict__ offsets, const long long* __restrict__ group_prim,
    const long long* __restrict__ group_start, const float* __restrict__ freq, const float* __restrict__ att,
    const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
    const float* __restrict__ b2, const float* __restrict__ W3, float scale, int segment,
    float* __restrict__ partial) {
  __shared__ __attribute__((aligned(16))) Vjp16Operands<T> w;
  __shared__ __attribute__((aligned(16))) Vjp16Masks s_mask;
  const int lane = threadIdx.x, n = lane & 31, g = lane >> 5;
  const long long group = blockIdx.x;
  const long long p = group_prim[group];
  const long long begin = group_start[group];
  const long long seg_end = begin + segment, list_end = offsets[p + 1];
  const long long end = seg_end < list_end ? seg_end : list_end;
  w.select(lane);
  w.load(W1, b1, W2, b2, W3, (size_t)p, lane);
  float kf[6];
#pragma unroll
  for (int f = 0; f < 6; ++f) kf[f] = (freq[f] * att[f]) * 0.159154943f;
  Vjp16Sums sum;
  sum.clear();
  for (long long base = begin; base < end; base += 32) {
    const long long rec = base + n;
    const bool live = rec < end;
    // this lane's record: three inputs of its group, the output adjoints, the mask words
    float x[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = live ? x6[rec * 6 + 3 * g + c] : 0.f;
    float4 d3 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (live && g == 0) d3 = *reinterpret_cast<const float4*>(grad4 + rec * 4);
    uint2 words = make_uint2(0u, 0u);
    if constexpr (SAVED) {
      if (live) words = make_uint2((uint32_t)masks[rec * 2], (uint32_t)masks[rec * 2 + 1]);
      s_mask.put(g, n, g ? words.y : words.x);
    }
    vjp16_block<T, SAVED>(w, sum, x, d3, live, s_mask, words.y, kf, scale, lane);
  }
  vjp16_store(sum, packed_grad_rows(partial + group * kGradFloats), 1.f / scale, lane);
}

// ---------------------------------------------------------------------------------------------
// The f32 path.  v_mfma_f32_32x32x2_f32 takes ONE element per lane and operand, so an operand can be read from
// LDS in either orientation and no transposed copies are needed; and the contraction over the block's records
// may run in any order, so the weight-gradient products take their A operand -- an adjoint tile, transposed --
// straight from the accumulator registers that hold it: register i of lane (column c, group g) is row
// rec(i, g) = 8 (i / 4) + 4 g + i % 4, which is used as "record 2 i + g" of the contraction, the B operand
// reading the same record's row.  Tiles in LDS: encoding, both hidden activations, d2 and d3 (row-major,
// [record][column]) and the weights in their own layout: 37 KB per wavefront, four wavefronts per CU.
// ---------------------------------------------------------------------------------------------
struct VjpTilesF32 {
  static constexpr int LD1 = 73, LD32 = 33, LD3 = 5;
  float w1[32 * LD1];    // [hid][k]
  float w2[32 * LD32];   // [hid2][hid]
  float w3[4 * LD32];    // [out][hid2]
  float enc[32 * LD1];   // [rec][k]
  float h1[32 * LD32];   // [rec][hid]
  float h2[32 * LD32];   // [rec][hid2]
  float d2[32 * LD32];   // [rec][hid2]
  float d3[32 * LD3];    // [rec][out]
  int32_t mask[2][32];
};

__device__ __forceinline__ vf32x16 mfma32(float a, float b, vf32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// acc += A B over STEPS MFMAs; element k of the operands at a[k * a_stride], b[k * b_stride] (the caller folds
// the lane's row/column and k-group into the pointers).  Operands are fetched CHUNK steps ahead of the MFMAs
// that use them: written as "load, wait, MFMA" per step the LDS latency is paid once per instruction.
template <int STEPS, int CHUNK>
__device__ __forceinline__ vf32x16 mma_f32(const float* a, int a_stride, const float* b, int b_stride, vf32x16 acc) {
  static_assert(STEPS % CHUNK == 0, "whole chunks");
#pragma unroll
  for (int c0 = 0; c0 < STEPS; c0 += CHUNK) {
    float av[CHUNK], bv[CHUNK];
#pragma unroll
    for (int s = 0; s < CHUNK; ++s) {
      av[s] = a[(c0 + s) * a_stride];
      bv[s] = b[(c0 + s) * b_stride];
    }
#pragma unroll
    for (int s = 0; s < CHUNK; ++s) acc = mfma32(av[s], bv[s], acc);
  }
  return acc;
}

__global__ __launch_bounds__(64) void grouped_vjp_f32_kernel(
    const float* __restrict__ x6, const float* __restrict__ grad4, const int32_t* __restrict__ masks,
    const long long* __restrict__ offsets, const long long* __restrict__ group_prim,
    const long long* __restrict__ group_start, const float* __restrict__ freq, const float* __restrict__ att,
    const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
    const float* __restrict__ b2, const float* __restrict__ W3, float scale, int segment,
    float* __restrict__ partial) {
  using TL = VjpTilesF32;
  __shared__ TL t;
  const int lane = threadIdx.x, n = lane & 31, g = lane >> 5;
  const long long group = blockIdx.x;
  const long long p = group_prim[group];
  const long long begin = group_start[group];
  const long long seg_end = begin + segment, list_end = offsets[p + 1];
  const long long end = seg_end < list_end ? seg_end : list_end;
  for (int i = lane; i < 32 * 72; i += 64) t.w1[(i / 72) * TL::LD1 + i % 72] = W1[p * 2304 + i];
  for (int i = lane; i < 32 * 32; i += 64) t.w2[(i >> 5) * TL::LD32 + (i & 31)] = W2[p * 1024 + i];
  for (int i = lane; i < 4 * 32; i += 64) t.w3[(i >> 5) * TL::LD32 + (i & 31)] = W3[p * 128 + i];
  const float bias1 = b1[p * 32 + n], bias2 = b2[p * 32 + n];
  __syncthreads();

  vf32x16 gw1[3], gw2, gw3;
#pragma unroll
  for (int i = 0; i < 16; ++i) gw1[0][i] = gw1[1][i] = gw1[2][i] = gw2[i] = gw3[i] = 0.f;
  float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f;
  const vf32x16 zero = gw2;
  const int n2 = n < 8 ? n : 0;    // column of the third 32-wide block of the 72 encoding columns (64 + n2)

  for (long long base = begin; base < end; base += 32) {
    const long long rec = base + n;
    const bool live = rec < end;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float x = live ? x6[rec * 6 + 3 * g + c] : 0.f;
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const int j = (3 * g + c) * 6 + f;
        float s, co;
        det_sincos((x * freq[f]) * att[f], s, co);
        t.enc[n * TL::LD1 + j] = live ? s : 0.f;
        t.enc[n * TL::LD1 + 36 + j] = live ? co : 0.f;
      }
    }
    if (g == 0) {
#pragma unroll
      for (int o = 0; o < 4; ++o) t.d3[n * TL::LD3 + o] = live ? grad4[rec * 4 + o] * scale : 0.f;
    } else if (masks) {
      t.mask[0][n] = live ? masks[rec * 2] : 0;
      t.mask[1][n] = live ? masks[rec * 2 + 1] : 0;
    }
    __syncthreads();

    // forward (accumulator column = hidden unit n, register i = record 8 (i/4) + 4 g + i%4)
    vf32x16 a1 = mma_f32<36, 18>(t.enc + n * TL::LD1 + g, 2, t.w1 + n * TL::LD1 + g, 2, zero);
    unsigned act1 = 0u, act2 = 0u;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i >> 2) + 4 * g + (i & 3);
      const float h = fmaxf(a1[i] + bias1, 0.f);
      t.h1[row * TL::LD32 + n] = h;
      act1 |= (masks ? ((unsigned)t.mask[0][row] >> n) & 1u : (h > 0.f ? 1u : 0u)) << i;
    }
    __syncthreads();
    vf32x16 a2 = mma_f32<16, 16>(t.h1 + n * TL::LD32 + g, 2, t.w2 + n * TL::LD32 + g, 2, zero);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i >> 2) + 4 * g + (i & 3);
      const float h = fmaxf(a2[i] + bias2, 0.f);
      t.h2[row * TL::LD32 + n] = h;
      act2 |= (masks ? ((unsigned)t.mask[1][row] >> n) & 1u : (h > 0.f ? 1u : 0u)) << i;
    }
    // backward
    vf32x16 dd2 = mma_f32<2, 2>(t.d3 + n * TL::LD3 + g, 2, t.w3 + g * TL::LD32 + n, 2 * TL::LD32, zero);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i >> 2) + 4 * g + (i & 3);
      dd2[i] = ((act2 >> i) & 1u) ? dd2[i] : 0.f;
      gb2 += dd2[i];
      t.d2[row * TL::LD32 + n] = dd2[i];
    }
    if (lane < 4) {
      for (int r = 0; r < 32; ++r) gb3 += t.d3[r * TL::LD3 + lane];
    }
    __syncthreads();
    vf32x16 dd1 = mma_f32<16, 16>(t.d2 + n * TL::LD32 + g, 2, t.w2 + g * TL::LD32 + n, 2 * TL::LD32, zero);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dd1[i] = ((act1 >> i) & 1u) ? dd1[i] : 0.f;
      gb1 += dd1[i];
    }
    // weight gradients: A = the adjoint tile from registers, B = the activation row of the same record
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += 4) {      // operands of four records ahead of their twenty MFMAs
      float e0[4], e1[4], e2[4], v1[4], v2[4], v3[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u, row = 8 * (i >> 2) + 4 * g + (i & 3);
        e0[u] = t.enc[row * TL::LD1 + n];
        e1[u] = t.enc[row * TL::LD1 + 32 + n];
        e2[u] = t.enc[row * TL::LD1 + 64 + n2];
        v1[u] = t.h1[row * TL::LD32 + n];
        v2[u] = t.h2[row * TL::LD32 + n];
        v3[u] = t.d3[row * TL::LD3 + (n < 4 ? n : 0)];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u;
        gw1[0] = mfma32(dd1[i], e0[u], gw1[0]);
        gw1[1] = mfma32(dd1[i], e1[u], gw1[1]);
        gw1[2] = mfma32(dd1[i], e2[u], gw1[2]);
        gw2 = mfma32(dd2[i], v1[u], gw2);
        gw3 = mfma32(n < 4 ? v3[u] : 0.f, v2[u], gw3);
      }
    }
    __syncthreads();
  }

  float* __restrict__ out = partial + group * kGradFloats;
  const float inv = 1.f / scale;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = 8 * (i >> 2) + 4 * g + (i & 3);
    out[row * 72 + n] = gw1[0][i] * inv;
    out[row * 72 + 32 + n] = gw1[1][i] * inv;
    if (n < 8) out[row * 72 + 64 + n] = gw1[2][i] * inv;
    out[2336 + row * 32 + n] = gw2[i] * inv;
    if (row < 4) out[3392 + row * 32 + n] = gw3[i] * inv;
  }
  gb1 += __shfl_xor(gb1, 32);
  gb2 += __shfl_xor(gb2, 32);
  if (g == 0) {
    out[2304 + n] = gb1 * inv;
    out[3360 + n] = gb2 * inv;
  }
  if (lane < 4) out[3520 + lane] = gb3 * inv;
}

}  // namespace mlpsp

using namespace mlpsp;

MLPSP_API int mlpsp_grouped_vjp(const float* x6_dev, const float* grad4_dev, const int32_t* relu_masks_dev,
                                const int64_t* csr_offsets_dev, const int64_t* group_primitives_dev,
                                const int64_t* group_starts_dev, int64_t num_groups, const float* freq_dev,
                                const float* att_dev, const float* W1, const float* b1, const float* W2,
                                const float* b2, const float* W3, int precision, float scale, int segment,
                                float* partial_dev, mlpsp_stream_t stream) {
  if (num_groups < 0 || num_groups > 2147483647LL || segment <= 0 || segment % 32 != 0) return MLPSP_E_ARGUMENT;
  if (precision < 0 || precision > 2 || !(scale > 0.f) || !(scale <= 3.4028235e38f)) return MLPSP_E_ARGUMENT;
  if (num_groups == 0) return MLPSP_OK;
  if (!x6_dev || !grad4_dev || !csr_offsets_dev || !group_primitives_dev || !group_starts_dev || !freq_dev ||
      !att_dev || !W1 || !b1 || !W2 || !b2 || !W3 || !partial_dev)
    return MLPSP_E_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)num_groups), block(64);
#define MLPSP_VJP_LAUNCH(T)                                                                                        \
  do {                                                                                                             \
    if (relu_masks_dev)                                                                                            \
      hipLaunchKernelGGL((grouped_vjp16_kernel<T, true>), grid, block, 0, s, x6_dev, grad4_dev, relu_masks_dev,    \
                         (const long long*)csr_offsets_dev, (const long long*)group_primitives_dev,                \
                         (const long long*)group_starts_dev, freq_dev, att_dev, W1, b1, W2, b2, W3, scale,         \
                         segment, partial_dev);                                                                    \
    else                                                                                                           \
      hipLaunchKernelGGL((grouped_vjp16_kernel<T, false>), grid, block, 0, s, x6_dev, grad4_dev, relu_masks_dev,   \
                         (const long long*)csr_offsets_dev, (const long long*)group_primitives_dev,                \
                         (const long long*)group_starts_dev, freq_dev, att_dev, W1, b1, W2, b2, W3, scale,         \
                         segment, partial_dev);                                                                    \
  } while (0)
  if (precision != 0 && ((reinterpret_cast<uintptr_t>(W1) | reinterpret_cast<uintptr_t>(W2) |
                          reinterpret_cast<uintptr_t>(b1) | reinterpret_cast<uintptr_t>(b2) |
                          reinterpret_cast<uintptr_t>(grad4_dev)) & 15) != 0)
    return MLPSP_E_ARGUMENT;      // the 16-bit kernels read weight rows and adjoints with 16-byte loads
  if (precision == 0)
    hipLaunchKernelGGL(grouped_vjp_f32_kernel, grid, block, 0, s, x6_dev, grad4_dev, relu_masks_dev,
                       (const long long*)csr_offsets_dev, (const long long*)group_primitives_dev,
                       (const long long*)group_starts_dev, freq_dev, att_dev, W1, b1, W2, b2, W3, scale, segment,
                       partial_dev);
  else if (precision == 1) MLPSP_VJP_LAUNCH(_Float16);
  else MLPSP_VJP_LAUNCH(__bf16);
#undef MLPSP_VJP_LAUNCH
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}

MLPSP_API int64_t mlpsp_segment_reduce_rows(int64_t num_groups) {
  return num_groups < 0 ? -1 : segment_reduce_rows(num_groups);
}

MLPSP_API int mlpsp_reduce_partials(const float* partial_dev, const int64_t* group_primitives_dev,
                                    const int64_t* group_offsets_dev, int64_t num_groups, int num_primitives,
                                    float* out_dev, int32_t* nonfinite_dev, mlpsp_stream_t stream) {
  if (!nonfinite_dev || num_primitives < 0) return MLPSP_E_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  MLPSP_HIP_TRY(clear_async(nonfinite_dev, sizeof(int32_t), s));
  ReduceDest dest{};
  dest.packed = out_dev;
  return segment_reduce<false>(partial_dev, group_primitives_dev, group_offsets_dev, num_groups, num_primitives,
                               kGradFloats, dest, nonfinite_dev, s);
}

MLPSP_API int mlpsp_reduce_partials_split(const float* partial_dev, const int64_t* group_primitives_dev,
                                          const int64_t* group_offsets_dev, int64_t num_groups, int num_primitives,
                                          float* gW1_dev, float* gb1_dev, float* gW2_dev, float* gb2_dev, float* gW3_dev,
                                          float* gb3_dev, int32_t* nonfinite_dev, mlpsp_stream_t stream) {
  if (!nonfinite_dev || num_primitives < 0) return MLPSP_E_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  MLPSP_HIP_TRY(clear_async(nonfinite_dev, sizeof(int32_t), s));
  ReduceDest dest{};
  float* parts[6] = {gW1_dev, gb1_dev, gW2_dev, gb2_dev, gW3_dev, gb3_dev};
  for (int i = 0; i < 6; ++i) dest.part[i] = parts[i];
  return segment_reduce<true>(partial_dev, group_primitives_dev, group_offsets_dev, num_groups, num_primitives,
                              kGradFloats, dest, nonfinite_dev, s);
}
