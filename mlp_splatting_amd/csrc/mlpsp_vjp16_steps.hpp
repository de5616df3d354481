// Weight gradients of the per-primitive 72->32->32->4 MLP over training steps in 16-bit operands (fp16 / bf16,
// v_mfma_f32_32x32x16, f32 accumulation): the roundings of mlpsp_vjp16.hpp -- encoding, weights, adjoints and hidden activations
// to the operand type, sums in f32 -- in the frame of mlpsp_vjp32.hpp: a workgroup shares a primitive's operands in LDS and deals
// its half steps to its wavefronts, and what a gradient needs with its records in the k-slots is read back from LDS with
// ds_read_b64_tr_b16 instead of being computed in both orientations or transposed by the matrix core: 16 large matrix
// instructions and ~250 vector instructions a block instead of 30 and 350.
//
// Bound by the vector instructions (the 36 sines and cosines are a third of their time).  Four wavefronts to a workgroup and
// two workgroups to a CU: while one changes primitives the other works, and two wavefronts to a SIMD hold everything in 186
// registers.  Gradient call of 648,000 steps: 1.90 ms; one workgroup of eight 2.12, four of two 2.31, three of four 2.9 (168
// registers: spills); with the block of mlpsp_vjp16.hpp, a wavefront to a chunk of 64 steps, 2.54.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_mfma16.hpp"
#include "mlpsp_vjp16.hpp"
#include "mlpsp_vjp32.hpp"

namespace mlpsp {

constexpr int kVjp16Waves = 4;
// As Vjp32Wave, one plane.
struct Vjp16Wave {
  __attribute__((aligned(16))) unsigned enc[32][32];
  __attribute__((aligned(16))) unsigned enc_tail[32][4];
  __attribute__((aligned(16))) unsigned tile[32][16];
  __attribute__((aligned(16))) unsigned d3[32][2];         // [record]: the four output adjoints, rounded
  Vjp16Masks mask;
  static constexpr int kRowBytes = 128;
};
template <typename T>
struct Vjp16Shared {
  u32x4 w1[5][64];               // W1[n][..]: words = pairs (sin, cos) 4 s + d of group g
  u32x4 w2[2][64], w2t[2][64];   // W2[n][u] over u = d_row(8 s + j, g); W2[u][n] over u = hidden_unit(8 s + j, g)
  u32x2 w3r[64];                 // W3 column of unit hidden_unit_of_row(n) (k-slots: the four outputs), group 0
  float bias1[32], bias2[32];
  __attribute__((aligned(16))) unsigned zero[4];
  Vjp16Wave wave[kVjp16Waves];
};
template <typename T>
union Vjp16StepsLds {
  Vjp16Shared<T> s;
  __attribute__((aligned(16))) float sums[kVjp16Waves][kGradFloats];    // in the end
};

// The primitive's weights into LDS, by the first six wavefronts.
template <typename T>
__device__ __forceinline__ void vjp16_load(const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
                                           const float* __restrict__ b2, const float* __restrict__ W3, size_t p, int wave, int lane,
                                           Vjp16Shared<T>& s) {
  asm volatile("" : "+v"(lane));         // (or the addresses are formed ahead of the loop over the runs, one by one)
  const int n = lane & 31, g = lane >> 5;
  for (int q = wave; q < 5; q += kVjp16Waves) {
    const float* __restrict__ row = W1 + p * 2304 + n * 72 + 18 * g;
    u32x4 v;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int t = 4 * q + d;
      v[d] = t < 18 ? Ops<T>::pack2(row[t < 18 ? t : 0], row[36 + (t < 18 ? t : 0)]) : 0u;
    }
    s.w1[q][lane] = v;
  }
  if (wave == 1 || wave == 2) {
    const int k = wave - 1;
    const float* __restrict__ row = W2 + p * 1024 + n * 32 + 16 * k + 4 * g;
    const float* __restrict__ col = W2 + p * 1024 + n;
    u32x4 a, b;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int j = 2 * d + (d & 2 ? 4 : 0);
      a[d] = Ops<T>::pack2(row[j], row[j + 1]);
      b[d] = Ops<T>::pack2(col[hidden_unit(8 * k + 2 * d, g) * 32], col[hidden_unit(8 * k + 2 * d + 1, g) * 32]);
    }
    s.w2[k][lane] = a;
    s.w2t[k][lane] = b;
  }
  if (wave == 3) {
    const float* __restrict__ r = W3 + p * 128 + hidden_unit_of_row(n);
    s.w3r[lane] = g ? u32x2{0u, 0u} : u32x2{Ops<T>::pack2(r[0], r[32]), Ops<T>::pack2(r[64], r[96])};
    (g ? s.bias2 : s.bias1)[n] = (g ? b2 : b1)[p * 32 + n];
  }
}

struct Vjp16StepSums {
  vf32x16 gw1[2], gw2;
  f32x4 gw1e, gw3, gb1, gb2;
  float gb3[4];
  __device__ __forceinline__ void clear() {
    gw1[0] = gw1[1] = gw2 = splat16(0.f);
    gw1e = gw3 = gb1 = gb2 = f32x4{0.f, 0.f, 0.f, 0.f};
    gb3[0] = gb3[1] = gb3[2] = gb3[3] = 0.f;
  }
};
__device__ __forceinline__ Pack8 transpose_tile(const Pack8& v, Vjp16Wave& s, int n, int g) {
  const char* const from = tile_reads(s.tile, n, g);
  *reinterpret_cast<u32x4*>(&s.tile[n][tile_place(2 * g, n)]) = v.s[0];
  *reinterpret_cast<u32x4*>(&s.tile[n][tile_place(2 * g + 1, n)]) = v.s[1];
  return Pack8{{read_records(from, 0, 64), read_records(from, 1, 64)}};
}
__device__ __forceinline__ f32x4 tail_product(u32x4 a, u32x4 b, f32x4 c, __bf16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 tail_product(u32x4 a, u32x4 b, f32x4 c, _Float16) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// One block of 32 records.  Lane (n, g): record n, x = its three inputs of group g; kf: the phase scales in revolutions.
template <typename T>
__device__ __forceinline__ void vjp16_step_block(const Vjp16Shared<T>& w, Vjp16StepSums& sum, Vjp16Wave& s, const float x[3],
                                                 float4 adjoint, uint32_t mask1, uint32_t mask2, const float (&kf)[6], float scale,
                                                 int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5;
  const vf32x16 zero = splat16(0.f);
  const u32x2 ones = {Ops<T>::kOneWord, Ops<T>::kOneWord};
  // ---- adjoints of layer 2: record in the lane, unit hidden_unit(i, g) in register i.  (Group 1 multiplies by zero.)
  s.mask.put(g, n, g ? mask2 : mask1);
  u32x4 d3 = {0u, 0u, 0u, 0u};
  d3[0] = Ops<T>::pack2(adjoint.x * scale, adjoint.y * scale);
  d3[1] = Ops<T>::pack2(adjoint.z * scale, adjoint.w * scale);
  if (g == 0) {
    *reinterpret_cast<u32x2*>(s.d3[n]) = u32x2{d3[0], d3[1]};
    sum.gb3[0] += Unpack<T>::lo(d3[0]);
    sum.gb3[1] += Unpack<T>::hi(d3[0]);
    sum.gb3[2] += Unpack<T>::lo(d3[1]);
    sum.gb3[3] += Unpack<T>::hi(d3[1]);
  }
  const u32x2 w3r = w.w3r[lane];
  const Pack8 d2 = and_tile(pack_tile<T>(Ops<T>::mfma(u32x4{w3r[0], w3r[1], 0u, 0u}, d3, zero)), mask_tile_record_major(mask2, g));
  const Pack8 d2t = transpose_tile(d2, s, n, g);
  // ---- adjoints of layer 1: unit in the lane
  const Pack8 d1 = and_tile(pack_tile<T>(mma2<T>(d2, Pack8{{w.w2t[0][lane], w.w2t[1][lane]}}, zero)),
                            mask_tile_unit_major(s.mask.half[0], n, g));
  // ---- encoding and layer 1: record in the lane
  vf32x16 a1 = bias_rows(w.bias1, g);
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    u32x4 e;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int t = 4 * k + d;
      const float rev = t < 18 ? x[t < 18 ? t / 6 : 0] * kf[t % 6] : 0.f;
      e[d] = t < 18 ? Ops<T>::pack2(__builtin_amdgcn_sinf(rev), __builtin_amdgcn_cosf(rev)) : 0u;
    }
    if (k < 4) *reinterpret_cast<u32x4*>(&s.enc[n][enc_place(2 * g + (k >> 1), k & 1, n)]) = e;
    else *reinterpret_cast<u32x2*>(&s.enc_tail[n][2 * g]) = u32x2{e[0], e[1]};
    a1 = Ops<T>::mfma(w.w1[k][lane], e, a1);
  }
  const Pack8 h1 = relu_tile(pack_tile<T>(a1));
  const Pack8 h1t = transpose_tile(h1, s, n, g);
  // ---- layer 2: unit in the lane, straight into the W3 gradient
  const Pack8 h2 = relu_tile(pack_tile<T>(mma2<T>(h1, Pack8{{w.w2[0][lane], w.w2[1][lane]}}, splat16(w.bias2[n]))));
  const char* const d3_from = reinterpret_cast<const char*>(s.d3[4 * g + ((n >> 2) & 3)]);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = q >> 1, d = 2 * (q & 1);
    sum.gw3 = Ops<T>::mfma4(read_transposed(d3_from + 8 * q * 8), u32x2{h2.s[k][d], h2.s[k][d + 1]}, sum.gw3);
    sum.gb2 = Ops<T>::mfma4(ones, u32x2{d2t.s[k][d], d2t.s[k][d + 1]}, sum.gb2);
    sum.gb1 = Ops<T>::mfma4(ones, u32x2{d1.s[k][d], d1.s[k][d + 1]}, sum.gb1);
  }
  sum.gw2 = mma2<T>(d2t, h1t, sum.gw2);
  // ---- the W1 gradient (addresses as in vjp32_block)
  const int rec = 4 * g + ((n >> 2) & 3);
  const bool last = ((n >> 1) & 1) == (n >> 4);
  const char* const last0 = last ? reinterpret_cast<const char*>(&s.enc_tail[rec][2 * (n & 1)]) : reinterpret_cast<const char*>(w.zero);
  const int last_row = last ? 16 : 0;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      sum.gw1[c] = Ops<T>::mfma(d1.s[k], read_records(enc_reads(s.enc, c, n, g), k, Vjp16Wave::kRowBytes), sum.gw1[c]);
    }
    sum.gw1e = tail_product(d1.s[k], read_records(last0, k, last_row), sum.gw1e, T{});
  }
}

// A wavefront's sums to a row of LDS, in the order of a packed row of gradients.
__device__ __forceinline__ void vjp16_park(const Vjp16StepSums& sum, float* to, int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5;
  const GradRows out = packed_grad_rows(to);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 8 * (i >> 2) + 4 * g + (i & 3);
    out.W1[r * 72 + enc_feature(n)] = sum.gw1[0][i];
    out.W1[r * 72 + enc_feature(32 + n)] = sum.gw1[1][i];
    out.W2[hidden_unit(r & 15, r >> 4) * 32 + tile_unit(n)] = sum.gw2[i];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    out.W1[((lane & 8 ? 16 : 0) + 4 * (lane >> 4) + r) * 72 + enc_feature(64 + (lane & 7))] = sum.gw1e[r];
    const float v = sum.gw3[r] + __shfl_xor(sum.gw3[r], 32);
    if (g == 0) out.W3[r * 32 + n] = v;
  }
  const float gb1 = sum.gb1[0] + __shfl_xor(sum.gb1[0], 32), gb2 = sum.gb2[0] + __shfl_xor(sum.gb2[0], 32);
  if (g == 0) out.b1[n] = gb1;
  else out.b2[hidden_unit(n & 15, n >> 4)] = gb2;
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    float v = sum.gb3[o];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    if (lane == o) out.b3[o] = v;
  }
}

}  // namespace mlpsp
