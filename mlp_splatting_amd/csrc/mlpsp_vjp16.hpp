// Weight gradients of the per-primitive 72->32->32->4 MLP over blocks of 32 records of one primitive, in 16-bit operands
// with f32 accumulation: what the grouped kernel over a CSR of records (mlpsp_grouped_vjp.hip) and the kernel over
// training steps (mlpsp_train_backward.hip) share.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_mfma16.hpp"

namespace mlpsp {

typedef float vf32x16 __attribute__((ext_vector_type(16)));

constexpr int kGradFloats = 3524;   // W1 2304 | b1 32 | W2 1024 | b2 32 | W3 128 | b3 4 (primitive_gemm.py:160-166)

// ---------------------------------------------------------------------------------------------
// The 16-bit paths (fp16 / bf16 operands, v_mfma_f32_32x32x16, f32 accumulation): everything in registers.
//
// An MFMA D = A B takes from lane (m, g) row m of A and column m of B, eight k-slots each (k = 8 g + 0..7
// of the K-step), and returns to lane (n, g) column n of D, rows d_row(i, g) = 8 (i/4) + 4 g + i%4 in
// register i.  Two consequences carry the whole kernel:
//  (1) Swapping the operands transposes the result: with X = the block's 32 records (one per lane, k-slots =
//      its inputs) and W = a weight matrix (one output unit per lane), mfma(W, X) puts a RECORD in every lane
//      and the units in its registers ("record-major" tile), mfma(X, W) a UNIT in every lane and the records
//      d_row(i, g) in its registers ("unit-major").  A record-major tile, rectified, rounded and packed in
//      pairs, is the X operand of the next layer; a unit-major tile packed the same way is an operand whose
//      k-slots are RECORDS -- which is what the weight gradients contract over.  Since both operands of a
//      weight-gradient product come from unit-major tiles, their k-slots name the same records, and nothing has
//      to be transposed through LDS: each forward/backward product is simply issued in both orientations.
//  (2) A tile that no product yields in the needed orientation (the encoding, the output adjoints) is
//      transposed by the matrix core itself: mfma(X, I) with a 0/1 selection operand I returns X unit-major,
//      exactly (one non-zero term per sum).
// Per block of 32 records: 32 MFMAs (34 without saved masks) against 20 for a formulation that transposes
// through LDS, and no LDS traffic except the 64 mask words: 11.3 -> 2.8 ms for 38.6 M records, with one
// wavefront per SIMD (342 registers; capped at 256 the compiler spills 84 and the kernel takes 4.5 ms).
//
// k-slot order of the encoding (both the X operand of layer 1 and W1's operand): lane group g owns input
// components 3g..3g+2; its slot q = 8 s + j of K-step s (q < 36) is pair t = q / 2 = 6 c + f (component
// 3g + c, frequency f), sin for even q, cos for odd.  Slots q = 36..39 are padding; slot q = 36 of group 0
// (k = 68) carries the constant 1, so that the layer-1 bias gradient falls out of the W1 product as one more
// column.  sin/cos use the native v_sin/v_cos in revolutions: their error (~1e-6) is far below the operand
// rounding, as in the forward kernels of this precision.
// ---------------------------------------------------------------------------------------------
typedef unsigned short vu16x2 __attribute__((ext_vector_type(2)));

template <typename T> struct Unpack;
template <> struct Unpack<__bf16> {
  static __device__ __forceinline__ float lo(unsigned w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float hi(unsigned w) { return __uint_as_float(w & 0xFFFF0000u); }
};
template <> struct Unpack<_Float16> {
  static __device__ __forceinline__ float lo(unsigned w) { return (float)__builtin_bit_cast(f16x2, w)[0]; }
  static __device__ __forceinline__ float hi(unsigned w) { return (float)__builtin_bit_cast(f16x2, w)[1]; }
};

// 0xFFFF in every half of `rectified` that is not zero (an active unit), 0 in the others
__device__ __forceinline__ unsigned active_halves(unsigned rectified) {
  const vu16x2 one = {1, 1}, all = {0xFFFF, 0xFFFF};
  return __builtin_bit_cast(unsigned, (vu16x2)(__builtin_elementwise_min(__builtin_bit_cast(vu16x2, rectified), one) * all));
}

struct Pack8 {
  u32x4 s[2];   // the two K-steps of a 32-deep contraction
};

template <typename T>
__device__ __forceinline__ Pack8 pack_tile(const vf32x16& v) {
  Pack8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) r.s[s][d] = Ops<T>::pack2(v[8 * s + 2 * d], v[8 * s + 2 * d + 1]);
  return r;
}
__device__ __forceinline__ Pack8 relu_tile(Pack8 r) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) r.s[s][d] = relu_packed(r.s[s][d]);
  return r;
}
__device__ __forceinline__ Pack8 and_tile(Pack8 r, const Pack8& m) {
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) r.s[s][d] &= m.s[s][d];
  return r;
}
__device__ __forceinline__ Pack8 active_tile(const Pack8& h) {
  Pack8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) r.s[s][d] = active_halves(h.s[s][d]);
  return r;
}
// AND-masks of a unit-major tile from saved mask words: w[i] = the mask word of the record in register i,
// bit = this lane's unit
__device__ __forceinline__ Pack8 mask_tile_unit_major(const int32_t w[16], int bit) {
  Pack8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int i = 8 * s + 2 * d;
      const unsigned lo = (unsigned)__builtin_amdgcn_sbfe(w[i], bit, 1), hi = (unsigned)__builtin_amdgcn_sbfe(w[i + 1], bit, 1);
      r.s[s][d] = (lo & 0xFFFFu) | (hi << 16);
    }
  return r;
}
// ... and of a record-major tile: `word` = the mask word of this lane's record, register i is unit d_row(i, g)
__device__ __forceinline__ Pack8 mask_tile_record_major(int32_t word, int g) {
  const int shifted = word >> (4 * g);
  Pack8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int i = 8 * s + 2 * d, u = 8 * (i / 4) + (i % 4);      // d_row(i, 0); i is even, so i + 1 is unit u + 1
      const unsigned lo = (unsigned)__builtin_amdgcn_sbfe(shifted, u, 1), hi = (unsigned)__builtin_amdgcn_sbfe(shifted, u + 1, 1);
      r.s[s][d] = (lo & 0xFFFFu) | (hi << 16);
    }
  return r;
}
template <typename T>
__device__ __forceinline__ float sum_tile(const Pack8& r) {
  float t = 0.f;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) t += Unpack<T>::lo(r.s[s][d]) + Unpack<T>::hi(r.s[s][d]);
  return t;
}
template <typename T>
__device__ __forceinline__ vf32x16 mma2(const Pack8& a, const Pack8& b, vf32x16 acc) {
  acc = Ops<T>::mfma(a.s[0], b.s[0], acc);
  return Ops<T>::mfma(a.s[1], b.s[1], acc);
}
__device__ __forceinline__ vf32x16 splat16(float v) {
  vf32x16 r;
#pragma unroll
  for (int i = 0; i < 16; ++i) r[i] = v;
  return r;
}

// The primitive's weights as operands, one unit (n) per lane, and the selection operands.
template <typename T>
struct Vjp16Operands {
  u32x4 w1op[5], w3op, out_sel, k_sel[2];
  Pack8 w2op, w2top;     // W2[n][u] and W2[u][n] over the units u = d_row(8 s + j, g) of this lane's k-slots
  float bias1, bias2;
  unsigned one_lo;

  __device__ __forceinline__ void select(int n, int g) {
    // out_sel returns the output adjoints unit-major (column n = output n < 4); k_sel[h] returns K-step 2c + h of the
    // encoding as columns 32c + n
    const unsigned one_hi = Ops<T>::pack2(0.f, 1.f);
    one_lo = Ops<T>::pack2(1.f, 0.f);
    out_sel = k_sel[0] = k_sel[1] = u32x4{0u, 0u, 0u, 0u};
    if (g == 0 && n < 4) out_sel[n >> 1] = (n & 1) ? one_hi : one_lo;
    const unsigned v = (n & 1) ? one_hi : one_lo;
    const bool mine = ((n >> 3) & 1) == g;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int d = 0; d < 4; ++d) k_sel[h][d] = (mine && (n >> 4) == h && ((n & 7) >> 1) == d) ? v : 0u;
  }

  __device__ __forceinline__ void load(const float* __restrict__ W1, const float* __restrict__ b1,
                                       const float* __restrict__ W2, const float* __restrict__ b2,
                                       const float* __restrict__ W3, long long p, int n, int g) {
    {
      const float* __restrict__ row = W1 + p * 2304 + n * 72 + 18 * g;
      float ws[18], wc[18];
#pragma unroll
      for (int t = 0; t < 18; t += 2) {
        const float2 a = *reinterpret_cast<const float2*>(row + t), c = *reinterpret_cast<const float2*>(row + 36 + t);
        ws[t] = a.x;
        ws[t + 1] = a.y;
        wc[t] = c.x;
        wc[t + 1] = c.y;
      }
#pragma unroll
      for (int s = 0; s < 5; ++s)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int t = 4 * s + d;
          w1op[s][d] = t < 18 ? Ops<T>::pack2(ws[t], wc[t]) : 0u;
        }
    }
    {
      const float* __restrict__ row = W2 + p * 1024 + n * 32;
      const float* __restrict__ col = W2 + p * 1024 + n;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float4 lo = *reinterpret_cast<const float4*>(row + 16 * s + 4 * g);
        const float4 hi = *reinterpret_cast<const float4*>(row + 16 * s + 8 + 4 * g);
        w2op.s[s] = u32x4{Ops<T>::pack2(lo.x, lo.y), Ops<T>::pack2(lo.z, lo.w), Ops<T>::pack2(hi.x, hi.y), Ops<T>::pack2(hi.z, hi.w)};
        float c[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) c[j] = col[(16 * s + 8 * (j / 4) + 4 * g + j % 4) * 32];
        w2top.s[s] = u32x4{Ops<T>::pack2(c[0], c[1]), Ops<T>::pack2(c[2], c[3]), Ops<T>::pack2(c[4], c[5]), Ops<T>::pack2(c[6], c[7])};
      }
    }
    // W3^T: k-slots = the four outputs (group 0, slots 0..3)
    w3op = u32x4{0u, 0u, 0u, 0u};
    if (g == 0) {
      const float* __restrict__ col = W3 + p * 128 + n;
      w3op[0] = Ops<T>::pack2(col[0], col[32]);
      w3op[1] = Ops<T>::pack2(col[64], col[96]);
    }
    bias1 = b1[p * 32 + n];
    bias2 = b2[p * 32 + n];
  }
};

struct Vjp16Sums {
  vf32x16 gw1[3], gw2, gw3;
  float gb2, gb3[4];
  __device__ __forceinline__ void clear() {
    gw1[0] = gw1[1] = gw1[2] = gw2 = gw3 = splat16(0.f);
    gb2 = gb3[0] = gb3[1] = gb3[2] = gb3[3] = 0.f;
  }
};

// One block of 32 records.  Lane (n, g): record n; x = its three inputs of group g, d3 = the record's output adjoints
// (lanes of group 0; zeros in group 1); SAVED: s_mask[g][n] holds mask word g of record n already.  b1r, b2r: the
// primitive's bias rows in global memory (L1-resident).
template <typename T, bool SAVED>
__device__ __forceinline__ void vjp16_block(const Vjp16Operands<T>& w, Vjp16Sums& sum, const float x[3], float4 d3,
                                            bool live, const int32_t (*s_mask)[32], const float kf[6],
                                            const float* __restrict__ b1r, const float* __restrict__ b2r, float scale,
                                            int n, int g) {
  const vf32x16 zero = splat16(0.f);
  // ---- encoding, record-major
  u32x4 enc[5];
#pragma unroll
  for (int s = 0; s < 5; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const int t = 4 * s + d;
      if (t < 18) {
        const float rev = x[t / 6] * kf[t % 6];
        enc[s][d] = live ? Ops<T>::pack2(__builtin_amdgcn_sinf(rev), __builtin_amdgcn_cosf(rev)) : 0u;
      } else if (t == 18) {
        enc[s][d] = (live && g == 0) ? w.one_lo : 0u;      // the constant input (k = 68): bias gradient of layer 1
      } else {
        enc[s][d] = 0u;
      }
    }
  u32x4 d3op = {0u, 0u, 0u, 0u};                        // rounded, scaled output adjoints (group 0)
  d3op[0] = Ops<T>::pack2(d3.x * scale, d3.y * scale);
  d3op[1] = Ops<T>::pack2(d3.z * scale, d3.w * scale);
  sum.gb3[0] += Unpack<T>::lo(d3op[0]);
  sum.gb3[1] += Unpack<T>::hi(d3op[0]);
  sum.gb3[2] += Unpack<T>::lo(d3op[1]);
  sum.gb3[3] += Unpack<T>::hi(d3op[1]);

  // ---- layer 1 in both orientations
  vf32x16 a_rec, a_unit = splat16(w.bias1);
  {
    // record-major: register i is unit d_row(i, g); its bias comes from global memory (L1-resident)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(b1r + 8 * q + 4 * g);
      a_rec[4 * q] = v.x;
      a_rec[4 * q + 1] = v.y;
      a_rec[4 * q + 2] = v.z;
      a_rec[4 * q + 3] = v.w;
    }
  }
#pragma unroll
  for (int s = 0; s < 5; ++s) {
    a_rec = Ops<T>::mfma(w.w1op[s], enc[s], a_rec);
    a_unit = Ops<T>::mfma(enc[s], w.w1op[s], a_unit);
  }
  const Pack8 h1_rec = relu_tile(pack_tile<T>(a_rec));
  const Pack8 h1_unit = relu_tile(pack_tile<T>(a_unit));
  // ---- layer 2: unit-major for the W3 gradient; record-major only to learn which units are active
  const Pack8 h2_unit = relu_tile(pack_tile<T>(mma2<T>(h1_rec, w.w2op, splat16(w.bias2))));
  Pack8 act1_unit, act2_unit, act2_rec;
  if constexpr (SAVED) {
    int32_t words[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 v = *reinterpret_cast<const int4*>(&s_mask[0][8 * q + 4 * g]);
      words[4 * q] = v.x;
      words[4 * q + 1] = v.y;
      words[4 * q + 2] = v.z;
      words[4 * q + 3] = v.w;
    }
    act1_unit = mask_tile_unit_major(words, n);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 v = *reinterpret_cast<const int4*>(&s_mask[1][8 * q + 4 * g]);
      words[4 * q] = v.x;
      words[4 * q + 1] = v.y;
      words[4 * q + 2] = v.z;
      words[4 * q + 3] = v.w;
    }
    act2_unit = mask_tile_unit_major(words, n);
    act2_rec = mask_tile_record_major(s_mask[1][n], g);
  } else {
    vf32x16 a2;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(b2r + 8 * q + 4 * g);
      a2[4 * q] = v.x;
      a2[4 * q + 1] = v.y;
      a2[4 * q + 2] = v.z;
      a2[4 * q + 3] = v.w;
    }
    act1_unit = active_tile(h1_unit);
    act2_unit = active_tile(h2_unit);
    act2_rec = active_tile(relu_tile(pack_tile<T>(mma2<T>(w.w2op, h1_rec, a2))));
  }
  // ---- backward: D2 in both orientations, D1 unit-major, the output adjoints unit-major
  const Pack8 d2_rec = and_tile(pack_tile<T>(Ops<T>::mfma(w.w3op, d3op, zero)), act2_rec);
  const Pack8 d2_unit = and_tile(pack_tile<T>(Ops<T>::mfma(d3op, w.w3op, zero)), act2_unit);
  const Pack8 d1_unit = and_tile(pack_tile<T>(mma2<T>(d2_rec, w.w2top, zero)), act1_unit);
  const Pack8 d3_unit = pack_tile<T>(Ops<T>::mfma(d3op, w.out_sel, zero));
  sum.gb2 += sum_tile<T>(d2_unit);
  // ---- weight gradients: contraction over the records in the k-slots of the unit-major tiles
  sum.gw2 = mma2<T>(d2_unit, h1_unit, sum.gw2);
  sum.gw3 = mma2<T>(d3_unit, h2_unit, sum.gw3);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    vf32x16 e = Ops<T>::mfma(enc[2 * c], w.k_sel[0], zero);
    if (c < 2) e = Ops<T>::mfma(enc[2 * c + 1], w.k_sel[1], e);
    sum.gw1[c] = mma2<T>(d1_unit, pack_tile<T>(e), sum.gw1[c]);
  }
}

// Where a primitive's gradients go: the six rows of a packed partial sum, or of the six gradient tensors.
struct GradRows {
  float *W1, *b1, *W2, *b2, *W3, *b3;
};
__device__ __forceinline__ GradRows packed_grad_rows(float* row) {
  return GradRows{row, row + 2304, row + 2336, row + 3360, row + 3392, row + 3520};
}

// accumulator column n, rows d_row(i, g) -> rows; returns whether a value was not finite
__device__ __forceinline__ bool vjp16_store(Vjp16Sums& sum, const GradRows& out, float inv, int lane) {
  const int n = lane & 31, g = lane >> 5;
  bool bad = false;
  const auto put = [&](float* dst, float v) {
    bad |= !(__builtin_fabsf(v) <= 3.4028235e38f);
    *dst = v;
  };
  int feature[3];       // W1 column of encoding slot k = 32 c + n; -1: padding, -2: the constant input
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const int k = 32 * c + n, q = 8 * (k >> 4) + (k & 7), gk = (k >> 3) & 1;
    feature[c] = q < 36 ? (q & 1) * 36 + 18 * gk + (q >> 1) : ((q == 36 && gk == 0) ? -2 : -1);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int row = 8 * (i >> 2) + 4 * g + (i & 3);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (feature[c] >= 0) put(out.W1 + row * 72 + feature[c], sum.gw1[c][i] * inv);
      else if (feature[c] == -2) put(out.b1 + row, sum.gw1[c][i] * inv);
    }
    put(out.W2 + row * 32 + n, sum.gw2[i] * inv);
    if (row < 4) put(out.W3 + row * 32 + n, sum.gw3[i] * inv);
  }
  const float gb2 = sum.gb2 + __shfl_xor(sum.gb2, 32);
  if (g == 0) put(out.b2 + n, gb2 * inv);
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    float v = sum.gb3[o];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    if (lane == o) put(out.b3 + o, v * inv);
  }
  return bad;
}

}  // namespace mlpsp
