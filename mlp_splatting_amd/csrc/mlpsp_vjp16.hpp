// Weight gradients of the per-primitive 72->32->32->4 MLP over blocks of 32 records of one primitive, in 16-bit operands
// with f32 accumulation: the grouped kernel over a CSR of records (mlpsp_grouped_vjp.hip), and what the kernel over
// training steps (mlpsp_vjp16_steps.hpp) takes from it.
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
// Per block of 32 records: 30 MFMAs of 32 clocks and 8 small ones (32 without saved masks) against 20 for a formulation
// that transposes through LDS.  The 4x32 gradient of W3 and the bias gradient of layer 2 are 4x4x4 products: their 4 rows
// would fill an eighth of a 32x32 tile.  Bound by the ~350 vector instructions of a block: a wavefront that is alone on its
// SIMD issues them at half the rate, so the weight operands lie in LDS and two wavefronts fit (252 registers; with the
// operands in registers 342 and one wavefront; over training steps, which ran these blocks before mlpsp_vjp16_steps.hpp, the one
// took 2.06 ms for 648,000 steps, the other 3.18).
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
// 0xFFFF in each half whose bit 15 - up is set, 0 in the other
__device__ __forceinline__ unsigned spread_bit(unsigned halves, vu16x2 up) {
  typedef short vi16x2 __attribute__((ext_vector_type(2)));
  const vu16x2 top = __builtin_bit_cast(vu16x2, halves) << up;
  return __builtin_bit_cast(unsigned, (vi16x2)(__builtin_bit_cast(vi16x2, top) >> (vi16x2){15, 15}));
}
// Mask words of the block's records, split in halves: half h of the word of record m at [h][m].  A lane that looks at
// unit n takes the half that holds bit n, four consecutive records in one 8-byte read, already paired as the packed
// tiles pair them.
struct Vjp16Masks {
  unsigned short half[2][2][32];     // [layer][half][record]
  __device__ __forceinline__ void put(int layer, int record, uint32_t word) {
    half[layer][0][record] = (unsigned short)word;
    half[layer][1][record] = (unsigned short)(word >> 16);
  }
};
__device__ __forceinline__ Pack8 mask_tile_unit_major(const unsigned short (*half)[32], int n, int g) {
  const unsigned short* __restrict__ src = half[n >> 4] + 4 * g;
  const unsigned short shift = (unsigned short)(15 - (n & 15));
  const vu16x2 up = {shift, shift};
  Pack8 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint2 v = *reinterpret_cast<const uint2*>(src + 8 * q);
    r.s[q >> 1][2 * (q & 1)] = spread_bit(v.x, up);
    r.s[q >> 1][2 * (q & 1) + 1] = spread_bit(v.y, up);
  }
  return r;
}
// ... and of a record-major tile whose register i holds unit hidden_unit(i, g): the two units of a pair are bits k and
// k + 16 of this lane's word
__device__ __forceinline__ Pack8 mask_tile_record_major(uint32_t word, int g) {
  const unsigned mine = (word >> (8 * g)) & 0x00ff00ffu;
  Pack8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned short shift = (unsigned short)(15 - (4 * s + d));
      r.s[s][d] = spread_bit(mine, vu16x2{shift, shift});
    }
  return r;
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

// The primitive's weights as operands, one unit (n) per lane, and the selection operands, in LDS: they change per primitive
// and are read once per block (15 reads of 16 bytes), which leaves the registers to the sums and the tiles.
template <typename T>
struct Vjp16Operands {
  u32x4 w1[5][64], w2[2][64], w2t[2][64];  // w2: W2[n][u] over the units u = d_row(8 s + j, g) of a lane's k-slots; w2t:
                                           // W2[u][n] over u = hidden_unit(8 s + j, g)
  u32x4 k_sel[2][64];                      // returns K-step 2c + h of the encoding as columns 32c + n
  u32x2 w3u[64], w3r[64];                  // W3 column of unit n, of unit hidden_unit_of_row(n) (k-slots: the four outputs)
  float bias1[32], bias2[32];

  // What is the same for every primitive.
  __device__ __forceinline__ void select(int lane) {
    const int n = lane & 31, g = lane >> 5;
    const unsigned v = (n & 1) ? Ops<T>::pack2(0.f, 1.f) : Ops<T>::pack2(1.f, 0.f);
    const bool mine = ((n >> 3) & 1) == g;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 k;
#pragma unroll
      for (int d = 0; d < 4; ++d) k[d] = (mine && (n >> 4) == h && ((n & 7) >> 1) == d) ? v : 0u;
      k_sel[h][lane] = k;
    }
  }

  __device__ __forceinline__ void load(const float* __restrict__ W1, const float* __restrict__ b1,
                                       const float* __restrict__ W2, const float* __restrict__ b2,
                                       const float* __restrict__ W3, size_t p, int lane) {
    const int n = lane & 31, g = lane >> 5;
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
      for (int s = 0; s < 5; ++s) {
        u32x4 v;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const int t = 4 * s + d;
          v[d] = t < 18 ? Ops<T>::pack2(ws[t], wc[t]) : 0u;
        }
        w1[s][lane] = v;
      }
    }
    {
      const float* __restrict__ row = W2 + p * 1024 + n * 32;
      const float* __restrict__ col = W2 + p * 1024 + n;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float4 lo = *reinterpret_cast<const float4*>(row + 16 * s + 4 * g);
        const float4 hi = *reinterpret_cast<const float4*>(row + 16 * s + 8 + 4 * g);
        w2[s][lane] = u32x4{Ops<T>::pack2(lo.x, lo.y), Ops<T>::pack2(lo.z, lo.w), Ops<T>::pack2(hi.x, hi.y), Ops<T>::pack2(hi.z, hi.w)};
        float c[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) c[j] = col[hidden_unit(8 * s + j, g) * 32];
        w2t[s][lane] = u32x4{Ops<T>::pack2(c[0], c[1]), Ops<T>::pack2(c[2], c[3]), Ops<T>::pack2(c[4], c[5]), Ops<T>::pack2(c[6], c[7])};
      }
    }
    // W3^T: k-slots = the four outputs (group 0, slots 0..3; group 1's are zero)
    {
      const float* __restrict__ u = W3 + p * 128 + n;
      const float* __restrict__ r = W3 + p * 128 + hidden_unit_of_row(n);
      w3u[lane] = g ? u32x2{0u, 0u} : u32x2{Ops<T>::pack2(u[0], u[32]), Ops<T>::pack2(u[64], u[96])};
      w3r[lane] = g ? u32x2{0u, 0u} : u32x2{Ops<T>::pack2(r[0], r[32]), Ops<T>::pack2(r[64], r[96])};
    }
    if (g == 0) {
      bias1[n] = b1[p * 32 + n];
      bias2[n] = b2[p * 32 + n];
    }
  }
};

struct Vjp16Sums {
  vf32x16 gw1[3], gw2;
  f32x4 gw3, gb2;
  float gb3[4];
  __device__ __forceinline__ void clear() {
    gw1[0] = gw1[1] = gw1[2] = gw2 = splat16(0.f);
    gw3 = gb2 = f32x4{0.f, 0.f, 0.f, 0.f};
    gb3[0] = gb3[1] = gb3[2] = gb3[3] = 0.f;
  }
};

// The four 4x4x4 products over the records of two packed unit-major tiles: every group of four lanes is a block of its
// own, row l % 4 of a against column l % 4 of b.
template <typename T>
__device__ __forceinline__ f32x4 mma4(const Pack8& a, const Pack8& b, f32x4 acc) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int s = q >> 1, d = 2 * (q & 1);
    acc = Ops<T>::mfma4(u32x2{a.s[s][d], a.s[s][d + 1]}, u32x2{b.s[s][d], b.s[s][d + 1]}, acc);
  }
  return acc;
}

// The bias of a record-major tile: register i holds unit d_row(i, g) (rows), or of a row order of the caller's
__device__ __forceinline__ vf32x16 bias_rows(const float* bias, int g) {
  vf32x16 r;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(bias + 8 * q + 4 * g);
#pragma unroll
    for (int k = 0; k < 4; ++k) r[4 * q + k] = v[k];
  }
  return r;
}

// One block of 32 records.  Lane (n, g): record n; x = its three inputs of group g, d3 = the record's output adjoints
// (lanes of group 0; zeros in group 1); SAVED: `masks` holds the mask words of the block's records, mask2 is that of
// record n and layer 2.
template <typename T, bool SAVED>
__device__ __forceinline__ void vjp16_block(const Vjp16Operands<T>& w, Vjp16Sums& sum, const float x[3], float4 d3,
                                            bool live, const Vjp16Masks& masks, uint32_t mask2, const float kf[6],
                                            float scale, int lane) {
  // (opaque: the operands are to be read here, not kept in registers from block to block)
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5;
  const vf32x16 zero = splat16(0.f);
  const unsigned one_lo = Ops<T>::pack2(1.f, 0.f), one_hi = Ops<T>::pack2(0.f, 1.f);
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
        enc[s][d] = (live && g == 0) ? one_lo : 0u;      // the constant input (k = 68): bias gradient of layer 1
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
  vf32x16 a_rec = bias_rows(w.bias1, g), a_unit = splat16(w.bias1[n]);
#pragma unroll
  for (int s = 0; s < 5; ++s) {
    const u32x4 w1 = w.w1[s][lane];
    a_rec = Ops<T>::mfma(w1, enc[s], a_rec);
    a_unit = Ops<T>::mfma(enc[s], w1, a_unit);
  }
  const Pack8 h1_rec = relu_tile(pack_tile<T>(a_rec));
  const Pack8 h1_unit = relu_tile(pack_tile<T>(a_unit));
  // ---- layer 2: unit-major for the W3 gradient; record-major only to learn which units are active
  const Pack8 w2 = {{w.w2[0][lane], w.w2[1][lane]}};
  const Pack8 h2_unit = relu_tile(pack_tile<T>(mma2<T>(h1_rec, w2, splat16(w.bias2[n]))));
  Pack8 act1_unit, act2_unit, act2_rec;
  if constexpr (SAVED) {
    act1_unit = mask_tile_unit_major(masks.half[0], n, g);
    act2_unit = mask_tile_unit_major(masks.half[1], n, g);
    act2_rec = mask_tile_record_major(mask2, g);
  } else {
    // rows of the product = units hidden_unit(i, g), as mask_tile_record_major has them
    const int m = (lane & 32) | hidden_unit_of_row(n);
    const Pack8 w2r = {{w.w2[0][m], w.w2[1][m]}};
    vf32x16 a2;
#pragma unroll
    for (int i = 0; i < 16; ++i) a2[i] = w.bias2[hidden_unit(i, 0) + 8 * g];
    act1_unit = active_tile(h1_unit);
    act2_unit = active_tile(h2_unit);
    act2_rec = active_tile(relu_tile(pack_tile<T>(mma2<T>(w2r, h1_rec, a2))));
  }
  // ---- backward: D2 in both orientations, D1 unit-major, the output adjoints unit-major (column n = output n % 4)
  const u32x2 w3r = w.w3r[lane], w3u = w.w3u[lane];
  const unsigned pick = (n & 1) ? one_hi : one_lo;
  const u32x4 out_sel = {(g == 0 && !(n & 2)) ? pick : 0u, (g == 0 && (n & 2)) ? pick : 0u, 0u, 0u};
  const Pack8 d2_rec = and_tile(pack_tile<T>(Ops<T>::mfma(u32x4{w3r[0], w3r[1], 0u, 0u}, d3op, zero)), act2_rec);
  const Pack8 d2_unit = and_tile(pack_tile<T>(Ops<T>::mfma(d3op, u32x4{w3u[0], w3u[1], 0u, 0u}, zero)), act2_unit);
  const Pack8 d3_unit = pack_tile<T>(Ops<T>::mfma(d3op, out_sel, zero));
  const Pack8 w2t = {{w.w2t[0][lane], w.w2t[1][lane]}};
  const Pack8 d1_unit = and_tile(pack_tile<T>(mma2<T>(d2_rec, w2t, zero)), act1_unit);
  // ---- weight gradients: contraction over the records in the k-slots of the unit-major tiles
  Pack8 ones;
#pragma unroll
  for (int d = 0; d < 4; ++d) ones.s[0][d] = ones.s[1][d] = Ops<T>::kOneWord;
  sum.gb2 = mma4<T>(ones, d2_unit, sum.gb2);
  sum.gw3 = mma4<T>(d3_unit, h2_unit, sum.gw3);
  sum.gw2 = mma2<T>(d2_unit, h1_unit, sum.gw2);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    vf32x16 e = Ops<T>::mfma(enc[2 * c], w.k_sel[0][lane], zero);
    if (c < 2) e = Ops<T>::mfma(enc[2 * c + 1], w.k_sel[1][lane], e);
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
  }
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    const float v = sum.gw3[o] + __shfl_xor(sum.gw3[o], 32);
    if (g == 0) put(out.W3 + o * 32 + n, v * inv);
  }
  const float gb2 = sum.gb2[0] + __shfl_xor(sum.gb2[0], 32);
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
