// Wave-level f32 evaluation of one primitive's 72->32->32->4 (or 72->16->16->4) MLP for the 64 pixels of a
// wavefront on the matrix cores, bit-identical to the scalar chain of mlp_fixed<32, 6> (mlp_fixed<16, 6>).
//
// v_mfma_f32_32x32x2_f32 computes, per output element, fma(a1, b1, fma(a0, b0, c)) with both steps
// rounded as IEEE f32 fused multiply-adds (no flush of denormals): one instruction is two consecutive links
// of the reference's accumulation chain (np_tile_kernels.cu:2050-2089), so 36 of them walk layer 1 in the
// order sin_j, cos_j and 16 walk layer 2 in the order h = 2i, 2i+1.
//
// Operand layout.  The wavefront's pixels form two column blocks (pixels 0..31 and 32..63), one accumulator
// tile each.  Lane (n = lane % 32, g = lane / 32) of a 32x32 f32 accumulator tile holds column n and rows
// 8q + 4g + r in register 4q + r.  The weight rows are fed in permuted order -- row 8q + 4g + r of the
// A operand is hidden unit 2(4q + r) + g -- so register i of lane (n, g) holds hidden unit 2i + g: exactly
// the B operand (k = g) of the next layer's i-th instruction.  Layer outputs therefore feed the next layer
// from registers, with a ReLU in between and no shuffles.  Layer-1 inputs are computed per lane = pixel and
// moved into operand position by one half-wave swap per sin/cos pair; the same swap brings the 32 layer-2
// outputs of a pixel onto its own lane for the 4-wide output layer, which runs on the vector ALU with
// scalar weight operands.
// 16 hidden units run on the 16x16x4 form (mlp_wave_mfma16x4 below).
#pragma once
#include "mlpsp_device.hpp"

namespace mlpsp {

typedef float mf32x16 __attribute__((ext_vector_type(16)));
typedef float mf32x4 __attribute__((ext_vector_type(4)));

// Exchanges lanes 32..63 of a with lanes 0..31 of b.
__device__ __forceinline__ void half_swap(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void half_swap(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Exchanges the odd rows of 16 lanes of a with the even rows of b.
__device__ __forceinline__ void row_swap(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}

// 16 consecutive floats at src + 16 g, as loaded (c[q] = floats 4q .. 4q+3)  ->  element i = src[2i + g]
// (g = lane / 32): eight swaps pair the even entries of the two half-waves.
__device__ __forceinline__ void interleave16(const mf32x4 c4[4], float v[16]) {
  float c[16];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    c[4 * q + 0] = c4[q][0];
    c[4 * q + 1] = c4[q][1];
    c[4 * q + 2] = c4[q][2];
    c[4 * q + 3] = c4[q][3];
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    half_swap(c[2 * t], c[2 * t + 1]);   // c[2t] = (src[2t], src[2t+1]), c[2t+1] = (src[16+2t], src[17+2t])
    v[t] = c[2 * t];
    v[8 + t] = c[2 * t + 1];
  }
}

// What one lane loads of a primitive's layers 1 and 2, as the loads deliver it: row `hid` of W1 (its half g) and
// the first bias vector (its half g); the same row of W2 and the second bias vector.  Requesting is separate from
// using, and layer 1 from layer 2: those of layer 2 arrive behind layer 1's instructions.
struct MlpLayer1 {
  mf32x4 a1[9], b1[4];
};
struct MlpLayer2 {
  mf32x4 a2[4], b2[4];
};
// Hidden unit whose weight row lane (m, g) supplies.
__device__ __forceinline__ int mfma32_hidden_row(int m) { return 8 * (m >> 3) + 2 * (m & 3) + ((m >> 2) & 1); }
__device__ __forceinline__ void request_layer1(const float* __restrict__ W1, const float* __restrict__ b1, int p,
                                               MlpLayer1& o) {
  const int lane = threadIdx.x & 63, m = lane & 31, g = lane >> 5;
  const mf32x4* __restrict__ s1 =
      reinterpret_cast<const mf32x4*>(W1 + (size_t)p * (32 * 72) + mfma32_hidden_row(m) * 72 + 36 * g);
#pragma unroll
  for (int q = 0; q < 9; ++q) o.a1[q] = s1[q];
  const mf32x4* __restrict__ sb1 = reinterpret_cast<const mf32x4*>(b1 + (size_t)p * 32 + 16 * g);
#pragma unroll
  for (int q = 0; q < 4; ++q) o.b1[q] = sb1[q];
}
__device__ __forceinline__ void request_layer2(const float* __restrict__ W2, const float* __restrict__ b2, int p,
                                               MlpLayer2& o) {
  const int lane = threadIdx.x & 63, m = lane & 31, g = lane >> 5;
  const mf32x4* __restrict__ s2 =
      reinterpret_cast<const mf32x4*>(W2 + (size_t)p * (32 * 32) + mfma32_hidden_row(m) * 32 + 16 * g);
  const mf32x4* __restrict__ sb2 = reinterpret_cast<const mf32x4*>(b2 + (size_t)p * 32 + 16 * g);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    o.a2[q] = s2[q];
    o.b2[q] = sb2[q];
  }
}

// max(x, +0): the same bits as x > 0 ? x : 0 for every x (NaN -> 0, -0 -> +0).  v_med3_f32 with 0 and +inf is one
// instruction; fmaxf() is two, because the compiler quiets a possible signalling NaN first (128 of the 1,150 vector
// instructions of a hit step).  The infinity is hidden from the compiler, which would turn a median with it into that
// maximum.  A builtin, not inline assembly: the compiler must see the instruction to keep the wait states between a
// matrix-core result and its first reader.
__device__ __forceinline__ float relu_limit() {
  float inf = __builtin_inff();
  asm("" : "+s"(inf));
  return inf;
}
__device__ __forceinline__ float relu_f32(float x, float inf) { return __builtin_amdgcn_fmed3f(x, 0.f, inf); }

// det_sincos() for |x| <= 65536, the same bits: no range check, the quadrant's signs by exclusive-or.
__device__ __forceinline__ void det_sincos_in_range(float x, float& s_out, float& c_out) {
  const float kf = __builtin_rintf(x * 0.636619772f);
  float r = fmaf(kf, -1.5703125f, x);
  r = fmaf(kf, -4.83751297e-04f, r);
  r = fmaf(kf, -7.54978995e-08f, r);
  const float z = r * r;
  float ps = 2.75573192e-06f;
  ps = fmaf(ps, z, -1.98412698e-04f);
  ps = fmaf(ps, z, 8.33333333e-03f);
  ps = fmaf(ps, z, -1.66666667e-01f);
  const float s = fmaf(r * z, ps, r);
  float pc = -2.75573192e-07f;
  pc = fmaf(pc, z, 2.48015873e-05f);
  pc = fmaf(pc, z, -1.38888889e-03f);
  pc = fmaf(pc, z, 4.16666667e-02f);
  const float c = fmaf(z * z, pc, fmaf(z, -0.5f, 1.0f));
  const uint32_t q = (uint32_t)(int)kf;
  const bool odd = (q & 1u) != 0u;
  const uint32_t turn = q << 30;             // bit 31: the sine's sign; one more quarter turn: the cosine's
  s_out = bits_to_float(float_to_bits(odd ? c : s) ^ (turn & 0x80000000u));
  c_out = bits_to_float(float_to_bits(odd ? s : c) ^ ((turn + 0x40000000u) & 0x80000000u));
}
// The six (sin, cos) pairs of one input component, bit for bit det_sincos((x freq_f) att_f).  One test covers the
// range of all six (a NaN fails it too); phases beyond it, which no scene has in earnest, are put right behind a branch
// that the whole wavefront skips.
__device__ __forceinline__ void encode_component(float x, const float* __restrict__ freq, const float* __restrict__ att,
                                                 float s[6], float c[6]) {
  float phase[6];
#pragma unroll
  for (int f = 0; f < 6; ++f) phase[f] = (x * freq[f]) * att[f];
  const float reach = ((__builtin_fabsf(phase[0]) + __builtin_fabsf(phase[1])) +
                       (__builtin_fabsf(phase[2]) + __builtin_fabsf(phase[3]))) +
                      (__builtin_fabsf(phase[4]) + __builtin_fabsf(phase[5]));
#pragma unroll
  for (int f = 0; f < 6; ++f) det_sincos_in_range(phase[f], s[f], c[f]);
  if (__ballot(!(reach <= 65536.0f)) != 0ull) {
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      float again = x;                       // (or the six comparisons are made ahead of the branch)
      asm volatile("" : "+v"(again));
      const bool ok = __builtin_fabsf((again * freq[f]) * att[f]) <= 65536.0f;
      s[f] = ok ? s[f] : __builtin_nanf("");
      c[f] = ok ? c[f] : __builtin_nanf("");
    }
  }
}

// The encoding of the ray direction (input components 0..2) does not depend on the primitive: its 18 sin/cos pairs are
// computed once per pixel and parked in LDS in B-operand position (after the half-wave swap), four instructions' worth
// per 16-byte read.  Written and read by one wavefront: no barrier.  (36 registers less than keeping them: a fourth
// wavefront per SIMD.)
struct DirOperands {
  mf32x4 q[9][64];       // [i]: pairs 2i and 2i + 1.  32 hidden units: blocks 0 and 1 of either = (b0[2i], b1[2i], b0[2i+1],
};                       // b1[2i+1]); 16: blocks 0 .. 3 of the two together (mlp_wave_mfma16x4)
// Four values of every pixel, exchanged between the four rows of 16 lanes: afterwards lane (c, q) holds in v[b] what lane
// (c, b) = pixel 16 b + c had in v[q].
__device__ __forceinline__ void row_transpose(float v[4]) {
  half_swap(v[0], v[2]);
  half_swap(v[1], v[3]);
  row_swap(v[0], v[1]);
  row_swap(v[2], v[3]);
}
template <int HID = 32>
__device__ __forceinline__ void encode_direction(float rdx, float rdy, float rdz, const float* __restrict__ freq,
                                                 const float* __restrict__ att, DirOperands& d) {
  const int lane = threadIdx.x & 63;
  const float x3[3] = {rdx, rdy, rdz};
  for (int c = 0; c < 3; ++c) {
    float s[6], co[6];
    encode_component(c == 0 ? x3[0] : c == 1 ? x3[1] : x3[2], freq, att, s, co);
    if constexpr (HID == 32) {
#pragma unroll
      for (int f = 0; f < 6; ++f) half_swap(s[f], co[f]);
    }
#pragma unroll
    for (int f = 0; f < 6; f += 2) {
      float v[4] = {s[f], co[f], s[f + 1], co[f + 1]};
      if constexpr (HID == 16) row_transpose(v);
      d.q[3 * c + f / 2][lane] = mf32x4{v[0], v[1], v[2], v[3]};
    }
  }
}

// `mask` shifted left by BITS, the lowest of which say whether the rectified value r is positive: the highest of them does, as the
// sign of 0 - r (+0 where r is a zero), the other is r's.  Two instructions a value; compared, selected and or-ed they are three,
// each of the slower kind, and layer 1's accumulators need not outlive layer 2 (168 -> 146 registers; training forward of the
// 200,000-primitive 1200x680 frame 4.08 -> 4.01 ms).
template <int BITS>
__device__ __forceinline__ uint32_t push_positive(uint32_t mask, float r) {
  return __builtin_amdgcn_alignbit(mask, float_to_bits(0.f - r), 32 - BITS);
}

// All 64 lanes must be active.  x6 is the lane's own pixel's input (components 0..2 enter through dir,
// which encode_direction() made from them); out is the lane's own pixel's output.  `w1` = the primitive's layer-1
// operands as request_layer1() loaded them; layer2(w2) requests those of layer 2.  REC selects the record kernels' layer-2
// rounding (bias added after a chain started at zero); MASKS fills masks[0..1] with the ReLU masks of the lane's pixel.
// (mlp_wave_mfma32 is the one caller.  With its requests written here the compiler places them otherwise: the f32 frame and the
// training forward are 0.4 to 0.7 % slower.)
template <bool REC, bool MASKS, typename RequestLayer2>
__device__ __forceinline__ void mlp_wave_mfma32_with(const MlpLayer1& w1, RequestLayer2&& layer2, const float x6[6],
                                                     const float* __restrict__ freq, const float* __restrict__ att,
                                                     const float* __restrict__ W3, const float* __restrict__ b3, int p,
                                                     const DirOperands& dir, float out[4], uint32_t* masks) {
  constexpr int H = 32, R = H / 2;    // R: accumulator registers (hidden units 2i + g)
  const int lane = threadIdx.x & 63, g = lane >> 5;
  const float inf = relu_limit();

  // A operands: lane (m, g) supplies row hid, k = g of every instruction.
  float a1[36];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    a1[4 * q + 0] = w1.a1[q][0];
    a1[4 * q + 1] = w1.a1[q][1];
    a1[4 * q + 2] = w1.a1[q][2];
    a1[4 * q + 3] = w1.a1[q][3];
  }
  float bias1[16];
  interleave16(w1.b1, bias1);

  mf32x16 d0, d1;
#pragma unroll
  for (int i = 0; i < 16; ++i) d0[i] = d1[i] = bias1[i];
  // (the lane index is made opaque so that the reads stay here and are not hoisted out of the primitive loop)
  int ll = lane;
  asm volatile("" : "+v"(ll));
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const mf32x4 q = dir.q[i][ll];
    d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[2 * i], q[0], d0, 0, 0, 0);
    d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[2 * i], q[1], d1, 0, 0, 0);
    d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[2 * i + 1], q[2], d0, 0, 0, 0);
    d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[2 * i + 1], q[3], d1, 0, 0, 0);
  }
  MlpLayer2 w2;
#pragma unroll
  for (int c = 3; c < 6; ++c) {
    // (layer 2's operands are requested behind five sixths of layer 1, and not before: 32 registers)
    if (c == 5) layer2(w2);
    float sn[6], cs[6];
    encode_component(x6[c], freq, att, sn, cs);
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      float s = sn[f], co = cs[f];
      half_swap(s, co);   // s: (sin, cos) of pixels 0..31, co: (sin, cos) of pixels 32..63
      d0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[c * 6 + f], s, d0, 0, 0, 0);
      d1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[c * 6 + f], co, d1, 0, 0, 0);
    }
  }

  float a2[16], bias2[16];
  interleave16(w2.a2, a2);
  interleave16(w2.b2, bias2);
  mf32x16 e0, e1;
#pragma unroll
  for (int i = 0; i < 16; ++i) e0[i] = e1[i] = REC ? 0.f : bias2[i];
  uint32_t lo = 0u, hi = 0u;   // bits 31 - 2i: unit 2i + g of blocks 0 and 1
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float r0 = relu_f32(d0[i], inf), r1 = relu_f32(d1[i], inf);
    e0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[i], r0, e0, 0, 0, 0);
    e1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[i], r1, e1, 0, 0, 0);
    if constexpr (MASKS) {
      lo = push_positive<2>(lo, r0);
      hi = push_positive<2>(hi, r1);
    }
  }
  if constexpr (REC) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      e0[i] = bias2[i] + e0[i];
      e1[i] = bias2[i] + e1[i];
    }
  }

  // Output layer on the lane's own pixel: register i of the two blocks, swapped, is (h2[2i], h2[2i+1]).
  const float* __restrict__ w3 = W3 + (size_t)p * (4 * H);
  const float* __restrict__ bb3 = b3 + (size_t)p * 4;
  float acc[4] = {bb3[0], bb3[1], bb3[2], bb3[3]};
  uint32_t m2 = 0u;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float even = relu_f32(e0[i], inf), odd = relu_f32(e1[i], inf);
    half_swap(even, odd);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      acc[k] = fmaf(w3[k * H + 2 * i], even, acc[k]);
      acc[k] = fmaf(w3[k * H + 2 * i + 1], odd, acc[k]);
    }
    if constexpr (MASKS) m2 = push_positive<1>(push_positive<1>(m2, even), odd);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = acc[k];
  if constexpr (MASKS) {
    half_swap(lo, hi);         // the lane's pixel: even units, odd units
    masks[0] = (__brev(lo) & 0x55555555u) | ((__brev(hi) & 0x55555555u) << 1);
    masks[1] = __brev(m2);
  }
}

// The 72->16->16->4 MLP, the same contract: v_mfma_f32_16x16x4_f32 is four consecutive links of the chain, k = 0 .. 3 (one
// rounding each, as the 32x32x2's two), in 32 clocks, and has no half-filled rows: four column blocks of 16 pixels, 18
// instructions a block for layer 1 and four for layer 2, 2,816 clocks per evaluation where half-filled 32x32x2 tiles take
// 5,632 (frame of 5,000 primitives, 160x120: 268 -> 242 us; nine exchanges of rows more take back a tenth).  Lane (c, q) = (lane % 16, lane / 16) of an accumulator tile holds column c and rows 4 q + r in register r; with row
// 4 q + r = hidden unit 4 r + q that is the operand (k = q) of the next layer's r-th instruction.
__device__ __forceinline__ void mlp_wave_mfma16x4(const float x6[6], const float* __restrict__ freq, const float* __restrict__ att,
                                                  const float* __restrict__ W1, const float* __restrict__ b1,
                                                  const float* __restrict__ W2, const float* __restrict__ b2,
                                                  const float* __restrict__ W3, const float* __restrict__ b3, int p,
                                                  const DirOperands& dir, float out[4]) {
  const int lane = threadIdx.x & 63, c16 = lane & 15, q = lane >> 4;
  const int unit = 4 * (c16 & 3) + (c16 >> 2);
  const float inf = relu_limit();
  // W1: k-slots 0 .. 3 of instruction j = sine and cosine of pairs 2 j, 2 j + 1: every other entry of a half row
  const mf32x4* __restrict__ s1 = reinterpret_cast<const mf32x4*>(W1 + (size_t)p * (16 * 72) + unit * 72 + 36 * (q & 1));
  float a1[18];
#pragma unroll
  for (int i = 0; i < 9; ++i) {
    const mf32x4 v = s1[i];
    a1[2 * i] = q & 2 ? v[1] : v[0];
    a1[2 * i + 1] = q & 2 ? v[3] : v[2];
  }
  float bias1[4], a2[4], bias2[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bias1[i] = b1[(size_t)p * 16 + 4 * i + q];
    a2[i] = W2[(size_t)p * 256 + unit * 16 + 4 * i + q];
    bias2[i] = b2[(size_t)p * 16 + 4 * i + q];
  }
  mf32x4 d[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) d[b] = mf32x4{bias1[0], bias1[1], bias1[2], bias1[3]};
  int ll = lane;                         // (opaque: the reads stay here and are not hoisted out of the primitive loop)
  asm volatile("" : "+v"(ll));
#pragma unroll
  for (int j = 0; j < 9; ++j) {
    const mf32x4 x = dir.q[j][ll];
#pragma unroll
    for (int b = 0; b < 4; ++b) d[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[j], x[b], d[b], 0, 0, 0);
  }
#pragma unroll
  for (int c = 3; c < 6; ++c) {
    float sn[6], cs[6];
    encode_component(x6[c], freq, att, sn, cs);
#pragma unroll
    for (int f = 0; f < 6; f += 2) {
      float v[4] = {sn[f], cs[f], sn[f + 1], cs[f + 1]};
      row_transpose(v);
#pragma unroll
      for (int b = 0; b < 4; ++b) d[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[3 * c + f / 2], v[b], d[b], 0, 0, 0);
    }
  }
  mf32x4 e[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) e[b] = mf32x4{bias2[0], bias2[1], bias2[2], bias2[3]};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b) e[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[i], relu_f32(d[b][i], inf), e[b], 0, 0, 0);
  // output layer on the lane's own pixel
  const float* __restrict__ w3 = W3 + (size_t)p * 64;
  const float* __restrict__ bb3 = b3 + (size_t)p * 4;
  float acc[4] = {bb3[0], bb3[1], bb3[2], bb3[3]};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float h[4] = {relu_f32(e[0][i], inf), relu_f32(e[1][i], inf), relu_f32(e[2][i], inf), relu_f32(e[3][i], inf)};
    row_transpose(h);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[k] = fmaf(w3[k * 16 + 4 * i + u], h[u], acc[k]);
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = acc[k];
}

// The same with the operands requested here.
template <bool REC = false, bool MASKS = REC, int HID = 32>
__device__ __forceinline__ void mlp_wave_mfma32(const float x6[6], const float* __restrict__ freq,
                                                const float* __restrict__ att, const float* __restrict__ W1,
                                                const float* __restrict__ b1, const float* __restrict__ W2,
                                                const float* __restrict__ b2, const float* __restrict__ W3,
                                                const float* __restrict__ b3, int p, const DirOperands& dir,
                                                float out[4], uint32_t* masks = nullptr) {
  static_assert(HID == 32 || (HID == 16 && !REC && !MASKS), "hidden width of the matrix-core f32 evaluation");
  if constexpr (HID == 16) {
    mlp_wave_mfma16x4(x6, freq, att, W1, b1, W2, b2, W3, b3, p, dir, out);
  } else {
    MlpLayer1 w1;
    request_layer1(W1, b1, p, w1);
    const auto layer2 = [&](MlpLayer2& w2) {
      __builtin_amdgcn_sched_barrier(0);
      request_layer2(W2, b2, p, w2);
    };
    mlp_wave_mfma32_with<REC, MASKS>(w1, layer2, x6, freq, att, W3, b3, p, dir, out, masks);
  }
}

}  // namespace mlpsp
