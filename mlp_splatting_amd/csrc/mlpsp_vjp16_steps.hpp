// Weight gradients of the per-primitive 72->32->32->4 MLP over training steps in 16-bit operands (fp16 / bf16,
// v_mfma_f32_32x32x16, f32 accumulation): the roundings of mlpsp_vjp16.hpp -- encoding, weights, adjoints and hidden activations
// to the operand type, sums in f32 -- in the frame of mlpsp_vjp32.hpp: a workgroup shares a primitive's operands in LDS and deals
// its half steps to its wavefronts, and what a gradient needs with its records in the k-slots is read back from LDS with
// ds_read_b64_tr_b16 instead of being computed in both orientations or transposed by the matrix core: 16 large matrix
// instructions and ~250 vector instructions a block instead of 30 and 350.
//
// Bound by the latency of a block's chain of products, conversions and LDS.  Four wavefronts to a workgroup and three workgroups
// to a CU: while one changes primitives the others work.  Three wavefronts to a SIMD have 168 registers, which is what a block
// needs if its parts stay one behind the other (sched_barrier) and neither the lane's number nor an address is kept from one
// block to the next (fresh_lane); a word that spills is waited for behind the record requested ahead (2.04 ms with seven).
// Gradient call of 648,000 steps: 1.84 ms; two workgroups of four 1.96, one of eight 2.12, four of two 2.31; with the block of
// mlpsp_vjp16.hpp, a wavefront to a chunk of 64 steps, 2.54.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_mfma16.hpp"
#include "mlpsp_vjp16.hpp"
#include "mlpsp_vjp32.hpp"

namespace mlpsp {

constexpr int kVjp16Waves = 4, kVjp16Slots = 2;
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
  __attribute__((aligned(16))) float sums[kVjp16Slots][kGradFloats];    // in the end, two wavefronts to a row
};

// What a lane loads of a primitive's weights, as Vjp32Request: of W1 the pairs 4 wave .. 4 wave + 3; then wavefront 0 the pairs 16
// and 17, 1 and 2 rows and columns of W2, 3 W3 and the biases.
struct Vjp16Request {
  f32x4 sines, cosines, a, b;
  float c[8];
};
__device__ __forceinline__ Vjp16Request vjp16_request(const float* __restrict__ W1, const float* __restrict__ b1,
                                                      const float* __restrict__ W2, const float* __restrict__ b2,
                                                      const float* __restrict__ W3, size_t p, int wave, int lane) {
  asm volatile("" : "+v"(lane));         // (or the addresses are formed ahead of the loop over the runs, one by one)
  const int n = lane & 31, g = lane >> 5, k = wave == 2 ? 1 : 0;
  const float* row1 = W1 + p * 2304 + n * 72 + 18 * g;
  const float* a = wave == 0 ? row1 + 14 : W2 + p * 1024 + n * 32 + 16 * k + 4 * g;
  Vjp16Request r{load4_here(row1 + 4 * wave), load4_here(row1 + 36 + 4 * wave), load4_here(a), load4_here(wave == 0 ? a + 36 : a + 8), {}};
  const float *col = W2 + p * 1024 + n, *out = W3 + p * 128 + hidden_unit_of_row(n), *bias = (g ? b2 : b1) + p * 32 + n;
#pragma unroll
  for (int i = 0; i < 8; ++i) r.c[i] = load_here(wave == 3 ? (i < 4 ? out + 32 * i : bias) : col + hidden_unit(8 * k + i, g) * 32);
  return r;
}
// The primitive's weights into LDS, by the whole workgroup.
template <typename T>
__device__ __forceinline__ void vjp16_load(const Vjp16Request& r, int wave, int lane, Vjp16Shared<T>& s) {
  asm volatile("" : "+v"(lane));         // (as in vjp16_request)
  const int n = lane & 31, g = lane >> 5;
  s.w1[wave][lane] = u32x4{Ops<T>::pack2(r.sines[0], r.cosines[0]), Ops<T>::pack2(r.sines[1], r.cosines[1]),
                           Ops<T>::pack2(r.sines[2], r.cosines[2]), Ops<T>::pack2(r.sines[3], r.cosines[3])};
  if (wave == 0) {
    s.w1[4][lane] = u32x4{Ops<T>::pack2(r.a[2], r.b[2]), Ops<T>::pack2(r.a[3], r.b[3]), 0u, 0u};
  } else if (wave < 3) {
    s.w2[wave - 1][lane] = u32x4{Ops<T>::pack2(r.a[0], r.a[1]), Ops<T>::pack2(r.a[2], r.a[3]),
                                 Ops<T>::pack2(r.b[0], r.b[1]), Ops<T>::pack2(r.b[2], r.b[3])};
    s.w2t[wave - 1][lane] = u32x4{Ops<T>::pack2(r.c[0], r.c[1]), Ops<T>::pack2(r.c[2], r.c[3]),
                                  Ops<T>::pack2(r.c[4], r.c[5]), Ops<T>::pack2(r.c[6], r.c[7])};
  } else {
    s.w3r[lane] = g ? u32x2{0u, 0u} : u32x2{Ops<T>::pack2(r.c[0], r.c[1]), Ops<T>::pack2(r.c[2], r.c[3])};
    (g ? s.bias2 : s.bias1)[n] = r.c[4];
  }
}

struct Vjp16StepSums {
  vf32x16 gw1[2], gw2;
  f32x4 gw1e, gw3, gb;       // gb: rows 0 and 1 = b2, b1
  float gb3[2];              // outputs 2 g, 2 g + 1
  __device__ __forceinline__ void clear() {
    gw1[0] = gw1[1] = gw2 = splat16(0.f);
    gw1e = gw3 = gb = f32x4{0.f, 0.f, 0.f, 0.f};
    gb3[0] = gb3[1] = 0.f;
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
  lane = fresh_lane();
  const int n = lane & 31, g = lane >> 5;
  const vf32x16 zero = splat16(0.f);
  // (row n % 4 of the small products' first operand)
  const unsigned row0 = (n & 3) == 0 ? Ops<T>::kOneWord : 0u, row1 = (n & 3) == 1 ? Ops<T>::kOneWord : 0u;
  // ---- adjoints of layer 2: record in the lane, unit hidden_unit(i, g) in register i.  (Group 1 multiplies by zero.)
  s.mask.put(g, n, g ? mask2 : mask1);
  u32x4 d3 = {0u, 0u, 0u, 0u};
  d3[0] = Ops<T>::pack2(adjoint.x * scale, adjoint.y * scale);
  d3[1] = Ops<T>::pack2(adjoint.z * scale, adjoint.w * scale);
  if (g == 0) *reinterpret_cast<u32x2*>(s.d3[n]) = u32x2{d3[0], d3[1]};
  const unsigned mine = g ? d3[1] : d3[0];
  sum.gb3[0] += Unpack<T>::lo(mine);
  sum.gb3[1] += Unpack<T>::hi(mine);
  const u32x2 w3r = w.w3r[lane];
  const Pack8 d2 = and_tile(pack_tile<T>(Ops<T>::mfma(u32x4{w3r[0], w3r[1], 0u, 0u}, d3, zero)), mask_tile_record_major(mask2, g));
  const Pack8 d2t = transpose_tile(d2, s, n, g);
  __builtin_amdgcn_sched_barrier(0);
  // ---- adjoints of layer 1: unit in the lane
  const Pack8 d1 = and_tile(pack_tile<T>(mma2<T>(d2, Pack8{{w.w2t[0][lane], w.w2t[1][lane]}}, zero)),
                            mask_tile_unit_major(s.mask.half[0], n, g));
  __builtin_amdgcn_sched_barrier(0);
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
  __builtin_amdgcn_sched_barrier(0);
  const Pack8 h1 = relu_tile(pack_tile<T>(a1));
  const Pack8 h1t = transpose_tile(h1, s, n, g);
  __builtin_amdgcn_sched_barrier(0);
  // ---- layer 2: unit in the lane, straight into the W3 gradient
  const Pack8 h2 = relu_tile(pack_tile<T>(mma2<T>(h1, Pack8{{w.w2[0][lane], w.w2[1][lane]}}, splat16(w.bias2[n]))));
  const char* const d3_from = reinterpret_cast<const char*>(s.d3[4 * g + ((n >> 2) & 3)]);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = q >> 1, d = 2 * (q & 1);
    sum.gw3 = Ops<T>::mfma4(read_transposed(d3_from + 8 * q * 8), u32x2{h2.s[k][d], h2.s[k][d + 1]}, sum.gw3);
    sum.gb = Ops<T>::mfma4(u32x2{row0, row0}, u32x2{d2t.s[k][d], d2t.s[k][d + 1]}, sum.gb);
    sum.gb = Ops<T>::mfma4(u32x2{row1, row1}, u32x2{d1.s[k][d], d1.s[k][d + 1]}, sum.gb);
  }
  sum.gw2 = mma2<T>(d2t, h1t, sum.gw2);
  __builtin_amdgcn_sched_barrier(0);
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

// A wavefront's sums to a row of LDS, in the order of a packed row of gradients; ADD: onto what is there.
template <bool ADD>
__device__ __forceinline__ void vjp16_park(const Vjp16StepSums& sum, float* to, int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5;
  const GradRows out = packed_grad_rows(to);
  const auto put = [](float& at, float v) { at = ADD ? at + v : v; };
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 8 * (i >> 2) + 4 * g + (i & 3);
    put(out.W1[r * 72 + enc_feature(n)], sum.gw1[0][i]);
    put(out.W1[r * 72 + enc_feature(32 + n)], sum.gw1[1][i]);
    put(out.W2[hidden_unit(r & 15, r >> 4) * 32 + tile_unit(n)], sum.gw2[i]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    put(out.W1[((lane & 8 ? 16 : 0) + 4 * (lane >> 4) + r) * 72 + enc_feature(64 + (lane & 7))], sum.gw1e[r]);
    const float v = sum.gw3[r] + __shfl_xor(sum.gw3[r], 32);
    if (g == 0) put(out.W3[r * 32 + n], v);
  }
  const float gb2 = sum.gb[0] + __shfl_xor(sum.gb[0], 32), gb1 = sum.gb[1] + __shfl_xor(sum.gb[1], 32);
  if (g == 0) put(out.b1[n], gb1);
  else put(out.b2[hidden_unit(n & 15, n >> 4)], gb2);
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    float v = sum.gb3[o];
#pragma unroll
    for (int m = 16; m > 0; m >>= 1) v += __shfl_xor(v, m);
    if (n == o) put(out.b3[2 * g + o], v);
  }
}

}  // namespace mlpsp
