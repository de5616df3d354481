// Weight gradients of the per-primitive 72->32->32->4 MLP over blocks of 32 records of one primitive in f32, on the bf16
// matrix cores: every f32 operand is the exact sum of three bf16 numbers.
//
// Why.  v_mfma_f32_32x32x2_f32 does 32 multiply-adds per clock and SIMD and keeps the vector ALU from working meanwhile; the
// bf16 instruction does 512 beside it.  x = h + m + l with h = bf16(x), m = bf16(x - h), l = x - h - m is exact (three times
// eight significant bits, of numbers down to 2^-100; kVjp32Lift), and of the nine products of two such sums the six of weight 2^-16 and more are
// kept: what is dropped is below 2^-24 of the product, a rounding of the f32 product itself.  A sum over K = 16 terms then
// takes six instructions of 32 clocks instead of eight of 64, and rounds its accumulator six times instead of sixteen.
// Error of the gradients against float64 at the same f32 phases, 2-norm over 2-norm, and of a primitive's W1 gradient in the
// median and at the most, f32 chains of v_mfma_f32_32x32x2_f32 -> here:
//                           W1                 b1                 W2                 b2                 W3           a primitive's W1
//   647,988 steps   3.9e-7 -> 2.3e-7   2.8e-7 -> 1.5e-7   3.4e-7 -> 1.8e-7   3.7e-7 -> 1.1e-7   2.8e-7 -> 1.5e-7   3.7e-7 -> 2.8e-7, 2.4e-6 -> 1.3e-6
//    51,614 steps   1.9e-7 -> 1.0e-7   2.3e-7 -> 1.1e-7   2.1e-7 -> 0.9e-7   2.2e-7 -> 0.7e-7   1.7e-7 -> 1.0e-7   1.9e-7 -> 1.3e-7, 4.2e-7 -> 4.0e-7
//   3 x 4,096       6.2e-7 -> 4.7e-7   6.8e-7 -> 3.9e-7   7.4e-7 -> 4.8e-7   8.8e-7 -> 4.0e-7   9.3e-7 -> 3.7e-7
// The part of it along the gradient (a bias of all elements together) is at most 2e-7 of the norm, of either sign, also where
// all adjoints have one sign; of the f32 chains as much, for b3 9e-7.
// Time of the whole gradient call (200,000 primitives, 1200x680 / 20,000, 320x240): 7.42 -> 5.11 ms, 0.72 -> 0.49 ms.
//
// Bound by the latency of a block's chain -- products, the ~1,090 vector instructions beside them (a third of them sines and
// cosines, a sixth the splits), LDS --, two wavefronts to a SIMD: 256 registers with the weights in LDS.  (Sines and cosines by
// det_sincos: 1,250 instructions instead of 920 with a table without remainders, and 3 % of the time.)  A wavefront with its own
// weights in registers spills (6.7 ms, waiting for its spills behind the records requested ahead), alone on its SIMD it is no
// faster for 512 registers (7.0).  The two belong to different workgroups, one of which works while the other changes primitives
// (one workgroup of eight: 5.23 and 0.52 ms instead of 5.17 and 0.48).
//
// Per block (lane (n, g) = record n, half g of its inputs; D(a, b) has the rows of a in its registers):
//   d2        D(W3, d): record in the lane, unit 8 (i / 4) + 4 g + i % 4 in register i, in f32 products
//   d1        D(d2, W2^T): unit in the lane, records in the registers = the operand order of the W1 gradient
//   encoding  18 (sin, cos) pairs per lane, split, parked in LDS as [plane][record][column]
//   h1        D(W1, enc): record in the lane -- the operand order of layer 2
//   h2        D(h1, W2): unit in the lane, records in the registers, straight into the W3 gradient (4x4x1 f32 products)
//   gW2, gW1  contract over records.  What has its records in the lanes (d2, h1, the encoding) is written to LDS as it
//             lies and read with ds_read_b64_tr_b16, which hands a lane four records of one column
//   The last 8 of the 72 columns: a 16x16x32 product whose k-slots are (units 0..15, units 16..31) x records; its other
//   operand holds the 8 columns twice, for either half of the units, zero elsewhere.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_mlp_mfma32.hpp"
#include "mlpsp_vjp16.hpp"

namespace mlpsp {

typedef short i16x4v __attribute__((ext_vector_type(4)));
typedef float f32x2v __attribute__((ext_vector_type(2)));

// The lane's number, made anew where it is asked for: no register keeps it in between.
__device__ __forceinline__ int fresh_lane() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}
// Pairs of f32 as packed bf16: h + m + l = the pair.
struct Split2 {
  unsigned h, m, l;
};
// (1, 0) and (0, 1) negated, as operands of the two-term dot product that takes a rounded half off its original in one
// instruction.  Hidden from the compiler: as a packed inline constant -1 would stand in both halves.
struct SplitUnits {
  unsigned lo, hi;
  __device__ __forceinline__ SplitUnits() : lo(0x0000bf80u), hi(0xbf800000u) { asm("" : "+s"(lo), "+s"(hi)); }
};
__device__ __forceinline__ float minus_half(float a, unsigned pair, unsigned unit) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, unit), a, false);
}
__device__ __forceinline__ Split2 split2(float a, float b, const SplitUnits& u) {
  Split2 r;
  r.h = Ops<__bf16>::pack2(a, b);
  const float a1 = minus_half(a, r.h, u.lo), b1 = minus_half(b, r.h, u.hi);
  r.m = Ops<__bf16>::pack2(a1, b1);
  r.l = Ops<__bf16>::pack2(minus_half(a1, r.m, u.lo), minus_half(b1, r.m, u.hi));
  return r;
}

// The three planes of an operand of a 32-deep contraction.
struct Split8 {
  Pack8 p[3];
};
__device__ __forceinline__ Split8 split_tile(const vf32x16& v, const SplitUnits& u) {
  Split8 r;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const Split2 t = split2(v[8 * s + 2 * d], v[8 * s + 2 * d + 1], u);
      r.p[0].s[s][d] = t.h;
      r.p[1].s[s][d] = t.m;
      r.p[2].s[s][d] = t.l;
    }
  return r;
}
// The products of two split operands: `big` takes h h, `small` the five others.  Apart, because the matrix core cuts off what
// lies far below the largest of an instruction's addends: with the small products on top of the sum of the large ones the
// result is biased towards zero.
struct SplitAcc {
  vf32x16 big, small;
  __device__ __forceinline__ vf32x16 sum() const { return big + small; }
};
__device__ __forceinline__ void mfma_split(const u32x4& ha, const u32x4& ma, const u32x4& la, const u32x4& hb,
                                           const u32x4& mb, const u32x4& lb, SplitAcc& acc) {
  acc.small = Ops<__bf16>::mfma(la, hb, acc.small);
  acc.big = Ops<__bf16>::mfma(ha, hb, acc.big);
  acc.small = Ops<__bf16>::mfma(ha, lb, acc.small);
  acc.small = Ops<__bf16>::mfma(ma, mb, acc.small);
  acc.small = Ops<__bf16>::mfma(ma, hb, acc.small);
  acc.small = Ops<__bf16>::mfma(ha, mb, acc.small);
}
__device__ __forceinline__ void mma_split(const Split8& a, const Split8& b, SplitAcc& acc) {
#pragma unroll
  for (int s = 0; s < 2; ++s) mfma_split(a.p[0].s[s], a.p[1].s[s], a.p[2].s[s], b.p[0].s[s], b.p[1].s[s], b.p[2].s[s], acc);
}
// ... onto one accumulator that is large against any one product: nothing of it can be cut off by the product beside it (the
// bias that is left is measured above)
__device__ __forceinline__ vf32x16 mfma_split_onto(const u32x4& ha, const u32x4& ma, const u32x4& la, const u32x4& hb,
                                                   const u32x4& mb, const u32x4& lb, vf32x16 acc) {
  acc = Ops<__bf16>::mfma(la, hb, acc);
  acc = Ops<__bf16>::mfma(ha, lb, acc);
  acc = Ops<__bf16>::mfma(ma, mb, acc);
  acc = Ops<__bf16>::mfma(ma, hb, acc);
  acc = Ops<__bf16>::mfma(ha, mb, acc);
  return Ops<__bf16>::mfma(ha, hb, acc);
}

// A workgroup of four wavefronts, two workgroups to a CU: 22 KB of operands and 2.5 KB of turns that its wavefronts read, 14 KB of each one's own.
constexpr int kVjp32Waves = 4;
// The third part of a number below 2^-100 is lost.  The adjoints, which scale with the loss, are multiplied by this first and
// their sums divided by it, which changes no bit of a number in range: with adjoints of 2^-120 (2^-112) the W1 gradient was off
// by 4e-3 (1.5e-5) of its norm, with f32 products by 4e-7 (3e-8).  Weights and encodings below 2^-100 stay as they are.
constexpr float kVjp32Lift = 0x1p32f;
constexpr int kCircleEntries = 320;       // of vjp32_sincos' table
union Vjp32Wave {
  struct {
    // Columns of the encoding: pair t of group g (sin, cos) is word 16 g + t of a record's 32 for t < 16, and word
    // 2 g + (t - 16) of its tail; enc_place says where in the record's row.
    __attribute__((aligned(16))) unsigned enc[3][32][32];
    __attribute__((aligned(16))) unsigned enc_tail[3][32][4];
    __attribute__((aligned(16))) uint32_t mask1[32];
  };
  // (in the encoding's first half of plane 0, which is not written yet or, of the records 16 on, read again)
  __attribute__((aligned(16))) unsigned tile[32][16];   // one plane: word 8 g + d of a record (tile_place) = registers 2 d, 2 d + 1 of group g
  __attribute__((aligned(16))) float d3[32][4];         // [record][output]
  __attribute__((aligned(16))) float sums[kGradFloats]; // in the end
  static constexpr int kRowBytes = 128, kPlaneBytes = 4096;
};
struct Vjp32Lds {
  u32x4 w1[3][4][64];            // W1[n][..]: slots 2 d, 2 d + 1 of K-step s = pair 4 s + d
  u32x4 w1_tail[2][64];          // pairs 16, 17 of two planes
  u32x2 w1_tail1[2][64];         // ... of one, against zeros for the other
  unsigned w2[3][32][16];        // W2[n][..]: 16 bytes 2 s + g (tile_place) = unit(8 s + j, g)
  __attribute__((aligned(16))) float w3[2][64];      // W3[2 j + g][n]: as it lies
  __attribute__((aligned(16))) float bias1[32], bias2[32];
  __attribute__((aligned(16))) unsigned zero[4];
  int beyond[kVjp32Waves];       // a wavefront's sums are not all finite
  f32x2v circle[kCircleEntries];
  Vjp32Wave wave[kVjp32Waves];
};
constexpr int kVjp32RestLds = 528;        // of the kernel's own: the primitives of a chunk's steps
static_assert(2 * (sizeof(Vjp32Lds) + kVjp32RestLds) <= 163840, "two workgroups per CU");
// W1 column of encoding column k = 2 w + (0 sin, 1 cos)
__device__ __forceinline__ int enc_feature(int k) {
  const int w = k >> 1, g = w < 32 ? w >> 4 : (w - 32) >> 1, t = w < 32 ? w & 15 : 16 + (w & 1);
  return (k & 1) * 36 + 18 * g + t;
}
// unit held in column c of `tile`
__device__ __forceinline__ int tile_unit(int c) { return 8 * ((c >> 2) & 3) + 4 * (c >> 4) + (c & 3); }

__device__ __forceinline__ u32x2 read_transposed(const void* p) {
  typedef __attribute__((address_space(3))) i16x4v LdsVec;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsVec*)p));
}
// Operand (column 16 (n / 16) + n % 16 of the lane, k-slots = records) of K-step s: `row0` = this lane's address for
// records 4 g .. 4 g + 3; `row` bytes per record.
__device__ __forceinline__ u32x4 read_records(const char* row0, int s, int row) {
  const u32x2 a = read_transposed(row0 + (16 * s) * row), b = read_transposed(row0 + (16 * s + 8) * row);
  return u32x4{a[0], a[1], b[0], b[1]};
}
// Where 16 bytes of a record lie in its row of `tile` (quarter q of 64 bytes) and of `enc` (half h of 32 bytes b), in words: a
// store of 16 bytes a lane and a transposed read then reach every bank equally often (13 and 2.2 clocks; in order a store to
// `tile` takes 32).  The same for records eight apart, whose reads differ by a constant.
__device__ __forceinline__ int tile_place(int q, int record) { return 4 * (q ^ ((record >> 1) & 3)); }
__device__ __forceinline__ int enc_place(int b, int h, int record) {
  return 8 * (b ^ ((record & 2) | ((record >> 2) & 1))) + 4 * (h ^ (record & 1));
}
// This lane's address of transposed reads: record 4 g + (lane / 4) % 4, columns 16 (n / 16) + 4 (lane % 4) on
__device__ __forceinline__ const char* tile_reads(const unsigned (*tile)[16], int n, int g) {
  const int rec = 4 * g + ((n >> 2) & 3);
  return reinterpret_cast<const char*>(&tile[rec][tile_place(2 * (n >> 4) + ((n >> 1) & 1), rec) + 2 * (n & 1)]);
}
// ... columns 32 c further on
__device__ __forceinline__ const char* enc_reads(const unsigned (*enc)[32], int c, int n, int g) {
  const int rec = 4 * g + ((n >> 2) & 3);
  return reinterpret_cast<const char*>(&enc[rec][enc_place((n >> 4) + 2 * c, (n >> 1) & 1, rec) + 2 * (n & 1)]);
}

// Four floats that need not be aligned to more than one.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef const __attribute__((address_space(1))) f32x4u* Float4Address;
// (An address of unknown origin: out of a tensor that nothing is written to, the load would be put off until its value is used.)
__device__ __forceinline__ f32x4 load4_here(const float* p) {
  uintptr_t at = reinterpret_cast<uintptr_t>(p);
  asm volatile("" : "+v"(at));
  return f32x4(*(Float4Address)at);
}
__device__ __forceinline__ float load_here(const float* p) {
  uintptr_t at = reinterpret_cast<uintptr_t>(p);
  asm volatile("" : "+v"(at));
  return *(const __attribute__((address_space(1))) float*)at;
}
// What a lane loads of a primitive's weights, asked for while the sums of the primitive before are put away, as is where its
// steps lie (a chain of six look-ups from one primitive to the next otherwise; kernel at 80,000 steps 675 -> 651 us, at 650,000
// 5.54 -> 5.49 ms, the 16-bit one 1.53 -> 1.52): the workgroup's four wavefronts share them out, each with the same four loads (no branch: where paths meet, loads are waited for).  Of W1,
// lane (n, g): pairs 4 wave .. 4 wave + 3; then wavefronts 0 and 1 rows of W2, 2 the pairs 16 and 17 (as elements 2 and 3: the
// four behind them may lie outside the tensor), 3 W3, b1 and b2 as they lie.
struct Vjp32Request {
  f32x4 sines, cosines, a, b;
};
__device__ __forceinline__ Vjp32Request vjp32_request(const float* __restrict__ W1, const float* __restrict__ b1,
                                                      const float* __restrict__ W2, const float* __restrict__ b2,
                                                      const float* __restrict__ W3, size_t p, int wave, int lane) {
  asm volatile("" : "+v"(lane));         // (as in vjp32_block)
  const int n = lane & 31, g = lane >> 5;
  const float* row1 = W1 + p * 2304 + n * 72 + 18 * g;
  const float* tail = lane < 32 ? W3 + p * 128 + 4 * lane : lane < 40 ? b1 + p * 32 + 4 * (lane - 32) : b2 + p * 32 + 4 * (min(lane, 47) - 40);
  const float* a = wave < 2 ? W2 + p * 1024 + n * 32 + 16 * wave + 4 * g : wave == 2 ? row1 + 14 : tail;
  const float* b = wave < 2 ? a + 8 : wave == 2 ? a + 36 : a;
  return Vjp32Request{load4_here(row1 + 4 * wave), load4_here(row1 + 36 + 4 * wave), load4_here(a), load4_here(b)};
}
// The primitive's weights into LDS, by the whole workgroup.
__device__ __forceinline__ void vjp32_load(const Vjp32Request& r, int wave, int lane, Vjp32Lds& s, const SplitUnits& u) {
  asm volatile("" : "+v"(lane));         // (as in vjp32_block)
  const int n = lane & 31, g = lane >> 5;
  u32x4 v[3];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const Split2 x = split2(r.sines[d], r.cosines[d], u);
    v[0][d] = x.h;
    v[1][d] = x.m;
    v[2][d] = x.l;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) s.w1[k][wave][lane] = v[k];
  if (wave < 2) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const f32x4& from = d < 2 ? r.a : r.b;
      const Split2 x = split2(from[2 * (d & 1)], from[2 * (d & 1) + 1], u);
      v[0][d] = x.h;
      v[1][d] = x.m;
      v[2][d] = x.l;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<u32x4*>(&s.w2[k][n][tile_place(2 * wave + g, n)]) = v[k];
  } else if (wave == 2) {
    const Split2 x = split2(r.a[2], r.b[2], u), y = split2(r.a[3], r.b[3], u);
    s.w1_tail1[0][lane] = u32x2{x.h, y.h};               // h h: against (h, m)
    s.w1_tail1[1][lane] = u32x2{x.l, y.l};               // l h: against (h, m)
    s.w1_tail[0][lane] = u32x4{x.m, y.m, x.h, y.h};      // m m, h l: against (m, l)
    s.w1_tail[1][lane] = u32x4{x.h, y.h, x.m, y.m};      // h m, m h: against (m, h)
  } else if (lane < 48) {
    reinterpret_cast<f32x4*>(lane < 32 ? &s.w3[0][0] : lane < 40 ? s.bias1 - 32 * 4 : s.bias2 - 40 * 4)[lane] = r.a;
  }
}
struct Vjp32Sums {
  vf32x16 gw1[2], gw2;
  f32x4 gw1e, gw3, gb2;
  float gb1, gb3[4];
  __device__ __forceinline__ void clear() {
    gw1[0] = gw1[1] = gw2 = splat16(0.f);
    gw1e = gw3 = gb2 = f32x4{0.f, 0.f, 0.f, 0.f};
    gb1 = gb3[0] = gb3[1] = gb3[2] = gb3[3] = 0.f;
  }
};

// The six (sin, cos) pairs of one input component, from the sine and cosine of the nearest of 256 turns k 2 pi / 256 and a
// rotation by the rest, |r| <= pi / 256: sin r = r - r^3 / 6 and cos r - 1 = -r^2 / 2 to 2e-12 and 1e-9.  The table holds the
// sine of 320 turns -- a cosine is the sine of the turn 64 further on -- as its f32 value and what that leaves over, which is
// added to the rotation's terms before the value itself: what a pair is off by is the rounding of that last sum.  Against
// float64 over phases up to 30: 1.5e-8 rms, 3.2e-8 at the most; det_sincos 2.1e-8 and 9.2e-8; a table without remainders
// 2.5e-8 and 8.9e-8.  20 instructions a pair and one LDS read of two entries, det_sincos 27.
//
// The phase is the forward's, (x freq) att with both roundings: with the factors multiplied first, the sine of a phase of 100
// is that of another number by 1e-5, and the gradient is off by 2.6e-6 of its norm.  Out of range (|phase| > 65536: a pair of
// NaN, as in det_sincos) without a comparison: the phase times the largest float / 65536 is infinite exactly there, and zero
// times that is added to the rest.
struct PhaseFactors {
  float freq[6], att[6];
};
struct CircleTable {
  float at[kCircleEntries][2];
  constexpr CircleTable() : at{} {
    for (int k = 0; k < kCircleEntries; ++k) {
      const double x = (k < 128 ? k : k - 256) * (6.283185307179586476925 / 256.0);
      double sine = 0.0, term = x;                       // x^i / i!
      for (int i = 1; i < 40; i += 2) {
        sine += i & 2 ? -term : term;
        term *= x * x / ((i + 1) * (i + 2));
      }
      at[k][0] = (float)sine;
      at[k][1] = (float)(sine - (double)at[k][0]);
    }
  }
};
static __device__ const CircleTable kCircle = CircleTable();
__device__ __forceinline__ void vjp32_sincos(const f32x2v* circle, float x, const PhaseFactors& k, float s_out[6], float c_out[6]) {
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const float phase = (x * k.freq[f]) * k.att[f];
    const float shifted = fmaf(phase, 40.7436654f, 12582912.0f);         // the nearest turn, in the low bits
    const float kf = shifted - 12582912.0f;
    float r = fmaf(kf, -0.0245436933f, phase);
    r = fmaf(kf, 6.82990470e-10f, r);
    r = fmaf(phase * 0x1.fffffep111f, 0.f, r);
    const f32x2v* const at = reinterpret_cast<const f32x2v*>(reinterpret_cast<const char*>(circle) + ((float_to_bits(shifted) << 3) & 0x7f8u));
    const f32x2v sv = at[0], cv = at[64];
    const float z = r * r, less = -0.5f * z, sine = fmaf(r * z, -0.166666667f, r);
    s_out[f] = sv[0] + fmaf(cv[0], sine, fmaf(sv[0], less, sv[1]));
    c_out[f] = cv[0] + fmaf(-sv[0], sine, fmaf(cv[0], less, cv[1]));
  }
}
// v where bit `bit` of word is set, else +0
__device__ __forceinline__ float where_bit(float v, uint32_t word, int bit) {
  return __uint_as_float(__float_as_uint(v) & (uint32_t)__builtin_amdgcn_sbfe((int)word, bit, 1));
}
// A tile whose lanes are records, transposed through LDS a plane at a time (a wavefront's LDS operations complete in order).
__device__ __forceinline__ Split8 transpose_tile(const Split8& v, Vjp32Wave& s, int n, int g) {
  asm volatile("" : "+v"(n));            // (or the addresses are kept from one transposition to the next, and registers spill)
  unsigned* const to = &s.tile[n][tile_place(2 * g, n)];
  unsigned* const to1 = &s.tile[n][tile_place(2 * g + 1, n)];
  const char* const from = tile_reads(s.tile, n, g);
  Split8 r;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    *reinterpret_cast<u32x4*>(to) = v.p[p].s[0];
    *reinterpret_cast<u32x4*>(to1) = v.p[p].s[1];
#pragma unroll
    for (int k = 0; k < 2; ++k) r.p[p].s[k] = read_records(from, k, 64);
  }
  return r;
}
// The operands of layer 2, W2[n][unit(8 s + j, g)] and, transposed, W2[unit(8 s + j, g)][n]
__device__ __forceinline__ Split8 read_w2(const Vjp32Lds& w, int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5;
  Split8 r;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const unsigned* const from = &w.w2[0][n][tile_place(2 * k + g, n)];
#pragma unroll
    for (int p = 0; p < 3; ++p) r.p[p].s[k] = *reinterpret_cast<const u32x4*>(from + 512 * p);
  }
  return r;
}
__device__ __forceinline__ Split8 read_w2_transposed(const Vjp32Lds& w, int lane) {
  asm volatile("" : "+v"(lane));
  const int n = lane & 31, g = lane >> 5, row = 4 * g + ((n >> 2) & 3);
  const char* const from = reinterpret_cast<const char*>(&w.w2[0][row][tile_place(2 * (n >> 4) + (n & 1), row) + (n & 2)]);
  Split8 r;
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int k = 0; k < 2; ++k) r.p[p].s[k] = read_records(from + 2048 * p, k, 64);
  return r;
}
struct SplitOperand {
  u32x4 p[3];
};
__device__ __forceinline__ SplitOperand read_step(const u32x4 (*b)[4][64], int k, int lane) {
  return SplitOperand{{b[0][k][lane], b[1][k][lane], b[2][k][lane]}};
}
__device__ __forceinline__ void mfma_split(const SplitOperand& a, const SplitOperand& b, SplitAcc& acc) {
  mfma_split(a.p[0], a.p[1], a.p[2], b.p[0], b.p[1], b.p[2], acc);
}
// Six pairs of the encoding as operands: e.p[..][t % 4] of K-step t / 4; a finished K-step goes to LDS and to `done`.
template <int C, typename Done>
__device__ __forceinline__ void vjp32_encode(const f32x2v* circle, float x, const PhaseFactors& factors, Vjp32Wave& s, int n, int g, const SplitUnits& u,
                                             SplitOperand& e, Done&& done) {
  float sn[6], cs[6];
  vjp32_sincos(circle, x, factors, sn, cs);
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const int t = 6 * C + f;
    const Split2 v = split2(sn[f], cs[f], u);
    e.p[0][t & 3] = v.h;
    e.p[1][t & 3] = v.m;
    e.p[2][t & 3] = v.l;
    if ((t & 3) == 3) {
      const int k = t >> 2;
      unsigned* const to = &s.enc[0][n][enc_place(2 * g + (k >> 1), k & 1, n)];
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x4*>(to + 1024 * p) = e.p[p];
      done(k, e);
    }
  }
}

// One block of 32 records.  Lane (n, g): record n, x = its three inputs of group g.  The parts stay one behind the other
// (sched_barrier): mixed by the compiler they need more registers than there are.  (Matrix and vector instructions of a part
// alternated by hand: no faster; the other wavefront of the SIMD fills the gaps.)
__device__ __forceinline__ void vjp32_block(const Vjp32Lds& w, Vjp32Sums& sum, Vjp32Wave& s, const float x[3], float4 adjoint,
                                            uint32_t mask1, uint32_t mask2, const PhaseFactors& factors, float scale,
                                            int lane, const SplitUnits& u) {
  asm volatile("" : "+v"(lane));         // (or the addresses are formed ahead of the loop over the blocks, one by one)
  const int n = lane & 31, g = lane >> 5;
  const float inf = relu_limit();
  const float d[4] = {adjoint.x * scale, adjoint.y * scale, adjoint.z * scale, adjoint.w * scale};
  if (g == 0) {
    s.mask1[n] = mask1;
#pragma unroll
    for (int o = 0; o < 4; ++o) sum.gb3[o] += d[o];
  }
  // ---- adjoints of layer 2: record in the lane.  (Four terms: two f32 products.  Their eight split products in two bf16
  // instructions are biased, see SplitAcc.)
  Split8 d2;
  {
    vf32x16 t = __builtin_amdgcn_mfma_f32_32x32x2f32(w.w3[0][lane], g ? d[1] : d[0], splat16(0.f), 0, 0, 0);
    t = __builtin_amdgcn_mfma_f32_32x32x2f32(w.w3[1][lane], g ? d[3] : d[2], t, 0, 0, 0);
    const uint32_t mine = mask2 >> (4 * g);
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i] = where_bit(t[i], mine, 8 * (i >> 2) + (i & 3));
    d2 = split_tile(t, u);
  }
  const Split8 d2t = transpose_tile(d2, s, n, g);
  __builtin_amdgcn_sched_barrier(0);
  // ---- adjoints of layer 1: unit in the lane; encoding and layer 1: record in the lane
  SplitAcc t1;
  t1.big = t1.small = splat16(0.f);
  SplitOperand e, e0, e1, e2, e3;
  mma_split(d2, read_w2_transposed(w, lane), t1);
  vjp32_encode<0>(w.circle, x[0], factors, s, n, g, u, e, [&](int, const SplitOperand& v) { e0 = v; });
  __builtin_amdgcn_sched_barrier(0);
  vf32x16 tsum = t1.sum();
  SplitAcc a1;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(&w.bias1[8 * q + 4 * g]);
#pragma unroll
    for (int k = 0; k < 4; ++k) a1.big[4 * q + k] = v[k];
  }
  a1.small = splat16(0.f);
  mfma_split(read_step(w.w1, 0, lane), e0, a1);
  vjp32_encode<1>(w.circle, x[1], factors, s, n, g, u, e, [&](int k, const SplitOperand& v) { (k == 1 ? e1 : e2) = v; });
  __builtin_amdgcn_sched_barrier(0);
  mfma_split(read_step(w.w1, 1, lane), e1, a1);
  mfma_split(read_step(w.w1, 2, lane), e2, a1);
  vjp32_encode<2>(w.circle, x[2], factors, s, n, g, u, e, [&](int, const SplitOperand& v) { e3 = v; });
#pragma unroll
  for (int p = 0; p < 3; ++p) *reinterpret_cast<u32x2*>(&s.enc_tail[p][n][2 * g]) = u32x2{e.p[p][0], e.p[p][1]};
  __builtin_amdgcn_sched_barrier(0);
  // ---- adjoints of layer 1 masked, beside the end of layer 1
  Split8 d1;
  mfma_split(read_step(w.w1, 3, lane), e3, a1);
  {
    const u32x4 hm = {e.p[0][0], e.p[0][1], e.p[1][0], e.p[1][1]};
    const u32x2 wh = w.w1_tail1[0][lane], wl = w.w1_tail1[1][lane];
    a1.big = Ops<__bf16>::mfma(u32x4{wh[0], wh[1], 0u, 0u}, hm, a1.big);
    a1.small = Ops<__bf16>::mfma(u32x4{wl[0], wl[1], 0u, 0u}, hm, a1.small);
    a1.small = Ops<__bf16>::mfma(w.w1_tail[0][lane], u32x4{e.p[1][0], e.p[1][1], e.p[2][0], e.p[2][1]}, a1.small);
    a1.small = Ops<__bf16>::mfma(w.w1_tail[1][lane], u32x4{e.p[1][0], e.p[1][1], e.p[0][0], e.p[0][1]}, a1.small);
  }
  {
    vf32x16 v = tsum;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int4 m = *reinterpret_cast<const int4*>(&s.mask1[8 * q + 4 * g]);
      v[4 * q] = where_bit(v[4 * q], (uint32_t)m.x, n);
      v[4 * q + 1] = where_bit(v[4 * q + 1], (uint32_t)m.y, n);
      v[4 * q + 2] = where_bit(v[4 * q + 2], (uint32_t)m.z, n);
      v[4 * q + 3] = where_bit(v[4 * q + 3], (uint32_t)m.w, n);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sum.gb1 += v[i];
    d1 = split_tile(v, u);
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- layer 1 rectified, beside the first half of the W1 gradient.  This lane's addresses of transposed reads: record
  // rec = 4 g + (lane / 4) % 4 (and 8 on), columns 32 c + 16 (n / 16) + 4 (lane % 4) on
  const int rec = 4 * g + ((n >> 2) & 3);
  // of the last columns: units 0..15 (n < 16) take them in the low half of the columns, units 16..31 in the high half
  const bool last = ((n >> 1) & 1) == (n >> 4);
  const char* const last0 = last ? reinterpret_cast<const char*>(&s.enc_tail[0][rec][2 * (n & 1)]) : reinterpret_cast<const char*>(w.zero);
  const int last_row = last ? 16 : 0, last_plane = last ? 32 * 16 : 0;
  const auto gradient1 = [&](int k) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const char* const at = enc_reads(s.enc[0], c, n, g);
      u32x4 b[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) b[p] = read_records(at + p * Vjp32Wave::kPlaneBytes, k, Vjp32Wave::kRowBytes);
      sum.gw1[c] = mfma_split_onto(d1.p[0].s[k], d1.p[1].s[k], d1.p[2].s[k], b[0], b[1], b[2], sum.gw1[c]);
    }
    bf16x8 b[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) b[p] = __builtin_bit_cast(bf16x8, read_records(last0 + p * last_plane, k, last_row));
    const auto product = [&](int i, int j) {
      sum.gw1e = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, d1.p[i].s[k]), b[j], sum.gw1e, 0, 0, 0);
    };
    product(2, 0);
    product(0, 2);
    product(1, 1);
    product(1, 0);
    product(0, 1);
    product(0, 0);
  };
  Split8 h1;
  gradient1(0);
  {
    vf32x16 v = a1.sum();
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = relu_f32(v[i], inf);
    h1 = split_tile(v, u);
  }
  __builtin_amdgcn_sched_barrier(0);
  const Split8 h1t = transpose_tile(h1, s, n, g);
  if (g == 0) *reinterpret_cast<f32x4*>(s.d3[n]) = f32x4{d[0], d[1], d[2], d[3]};
  const float bias2 = w.bias2[n];
  gradient1(1);
  __builtin_amdgcn_sched_barrier(0);
  // ---- layer 2: unit in the lane; the W2 gradient
  SplitAcc o2;
  o2.big = splat16(bias2);
  o2.small = splat16(0.f);
  mma_split(h1, read_w2(w, lane), o2);
  const u32x2 ones = {Ops<__bf16>::kOneWord, Ops<__bf16>::kOneWord};
#pragma unroll
  for (int k = 0; k < 2; ++k) {
#pragma unroll
    for (int p = 2; p >= 0; --p) {
      const u32x4 v = d2t.p[p].s[k];
      sum.gb2 = Ops<__bf16>::mfma4(ones, u32x2{v[0], v[1]}, sum.gb2);
      sum.gb2 = Ops<__bf16>::mfma4(ones, u32x2{v[2], v[3]}, sum.gb2);
    }
    sum.gw2 = mfma_split_onto(d2t.p[0].s[k], d2t.p[1].s[k], d2t.p[2].s[k], h1t.p[0].s[k], h1t.p[1].s[k], h1t.p[2].s[k], sum.gw2);
  }
  // ... straight into the W3 gradient, in four chains
  {
    const vf32x16 v = o2.sum();
    const float* d3 = &s.d3[4 * g][n & 3];
    f32x4 part[4] = {sum.gw3, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int i = 0; i < 16; ++i)
      part[i & 3] = __builtin_amdgcn_mfma_f32_4x4x1f32(d3[4 * (8 * (i >> 2) + (i & 3))], relu_f32(v[i], inf), part[i & 3], 0, 0, 0);
    sum.gw3 = (part[0] + part[1]) + (part[2] + part[3]);
  }
}

// A wavefront's sums to `row` in LDS, in the order of a packed row of gradients.
__device__ __forceinline__ void vjp32_park(const Vjp32Sums& sum, float* row, int lane) {
  asm volatile("" : "+v"(lane));         // (as in vjp32_block)
  const int n = lane & 31, g = lane >> 5;
  const GradRows out = packed_grad_rows(row);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 8 * (i >> 2) + 4 * g + (i & 3);
    out.W1[r * 72 + enc_feature(n)] = sum.gw1[0][i];
    out.W1[r * 72 + enc_feature(32 + n)] = sum.gw1[1][i];
    out.W2[tile_unit(r) * 32 + tile_unit(n)] = sum.gw2[i];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    out.W1[((lane & 8 ? 16 : 0) + 4 * (lane >> 4) + r) * 72 + enc_feature(64 + (lane & 7))] = sum.gw1e[r];
    const float v = sum.gw3[r] + __shfl_xor(sum.gw3[r], 32);
    if (g == 0) out.W3[r * 32 + n] = v;
  }
  const float gb1 = sum.gb1 + __shfl_xor(sum.gb1, 32), gb2 = sum.gb2[0] + __shfl_xor(sum.gb2[0], 32);
  if (g == 0) out.b1[n] = gb1;
  else out.b2[tile_unit(n)] = gb2;
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    float v = sum.gb3[o];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    if (lane == o) out.b3[o] = v;
  }
}
// The sums in `rows` rows of LDS, `stride` floats apart, added up by the workgroup and stored; returns whether a value was not
// finite.
__device__ __forceinline__ bool store_row_sums(const float* first, int stride, int rows, const GradRows& out, float inv, int t,
                                               int threads) {
  asm volatile("" : "+v"(t));
  bool bad = false;
  for (int k = t; k < kGradFloats / 4; k += threads) {
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < rows; ++w) v += *reinterpret_cast<const f32x4*>(first + w * stride + 4 * k);
    v *= inv;
#pragma unroll
    for (int q = 0; q < 4; ++q) bad |= !(__builtin_fabsf(v[q]) <= 3.4028235e38f);
    // float4 ranges of the parts: [0,576) W1, [576,584) b1, [584,840) W2, [840,848) b2, [848,880) W3, 880 b3
    f32x4* to;
    if (k < 576) to = reinterpret_cast<f32x4*>(out.W1) + k;
    else if (k < 584) to = reinterpret_cast<f32x4*>(out.b1) + (k - 576);
    else if (k < 840) to = reinterpret_cast<f32x4*>(out.W2) + (k - 584);
    else if (k < 848) to = reinterpret_cast<f32x4*>(out.b2) + (k - 840);
    else if (k < 880) to = reinterpret_cast<f32x4*>(out.W3) + (k - 848);
    else to = reinterpret_cast<f32x4*>(out.b3);
    *to = v;
  }
  return bad;
}

}  // namespace mlpsp
