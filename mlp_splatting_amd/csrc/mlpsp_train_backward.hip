// libmlpsp_hip: backward pass over the training steps of a frame (mlpsp_train.hpp): reverse compositing, then geometry
// and MLP weight gradients per primitive.  Counterpart of the reference's reverse walk (primitive_records.cuh:3-46) and
// grouped gradient kernels (scannet/primitive_gemm.py:101-183) in one pipeline whose unit is a step, not a record.
//
// The steps are sorted by primitive (S = 0.65 M at the 200,000-primitive 1200x680 frame) and cut into chunks of equal
// length.  A workgroup walks one chunk; where the primitive changes it writes its sums: straight to the gradients if the
// primitive's steps all lie in the chunk, else to the chunk's tail row (the primitive goes on in the next chunk) or head row
// (it ended here).  One more launch adds the rows of the primitives that span chunks; the zeros of those without a step are
// written by the weight gradient kernels too, or by a launch of their own where these have few wavefronts (kZeroShare32).  No
// atomics, a fixed order of every sum.
//
// Measured at 200,000 primitives, 1200x680, f32, against the record pipeline (ms): reverse 0.47 (1.8), sort and grouping
// 0.11 (sort 1.7, gathers 2.85), geometry 0.16 (1.3), weight gradients with the zeros beside them 5.1 (12.8 and 0.8), joining rows 0.04.
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mlp_mfma32.hpp"
#include "mlpsp_train.hpp"
#include "mlpsp_vjp16.hpp"
#include "mlpsp_vjp16_steps.hpp"
#include "mlpsp_vjp32.hpp"

namespace mlpsp {

// ---------------------------------------------------------------------------------------------
// reverse compositing: one wavefront per tile, its steps last to first; per step and lane d4 = the adjoints of the four
// pre-activation outputs and the falloff adjoint dL/d(decay) decay (the expressions of records_reverse_kernel).  Bound by
// memory: 2 KB read and 1.25 KB written per step, both contiguous, where there are many tiles (200,000 primitives, 1200x680:
// 0.50 ms, 4.4 TB/s); where there are few, by the time a step's planes take to arrive, so four steps are asked for ahead, without
// a wait for the chunk table between them (1,200 tiles: 88 us with one, 55).
// ---------------------------------------------------------------------------------------------
constexpr int kReverseAhead = 4;
__global__ __launch_bounds__(64) void train_reverse_kernel(
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ tile_base, const int32_t* __restrict__ chunk_table,
    const unsigned char* __restrict__ records, const float* __restrict__ grgb, const float* __restrict__ gt, int W, int H,
    int ntx, int nty, float4* __restrict__ d4, float* __restrict__ falloff) {
  const int tile = superblock_tile(blockIdx.x, ntx, nty);
  if (tile < 0) return;
  const int l = threadIdx.x;
  const int base = tile_base[tile], count = tile_base[tile + 1] - base;
  if (count == 0) return;
  const int x = (tile % ntx) * 8 + (l & 7), y = (tile / ntx) * 8 + (l >> 3);
  const bool valid = (x < W) && (y < H);
  const int pix = valid ? (y * W + x) : 0;
  const Float3 g = valid ? load3(grgb, pix) : Float3{0.f, 0.f, 0.f};
  float next = valid ? gt[pix] : 0.f;
  // The tile's entries of the chunk table, 64 at a time, an entry in each lane; the planes of the next kReverseAhead steps.
  const int table = step_table(offsets[tile], tile), last = (count - 1) >> StepGroups::kLog2;
  int window = -1, chunks = 0;
  const auto request = [&](int m, float4& a, float4& b) {
    const int c = m >> StepGroups::kLog2;
    if ((c & ~63) != window) {
      window = c & ~63;
      chunks = chunk_table[table + min(window + l, last)];
      asm volatile("" : "+v"(chunks));           // (waited for here, not in every turn)
    }
    const int slot = __builtin_amdgcn_readlane(chunks, c & 63) * kStepChunk + (m & (kStepChunk - 1));
    const float4* src = reinterpret_cast<const float4*>(records + (size_t)slot * kStepBytes) + l;
    a = src[0];
    b = src[64];
  };
  float4 a[kReverseAhead], b[kReverseAhead];
#pragma unroll
  for (int k = 0; k < kReverseAhead; ++k) request(max(count - 1 - k, 0), a[k], b[k]);
  for (int first = count - 1; first >= 0; first -= kReverseAhead) {
#pragma unroll
    for (int k = 0; k < kReverseAhead; ++k) {
      const int m = first - k;                   // (below zero at the end: the first step again, nothing stored)
      const float R = a[k].x, G = a[k].y, B = a[k].z, sigma_raw = a[k].w, trans = b[k].x, alpha = b[k].y, decay = b[k].z;
      // A lane that the primitive missed holds zeros (a hit's transmittance is at least the floor), and its adjoint may be
      // anything -- the derivative of a root at a black pixel is infinite --: zeros come of it, not 0 inf.
      const bool hit = trans != 0.f;
      const float dotg = (g.x * R + g.y * G) + g.z * B;
      const float grad_alpha = trans * (dotg - next);
      next = hit ? next * (1.f - alpha) + dotg * alpha : next;
      const float grad_sigma = grad_alpha * det_exp(-sigma_raw * decay);
      const float grad_decay = grad_sigma * sigma_raw;
      float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
      if (hit) {
        d.x = g.x * (trans * alpha) * R * (1.f - R);
        d.y = g.y * (trans * alpha) * G * (1.f - G);
        d.z = g.z * (trans * alpha) * B * (1.f - B);
        d.w = grad_sigma * decay * sigmoid(b[k].w);
      }
      float f = hit ? grad_decay * decay : 0.f;
      asm volatile("" : "+v"(d.x), "+v"(d.y), "+v"(d.z), "+v"(d.w), "+v"(f), "+v"(next));   // (done with the planes' registers)
      request(max(m - kReverseAhead, 0), a[k], b[k]);
      if (m >= 0) {
        const size_t at = (size_t)(base + m) * 64 + l;
        d4[at] = d;
        falloff[at] = f;
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// steps sorted by primitive: a stable radix sort of the S primitive numbers in tile order, in digits of equal width (two of
// nine bits at 200,000 primitives).  A wavefront takes an eighth of its block's steps in rounds of 64, whose equal digits are
// found with a ballot per bit.  Eight launches, 110 us at 650,000 steps (the two sums over blocks x digits, one workgroup
// each, 18 of them, the two scatters 58); the library's sort took 22 launches and 200 us with the gather behind it.
// ---------------------------------------------------------------------------------------------
constexpr int kSortBlock = 512, kSortBits = 10;
// Steps of a block: 8,192, a quarter of that where this would leave a chip of 256 CUs fewer than 32 blocks (16 rounds one
// after the other took 33 us at 80,000 steps); the sums over blocks x digits grow with the blocks.
inline int sort_keys(int64_t S) { return S >= 32 * 8192 ? 8192 : 2048; }

// keys and particulars of the steps in tile order
__global__ __launch_bounds__(256) void step_list_kernel(const int32_t* __restrict__ offsets, const int32_t* __restrict__ tile_base,
                                                        const int32_t* __restrict__ chunk_table, const int32_t* __restrict__ ids,
                                                        int T, int W, int ntx, int32_t* __restrict__ keys, int4* __restrict__ info) {
  const int tile = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if (tile >= T) return;
  const int base = tile_base[tile], count = tile_base[tile + 1] - base, table = step_table(offsets[tile], tile);
  const int pixel = (tile / ntx) * 8 * W + (tile % ntx) * 8;
  for (int m = lane; m < count; m += 64) {
    const int slot = step_slot(chunk_table, table, m);
    keys[base + m] = ids[slot];
    info[base + m] = make_int4(slot, base + m, tile, pixel);
  }
}

__global__ __launch_bounds__(kSortBlock) void step_hist_kernel(const int32_t* __restrict__ keys, int S, int share, int shift,
                                                               int bits, int blocks, int32_t* __restrict__ hist) {
  __shared__ int s_count[1 << kSortBits];
  const int R = 1 << bits;
  for (int d = threadIdx.x; d < R; d += kSortBlock) s_count[d] = 0;
  __syncthreads();
  const int end = min(S, (int)(blockIdx.x + 1) * share);
  for (int i = (int)blockIdx.x * share + threadIdx.x; i < end; i += kSortBlock)
    atomicAdd(&s_count[(keys[i] >> shift) & (R - 1)], 1);
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kSortBlock) hist[d * blocks + blockIdx.x] = s_count[d];
}

// exclusive sums of n counts, in place; one workgroup, kSumRounds of 4,096 counts behind one barrier.  Us a launch (traced,
// 200,000 primitives), a round at a time, its loads and two barriers one after the other / 6 / 10 / 16 rounds:
//     steps    1,600   80,000  250,000  650,000  750,000  1,000,000  1,300,000  2,000,000
//     one        2.1     12.9     37.4     24.3     28.2       36.6       47.2       70.3
//     6          2.7      4.7     12.6      8.3      9.4       12.4       15.5       23.2
//     10         3.2      4.9     12.5      8.3     10.5       12.4       15.0       23.7
//     16         3.9      5.6     11.9      8.2      9.4       11.8       15.9       21.4
constexpr int kSumRounds = 6;
__global__ __launch_bounds__(1024) void step_sums_kernel(int32_t* __restrict__ v, int n) {
  __shared__ int s_wave[2][kSumRounds * 16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int carry = 0;
  for (int base = 0, turn = 0; base < n; base += kSumRounds * 4096, turn ^= 1) {
    int4 x[kSumRounds];
#pragma unroll
    for (int u = 0; u < kSumRounds; ++u) {
      const int i = base + 4096 * u + 4 * t;
      x[u] = i + 3 < n ? *reinterpret_cast<const int4*>(v + i)
                       : make_int4(i < n ? v[i] : 0, i + 1 < n ? v[i + 1] : 0, i + 2 < n ? v[i + 2] : 0, 0);
    }
    int incl[kSumRounds];
#pragma unroll
    for (int u = 0; u < kSumRounds; ++u) {
      if (base + 4096 * u >= n) break;
      incl[u] = (x[u].x + x[u].y) + (x[u].z + x[u].w);
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl[u], d);
        if (lane >= d) incl[u] += up;
      }
      if (lane == 63) s_wave[turn][16 * u + wave] = incl[u];
    }
    __syncthreads();                   // (the one barrier of a turn: the next writes the other half)
    // lane = wavefront of a round; all rounds' sums up to and with it
    int total = carry;
#pragma unroll
    for (int u = 0; u < kSumRounds; ++u) {
      if (base + 4096 * u >= n) break;
      int w = s_wave[turn][16 * u + (lane & 15)];
      const int own = w;
#pragma unroll
      for (int d = 1; d < 16; d <<= 1) {
        const int up = __shfl_up(w, d);
        if ((lane & 15) >= d) w += up;
      }
      const int i = base + 4096 * u + 4 * t;
      int run = total + __builtin_amdgcn_readlane(w - own, wave) + incl[u] - ((x[u].x + x[u].y) + (x[u].z + x[u].w));
      total += __builtin_amdgcn_readlane(w, 15);
      const int4 out = make_int4(run, run + x[u].x, run + x[u].x + x[u].y, run + x[u].x + x[u].y + x[u].z);
      if (i + 3 < n) {
        *reinterpret_cast<int4*>(v + i) = out;
      } else {
        if (i < n) v[i] = out.x;
        if (i + 1 < n) v[i + 1] = out.y;
        if (i + 2 < n) v[i + 2] = out.z;
      }
    }
    carry = total;
  }
}

// order: numbers of the keys (null: their places).  The last digit's pass writes the sorted primitives and particulars.
template <bool LAST>
__global__ __launch_bounds__(kSortBlock) void step_scatter_kernel(const int32_t* __restrict__ keys, const int32_t* __restrict__ order,
                                                                  int S, int share, int shift, int bits, int blocks,
                                                                  const int32_t* __restrict__ sums, const int4* __restrict__ info,
                                                                  int32_t* __restrict__ out_keys, int32_t* __restrict__ out_order,
                                                                  int4* __restrict__ out_step) {
  constexpr int kWaves = kSortBlock / 64;
  __shared__ int s_at[kWaves][1 << kSortBits];
  const int R = 1 << bits, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int d = threadIdx.x; d < R; d += kSortBlock) {
#pragma unroll
    for (int w = 0; w < kWaves; ++w) s_at[w][d] = 0;
  }
  __syncthreads();
  const int begin = (int)blockIdx.x * share + wave * (share / kWaves), end = min(S, begin + share / kWaves);
  for (int i = begin + lane; i < end; i += 64) atomicAdd(&s_at[wave][(keys[i] >> shift) & (R - 1)], 1);
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kSortBlock) {
    int run = sums[d * blocks + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const int c = s_at[w][d];
      s_at[w][d] = run;
      run += c;
    }
  }
  __syncthreads();
  for (int base = begin; base < end; base += 64) {
    const int i = base + lane;
    const bool valid = i < end;
    const int key = valid ? keys[i] : 0, digit = (key >> shift) & (R - 1);
    unsigned long long same = __ballot(valid);
    for (int b = 0; b < bits; ++b) {
      const bool set = (digit >> b) & 1;
      const unsigned long long m = __ballot(set);
      same &= set ? m : ~m;
    }
    if (!valid) continue;
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    const int at = s_at[wave][digit] + rank;
    if (rank == 0) s_at[wave][digit] = at + (int)__popcll(same);
    const int number = order ? order[i] : i;
    out_keys[at] = key;
    if constexpr (LAST) out_step[at] = info[number];
    else out_order[at] = number;
  }
}

// first[p] = first sorted position whose primitive is >= p
__global__ __launch_bounds__(256) void step_first_kernel(const int32_t* __restrict__ prim, int S, int N, int32_t* __restrict__ first) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i > N) return;
  int lo = 0, hi = S;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (prim[mid] < i) lo = mid + 1;
    else hi = mid;
  }
  first[i] = lo;
}

struct StepIndex {
  const int32_t* prim;    // of StepSort
  const int32_t* first;
  const int4* step;
};

constexpr int kGeoFloats = 16;                            // 15 geometry sums, one pad
constexpr int kRowFloats = kGradFloats + kGeoFloats;      // of a head or tail row
constexpr int kTrainChunk = 128;                          // steps of a chunk, at the most (train_chunk_steps)

// A chunk's run of one primitive: steps [begin, end), and where its sums belong.
struct StepRun {
  int p, begin, end;
  bool complete, goes_on;
};
// A chunk's workgroup keeps the primitives of its steps in LDS, and those of the step before and of the one behind (-1: there is
// none): where a run ends is seen without a look-up that would have to be waited for.
struct ChunkPrims {
  int prim[kTrainChunk + 2];
};
__device__ __forceinline__ void load_chunk(const StepIndex& ix, int S, int begin, int end, int t, int threads, ChunkPrims& s) {
  for (int k = t; k < end - begin + 2; k += threads) {
    const int i = begin - 1 + k;
    s.prim[k] = i >= 0 && i < S ? ix.prim[i] : -1;
  }
}
__device__ __forceinline__ StepRun chunk_run(const ChunkPrims& s, int pos, int chunk_begin, int chunk_end, int lane) {
  static_assert(kTrainChunk <= 128, "two looks");
  asm volatile("" : "+v"(lane));         // (or addresses are formed ahead of the loop over the runs and kept)
  const int n = chunk_end - chunk_begin, at = pos - chunk_begin;        // prim[at + 1] is that of step pos
  StepRun r;
  r.p = __builtin_amdgcn_readfirstlane(s.prim[at + 1]);
  const int near = at + lane, far = near + 64;
  const unsigned long long a = __ballot(near >= n || s.prim[min(near, n) + 1] != r.p);
  const unsigned long long b = __ballot(far >= n || s.prim[min(far, n) + 1] != r.p);
  r.begin = pos;
  r.end = a ? pos + (int)__builtin_ctzll(a) : b ? pos + 64 + (int)__builtin_ctzll(b) : chunk_end;
  r.goes_on = r.end == chunk_end && __builtin_amdgcn_readfirstlane(s.prim[n + 1]) == r.p;
  r.complete = !r.goes_on && __builtin_amdgcn_readfirstlane(s.prim[at]) != r.p;
  return r;
}
// Where the steps first, first + STRIDE, ... of a run lie, a step in each lane; the last one's in those that have none.
template <int STRIDE>
__device__ __forceinline__ int4 walk_steps(const StepIndex& ix, int first, int end, int lane) {
  static_assert(kTrainChunk <= 64 * STRIDE, "a lane for every step");
  asm volatile("" : "+v"(lane));         // (as in chunk_run)
  return ix.step[min(first + STRIDE * lane, end - 1)];
}
// head rows come first, then tail rows
__device__ __forceinline__ float* run_row(float* rows, const StepRun& r, int chunk, int num_chunks) {
  return rows + (size_t)(r.goes_on ? num_chunks + chunk : chunk) * kRowFloats;
}
__device__ __forceinline__ GradRows run_dest(float* rows, const GradRows& grads, const StepRun& r, int chunk, int num_chunks) {
  if (!r.complete) return packed_grad_rows(run_row(rows, r, chunk, num_chunks));
  const size_t p = (size_t)r.p;
  return GradRows{grads.W1 + p * 2304, grads.b1 + p * 32, grads.W2 + p * 1024, grads.b2 + p * 32, grads.W3 + p * 128, grads.b3 + p * 4};
}

// ---------------------------------------------------------------------------------------------
// geometry: the terms of geometry_partials_kernel (mlpsp_records_reverse.hip) over a chunk's steps, lane = pixel
// ---------------------------------------------------------------------------------------------
struct GeoGrads {
  float *pos, *scale, *quat;
};
// The per-primitive linear maps of the local-frame sums (np_tile_kernels.cu:439-479).
__device__ __forceinline__ void geometry_store(const float v[15], float qw, float qx, float qy, float qz, size_t p,
                                               const GeoGrads& out) {
  const Vec3 gd = quat_rotate(qw, qx, qy, qz, Vec3{v[0], v[1], v[2]});
  out.pos[p * 3] = gd.x;
  out.pos[p * 3 + 1] = gd.y;
  out.pos[p * 3 + 2] = gd.z;
  out.scale[p * 3] = v[3];
  out.scale[p * 3 + 1] = v[4];
  out.scale[p * 3 + 2] = v[5];
  const float r00 = v[6], r01 = v[7], r02 = v[8], r10 = v[9], r11 = v[10], r12 = v[11], r20 = v[12], r21 = v[13],
              r22 = v[14];
  out.quat[p * 4] = r01 * (-2.f * qz) + r02 * (2.f * qy) + r10 * (2.f * qz) + r12 * (-2.f * qx) + r20 * (-2.f * qy) +
                    r21 * (2.f * qx);
  out.quat[p * 4 + 1] = r01 * (2.f * qy) + r02 * (2.f * qz) + r10 * (2.f * qy) + r11 * (-4.f * qx) + r12 * (-2.f * qw) +
                        r20 * (2.f * qz) + r21 * (2.f * qw) + r22 * (-4.f * qx);
  out.quat[p * 4 + 2] = r00 * (-4.f * qy) + r01 * (2.f * qx) + r02 * (2.f * qw) + r10 * (2.f * qx) + r12 * (2.f * qz) +
                        r20 * (-2.f * qw) + r21 * (2.f * qz) + r22 * (-4.f * qy);
  out.quat[p * 4 + 3] = r00 * (-4.f * qz) + r01 * (-2.f * qw) + r02 * (2.f * qx) + r10 * (2.f * qw) + r11 * (-4.f * qz) +
                        r12 * (2.f * qy) + r20 * (2.f * qx) + r21 * (2.f * qy);
}

// A workgroup per chunk, the steps of a run to its wavefronts in turn.  Bound by memory (1,280 bytes a step) where there are many
// steps, by the chain of look-ups, loads and sums of a run where there are few: a lane knows where a step lies, four steps are asked
// for together, and a run's 15 sums do not go through LDS.  650,000 steps: 185 -> 174 us, 4.8 TB/s; 80,000: 36 -> 28.
constexpr int kGeoWaves = 4, kGeoAhead = 4;
__global__ __launch_bounds__(64 * kGeoWaves) void train_geometry_kernel(
    StepIndex ix, int S, int chunk_steps, int num_chunks, const unsigned char* __restrict__ records,
    const float* __restrict__ falloff, const float* __restrict__ logs, const float* __restrict__ quats,
    float* __restrict__ rows, GeoGrads out) {
  __shared__ __attribute__((aligned(16))) float s_sum[2][kGeoWaves][16];
  __shared__ ChunkPrims prims;
  const int chunk = (int)blockIdx.x, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = threadIdx.x & 63;
  const int chunk_begin = chunk * chunk_steps, chunk_end = min(S, chunk_begin + chunk_steps);
  load_chunk(ix, S, chunk_begin, chunk_end, threadIdx.x, 64 * kGeoWaves, prims);
  __syncthreads();
  int turn = 0;
  for (int pos = chunk_begin; pos < chunk_end; turn ^= 1) {
    const StepRun run = chunk_run(prims, pos, chunk_begin, chunk_end, l);
    const size_t p = (size_t)run.p;
    const int4 where = walk_steps<kGeoWaves>(ix, run.begin + wave, run.end, l);
    const int count = (run.end - run.begin - wave + kGeoWaves - 1) / kGeoWaves;
    const float qw = quats[p * 4], qx = quats[p * 4 + 1], qy = quats[p * 4 + 2], qz = quats[p * 4 + 3];
    const float mx = det_exp(-2.f * logs[p * 3]), my = det_exp(-2.f * logs[p * 3 + 1]), mz = det_exp(-2.f * logs[p * 3 + 2]);
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = 0.f;
    for (int first = 0; first < count; first += kGeoAhead) {
      float4 offset[kGeoAhead];
      float fall[kGeoAhead];
#pragma unroll
      for (int u = 0; u < kGeoAhead; ++u) {
        const int k = min(first + u, count - 1);
        offset[u] = reinterpret_cast<const float4*>(records + (size_t)__builtin_amdgcn_readlane(where.x, k) * kStepBytes + kStepPlaneC)[l];
        fall[u] = falloff[(size_t)__builtin_amdgcn_readlane(where.y, k) * 64 + l];
      }
#pragma unroll
      for (int u = 0; u < kGeoAhead; ++u) {
        if (first + u >= count) break;
        const float a = fall[u], dx = offset[u].x, dy = offset[u].y, dz = offset[u].z;
        const Vec3 q = quat_rotate_conj(qw, qx, qy, qz, Vec3{dx, dy, dz});
        const float gx = -a * mx * q.x, gy = -a * my * q.y, gz = -a * mz * q.z;
        v[0] += gx;
        v[1] += gy;
        v[2] += gz;
        v[3] += a * mx * q.x * q.x;
        v[4] += a * my * q.y * q.y;
        v[5] += a * mz * q.z * q.z;
        v[6] += dx * gx; v[7] += dx * gy; v[8] += dx * gz;
        v[9] += dy * gx; v[10] += dy * gy; v[11] += dy * gz;
        v[12] += dz * gx; v[13] += dz * gy; v[14] += dz * gz;
      }
    }
#pragma unroll
    for (int k = 0; k < 15; ++k) v[k] = sum_up_to_lane<false>(v[k]);      // (the last lane has all)
    if (l == 63) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        *reinterpret_cast<float4*>(&s_sum[turn][wave][4 * k]) = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
    }
    __syncthreads();                   // (the one barrier of a turn: the next writes the other half)
    if (wave == 0) {
      float total = 0.f;
      if (l < 15) {
#pragma unroll
        for (int w = 0; w < kGeoWaves; ++w) total += s_sum[turn][w][l];
      }
      if (!run.complete) {
        if (l < 15) run_row(rows, run, chunk, num_chunks)[kGradFloats + l] = total;
      } else {
#pragma unroll
        for (int k = 0; k < 15; ++k) v[k] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(total), k));
        if (l == 0) geometry_store(v, qw, qx, qy, qz, p, out);
      }
    }
    pos = run.end;
  }
}

// ---------------------------------------------------------------------------------------------
// MLP weight gradients, 16-bit operands: the blocks of mlpsp_vjp16_steps.hpp.  A workgroup per chunk, half a step to a wavefront.
// ---------------------------------------------------------------------------------------------
// What lane (n, g) needs of record n of half h of a step: its group's three inputs (the ray direction, the hit offset), the
// output adjoints, the masks.  Each lane asks for its own inputs only: chosen behind the loads of both, every request was
// waited for as soon as it was made (f32 / 16-bit gradient call of 648,000 steps 5.40 -> 5.32 / 2.32 -> 2.18 ms).
struct StepRecord {
  float x[3];
  float4 d;
  uint32_t mask1, mask2;
};
__device__ __forceinline__ StepRecord step_record(const unsigned char* __restrict__ records, const float4* __restrict__ d4,
                                                  const float* __restrict__ rays_d, int4 at, int half, int n, int g, int W,
                                                  int pixels) {
  StepRecord r;
  const int px = 32 * half + n;
  const unsigned char* __restrict__ rec = records + (size_t)at.x * kStepBytes;
  r.d = d4[(size_t)at.y * 64 + px];
  const unsigned char* offset = rec + kStepPlaneC + 16 * px;
  const float* dir = rays_d + 3 * (size_t)min(at.w + (px >> 3) * W + (px & 7), pixels - 1);      // (whatever it is outside the image)
  const Float3 x = load3(g ? reinterpret_cast<const float*>(offset) : dir, 0);
  r.x[0] = x.x;
  r.x[1] = x.y;
  r.x[2] = x.z;
  r.mask1 = *reinterpret_cast<const uint32_t*>(offset + 12);
  r.mask2 = reinterpret_cast<const uint32_t*>(rec + kStepPlaneD)[px];
  return r;
}
// A wavefront's share of a run: one half of every STRIDE-th step, from `first` on (walk_steps).  The first record is requested
// beside the run's weights (walk_record), and walk_halves has the next record under way while one is worked on (two or three: no
// faster): work(record) for those that have an adjoint.  Records without one get inputs of zero, whatever ray their lane has.  A
// wavefront without a step (first >= end) asks for the last one's and drops it.
__device__ __forceinline__ StepRecord walk_record(const int4& where, int k, int half, const unsigned char* __restrict__ records,
                                                  const float4* __restrict__ d4, const float* __restrict__ rays_d, int W,
                                                  int pixels, int lane) {
  return step_record(records, d4, rays_d, make_int4(__builtin_amdgcn_readlane(where.x, k), __builtin_amdgcn_readlane(where.y, k), 0,
                                                    __builtin_amdgcn_readlane(where.w, k)), half, lane & 31, lane >> 5, W, pixels);
}
template <int STRIDE, bool FRESH, typename Work>
__device__ __forceinline__ void walk_halves(const int4& where, StepRecord next, int first, int end, int half,
                                            const unsigned char* __restrict__ records, const float4* __restrict__ d4,
                                            const float* __restrict__ rays_d, int W, int pixels, int lane, Work&& work) {
  const int count = (end - first + STRIDE - 1) / STRIDE;
  for (int i = 0; i < count; ++i) {
    StepRecord r = next;
    // (at the end the last one again: under a condition the request is waited for)
    next = walk_record(where, min(i + 1, count - 1), half, records, d4, rays_d, W, pixels, FRESH ? fresh_lane() : lane);
    const bool adjoint = r.d.x != 0.f || r.d.y != 0.f || r.d.z != 0.f || r.d.w != 0.f;
    if (__ballot(adjoint) == 0ull) continue;
#pragma unroll
    for (int c = 0; c < 3; ++c) r.x[c] = adjoint ? r.x[c] : 0.f;
    work(r);
  }
}

// A wavefront's share of the rows of primitives without a step, stored behind its chunk: the chunks end at different times, and
// the stores go on beside the products of the others.  The whole call at 648,000 steps of 200,000 primitives with these 2.8 GB in
// a launch behind it / here / here past the caches: f32 5.54 / 5.31 / 5.30 ms, fp16 1.94 / 1.74 / 1.70; a primitive per block of
// products 5.34 and 1.83.  Ahead of the chunk its first record is waited for behind the stores: the f32 kernel of 80,000 steps
// takes 676 us instead of 663.  With the rows of the attributes' gradient (512 channels, four slots: 1.6 GB more) fp16 1.52 -> 1.62.
// What a wavefront may be given of them: few steps make few chunks, and the four wavefronts of one would store all rows alone
// (16 steps of 200,000 primitives 56 ms, in a launch of their own 0.7).  Above it that launch, behind the gradients.  Call in us,
// a launch / here, at KB per wavefront:
//   f32    200,000 primitives  4,000 steps  2,761   628 /   649     8,000  1,380   651 / 648    16,000  690   735 /   677
//           60,000             1,008        3,287   270 /   382     2,400  1,380   267 / 271     4,000  828   274 /   270
//           20,000             1,008        1,096   169 /   203     2,400    460   166 / 163     8,000  138   193 /   169
//   fp16   200,000            16,000          690   641 /   652    24,000    460   663 / 678    32,000  345   703 /   701
//           60,000             1,008        3,287   244 /   358     4,000    828   240 / 243     8,000  414   251 /   243
//          and 512 attribute channels of four slots, 200,000: 32,000  545   997 / 1,006    48,000  363  1,056 / 1,049    80,000  436  1,165 / 1,116
constexpr int64_t kZeroShare32 = 1024 * 1024, kZeroShare16 = 448 * 1024;
template <int WAVES>
__device__ __forceinline__ void zero_share(const StepIndex& ix, int N, const ZeroRows& zero, int chunk, int num_chunks, int wave,
                                           int lane) {
  for (int group = chunk * WAVES + wave; group * kZeroGroup < N; group += num_chunks * WAVES) zero_rows<true>(ix.first, N, zero, group, lane);
}

template <typename T>
__global__ __launch_bounds__(64 * kVjp16Waves) __attribute__((amdgpu_waves_per_eu(3, 3))) void train_vjp16_kernel(
    StepIndex ix, int S, int chunk_steps, int num_chunks, const unsigned char* __restrict__ records,
    const float4* __restrict__ d4, const float* __restrict__ rays_d, int W, int H, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
    const float* __restrict__ b2, const float* __restrict__ W3, float scale, float* __restrict__ rows, GradRows grads,
    int32_t* __restrict__ nonfinite, int N, ZeroRows zero) {
  __shared__ Vjp16StepsLds<T> lds;
  __shared__ ChunkPrims prims;
  Vjp16Shared<T>& s = lds.s;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int chunk = blockIdx.x, chunk_end = min(S, (chunk + 1) * chunk_steps);
  float kf[6];
#pragma unroll
  for (int f = 0; f < 6; ++f)
    kf[f] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint((freq[f] * att[f]) * 0.159154943f)));
  const int chunk_begin = chunk * chunk_steps, first = wave >> 1;
  load_chunk(ix, S, chunk_begin, chunk_end, t, 64 * kVjp16Waves, prims);
  __syncthreads();
  StepRun run = chunk_run(prims, chunk_begin, chunk_begin, chunk_end, lane);
  Vjp16Request weights = vjp16_request(W1, b1, W2, b2, W3, (size_t)run.p, wave, lane);
  int4 where = walk_steps<kVjp16Waves / 2>(ix, run.begin + first, run.end, lane);
  bool bad = false;
  for (;;) {
    StepRecord record = walk_record(where, 0, wave & 1, records, d4, rays_d, W, W * H, lane);
    vjp16_load<T>(weights, wave, lane, s);
    if (t < 4) s.zero[t] = 0u;
    Vjp16StepSums sum;
    sum.clear();
    __syncthreads();
    walk_halves<kVjp16Waves / 2, true>(where, record, run.begin + first, run.end, wave & 1, records, d4, rays_d, W, W * H, lane, [&](const StepRecord& r) {
      vjp16_step_block<T>(s, sum, s.wave[wave], r.x, r.d, r.mask1, r.mask2, kf, scale, lane);
    });
    const StepRun next = run.end < chunk_end ? chunk_run(prims, run.end, chunk_begin, chunk_end, lane) : run;
    weights = vjp16_request(W1, b1, W2, b2, W3, (size_t)next.p, wave, lane);
    where = walk_steps<kVjp16Waves / 2>(ix, next.begin + first, next.end, lane);
    const int waves = min(2 * (run.end - run.begin), kVjp16Waves), slots = min(waves, kVjp16Slots);
    __syncthreads();
    if (wave < slots) vjp16_park<false>(sum, lds.sums[wave], lane);
    if (waves > slots) {
      __syncthreads();
      if (wave >= slots && wave < waves) vjp16_park<true>(sum, lds.sums[wave - slots], lane);
    }
    __syncthreads();
    bad |= store_row_sums(lds.sums[0], kGradFloats, slots, run_dest(rows, grads, run, chunk, num_chunks), 1.f / scale, t,
                          64 * kVjp16Waves);
    if (run.end >= chunk_end) break;
    run = next;
    __syncthreads();
  }
  zero_share<kVjp16Waves>(ix, N, zero, chunk, num_chunks, wave, lane);
  if (__ballot(bad) != 0ull && lane == 0) atomicOr(nonfinite, 1);
}

// ---------------------------------------------------------------------------------------------
// MLP weight gradients in f32: the blocks of mlpsp_vjp32.hpp.  A workgroup per chunk, half a step to a wavefront.
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(64 * kVjp32Waves) __attribute__((amdgpu_waves_per_eu(2, 2))) void train_vjp_f32_kernel(
    StepIndex ix, int S, int chunk_steps, int num_chunks, const unsigned char* __restrict__ records,
    const float4* __restrict__ d4, const float* __restrict__ rays_d, int W, int H, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
    const float* __restrict__ b2, const float* __restrict__ W3, float scale, float* __restrict__ rows, GradRows grads,
    int32_t* __restrict__ nonfinite, int N, ZeroRows zero) {
  __shared__ Vjp32Lds s;
  __shared__ ChunkPrims prims;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int chunk = blockIdx.x, chunk_end = min(S, (chunk + 1) * chunk_steps);
  const SplitUnits u;
  PhaseFactors factors;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    factors.freq[f] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(freq[f])));
    factors.att[f] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(att[f])));
  }
  if (t < 4) s.zero[t] = 0u;
  for (int k = t; k < kCircleEntries; k += 64 * kVjp32Waves) s.circle[k] = f32x2v{kCircle.at[k][0], kCircle.at[k][1]};
  const int chunk_begin = chunk * chunk_steps, first = wave >> 1;
  load_chunk(ix, S, chunk_begin, chunk_end, t, 64 * kVjp32Waves, prims);
  __syncthreads();
  StepRun run = chunk_run(prims, chunk_begin, chunk_begin, chunk_end, lane);
  Vjp32Request weights = vjp32_request(W1, b1, W2, b2, W3, (size_t)run.p, wave, lane);
  int4 where = walk_steps<kVjp32Waves / 2>(ix, run.begin + first, run.end, lane);
  bool bad = false;
  // The adjoints lifted first; a run whose sums this takes out of range is gone through again without.
  float by = scale * kVjp32Lift;
  for (;;) {
    const StepRecord record = walk_record(where, 0, wave & 1, records, d4, rays_d, W, W * H, lane);
    vjp32_load(weights, wave, lane, s, u);
    Vjp32Sums sum;
    sum.clear();
    __syncthreads();
    walk_halves<kVjp32Waves / 2, false>(where, record, run.begin + first, run.end, wave & 1, records, d4, rays_d, W, W * H, lane, [&](const StepRecord& r) {
      vjp32_block(s, sum, s.wave[wave], r.x, r.d, r.mask1, r.mask2, factors, by, lane, u);
    });
    StepRun next = run.end < chunk_end ? chunk_run(prims, run.end, chunk_begin, chunk_end, lane) : run;
    weights = vjp32_request(W1, b1, W2, b2, W3, (size_t)next.p, wave, lane);
    where = walk_steps<kVjp32Waves / 2>(ix, next.begin + first, next.end, lane);
    const int waves = min(2 * (run.end - run.begin), kVjp32Waves);
    if (wave < waves) vjp32_park(sum, reinterpret_cast<float*>(&s.wave[wave]), lane);
    __syncthreads();
    const bool beyond = store_row_sums(reinterpret_cast<const float*>(&s.wave[0]), sizeof(Vjp32Wave) / 4, waves,
                                       run_dest(rows, grads, run, chunk, num_chunks), 1.f / by, t, 64 * kVjp32Waves);
    if (lane == 0) s.beyond[wave] = __ballot(beyond) != 0ull;
    __syncthreads();
    const bool again = __builtin_amdgcn_readfirstlane(s.beyond[0] | s.beyond[1] | s.beyond[2] | s.beyond[3]) != 0;
    if (again && by != scale) {
      by = scale;
      weights = vjp32_request(W1, b1, W2, b2, W3, (size_t)run.p, wave, lane);
      where = walk_steps<kVjp32Waves / 2>(ix, run.begin + first, run.end, lane);
      continue;
    }
    bad |= again;
    if (run.end >= chunk_end) break;
    by = scale * kVjp32Lift;
    run = next;
  }
  zero_share<kVjp32Waves>(ix, N, zero, chunk, num_chunks, wave, lane);
  if (__ballot(bad) != 0ull && lane == 0) atomicOr(nonfinite, 1);
}

// ---------------------------------------------------------------------------------------------
// One workgroup per chunk and quarter of a row: the sum of the rows of the primitive whose steps begin in the chunk and go
// on in the next (its tail row here, tails in between, the head row of its last chunk); nothing if there is none.  What
// lasts is a primitive with steps in most tiles, hundreds of rows one after the other: sixteen of them are in flight, and
// its columns are shared out (650,000 steps in chunks of 64: one workgroup and eight in flight 0.35 ms, this 0.21; in chunks of
// 128 as now 0.035).
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void train_join_kernel(StepIndex ix, int S, int chunk_steps, int num_chunks,
                                                         const float* __restrict__ rows, const float* __restrict__ quats,
                                                         GradRows grads, GeoGrads geo, int32_t* __restrict__ nonfinite) {
  const int t = threadIdx.x, cf = blockIdx.x, k = blockIdx.y * 256 + t;
  const SpanningRun run = spanning_run(ix.prim, ix.first, S, cf, chunk_steps);
  if (run.p < 0) return;
  const int cl = run.last_chunk;
  const size_t np = (size_t)run.p;
  __shared__ float s_geo[16][kGeoFloats];
  bool bad = false;
  const auto row = [&](int c) { return rows + (size_t)(c < cl ? num_chunks + c : c) * kRowFloats; };
  if (k < kGradFloats / 4) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 16
    for (int c = cf; c <= cl; ++c) {
      const float4 v = reinterpret_cast<const float4*>(row(c))[k];
      acc.x += v.x;
      acc.y += v.y;
      acc.z += v.z;
      acc.w += v.w;
    }
    bad |= !(__builtin_fabsf(acc.x) <= 3.4028235e38f) || !(__builtin_fabsf(acc.y) <= 3.4028235e38f) ||
           !(__builtin_fabsf(acc.z) <= 3.4028235e38f) || !(__builtin_fabsf(acc.w) <= 3.4028235e38f);
    // float4 ranges of the parts: [0,576) W1, [576,584) b1, [584,840) W2, [840,848) b2, [848,880) W3, 880 b3
    float4* dst;
    if (k < 576) dst = reinterpret_cast<float4*>(grads.W1) + np * 576 + k;
    else if (k < 584) dst = reinterpret_cast<float4*>(grads.b1) + np * 8 + (k - 576);
    else if (k < 840) dst = reinterpret_cast<float4*>(grads.W2) + np * 256 + (k - 584);
    else if (k < 848) dst = reinterpret_cast<float4*>(grads.b2) + np * 8 + (k - 840);
    else if (k < 880) dst = reinterpret_cast<float4*>(grads.W3) + np * 32 + (k - 848);
    else dst = reinterpret_cast<float4*>(grads.b3) + np;
    *dst = acc;
  }
  if (__ballot(bad) != 0ull && (t & 63) == 0) atomicOr(nonfinite, 1);
  if (blockIdx.y != 3) return;         // (the last quarter is the shortest)
  float v = 0.f;
  for (int c = cf + (t >> 4); c <= cl; c += 16) v += (t & 15) < 15 ? row(c)[kGradFloats + (t & 15)] : 0.f;
  s_geo[t >> 4][t & 15] = v;
  __syncthreads();
  if (t == 0) {
    float sums[15];
    for (int k = 0; k < 15; ++k) {
      float a = 0.f;
      for (int j = 0; j < 16; ++j) a += s_geo[j][k];
      sums[k] = a;
    }
    geometry_store(sums, quats[np * 4], quats[np * 4 + 1], quats[np * 4 + 2], quats[np * 4 + 3], np, geo);
  }
}

// Steps per chunk: as many as a wavefront has lanes for (twice that is no faster), fewer where that would leave fewer than four
// chunks for each of the 512 workgroups that run at once (f32; 768 in 16 bits), 16 at the least.  Gradient call in us, f32, a half, as much and
// twice as much of that rule at 51,600 steps: 494, 489, 526.
inline int train_chunk_steps(int64_t S) {
  const int64_t per = S / 2048 / 8 * 8;
  return per >= kTrainChunk ? kTrainChunk : per <= 16 ? 16 : (int)per;
}

// The sorted steps, then head and tail rows of every chunk.
struct TrainScratch : StepSort {
  float* rows;
  int chunk_steps, num_chunks;
};
inline TrainScratch train_scratch(void* base, int64_t S, int N) {
  TrainScratch t{};
  static_cast<StepSort&>(t) = step_sort(base, S, N);
  t.rows = (float*)((unsigned char*)base + t.bytes);
  t.chunk_steps = train_chunk_steps(S);
  t.num_chunks = (int)((S + t.chunk_steps - 1) / t.chunk_steps);
  t.bytes += step_align((size_t)2 * t.num_chunks * kRowFloats * 4);
  return t;
}

}  // namespace mlpsp

using namespace mlpsp;

MLPSP_API int mlpsp_train_reverse(const int32_t* tile_offsets_dev, int64_t num_pairs, int width, int height,
                                  const void* workspace_dev, size_t workspace_bytes, const float* grad_rgb_dev,
                                  const float* grad_t_dev, float* d4_dev, float* falloff_dev, mlpsp_stream_t stream) {
  const int64_t T = checked_num_tiles(width, height, 8, 8);
  if (T <= 0 || T > 2147483647LL - 8 || num_pairs < 0 || num_pairs > 2147483647LL) return MLPSP_E_ARGUMENT;
  if (!workspace_dev || workspace_bytes < step_tables_bytes(num_pairs, T)) return MLPSP_E_SCRATCH;
  if (!tile_offsets_dev || !grad_rgb_dev || !grad_t_dev || !d4_dev || !falloff_dev || ((uintptr_t)d4_dev & 15u))
    return MLPSP_E_ARGUMENT;
  const StepPool sp = step_pool_carve(const_cast<void*>(workspace_dev), workspace_bytes, num_pairs, T);
  const int ntx = ceil_div(width, 8), nty = ceil_div(height, 8);
  hipLaunchKernelGGL(train_reverse_kernel, dim3(superblock_grid(ntx, nty)), dim3(64), 0, (hipStream_t)stream, tile_offsets_dev,
                     sp.tile_base, sp.chunk_table, sp.records, grad_rgb_dev, grad_t_dev, width, height, ntx, nty,
                     (float4*)d4_dev, falloff_dev);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}

MLPSP_API size_t mlpsp_train_scratch_bytes(int64_t num_steps, int num_primitives) {
  if (num_steps < 0 || num_steps > 2147483647LL || num_primitives < 0) return 0;
  return train_scratch(nullptr, num_steps, num_primitives).bytes;
}

MLPSP_API int mlpsp_train_group(const int32_t* tile_offsets_dev, int64_t num_pairs, int width, int height,
                                const void* workspace_dev, size_t workspace_bytes, int64_t num_steps, int num_primitives,
                                void* scratch_dev, size_t scratch_bytes, mlpsp_stream_t stream) {
  const int64_t T = checked_num_tiles(width, height, 8, 8);
  if (T <= 0 || T > 2147483647LL - 8 || num_pairs < 0 || num_pairs > 2147483647LL || num_steps < 0 ||
      num_steps > 2147483647LL - 8192 || num_primitives < 0 || !tile_offsets_dev)
    return MLPSP_E_ARGUMENT;
  if (!workspace_dev || workspace_bytes < step_tables_bytes(num_pairs, T)) return MLPSP_E_SCRATCH;
  const TrainScratch t = train_scratch(scratch_dev, num_steps, num_primitives);
  if (!scratch_dev || reinterpret_cast<uintptr_t>(scratch_dev) % 256 != 0 || scratch_bytes < t.bytes) return MLPSP_E_SCRATCH;
  const StepPool sp = step_pool_carve(const_cast<void*>(workspace_dev), workspace_bytes, num_pairs, T);
  hipStream_t s = (hipStream_t)stream;
  const int S = (int)num_steps;
  if (S > 0) {
    int bits = 1;
    while (bits < 31 && (1 << bits) < num_primitives) ++bits;
    const int passes = (bits + kSortBits - 1) / kSortBits, width_bits = (bits + passes - 1) / passes;
    const int share = sort_keys(S), blocks = (S + share - 1) / share;
    // (the rows are written after the sort: its buffers lie there)
    unsigned char* p = (unsigned char*)t.rows;
    int4* info = (int4*)p;
    p += step_align((size_t)S * 16);
    int32_t *keys[2], *order[2];
    for (int k = 0; k < 2; ++k) {
      keys[k] = (int32_t*)p;
      p += step_align((size_t)S * 4);
      order[k] = (int32_t*)p;
      p += step_align((size_t)S * 4);
    }
    int32_t* hist = (int32_t*)p;
    p += (size_t)blocks * (1 << width_bits) * 4;
    // (cannot be: 220 bytes of rows per step at least, 34 of these)
    if ((size_t)(p - (unsigned char*)scratch_dev) > t.bytes) return MLPSP_E_SCRATCH;
    hipLaunchKernelGGL(step_list_kernel, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, s, tile_offsets_dev, sp.tile_base,
                       sp.chunk_table, sp.ids, (int)T, width, ceil_div(width, 8), keys[0], info);
    MLPSP_LAUNCH_CHECK();
    for (int pass = 0; pass < passes; ++pass) {
      const int32_t *in = keys[pass & 1], *numbers = pass == 0 ? nullptr : order[pass & 1];
      hipLaunchKernelGGL(step_hist_kernel, dim3((unsigned)blocks), dim3(kSortBlock), 0, s, in, S, share, pass * width_bits,
                         width_bits, blocks, hist);
      MLPSP_LAUNCH_CHECK();
      hipLaunchKernelGGL(step_sums_kernel, dim3(1), dim3(1024), 0, s, hist, blocks << width_bits);
      MLPSP_LAUNCH_CHECK();
      if (pass + 1 == passes)
        hipLaunchKernelGGL(step_scatter_kernel<true>, dim3((unsigned)blocks), dim3(kSortBlock), 0, s, in, numbers, S, share,
                           pass * width_bits, width_bits, blocks, hist, info, t.prim, (int32_t*)nullptr, t.step);
      else
        hipLaunchKernelGGL(step_scatter_kernel<false>, dim3((unsigned)blocks), dim3(kSortBlock), 0, s, in, numbers, S, share,
                           pass * width_bits, width_bits, blocks, hist, info, keys[(pass + 1) & 1], order[(pass + 1) & 1],
                           (int4*)nullptr);
      MLPSP_LAUNCH_CHECK();
    }
  }
  hipLaunchKernelGGL(step_first_kernel, dim3((unsigned)((num_primitives + 256) / 256)), dim3(256), 0, s, t.prim, S, num_primitives,
                     t.first);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}

namespace {
int train_gradients(int64_t num_steps, int64_t num_pairs, int width,
                                    int height, const void* workspace_dev, size_t workspace_bytes, const float* d4_dev,
                                    const float* falloff_dev, const float* rays_d_dev, const float* freq_dev,
                                    const float* att_dev, const float* W1, const float* b1, const float* W2, const float* b2,
                                    const float* W3, const float* log_scales_dev, const float* quats_dev, int num_primitives,
                                    int precision, float scale, void* scratch_dev, size_t scratch_bytes, float* gW1_dev,
                                    float* gb1_dev, float* gW2_dev, float* gb2_dev, float* gW3_dev, float* gb3_dev,
                                    float* grad_positions_dev, float* grad_log_scales_dev, float* grad_quats_dev,
                                    int32_t* nonfinite_dev, float* rows_dev, int row_floats, hipStream_t s) {
  const int64_t T = checked_num_tiles(width, height, 8, 8);
  if (T <= 0 || num_pairs < 0 || num_pairs > 2147483647LL || num_steps < 0 || num_steps > 2147483647LL || num_primitives <= 0)
    return MLPSP_E_ARGUMENT;
  if (precision < 0 || precision > 2 || !(scale > 0.f) || !(scale <= 3.4028235e38f)) return MLPSP_E_ARGUMENT;
  if (!workspace_dev || workspace_bytes < step_tables_bytes(num_pairs, T)) return MLPSP_E_SCRATCH;
  const TrainScratch t = train_scratch(scratch_dev, num_steps, num_primitives);
  if (!scratch_dev || reinterpret_cast<uintptr_t>(scratch_dev) % 256 != 0 || scratch_bytes < t.bytes) return MLPSP_E_SCRATCH;
  if (!rays_d_dev || !freq_dev || !att_dev || !W1 || !b1 || !W2 || !b2 || !W3 || !log_scales_dev || !quats_dev || !gW1_dev ||
      !gb1_dev || !gW2_dev || !gb2_dev || !gW3_dev || !gb3_dev || !grad_positions_dev || !grad_log_scales_dev ||
      !grad_quats_dev || !nonfinite_dev || (num_steps > 0 && (!d4_dev || !falloff_dev)))
    return MLPSP_E_ARGUMENT;
  if (((uintptr_t)W1 | (uintptr_t)b1 | (uintptr_t)W2 | (uintptr_t)b2 | (uintptr_t)d4_dev | (uintptr_t)gW1_dev |
       (uintptr_t)gb1_dev | (uintptr_t)gW2_dev | (uintptr_t)gb2_dev | (uintptr_t)gW3_dev | (uintptr_t)gb3_dev) & 15u)
    return MLPSP_E_ARGUMENT;
  const StepPool sp = step_pool_carve(const_cast<void*>(workspace_dev), workspace_bytes, num_pairs, T);
  MLPSP_HIP_TRY(clear_async(nonfinite_dev, sizeof(int32_t), s));
  const StepIndex ix{t.prim, t.first, t.step};
  const GradRows grads{gW1_dev, gb1_dev, gW2_dev, gb2_dev, gW3_dev, gb3_dev};
  const GeoGrads geo{grad_positions_dev, grad_log_scales_dev, grad_quats_dev};
  const int S = (int)num_steps;
  const int chunk_steps = t.chunk_steps, num_chunks = t.num_chunks;
  ZeroRows zero{};
  zero.add(gW1_dev, 2304);
  zero.add(gb1_dev, 32);
  zero.add(gW2_dev, 1024);
  zero.add(gb2_dev, 32);
  zero.add(gW3_dev, 128);
  zero.add(gb3_dev, 4);
  zero.add(grad_positions_dev, 3);
  zero.add(grad_log_scales_dev, 3);
  zero.add(grad_quats_dev, 4);
  if (rows_dev) zero.add(rows_dev, row_floats);
  const int64_t row_bytes = 4LL * (kGradFloats + 10 + (rows_dev ? row_floats : 0));
  const int64_t room = num_chunks * (precision == 0 ? kZeroShare32 * kVjp32Waves : kZeroShare16 * kVjp16Waves);
  const bool beside = num_primitives * row_bytes <= room;
  if (num_chunks > 0) {
    const int zeros_here = beside ? num_primitives : 0;
#define MLPSP_TRAIN_VJP(KERNEL, THREADS)                                                                                \
  hipLaunchKernelGGL(KERNEL, dim3((unsigned)num_chunks), dim3(THREADS), 0, s, ix, S, chunk_steps, num_chunks, sp.records, \
                     (const float4*)d4_dev, rays_d_dev, width, height, freq_dev, att_dev, W1, b1, W2, b2, W3, scale,   \
                     t.rows, grads, nonfinite_dev, zeros_here, zero)
    if (precision == 0) MLPSP_TRAIN_VJP(train_vjp_f32_kernel, 64 * kVjp32Waves);
    else if (precision == 1) MLPSP_TRAIN_VJP((train_vjp16_kernel<_Float16>), 64 * kVjp16Waves);
    else MLPSP_TRAIN_VJP((train_vjp16_kernel<__bf16>), 64 * kVjp16Waves);
#undef MLPSP_TRAIN_VJP
    MLPSP_LAUNCH_CHECK();
    hipLaunchKernelGGL(train_geometry_kernel, dim3((unsigned)num_chunks), dim3(64 * kGeoWaves), 0, s, ix, S, chunk_steps,
                       num_chunks, sp.records, falloff_dev, log_scales_dev, quats_dev, t.rows, geo);
    MLPSP_LAUNCH_CHECK();
    hipLaunchKernelGGL(train_join_kernel, dim3((unsigned)num_chunks, 4), dim3(256), 0, s, ix, S, chunk_steps, num_chunks,
                       t.rows, quats_dev, grads, geo, nonfinite_dev);
    MLPSP_LAUNCH_CHECK();
  }
  if (!beside) {
    launch_zero_rows(t.first, num_primitives, zero, s);
    MLPSP_LAUNCH_CHECK();
  }
  return MLPSP_OK;
}
}  // namespace

MLPSP_API int mlpsp_train_gradients(int64_t num_steps, int64_t num_pairs, int width, int height, const void*
    workspace_dev, size_t workspace_bytes, const float* d4_dev, const float* falloff_dev, const float* rays_d_dev, const
    float* freq_dev, const float* att_dev, const float* W1, const float* b1, const float* W2, const float* b2, const
    float* W3, const float* log_scales_dev, const float* quats_dev, int num_primitives, int precision, float scale, void*
    scratch_dev, size_t scratch_bytes, float* gW1_dev, float* gb1_dev, float* gW2_dev, float* gb2_dev, float* gW3_dev,
    float* gb3_dev, float* grad_positions_dev, float* grad_log_scales_dev, float* grad_quats_dev, int32_t* nonfinite_dev,
    mlpsp_stream_t stream) {
  return train_gradients(num_steps, num_pairs, width, height, workspace_dev, workspace_bytes, d4_dev, falloff_dev,
                         rays_d_dev, freq_dev, att_dev, W1, b1, W2, b2, W3, log_scales_dev, quats_dev, num_primitives,
                         precision, scale, scratch_dev, scratch_bytes, gW1_dev, gb1_dev, gW2_dev, gb2_dev, gW3_dev,
                         gb3_dev, grad_positions_dev, grad_log_scales_dev, grad_quats_dev, nonfinite_dev, nullptr, 0,
                         (hipStream_t)stream);
}

MLPSP_API int mlpsp_train_gradients_beside(int64_t num_steps, int64_t num_pairs, int width, int height, const void*
    workspace_dev, size_t workspace_bytes, const float* d4_dev, const float* falloff_dev, const float* rays_d_dev, const
    float* freq_dev, const float* att_dev, const float* W1, const float* b1, const float* W2, const float* b2, const
    float* W3, const float* log_scales_dev, const float* quats_dev, int num_primitives, int precision, float scale, void*
    scratch_dev, size_t scratch_bytes, float* gW1_dev, float* gb1_dev, float* gW2_dev, float* gb2_dev, float* gW3_dev,
    float* gb3_dev, float* grad_positions_dev, float* grad_log_scales_dev, float* grad_quats_dev, int32_t* nonfinite_dev,
    float* rows_dev, int row_floats, mlpsp_stream_t stream) {
  if (!rows_dev || row_floats <= 0) return MLPSP_E_ARGUMENT;
  return train_gradients(num_steps, num_pairs, width, height, workspace_dev, workspace_bytes, d4_dev, falloff_dev,
                         rays_d_dev, freq_dev, att_dev, W1, b1, W2, b2, W3, log_scales_dev, quats_dev, num_primitives,
                         precision, scale, scratch_dev, scratch_bytes, gW1_dev, gb1_dev, gW2_dev, gb2_dev, gW3_dev,
                         gb3_dev, grad_positions_dev, grad_log_scales_dev, grad_quats_dev, nonfinite_dev, rows_dev,
                         row_floats, (hipStream_t)stream);
}
