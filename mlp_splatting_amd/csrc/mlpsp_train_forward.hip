// libmlpsp_hip: forward pass of a differentiable frame on 8x8 tiles with the 72->32->32->4 MLP, keeping its steps
// (mlpsp_train.hpp).  One traversal: image, alpha and everything the backward needs; the counterpart of the reference's
// record forward (np_tile_kernels.cu:2925-3206; training_wmma.cuh:62-253), which walks the frame twice -- count, then
// emit at scanned offsets -- because per-pixel records must lie pixel after pixel.
//
// Geometry, order, activations and compositing are the f32 expressions of the render (f32 MLP: its bits with
// `render_order`, the record kernels' rounding of layer 2 without).  Bound by the MLP; the steps add 3.3 KB of contiguous
// stores per hit step.  200,000 primitives, 1200x680, f32: 4.7 ms, against 4.4 + 6.6 ms of the record forward's two walks.
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mfma16.hpp"
#include "mlpsp_mlp_mfma32.hpp"
#include "mlpsp_train.hpp"
#include "mlpsp_walk_f32.hpp"

namespace mlpsp {

struct TrainOut {
  float* rgb;
  float* alpha;
};

__device__ __forceinline__ bool train_not_finite(float v) { return !(__builtin_fabsf(v) <= 3.4028235e38f); }

// T = float: the MLP in exact f32 (REC: layer 2 rounded as the record kernels do); _Float16 / __bf16: reduced operands.
// All but the exact forward in the render's order report what is not finite, as the reduced-precision record forward does.
template <typename T> struct TrainLds { DirWords dir; };
template <> struct TrainLds<float> { DirOperands dir; };

template <typename T, bool REC>
__device__ __forceinline__ void train_forward_body(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, const unsigned char* __restrict__ packed, int N, int W, int H, int ntx, int nty,
    float thr, int max_hits, const StepPool& sp, TrainOut out, TrainLds<T>& s, WalkLds& s_walk) {
  constexpr bool F32 = sizeof(T) == 4;
  constexpr bool CHECKED = !F32 || REC;
  const int tile = superblock_tile(blockIdx.x, ntx, nty);
  if (tile < 0) return;
  const int l = threadIdx.x;
  const int x = (tile % ntx) * 8 + (l & 7), y = (tile / ntx) * 8 + (l >> 3);
  const bool valid = (x < W) && (y < H);
  const int pix = valid ? (y * W + x) : 0;
  const Float3 ro = valid ? load3(rays_o, pix) : Float3{0.f, 0.f, 0.f}, rd = valid ? load3(rays_d, pix) : Float3{0.f, 0.f, 0.f};
  float kf[3] = {0.f, 0.f, 0.f};
  if constexpr (F32) {
    encode_direction(rd.x, rd.y, rd.z, freq, att, s.dir);
  } else {
    phase_scales(freq, att, l >> 5, kf);
    encode_direction_words<T>(rd.x, rd.y, rd.z, kf, l, s.dir);
  }
  const int start = offsets[tile], end = offsets[tile + 1];
  float trans = 1.f, cr = 0.f, cg = 0.f, cb = 0.f;
  int used = 0;
  bool over = false, bad = false;
  StepWriter writer = step_writer_begin(start, tile);
  walk_tile_f32(
      order, start, end, N, prims, valid, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, thr, s_walk,
      [&]() { return valid && (trans >= kTransmittanceFloor) && (used < max_hits); },
      [&](int p, bool hit, const HitInfo& h, unsigned long long mask) {
        if (mask == 0ull) return true;
        const float dx = hit ? h.dx : 0.f, dy = hit ? h.dy : 0.f, dz = hit ? h.dz : 0.f;
        float o[4];
        uint32_t mk[2] = {0u, 0u};
        if constexpr (F32) {
          const float x6[6] = {rd.x, rd.y, rd.z, dx, dy, dz};
          mlp_wave_mfma32<REC, true, 32>(x6, freq, att, W1, b1, W2, b2, W3, b3, p, s.dir, o, mk);
        } else {
          bad |= mlp_wave_mfma16<T, true, true>(packed + (size_t)p * kPackStride, mask, l, dx, dy, dz, kf, s.dir, o, mk);
        }
        if constexpr (CHECKED) bad |= hit && (train_not_finite((dx + dy) + dz) || train_not_finite(h.decay));
        const int slot = step_writer_next(sp, writer, l);
        float R = 0.f, G = 0.f, Bc = 0.f, sigma_raw = 0.f, alpha = 0.f;
        const float before = trans;
        if (hit) {
          R = sigmoid(o[0]);
          G = sigmoid(o[1]);
          Bc = sigmoid(o[2]);
          sigma_raw = softplus(o[3]);
          alpha = 1.f - det_exp(-(sigma_raw * h.decay));
          if constexpr (CHECKED)
            bad |= train_not_finite((o[0] + o[1]) + (o[2] + o[3])) || train_not_finite((R + G) + (Bc + sigma_raw)) ||
                   train_not_finite(alpha);
          const float weight = trans * alpha;
          cr = fmaf(weight, R, cr);
          cg = fmaf(weight, G, cg);
          cb = fmaf(weight, Bc, cb);
          trans = trans * (1.f - alpha);
          ++used;
          if constexpr (CHECKED) bad |= train_not_finite(trans);
        }
        if (slot >= 0) step_store(sp, slot, l, p, hit, R, G, Bc, sigma_raw, before, alpha, h.decay, o[3], dx, dy, dz, mk[0], mk[1]);
        const bool live = valid && (trans >= kTransmittanceFloor);
        over |= live && (used >= max_hits);      // np_tile_kernels.cu:3166-3168: refused, never truncated silently
        return __ballot(live) != 0ull;
      });
  if constexpr (CHECKED) bad |= train_not_finite((cr + cg) + cb);
  if (l == 0) sp.tile_steps[tile] = writer.count;
  int bits = 0;
  if (__ballot(over) != 0ull) bits |= kTrainCapacity;
  if (__ballot(bad) != 0ull) bits |= kTrainNumeric;
  if (bits != 0 && l == 0) atomicOr(sp.head + 1, bits);
  if (valid) {
    store3(out.rgb, pix, cr, cg, cb);
    out.alpha[pix] = 1.f - trans;
  }
}

template <bool REC>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 3))) void train_forward_f32_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, int W, int H, int ntx, int nty, float thr, int max_hits, StepPool sp, TrainOut out) {
  __shared__ TrainLds<float> s;
  __shared__ WalkLds s_walk;
  train_forward_body<float, REC>(rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, nullptr, N, W, H,
                                 ntx, nty, thr, max_hits, sp, out, s, s_walk);
}

template <typename T>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 4))) void train_forward_mfma_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const unsigned char* __restrict__ packed, int N, int W, int H, int ntx, int nty, float thr,
    int max_hits, StepPool sp, TrainOut out) {
  __shared__ TrainLds<T> s;
  __shared__ WalkLds s_walk;
  train_forward_body<T, false>(rays_o, rays_d, prims, order, offsets, freq, att, nullptr, nullptr, nullptr, nullptr, nullptr,
                               nullptr, packed, N, W, H, ntx, nty, thr, max_hits, sp, out, s, s_walk);
}

// tile_base = exclusive sums of tile_steps, head[2] = their total; one workgroup (12,750 tiles: 6 us).
__global__ __launch_bounds__(1024) void step_scan_kernel(const int32_t* __restrict__ tile_steps, int T,
                                                         int32_t* __restrict__ tile_base, int32_t* __restrict__ head) {
  __shared__ int32_t s_wave[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int per = (T + 1023) / 1024, first = min(T, t * per), last = min(T, first + per);
  int sum = 0;
  for (int i = first; i < last; ++i) sum += tile_steps[i];
  int incl = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (lane >= d) incl += v;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  int before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    before += w < wave ? s_wave[w] : 0;
    total += s_wave[w];
  }
  int run = before + incl - sum;
  for (int i = first; i < last; ++i) {
    tile_base[i] = run;
    run += tile_steps[i];
  }
  if (t == 0) {
    tile_base[T] = total;
    head[2] = total;
  }
}

// Steps in tile order: primitive, pool slot and tile of each.
__global__ __launch_bounds__(256) void step_list_kernel(const int32_t* __restrict__ offsets, const int32_t* __restrict__ tile_base,
                                                        const int32_t* __restrict__ chunk_table, const int32_t* __restrict__ ids,
                                                        int T, int32_t* __restrict__ step_prim,
                                                        int32_t* __restrict__ step_slot_of, int32_t* __restrict__ step_tile) {
  const int tile = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if (tile >= T) return;
  const int base = tile_base[tile], count = tile_base[tile + 1] - base, table = (offsets[tile] >> 4) + tile;
  for (int m = lane; m < count; m += 64) {
    const int slot = step_slot(chunk_table, table, m);
    step_prim[base + m] = ids[slot];
    step_slot_of[base + m] = slot;
    step_tile[base + m] = tile;
  }
}

}  // namespace mlpsp

using namespace mlpsp;

namespace {
struct TrainFrame {
  int64_t T;
  int ntx, nty;
  StepPool sp;
};
int train_frame(int width, int height, int64_t num_pairs, void* workspace_dev, size_t workspace_bytes, TrainFrame& f) {
  f.T = checked_num_tiles(width, height, 8, 8);
  if (f.T <= 0 || f.T > 2147483647LL - 8 || num_pairs < 0 || num_pairs > 2147483647LL) return MLPSP_E_ARGUMENT;
  if (!workspace_dev || reinterpret_cast<uintptr_t>(workspace_dev) % 256 != 0 ||
      workspace_bytes < step_tables_bytes(num_pairs, f.T))
    return MLPSP_E_SCRATCH;
  f.ntx = ceil_div(width, 8);
  f.nty = ceil_div(height, 8);
  f.sp = step_pool_carve(workspace_dev, workspace_bytes, num_pairs, f.T);
  return MLPSP_OK;
}
int train_scan(const TrainFrame& f, hipStream_t s) {
  hipLaunchKernelGGL(step_scan_kernel, dim3(1), dim3(1024), 0, s, f.sp.tile_steps, (int)f.T, f.sp.tile_base, f.sp.head);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}
}  // namespace

MLPSP_API size_t mlpsp_train_workspace_bytes(int64_t num_pairs, int width, int height, int64_t pool_steps) {
  const int64_t T = checked_num_tiles(width, height, 8, 8);
  if (T <= 0 || num_pairs < 0) return 0;
  const int64_t worst = num_pairs + (int64_t)(kStepChunk * kStepGrab - 1) * T + kStepChunk * kStepGrab;
  if (pool_steps < 0 || pool_steps > worst) pool_steps = worst;
  return step_pool_bytes(num_pairs, T, pool_steps);
}

MLPSP_API int mlpsp_train_forward_f32(const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev,
                                      const int32_t* order_dev, const int32_t* tile_offsets_dev, int64_t num_pairs,
                                      const float* freq_dev, const float* att_dev, const float* W1, const float* b1,
                                      const float* W2, const float* b2, const float* W3, const float* b3,
                                      int num_primitives, int width, int height, float threshold, int max_hits,
                                      int render_order, void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev,
                                      float* out_alpha_dev, mlpsp_stream_t stream) {
  TrainFrame f;
  const int rc = train_frame(width, height, num_pairs, workspace_dev, workspace_bytes, f);
  if (rc != MLPSP_OK) return rc;
  if (!rays_o_dev || !rays_d_dev || !tile_offsets_dev || !freq_dev || !att_dev || !out_rgb_dev || !out_alpha_dev ||
      num_primitives < 0 || max_hits <= 0)
    return MLPSP_E_ARGUMENT;
  if (num_primitives > 0 && (!prim_records_dev || !W1 || !b1 || !W2 || !b2 || !W3 || !b3)) return MLPSP_E_ARGUMENT;
  if (((uintptr_t)W1 | (uintptr_t)b1 | (uintptr_t)W2 | (uintptr_t)b2) & 15u) return MLPSP_E_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  MLPSP_HIP_TRY(hipMemsetAsync(f.sp.head, 0, 64 * sizeof(int32_t), s));
  const dim3 grid(superblock_grid(f.ntx, f.nty)), block(64);
#define MLPSP_TRAIN_LAUNCH(REC)                                                                                       \
  hipLaunchKernelGGL((train_forward_f32_kernel<REC>), grid, block, 0, s, rays_o_dev, rays_d_dev,                      \
                     (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev, W1, b1, W2, b2, \
                     W3, b3, num_primitives, width, height, f.ntx, f.nty, threshold, max_hits, f.sp,                    \
                     TrainOut{out_rgb_dev, out_alpha_dev})
  if (render_order) MLPSP_TRAIN_LAUNCH(false);
  else MLPSP_TRAIN_LAUNCH(true);
#undef MLPSP_TRAIN_LAUNCH
  MLPSP_LAUNCH_CHECK();
  return train_scan(f, s);
}

MLPSP_API int mlpsp_train_forward_mfma(const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev,
                                       const int32_t* order_dev, const int32_t* tile_offsets_dev, int64_t num_pairs,
                                       const float* freq_dev, const float* att_dev, const void* packed_dev,
                                       int num_primitives, int width, int height, float threshold, int max_hits,
                                       int use_bf16, void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev,
                                       float* out_alpha_dev, mlpsp_stream_t stream) {
  TrainFrame f;
  const int rc = train_frame(width, height, num_pairs, workspace_dev, workspace_bytes, f);
  if (rc != MLPSP_OK) return rc;
  if (!rays_o_dev || !rays_d_dev || !tile_offsets_dev || !freq_dev || !att_dev || !out_rgb_dev || !out_alpha_dev ||
      num_primitives < 0 || max_hits <= 0)
    return MLPSP_E_ARGUMENT;
  if (num_primitives > 0 && (!prim_records_dev || !packed_dev)) return MLPSP_E_ARGUMENT;
  if (((uintptr_t)prim_records_dev % 128) != 0 || ((uintptr_t)packed_dev % 16) != 0) return MLPSP_E_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  MLPSP_HIP_TRY(hipMemsetAsync(f.sp.head, 0, 64 * sizeof(int32_t), s));
  const dim3 grid(superblock_grid(f.ntx, f.nty)), block(64);
#define MLPSP_TRAIN_LAUNCH(T)                                                                                         \
  hipLaunchKernelGGL((train_forward_mfma_kernel<T>), grid, block, 0, s, rays_o_dev, rays_d_dev,                       \
                     (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev,              \
                     (const unsigned char*)packed_dev, num_primitives, width, height, f.ntx, f.nty, threshold, max_hits, \
                     f.sp, TrainOut{out_rgb_dev, out_alpha_dev})
  if (use_bf16) MLPSP_TRAIN_LAUNCH(__bf16);
  else MLPSP_TRAIN_LAUNCH(_Float16);
#undef MLPSP_TRAIN_LAUNCH
  MLPSP_LAUNCH_CHECK();
  return train_scan(f, s);
}

MLPSP_API int mlpsp_train_list_steps(const int32_t* tile_offsets_dev, int64_t num_pairs, int width, int height,
                                     const void* workspace_dev, size_t workspace_bytes, int32_t* step_prim_dev,
                                     int32_t* step_slot_dev, int32_t* step_tile_dev, mlpsp_stream_t stream) {
  TrainFrame f;
  const int rc = train_frame(width, height, num_pairs, const_cast<void*>(workspace_dev), workspace_bytes, f);
  if (rc != MLPSP_OK) return rc;
  if (!tile_offsets_dev || !step_prim_dev || !step_slot_dev || !step_tile_dev) return MLPSP_E_ARGUMENT;
  hipLaunchKernelGGL(step_list_kernel, dim3((unsigned)((f.T + 3) / 4)), dim3(256), 0, (hipStream_t)stream, tile_offsets_dev,
                     f.sp.tile_base, f.sp.chunk_table, f.sp.ids, (int)f.T, step_prim_dev, step_slot_dev, step_tile_dev);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}
