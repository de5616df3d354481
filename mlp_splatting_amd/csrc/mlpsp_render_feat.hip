// libmlpsp_hip: tile-centre-order forward with the gated per-primitive feature channel, scalar f32.
//
// The reference read-modify-writes a C-float row of global memory per hit and per pixel
// (np_tile_kernels.cu:6036-6075).  Here the work is split in two kernels that keep the reference's
// arithmetic order per pixel and channel (feat = fma(w, mix, feat), mix the fma chain over the slots),
// so the result is bit-identical to a sequential evaluation:
//   1. the f32 render kernel (lane = pixel, mlpsp_render_f32.hpp) composites RGB and emits, per wavefront,
//      the primitives that hit and per pixel the weight w and the four gates (hit records,
//      mlpsp_hitrec.hpp): float[K][64] with K = 5 (w, g0..g3) or 1 (w), w = -1 where the primitive missed;
//   2. feat_accumulate_kernel turns the roles around: lane = channel.  A 256-thread block owns one
//      64-pixel item, a wavefront up to 128 channels of 32 or 16 of its pixels.  Per record the attribute rows
//      are two coalesced loads per slot, the per-pixel weight and gates are wave-uniform scalar operands, a
//      pixel the primitive missed costs one scalar branch, and every output row is written exactly once.
#include "mlpsp_device.hpp"
#include "mlpsp_hitrec.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mlp.hpp"
#include "mlpsp_render_f32.hpp"

namespace mlpsp {

typedef float f32x8 __attribute__((ext_vector_type(8)));

// The mix of a primitive's attribute rows r by a pixel's gates g (np_tile_kernels.cu:6037-6070).
template <int SLOTS>
__device__ __forceinline__ float feat_mix(const float r[SLOTS], float g0, float g1, float g2, float g3) {
  if constexpr (SLOTS == 1) return r[0];
  constexpr int k = SLOTS == 5 ? 1 : 0;
  float m = SLOTS == 5 ? fmaf(g0, r[k], r[0]) : fmaf(g0, r[k], 0.f);
  m = fmaf(g1, r[k + 1], m);
  m = fmaf(g2, r[k + 2], m);
  return fmaf(g3, r[k + 3], m);
}

// SLOTS = 1, 4 or 5.  PX: pixels per wavefront, 16 or 32; 64 / PX wavefronts share
// 128 channels.  Bound by latency and, with wave-uniform weights and gates (an operand out of a scalar register costs an
// instruction twice its time), by the two to ten operations per hit and 64 channels.
// Few pixels per wavefront mean more wavefronts (all four of a block have channels at 128 already) on smaller
// accumulators (58 to 73 registers at 16 pixels, 150 at 64), at the price of fetching the rows 64 / PX times.
// 333x251, 30,000 primitives, 67 channels: 433 us with 64 pixels and one slot fetch per record, 187 us with 16.
// Fetching the next record's rows ahead gained nothing at either size.
//
// HALVES: 64 channels or 128.  TAIL (64 channels, 16 pixels): the up to 4 TAIL channels behind them, with a lane's 4 TAIL-th of
// the wavefront for each of 16 / TAIL pixels at a time, TAIL times: the few channels of a ragged count then cost a few
// operations per hit and not as many as the first 64 (67 channels as above: 146 us; in the frame no channel count below 81
// is slower than with 128 of them reckoned, and 81 or more have no such form).
template <int SLOTS, int PX, int HALVES, int TAIL>
__global__ __launch_bounds__(256) void feat_accumulate_kernel(const float* __restrict__ feat_attr, int C, HitPool hp,
                                                              const int32_t* __restrict__ offsets, TileGeom g,
                                                              int waves_per_tile, float* __restrict__ out_feat) {
  static_assert(TAIL == 0 || (HALVES == 1 && PX == 16 && (TAIL == 1 || TAIL == 2 || TAIL == 4)), "a tail of up to 16 channels");
  constexpr int kShare = 64 / PX, kTailChannels = 4 * TAIL, kTailPixels = TAIL ? 16 / TAIL : 0;
  // (the render's mapping: what a tile's wavefront wrote lies in this XCD's L2)
  const int unit = (int)(blockIdx.x / kNumXcd), wslot = unit % waves_per_tile;
  const int tile = superblock_tile_of((int)(blockIdx.x % kNumXcd), unit / waves_per_tile, g.ntx, g.nty);
  if (tile < 0) return;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = threadIdx.x & 63;
  const int c0 = ((int)blockIdx.y * (4 / kShare) + wave / kShare) * 128, px0 = (wave % kShare) * PX;
  if (c0 >= C) return;
  const int hits = hp.item_hits[tile * waves_per_tile + wslot];
  const int table_base = wslot * hp.table_stride + (offsets[tile] >> 4) + tile;
  const int ca = c0 + l, cb = c0 + 64 + l;
  const bool has_a = ca < C, has_b = HALVES == 2 && cb < C;
  const int ct = c0 + 64 + (TAIL ? l % (TAIL ? kTailChannels : 1) : 0), tail_px = TAIL ? l / (TAIL ? kTailChannels : 1) : 0;
  const bool has_t = TAIL > 0 && ct < C;
  constexpr bool GATED = SLOTS > 1;

  float acc[PX][HALVES], tail[TAIL ? TAIL : 1];
#pragma unroll
  for (int px = 0; px < PX; ++px) {
#pragma unroll
    for (int h = 0; h < HALVES; ++h) acc[px][h] = 0.f;
  }
#pragma unroll
  for (int q = 0; q < TAIL; ++q) tail[q] = 0.f;

  int slots = 0, ids = 0;               // of 64 records, one per lane
  for (int m = 0; m < hits; ++m) {
    if ((m & 63) == 0) {
      slots = m + l < hits ? hit_slot(hp, table_base, m + l) : 0;
      ids = m + l < hits ? hp.hit_ids[slots] : 0;
    }
    const int rs = __builtin_amdgcn_readlane(slots, m & 63), p = __builtin_amdgcn_readlane(ids, m & 63);
    const float* __restrict__ rows = feat_attr + (size_t)p * SLOTS * C;
    float ra[SLOTS], rb[SLOTS], rt[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      ra[s] = has_a ? rows[(size_t)s * C + ca] : 0.f;
      rb[s] = has_b ? rows[(size_t)s * C + cb] : 0.f;
      rt[s] = has_t ? rows[(size_t)s * C + ct] : 0.f;
    }
    const float* __restrict__ rec = reinterpret_cast<const float*>(hp.records + (size_t)rs * hp.record_bytes) + px0;
    float wt[TAIL ? TAIL : 1], gt[TAIL ? TAIL : 1][4];
#pragma unroll
    for (int q = 0; q < TAIL; ++q) {
      const int px = q * kTailPixels + tail_px;
      wt[q] = rec[px];
#pragma unroll
      for (int k = 0; k < 4; ++k) gt[q][k] = GATED ? rec[64 * (k + 1) + px] : 0.f;
    }
    // weights and gates of 8 pixels at a time: wave-uniform 32-byte scalar loads, issued unconditionally
    // so that their latency overlaps the previous group's arithmetic
#pragma unroll
    for (int q = 0; q < PX / 8; ++q) {
      const f32x8 w8 = *reinterpret_cast<const f32x8*>(rec + 8 * q);
      f32x8 g8[4];
      if constexpr (GATED) {
#pragma unroll
        for (int k = 0; k < 4; ++k) g8[k] = *reinterpret_cast<const f32x8*>(rec + 64 * (k + 1) + 8 * q);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int px = 8 * q + j;
        const float w = w8[j];
        if (w >= 0.f) {
          acc[px][0] = fmaf(w, feat_mix<SLOTS>(ra, g8[0][j], g8[1][j], g8[2][j], g8[3][j]), acc[px][0]);
          if constexpr (HALVES == 2)
            acc[px][1] = fmaf(w, feat_mix<SLOTS>(rb, g8[0][j], g8[1][j], g8[2][j], g8[3][j]), acc[px][1]);
        }
      }
    }
#pragma unroll
    for (int q = 0; q < TAIL; ++q) {
      const float v = fmaf(wt[q], feat_mix<SLOTS>(rt, gt[q][0], gt[q][1], gt[q][2], gt[q][3]), tail[q]);
      tail[q] = wt[q] >= 0.f ? v : tail[q];
    }
  }

  const int tx = tile % g.ntx, ty = tile / g.ntx;
  const auto row = [&](int px) -> float* {          // a pixel's row of the image, null outside
    const int slot = wslot * 64 + px0 + px;
    const int x = tx * g.TW + slot % g.TW, y = ty * g.TH + slot / g.TW;
    return slot < g.TW * g.TH && x < g.W && y < g.H ? out_feat + (size_t)(y * g.W + x) * C : nullptr;
  };
#pragma unroll
  for (int px = 0; px < PX; ++px) {
    if (float* __restrict__ dst = row(px)) {
      if (has_a) dst[ca] = acc[px][0];
      if constexpr (HALVES == 2) {
        if (has_b) dst[cb] = acc[px][1];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < TAIL; ++q) {
    float* __restrict__ dst = row(q * kTailPixels + tail_px);
    if (dst && has_t) dst[ct] = tail[q];
  }
}

}  // namespace mlpsp

using namespace mlpsp;

MLPSP_API size_t mlpsp_feat_workspace_bytes(int64_t num_pairs, int width, int height, int tile_w, int tile_h,
                                            int feat_slots, int fp16_records, int64_t pool_records) {
  const int64_t T = checked_num_tiles(width, height, tile_w, tile_h);
  const int64_t tile_px = (int64_t)tile_w * tile_h;
  if (T <= 0 || tile_px <= 0 || tile_px > 256 || num_pairs < 0 || !(feat_slots == 1 || feat_slots == 4 || feat_slots == 5))
    return 0;
  const int wpt = (int)((tile_px + 63) / 64);
  const int rec = fp16_records ? 64 * 2 * (feat_slots == 5 ? 8 : 4) : 64 * 4 * (feat_slots > 1 ? 5 : 1);
  // every wavefront draws records 64 at a time: its last draw can stay 63 short of full
  const int64_t worst = num_pairs * wpt + (int64_t)(kHitChunk * kHitGrab - 1) * T * wpt + kHitChunk * kHitGrab;
  if (pool_records < 0 || pool_records > worst) pool_records = worst;
  return hitpool_bytes(num_pairs, T, wpt, pool_records, rec);
}

MLPSP_API int mlpsp_render_tilecenter_feat_f32(
    const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev, const int32_t* order_dev,
    const int32_t* tile_offsets_dev, const float* freq_dev, const float* att_dev, int num_frequencies,
    const float* W1, const float* b1, const float* W2, const float* b2, const float* W3, const float* b3,
    int num_primitives, int hidden, const float* feat_attr_dev, int feat_slots, int feat_channels, float gating_beta,
    float gating_temp, int width, int height, int tile_w, int tile_h, float threshold, int64_t num_pairs,
    void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev, float* out_alpha_dev, float* out_feat_dev,
    int32_t* status_dev, mlpsp_stream_t stream) {
  const int64_t T = checked_num_tiles(width, height, tile_w, tile_h);
  if (T <= 0) return MLPSP_E_ARGUMENT;
  const int64_t tile_px = (int64_t)tile_w * tile_h;
  if (tile_px <= 0 || tile_px > 256) return MLPSP_E_ARGUMENT;
  if (num_frequencies <= 0 || num_frequencies > 16 || hidden <= 0 || hidden > 64 || num_primitives < 0)
    return MLPSP_E_ARGUMENT;
  if (!(feat_slots == 1 || feat_slots == 4 || feat_slots == 5) || feat_channels <= 0 || feat_channels > 512)
    return MLPSP_E_ARGUMENT;
  if (!rays_o_dev || !rays_d_dev || !tile_offsets_dev || !out_rgb_dev || !out_alpha_dev || !out_feat_dev ||
      !status_dev || num_pairs < 0 || num_pairs > 2147483647LL)
    return MLPSP_E_ARGUMENT;
  if (num_primitives > 0 && !feat_attr_dev) return MLPSP_E_ARGUMENT;
  const int wpt = (int)((tile_px + 63) / 64);
  const int64_t items = T * wpt;
  if (items > 2147483647LL - 8) return MLPSP_E_ARGUMENT;
  if (!workspace_dev || reinterpret_cast<uintptr_t>(workspace_dev) % 256 != 0 ||
      workspace_bytes < hitpool_min_bytes(num_pairs, T, wpt))
    return MLPSP_E_SCRATCH;
  const int rec_bytes = 64 * 4 * (feat_slots > 1 ? 5 : 1);
  const HitPool hp = hitpool_carve(workspace_dev, workspace_bytes, num_pairs, T, wpt, rec_bytes);
  hipStream_t s = (hipStream_t)stream;
  MLPSP_HIP_TRY(clear_async(hp.counters, 64 * sizeof(int32_t), s));
  const int per_xcd = (int)((items + kNumXcd - 1) / kNumXcd);
  TileGeom g{width, height, tile_w, tile_h, ceil_div(width, tile_w), ceil_div(height, tile_h)};
  const dim3 grid((unsigned)(per_xcd * kNumXcd)), block(64);
#define MLPSP_EMIT_LAUNCH(HT, FT, EM, ...)                                                                        \
  hipLaunchKernelGGL((render_tilecenter_f32_kernel<HT, FT, EM, ##__VA_ARGS__>), grid, block, 0, s, rays_o_dev, rays_d_dev,       \
                     (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev,         \
                     num_frequencies, W1, b1, W2, b2, W3, b3, num_primitives, hidden, g, wpt, per_xcd, (int)items, threshold,          \
                     out_rgb_dev, out_alpha_dev, (float*)nullptr, (unsigned long long*)nullptr, gating_beta,      \
                     gating_temp, hp)
#define MLPSP_EMIT_ARGS                                                                                           \
  rays_o_dev, rays_d_dev, (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev, W1, b1, W2, \
      b2, W3, b3, num_primitives, g, wpt, threshold, out_rgb_dev, out_alpha_dev, (float*)nullptr,                   \
      (unsigned long long*)nullptr, gating_beta, gating_temp, hp
#define MLPSP_EMIT_TEAM(EM, TEAM)                                                                                   \
  hipLaunchKernelGGL((render_team_f32_kernel<32, EM, TEAM>), dim3(plan.grid), dim3(64 * TEAM), 0, s, MLPSP_EMIT_ARGS)
#define MLPSP_EMIT_GO(EM)                                                                                         \
  do {                                                                                                            \
    if (plan.team == 12) MLPSP_EMIT_TEAM(EM, 12);                                                                 \
    else if (plan.team == 8) MLPSP_EMIT_TEAM(EM, 8);                                                              \
    else                                                                                                          \
      hipLaunchKernelGGL((render_mixed_f32_kernel<32, EM>), dim3(plan.grid), dim3(256), 0, s, MLPSP_EMIT_ARGS, plan.body); \
  } while (0)
  const bool gated = feat_slots > 1;
  if (hidden == 32 && use_mfma32(hidden, num_frequencies, W1, b1, W2, b2)) {
    const PlanF32 plan = plan_f32(g, wpt, items, true);
    if (gated) MLPSP_EMIT_GO(2);
    else MLPSP_EMIT_GO(1);
  } else if (hidden == 32 && num_frequencies == 6) {
    if (gated) MLPSP_EMIT_LAUNCH(32, 6, 2);
    else MLPSP_EMIT_LAUNCH(32, 6, 1);
  } else {
    if (gated) MLPSP_EMIT_LAUNCH(0, 0, 2);
    else MLPSP_EMIT_LAUNCH(0, 0, 1);
  }
#undef MLPSP_EMIT_GO
#undef MLPSP_EMIT_TEAM
#undef MLPSP_EMIT_ARGS
#undef MLPSP_EMIT_LAUNCH
  MLPSP_LAUNCH_CHECK();
#define MLPSP_ACC_LAUNCH(SL, PX, HALVES, TAIL)                                                                      \
  hipLaunchKernelGGL((feat_accumulate_kernel<SL, PX, HALVES, TAIL>), dim3(superblock_grid(g.ntx, g.nty) * (unsigned)wpt,            \
                     (unsigned)ceil_div(feat_channels, 8 * PX)), dim3(256), 0, s, feat_attr_dev, feat_channels, hp,   \
                     tile_offsets_dev, g, wpt, out_feat_dev)
  // 16 pixels per wavefront unless the rows are long and the launch fills the chip anyway: four times the wavefronts for
  // four times the row fetches.  Render and product in us with 16 / 32 pixels (runs differ by about 1 %):
  //    items   64 channels      128           192           256           384           512
  //    1,200   1,019 / 1,111  1,010 / 1,109  1,114 / 1,134  1,108 / 1,137  1,203 / 1,287  1,304 / 1,342
  //    2,640   1,428 / 1,537  1,441 / 1,545  1,637 / 1,673  1,651 / 1,693  1,869 / 1,948  2,083 / 2,085
  //    3,500   1,821 / 1,928  1,821 / 1,927  2,118 / 2,132  2,103 / 2,134  2,438 / 2,496  2,741 / 2,659
  //    4,800   2,360 / 2,525  2,417 / 2,552  2,815 / 2,775  2,812 / 2,778  3,268 / 3,329  3,713 / 3,560
  //    8,190   3,569 / 3,763  3,542 / 3,759  4,337 / 4,135  4,321 / 4,153  5,078 / 5,051  5,764 / 5,439
  //   12,750   5,408 / 5,678  5,464 / 5,659  6,602 / 6,404  6,667 / 6,380  7,847 / 7,722  8,970 / 8,389
  // (384 channels are one and a half of the 256 that a workgroup of 32-pixel wavefronts takes.)
  const bool sixteen = feat_channels <= 128 || items <= 3072;
  // Up to 80 channels reckon only those that there are (in fours behind the 64th).  Whole frame of 333x251 and 30,000
  // primitives in us, 128 channels reckoned / as here (96 channels, the same kernel on both sides: 962 / 962):
  //    16 channels   957 / 914      40   960 / 909      64   959 / 915      67   961 / 922      72   960 / 926      80   960 / 930
  //    800x640 and 100,000:  33   3,506 / 3,452      70   3,510 / 3,314
  // Above, 32 channels behind the 64th, two pixels at a time, are no faster than 64: 84, 88 and 96 channels 1,136 / 1,150, 1,141 /
  // 1,160 and 1,141 / 1,146 at 30,000 primitives, 3,556 / 3,611, 3,544 / 3,617 and 3,565 / 3,615 at 100,000.
#define MLPSP_ACC_GO(SL)                                          \
  do {                                                            \
    if (!sixteen) MLPSP_ACC_LAUNCH(SL, 32, 2, 0);                 \
    else if (feat_channels <= 64) MLPSP_ACC_LAUNCH(SL, 16, 1, 0); \
    else if (feat_channels <= 68) MLPSP_ACC_LAUNCH(SL, 16, 1, 1); \
    else if (feat_channels <= 72) MLPSP_ACC_LAUNCH(SL, 16, 1, 2); \
    else if (feat_channels <= 80) MLPSP_ACC_LAUNCH(SL, 16, 1, 4); \
    else MLPSP_ACC_LAUNCH(SL, 16, 2, 0);                          \
  } while (0)
  if (feat_slots == 4) MLPSP_ACC_GO(4);
  else if (feat_slots == 5) MLPSP_ACC_GO(5);
  else MLPSP_ACC_GO(1);
#undef MLPSP_ACC_GO
#undef MLPSP_ACC_LAUNCH
  MLPSP_LAUNCH_CHECK();
  // status_dev[0] = 1 if the record pool was too small (the feature image is then incomplete)
  MLPSP_HIP_TRY(hipMemcpyAsync(status_dev, hp.counters + 1, sizeof(int32_t), hipMemcpyDeviceToDevice, s));
  return MLPSP_OK;
}
