// The scalar-f32 tile-centre render kernel (shared by the RGB entry point and the feature entry point,
// which asks it to emit hit records).
#pragma once
#include <cstdlib>
#include "mlpsp_device.hpp"
#include "mlpsp_hitrec.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mlp.hpp"
#include "mlpsp_mlp_mfma32.hpp"
#include "mlpsp_team.hpp"
#include "mlpsp_walk_f32.hpp"

namespace mlpsp {

// EMIT = 0: image only.  EMIT = 1 / 2: also emit one hit record per primitive that hits a pixel of this
// wavefront, float[K][64] with K = 1 (the compositing weight w) / K = 5 (w and the four tetrahedral
// gates); w = -1 marks a pixel the primitive did not hit (weights are never negative).
//
// STATS: also accumulate the pruning statistics of np_tile_kernels.cu:2139-2519: per processed primitive
// the wavefront reduces over its pixels  w,  max w,  [w > 1e-8],  [w > 0.1] * w * err  and  [w > 0.1]
// (err = L1 colour error of the pixel after this blend step against gt_rgb) and adds them to the five
// per-primitive buffers with atomics, as the reference does per block (:2435-2456).
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) v += __shfl_xor(v, d);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) v = fmaxf(v, __shfl_xor(v, d));
  return v;
}

// This kernel evaluates the MLP on the vector ALU (shapes and alignments the matrix-core kernel below does not take).
template <int HT, int FT, int EMIT, bool STATS = false>
__global__ __launch_bounds__(64) void render_tilecenter_f32_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, int F, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, int H, TileGeom g, int waves_per_tile, int per_xcd,
    int num_items, float thr, float* __restrict__ out_rgb, float* __restrict__ out_alpha, float* __restrict__ out_t,
    unsigned long long* __restrict__ counters, float beta, float temp, HitPool hp,
    const float* __restrict__ gt_rgb = nullptr, float* __restrict__ stat_sum_w = nullptr,
    float* __restrict__ stat_max_w = nullptr, int32_t* __restrict__ stat_hits = nullptr,
    float* __restrict__ stat_sum_werr = nullptr, int32_t* __restrict__ stat_contrib = nullptr) {
  // The weight pointers are separate __restrict__ parameters (not a struct): only then does the compiler
  // know that the record stores below cannot alias them and keeps fetching weights with scalar loads.
  const MlpPtrs mlp{W1, b1, W2, b2, W3, b3};
  // XCD-aware work assignment: XCD k (blockIdx.x % 8) walks items [k*per_xcd, (k+1)*per_xcd).
  const int item = (blockIdx.x % kNumXcd) * per_xcd + blockIdx.x / kNumXcd;
  if (item >= num_items) return;
  const int tile = item / waves_per_tile, wslot = item % waves_per_tile;
  const int slot = wslot * 64 + threadIdx.x;
  const int tx = tile % g.ntx, ty = tile / g.ntx;
  const int lx = slot % g.TW, ly = slot / g.TW;
  const int x = tx * g.TW + lx, y = ty * g.TH + ly;
  const bool valid = (slot < g.TW * g.TH) && (x < g.W) && (y < g.H);
  const int pix = valid ? (y * g.W + x) : 0;

  const float rox = valid ? rays_o[pix * 3 + 0] : 0.f;
  const float roy = valid ? rays_o[pix * 3 + 1] : 0.f;
  const float roz = valid ? rays_o[pix * 3 + 2] : 0.f;
  const float rdx = valid ? rays_d[pix * 3 + 0] : 0.f;
  const float rdy = valid ? rays_d[pix * 3 + 1] : 0.f;
  const float rdz = valid ? rays_d[pix * 3 + 2] : 0.f;

  const int start = offsets[tile];
  const int end = offsets[tile + 1];

  PixelAcc acc = {0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
  unsigned n_proc = 0, n_proc_hit = 0, n_hits = 0;
  float gtr = 0.f, gtg = 0.f, gtb = 0.f;
  if constexpr (STATS) {
    if (valid) {
      gtr = gt_rgb[pix * 3 + 0];
      gtg = gt_rgb[pix * 3 + 1];
      gtb = gt_rgb[pix * 3 + 2];
    }
  }
  HitEmitter em = hit_emitter_begin(hp, wslot, start, tile);

  for (int i = start; i < end; ++i) {
    const int p = __builtin_amdgcn_readfirstlane(order[i]);
    if (p < 0 || p >= N) continue;
    const PrimRecord P = prims[p];
    HitInfo h;
    const bool live = valid && (acc.trans >= kTransmittanceFloor);
    const bool hit = live && hit_rot(rox, roy, roz, rdx, rdy, rdz, P, thr, h);
    const unsigned long long hit_mask = __ballot(hit);
    ++n_proc;
    if (hit_mask != 0ull) {
      ++n_proc_hit;
      n_hits += __popcll(hit_mask);
      int rs = -1;
      float w_stat = 0.f;
      if constexpr (EMIT > 0) rs = hit_emitter_next(hp, em, (int)threadIdx.x);
      float* __restrict__ rec = reinterpret_cast<float*>(hp.records + (size_t)(rs < 0 ? 0 : rs) * hp.record_bytes);
      const float x6[6] = {rdx, rdy, rdz, h.dx, h.dy, h.dz};
      float o[4];
      if (hit) {
        mlp_eval<HT, FT>(x6, freq, att, F, H, mlp, p, o);
        const float w = blend_step(acc, o[0], o[1], o[2], o[3], h.decay, h.t);
        w_stat = w;
        if constexpr (EMIT > 0) {
          if (rs >= 0) {
            rec[threadIdx.x] = w;
            if constexpr (EMIT > 1) {
              float gt[4];
              tetra_gates(h.qlx, h.qly, h.qlz, P.lgx, P.lgy, P.lgz, beta, temp, gt);
#pragma unroll
              for (int k = 0; k < 4; ++k) rec[(k + 1) * 64 + threadIdx.x] = gt[k];
            }
          }
        }
      } else if constexpr (EMIT > 0) {
        if (rs >= 0) rec[threadIdx.x] = -1.f;       // the gates of a missed pixel are never read
      }
      if constexpr (EMIT > 0) {
        if (rs >= 0 && threadIdx.x == 0) hp.hit_ids[rs] = p;
      }
      if constexpr (STATS) {
        const float lw = hit ? w_stat : 0.f;
        const bool contrib = hit && (lw > 1e-1f);
        float lerr = 0.f;
        if (contrib) lerr = lw * ((fabsf(acc.cr - gtr) + fabsf(acc.cg - gtg)) + fabsf(acc.cb - gtb));
        const float s_w = wave_sum(lw), m_w = wave_max(lw), s_err = wave_sum(lerr);
        const int n_hit = __popcll(__ballot(hit && (lw > 1e-8f))), n_con = __popcll(__ballot(contrib));
        if (threadIdx.x == 0) {
          atomicAdd(stat_sum_w + p, s_w);
          atomicMax(reinterpret_cast<int*>(stat_max_w + p), __float_as_int(m_w));   // weights are >= 0
          atomicAdd(stat_hits + p, n_hit);
          if (stat_sum_werr) atomicAdd(stat_sum_werr + p, s_err);
          if (stat_contrib) atomicAdd(stat_contrib + p, n_con);
        }
      }
    }
    if (__ballot(valid && (acc.trans >= kTransmittanceFloor)) == 0ull) break;
  }

  if (valid) {
    out_rgb[pix * 3 + 0] = acc.cr;
    out_rgb[pix * 3 + 1] = acc.cg;
    out_rgb[pix * 3 + 2] = acc.cb;
    out_alpha[pix] = 1.f - acc.trans;
    if (out_t) out_t[pix] = acc.t_acc / (acc.w_acc > 1e-8f ? acc.w_acc : 1.f);
  }
  if constexpr (EMIT > 0) {
    if (threadIdx.x == 0) hp.item_hits[item] = em.count;
  }
  if (counters && threadIdx.x == 0) {
    atomicAdd(counters + 1, (unsigned long long)n_proc);
    atomicAdd(counters + 2, (unsigned long long)n_proc_hit);
    atomicAdd(counters + 3, (unsigned long long)n_hits);
  }
}

// The 72->{32,16}->{32,16}->4 MLP of a hit on the matrix cores for all 64 pixels at once (mlp_wave_mfma32, same bits);
// needs 16-byte aligned weight arrays.
//
// What bounds it: v_mfma_f32_32x32x2 and vector instructions do NOT run beside one another on this chip, neither in one
// wavefront nor across the wavefronts of a SIMD (a probe of four wavefronts per SIMD: 8 MFMAs 516 clocks, 64
// independent FMAs 183, the two interleaved 691), so a hit step costs the sum: 104 x 64 clocks of matrix work plus 2.9
// for every vector instruction, and every instruction removed shows: the walk of mlpsp_walk_f32.hpp, sin/cos pairs without
// their range selects, a one-instruction ReLU (1,575 -> 1,360 vector instructions per hit step, 106 of them MFMAs) and
// super-blocks of tiles dealt to the XCDs instead of bands of image rows took the 200,000-primitive 1200x680 frame from 4.33 to 3.93
// ms and a 30,000-primitive 333x251 feature frame from 1.77 to 1.47.  The sum is 10,400 of the 13,500 clocks that a hit step
// takes; the rest are waits of the three wavefronts per SIMD: four would need 10 KB of LDS per wavefront, and two less
// registers, and measured within 1 % of three.
struct ItemF32Lds {
  DirOperands dir;
  WalkLds walk;
};
struct StatsF32 {
  const float* gt_rgb;
  float *sum_w, *max_w;
  int32_t* hits;
  float* sum_werr;
  int32_t* contrib;
};
template <int HT, int EMIT, bool STATS>
__device__ __forceinline__ void render_item_f32(
    const int tile, const int wslot, const int lane, ItemF32Lds& lds,
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, TileGeom g, int waves_per_tile, float thr, float* __restrict__ out_rgb,
    float* __restrict__ out_alpha, float* __restrict__ out_t, unsigned long long* __restrict__ counters, float beta,
    float temp, HitPool hp, const StatsF32& stats) {
  DirOperands& s_dir = lds.dir;
  WalkLds& s_walk = lds.walk;
  const int slot = wslot * 64 + lane;
  const int tx = tile % g.ntx, ty = tile / g.ntx;
  const int x = tx * g.TW + slot % g.TW, y = ty * g.TH + slot / g.TW;
  const bool valid = (slot < g.TW * g.TH) && (x < g.W) && (y < g.H);
  const int pix = valid ? (y * g.W + x) : 0;
  const Float3 ro = valid ? load3(rays_o, pix) : Float3{0.f, 0.f, 0.f}, rd = valid ? load3(rays_d, pix) : Float3{0.f, 0.f, 0.f};
  const int start = offsets[tile], end = offsets[tile + 1];

  PixelAcc acc = {0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
  unsigned n_proc = 0, n_proc_hit = 0, n_hits = 0;
  Float3 gt = {0.f, 0.f, 0.f};
  if constexpr (STATS) {
    if (valid) gt = load3(stats.gt_rgb, pix);
  }
  HitEmitter em = hit_emitter_begin(hp, wslot, start, tile);
  encode_direction<HT>(rd.x, rd.y, rd.z, freq, att, s_dir);

  walk_tile_f32(
      order, start, end, N, prims, valid, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, thr, s_walk,
      [&]() { return valid && (acc.trans >= kTransmittanceFloor); },
      [&](int p, bool hit, const HitInfo& h, unsigned long long mask) {
        ++n_proc;
        if (mask == 0ull) return true;
        ++n_proc_hit;
        n_hits += __popcll(mask);
        int rs = -1;
        if constexpr (EMIT > 0) rs = hit_emitter_next(hp, em, lane);
        // (lanes that did not hit carry no hit point; the matrix-core evaluation runs on all 64 lanes)
        const float x6[6] = {rd.x, rd.y, rd.z, hit ? h.dx : 0.f, hit ? h.dy : 0.f, hit ? h.dz : 0.f};
        float o[4];
        mlp_wave_mfma32<false, false, HT>(x6, freq, att, W1, b1, W2, b2, W3, b3, p, s_dir, o);
        float w = 0.f;
        if (hit) w = blend_step(acc, o[0], o[1], o[2], o[3], h.decay, h.t);
        if constexpr (EMIT > 0) {
          if (rs >= 0) {
            float* __restrict__ rec = reinterpret_cast<float*>(hp.records + (size_t)rs * hp.record_bytes);
            rec[lane] = hit ? w : -1.f;
            if constexpr (EMIT > 1) {
              if (hit) {          // the gates of a missed pixel are never read
                const PrimRecord& P = prims[p];
                float gates[4];
                tetra_gates(h.qlx, h.qly, h.qlz, P.lgx, P.lgy, P.lgz, beta, temp, gates);
#pragma unroll
                for (int k = 0; k < 4; ++k) rec[(k + 1) * 64 + lane] = gates[k];
              }
            }
            if (lane == 0) hp.hit_ids[rs] = p;
          }
        }
        if constexpr (STATS) {
          const bool contrib = hit && (w > 1e-1f);
          float lerr = 0.f;
          if (contrib) lerr = w * ((fabsf(acc.cr - gt.x) + fabsf(acc.cg - gt.y)) + fabsf(acc.cb - gt.z));
          const float s_w = wave_sum(w), m_w = wave_max(w), s_err = wave_sum(lerr);
          const int n_hit = __popcll(__ballot(hit && (w > 1e-8f))), n_con = __popcll(__ballot(contrib));
          if (lane == 0) {
            atomicAdd(stats.sum_w + p, s_w);
            atomicMax(reinterpret_cast<int*>(stats.max_w + p), __float_as_int(m_w));   // weights are >= 0
            atomicAdd(stats.hits + p, n_hit);
            if (stats.sum_werr) atomicAdd(stats.sum_werr + p, s_err);
            if (stats.contrib) atomicAdd(stats.contrib + p, n_con);
          }
        }
        return __ballot(valid && (acc.trans >= kTransmittanceFloor)) != 0ull;
      });

  if (valid) {
    store3(out_rgb, pix, acc.cr, acc.cg, acc.cb);
    out_alpha[pix] = 1.f - acc.trans;
    if (out_t) out_t[pix] = acc.t_acc / (acc.w_acc > 1e-8f ? acc.w_acc : 1.f);
  }
  if constexpr (EMIT > 0) {
    if (lane == 0) hp.item_hits[tile * waves_per_tile + wslot] = em.count;
  }
  if (counters && lane == 0) {
    atomicAdd(counters + 1, (unsigned long long)n_proc);
    atomicAdd(counters + 2, (unsigned long long)n_proc_hit);
    atomicAdd(counters + 3, (unsigned long long)n_hits);
  }
}
// The pruning statistics beside the image: one wavefront per item.
template <int HT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 3))) void render_stats_f32_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, TileGeom g, int waves_per_tile, float thr, float* __restrict__ out_rgb,
    float* __restrict__ out_alpha, float* __restrict__ out_t, unsigned long long* __restrict__ counters, float beta,
    float temp, HitPool hp, StatsF32 stats) {
  __shared__ ItemF32Lds s;
  const int unit = (int)(blockIdx.x / kNumXcd);
  const int tile = superblock_tile_of((int)(blockIdx.x % kNumXcd), unit / waves_per_tile, g.ntx, g.nty);
  if (tile < 0) return;
  render_item_f32<HT, 0, true>(tile, unit % waves_per_tile, (int)threadIdx.x, s, rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, N, g, waves_per_tile, thr, out_rgb, out_alpha, out_t, counters,
      beta, temp, hp, stats);
}

// The same item by a team of wavefronts (mlpsp_team.hpp).  Wavefront 0 adds up image and depth, in list order and with the
// roundings of the single wavefront; each wavefront writes the record of its own entry.
template <int TEAM>
struct TeamF32Lds {
  DirOperands dir;
  TeamWalkLds<TEAM> walk;
  float pay[2][TEAM][5][64];        // opacity, colour, ray parameter
  int chunk;
};
template <int HT, int EMIT, int TEAM>
__device__ __forceinline__ void render_team_item_f32(
    const int tile, const int wslot, const int k, const int lane, TeamF32Lds<TEAM>& s,
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, TileGeom g, int waves_per_tile, float thr, float* __restrict__ out_rgb,
    float* __restrict__ out_alpha, float* __restrict__ out_t, unsigned long long* __restrict__ counters, float beta,
    float temp, HitPool hp) {
  const int slot = wslot * 64 + lane;
  const int tx = tile % g.ntx, ty = tile / g.ntx;
  const int x = tx * g.TW + slot % g.TW, y = ty * g.TH + slot / g.TW;
  const bool valid = (slot < g.TW * g.TH) && (x < g.W) && (y < g.H);
  const int pix = valid ? (y * g.W + x) : 0;
  const Float3 ro = valid ? load3(rays_o, pix) : Float3{0.f, 0.f, 0.f}, rd = valid ? load3(rays_d, pix) : Float3{0.f, 0.f, 0.f};
  const int start = offsets[tile], end = offsets[tile + 1];
  PixelAcc acc = {0.f, 0.f, 0.f, 1.f, 0.f, 0.f};
  unsigned n_proc = 0, n_proc_hit = 0, n_hits = 0;
  TeamSlots slots{wslot * hp.table_stride + (start >> 4) + tile, 0, 0, 0, 0};
  if (k == 0) encode_direction<HT>(rd.x, rd.y, rd.z, freq, att, s.dir);

  int p_mine = 0;
  float gates[4];
  walk_team_f32<TEAM>(
      order, start, end, N, prims, valid, ro.x, ro.y, ro.z, rd.x, rd.y, rd.z, thr, s.walk, k, lane,
      [&]() { return valid && (acc.trans >= kTransmittanceFloor); },
      [&](int p, bool hit, const HitInfo& h, unsigned long long, int buf) {
        p_mine = p;
        const float x6[6] = {rd.x, rd.y, rd.z, hit ? h.dx : 0.f, hit ? h.dy : 0.f, hit ? h.dz : 0.f};
        float o[4];
        mlp_wave_mfma32<false, false, HT>(x6, freq, att, W1, b1, W2, b2, W3, b3, p, s.dir, o);
        float(&pay)[5][64] = s.pay[buf][k];
        if (hit) {
          const float sigma = softplus(o[3]) * h.decay;
          pay[0][lane] = 1.f - det_exp(-sigma);
          pay[1][lane] = sigmoid(o[0]);
          pay[2][lane] = sigmoid(o[1]);
          pay[3][lane] = sigmoid(o[2]);
          pay[4][lane] = h.t;
          if constexpr (EMIT > 1) {
            const PrimRecord& P = prims[p];
            tetra_gates(h.qlx, h.qly, h.qlz, P.lgx, P.lgy, P.lgz, beta, temp, gates);
          }
        }
      },
      [&](const unsigned long long* masks, int entries, int buf) {
        int kept = 0, mine = -1;
        float w_mine = -1.f;
#pragma unroll
        for (int i = 0; i < TEAM; ++i) {
          if (i == k && i < entries) n_proc += __ballot(valid && acc.trans >= kTransmittanceFloor) != 0ull;
          const unsigned long long m = masks[i];
          const unsigned long long um = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)m) |
                                        ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(m >> 32)) << 32);
          if (um == 0ull) continue;
          const bool hit = ((um >> lane) & 1ull) && (acc.trans >= kTransmittanceFloor);
          const unsigned long long blended = __ballot(hit);
          if (blended == 0ull) continue;           // (behind the last entry that counts)
          const float(&pay)[5][64] = s.pay[buf][i];
          const float alpha = pay[0][lane], w = acc.trans * alpha;
          if (i == k) {
            ++n_proc_hit;
            n_hits += __popcll(blended);
            mine = kept;
            w_mine = hit ? w : -1.f;
          }
          ++kept;
          if (hit) {
            if (k == 0) {
              acc.w_acc = fmaf(1.f, w, acc.w_acc);
              acc.t_acc = fmaf(w, pay[4][lane], acc.t_acc);
              acc.cr = fmaf(w, pay[1][lane], acc.cr);
              acc.cg = fmaf(w, pay[2][lane], acc.cg);
              acc.cb = fmaf(w, pay[3][lane], acc.cb);
            }
            acc.trans = acc.trans * (1.f - alpha);
          }
        }
        if constexpr (EMIT > 0) {
          const int rs = team_slot<HitGroups, true>(slots, kept, mine, k, lane, hp.counters, hp.chunk_table, hp.pool_chunks, s.chunk);
          if (rs >= 0) {
            float* __restrict__ rec = reinterpret_cast<float*>(hp.records + (size_t)rs * hp.record_bytes);
            rec[lane] = w_mine;
            if constexpr (EMIT > 1) {
              if (w_mine >= 0.f) {          // the gates of a missed pixel are never read
#pragma unroll
                for (int c = 0; c < 4; ++c) rec[(c + 1) * 64 + lane] = gates[c];
              }
            }
            if (lane == 0) hp.hit_ids[rs] = p_mine;
          }
        }
        return __ballot(valid && (acc.trans >= kTransmittanceFloor)) != 0ull;
      });

  if (k == 0 && valid) {
    store3(out_rgb, pix, acc.cr, acc.cg, acc.cb);
    out_alpha[pix] = 1.f - acc.trans;
    if (out_t) out_t[pix] = acc.t_acc / (acc.w_acc > 1e-8f ? acc.w_acc : 1.f);
  }
  if constexpr (EMIT > 0) {
    if (k == 0 && lane == 0) hp.item_hits[tile * waves_per_tile + wslot] = slots.count;
  }
  if (counters && lane == 0) {
    atomicAdd(counters + 1, (unsigned long long)n_proc);
    atomicAdd(counters + 2, (unsigned long long)n_proc_hit);
    atomicAdd(counters + 3, (unsigned long long)n_hits);
  }
}

// Every item by a team.  Twelve wavefronts: three on a SIMD, as many as a workgroup of that size leaves room for.  Four and eight:
// four on a SIMD, 128 registers (EMIT 0: at most twelve bytes spilled), 34 KB of LDS and less.
constexpr int team_waves_per_simd(int team) { return team == 12 ? 3 : 4; }
template <int HT, int EMIT, int TEAM>
__global__ __launch_bounds__(64 * TEAM) __attribute__((amdgpu_waves_per_eu(team_waves_per_simd(TEAM), team_waves_per_simd(TEAM)))) void render_team_f32_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, TileGeom g, int waves_per_tile, float thr, float* __restrict__ out_rgb,
    float* __restrict__ out_alpha, float* __restrict__ out_t, unsigned long long* __restrict__ counters, float beta,
    float temp, HitPool hp) {
  __shared__ TeamF32Lds<TEAM> s;
  const int unit = (int)(blockIdx.x / kNumXcd);
  const int tile = superblock_tile_of((int)(blockIdx.x % kNumXcd), unit / waves_per_tile, g.ntx, g.nty);
  if (tile < 0) return;
  render_team_item_f32<HT, EMIT, TEAM>(tile, unit % waves_per_tile, __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6),
                                       (int)threadIdx.x & 63, s, rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, N, g, waves_per_tile, thr, out_rgb, out_alpha, out_t, counters,
      beta, temp, hp);
}

// A wavefront per item, four items to a workgroup, but for the last ones: the workgroups from `body` on (per XCD) take one
// item each, as a team.
template <int HT, int EMIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void render_mixed_f32_kernel(
    const float* __restrict__ rays_o, const float* __restrict__ rays_d, const PrimRecord* __restrict__ prims,
    const int32_t* __restrict__ order, const int32_t* __restrict__ offsets, const float* __restrict__ freq,
    const float* __restrict__ att, const float* __restrict__ W1, const float* __restrict__ b1,
    const float* __restrict__ W2, const float* __restrict__ b2, const float* __restrict__ W3,
    const float* __restrict__ b3, int N, TileGeom g, int waves_per_tile, float thr, float* __restrict__ out_rgb,
    float* __restrict__ out_alpha, float* __restrict__ out_t, unsigned long long* __restrict__ counters, float beta,
    float temp, HitPool hp, int body) {
  union Lds {
    ItemF32Lds item[4];
    TeamF32Lds<4> team;
  };
  __shared__ Lds s;
  const int unit = (int)(blockIdx.x / kNumXcd), xcd = (int)(blockIdx.x % kNumXcd);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
  const bool alone = unit < body;
  const int item = alone ? unit * 4 + wave : body * 4 + (unit - body);
  const int tile = superblock_tile_of(xcd, item / waves_per_tile, g.ntx, g.nty);
  if (tile < 0) return;
  if (alone)
    render_item_f32<HT, EMIT, false>(tile, item % waves_per_tile, lane, s.item[wave], rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, N, g, waves_per_tile, thr, out_rgb, out_alpha, out_t, counters,
      beta, temp, hp, StatsF32{});
  else
    render_team_item_f32<HT, EMIT, 4>(tile, item % waves_per_tile, wave, lane, s.team, rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, N, g, waves_per_tile, thr, out_rgb, out_alpha, out_t, counters,
      beta, temp, hp);
}

// Launch of `items` 64-pixel items on the matrix cores.  An evaluation keeps its SIMD's matrix core busy, so a team is a
// multiple of four, one wavefront on each SIMD of a CU (3 and 6 were slower than 4, 2 as well): twelve where the items are no more
// than the CUs; eight up to 640 items, two tiles to a CU and four wavefronts to a SIMD; four up to 1,920.  Above, the mixed kernel
// with a team for each of the last items, which shortens the tail of the launch: what is left when the queue is empty lasts a
// third as long.  With hit records the kernels of four wavefronts to a SIMD spill 44 bytes and more: the mixed kernel from
// 641 items on.  Whole frames in us (5,000 to 50,000 primitives; the mixed kernel's three wavefronts to a
// SIMD as teams throughout below 1,280 items, else with 1,024 teams):
//                 hidden 32                            hidden 16               hidden 32, feature image of 67 channels
//      items   twelve  eight  four  mixed   items   eight  four  mixed    items   twelve  eight  four  mixed
//        180     240    247    276     --     180     213   240     --      180     416    431   472     --
//        272     282    261    276    280     272     211   230    230      272     460    440   463    455
//        400     330    310    331    335     300     225   245    244      400     544    525   554    543
//        500     499    452    472    476     588     356   364    362      500     802    765   809    789
//        690     547    509    506    511     960     446   426    456      690   1,472  1,416 1,400  1,364
//      1,200     796    679    687    704   1,200     476   457    474    1,344   1,264  1,149 1,154  1,163
//      1,610     967    804    770    824   1,610     580   544    556    1,610   1,382  1,218 1,184  1,228
//      2,016   1,134    949    935    922   2,560     793   731    706    2,016   1,625  1,430 1,378  1,381
// How many of the last items: a CU that is ahead takes one more of them, and a wavefront's item lasts a millisecond of the four
// that 12,750 items take.  With a wavefront per item throughout 4,034 us; with teams for the last
//      items    1,024   1,536   2,048   2,560   3,072
//      2,560    1,032   1,022   1,051   1,066   1,064
//      4,860    1,780   1,733   1,765   1,799   1,809
//      8,000    2,525   2,452   2,473   2,470   2,506
//     12,750    3,971   3,965   3,919   3,927   3,962
//     30,000    8,206   8,219   8,235   8,245   8,281
// and with a feature image of 67 channels 1,523 / 1,492 / 1,507 at 2,560 items, 3,605 / 3,534 / 3,557 at 8,000.
// MLPSP_F32_AHEAD=0 / 1 / 2 in the environment: a wavefront per item throughout / four / twelve (comparison runs, tests).
struct PlanF32 {
  int team;          // wavefronts of the kernel that gives every item a team; 0: the mixed kernel
  int body;          // workgroups per XCD with an item per wavefront (mixed kernel)
  unsigned grid;
};
inline PlanF32 plan_f32(const TileGeom& g, int waves_per_tile, int64_t items, bool records) {
  const unsigned slots = superblock_grid(g.ntx, g.nty) * (unsigned)waves_per_tile;
  const char* e = getenv("MLPSP_F32_AHEAD");
  const int forced = e && e[0] >= '0' && e[0] <= '2' ? e[0] - '0' : -1;
  const int team = forced == 2 || (forced < 0 && items <= 256) ? 12
                   : forced < 0 && items <= 640               ? 8
                   : !records && (forced == 1 || (forced < 0 && items <= 1920)) ? 4 : 0;
  if (team != 0) return PlanF32{team, 0, slots};
  const int per_xcd = (int)(slots / kNumXcd);
  const int teams = forced == 0 ? 0 : forced == 1 ? per_xcd : min(per_xcd, (items <= 8192 ? 1536 : 2048) / kNumXcd);
  const int body = forced == 0 ? (per_xcd + 3) / 4 : (per_xcd - teams) / 4;
  return PlanF32{0, body, (unsigned)(kNumXcd * (body + max(0, per_xcd - 4 * body)))};
}

// Whether the matrix-core f32 evaluation applies: the 72->32->32->4 or 72->16->16->4 shape, weight arrays that can be
// read 16 bytes at a time, and no request for the scalar kernel (environment MLPSP_F32_SCALAR=1, which
// exists for comparison runs).
inline bool use_mfma32(int hidden, int num_frequencies, const float* W1, const float* b1, const float* W2,
                       const float* b2) {
  if ((hidden != 32 && hidden != 16) || num_frequencies != 6) return false;
  if (((uintptr_t)W1 | (uintptr_t)b1 | (uintptr_t)W2 | (uintptr_t)b2) & 15u) return false;
  const char* e = getenv("MLPSP_F32_SCALAR");
  return !(e && e[0] == '1');
}

}  // namespace mlpsp

