// libmlpsp_hip: forward pass of a differentiable frame on 8x8 tiles with the 72->32->32->4 MLP, keeping its steps
// (mlpsp_train.hpp).  One traversal: image, alpha and everything the backward needs; the counterpart of the reference's
// record forward (np_tile_kernels.cu:2925-3206; training_wmma.cuh:62-253), which walks the frame twice -- count, then
// emit at scanned offsets -- because per-pixel records must lie pixel after pixel.
//
// Geometry, order, activations and compositing are the f32 expressions of the render (f32 MLP: its bits with
// `render_order`, the record kernels' rounding of layer 2 without).  Bound by the MLP; the steps add 3.3 KB of contiguous
// stores per hit step.  200,000 primitives, 1200x680, f32: 3.9 ms, against 4.0 + 6.0 of the record forward's two walks;
// 20,000 primitives, 320x240: 0.57 to 0.69 ms by camera, in teams of four (see train_plan).
#include <type_traits>

#include "mlpsp_device.hpp"
#include "mlpsp_finite.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mfma16.hpp"
#include "mlpsp_mlp_mfma32.hpp"
#include "mlpsp_team.hpp"
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
template <typename T> struct TrainDir { typedef DirWords type; };
template <> struct TrainDir<float> { typedef DirOperands type; };

struct TrainScene {
  const float *rays_o, *rays_d;
  const PrimRecord* prims;
  const int32_t *order, *offsets;
  const float *freq, *att, *W1, *b1, *W2, *b2, *W3, *b3;
  const unsigned char* packed;
  int N, W, H, ntx, nty;
  float thr;
  int max_hits;
};
// In f32 the walk parks 16 entries at a time: four workgroups' LDS is then a CU's (40,960 bytes each; three with 64), and at 128
// registers, with fifteen spills outside the products, four wavefronts run on a SIMD.  Forward of the 20,000-primitive 320x240
// frame, all teams: 776 -> 676 us for one camera, 582 -> 573 in the mean of five as traced; 200,000 at 1200x680 4.01 ms as before:
// there the matrix and vector pipes, which exclude each other, are taken.  (The f32 renders: frame of 200,000 0.5 % faster,
// feature frame of 30,000 with its hit records up to 4 % slower.)
template <typename T>
struct TrainItemLds {
  typename TrainDir<T>::type dir;
  WalkLdsOf<std::is_same_v<T, float> ? 16 : 64> walk;
};
template <typename T, int TEAM>
struct TrainTeamLds {
  typename TrainDir<T>::type dir;
  TeamWalkLds<TEAM> walk;
  float pay[2][TEAM][4][64];       // opacity, colour
  int chunk;
};

// A lane's pixel and the encoding of its ray.
struct TrainPixel {
  bool valid;
  int pix;
  Float3 ro, rd;
  float kf[3];
};
__device__ __forceinline__ TrainPixel train_pixel(const TrainScene& c, int tile, int l) {
  TrainPixel t;
  const int x = (tile % c.ntx) * 8 + (l & 7), y = (tile / c.ntx) * 8 + (l >> 3);
  t.valid = (x < c.W) && (y < c.H);
  t.pix = t.valid ? (y * c.W + x) : 0;
  t.ro = t.valid ? load3(c.rays_o, t.pix) : Float3{0.f, 0.f, 0.f};
  t.rd = t.valid ? load3(c.rays_d, t.pix) : Float3{0.f, 0.f, 0.f};
  t.kf[0] = t.kf[1] = t.kf[2] = 0.f;
  return t;
}
template <typename T>
__device__ __forceinline__ void train_encode(const TrainScene& c, const TrainPixel& t, int l, typename TrainDir<T>::type& dir) {
  if constexpr (sizeof(T) == 4) encode_direction(t.rd.x, t.rd.y, t.rd.z, c.freq, c.att, dir);
  else encode_direction_words<T>(t.rd.x, t.rd.y, t.rd.z, t.kf, l, dir);
}
// What an entry computes for a lane's pixel; zeros in the lanes that it does not hit, but for the masks.
struct TrainEntry {
  float R, G, B, sigma_raw, alpha, decay, logit, dx, dy, dz;
  uint32_t mask[2];
};
// bad: this lane's pixel yields something that is not finite; mlp_bad: some pixel's hidden layers do.
template <typename T, bool REC>
__device__ __forceinline__ TrainEntry train_entry(const TrainScene& c, const TrainPixel& t, int p, bool hit, const HitInfo& h,
                                                  unsigned long long mask, int l, const typename TrainDir<T>::type& dir,
                                                  bool& bad, bool& mlp_bad) {
  constexpr bool F32 = sizeof(T) == 4;
  TrainEntry e{};
  e.dx = hit ? h.dx : 0.f;
  e.dy = hit ? h.dy : 0.f;
  e.dz = hit ? h.dz : 0.f;
  e.decay = h.decay;
  float o[4];
  bad = mlp_bad = false;
  if constexpr (F32) {
    const float x6[6] = {t.rd.x, t.rd.y, t.rd.z, e.dx, e.dy, e.dz};
    mlp_wave_mfma32<REC, true, 32>(x6, c.freq, c.att, c.W1, c.b1, c.W2, c.b2, c.W3, c.b3, p, dir, o, e.mask);
  } else {
    mlp_bad = mlp_wave_mfma16<T, true, true>(c.packed + (size_t)p * kPackStride, mask, l, e.dx, e.dy, e.dz, t.kf, dir, o, e.mask);
  }
  e.logit = o[3];
  if (hit) {
    e.R = sigmoid(o[0]);
    e.G = sigmoid(o[1]);
    e.B = sigmoid(o[2]);
    e.sigma_raw = softplus(o[3]);
    e.alpha = 1.f - det_exp(-(e.sigma_raw * h.decay));
    if constexpr (!F32 || REC)
      bad = train_not_finite((e.dx + e.dy) + e.dz) || train_not_finite(h.decay) ||
            train_not_finite((o[0] + o[1]) + (o[2] + o[3])) || train_not_finite((e.R + e.G) + (e.B + e.sigma_raw)) ||
            train_not_finite(e.alpha);
  }
  return e;
}
__device__ __forceinline__ void train_store(const StepPool& sp, int slot, int l, int p, bool hit, float before, const TrainEntry& e) {
  if (slot >= 0)
    step_store(sp, slot, l, p, hit, e.R, e.G, e.B, e.sigma_raw, before, e.alpha, e.decay, e.logit, e.dx, e.dy, e.dz, e.mask[0], e.mask[1]);
}
__device__ __forceinline__ void train_status(const StepPool& sp, bool over, bool bad, int l) {
  int bits = 0;
  if (__ballot(over) != 0ull) bits |= kTrainCapacity;
  if (__ballot(bad) != 0ull) bits |= kTrainNumeric;
  if (bits != 0 && l == 0) atomicOr(sp.head + 1, bits);
}

// One tile by one wavefront.
template <typename T, bool REC>
__device__ __forceinline__ void train_tile(const int tile, const int l, TrainItemLds<T>& s, const TrainScene& c,
                                           const StepPool& sp, const TrainOut& out) {
  constexpr bool CHECKED = sizeof(T) != 4 || REC;
  TrainPixel t = train_pixel(c, tile, l);
  if constexpr (sizeof(T) != 4) phase_scales(c.freq, c.att, l >> 5, t.kf);
  train_encode<T>(c, t, l, s.dir);
  const int start = c.offsets[tile], end = c.offsets[tile + 1];
  float trans = 1.f, cr = 0.f, cg = 0.f, cb = 0.f;
  int used = 0;
  bool over = false, bad = false;
  StepWriter writer = step_writer_begin(start, tile);
  walk_tile_f32(
      c.order, start, end, c.N, c.prims, t.valid, t.ro.x, t.ro.y, t.ro.z, t.rd.x, t.rd.y, t.rd.z, c.thr, s.walk,
      [&]() { return t.valid && (trans >= kTransmittanceFloor) && (used < c.max_hits); },
      [&](int p, bool hit, const HitInfo& h, unsigned long long mask) {
        if (mask == 0ull) return true;
        bool lane_bad, mlp_bad;
        const TrainEntry e = train_entry<T, REC>(c, t, p, hit, h, mask, l, s.dir, lane_bad, mlp_bad);
        if constexpr (CHECKED) bad |= lane_bad | mlp_bad;
        const int slot = step_writer_next(sp, writer, l);
        const float before = trans;
        if (hit) {
          const float weight = trans * e.alpha;
          cr = fmaf(weight, e.R, cr);
          cg = fmaf(weight, e.G, cg);
          cb = fmaf(weight, e.B, cb);
          trans = trans * (1.f - e.alpha);
          ++used;
          if constexpr (CHECKED) bad |= train_not_finite(trans);
        }
        train_store(sp, slot, l, p, hit, before, e);
        const bool live = t.valid && (trans >= kTransmittanceFloor);
        over |= live && (used >= c.max_hits);      // np_tile_kernels.cu:3166-3168: refused, never truncated silently
        return __ballot(live) != 0ull;
      });
  if constexpr (CHECKED) bad |= train_not_finite((cr + cg) + cb);
  if (l == 0) sp.tile_steps[tile] = writer.count;
  train_status(sp, over, bad, l);
  if (t.valid) {
    store3(out.rgb, t.pix, cr, cg, cb);
    out.alpha[t.pix] = 1.f - trans;
  }
}

// One tile by a team (mlpsp_team.hpp): wavefront 0 adds up the colours, each wavefront writes the step of its own entry.
template <typename T, bool REC, int TEAM>
__device__ __forceinline__ void train_tile_team(const int tile, const int k, const int l, TrainTeamLds<T, TEAM>& s,
                                                const TrainScene& c, const StepPool& sp, const TrainOut& out) {
  constexpr bool CHECKED = sizeof(T) != 4 || REC;
  TrainPixel t = train_pixel(c, tile, l);
  if constexpr (sizeof(T) != 4) phase_scales(c.freq, c.att, l >> 5, t.kf);
  if (k == 0) train_encode<T>(c, t, l, s.dir);
  const int start = c.offsets[tile], end = c.offsets[tile + 1];
  float trans = 1.f, cr = 0.f, cg = 0.f, cb = 0.f;
  int used = 0, p_mine = 0;
  bool over = false, bad = false, lane_bad = false, mlp_bad = false;
  TeamSlots slots{step_table(start, tile), 0, 0, 0, 0};
  TrainEntry e{};
  walk_team_f32<TEAM>(
      c.order, start, end, c.N, c.prims, t.valid, t.ro.x, t.ro.y, t.ro.z, t.rd.x, t.rd.y, t.rd.z, c.thr, s.walk, k, l,
      [&]() { return t.valid && (trans >= kTransmittanceFloor) && (used < c.max_hits); },
      [&](int p, bool hit, const HitInfo& h, unsigned long long mask, int buf) {
        p_mine = p;
        e = train_entry<T, REC>(c, t, p, hit, h, mask, l, s.dir, lane_bad, mlp_bad);
        s.pay[buf][k][0][l] = e.alpha;
        s.pay[buf][k][1][l] = e.R;
        s.pay[buf][k][2][l] = e.G;
        s.pay[buf][k][3][l] = e.B;
      },
      [&](const unsigned long long* masks, int, int buf) {
        int kept = 0, mine = -1;
        float before = 0.f;
        bool hit_mine = false;
#pragma unroll
        for (int i = 0; i < TEAM; ++i) {
          const unsigned long long m = masks[i];
          const unsigned long long um = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)m) |
                                        ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(m >> 32)) << 32);
          if (um == 0ull) continue;
          const bool hit = ((um >> l) & 1ull) && (trans >= kTransmittanceFloor) && (used < c.max_hits);
          if (__ballot(hit) == 0ull) continue;           // (behind the last entry that counts)
          const float alpha = s.pay[buf][i][0][l];
          if (i == k) {
            mine = kept;
            before = trans;
            hit_mine = hit;
          }
          ++kept;
          if (hit) {
            if (k == 0) {
              const float weight = trans * alpha;
              cr = fmaf(weight, s.pay[buf][i][1][l], cr);
              cg = fmaf(weight, s.pay[buf][i][2][l], cg);
              cb = fmaf(weight, s.pay[buf][i][3][l], cb);
            }
            trans = trans * (1.f - alpha);
            ++used;
            if constexpr (CHECKED) bad |= train_not_finite(trans);
          }
          over |= t.valid && (trans >= kTransmittanceFloor) && (used >= c.max_hits);
        }
        if constexpr (CHECKED) bad |= (hit_mine && lane_bad) || (mine >= 0 && mlp_bad);
        const int slot = team_slot<StepGroups, false>(slots, kept, mine, k, l, sp.head, sp.chunk_table, sp.pool_chunks, s.chunk);
        train_store(sp, slot, l, p_mine, hit_mine, before, e);
        return __ballot(t.valid && (trans >= kTransmittanceFloor)) != 0ull;
      });
  if constexpr (CHECKED) bad |= train_not_finite((cr + cg) + cb);
  if (k == 0 && l == 0) sp.tile_steps[tile] = slots.count;
  train_status(sp, over, bad, l);
  if (k == 0 && t.valid) {
    store3(out.rgb, t.pix, cr, cg, cb);
    out.alpha[t.pix] = 1.f - trans;
  }
}

// A wavefront per tile, four tiles to a workgroup, but for the last ones: the workgroups from `body` on (per XCD) take a tile
// each, as a team.
constexpr int kTrainTeam = 4;
constexpr int kTrainLarge = 8;           // a team's wavefronts where tiles are few
static_assert(kTrainTeam <= kStepChunk && kTrainLarge <= kStepChunk, "a round of a team begins one chunk at most");
template <typename T, bool REC>
__device__ __forceinline__ void train_forward_body(const TrainScene& c, const StepPool& sp, const TrainOut& out, int body) {
  union Lds {
    TrainItemLds<T> item[kTrainTeam];
    TrainTeamLds<T, kTrainTeam> team;
  };
  __shared__ Lds s;
  const int unit = (int)(blockIdx.x / kNumXcd), xcd = (int)(blockIdx.x % kNumXcd);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), l = (int)threadIdx.x & 63;
  const bool alone = unit < body;
  const int tile = superblock_tile_of(xcd, alone ? unit * kTrainTeam + wave : body * kTrainTeam + (unit - body), c.ntx, c.nty);
  if (tile < 0) return;
  if (alone) train_tile<T, REC>(tile, l, s.item[wave], c, sp, out);
  else train_tile_team<T, REC, kTrainTeam>(tile, wave, l, s.team, c, sp, out);
}
// Every tile by a team.
template <typename T, bool REC, int TEAM>
__device__ __forceinline__ void train_forward_teams(const TrainScene& c, const StepPool& sp, const TrainOut& out) {
  __shared__ TrainTeamLds<T, TEAM> s;
  const int tile = superblock_tile(blockIdx.x, c.ntx, c.nty);
  if (tile < 0) return;
  train_tile_team<T, REC, TEAM>(tile, __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), (int)threadIdx.x & 63, s, c, sp, out);
}
// (The kernels take their pointers one by one, __restrict__: as members of an argument structure the output layer's weights,
// the same for all lanes, would be read through the vector memory path behind the stores of the steps.)
#define MLPSP_TRAIN_PARAMS                                                                                             \
  const float *__restrict__ rays_o, const float *__restrict__ rays_d, const PrimRecord *__restrict__ prims,             \
      const int32_t *__restrict__ order, const int32_t *__restrict__ offsets, const float *__restrict__ freq,           \
      const float *__restrict__ att
#define MLPSP_TRAIN_TAIL int N, int W, int H, int ntx, int nty, float thr, int max_hits, StepPool sp, TrainOut out, int body
// TEAM: every tile by a team of so many wavefronts; 0: most by one (train_forward_body).
constexpr int train_workgroup(int team) { return 64 * (team == 0 ? kTrainTeam : team); }
template <bool REC, int TEAM>
__global__ __launch_bounds__(train_workgroup(TEAM)) __attribute__((amdgpu_waves_per_eu(4, 4))) void train_forward_f32_kernel(
    MLPSP_TRAIN_PARAMS, const float* __restrict__ W1, const float* __restrict__ b1, const float* __restrict__ W2,
    const float* __restrict__ b2, const float* __restrict__ W3, const float* __restrict__ b3, MLPSP_TRAIN_TAIL) {
  const TrainScene c{rays_o, rays_d, prims, order, offsets, freq, att, W1, b1, W2, b2, W3, b3, nullptr, N, W, H, ntx, nty, thr, max_hits};
  if constexpr (TEAM == 0) train_forward_body<float, REC>(c, sp, out, body);
  else train_forward_teams<float, REC, TEAM>(c, sp, out);
}
template <typename T, int TEAM>
__global__ __launch_bounds__(train_workgroup(TEAM)) __attribute__((amdgpu_waves_per_eu(4, 4))) void train_forward_mfma_kernel(
    MLPSP_TRAIN_PARAMS, const unsigned char* __restrict__ packed, MLPSP_TRAIN_TAIL, FiniteScanInputs scan,
    int32_t* __restrict__ nonfinite) {
  const TrainScene c{rays_o, rays_d, prims, order, offsets, freq, att, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, packed,
                     N, W, H, ntx, nty, thr, max_hits};
  if constexpr (TEAM == 0) {
    train_forward_body<T, false>(c, sp, out, body);
    const int unit = (int)(blockIdx.x / kNumXcd), workgroup = 64 * kTrainTeam;
    if (scan.count > 0 && unit < body)
      finite_scan(scan, (long long)blockIdx.x * workgroup + threadIdx.x, (long long)kNumXcd * body * workgroup, nonfinite);
  } else {
    train_forward_teams<T, false, TEAM>(c, sp, out);
  }
}
#undef MLPSP_TRAIN_PARAMS
#undef MLPSP_TRAIN_TAIL
// A team of eight for every tile up to 640 tiles (two workgroups to a CU), of four up to 2,048; above, teams of four for the last
// tiles, so that a CU that is ahead can take one more of them: a wavefront's tile lasts a millisecond of the four that 12,750 take
// in f32.  Forward in us, f32 / fp16 operands:
//     tiles    a wavefront per tile   teams of eight    of four    for the last 1,024   1,536          2,048          2,560          3,072
//       300       641 / 245             240 / 101      259 / 115
//       500                             441 / 164      470 / 179
//     1,000                             643 / 228      644 / 227
//     1,610                             812 / 284      763 / 263
//     2,016                             973 / 334      906 / 311
//     2,560                           1,102 / --     1,012 / --     1,043 / 362    1,011 / 335    1,003 / 328
//     3,150                                                         1,265 / 402    1,172 / 386    1,185 / 392    1,202 / 396    1,224 / 394
//     4,860     1,783 / 639                                         1,855 / 574    1,708 / 532    1,719 / 537    1,759 / 547    1,770 / 544
//     8,000                                                         2,579 / 775    2,473 / 759    2,490 / 758    2,446 / 751    2,468 / 763
//    12,750     4,211 / 1,356                        5,396 / 1,695  4,001 / 1,181  3,984 / 1,183  3,915 / 1,179  3,906 / 1,160  3,924 / 1,173
//    30,000                                                         8,215          8,204          8,209          8,197          8,231
struct TrainPlan {
  int team;          // wavefronts of every tile's team; 0: the mixed kernel
  int body;          // its workgroups per XCD with a tile per wavefront
  unsigned grid;
};
inline TrainPlan train_plan(int ntx, int nty, int64_t T) {
  const unsigned slots = superblock_grid(ntx, nty);
  if (T <= 2048) return TrainPlan{T <= 640 ? kTrainLarge : kTrainTeam, 0, slots};
  const int per_xcd = (int)(slots / kNumXcd);
  const int teams = min(per_xcd, (T < 2816 ? 2048 : T <= 6400 ? 1536 : 2560) / kNumXcd), body = (per_xcd - teams) / kTrainTeam;
  return TrainPlan{0, body, (unsigned)(kNumXcd * (body + per_xcd - kTrainTeam * body))};
}

// What a wavefront that is done with its tile may look through for what is not finite, while the others' products leave memory
// idle; where it would be more -- most tiles in teams, which do not look, and many primitives --, a launch of its own.  Forward
// and look in us, fp16, in a launch of its own / beside:
//     50,000 primitives, 4,860 tiles, 212 KB a wavefront   645 /   597      200,000, 12,750, 280 KB   1,609 / 1,416
//    100,000,            4,860,       424 KB               749 /   695      200,000,  7,000, 635 KB   1,219 / 1,186
//     30,000,            2,400,     1,060 KB               378 /   385
constexpr int64_t kScanShare = 768 * 1024;

// tile_base = exclusive sums of tile_steps, head[2] = their total; one workgroup, four tiles to a thread and up to 16,384 behind
// one barrier, their counts on the way together.  Us (traced), consecutive tiles to a thread, one load after the other / 2 / 4 / 8
// rounds behind a barrier:
//     tiles     300   1,200   4,096  12,750  16,500  20,000  32,768  51,000  100,000
//     that      3.9     5.9     6.0    14.1    20.4    26.9    59.2    92.8    206.1
//     2         3.9     5.9     6.0     6.1     7.8     8.0    10.6    16.5     29.6
//     4         3.8     5.9     5.9     6.0     8.6     8.7     9.7    15.9     27.2
//     8         6.4     7.6     7.7     8.4     8.9     9.0     9.5    15.6     28.1
__global__ __launch_bounds__(1024) void step_scan_kernel(const int32_t* __restrict__ tile_steps, int T,
                                                         int32_t* __restrict__ tile_base, int32_t* __restrict__ head) {
  constexpr int kRounds = 4;
  __shared__ int32_t s_wave[2][kRounds][16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int carry = 0;
  for (int base = 0, turn = 0; base < T; base += kRounds * 4096, turn ^= 1) {
    int4 x[kRounds];
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
      // (the counts lie in whole 256 bytes: four at a multiple of four are inside)
      const int i = base + 4096 * u + 4 * t, at = min(i, (T - 1) & ~3);
      x[u] = *reinterpret_cast<const int4*>(tile_steps + at);
      x[u] = make_int4(i < T ? x[u].x : 0, i + 1 < T ? x[u].y : 0, i + 2 < T ? x[u].z : 0, i + 3 < T ? x[u].w : 0);
    }
    int incl[kRounds];
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
      incl[u] = (x[u].x + x[u].y) + (x[u].z + x[u].w);
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(incl[u], d);
        if (lane >= d) incl[u] += v;
      }
      if (lane == 63) s_wave[turn][u][wave] = incl[u];
    }
    __syncthreads();                     // (the one barrier of a turn: the next writes the other half)
#pragma unroll
    for (int u = 0; u < kRounds; ++u) {
      int before = carry;
#pragma unroll
      for (int w = 0; w < 16; ++w) {
        const int v = s_wave[turn][u][w];
        before += w < wave ? v : 0;
        carry += v;
      }
      const int i = base + 4096 * u + 4 * t, run = before + incl[u] - ((x[u].x + x[u].y) + (x[u].z + x[u].w));
      const int4 out = make_int4(run, run + x[u].x, run + x[u].x + x[u].y, run + x[u].x + x[u].y + x[u].z);
      if (i + 3 < T) {
        *reinterpret_cast<int4*>(tile_base + i) = out;
      } else {
        if (i < T) tile_base[i] = out.x;
        if (i + 1 < T) tile_base[i + 1] = out.y;
        if (i + 2 < T) tile_base[i + 2] = out.z;
      }
    }
  }
  if (t == 0) {
    tile_base[T] = carry;
    head[2] = carry;
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
  // k steps of a tile take up to k + 31 slots, and no more than the larger of a chunk and 2 k
  const int64_t full = num_pairs + (int64_t)(StepGroups::kMost - 1) * T, sparse = 2 * num_pairs + (int64_t)kStepChunk * T;
  const int64_t worst = (full < sparse ? full : sparse) + StepGroups::kMost;
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
  MLPSP_HIP_TRY(clear_async(f.sp.head, 64 * sizeof(int32_t), s));
  const TrainPlan plan = train_plan(f.ntx, f.nty, f.T);
#define MLPSP_TRAIN_TEAM(REC, TEAM)                                                                                    \
  hipLaunchKernelGGL((train_forward_f32_kernel<REC, TEAM>), dim3(plan.grid), dim3(train_workgroup(TEAM)), 0, s, rays_o_dev, rays_d_dev, \
                     (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev, W1, b1, W2, b2,  \
                     W3, b3, num_primitives, width, height, f.ntx, f.nty, threshold, max_hits, f.sp,                      \
                     TrainOut{out_rgb_dev, out_alpha_dev}, plan.body)
#define MLPSP_TRAIN_LAUNCH(REC)                                    \
  do {                                                             \
    if (plan.team == 0) MLPSP_TRAIN_TEAM(REC, 0);                  \
    else if (plan.team == kTrainTeam) MLPSP_TRAIN_TEAM(REC, kTrainTeam); \
    else MLPSP_TRAIN_TEAM(REC, kTrainLarge);                       \
  } while (0)
  if (render_order) MLPSP_TRAIN_LAUNCH(false);
  else MLPSP_TRAIN_LAUNCH(true);
#undef MLPSP_TRAIN_LAUNCH
#undef MLPSP_TRAIN_TEAM
  MLPSP_LAUNCH_CHECK();
  return train_scan(f, s);
}

namespace {
int train_forward_mfma(const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev, const int32_t* order_dev,
                       const int32_t* tile_offsets_dev, int64_t num_pairs, const float* freq_dev, const float* att_dev,
                       const void* packed_dev, int num_primitives, int width, int height, float threshold, int max_hits,
                       int use_bf16, void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev, float* out_alpha_dev,
                       FiniteScanInputs scan, int32_t* nonfinite_dev, hipStream_t s) {
  TrainFrame f;
  const int rc = train_frame(width, height, num_pairs, workspace_dev, workspace_bytes, f);
  if (rc != MLPSP_OK) return rc;
  if (!rays_o_dev || !rays_d_dev || !tile_offsets_dev || !freq_dev || !att_dev || !out_rgb_dev || !out_alpha_dev ||
      num_primitives < 0 || max_hits <= 0)
    return MLPSP_E_ARGUMENT;
  if (num_primitives > 0 && (!prim_records_dev || !packed_dev)) return MLPSP_E_ARGUMENT;
  if (((uintptr_t)prim_records_dev % 128) != 0 || ((uintptr_t)packed_dev % 16) != 0) return MLPSP_E_ARGUMENT;
  MLPSP_HIP_TRY(clear_async(f.sp.head, 64 * sizeof(int32_t), s));
  const TrainPlan plan = train_plan(f.ntx, f.nty, f.T);
  if (scan.count > 0 && finite_scan_bytes(scan) > kScanShare * kNumXcd * kTrainTeam * plan.body) {
    launch_finite_scan(scan, nonfinite_dev, s);
    MLPSP_LAUNCH_CHECK();
    scan.count = 0;
  }
#define MLPSP_TRAIN_TEAM(T, TEAM)                                                                                      \
  hipLaunchKernelGGL((train_forward_mfma_kernel<T, TEAM>), dim3(plan.grid), dim3(train_workgroup(TEAM)), 0, s, rays_o_dev, rays_d_dev, \
                     (const PrimRecord*)prim_records_dev, order_dev, tile_offsets_dev, freq_dev, att_dev,                \
                     (const unsigned char*)packed_dev, num_primitives, width, height, f.ntx, f.nty, threshold, max_hits, f.sp, \
                     TrainOut{out_rgb_dev, out_alpha_dev}, plan.body, scan, nonfinite_dev)
#define MLPSP_TRAIN_LAUNCH(T)                                      \
  do {                                                             \
    if (plan.team == 0) MLPSP_TRAIN_TEAM(T, 0);                    \
    else if (plan.team == kTrainTeam) MLPSP_TRAIN_TEAM(T, kTrainTeam); \
    else MLPSP_TRAIN_TEAM(T, kTrainLarge);                         \
  } while (0)
  if (use_bf16) MLPSP_TRAIN_LAUNCH(__bf16);
  else MLPSP_TRAIN_LAUNCH(_Float16);
#undef MLPSP_TRAIN_LAUNCH
#undef MLPSP_TRAIN_TEAM
  MLPSP_LAUNCH_CHECK();
  return train_scan(f, s);
}
}  // namespace

MLPSP_API int mlpsp_train_forward_mfma(const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev,
                                       const int32_t* order_dev, const int32_t* tile_offsets_dev, int64_t num_pairs,
                                       const float* freq_dev, const float* att_dev, const void* packed_dev,
                                       int num_primitives, int width, int height, float threshold, int max_hits,
                                       int use_bf16, void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev,
                                       float* out_alpha_dev, mlpsp_stream_t stream) {
  return train_forward_mfma(rays_o_dev, rays_d_dev, prim_records_dev, order_dev, tile_offsets_dev, num_pairs, freq_dev, att_dev,
                            packed_dev, num_primitives, width, height, threshold, max_hits, use_bf16, workspace_dev,
                            workspace_bytes, out_rgb_dev, out_alpha_dev, FiniteScanInputs{}, nullptr, (hipStream_t)stream);
}

MLPSP_API int mlpsp_train_forward_mfma_checked(const float* rays_o_dev, const float* rays_d_dev, const void* prim_records_dev,
                                       const int32_t* order_dev, const int32_t* tile_offsets_dev, int64_t num_pairs,
                                       const float* freq_dev, const float* att_dev, const void* packed_dev,
                                       int num_primitives, int width, int height, float threshold, int max_hits,
                                       int use_bf16, void* workspace_dev, size_t workspace_bytes, float* out_rgb_dev,
                                       float* out_alpha_dev, const float* const* arrays_dev,
                                       const int64_t* lengths, int num_arrays, int32_t* flag_dev, mlpsp_stream_t stream) {
  FiniteScanInputs scan{};
  if (!flag_dev || !finite_scan_inputs(arrays_dev, lengths, num_arrays, scan)) return MLPSP_E_ARGUMENT;
  return train_forward_mfma(rays_o_dev, rays_d_dev, prim_records_dev, order_dev, tile_offsets_dev, num_pairs, freq_dev, att_dev,
                            packed_dev, num_primitives, width, height, threshold, max_hits, use_bf16, workspace_dev,
                            workspace_bytes, out_rgb_dev, out_alpha_dev, scan, flag_dev, (hipStream_t)stream);
}
