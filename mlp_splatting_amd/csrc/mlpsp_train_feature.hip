// libmlpsp_hip: streamed feature L1 loss over the training steps of a frame (mlpsp_train.hpp) and its gradient with
// respect to the feature attributes: what the reference's _stream_l1, _feature_vjp and _feature_reduce
// (scannet/record_feature_loss.py:12-162) compute from per-pixel records.
//
// The value of target pixel t and channel c is  sum over steps, slots  k[t][step][slot] attr[primitive][slot][c]  with
//   k[t][step][slot] = sum over the (up to) four bilinear taps q of t:  weight_q  T alpha(step, q)  gate_slot(step, q),
// and the gradient of the attributes is the transposed product  sum over t  k[t][step][slot] sign(t, c).  So the taps are
// gathered once, into k -- per step and tile one number for each of the tile's targets and slots, 64 bytes where a
// target is a quarter of the image's resolution --, and what runs over the channels is a product of small matrices, not
// four walks over four pixels' record lists.  Both directions use the same k, in f32.
//
//   train_feature_blend_kernel  k of a tile's steps (kept for the backward); the tile's share of its targets' values
//   train_feature_join_kernel   the shares of a target (its taps lie in one, two or four tiles), residual, sign, loss
//   train_attr_kernel           steps sorted by primitive, in chunks as in mlpsp_train_backward.hip
//   train_attr_join_kernel      rows of primitives that span chunks
//
// All are bound by memory traffic: attribute rows out of L2 in the blend (8 KB per step at 512 channels, four slots), sign
// rows (2 KB) in the gradient; then come the zeros of the primitives without a step (8 KB each), in a launch of their own or,
// where weight gradients are asked for too, by their kernel (_listed: 0.26 ms less here, 0.10 more there, and what comes next
// does not meet the last of them on their way).  At 200,000 primitives, 1200x680, a 300x170 target of 512 channels: 0.45, 0.06,
// 0.20 and 0.26 ms; the record kernels took 4.95 ms for the loss and 8.1 ms for the gradient.
#include <type_traits>
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"
#include "mlpsp_mfma16.hpp"
#include "mlpsp_train.hpp"

namespace mlpsp {

// Bilinear source pixels of low-resolution index i (F.interpolate, align_corners=False): the same on host and device.
struct Taps {
  int i0, i1;
  float w;      // of i1
};
__host__ __device__ inline Taps feature_taps(int i, float scale, int size) {
  float v = ((float)i + .5f) * scale - .5f;
  v = v > 0.f ? v : 0.f;
  Taps t;
  t.i0 = (int)v;
  if (t.i0 > size - 1) t.i0 = size - 1;
  t.i1 = t.i0 + 1 < size ? t.i0 + 1 : size - 1;
  t.w = v - (float)t.i0;
  return t;
}
// Targets with a tap in [8 tile, 8 tile + 7]: the first one and their number (taps never decrease with i).
struct AxisSpan {
  int lo, n;
};
__host__ __device__ inline AxisSpan feature_axis_span(int tile, float scale, int size, int targets) {
  int lo = (int)((8.f * (float)tile - .5f) / scale) - 3;
  if (lo < 0) lo = 0;
  while (lo < targets && feature_taps(lo, scale, size).i1 < 8 * tile) ++lo;
  int hi = lo;
  while (hi < targets && feature_taps(hi, scale, size).i0 <= 8 * tile + 7) ++hi;
  return AxisSpan{lo, hi - lo};
}

constexpr int kBlendSteps = 16;     // steps per round of a blend workgroup
constexpr int kFeatWaves = 4;       // wavefronts of a blend workgroup, 256 channels each, at most

struct FeatShape {
  int W, H, ntx, nty, WF, HF, C, Cp, slots, NT;   // Cp: C rounded up to 4; NT: targets per tile, rounded up to 4
  float sx, sy;
  int64_t T;
};
inline bool feat_shape(int width, int height, int wf, int hf, int channels, int slots, FeatShape& f) {
  f.T = checked_num_tiles(width, height, 8, 8);
  if (f.T <= 0 || f.T > 2147483647LL - 8 || wf <= 0 || hf <= 0 || wf > width || hf > height || channels <= 0 ||
      channels > (1 << 20) || (slots != 1 && slots != 4 && slots != 5) || (int64_t)wf * hf > 2147483647LL)
    return false;
  f.W = width, f.H = height, f.WF = wf, f.HF = hf, f.C = channels, f.slots = slots;
  f.ntx = ceil_div(width, 8), f.nty = ceil_div(height, 8);
  f.Cp = (channels + 3) & ~3;
  f.sx = (float)width / (float)wf, f.sy = (float)height / (float)hf;
  int nx = 0, ny = 0;
  for (int t = 0; t < f.ntx; ++t) { const int n = feature_axis_span(t, f.sx, width, wf).n; nx = n > nx ? n : nx; }
  for (int t = 0; t < f.nty; ++t) { const int n = feature_axis_span(t, f.sy, height, hf).n; ny = n > ny ? n : ny; }
  f.NT = (nx * ny + 3) & ~3;
  return true;
}
// Kept for the backward: spans int32[2 (ntx + nty)] | groups of four targets of every tile int32[T] | signs int8[T][NT][Cp]
// | k float[S][NT / 4][slots][4].  Scratch of the forward: shares float[T][NT][Cp].
// A sign is the upper byte of a bf16 2, 0 or -2 (the lower one is zero): an integer of kSignUnit, 0 or -kSignUnit.
constexpr int kSignUnit = 64;
constexpr float kSignValue = 2.f;        // as bf16
struct FeatKept {
  int2 *columns, *rows;
  int32_t* groups;
  int8_t* signs;
  float* k;
  size_t bytes;
};
inline FeatKept feat_kept(void* base, const FeatShape& f, int64_t S) {
  FeatKept o{};
  unsigned char* p = (unsigned char*)base;
  o.columns = (int2*)p;
  p += step_align((size_t)f.ntx * 8);
  o.rows = (int2*)p;
  p += step_align((size_t)f.nty * 8);
  o.groups = (int32_t*)p;
  p += step_align((size_t)f.T * 4);
  o.signs = (int8_t*)p;
  p += step_align((size_t)f.T * f.NT * f.Cp);
  o.k = (float*)p;
  p += step_align((size_t)S * f.NT * f.slots * 4);
  o.bytes = (size_t)(p - (unsigned char*)base);
  return o;
}

__global__ __launch_bounds__(256) void feature_span_kernel(FeatShape f, FeatKept o) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x);
  if (i < f.ntx) {
    const AxisSpan s = feature_axis_span(i, f.sx, f.W, f.WF);
    o.columns[i] = make_int2(s.lo, s.n);
  }
  if (i < f.nty) {
    const AxisSpan s = feature_axis_span(i, f.sy, f.H, f.HF);
    o.rows[i] = make_int2(s.lo, s.n);
  }
  if (i < f.T)
    o.groups[i] = (feature_axis_span(i % f.ntx, f.sx, f.W, f.WF).n * feature_axis_span(i / f.ntx, f.sy, f.H, f.HF).n + 3) >> 2;
}

// Four consecutive channels of an attribute row: one load where the rows are 16-byte aligned (VEC), else four, those past
// the last channel clamped to it (what they yield is never used).
template <bool VEC>
__device__ __forceinline__ float4 four_channels(const float* __restrict__ row, int c, int C) {
  if constexpr (VEC) {
    return *reinterpret_cast<const float4*>(row + min(c, C - 4));
  } else {
    return make_float4(row[min(c, C - 1)], row[min(c + 1, C - 1)], row[min(c + 2, C - 1)], row[min(c + 3, C - 1)]);
  }
}
// Lanes per step, as a power of two: a row of up to 64, 128 or 256 channels takes 16, 32 or 64 lanes (four channels each),
// and the 4, 2 or 1 lane groups of a wavefront take steps in turn.
inline int lanes_per_row_log2(int Cp) { return Cp <= 64 ? 4 : Cp <= 128 ? 5 : 6; }

// One workgroup = one tile, four of its targets (blockIdx.y), up to 1,024 channels (blockIdx.z).  Sixteen steps at a time:
// every group of 16 lanes computes k of one step -- lane = (target, tap), the taps' sum two DPP
// adds --, then every lane adds the sixteen steps to its four channels.
template <int SLOTS, bool VEC>
__global__ __launch_bounds__(64 * kFeatWaves) void train_feature_blend_kernel(
    FeatShape f, FeatKept o, const int32_t* __restrict__ offsets, const int32_t* __restrict__ tile_base,
    const int32_t* __restrict__ chunk_table, const int32_t* __restrict__ ids, const unsigned char* __restrict__ records,
    const PrimRecord* __restrict__ prims, const float* __restrict__ attr, int lpr_log2, float beta, float temp,
    float* __restrict__ shares) {
  __shared__ __attribute__((aligned(16))) float s_k[2][kBlendSteps][SLOTS][4];
  __shared__ int s_p[2][kBlendSteps];
  const int tile = superblock_tile(blockIdx.x, f.ntx, f.nty);
  if (tile < 0) return;
  const int group = blockIdx.y, tx = tile % f.ntx, ty = tile / f.ntx, tid = threadIdx.x, lane = tid & 63;
  const int2 col = o.columns[tx], row = o.rows[ty];
  const int nt = col.y * row.y;
  if (group * 4 >= nt) return;
  const int base = tile_base[tile], count = tile_base[tile + 1] - base, table = step_table(offsets[tile], tile);

  // this lane's target and tap
  const int q = tid & 3, j = (tid >> 2) & 3, t = group * 4 + j;
  float weight = 0.f;
  int px = 0;
  if (t < nt) {
    const Taps x = feature_taps(col.x + t % col.y, f.sx, f.W), y = feature_taps(row.x + t / col.y, f.sy, f.H);
    const int xx = (q & 1) ? x.i1 : x.i0, yy = (q & 2) ? y.i1 : y.i0;
    const float w = ((q & 1) ? x.w : 1.f - x.w) * ((q & 2) ? y.w : 1.f - y.w);
    if ((xx >> 3) == tx && (yy >> 3) == ty) {
      weight = w;
      px = (yy & 7) * 8 + (xx & 7);
    }
  }
  const int lpr = 1 << lpr_log2, sub = lane >> lpr_log2, nsub = 64 >> lpr_log2;
  const int c = (blockIdx.z * (int)(blockDim.x >> 6) + (tid >> 6)) * 256 + (lane & (lpr - 1)) * 4;
  const bool channels = c < f.C;
  float4 acc[4];

  // A target of the tile that does not sample a step has a coefficient of 0, and 0 a = 0 unless the attribute a is infinite
  // or NaN: then the sums below are not finite, and the tile's are formed again without those products (SELECT), so that
  // such an attribute stays with the targets that sample it.
  const auto blend = [&](auto select) {
    constexpr bool SELECT = decltype(select)::value;
    const auto add = [](float k, float a, float& sum) {
      const float v = fmaf(k, a, sum);
      sum = SELECT && k == 0.f ? sum : v;
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int m = 0; m < count; m += kBlendSteps) {
      const int n = min(kBlendSteps, count - m), buf = (m / kBlendSteps) & 1;
      for (int i = tid >> 4; i < n; i += (int)(blockDim.x >> 4)) {
        const int slot = step_slot(chunk_table, table, m + i), p = ids[slot];
        float v[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        if (weight != 0.f) {
          const unsigned char* __restrict__ rec = records + (size_t)slot * kStepBytes;
          const float2 ta = *reinterpret_cast<const float2*>(rec + kStepPlaneB + px * 16);
          v[4] = weight * (ta.x * ta.y);
          if constexpr (SLOTS != 1) {
            const float4 d = *reinterpret_cast<const float4*>(rec + kStepPlaneC + px * 16);
            const PrimRecord& P = prims[p];
            const Vec3 ql = quat_rotate_conj(P.qw, P.qx, P.qy, P.qz, Vec3{d.x, d.y, d.z});
            float g[4];
            tetra_gates(ql.x, ql.y, ql.z, P.lgx, P.lgy, P.lgz, beta, temp, g);
#pragma unroll
            for (int s = 0; s < 4; ++s) v[s] = v[4] * g[s];
          }
        }
#pragma unroll
        for (int s = 0; s < 5; ++s) {
          v[s] += __shfl_xor(v[s], 1);
          v[s] += __shfl_xor(v[s], 2);
        }
        float* __restrict__ keep = o.k + (((size_t)(base + m + i) * (f.NT >> 2) + group) * SLOTS) * 4 + j;
        const bool writes = blockIdx.z == 0;
        if constexpr (SLOTS != 1) {
          const float mine = (q & 2) ? ((q & 1) ? v[3] : v[2]) : ((q & 1) ? v[1] : v[0]);
          const int s = q + (SLOTS == 5 ? 1 : 0);
          s_k[buf][i][s][j] = mine;
          if (writes) keep[s * 4] = mine;
        }
        if (SLOTS != 4 && q == 0) {
          s_k[buf][i][0][j] = v[4];
          if (writes) keep[0] = v[4];
        }
        if ((tid & 15) == 0) s_p[buf][i] = p;
      }
      __syncthreads();
      if (channels) {
#pragma unroll 4
        for (int i = sub; i < n; i += nsub) {
          const float* __restrict__ src = attr + (size_t)s_p[buf][i] * SLOTS * f.C;
#pragma unroll
          for (int s = 0; s < SLOTS; ++s) {
            const float4 a = four_channels<VEC>(src + (size_t)s * f.C, c, f.C);
            const float4 k = *reinterpret_cast<const float4*>(&s_k[buf][i][s][0]);
            add(k.x, a.x, acc[0].x), add(k.x, a.y, acc[0].y);
            add(k.x, a.z, acc[0].z), add(k.x, a.w, acc[0].w);
            add(k.y, a.x, acc[1].x), add(k.y, a.y, acc[1].y);
            add(k.y, a.z, acc[1].z), add(k.y, a.w, acc[1].w);
            add(k.z, a.x, acc[2].x), add(k.z, a.y, acc[2].y);
            add(k.z, a.z, acc[2].z), add(k.z, a.w, acc[2].w);
            add(k.w, a.x, acc[3].x), add(k.w, a.y, acc[3].y);
            add(k.w, a.z, acc[3].z), add(k.w, a.w, acc[3].w);
          }
        }
      }
    }
  };
  blend(std::false_type{});
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    finite &= __builtin_fabsf(acc[i].x) <= 3.4028235e38f && __builtin_fabsf(acc[i].y) <= 3.4028235e38f &&
              __builtin_fabsf(acc[i].z) <= 3.4028235e38f && __builtin_fabsf(acc[i].w) <= 3.4028235e38f;
  if (__syncthreads_or(!finite)) blend(std::true_type{});
  for (int d = lpr; d < 64; d <<= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      acc[i].x += __shfl_xor(acc[i].x, d);
      acc[i].y += __shfl_xor(acc[i].y, d);
      acc[i].z += __shfl_xor(acc[i].z, d);
      acc[i].w += __shfl_xor(acc[i].w, d);
    }
  }
  if (channels && sub == 0) {
    float* __restrict__ dst = shares + ((size_t)tile * f.NT + group * 4) * f.Cp + c;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<float4*>(dst + (size_t)i * f.Cp) = acc[i];
  }
}

// One lane = four channels of one target.  loss: one partial per workgroup, already divided by the number of residuals.
template <typename T>
__global__ __launch_bounds__(256) void train_feature_join_kernel(FeatShape f, FeatKept o, const float* __restrict__ shares,
                                                                 const T* __restrict__ target, float* __restrict__ loss) {
  __shared__ float s_part[4];
  const int quads = f.Cp >> 2;
  const long long at = (long long)blockIdx.x * 256 + threadIdx.x;
  float part = 0.f;
  if (at < (long long)f.WF * f.HF * quads) {
    const int pix = (int)(at / quads), c = (int)(at - (long long)pix * quads) * 4;
    const int ix = pix % f.WF, iy = pix / f.WF;
    const Taps x = feature_taps(ix, f.sx, f.W), y = feature_taps(iy, f.sy, f.H);
    const int x0 = x.i0 >> 3, x1 = x.i1 >> 3, y0 = y.i0 >> 3, y1 = y.i1 >> 3;
    const auto place = [&](int tx, int ty) {
      const int2 col = o.columns[tx], row = o.rows[ty];
      return ((size_t)(ty * f.ntx + tx) * f.NT + (iy - row.x) * col.y + (ix - col.x)) * f.Cp + c;
    };
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int ty = y0; ty <= y1; ++ty)
      for (int tx = x0; tx <= x1; ++tx) {
        const float4 s = *reinterpret_cast<const float4*>(shares + place(tx, ty));
        v[0] += s.x, v[1] += s.y, v[2] += s.z, v[3] += s.w;
      }
    const T* __restrict__ want = target + (size_t)pix * f.C;
    uint32_t signs = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (c + k < f.C) {
        const float delta = v[k] - (float)want[c + k];
        signs |= (uint32_t)(uint8_t)(int8_t)(kSignUnit * ((delta > 0.f) - (delta < 0.f))) << (8 * k);
        part += __builtin_fabsf(delta);
      }
    }
    for (int ty = y0; ty <= y1; ++ty)
      for (int tx = x0; tx <= x1; ++tx) *reinterpret_cast<uint32_t*>(o.signs + place(tx, ty)) = signs;
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) part += __shfl_xor(part, d);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = part;
  __syncthreads();
  if (threadIdx.x == 0)
    loss[blockIdx.x] = ((s_part[0] + s_part[1]) + (s_part[2] + s_part[3])) / (float)((long long)f.HF * f.WF * f.C);
}

// One wavefront = one chunk of the sorted steps x 256 channels: sum over the steps' targets of k[slot][target] sign.
template <int SLOTS, bool VEC>
__global__ __launch_bounds__(256) void train_attr_kernel(FeatShape f, FeatKept o, const int32_t* __restrict__ prim,
                                                         const int32_t* __restrict__ first, const int4* __restrict__ step, int S,
                                                         int chunk_steps, int num_chunks, int lpr_log2,
                                                         const float* __restrict__ adjoint, float* __restrict__ rows, float* __restrict__ out) {
  const int chunk = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
  if (chunk >= num_chunks) return;
  const int chunk_end = min(S, (chunk + 1) * chunk_steps);
  const int lpr = 1 << lpr_log2, sub = lane >> lpr_log2, nsub = 64 >> lpr_log2;
  const int c = (int)blockIdx.y * 256 + (lane & (lpr - 1)) * 4;
  const bool channels = c < f.C;
  const int cs = channels ? c : 0;
  const float norm = (float)((long long)f.WF * f.HF * f.C) * kSignUnit, scale = adjoint[0];
  const size_t k_stride = (size_t)f.NT * SLOTS;
  for (int pos = chunk * chunk_steps; pos < chunk_end;) {
    const int p = __builtin_amdgcn_readfirstlane(prim[pos]);
    const int all_end = first[p + 1], end = min(all_end, chunk_end);
    const bool goes_on = all_end > chunk_end, complete = first[p] == pos && !goes_on;
    float4 acc[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) acc[s] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int i = pos + sub; i < end; i += nsub) {
      const int4 at = step[i];
      const int tile = at.z, groups = o.groups[tile];
      const float* __restrict__ k = o.k + (size_t)at.y * k_stride;
      const int8_t* __restrict__ sg = o.signs + (size_t)tile * f.NT * f.Cp + cs;
      for (int g = 0; g < groups; ++g, k += 4 * SLOTS, sg += 4 * f.Cp) {
        int word[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) word[t] = *reinterpret_cast<const int*>(sg + t * f.Cp);
        float4 kk[SLOTS];
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) kk[s] = *reinterpret_cast<const float4*>(k + 4 * s);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float s0 = (float)(int8_t)word[t], s1 = (float)(int8_t)(word[t] >> 8), s2 = (float)(int8_t)(word[t] >> 16),
                      s3 = (float)(word[t] >> 24);
#pragma unroll
          for (int s = 0; s < SLOTS; ++s) {
            const float v = t == 0 ? kk[s].x : t == 1 ? kk[s].y : t == 2 ? kk[s].z : kk[s].w;
            acc[s].x = fmaf(v, s0, acc[s].x);
            acc[s].y = fmaf(v, s1, acc[s].y);
            acc[s].z = fmaf(v, s2, acc[s].z);
            acc[s].w = fmaf(v, s3, acc[s].w);
          }
        }
      }
    }
    for (int d = lpr; d < 64; d <<= 1) {
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) {
        acc[s].x += __shfl_xor(acc[s].x, d);
        acc[s].y += __shfl_xor(acc[s].y, d);
        acc[s].z += __shfl_xor(acc[s].z, d);
        acc[s].w += __shfl_xor(acc[s].w, d);
      }
    }
    if (channels && sub == 0) {
      if (complete) {
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) {
          float* __restrict__ dst = out + ((size_t)p * SLOTS + s) * f.C + c;
          const float4 v = make_float4(acc[s].x / norm * scale, acc[s].y / norm * scale, acc[s].z / norm * scale,
                                       acc[s].w / norm * scale);
          if constexpr (VEC) {
            *reinterpret_cast<float4*>(dst) = v;
          } else {
            dst[0] = v.x;
            if (c + 1 < f.C) dst[1] = v.y;
            if (c + 2 < f.C) dst[2] = v.z;
            if (c + 3 < f.C) dst[3] = v.w;
          }
        }
      } else {
        float* __restrict__ dst = rows + ((size_t)(goes_on ? num_chunks + chunk : chunk) * SLOTS) * f.Cp + c;
#pragma unroll
        for (int s = 0; s < SLOTS; ++s) *reinterpret_cast<float4*>(dst + (size_t)s * f.Cp) = acc[s];
      }
    }
    pos = end;
  }
}

// The same for four slots and sixteens of channels on the matrix cores (attr_on_matrix_cores): a product of k (four slots x
// steps and targets) and signs (steps and targets x channels) in 16x16x32 bf16 products.  Exact in its factors: a sign is a
// bf16 number, k the sum of three (mlpsp_vjp32.hpp), which take three times four of the sixteen rows and have accumulators of
// their own.  (A k below 2^-100 loses the third; its gradient, divided by the number of residuals, lies at the end of f32's range.)
// One wavefront = one chunk x 256 channels, eight steps at a time: lane (n, q) has two steps, and of their signs the
// channels 16 n .. 16 n + 15 -- sixteen bytes of a row a load; product j takes byte j of each, one byte permutation a word.
// The lanes hold the chunk's steps and their tiles' groups; a step's rows are not behind a chain of reads.
// Bound by the latency of those rows (2 KB a step at 512 channels), three wavefronts to a SIMD.  648,000 steps, 512 channels:
// 440 -> 200 us; error against float64 1.4e-7 -> 1.3e-7 of the gradient's norm, of a primitive's 1.4e-7 -> 0.6e-7 (median).
__global__ __launch_bounds__(256) void train_attr_mfma_kernel(FeatShape f, FeatKept o, const int32_t* __restrict__ prim,
                                                              const int32_t* __restrict__ first, const int4* __restrict__ step,
                                                              int S, int chunk_steps, int num_chunks,
                                                              const float* __restrict__ adjoint, float* __restrict__ rows,
                                                              float* __restrict__ out) {
  const int chunk = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63, n = lane & 15, q = lane >> 4;
  if (chunk >= num_chunks) return;
  const int chunk_begin = chunk * chunk_steps, chunk_end = min(S, chunk_begin + chunk_steps);
  const int c = (int)blockIdx.y * 256 + 16 * n, cs = c < f.C ? c : 0;
  const float norm = (float)((long long)f.WF * f.HF * f.C) * kSignValue, scale = adjoint[0];
  const int4 mine = step[min(chunk_begin + lane, chunk_end - 1)];       // (of up to 64)
  const int my_groups = o.groups[mine.z], parts = f.NT >> 2;
  for (int pos = chunk_begin; pos < chunk_end;) {
    const int p = __builtin_amdgcn_readfirstlane(prim[pos]);
    const int all_end = first[p + 1], end = min(all_end, chunk_end);
    const bool goes_on = all_end > chunk_end, complete = first[p] == pos && !goes_on;
    f32x4 acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = pos; i < end; i += 8) {
      int number[2], tile[2], groups[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int at = i + 2 * q + t, from = min(at, end - 1) - chunk_begin;
        number[t] = __shfl(mine.y, from);
        tile[t] = __shfl(mine.z, from);
        groups[t] = __shfl(my_groups, from);
        if (at >= end) groups[t] = 0;
      }
      for (int g = 0; g < parts && __ballot(groups[0] > g || groups[1] > g) != 0ull; ++g) {
        u32x4 sign[2][4];
        float4 k[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int8_t* __restrict__ from = o.signs + ((size_t)tile[t] * f.NT + 4 * g) * f.Cp + cs;
#pragma unroll
          for (int r = 0; r < 4; ++r) sign[t][r] = *reinterpret_cast<const u32x4*>(from + (size_t)r * f.Cp);
          k[t] = *reinterpret_cast<const float4*>(o.k + ((size_t)number[t] * parts + g) * 16 + 4 * (n & 3));
        }
        // row n of the one operand: part n / 4 of slot n % 4
        float v[8] = {k[0].x, k[0].y, k[0].z, k[0].w, k[1].x, k[1].y, k[1].z, k[1].w};
        u32x4 a;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const bool live = groups[d >> 1] > g && n < 12;
          float x = live ? v[2 * d] : 0.f, y = live ? v[2 * d + 1] : 0.f;
#pragma unroll
          for (int part = 0; part < 2; ++part) {
            const unsigned h = Ops<__bf16>::pack2(x, y);
            if ((n >> 2) > part) {
              x -= __uint_as_float(h << 16);
              y -= __uint_as_float(h & 0xffff0000u);
            }
          }
          a[d] = Ops<__bf16>::pack2(x, y);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const unsigned byte = 0x040c000cu + 0x01000100u * (unsigned)(j & 3);
          u32x4 b;
#pragma unroll
          for (int d = 0; d < 4; ++d)
            b[d] = __builtin_amdgcn_perm(sign[d >> 1][2 * (d & 1) + 1][j >> 2], sign[d >> 1][2 * (d & 1)][j >> 2], byte);
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc[j],
                                                           0, 0, 0);
        }
      }
    }
    // rows 4 q + slot of a product lie in lane group q: the three parts added up, slot q to group q
    float sum[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float even = sum_of_halves(acc[j][0], acc[j][2]), odd = sum_of_halves(acc[j][1], acc[j][3]);
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(even), __float_as_uint(odd), false, false);
      const unsigned lo = r[0], hi = r[1];
      sum[j] = __uint_as_float(lo) + __uint_as_float(hi);
    }
    if (c < f.C) {
      float* __restrict__ dst = complete ? out + ((size_t)p * 4 + q) * f.C + c
                                         : rows + ((size_t)(goes_on ? num_chunks + chunk : chunk) * 4 + q) * f.Cp + c;
#pragma unroll
      for (int j = 0; j < 16; j += 4) {
        float4 v = make_float4(sum[j], sum[j + 1], sum[j + 2], sum[j + 3]);
        if (complete) v = make_float4(v.x / norm * scale, v.y / norm * scale, v.z / norm * scale, v.w / norm * scale);
        *reinterpret_cast<float4*>(dst + j) = v;
      }
    }
    pos = end;
  }
}

// One workgroup per chunk, lane = four channels of one slot: the rows of the primitive that begins in it and goes on.
template <bool VEC>
__global__ __launch_bounds__(256) void train_attr_join_kernel(FeatShape f, const int32_t* __restrict__ prim,
                                                              const int32_t* __restrict__ first, int S, int chunk_steps,
                                                              int num_chunks, float unit, const float* __restrict__ adjoint,
                                                              const float* __restrict__ rows, float* __restrict__ out) {
  const int cf = blockIdx.x;
  const SpanningRun run = spanning_run(prim, first, S, cf, chunk_steps);
  if (run.p < 0) return;
  const int cl = run.last_chunk;
  const float norm = (float)((long long)f.WF * f.HF * f.C) * unit, scale = adjoint[0];
  const int quads = f.Cp >> 2;
  for (int i = threadIdx.x; i < quads * f.slots; i += 256) {
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
    for (int c = cf; c <= cl; ++c) {
      const float4 v = reinterpret_cast<const float4*>(rows + ((size_t)(c < cl ? num_chunks + c : c) * f.slots) * f.Cp)[i];
      acc.x += v.x, acc.y += v.y, acc.z += v.z, acc.w += v.w;
    }
    acc = make_float4(acc.x / norm * scale, acc.y / norm * scale, acc.z / norm * scale, acc.w / norm * scale);
    if constexpr (VEC) {
      reinterpret_cast<float4*>(out + (size_t)run.p * f.slots * f.C)[i] = acc;
    } else {
      const int s = i / quads, c = (i - s * quads) * 4;
      float* __restrict__ dst = out + ((size_t)run.p * f.slots + s) * f.C + c;
      dst[0] = acc.x;
      if (c + 1 < f.C) dst[1] = acc.y;
      if (c + 2 < f.C) dst[2] = acc.z;
      if (c + 3 < f.C) dst[3] = acc.w;
    }
  }
}

// Steps per wavefront of the gradient: 64, fewer where that would leave fewer than sixteen wavefronts for each SIMD.
inline int attr_chunk_steps(int64_t S, int C) {
  const int64_t per = S * ceil_div(C, 256) / 16384;
  return per >= 64 ? 64 : per <= 4 ? 4 : (int)per;
}
// Which of the two attribute kernels (four slots).  A lane of the matrix-core kernel takes sixteen signs a load, hence sixteens
// of channels, and a product eight steps; the other kernel takes one, two or four steps at a time, for rows of up to 256, 128
// and 64 channels.  Whole gradient call in us, f32 FMA / matrix cores, by steps of a chunk:
//     64 channels    4: 49 / 58      12:  54 / 64     43: 114 / 118
//    128             4: 58 / 70      12:  73 / 73     16:  88 / 80      43: 226 / 174
//    192 (256)       4: 58 / 62      5:   68 / 68 (73 / 76)      7: 78 / 71 (84 / 79)     43: 361 / 217 (404 / 270)
//    272 (512)       4: 63 / 74 (74 / 89)     7: 74 / 70 (86 / 85)     10: 93 / 80 (106 / 95)     64: 592 / 344 (740 / 506)
//    528             7: 78 / 80      11: 100 / 88     36: 260 / 160
inline bool attr_on_matrix_cores(int channels, int Cp, int chunk_steps) {
  return channels % 16 == 0 && channels > 64 && chunk_steps >= 7 * (64 >> lanes_per_row_log2(Cp));
}

}  // namespace mlpsp

using namespace mlpsp;

MLPSP_API size_t mlpsp_train_feature_bytes(int width, int height, int target_width, int target_height, int channels, int slots,
                                           int64_t num_steps, size_t* share_bytes, int64_t* loss_partials, size_t* row_bytes) {
  FeatShape f;
  if (!feat_shape(width, height, target_width, target_height, channels, slots, f) || num_steps < 0 || num_steps > 2147483647LL)
    return 0;
  if (share_bytes) *share_bytes = (size_t)f.T * f.NT * f.Cp * 4;
  if (loss_partials) *loss_partials = ((int64_t)f.WF * f.HF * (f.Cp >> 2) + 255) / 256;
  if (row_bytes) {
    const int per = attr_chunk_steps(num_steps, channels);
    *row_bytes = (size_t)2 * ((num_steps + per - 1) / per) * slots * f.Cp * 4;
  }
  return feat_kept(nullptr, f, num_steps).bytes;
}

MLPSP_API int mlpsp_train_feature_l1(const int32_t* tile_offsets_dev, int64_t num_pairs, int width, int height,
                                     const void* workspace_dev, size_t workspace_bytes, int64_t num_steps,
                                     const void* prim_records_dev, const float* attributes_dev, const void* target_dev,
                                     int target_is_half, int target_width, int target_height, int channels, int slots,
                                     float beta, float temp, void* kept_dev, size_t kept_bytes, float* shares_dev,
                                     float* loss_partials_dev, mlpsp_stream_t stream) {
  FeatShape f;
  if (!feat_shape(width, height, target_width, target_height, channels, slots, f) || num_pairs < 0 ||
      num_pairs > 2147483647LL || num_steps < 0 || num_steps > 2147483647LL)
    return MLPSP_E_ARGUMENT;
  if (!workspace_dev || workspace_bytes < step_tables_bytes(num_pairs, f.T)) return MLPSP_E_SCRATCH;
  const FeatKept o = feat_kept(kept_dev, f, num_steps);
  if (!kept_dev || reinterpret_cast<uintptr_t>(kept_dev) % 256 != 0 || kept_bytes < o.bytes) return MLPSP_E_SCRATCH;
  if (!tile_offsets_dev || !target_dev || !shares_dev || !loss_partials_dev || ((uintptr_t)shares_dev & 15u) ||
      (num_steps > 0 && (!prim_records_dev || !attributes_dev || (uintptr_t)prim_records_dev % 128 != 0)))
    return MLPSP_E_ARGUMENT;
  const StepPool sp = step_pool_carve(const_cast<void*>(workspace_dev), workspace_bytes, num_pairs, f.T);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(feature_span_kernel, dim3((unsigned)((f.T + 255) / 256)), dim3(256), 0, s, f, o);
  MLPSP_LAUNCH_CHECK();
  const int waves = min(kFeatWaves, ceil_div(channels, 256));
  const dim3 grid(superblock_grid(f.ntx, f.nty), (unsigned)(f.NT >> 2), (unsigned)ceil_div(channels, 256 * waves));
  const bool vec = channels % 4 == 0 && ((uintptr_t)attributes_dev & 15u) == 0;
  if (f.NT > 0) {
#define MLPSP_BLEND(SL, VEC)                                                                                            \
  hipLaunchKernelGGL((train_feature_blend_kernel<SL, VEC>), grid, dim3(64 * waves), 0, s, f, o, tile_offsets_dev, sp.tile_base, \
                     sp.chunk_table, sp.ids, sp.records, (const PrimRecord*)prim_records_dev, attributes_dev,            \
                     lanes_per_row_log2(f.Cp), beta, temp, shares_dev)
    if (slots == 1) { if (vec) MLPSP_BLEND(1, true); else MLPSP_BLEND(1, false); }
    else if (slots == 4) { if (vec) MLPSP_BLEND(4, true); else MLPSP_BLEND(4, false); }
    else { if (vec) MLPSP_BLEND(5, true); else MLPSP_BLEND(5, false); }
#undef MLPSP_BLEND
    MLPSP_LAUNCH_CHECK();
  }
  const dim3 join((unsigned)(((int64_t)f.WF * f.HF * (f.Cp >> 2) + 255) / 256));
  if (target_is_half)
    hipLaunchKernelGGL(train_feature_join_kernel<_Float16>, join, dim3(256), 0, s, f, o, shares_dev,
                       (const _Float16*)target_dev, loss_partials_dev);
  else
    hipLaunchKernelGGL(train_feature_join_kernel<float>, join, dim3(256), 0, s, f, o, shares_dev, (const float*)target_dev,
                       loss_partials_dev);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}

namespace {
int train_feature_gradients(int64_t num_steps, int width, int height, int target_width, int target_height, int channels, int slots,
                            const void* kept_dev, size_t kept_bytes, const void* scratch_dev, size_t scratch_bytes,
                            int num_primitives, const float* loss_adjoint_dev, float* rows_dev, float* out_dev, bool zeros,
                            hipStream_t s) {
  FeatShape f;
  if (!feat_shape(width, height, target_width, target_height, channels, slots, f) || num_steps < 0 ||
      num_steps > 2147483647LL || num_primitives < 0)
    return MLPSP_E_ARGUMENT;
  const FeatKept o = feat_kept(const_cast<void*>(kept_dev), f, num_steps);
  if (!kept_dev || kept_bytes < o.bytes) return MLPSP_E_SCRATCH;
  const StepSort t = step_sort(const_cast<void*>(scratch_dev), num_steps, num_primitives);
  if (!scratch_dev || scratch_bytes < t.bytes) return MLPSP_E_SCRATCH;
  if (num_primitives == 0) return MLPSP_OK;
  if (!loss_adjoint_dev || !out_dev || (num_steps > 0 && (!rows_dev || ((uintptr_t)rows_dev & 15u))))
    return MLPSP_E_ARGUMENT;
  const bool vec = channels % 4 == 0 && ((uintptr_t)out_dev & 15u) == 0;
  const int per = attr_chunk_steps(num_steps, channels), chunks = (int)((num_steps + per - 1) / per);
  if (chunks > 0) {
    const dim3 grid((unsigned)ceil_div(chunks, 4), (unsigned)ceil_div(channels, 256));
#define MLPSP_ATTR(SL, VEC)                                                                                              \
  hipLaunchKernelGGL((train_attr_kernel<SL, VEC>), grid, dim3(256), 0, s, f, o, t.prim, t.first, t.step,         \
                     (int)num_steps, per, chunks, lanes_per_row_log2(f.Cp), loss_adjoint_dev, rows_dev, out_dev)
    const bool wide = slots == 4 && vec && attr_on_matrix_cores(channels, f.Cp, per) && ((uintptr_t)kept_dev & 15u) == 0;
    const float unit = wide ? kSignValue : (float)kSignUnit;
    if (wide)
      hipLaunchKernelGGL(train_attr_mfma_kernel, grid, dim3(256), 0, s, f, o, t.prim, t.first, t.step, (int)num_steps, per, chunks,
                         loss_adjoint_dev, rows_dev, out_dev);
    else if (slots == 1) { if (vec) MLPSP_ATTR(1, true); else MLPSP_ATTR(1, false); }
    else if (slots == 4) { if (vec) MLPSP_ATTR(4, true); else MLPSP_ATTR(4, false); }
    else { if (vec) MLPSP_ATTR(5, true); else MLPSP_ATTR(5, false); }
#undef MLPSP_ATTR
    MLPSP_LAUNCH_CHECK();
    if (vec)
      hipLaunchKernelGGL(train_attr_join_kernel<true>, dim3((unsigned)chunks), dim3(256), 0, s, f, t.prim, t.first,
                         (int)num_steps, per, chunks, unit, loss_adjoint_dev, rows_dev, out_dev);
    else
      hipLaunchKernelGGL(train_attr_join_kernel<false>, dim3((unsigned)chunks), dim3(256), 0, s, f, t.prim, t.first,
                         (int)num_steps, per, chunks, unit, loss_adjoint_dev, rows_dev, out_dev);
    MLPSP_LAUNCH_CHECK();
  }
  if (!zeros) return MLPSP_OK;
  ZeroRows zero{};
  zero.add(out_dev, slots * channels);
  launch_zero_rows(t.first, num_primitives, zero, s);
  MLPSP_LAUNCH_CHECK();
  return MLPSP_OK;
}
}  // namespace

#define MLPSP_FEATURE_GRADIENTS(NAME, ZEROS)                                                                                \
  MLPSP_API int NAME(int64_t num_steps, int width, int height, int target_width, int target_height, int channels, int slots, \
                     const void* kept_dev, size_t kept_bytes, const void* scratch_dev, size_t scratch_bytes,                 \
                     int num_primitives, const float* loss_adjoint_dev, float* rows_dev, float* out_dev,                     \
                     mlpsp_stream_t stream) {                                                                                \
    return train_feature_gradients(num_steps, width, height, target_width, target_height, channels, slots, kept_dev,         \
                                   kept_bytes, scratch_dev, scratch_bytes, num_primitives, loss_adjoint_dev, rows_dev,       \
                                   out_dev, ZEROS, (hipStream_t)stream);                                                     \
  }
MLPSP_FEATURE_GRADIENTS(mlpsp_train_feature_gradients, true)
MLPSP_FEATURE_GRADIENTS(mlpsp_train_feature_gradients_listed, false)
#undef MLPSP_FEATURE_GRADIENTS
