// The walk of one wavefront (64 pixels of a tile) through its tile's sorted list in exact f32 arithmetic, shared by
// the f32 render kernels and the f32 training forward.
//
// The list is read 64 entries at a time, one coalesced load; culled (negative) entries never get a turn.  Lane j
// fetches the geometry of entry j, PARK of them at a time, and parks the ten words that the hit test needs in LDS, with -- where the tile's rays
// share their origin (a pinhole camera: always) -- the rotated offset centre - origin, which depends on the entry alone
// (same expressions on the same operands as hit_rot(), so the same bits).  An entry's turn then begins with four
// broadcast reads instead of a chain list entry -> record -> test, and a fifth of the test is done already.  (Scalar
// loads of the next entry's record, a turn ahead as in the reduced-precision render, do not work here: the output
// layer's scalar weights leave too few scalar registers, and the compiler spills registers that are being loaded.)
#pragma once
#include "mlpsp_device.hpp"

namespace mlpsp {

typedef float wf32x4 __attribute__((ext_vector_type(4)));

template <int PARK>
struct WalkLdsOf {
  wf32x4 e[PARK][4];      // centre, precision diagonal, quaternion (words 0..9 of the record), rotated offset
};

typedef WalkLdsOf<64> WalkLds;

// hit_rot() with the record's words as q[] and the rotated offset vl = R(q)^T (c - o) given.
__device__ __forceinline__ bool hit_rot_from(const wf32x4 q[3], Vec3 vl, float rox, float roy, float roz, float rdx,
                                             float rdy, float rdz, float thr, HitInfo& h) {
  const float mx = q[0][3], my = q[1][0], mz = q[1][1], qw = q[1][2], qx = q[1][3], qy = q[2][0], qz = q[2][1];
  const Vec3 dl = quat_rotate_conj(qw, qx, qy, qz, Vec3{rdx, rdy, rdz});
  const float denom = fmaf(dl.x * dl.x, mx, fmaf(dl.y * dl.y, my, (dl.z * dl.z) * mz));
  const float numer = fmaf(dl.x * vl.x, mx, fmaf(dl.y * vl.y, my, (dl.z * vl.z) * mz));
  const float t = numer / denom;
  const float px = rox + t * rdx;
  const float py = roy + t * rdy;
  const float pz = roz + t * rdz;
  h.t = t;
  h.dx = q[0][0] - px;
  h.dy = q[0][1] - py;
  h.dz = q[0][2] - pz;
  const Vec3 ql = quat_rotate_conj(qw, qx, qy, qz, Vec3{h.dx, h.dy, h.dz});
  h.qlx = ql.x;
  h.qly = ql.y;
  h.qlz = ql.z;
  const float r2 = fmaxf(((ql.x * ql.x) * mx + (ql.y * ql.y) * my) + (ql.z * ql.z) * mz, 0.f);
  h.decay = det_exp(-0.5f * r2);
  return !(denom <= 1e-20f) && !(t <= 0.f) && (h.decay > thr);
}

// can(): may this lane still take a hit?  step(p, hit, h, mask): called for every entry that was tested, with the
// ballot of its hits; returns false when the walk is over.  Call with all 64 lanes of a wavefront, and with an `s` that no
// other wavefront of its workgroup touches (a wavefront's LDS operations are in order: no barrier).
template <int PARK, typename Can, typename Step>
__device__ __forceinline__ void walk_tile_f32(const int32_t* __restrict__ order, int start, int end, int N,
                                              const PrimRecord* __restrict__ prims, bool valid, float rox, float roy,
                                              float roz, float rdx, float rdy, float rdz, float thr, WalkLdsOf<PARK>& s,
                                              Can&& can, Step&& step) {
  const int l = threadIdx.x & 63;
  const unsigned long long in_image = __ballot(valid);
  const int lane0 = in_image ? (int)__builtin_ctzll(in_image) : 0;
  const float ox = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(rox), lane0)),
              oy = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(roy), lane0)),
              oz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(roz), lane0));
  const bool one_origin = __ballot(valid && !(rox == ox && roy == oy && roz == oz)) == 0ull;
  for (int base = start; base < end; base += 64) {
    const int id_lane = (base + l < end) ? order[base + l] : -1;
    const bool usable = id_lane >= 0 && id_lane < N;
    unsigned long long todo = __ballot(usable);
    const auto park = [&](bool mine) {
      if (!mine) return;
      const wf32x4* __restrict__ src = reinterpret_cast<const wf32x4*>(prims + id_lane);
      const wf32x4 a = src[0], b = src[1];
      wf32x4 c = src[2];
      const Vec3 vl = quat_rotate_conj(b[2], b[3], c[0], c[1], Vec3{a[0] - ox, a[1] - oy, a[2] - oz});
      c[2] = vl.x;
      c[3] = vl.y;
      s.e[l % PARK][0] = a;
      s.e[l % PARK][1] = b;
      s.e[l % PARK][2] = c;
      s.e[l % PARK][3][0] = vl.z;
    };
    int parked = -1;
    while (todo != 0ull) {
      const int j = (int)__builtin_ctzll(todo);
      todo &= todo - 1ull;
      if (j / PARK != parked) {
        parked = j / PARK;
        park(usable && l / PARK == parked);
      }
      const wf32x4* __restrict__ e = s.e[j % PARK];
      const wf32x4 q[3] = {e[0], e[1], e[2]};
      Vec3 vl = {q[2][2], q[2][3], e[3][0]};
      if (!one_origin)
        vl = quat_rotate_conj(q[1][2], q[1][3], q[2][0], q[2][1], Vec3{q[0][0] - rox, q[0][1] - roy, q[0][2] - roz});
      HitInfo h;
      const bool hit = hit_rot_from(q, vl, rox, roy, roz, rdx, rdy, rdz, thr, h) && can();
      if (!step(__builtin_amdgcn_readlane(id_lane, j), hit, h, __ballot(hit))) return;
    }
  }
}

}  // namespace mlpsp
