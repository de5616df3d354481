// A tile's wavefronts as a team.  What an entry of the list contributes to a pixel does not depend on the entries in front
// of it, only the weight it gets does: wavefront k of TEAM tests and evaluates entries k, k + TEAM, ... of the list, and
// after every round of TEAM entries each wavefront goes through their opacities in list order.  All of them then know the
// transmittances, whether a pixel was still open at an entry's turn, and when the tile is done.
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_walk_f32.hpp"

namespace mlpsp {

// (orders LDS alone: requests to memory stay in flight across it)
__device__ __forceinline__ void team_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The walk of mlpsp_walk_f32.hpp by a team: `s` belongs to the workgroup, k is this wavefront's number.  evaluate(p, hit, h,
// mask, buf): this wavefront's entry of a round was hit by the lanes of `mask` (among those that can()); what it computes
// for the others it leaves in LDS buffer buf (0 or 1).  blend(masks, entries, buf): the round's entries, masks[i] = lanes
// that hit entry i; returns false when the tile is done.
template <int TEAM>
struct TeamWalkLds {
  WalkLds walk;
  unsigned long long mask[2][TEAM];
};
template <int TEAM, typename Can, typename Evaluate, typename Blend>
__device__ __forceinline__ void walk_team_f32(const int32_t* __restrict__ order, int start, int end, int N,
                                              const PrimRecord* __restrict__ prims, bool valid, float rox, float roy, float roz,
                                              float rdx, float rdy, float rdz, float thr, TeamWalkLds<TEAM>& s, int k, int l,
                                              Can&& can, Evaluate&& evaluate, Blend&& blend) {
  const unsigned long long in_image = __ballot(valid);
  const int lane0 = in_image ? (int)__builtin_ctzll(in_image) : 0;
  const float ox = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(rox), lane0)),
              oy = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(roy), lane0)),
              oz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(roz), lane0));
  const bool one_origin = __ballot(valid && !(rox == ox && roy == oy && roz == oz)) == 0ull;
  int buf = 0;
  for (int base = start; base < end; base += 64) {
    const int id_lane = (base + l < end) ? order[base + l] : -1;
    const bool usable = id_lane >= 0 && id_lane < N;
    unsigned long long todo = __ballot(usable);
    if (todo == 0ull) continue;
    if (usable && l % TEAM == k) {         // the entries' geometry, shared out
      const wf32x4* __restrict__ src = reinterpret_cast<const wf32x4*>(prims + id_lane);
      const wf32x4 a = src[0], b = src[1];
      wf32x4 c = src[2];
      const Vec3 vl = quat_rotate_conj(b[2], b[3], c[0], c[1], Vec3{a[0] - ox, a[1] - oy, a[2] - oz});
      c[2] = vl.x;
      c[3] = vl.y;
      s.walk.e[l][0] = a;
      s.walk.e[l][1] = b;
      s.walk.e[l][2] = c;
      s.walk.e[l][3][0] = vl.z;
    }
    int entries = (int)__builtin_popcountll(todo);
    for (int i = 0; i < k; ++i) todo &= todo - 1ull;
    team_barrier();
    for (; entries > 0; entries -= TEAM) {
      unsigned long long mask = 0ull;
      if (todo != 0ull) {
        const int j = (int)__builtin_ctzll(todo);
#pragma unroll
        for (int i = 0; i < TEAM; ++i) todo &= todo - 1ull;
        const wf32x4 q[3] = {s.walk.e[j][0], s.walk.e[j][1], s.walk.e[j][2]};
        Vec3 vl = {q[2][2], q[2][3], s.walk.e[j][3][0]};
        if (!one_origin)
          vl = quat_rotate_conj(q[1][2], q[1][3], q[2][0], q[2][1], Vec3{q[0][0] - rox, q[0][1] - roy, q[0][2] - roz});
        HitInfo h;
        const bool hit = hit_rot_from(q, vl, rox, roy, roz, rdx, rdy, rdz, thr, h) && can();
        mask = __ballot(hit);
        if (mask != 0ull) evaluate(__builtin_amdgcn_readlane(id_lane, j), hit, h, mask, buf);
      }
      if (l == 0) s.mask[buf][k] = mask;
      team_barrier();
      if (!blend(s.mask[buf], min(entries, TEAM), buf)) return;
      buf ^= 1;
    }
    team_barrier();                        // the entries' geometry is free again
  }
}

// Slots of a pool that hands out chunks in groups (mlpsp_hitrec.hpp, mlpsp_train.hpp), drawn by a team: the entries of a
// round that are kept get consecutive numbers in list order; a round that begins a new group lets wavefront 0 draw it (one
// atomic and one barrier per group).  GROUPS: kLog2, of the slots of a chunk, and slots(n), of the group that begins at
// number n; no fewer than a team has wavefronts, so that a round begins one chunk and one group at most.
struct TeamSlots {
  int table_base, count, chunk;      // chunk: first of the current group, -1 once the pool is exhausted
  int begin, end;                    // the numbers of the current group
};
// kept: entries of the round that are kept; mine: rank of this wavefront's entry among them, -1 if it is not.  Returns its
// slot, -1 if there is none.  Called by the whole team.  STOPS: nothing is counted once the pool is exhausted
// (counters[1] = 1 says so); else the draws go on.
template <typename GROUPS, bool STOPS>
__device__ __forceinline__ int team_slot(TeamSlots& w, int kept, int mine, int k, int l, int32_t* __restrict__ counters,
                                         int32_t* __restrict__ chunk_table, int pool_chunks, int& s_chunk) {
  constexpr int kLog2 = GROUPS::kLog2, kChunk = 1 << kLog2;
  if (kept == 0 || (STOPS && w.chunk < 0)) return -1;
  const int before = w.count, after = before + kept;
  const int group = w.end, entry = (before + kChunk - 1) & ~(kChunk - 1);   // next beginnings at or behind `before`
  const int old_chunk = w.chunk, old_begin = w.begin;
  w.count = after;
  if (group < after) {
    const int draw = GROUPS::slots(group) >> kLog2;
    team_barrier();                  // (the number drawn before has been read by all)
    if (k == 0 && l == 0) s_chunk = atomicAdd(counters, draw);
    team_barrier();
    w.chunk = __builtin_amdgcn_readfirstlane(s_chunk);
    w.begin = group;
    w.end = group + (draw << kLog2);
    if (w.chunk + draw > pool_chunks) {
      w.chunk = -1;
      if (STOPS) {
        w.count = group;
        if (k == 0 && l == 0) atomicExch(counters + 1, 1);
      }
    }
  }
  const auto chunk_of = [&](int number) {
    const int c = number >= group ? w.chunk : old_chunk;
    return c < 0 ? -1 : c + ((number - (number >= group ? group : old_begin)) >> kLog2);
  };
  if (entry < after && k == 0 && l == 0 && chunk_of(entry) >= 0) chunk_table[w.table_base + (entry >> kLog2)] = chunk_of(entry);
  if (mine < 0) return -1;
  const int chunk = chunk_of(before + mine);
  return chunk < 0 ? -1 : (chunk << kLog2) + ((before + mine) & (kChunk - 1));
}

}  // namespace mlpsp
