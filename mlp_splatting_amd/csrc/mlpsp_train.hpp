// Training steps: what a differentiable frame keeps between its forward and its backward pass.
//
// The forward writes one STEP per (8x8 tile, primitive that hits one of its pixels): 64 lanes = the tile's pixels, in
// planes of 64 so that every access of a wavefront is contiguous.  A lane that the primitive did not hit holds zeros
// (its transmittance among them, which no hit has): neutral beside finite numbers; the reverse walk and the feature blend,
// which meet adjoints and attributes that may be infinite, see to it that 0 inf does not come up.  58 of 64 lanes hit at
// the 200,000-primitive 1200x680 frame.  Everything downstream works on steps: the reverse walk goes through a tile's steps last to first, and the
// per-primitive gradient sums need an ordering of 0.65 M steps instead of one of 38 M per-pixel records -- whose sort,
// gathers and scattered stores were a third of a training step (the per-pixel records of mlpsp_records_* stay for
// callers that take records in their hands).
//
//   plane A  float4[64]  R, G, B, sigma_raw
//   plane B  float4[64]  T before the hit, alpha, decay, sigma logit
//   plane C  float4[64]  hit offset centre - point (MLP inputs 3..5), ReLU mask of layer 1 (bits)
//   plane D  uint32[64]  ReLU mask of layer 2
//
// How many steps a tile will have is known only when it is done, so steps come from a pool in chunks, one atomic for a
// group of them: a group per chunk at first, up to 32 steps in the end, so that a tile with a single hit takes one chunk
// and a long one few atomics.  (Training step of 50,000 small primitives, 2400x1360, 45 % of the pixels hit: 7.6 GiB with
// 32 steps from the start, 1.7 now; full frames take what they did, in the same time, and chunks of four are no better
// than of eight.)  The draw goes on when the pool is exhausted, so that the caller learns how many chunks the frame needs.
//
// A step is as large for five hits as for 64.  A primitive of few hits per tile is small on the screen, though, and hits
// few tiles: its steps are bounded by a few times the 28 KB of its weights and their gradients.
//
// Workspace: head int32[64] {chunks drawn, status bits, steps in all} | tile_steps int32[T] | tile_base int32[T + 1] |
// chunk_table int32[P / chunk + T + 1] | ids int32[pool] | records
#pragma once
#include "mlpsp_device.hpp"
#include "mlpsp_host.hpp"

namespace mlpsp {

constexpr int kStepBytes = 3328;
constexpr int kStepPlaneB = 1024, kStepPlaneC = 2048, kStepPlaneD = 3072;
struct StepGroups {              // as mlpsp_team.hpp takes them: groups begin at 0, c, 2 c, 4 c .. 32, 64, 96 ..
  static constexpr int kLog2 = 3, kMost = 32;
  __host__ __device__ static constexpr int slots(int begin) {
    return begin < (1 << kLog2) ? 1 << kLog2 : begin < kMost ? begin : kMost;
  }
};
constexpr int kStepChunk = 1 << StepGroups::kLog2;
static_assert(kStepChunk == MLPSP_STEP_CHUNK, "the unit of the workspace's first word");
constexpr int kTrainNumeric = 1, kTrainCapacity = 2;   // status bits

struct StepPool {
  int32_t* head;
  int32_t* tile_steps;
  int32_t* tile_base;
  int32_t* chunk_table;
  int32_t* ids;
  unsigned char* records;
  int pool_chunks;
};

inline size_t step_align(size_t v) { return (v + 255) & ~(size_t)255; }
inline size_t step_tables_bytes(int64_t num_pairs, int64_t num_tiles) {
  return step_align(64 * 4) + step_align((size_t)num_tiles * 4) + step_align((size_t)(num_tiles + 1) * 4) +
         step_align((size_t)(num_pairs / kStepChunk + num_tiles + 1) * 4);
}
inline size_t step_pool_bytes(int64_t num_pairs, int64_t num_tiles, int64_t pool_steps) {
  const size_t chunks = (size_t)((pool_steps + kStepChunk - 1) / kStepChunk);
  return step_tables_bytes(num_pairs, num_tiles) + step_align(chunks * kStepChunk * 4) + chunks * kStepChunk * (size_t)kStepBytes;
}
inline StepPool step_pool_carve(void* workspace, size_t bytes, int64_t num_pairs, int64_t num_tiles) {
  StepPool sp{};
  unsigned char* p = (unsigned char*)workspace;
  sp.head = (int32_t*)p;
  p += step_align(64 * 4);
  sp.tile_steps = (int32_t*)p;
  p += step_align((size_t)num_tiles * 4);
  sp.tile_base = (int32_t*)p;
  p += step_align((size_t)(num_tiles + 1) * 4);
  sp.chunk_table = (int32_t*)p;
  p += step_align((size_t)(num_pairs / kStepChunk + num_tiles + 1) * 4);
  const size_t left = bytes - step_tables_bytes(num_pairs, num_tiles);
  size_t chunks = left / ((size_t)kStepChunk * (kStepBytes + 4));
  while (chunks > 0 && step_align(chunks * kStepChunk * 4) + chunks * kStepChunk * (size_t)kStepBytes > left) --chunks;
  if (chunks > 0x7fffffffull / kStepChunk) chunks = 0x7fffffffull / kStepChunk;
  sp.pool_chunks = (int)chunks;
  sp.ids = (int32_t*)p;
  sp.records = p + step_align(chunks * kStepChunk * 4);
  return sp;
}

// The steps sorted by primitive: first sorted position of every primitive [N + 1]; of the sorted steps [S] the primitive, and
// pool slot, number in tile order, tile and pixel number of the tile's first pixel -- one 16-byte read.  Every buffer that
// holds them begins with them.
struct StepSort {
  int32_t *first, *prim;
  int4* step;
  size_t bytes;
};
inline StepSort step_sort(void* base, int64_t S, int N) {
  StepSort t{};
  unsigned char* p = (unsigned char*)base;
  t.first = (int32_t*)p;
  p += step_align(((size_t)N + 1) * 4);
  t.prim = (int32_t*)p;
  p += step_align((size_t)S * 4);
  t.step = (int4*)p;
  p += step_align((size_t)S * 16);
  t.bytes = (size_t)(p - (unsigned char*)base);
  return t;
}

#if defined(__HIPCC__)
// Wave-uniform writer state of one tile: its steps so far, and the first chunk (-1: the pool is exhausted) and the numbers of
// the group they are in.
struct StepWriter {
  int table_base, count, chunk, begin, end;
};
__device__ __forceinline__ int step_table(int list_start, int tile) { return (list_start >> StepGroups::kLog2) + tile; }
__device__ __forceinline__ StepWriter step_writer_begin(int list_start, int tile) {
  return StepWriter{step_table(list_start, tile), 0, 0, 0, 0};
}
// Slot of the tile's next step, or -1 if the pool is exhausted.  Call with the whole wavefront active.
__device__ __forceinline__ int step_writer_next(const StepPool& sp, StepWriter& w, int lane) {
  if (w.count == w.end) {
    const int steps = StepGroups::slots(w.count), draw = steps >> StepGroups::kLog2;
    int c = 0;
    if (lane == 0) c = atomicAdd(sp.head, draw);
    c = __builtin_amdgcn_readfirstlane(c);
    w.chunk = c + draw <= sp.pool_chunks ? c : -1;
    w.begin = w.count;
    w.end = w.count + steps;
  }
  const int number = w.count++;
  if (w.chunk < 0) return -1;
  const int within = number - w.begin;
  if ((within & (kStepChunk - 1)) == 0 && lane == 0)
    sp.chunk_table[w.table_base + (number >> StepGroups::kLog2)] = w.chunk + (within >> StepGroups::kLog2);
  return w.chunk * kStepChunk + within;
}
__device__ __forceinline__ int step_slot(const int32_t* __restrict__ chunk_table, int table_base, int m) {
  return chunk_table[table_base + (m >> StepGroups::kLog2)] * kStepChunk + (m & (kStepChunk - 1));
}
// One lane's part of a step.
__device__ __forceinline__ void step_store(const StepPool& sp, int slot, int lane, int p, bool hit, float R, float G,
                                           float B, float sigma_raw, float trans, float alpha, float decay, float logit,
                                           float dx, float dy, float dz, uint32_t mask1, uint32_t mask2) {
  unsigned char* __restrict__ rec = sp.records + (size_t)slot * kStepBytes;
  float4* __restrict__ a = reinterpret_cast<float4*>(rec);
  a[lane] = hit ? make_float4(R, G, B, sigma_raw) : make_float4(0.f, 0.f, 0.f, 0.f);
  a[64 + lane] = hit ? make_float4(trans, alpha, decay, logit) : make_float4(0.f, 0.f, 0.f, 0.f);
  a[128 + lane] = hit ? make_float4(dx, dy, dz, __uint_as_float(mask1)) : make_float4(0.f, 0.f, 0.f, 0.f);
  reinterpret_cast<uint32_t*>(rec + kStepPlaneD)[lane] = hit ? mask2 : 0u;
  if (lane == 0) sp.ids[slot] = p;
}
// Zero rows of the primitives that have no step, in every gradient tensor: a wavefront takes eight primitives, so that a
// row of a few floats fills its stores too.  Bound by the stores (6.3 TB/s for a plain fill on this card) where it is a launch
// of its own; the weight gradient kernels, which leave memory three quarters idle, do it beside their products (BESIDE: past the
// caches, where what they read lies; a launch of its own is 2 % slower that way).
struct ZeroRows {
  float* base[10];
  int len[10];       // floats per primitive
  int count;
  void add(float* p, int floats) {
    base[count] = p;
    len[count++] = floats;
  }
};
constexpr int kZeroGroup = 8;          // primitives a wavefront takes at a time
template <bool BESIDE>
__device__ __forceinline__ void zero_rows(const int32_t* __restrict__ first, int N, const ZeroRows& z, int group, int lane) {
  const int p0 = group * kZeroGroup;
  if (p0 >= N) return;
  const int p = min(p0 + (lane & 7), N - 1);
  const unsigned empty = (unsigned)__ballot(lane < 8 && p0 + lane < N && first[p] == first[p + 1]);
  if (empty == 0u) return;
  typedef float quad __attribute__((ext_vector_type(4)));
  const quad zero = {0.f, 0.f, 0.f, 0.f};
  for (int a = 0; a < z.count; ++a) {
    float* __restrict__ dst = z.base[a] + (size_t)p0 * z.len[a];
    const bool quads = (z.len[a] & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
    const int n = quads ? z.len[a] >> 2 : z.len[a];          // items per primitive
    if (n >= 64) {
      for (unsigned todo = empty; todo; todo &= todo - 1u) {
        const size_t at = (size_t)__builtin_ctz(todo) * n;
        for (int i = lane; i < n; i += 64) {
          if (!quads) dst[at + i] = 0.f;
          else if (BESIDE) __builtin_nontemporal_store(zero, reinterpret_cast<quad*>(dst) + at + i);
          else reinterpret_cast<quad*>(dst)[at + i] = zero;
        }
      }
    } else {
      for (int i = lane; i < 8 * n; i += 64) {
        if (!((empty >> (i / n)) & 1u)) continue;
        if (quads) reinterpret_cast<quad*>(dst)[i] = zero;
        else dst[i] = 0.f;
      }
    }
  }
}
static __global__ __launch_bounds__(256) void zero_rows_kernel(const int32_t* __restrict__ first, int N, ZeroRows z) {
  zero_rows<false>(first, N, z, (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), threadIdx.x & 63);
}
inline void launch_zero_rows(const int32_t* first, int N, const ZeroRows& z, hipStream_t s) {
  hipLaunchKernelGGL(zero_rows_kernel, dim3((unsigned)((N + 31) / 32)), dim3(256), 0, s, first, N, z);
}
// The primitive whose steps begin in chunk `chunk` and go on in the next (at most one): its number, or -1.
struct SpanningRun {
  int p, last_chunk;
};
__device__ __forceinline__ SpanningRun spanning_run(const int32_t* __restrict__ prim, const int32_t* __restrict__ first, int S,
                                                    int chunk, int chunk_steps) {
  const int chunk_end = (chunk + 1) * chunk_steps;
  if (chunk_end >= S) return SpanningRun{-1, 0};
  const int p = prim[chunk_end - 1], begin = first[p], end = first[p + 1];
  if (begin < chunk * chunk_steps || end <= chunk_end) return SpanningRun{-1, 0};
  return SpanningRun{p, (end - 1) / chunk_steps};
}
#endif

}  // namespace mlpsp
