// Host-side helpers shared by the translation units of libmlpsp_hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/mlpsp.h"

#define MLPSP_API extern "C" __attribute__((visibility("default")))

// A failed HIP call maps to MLPSP_E_RUNTIME; the sticky error is cleared so that the caller's
// context stays usable (the reference's tests synchronise after every rejected call).
#define MLPSP_HIP_TRY(expr)                  \
  do {                                       \
    hipError_t e__ = (expr);                 \
    if (e__ != hipSuccess) {                 \
      (void)hipGetLastError();               \
      return MLPSP_E_RUNTIME;                \
    }                                        \
  } while (0)

#define MLPSP_LAUNCH_CHECK() MLPSP_HIP_TRY(hipGetLastError())

namespace mlpsp {

// Zeros in place of hipMemsetAsync: as a node of a captured graph a memset has left wrong contents on replays after the
// first, and every entry point but those that read back may be captured.  W: the widest word that pointer and size allow.
template <typename W>
__global__ __launch_bounds__(256) void clear_kernel(W* __restrict__ p, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = W{};
}
inline hipError_t clear_async(void* dev, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  const auto launch = [&](auto* p) {
    const size_t n = bytes / sizeof(*p), blocks = (n + 255) / 256;
    hipLaunchKernelGGL(clear_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, s, p, n);
    return hipGetLastError();
  };
  const uintptr_t bits = (uintptr_t)dev | (uintptr_t)bytes;
  if ((bits & 15) == 0) return launch((uint4*)dev);
  if ((bits & 3) == 0) return launch((uint32_t*)dev);
  return launch((unsigned char*)dev);
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// tiles_x * tiles_y with the overflow checks of np_tile_kernels.cu:4542-4551; 0 if unusable.
inline int64_t checked_num_tiles(int64_t W, int64_t H, int64_t TW, int64_t TH) {
  if (W <= 0 || H <= 0 || TW <= 0 || TH <= 0) return 0;
  const int64_t tx = 1 + (W - 1) / TW, ty = 1 + (H - 1) / TH;
  if (tx > 2147483647LL || ty > 2147483647LL || tx > 2147483647LL / ty) return 0;
  return tx * ty;
}

// The chip hands consecutive workgroup ids to its 8 XCDs in turn, and each XCD has its own L2.
// Kernels that want neighbouring work items to share an L2 launch 8*per_xcd workgroups and map
// blockIdx.x -> (blockIdx.x % 8) * per_xcd + blockIdx.x / 8, so XCD k owns the contiguous range
// [k*per_xcd, (k+1)*per_xcd) of logical work items.
constexpr int kNumXcd = 8;

// Tile kernels whose neighbouring tiles share most of their primitives use a two-dimensional version of the same
// idea: the tile grid is cut into square super-blocks and the super-blocks are dealt to the XCDs in turn, so the (up
// to) 64 tiles of a super-block run on one L2 while every XCD still gets an equal share of every image region.
// Workgroup b belongs to XCD b % 8; it is that XCD's j-th workgroup, j = b / 8, and takes tile j % side^2 of the XCD's
// (j / side^2)-th super-block.  Tiles outside the image return -1.
// A side is 8 tiles (16 measured 7 to 10 % slower, 4 within 1 %), or fewer on an image that has fewer than eight
// super-blocks of that size for every XCD (2 at the least: the render takes four slots at a time): 40x30 tiles are 20
// super-blocks of 8x8, three for some XCDs and two for the others, but 80 of 4x4.
constexpr int kSuperLog2 = 3;

__host__ __device__ inline int superblock_log2(int ntx, int nty) {
  int sl = kSuperLog2;
  while (sl > 1 && (int64_t)((ntx + (1 << sl) - 1) >> sl) * ((nty + (1 << sl) - 1) >> sl) < 8 * kNumXcd) --sl;
  return sl;
}

inline unsigned superblock_grid(int ntx, int nty) {
  const int sl = superblock_log2(ntx, nty);
  const int nsb = ((ntx + (1 << sl) - 1) >> sl) * ((nty + (1 << sl) - 1) >> sl);
  return (unsigned)((((nsb + kNumXcd - 1) / kNumXcd) * kNumXcd) << (2 * sl));
}

// j-th tile slot of XCD xcd
__device__ __forceinline__ int superblock_tile_of(int xcd, int j, int ntx, int nty) {
  const int sl = superblock_log2(ntx, nty), side = 1 << sl;
  const int nsx = (ntx + side - 1) >> sl, nsy = (nty + side - 1) >> sl;
  const int sb = kNumXcd * (j >> (2 * sl)) + xcd, within = j & (side * side - 1);
  if (sb >= nsx * nsy) return -1;
  const int stx = ((sb % nsx) << sl) + (within & (side - 1)), sty = ((sb / nsx) << sl) + (within >> sl);
  return (stx < ntx && sty < nty) ? sty * ntx + stx : -1;
}

__device__ __forceinline__ int superblock_tile(unsigned block, int ntx, int nty) {
  return superblock_tile_of((int)(block % kNumXcd), (int)(block / kNumXcd), ntx, nty);
}

}  // namespace mlpsp
