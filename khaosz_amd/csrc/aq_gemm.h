// What the tiled GEMM kernels share: arguments, the matrix-core product of either type, waits and the bare barrier.
#ifndef AQ_GEMM_H
#define AQ_GEMM_H

#include <type_traits>

#include "aq_common.h"

namespace aq {

constexpr int NUM_XCD = 8;
constexpr int GROUP_M = 4;

enum { OUT_I32 = 0, OUT_F32 = 1, OUT_BF16 = 2 };

struct GemmArgs {
  const uint8_t* A;
  const uint8_t* B;
  void* C;
  int M, N, K;
  int lda;           // bytes between rows of A: K, or more (rows that begin on lines)
  int tiles_m, tiles_n;
  const float* sx;   // int8: [M]; fp8: [1]
  const float* sw;   // int8: [N]; fp8: [1]
  const void* bias;  // [N] or null
  int bias_dtype;
  const void* res;   // [M, N] residual in the output's type, or null; may be C itself
};

// Workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2.
// Re-number them so that one XCD owns a contiguous run of tile ids, and walk
// tile ids in GROUP_M-tall column-major groups, so the tiles resident on an
// XCD at one time share A rows and B rows (4 x 8 tiles = 2 MB + 2 MB of
// operands for the 4096 x 2048 x 2048 case).
__device__ __forceinline__ void tile_of_block(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int nt = tiles_m * tiles_n;
  const int per = nt / NUM_XCD, rem = nt % NUM_XCD;
  const int xcd = pid % NUM_XCD, idx = pid / NUM_XCD;
  const int tile = xcd * per + (xcd < rem ? xcd : rem) + idx;
  const int group_sz = GROUP_M * tiles_n;
  const int group = tile / group_sz;
  const int first_m = group * GROUP_M;
  const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_group = tile - group * group_sz;
  tm = first_m + in_group % gm;
  tn = in_group / gm;
}

template <bool FP8>
struct Acc {
  using type = v16i;
};
template <>
struct Acc<true> {
  using type = v16f;
};

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding:
// vmcnt in bits 3:0 and 15:14, expcnt 6:4 and lgkmcnt 11:8 left at their maxima).
#define AQ_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0f70 | ((n) & 15) | (((n) >> 4) << 14))
// Workgroup barrier without the memory fence of __syncthreads(): the fence
// would drain every outstanding global->LDS load, including the ones issued
// two K steps ahead on purpose.  The empty asm statements stop the compiler
// from moving LDS accesses across it.
#define AQ_BARRIER()                   \
  do {                                 \
    asm volatile("" ::: "memory");     \
    __builtin_amdgcn_s_barrier();      \
    asm volatile("" ::: "memory");     \
  } while (0)

typedef __attribute__((address_space(3))) void lds_void;

template <bool FP8>
struct Frag {
  using type = v4i;  // 16 bytes of K per lane: v_mfma_i32_32x32x32_i8
};
template <>
struct Frag<true> {
  using type = v8i;  // 32 bytes of K per lane: v_mfma_scale_f32_32x32x64_f8f6f4
};

#ifndef AQ_FP8_SCALE
#define AQ_FP8_SCALE 0
#endif
template <bool FP8>
__device__ __forceinline__ typename Acc<FP8>::type mma(const typename Frag<FP8>::type& a,
                                                       const typename Frag<FP8>::type& b,
                                                       const typename Acc<FP8>::type& c) {
  if constexpr (!FP8) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  } else {
    // E8M0 scale 127 = 2^0 for both operands: plain e4m3 x e4m3.
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, AQ_FP8_SCALE, 0, AQ_FP8_SCALE);
  }
}

// gemm_slices.hip: small tiles, K cut among a workgroup's wavefronts
// (numbered on from gemm_mfma.hip's TileKind)
enum SlicesTile {
  SLICES_FIRST = 34, SLICES_32X32 = SLICES_FIRST, SLICES_64X32, SLICES_48X32, SLICES_32X48, SLICES_32X64, SLICES_48X48, SLICES_16X16, SLICES_16X32,
  SLICES_32X16, SLICES_16X64, SLICES_LAST = SLICES_16X64
};
int gemm_slices_tile(int64_t M, int64_t N, int64_t K, int64_t cus);
template <bool FP8, int OUT>
int gemm_slices_launch(GemmArgs& a, int tile, hipStream_t st);

// gemm_walk.hip
// The last round of 256 x 128 tiles is cut in two behind three rounds or more, when at most half the compute units have a tile in it.
inline bool gemm_walk_halves(int64_t tiles, int64_t cus) { return tiles % cus != 0 && tiles % cus <= cus / 2 && tiles >= 3 * cus; }
bool gemm_walk_ok(const GemmArgs& a, int out);
template <bool FP8, int OUT>
int gemm_walk_launch(const GemmArgs& a, hipStream_t st, int width);

}  // namespace aq

#endif  // AQ_GEMM_H
