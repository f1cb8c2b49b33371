// What the decode kernels (gemv.hip, gemv_rows.hip) share: their arguments, the epilogue's operands and the launch helpers.
#pragma once
#include "aq_common.h"

namespace aq {

struct GemvArgs {
  const void* x;      // [M, K] bf16 activations (fused-quantise kernels), row stride K
  const int8_t* xq;   // [M, K] codes (kernels that take codes)
  const float* sx;    // [M]
  const int8_t* wq;   // [N, K]
  const float* sw;    // [N]
  const void* bias;   // [N] or null
  const void* res;    // [M, N] residual in y's dtype (row stride ldr), or null; may be y itself
  void* y;            // [M, N]
  int64_t ldr;
  int M, N, K;
  int bias_dtype, y_dtype;
  int ksplit, groups;  // matrix-core variant: wavefronts sharing a row group, row groups per workgroup
  const void* gamma;   // NORM kernels: RMSNorm gain [K] in x's dtype
  float eps;
  const float* parts;  // attention partial results in place of x (gemv_rows_kernel<.., WPR>)
  int parts_ns, parts_d;
  int tile_rows;       // gemv_rows_kernel: rows of a tile (blockIdx.y), at most 16; 0: all M are one
};

// y (+ residual): the projection is rounded to the output type first and the
// sum rounded again, the bits a separate elementwise add of the two tensors gives.
__device__ __forceinline__ float add_residual_bf16(float y, uint32_t res_bits) {
  return __fadd_rn(bf16_bits_to_f32((uint16_t)f32_to_bf16_bits(y)), bf16_bits_to_f32((uint16_t)res_bits));
}

// Epilogue operands (activation scale, weight scale, bias, residual) are requested at the very start of a
// kernel through buffer descriptors, without a branch: a descriptor of size 0 (no bias, no residual, a
// wavefront or lane that stores nothing) makes the load return 0 without touching memory.  Written as
// `if (bias) load`, the compiler waited for the loads at every join of those branches -- a full memory
// round trip in front of the weight stream whenever a bf16 bias was given.
struct EpiOperands {
  __amdgpu_buffer_rsrc_t sx, sw, bias_f32, bias_bf16, res_f32, res_bf16;
  __device__ __forceinline__ EpiOperands(const GemvArgs& p, bool live, bool want_sx, bool want_res) {
    const bool has_bias = p.bias != nullptr;
    const bool bias_is_bf16 = p.bias_dtype == AQ_BF16, res_is_bf16 = p.y_dtype == AQ_BF16;
    const uint32_t n = (uint32_t)p.N;
    sx = make_rsrc(want_sx ? (const void*)p.sx : (const void*)p.sw, live && want_sx ? (uint32_t)p.M * 4u : 0u);
    sw = make_rsrc(p.sw, live ? n * 4u : 0u);
    bias_f32 = make_rsrc(has_bias ? p.bias : (const void*)p.sw, live && has_bias && !bias_is_bf16 ? n * 4u : 0u);
    bias_bf16 = make_rsrc(has_bias ? p.bias : (const void*)p.sw, live && has_bias && bias_is_bf16 ? n * 2u : 0u);
    const bool has_res = want_res && p.res != nullptr;
    const uint32_t res_elems = (uint32_t)p.M * (uint32_t)p.ldr;
    res_f32 = make_rsrc(has_res ? p.res : (const void*)p.sw, live && has_res && !res_is_bf16 ? res_elems * 4u : 0u);
    res_bf16 = make_rsrc(has_res ? p.res : (const void*)p.sw, live && has_res && res_is_bf16 ? res_elems * 2u : 0u);
  }
  __device__ __forceinline__ float load_sx(int m, bool ok) const {
    return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(sx, ok ? m * 4 : (int)OOB_OFFSET, 0, 0));
  }
  __device__ __forceinline__ float load_sw(int n, bool ok) const {
    return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(sw, ok ? n * 4 : (int)OOB_OFFSET, 0, 0));
  }
  // Both element sizes are requested; only the descriptor of the operand's own type has a size, the other
  // load returns 0, and the two results are OR-ed: no select on the type (which the compiler turns back
  // into a branch around each load, with a wait at its join).
  __device__ __forceinline__ float load_bias(int n, bool ok) const {
    const uint32_t f = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(bias_f32, ok ? n * 4 : (int)OOB_OFFSET, 0, 0);
    const uint32_t h = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(bias_bf16, ok ? n * 2 : (int)OOB_OFFSET, 0, 0);
    return __uint_as_float(f | (h << 16));
  }
  __device__ __forceinline__ uint32_t load_res(int m, int n, bool ok, int ldr) const {  // raw bits of one element
    const int e = m * ldr + n;
    const uint32_t f = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(res_f32, ok ? e * 4 : (int)OOB_OFFSET, 0, 0);
    const uint32_t h = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(res_bf16, ok ? e * 2 : (int)OOB_OFFSET, 0, 0);
    return f | (h & 0xffffu);
  }
};

// Weight loads are marked as streaming (nt): every byte is read exactly once per launch.  Measured 0.05 - 0.35 us
// per launch against plain loads (M = 1: 5.50 -> 5.15 us; a one-shot 16 MiB read: 4.4 -> 4.0 us).
#define GV_WLOAD buffer_load_16_stream
#define GV_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(0x0f70 | ((n) & 15) | (((n) >> 4) << 14))

// A kernel whose dynamic LDS may exceed 64 KiB is opted in to the whole 160 KiB of a compute unit the first
// time a launch on a device needs it (one attribute call per kernel and device instead of one per launch).
// Two threads racing here both make the idempotent call.
struct LdsOptIn {
  bool done[64] = {};
  int ensure(const void* fn) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = -1;
    if (dev >= 0 && done[dev]) return 0;
    const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return (int)e;
    if (dev >= 0) done[dev] = true;
    return 0;
  }
};

constexpr int64_t GV_MAX_LDS = 160 * 1024;  // LDS of one gfx950 CU

// gemv_rows.hip: the decode GEMV that quantises its rows itself, by what it makes of them.  a.x (and a.gamma) name the
// rows; launch only what gemv_rows_ok admits.
enum RowsKind { ROWS_I8, ROWS_I8_NORM, ROWS_I8_F32, ROWS_FP8 };
bool gemv_rows_ok(RowsKind kind, int64_t M, int64_t K);
int launch_gemv_rows(const GemvArgs& a, RowsKind kind, hipStream_t st);  // a.M above 16: in tiles (gemv_rows_tiled)
enum Tiling { TILED_NOT, TILED, TILED_ALONE };  // ALONE: the faster form only where the host's time for a launch counts
Tiling gemv_rows_tiled(RowsKind kind, int64_t M, int64_t N, int64_t K);
int launch_gemv_rows_swiglu(const GemvArgs& a, hipStream_t st);
int launch_gemv_rows_attn(const GemvArgs& a, hipStream_t st);  // rows from a.parts; M <= 8, K <= 2048

}  // namespace aq
