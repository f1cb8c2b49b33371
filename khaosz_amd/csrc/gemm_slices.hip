// The GEMM of a few dozen to a few hundred rows: tiles of 32 x 32 or 64 x 32, K cut among the wavefronts of a workgroup.
//
// What bounds it: with few rows a compute unit has at most one small tile, and in a K loop shared by a workgroup's
// wavefronts every K step costs the latency of its barrier, its LDS reads and its waits, 430 to 450 cycles for 128 to 256
// of products (64 x 2048 x 2048: 16 steps, 6.8 k of 10 k cycles).  Here a wavefront takes every fourth (eighth) step by
// itself: the whole tile's products of its own slice of K, from its own LDS stages, with its own waits and no barrier.
// The chains run side by side, and the partial sums meet in LDS at the end.  int8 sums are whole numbers, in any order the
// same; FP8 sums are added in the order of the wavefronts.
//
// us, 64 x 32 tile of gemm_kernel (or the weight-streaming GEMV up to 32 rows) -> here: 32 x 2048 x 2048 4.8 -> 3.8,
// 64 x 2048 x 2048 5.4 -> 3.85, 64 x 1536 x 6912 10.4 -> 6.0, 128 x 2048 x 8192 11.8 -> 8.2, weights from HBM 13.9 -> 9.9;
// 200 x 1536 x 6912 10.5 -> 9.1 (64 x 32).  Wider tiles (64 x 64), 64-byte steps, three and four stages, eight wavefronts on
// the 32 x 32 tile measured 0 to 40 % slower.
#include "aq_gemm.h"

namespace aq {

template <int W, int TM, int TN, int BK, int NST>
struct SliceShape {
  static constexpr int BM = 32 * TM, BN = 32 * TN;
  static constexpr int STAGE = (BM + BN) * BK;         // bytes of a K step, of one wavefront
  static constexpr int WAVE_LDS = NST * STAGE > TM * TN * 4096 ? NST * STAGE : TM * TN * 4096;
  static constexpr int LOADS = STAGE / 1024;
  static_assert(W * WAVE_LDS <= 160 * 1024 && NST * LOADS <= 63, "LDS and the vector-memory counter");
};

template <bool FP8, int OUT, int W, int TM, int TN, int BK, int NST>
__global__ __launch_bounds__(W * 64) void gemm_slices_kernel(GemmArgs p) {
  using S = SliceShape<W, TM, TN, BK, NST>;
  constexpr int BM = S::BM, BN = S::BN, LOADS = S::LOADS;
  constexpr int PPR = BK / 16, RPL = 256 / BK, RPG = 1024 / BK;  // 16-byte pieces of a row; rows of a bank line, of a load
  constexpr int A_LOADS = BM / RPG;
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * S::WAVE_LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N, K = p.K;
  int tile_m, tile_n;
  tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // What the epilogue needs, requested first.  Of each 32 x 32 sub-tile a thread finishes one pair of columns of one row:
  // accumulator register r of lanes 2 c and 2 c + 1.
  constexpr int IT = 512 / (W * 64);  // items of a sub-tile per thread: rows 16 / IT registers apart
  const int er = tid >> 5, ec = tid & 31;
  auto row_of = [&](int t) { const int r = er + t * (16 / IT); return (r / 4) * 8 + (ec / 16) * 4 + r % 4; };
  const int col_in = 2 * (ec % 16);
  constexpr int ESZ = OUT == OUT_BF16 ? 2 : 4;
  const bool has_bias = p.bias != nullptr, bias_bf16 = p.bias_dtype == AQ_BF16, pairs = (N & 1) == 0;
  float sx[TM][IT], sw[TN][2];
  uint32_t bias[TN][2];  // raw: a conversion here would wait for the load
  uint2 res[TM][TN][IT];
  {
    const __amdgpu_buffer_rsrc_t Sr = make_rsrc(p.sx, (uint32_t)(FP8 ? 1 : M) * 4u), Wr = make_rsrc(p.sw, (uint32_t)(FP8 ? 1 : N) * 4u);
    const __amdgpu_buffer_rsrc_t Br = make_rsrc(has_bias ? p.bias : (const void*)p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
    const __amdgpu_buffer_rsrc_t Rr =
        make_rsrc(p.res ? reinterpret_cast<const uint8_t*>(p.res) + (int64_t)m0 * N * ESZ : (const void*)p.sw,
                  p.res ? (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)N * ESZ : 0u);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int t = 0; t < IT; ++t)
        sx[i][t] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Sr, FP8 ? 0 : (m0 + i * 32 + row_of(t)) * 4, 0, 0));
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int n = n0 + j * 32 + col_in + e;
        sw[j][e] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Wr, FP8 ? 0 : n * 4, 0, 0));
        bias[j][e] = bias_bf16 ? (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Br, n * 2, 0, 0)
                               : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Br, n * 4, 0, 0);
      }
    if (p.res) {  // uniform
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jt = 0; jt < TN * IT; ++jt) {
          const int j = jt / IT, t = jt % IT, n = n0 + j * 32 + col_in;
          const uint32_t at = ((uint32_t)(i * 32 + row_of(t)) * (uint32_t)N + (uint32_t)n) * ESZ;
          const uint32_t at0 = n < N ? at : OOB_OFFSET, at1 = n + 1 < N ? at + ESZ : OOB_OFFSET;
          if constexpr (OUT == OUT_BF16) {
            res[i][j][t].y = 0;
            if (pairs) {  // uniform
              res[i][j][t].x = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at0, 0, 0);
            } else {
              res[i][j][t].x = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Rr, at0, 0, 0);
              res[i][j][t].y = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Rr, at1, 0, 0);
            }
          } else {
            res[i][j][t].x = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at0, 0, 0);
            res[i][j][t].y = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at1, 0, 0);
          }
        }
    }
    asm volatile("" ::: "memory");
  }

  const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A + (int64_t)m0 * p.lda, (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)p.lda);
  const __amdgpu_buffer_rsrc_t Br = make_rsrc(p.B + (int64_t)n0 * K, (uint32_t)(N - n0 < BN ? N - n0 : BN) * (uint32_t)K);
  const int steps = (K + BK - 1) / BK;
  uint8_t* const mine = smem + wave * S::WAVE_LDS;
  // Rows of a stage: the tile's BM rows of A, then its BN rows of B; a load brings RPG of them.  Piece c of row r sits at
  // slot c ^ (r / RPL % PPR) (see gemm_kernel).
  auto issue = [&](int step, int buf) {
    const int k0 = step * BK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int ia = i < A_LOADS ? i : i - A_LOADS;
      const int row = ia * RPG + lane / PPR;
      const int k = k0 + ((lane % PPR) ^ (row / RPL % PPR)) * 16;
      const uint32_t off = k < K ? (uint32_t)row * (uint32_t)(i < A_LOADS ? p.lda : K) + (uint32_t)k : OOB_OFFSET;  // past K (or the last step): zeros
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < A_LOADS ? Ar : Br, (lds_void*)(mine + buf * S::STAGE + i * 1024), 16, off, 0, 0, 0);
    }
  };
#pragma unroll
  for (int s = 0; s < NST; ++s) issue(wave + s * W, s);

  using acc_t = typename Acc<FP8>::type;
  using frag_t = typename Frag<FP8>::type;
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
  const int col = lane & 31, half = lane >> 5, fsw = col / RPL % PPR;
  constexpr int KSUB = FP8 ? 64 : 32, NKS = BK / KSUB;
  int buf = 0;
  for (int step = wave; step < steps; step += W) {
    AQ_WAIT_VMCNT((NST - 1) * LOADS);  // this step's rows have landed
    asm volatile("" ::: "memory");
    const uint8_t* st = mine + buf * S::STAGE;
    frag_t f[NKS][TM + TN];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int i = 0; i < TM + TN; ++i) {
        const uint8_t* row = st + (i * 32 + col) * BK;
        if constexpr (!FP8) {
          f[ks][i] = *reinterpret_cast<const v4i*>(row + (((ks * 2 + half) ^ fsw) << 4));
        } else {
          const v4i lo = *reinterpret_cast<const v4i*>(row + (((ks * 4 + half * 2) ^ fsw) << 4));
          const v4i hi = *reinterpret_cast<const v4i*>(row + (((ks * 4 + half * 2 + 1) ^ fsw) << 4));
          f[ks][i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
      }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stage has been read
    asm volatile("" ::: "memory");
    issue(step + NST * W, buf);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mma<FP8>(f[ks][i], f[ks][TM + j], acc[i][j]);
    buf = buf == NST - 1 ? 0 : buf + 1;
  }
  AQ_WAIT_VMCNT(0);  // loads past the last step land in LDS too

  // the partial sums: [sub-tile][register][lane] words of each wavefront, in its own stages
  asm volatile("" ::: "memory");
  using word_t = std::conditional_t<FP8, float, int>;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) reinterpret_cast<word_t*>(mine)[((i * TN + j) * 16 + r) * 64 + lane] = acc[i][j][r];
  __syncthreads();
  const __amdgpu_buffer_rsrc_t Cr = make_rsrc(reinterpret_cast<uint8_t*>(p.C) + (int64_t)m0 * N * ESZ,
                                              (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)N * ESZ);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jt = 0; jt < TN * IT; ++jt) {
      const int j = jt / IT, t = jt % IT;
      word_t a0 = 0, a1 = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        typedef word_t pair_t __attribute__((ext_vector_type(2)));
        const pair_t v = *reinterpret_cast<const pair_t*>(smem + w * S::WAVE_LDS + (((i * TN + j) * 16 + er + t * (16 / IT)) * 64 + 2 * ec) * 4);
        a0 += v.x;
        a1 += v.y;
      }
      // three separately rounded fp32 operations (see gemm_kernel); rows past M fall outside the descriptor
      const float b0 = !has_bias ? 0.0f : __uint_as_float(bias_bf16 ? bias[j][0] << 16 : bias[j][0]);
      const float b1 = !has_bias ? 0.0f : __uint_as_float(bias_bf16 ? bias[j][1] << 16 : bias[j][1]);
      float y0 = __fadd_rn(__fmul_rn(__fmul_rn((float)a0, sx[i][t]), sw[j][0]), b0);
      float y1 = __fadd_rn(__fmul_rn(__fmul_rn((float)a1, sx[i][t]), sw[j][1]), b1);
      const int n = n0 + j * 32 + col_in;
      const uint32_t at = ((uint32_t)(i * 32 + row_of(t)) * (uint32_t)N + (uint32_t)n) * ESZ;
      const uint32_t at0 = n < N ? at : OOB_OFFSET, at1 = n + 1 < N ? at + ESZ : OOB_OFFSET;
      if constexpr (OUT == OUT_BF16) {
        uint32_t pk = pack_bf16x2(y0, y1);
        if (p.res)
          pk = pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(res[i][j][t].x << 16)),
                           __fadd_rn(__uint_as_float(pk & 0xffff0000u),
                                     __uint_as_float(pairs ? res[i][j][t].x & 0xffff0000u : res[i][j][t].y << 16)));
        if (pairs) {
          __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, at0, 0, STORE_WT);
        } else {
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)pk, Cr, at0, 0, STORE_WT);
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(pk >> 16), Cr, at1, 0, STORE_WT);
        }
      } else {
        if (p.res) y0 = __fadd_rn(y0, __uint_as_float(res[i][j][t].x)), y1 = __fadd_rn(y1, __uint_as_float(res[i][j][t].y));
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y0), Cr, at0, 0, STORE_WT);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y1), Cr, at1, 0, STORE_WT);
      }
    }
}

template <bool FP8, int OUT, int W, int TM, int TN, int BK, int NST>
static int launch_slices(GemmArgs& a, hipStream_t st) {
  a.tiles_m = (a.M + 32 * TM - 1) / (32 * TM);
  a.tiles_n = (a.N + 32 * TN - 1) / (32 * TN);
  aq::queue_kernel((gemm_slices_kernel<FP8, OUT, W, TM, TN, BK, NST>), dim3((unsigned)(a.tiles_m * a.tiles_n)), dim3(W * 64), 0,
                     st, a);
  return (int)hipGetLastError();
}

// 1: 32 x 32 tiles, 2: 64 x 32, 0: neither.  One tile per compute unit: a second round costs as much as the first, and the
// kernels with larger tiles move fewer bytes.  Up to 16 rows have kernels of their own.
//
// Measured, us, the path before (gemm_kernel's tiles; up to 32 rows the weight-streaming GEMV) -> here, weights in the
// last-level cache | streamed from HBM:
//   32 x 32, more than 32 rows: faster at every size tried (N 512 to 4096, K 512 to 8192), 64 x 2048 x 512 3.5 -> 3.1 | 3.9 -> 3.4,
//     64 x 4096 x 8192 12.2 -> 8.9 | 17.4 -> 12.7, 333 x 512 x 6912 10.5 -> 6.1 | 10.6 -> 7.7.
//   32 x 32, 17..32 rows: 32 x 256 x 2048 4.6 -> 3.7 | 4.7 -> 4.7, 32 x 2048 x 2048 5.1 -> 3.7 | 5.2 -> 5.4, 24 x 512 x 8192
//     9.9 -> 6.2 | 9.6 -> 10.8, 32 x 2048 x 8192 10.3 -> 6.7 | 10.4 -> 12.1, 32 x 8192 x 4096 8.2 -> 6.2 | 9.3 -> 9.5: a fifth to two
//     thirds faster from the cache, level to 16 % slower from HBM, where the GEMV has more loads in flight.
//   64 x 32: every tile reads all 64 rows of A.  K below 1536 is over before that is hidden (64 x 6144 x 512 3.5 -> 3.8 |
//     4.0 -> 4.3, x 1024 4.1 -> 4.3 | 5.5 -> 5.7, x 1536 4.6 -> 4.6 | 6.4 -> 6.3; 1000 x 512 x 1024 4.1 -> 4.4 | 4.5 -> 4.6), and so
//     is not a wide matrix whose weights alone keep the memory busy (64 x 8192 x 6912 11.5 -> 12.9 | 16.8 -> 17.4, 64 x 5632 x 6912
//     11.1 -> 11.5 | 15.8 -> 16.3, 40 x 8192 x 5120 9.5 -> 10.1 | 12.8 -> 13.0): those stay with the larger tiles.  Between them
//     64 x 5120 x 5120 8.9 -> 7.8 | 13.7 -> 13.0, 40 x 6912 x 6912 11.0 -> 10.7 | 14.3 -> 14.6, 200 x 2048 x 6912 10.8 -> 9.4 |
//     11.9 -> 11.8, 128 x 4096 x 8192 12.4 -> 11.9 | 17.3 -> 16.5.
int gemm_slices_rows(int64_t M, int64_t N, int64_t K, int64_t cus) {
  const int64_t n32 = (N + 31) / 32, tiles = (M + 63) / 64 * n32;
  if (M <= 16) return 0;
  if ((M + 31) / 32 * n32 <= cus) return 1;
  const bool streams = M <= 64 && N * K > (32 << 20) && M * tiles > 9600;  // much weight, and many tiles that each read A
  return tiles <= cus && K >= 1536 && !streams ? 2 : 0;
}

template <bool FP8, int OUT>
int gemm_slices_launch(GemmArgs& a, int tm, hipStream_t st) {
  if (tm == 1) return launch_slices<FP8, OUT, 4, 1, 1, 128, 2>(a, st);
  return launch_slices<FP8, OUT, 8, 2, 1, 128, 1>(a, st);
}
template int gemm_slices_launch<false, OUT_F32>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<false, OUT_BF16>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<true, OUT_F32>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<true, OUT_BF16>(GemmArgs&, int, hipStream_t);

}  // namespace aq
