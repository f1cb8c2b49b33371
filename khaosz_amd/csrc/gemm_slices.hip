// The GEMM of up to a few hundred rows: tiles of 16 x 16 to 48 x 48, K cut among the wavefronts of a workgroup.
//
// What bounds it: with few rows a compute unit has at most one small tile, and in a K loop shared by a workgroup's
// wavefronts every K step costs the latency of its barrier, its LDS reads and its waits, 430 to 450 cycles for 128 to 256
// of products (64 x 2048 x 2048: 16 steps, 6.8 k of 10 k cycles).  Here a wavefront takes every fourth (eighth) step by
// itself: the whole tile's products of its own slice of K, from its own LDS stages, with its own waits and no barrier.
// The chains run side by side, and the partial sums meet in LDS at the end.  int8 sums are whole numbers, in any order the
// same; FP8 sums are added in the order of the wavefronts.  What is left is the load of (rows + outputs) K bytes into each compute
// unit, 75 to 90 GB/s, and so the tile is the smallest of which every compute unit has at most one: hence products of 16 x 16, of
// which tiles come in steps of 16.
//
// us, 64 x 32 tile of gemm_kernel (or the weight-streaming GEMV up to 32 rows) -> here: 32 x 2048 x 2048 4.8 -> 2.9,
// 64 x 2048 x 2048 5.4 -> 3.2, 64 x 1536 x 6912 10.4 -> 5.2, 128 x 2048 x 8192 11.8 -> 8.1, weights from HBM 13.9 -> 9.8;
// 200 x 1536 x 6912 10.5 -> 9.2 (48 x 32).  Wider tiles (64 x 48, 64 x 64), 64-byte steps, three and four stages, eight wavefronts on
// the 32 x 32 tile measured 0 to 40 % slower.  Products of 32 x 32, and a compare and a select in every load, which only a step in
// which K ends needs: 32 x 32 tiles 3 to 4 % slower (64 x 2048 x 2048 3.83, K 2032 3.84 | 3.79), 64 x 32 1 to 2 % (200 x 1536 x 6912 10.26 | 10.12).
#include "aq_gemm.h"

namespace aq {

template <int W, int TM, int TN, int BK, int NST>
struct SliceShape {
  static constexpr int BM = 16 * TM, BN = 16 * TN;
  static constexpr int STAGE = (BM + BN) * BK;         // bytes of a K step, of one wavefront
  static constexpr int WAVE_LDS = NST * STAGE > TM * TN * 1024 ? NST * STAGE : TM * TN * 1024;
  static constexpr int LOADS = STAGE / 1024;
  static_assert(BM * BK % 1024 == 0 && BN * BK % 1024 == 0, "whole loads of A and of B");
  static_assert(W * WAVE_LDS <= 160 * 1024 && NST * LOADS <= 63, "LDS and the vector-memory counter");
};

template <bool FP8>
__device__ __forceinline__ std::conditional_t<FP8, v4f, v4i> mma16(const typename Frag<FP8>::type& a, const typename Frag<FP8>::type& b,
                                                                   const std::conditional_t<FP8, v4f, v4i>& c) {
  if constexpr (!FP8)
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, AQ_FP8_SCALE, 0, AQ_FP8_SCALE);
}

template <bool FP8, int OUT, int W, int TM, int TN, int BK, int NST>
__device__ __forceinline__ void gemm_slices_body(const GemmArgs& p, uint8_t* smem) {
  using S = SliceShape<W, TM, TN, BK, NST>;
  constexpr int BM = S::BM, BN = S::BN, LOADS = S::LOADS;
  constexpr int PPR = BK / 16, RPL = 256 / BK, RPG = 1024 / BK;  // 16-byte pieces of a row; rows of a bank line, of a load
  constexpr int A_LOADS = BM / RPG;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N, K = p.K;
  int tile_m, tile_n;
  tile_of_block(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // What the epilogue needs, requested first.  A thread finishes every (64 W)th pair of neighbouring columns of the tile, row by row.
  constexpr int PAIRS = BM * BN / 2, IT = (PAIRS + W * 64 - 1) / (W * 64);
  constexpr int ESZ = OUT == OUT_BF16 ? 2 : 4;
  auto row_of = [&](int t) { return (tid + t * W * 64) / (BN / 2); };
  auto col_of = [&](int t) { return (tid + t * W * 64) % (BN / 2) * 2; };
  const bool has_bias = p.bias != nullptr, bias_bf16 = p.bias_dtype == AQ_BF16, pairs = (N & 1) == 0;
  // byte offset of element (row, column + e), from the tile's first row; out of range past the tile or N (past M: outside the descriptor)
  auto at = [&](int t, int e) {
    const int n = n0 + col_of(t) + e;
    return n < N && (PAIRS % (W * 64) == 0 || tid + t * W * 64 < PAIRS) ? ((uint32_t)row_of(t) * (uint32_t)N + (uint32_t)n) * ESZ : OOB_OFFSET;
  };
  float sx[IT], sw[IT][2];
  uint32_t bias[IT][2];  // raw: a conversion here would wait for the load
  uint2 res[IT];
  {
    const __amdgpu_buffer_rsrc_t Sr = make_rsrc(p.sx, (uint32_t)(FP8 ? 1 : M) * 4u), Wr = make_rsrc(p.sw, (uint32_t)(FP8 ? 1 : N) * 4u);
    const __amdgpu_buffer_rsrc_t Br = make_rsrc(has_bias ? p.bias : (const void*)p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
    const __amdgpu_buffer_rsrc_t Rr =
        make_rsrc(p.res ? reinterpret_cast<const uint8_t*>(p.res) + (int64_t)m0 * N * ESZ : (const void*)p.sw,
                  p.res ? (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)N * ESZ : 0u);
#pragma unroll
    for (int t = 0; t < IT; ++t) {
      sx[t] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Sr, FP8 ? 0 : (m0 + row_of(t)) * 4, 0, 0));
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int n = n0 + col_of(t) + e;
        sw[t][e] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Wr, FP8 ? 0 : n * 4, 0, 0));
        bias[t][e] = bias_bf16 ? (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Br, n * 2, 0, 0)
                               : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Br, n * 4, 0, 0);
      }
    }
    if (p.res) {  // uniform
#pragma unroll
      for (int t = 0; t < IT; ++t) {
        if constexpr (OUT == OUT_BF16) {
          res[t].y = 0;
          if (pairs) {  // uniform
            res[t].x = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at(t, 0), 0, 0);
          } else {
            res[t].x = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Rr, at(t, 0), 0, 0);
            res[t].y = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(Rr, at(t, 1), 0, 0);
          }
        } else {
          res[t].x = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at(t, 0), 0, 0);
          res[t].y = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at(t, 1), 0, 0);
        }
      }
    }
    asm volatile("" ::: "memory");
  }

  const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A + (int64_t)m0 * p.lda, (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)p.lda);
  const __amdgpu_buffer_rsrc_t Br = make_rsrc(p.B + (int64_t)n0 * K, (uint32_t)(N - n0 < BN ? N - n0 : BN) * (uint32_t)K);
  const int steps = (K + BK - 1) / BK;
  uint8_t* const mine = smem + wave * S::WAVE_LDS;
  const int whole = K / BK;  // steps that K does not end in
  // Rows of a stage: the tile's BM rows of A, then its BN rows of B; a load brings RPG of them.  Piece c of row r sits at
  // slot c ^ (r / RPL % PPR) (see gemm_kernel).
  uint32_t vo[LOADS];
  auto row_in = [&](int i) { return (i < A_LOADS ? i : i - A_LOADS) * RPG + lane / PPR; };
  auto piece = [&](int i) { return ((lane % PPR) ^ (row_in(i) / RPL % PPR)) * 16; };
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    vo[i] = (uint32_t)row_in(i) * (uint32_t)(i < A_LOADS ? p.lda : K) + (uint32_t)piece(i);
  auto issue = [&](int step, int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < A_LOADS ? Ar : Br, (lds_void*)(mine + buf * S::STAGE + i * 1024), 16, vo[i], step * BK, 0, 0);
  };
  auto issue_last = [&](int step, int buf) {  // a step in which K ends: zeros behind it
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < A_LOADS ? Ar : Br, (lds_void*)(mine + buf * S::STAGE + i * 1024), 16,
                                               step * BK + piece(i) < K ? vo[i] : OOB_OFFSET, step * BK, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < NST; ++s) {
    const int step = wave + s * W;
    if (step < whole)
      issue(step, s);
    else if (step < steps)
      issue_last(step, s);
  }

  using acc_t = std::conditional_t<FP8, v4f, v4i>;
  using frag_t = typename Frag<FP8>::type;
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
  const int col = lane & 15, quarter = lane >> 4, fsw = col / RPL % PPR;
  constexpr int KSUB = FP8 ? 128 : 64, NKS = BK / KSUB;
  int buf = 0;
  // the products of the step in buffer `buf`, which step `next` then refills
  auto products = [&](bool next_whole, int next) __attribute__((always_inline)) {
    const uint8_t* st = mine + buf * S::STAGE;
    frag_t f[NKS][TM + TN];
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int i = 0; i < TM + TN; ++i) {
        const uint8_t* row = st + (i * 16 + col) * BK;
        if constexpr (!FP8) {
          f[ks][i] = *reinterpret_cast<const v4i*>(row + (((ks * 4 + quarter) ^ fsw) << 4));
        } else {
          const v4i lo = *reinterpret_cast<const v4i*>(row + (((ks * 8 + quarter * 2) ^ fsw) << 4));
          const v4i hi = *reinterpret_cast<const v4i*>(row + (((ks * 8 + quarter * 2 + 1) ^ fsw) << 4));
          f[ks][i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
      }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stage has been read
    asm volatile("" ::: "memory");
    if (next_whole)
      issue(next, buf);
    else if (next < steps)
      issue_last(next, buf);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = mma16<FP8>(f[ks][i], f[ks][TM + j], acc[i][j]);
    buf = buf == NST - 1 ? 0 : buf + 1;
  };
  int step = wave;
  for (; step + NST * W < whole; step += W) {
    AQ_WAIT_VMCNT((NST - 1) * LOADS);  // this step's rows have landed
    asm volatile("" ::: "memory");
    products(true, step + NST * W);
  }
  static_assert(NST <= 2, "at most one step behind this one in flight");
  for (; step < steps; step += W) {
    if (NST == 2 && step + W < steps)
      AQ_WAIT_VMCNT((NST - 1) * LOADS);
    else
      AQ_WAIT_VMCNT(0);
    asm volatile("" ::: "memory");
    products(false, step + NST * W);
  }

  // the partial sums: [16 x 16 block][register][lane] words of each wavefront, in its own stages
  asm volatile("" ::: "memory");
  using word_t = std::conditional_t<FP8, float, int>;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) reinterpret_cast<word_t*>(mine)[((i * TN + j) * 4 + r) * 64 + lane] = acc[i][j][r];
  __syncthreads();
  const __amdgpu_buffer_rsrc_t Cr = make_rsrc(reinterpret_cast<uint8_t*>(p.C) + (int64_t)m0 * N * ESZ,
                                              (uint32_t)(M - m0 < BM ? M - m0 : BM) * (uint32_t)N * ESZ);
#pragma unroll
  for (int t = 0; t < IT; ++t) {
    if (PAIRS % (W * 64) != 0 && tid + t * W * 64 >= PAIRS) break;
    const int r = row_of(t), c = col_of(t);
    const uint8_t* sums = smem + (((r / 16 * TN + c / 16) * 4 + r % 4) * 64 + r % 16 / 4 * 16 + c % 16) * 4;
    word_t a0 = 0, a1 = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      typedef word_t pair_t __attribute__((ext_vector_type(2)));
      const pair_t v = *reinterpret_cast<const pair_t*>(sums + w * S::WAVE_LDS);
      a0 += v.x;
      a1 += v.y;
    }
    // three separately rounded fp32 operations (see gemm_kernel); rows past M fall outside the descriptor
    const float b0 = !has_bias ? 0.0f : __uint_as_float(bias_bf16 ? bias[t][0] << 16 : bias[t][0]);
    const float b1 = !has_bias ? 0.0f : __uint_as_float(bias_bf16 ? bias[t][1] << 16 : bias[t][1]);
    float y0 = __fadd_rn(__fmul_rn(__fmul_rn((float)a0, sx[t]), sw[t][0]), b0);
    float y1 = __fadd_rn(__fmul_rn(__fmul_rn((float)a1, sx[t]), sw[t][1]), b1);
    if constexpr (OUT == OUT_BF16) {
      uint32_t pk = pack_bf16x2(y0, y1);
      if (p.res)
        pk = pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(res[t].x << 16)),
                         __fadd_rn(__uint_as_float(pk & 0xffff0000u),
                                   __uint_as_float(pairs ? res[t].x & 0xffff0000u : res[t].y << 16)));
      if (pairs) {
        __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, at(t, 0), 0, STORE_WT);
      } else {
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)pk, Cr, at(t, 0), 0, STORE_WT);
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(pk >> 16), Cr, at(t, 1), 0, STORE_WT);
      }
    } else {
      if (p.res) y0 = __fadd_rn(y0, __uint_as_float(res[t].x)), y1 = __fadd_rn(y1, __uint_as_float(res[t].y));
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y0), Cr, at(t, 0), 0, STORE_WT);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y1), Cr, at(t, 1), 0, STORE_WT);
    }
  }
}

template <bool FP8, int OUT, int W, int TM, int TN, int BK, int NST>
__global__ __launch_bounds__(W * 64) void gemm_slices_kernel(GemmArgs p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[W * SliceShape<W, TM, TN, BK, NST>::WAVE_LDS];
  gemm_slices_body<FP8, OUT, W, TM, TN, BK, NST>(p, smem);
}

template <bool FP8, int OUT, int W, int TM, int TN, int BK, int NST>
static int launch_slices(GemmArgs& a, hipStream_t st) {
  a.tiles_m = (a.M + 16 * TM - 1) / (16 * TM);
  a.tiles_n = (a.N + 16 * TN - 1) / (16 * TN);
  aq::queue_kernel((gemm_slices_kernel<FP8, OUT, W, TM, TN, BK, NST>), dim3((unsigned)(a.tiles_m * a.tiles_n)), dim3(W * 64), 0,
                     st, a);
  return (int)hipGetLastError();
}

// The tile of a launch, 0: none of them.  One tile per compute unit: a second round costs as much as the first, and the
// kernels with larger tiles move fewer bytes.
//
// Measured, us, the path before (gemm_kernel's tiles; up to 32 rows the weight-streaming GEMV) -> here, weights in the
// last-level cache | streamed from HBM:
//   16 x 16, 16 x 32 and 32 x 16 against 32 x 32 (520 sizes drawn from 17..130 rows, N 100 to 9000, K 256 to 9000): 0.84 | 0.86 in the mean, by
//     K 0.89 to 0.70, none slower.  Four wavefronts; eight on 16 x 16 0.93 of these from HBM with K from 4096, 1.06 from the cache.
//   Up to 16 rows (codes whose quantiser is a launch of its own, of rows too long or too wide for the kernels that round them): FP8 and tiles of
//     gemm_kernel 0.57 | 0.63 (181 sizes of 9..16 rows, the GEMV on codes or 64 x 32 tiles before), none slower: 12 x 816 x 6416 11.4 -> 4.3 | 11.6 -> 5.2, 9 x
//     5820 x 5120 18.4 -> 7.1 | 18.1 -> 8.5; 1..8 rows 0.56 | 0.68.  Beyond 8192 outputs 16 x 64 (0.71 | 0.78 for 59 sizes up to 16384, two of them
//     slower, by 4 and 5 %), then rounds of 16 x 32 (0.74 | 0.81).  12 x 4096 x 11008 16.1 -> 10.1 | 16.5 -> 13.1 (the weight-streaming kernel).
//   32 x 32, more than 32 rows: faster at every size tried (N 512 to 4096, K 512 to 8192), 64 x 2048 x 512 3.5 -> 3.1 | 3.9 -> 3.4,
//     64 x 4096 x 8192 12.2 -> 8.8 | 17.4 -> 12.6, 333 x 512 x 6912 10.5 -> 6.0 | 10.6 -> 7.6.
//   17..32 rows, the GEMV -> the smallest tile that fits (32 x 2048 is 16 x 16): 32 x 256 x 2048 4.6 -> 2.9 | 4.7 -> 3.3, 32 x 2048 x 2048 5.1 -> 2.9 |
//     5.2 -> 4.0, 24 x 512 x 8192 9.9 -> 4.3 | 9.6 -> 6.4, 32 x 8192 x 4096 8.2 -> 6.1 | 9.3 -> 9.3 (32 x 32).
//   48 x 32 and 32 x 48, where 32 x 32 are too many (120 sizes drawn from 17..800 rows, N 256 to 16384, K 256 to 9000): 0.90 | 0.92 in the
//     mean, 200 x 1536 x 6912 10.3 -> 9.2 | 11.7 -> 10.2 (64 x 32 tiles before), 22 x 9456 x 1280 FP8 0.66 | 0.77 (the GEMV before); the slowest 0.95 | 1.06
//     (24 x 10912 x 768).
//   64 x 32: every tile reads all 64 rows of A.  K below 1536 is over before that is hidden (64 x 6144 x 512 3.5 -> 3.8 |
//     4.0 -> 4.3, x 1024 4.1 -> 4.3 | 5.5 -> 5.7, x 1536 4.6 -> 4.6 | 6.4 -> 6.3; 1000 x 512 x 1024 4.1 -> 4.4 | 4.5 -> 4.6), and so
//     is not a wide matrix whose weights alone keep the memory busy (64 x 8192 x 6912 11.5 -> 12.9 | 16.8 -> 17.4, 57 x 7872 x 7552
//     12.7 -> 13.2 | 17.2 -> 17.7): those stay with the larger tiles.  Between them 64 x 5120 x 5120 8.9 -> 7.7 | 13.7 -> 13.0, 200 x 2048 x 6912
//     10.8 -> 9.3 | 11.9 -> 11.7, 128 x 4096 x 8192 12.4 -> 11.8 | 17.3 -> 16.4.
//   32 x 64 beyond (65..96 rows and such), K from 512: 0.94 | 0.94 in the mean of 15, none slower.
//   48 x 48 beyond, K from 3072, where the barriers of gemm_kernel's 64 x 64 tiles cost more than the larger share of a load: 333 x 1536 x 6912 12.8 ->
//     11.1 | 17.1 -> 13.2, FP8 12.6 -> 11.1 | 15.3 -> 12.4; with K 1536 to 3072 1.07 | 1.05 in the mean, and up to 64 rows 39 x 11824 x 3840 9.9 -> 10.9 | 13.7 ->
//     12.9.
int gemm_slices_tile(int64_t M, int64_t N, int64_t K, int64_t cus) {
  auto fits = [&](int64_t bm, int64_t bn) { return (M + bm - 1) / bm * ((N + bn - 1) / bn) <= cus; };
  if (fits(16, 16)) return SLICES_16X16;
  if (fits(16, 32)) return SLICES_16X32;
  if (M <= 16) return fits(16, 64) ? SLICES_16X64 : SLICES_16X32;
  if (fits(32, 16)) return SLICES_32X16;
  if (fits(32, 32)) return SLICES_32X32;
  if (fits(48, 32)) return SLICES_48X32;
  if (fits(32, 48)) return SLICES_32X48;
  const bool streams = M <= 64 && N * K > (32 << 20) && M * ((N + 31) / 32) > 9600;  // much weight, and many tiles that each read A
  if (fits(64, 32)) return K >= 1536 && !streams ? SLICES_64X32 : 0;
  if (M > 64 && K >= 512 && fits(32, 64)) return SLICES_32X64;
  return M > 64 && K >= 3072 && fits(48, 48) ? SLICES_48X48 : 0;
}

template <bool FP8, int OUT>
int gemm_slices_launch(GemmArgs& a, int tile, hipStream_t st) {
  switch (tile) {
    case SLICES_16X16: return launch_slices<FP8, OUT, 4, 1, 1, 128, 2>(a, st);
    case SLICES_16X32: return launch_slices<FP8, OUT, 4, 1, 2, 128, 2>(a, st);
    case SLICES_16X64: return launch_slices<FP8, OUT, 8, 1, 4, 128, 1>(a, st);
    case SLICES_32X16: return launch_slices<FP8, OUT, 4, 2, 1, 128, 2>(a, st);
    case SLICES_32X32: return launch_slices<FP8, OUT, 4, 2, 2, 128, 2>(a, st);
    case SLICES_48X32: return launch_slices<FP8, OUT, 4, 3, 2, 128, 2>(a, st);
    case SLICES_32X48: return launch_slices<FP8, OUT, 4, 2, 3, 128, 2>(a, st);
    case SLICES_64X32: return launch_slices<FP8, OUT, 8, 4, 2, 128, 1>(a, st);
    case SLICES_32X64: return launch_slices<FP8, OUT, 8, 2, 4, 128, 1>(a, st);
    default: return launch_slices<FP8, OUT, 8, 3, 3, 128, 1>(a, st);
  }
}
template int gemm_slices_launch<false, OUT_F32>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<false, OUT_BF16>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<true, OUT_F32>(GemmArgs&, int, hipStream_t);
template int gemm_slices_launch<true, OUT_BF16>(GemmArgs&, int, hipStream_t);

}  // namespace aq
