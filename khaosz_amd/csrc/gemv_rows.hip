// Decode path, one launch for rows of any length: a weight-streaming GEMV on the matrix core that quantises its own
// token rows -- up to 16 of them, bf16 or fp32, K any multiple of 16 up to 8192 -- while its weights are in flight.
// int8 (per-token scales, exact int32 sums: the bits of row quantiser + GEMV) and FP8 (e4m3, one scale per tensor,
// fp32 sums in a fixed order), with the RMSNorm in front and the residual or the SwiGLU behind folded in.
//
// A workgroup of 8 wavefronts owns 8, 16, 32 or 64 weight rows: KS K parts x GR groups of R rows.  Every wavefront
// requests its token rows, its share of the epilogue's operands and then ALL its weights (up to 16 loads of 16 bytes
// per lane; longer parts rotate two register batches), rounds its token rows into LDS, and multiplies behind one
// barrier; the K parts' sums meet in LDS and every thread finishes one output.
//
// What bounds it: at decode sizes the launch (1.8 us) and the latency of the token rows and weights, then how many
// requests a compute unit has to take in.  The number of loads is therefore cut to the line: a kernel is built for
// each row length class, so that no wavefront sends loads that fall outside its part.  An empty load (an offset past
// the descriptor) returns zero without touching memory but still takes its turn in the address path: with a fixed 16
// weight loads per lane and the epilogue's operands asked for by one wavefront in KS (20 small loads, most empty), the
// same kernel took 1.5 to 2.5 us longer.  Measured (us, graph replay, weights from HBM, before -> now):
//   bf16 16 x 2048 -> 8192 8.1 -> 6.5, 11 x 1536 -> 1536 5.9 -> 3.8, 8 x 2048 -> 3072 5.0 -> 3.9, 8 x 5632 -> 2048 7.3 -> 6.1;
//   rows that took a quantiser launch of their own: 11 x 6912 -> 1536 13.6 -> 7.7, 16 x 1840 -> 9152 15.7 -> 8.9,
//   11 x 5712 -> 4832 20.4 -> 13.8, fp32 8 x 6912 -> 1536 25 -> 8.3, 8 x 1536 -> 1536 6.7 -> 3.7;
//   FP8 8 x 2048 -> 8192 7.4 -> 5.6, 4 x 688 -> 3520 8.7 -> 3.0, 8 x 6912 -> 1536 17.5 -> 8.2;
//   up/gate + SwiGLU with the norm: 4 x 1536 -> 2 x 6912 7.3 -> 6.4, 8 x 2048 -> 2 x 5632 8.2 -> 7.6.
#include <type_traits>

#include "aq_common.h"
#include "aq_gemv.h"
#include "aq_rows.h"

namespace aq {

#ifdef AQ_LAB
// Lab build only (csrc/aq_lab.h): where the wavefronts leave time stamps of the 100 MHz counter, 8 per wavefront, and a
// switch that makes the kernel request no weight bytes (products of zeros).  The product library has neither.
__device__ long long* gv_timeline = nullptr;
__device__ int gv_skip_weights = 0;
#define GV_STAMP(slot)                                                                                         \
  do {                                                                                                         \
    if (gv_timeline && lane == 0) gv_timeline[((size_t)blockIdx.x * 16 + wave) * 8 + (slot)] = wall_clock64(); \
  } while (0)
#else
#define GV_STAMP(slot) \
  do {                 \
  } while (0)
#endif

constexpr int GX_WAVES = 8;  // wavefronts per workgroup
constexpr int64_t GX_MAX_K = 8192;

// KS K parts x GX_WAVES / KS groups of R weight rows.  RPW: token rows per wavefront (fp32 rows, twice as long in
// registers, go one after the other instead), VPL: 16-byte vectors per lane and row -- together the row length class.
// R = 8 fills half of a matrix-core operand (the other half repeats other pieces of the same rows and is not stored):
// for short matrices, so that twice the compute units stream weights.
// SWI: the weight is an MLP's up and gate projections stacked, rows [0, F) up and [F, 2F) gate; the first half of the
// row groups takes rows of up, the second half the same rows of gate, and the output is up * silu(gate), the two as the
// projections would have been stored (rounded to the output type first).
// WPR > 0: the rows (up to 8, of up to 2048) are a decode step's attention output, combined here from the attention kernel's partial
// results of up to 4 slices (p.parts), WPR wavefronts to a row: 4 rows of 1536 in 3 slices are 78 KB to request, and all
// eight wavefronts ask for them at once (whole rows in 4 of 4 wavefronts, vector ALU products, N = 1536: 5.8 us; 5.3).
// TILED: more than 16 rows, a tile of p.tile_rows of them per blockIdx.y.  FP8: the scale is the maximum of all rows', the other tiles'
// read besides.  (Kernels of their own: 25 registers more (FP8), and 0.03 to 0.05 us a launch for the tile's place.)
template <int KS, int R, bool BF16, int RPW, int VPL, bool NORM, bool FP8, bool SWI = false, int WPR = 0, bool TILED = false>
__global__ __launch_bounds__(GX_WAVES * 64) void gemv_rows_kernel(GemvArgs p) {
  constexpr int GR = GX_WAVES / KS;
  // rows rounded without a branch around each vector (see RowsToLds), where the registers allow it: with 16 vectors beside
  // the weights of 16-row groups they spill (8 x 6912 -> 9000: 19.7 us, with the branches 18.5)
  constexpr bool WHOLE = RPW == 1 && (VPL <= 8 || R == 8);
  constexpr int HALVES = R / 8;                          // 8-row halves of a row group: loads per line
  constexpr int MOST = VPL * (BF16 ? 4 : 2) / KS;        // lines of 128 bytes of a wavefront's K part, at most
  constexpr int PART = MOST > 0 ? MOST * HALVES : HALVES;
  constexpr int DEEP = RPW * VPL >= 32 ? 8 : 16;         // 16-byte weight loads in flight per lane, at most
  constexpr bool LOOP = PART > DEEP;                     // longer parts rotate two register batches
  constexpr int LOADS = LOOP ? DEEP / 2 : PART;          // loads per register batch
  constexpr int LINES = LOADS / HALVES;                  // lines per register batch
  static_assert(R == 8 || R == 16, "rows of one matrix-core operand, or half of them");
  static_assert(!(FP8 && (NORM || !BF16)), "the FP8 cast takes bf16 rows as they are");
  extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [M][pitch] token codes, [16] scales; later the partial sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / KS, kh = wave % KS;
  const int K = p.K, N = p.N;
  [[maybe_unused]] const void* const all_x = p.x;  // FP8: the tensor whose maximum sets the scale
  [[maybe_unused]] const int all_rows = p.M;
  if constexpr (TILED) {
    const int first = blockIdx.y * p.tile_rows;
    p.M = all_rows - first < p.tile_rows ? all_rows - first : p.tile_rows;
    p.x = static_cast<const uint8_t*>(p.x) + (int64_t)first * K * (BF16 ? 2 : 4);
    const int64_t out = (int64_t)first * (SWI ? N >> 1 : N) * (p.y_dtype == AQ_BF16 ? 2 : 4);
    p.y = static_cast<uint8_t*>(p.y) + out;
    if (p.res) p.res = static_cast<const uint8_t*>(p.res) + out;
  }
  const int M = p.M;
  const int nline_all = (K + 127) >> 7;
  const int pitch = (nline_all << 7) + 16;  // 16 token rows then start 4 banks apart
  const int per = (nline_all + KS - 1) / KS;
  const int lbeg = kh * per, lend = lbeg + per < nline_all ? lbeg + per : nline_all;  // this wavefront's lines (none is possible)
  const int FH = SWI ? N >> 1 : N;  // outputs per token
  constexpr int GO = SWI ? GR / 2 : GR;
  const int half = SWI && grp >= GO ? FH : 0;
  const int n0 = __builtin_amdgcn_readfirstlane(half + (blockIdx.x * GO + (SWI ? grp % GO : grp)) * R);
  const int nlim = half + FH;

  // The outputs of the workgroup, GR * R weight rows of up to 16 tokens, are dealt out one to a thread (OPT of them):
  // thread t takes row t % (GR R) of token t / (GR R).  Every wavefront then requests its share of the epilogue's
  // operands; with four outputs per lane of one wavefront in KS, each wavefront sent out 20 small loads, most of them
  // empty, ahead of its weights.
  constexpr int OUT = GO * R, OPT = (OUT * 16 + GX_WAVES * 64 - 1) / (GX_WAVES * 64);
  const int tok = lane & 15;  // of the products
  const int b0 = blockIdx.x * OUT;
  float swv[OPT], bv[OPT], swg[SWI ? OPT : 1], bg[SWI ? OPT : 1], sxv = 1.0f;
  uint32_t rv[OPT];
  const EpiOperands epi(p, true, false, !SWI);
  auto load_epi = [&]() {
#pragma unroll
    for (int i = 0; i < OPT; ++i) {
      const int t = tid + i * GX_WAVES * 64;
      const int m = t / OUT, n = b0 + t % OUT;
      const bool ok = m < M && n < FH;
      swv[i] = epi.load_sw(FP8 ? 0 : n, FP8 || ok);
      bv[i] = epi.load_bias(n, ok);
      if constexpr (SWI) {
        swg[i] = epi.load_sw(FH + n, ok);
        bg[i] = epi.load_bias(FH + n, ok);
      } else {
        rv[i] = epi.load_res(m, n, ok, (int)p.ldr);
      }
    }
  };

  // weight stream: an instruction covers one line of 8 rows (lane l: row l % 8, 16-byte piece l / 8)
  const int rows = n0 < nlim ? ((nlim - n0) < R ? (nlim - n0) : R) : 0;
#ifdef AQ_LAB
  const __amdgpu_buffer_rsrc_t Wr = make_rsrc(p.wq + (int64_t)(n0 < nlim ? n0 : 0) * K, gv_skip_weights ? 0u : (uint32_t)rows * (uint32_t)K);
#else
  const __amdgpu_buffer_rsrc_t Wr = make_rsrc(p.wq + (int64_t)(n0 < nlim ? n0 : 0) * K, (uint32_t)rows * (uint32_t)K);
#endif
  const uint32_t woff = (uint32_t)(lane & 7) * (uint32_t)K, woff8 = 8u * (uint32_t)K;
  const int piece = (lane >> 3) * 16;
  uint4 wa[LOADS], wb[LOOP ? LOADS : 1];
  auto wload = [&](int line0, uint4* dst) {
#pragma unroll
    for (int t = 0; t < LINES; ++t) {
      const int kb = (line0 + t) * 128 + piece;
      const bool ok = (line0 + t) < lend && kb < K;  // past K the offset would alias the next row
      const uint32_t o = woff + (uint32_t)kb;
      dst[t * HALVES] = buffer_load_16_stream(Wr, ok ? o : OOB_OFFSET);
      if constexpr (HALVES == 2) dst[t * HALVES + 1] = buffer_load_16_stream(Wr, ok ? o + woff8 : OOB_OFFSET);
    }
  };

  float* const sx_lds = reinterpret_cast<float*>(xs + M * pitch);
  GV_STAMP(0);
  if constexpr (WPR > 0) {
    static_assert(BF16 && RPW == 1 && VPL == 4 && !NORM && !FP8 && !SWI, "attention rows");
    constexpr int VR = WPR < 4 ? 4 / WPR : 1;  // vectors of a row per lane
    const int m = wave / WPR, q = wave % WPR;
    AttnRows<VR, AQ_GEMV_ATTN_MAX_SLICES> ar;
    ar.issue(p.parts, m < M, m, K, p.parts_d, p.parts_ns, q * 64, WPR * 64, lane);
    asm volatile("" ::: "memory");  // request order: token rows, epilogue operands, the weight stream
    load_epi();
    asm volatile("" ::: "memory");
    wload(lbeg, wa);
    static_assert(!LOOP, "all weights are in flight");
    asm volatile("" ::: "memory");
    uint4 c[VR];
    ar.merge(c, m < M, K, p.parts_ns, q * 64, WPR * 64, lane);
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      float f[8];
      RowIn<true>::unpack(c[i], f);
      amax = fmaxf(amax, vec_amax<8>(f));
    }
    amax = wave_max(amax);
    if constexpr (WPR > 1) {  // the row's wavefronts
      if (lane == 0) sx_lds[8 + wave] = amax;
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();  // no memory fence: the weight loads stay in flight
      asm volatile("" ::: "memory");
#pragma unroll
      for (int w = 0; w < WPR; ++w) amax = fmaxf(amax, sx_lds[8 + m * WPR + w]);
    }
    constexpr int STEPS = quant_steps<true, false>();
    const RowScale rsc = row_scale<STEPS>(amax);
    if (lane == 0 && q == 0 && m < M) sx_lds[m] = rsc.s;
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      const int v = (i * WPR + q) * 64 + lane;
      if (m < M && v < K / 8) {
        float f[8];
        uint32_t code[2];
        RowIn<true>::unpack(c[i], f);
        quant_codes_packed<8, STEPS>(f, rsc.s, rsc.rs, rsc.fast_ok, code);
        *reinterpret_cast<uint2*>(xs + m * pitch + v * 8) = make_uint2(code[0], code[1]);
      }
    }
  } else if constexpr (BF16) {
    RowsToLds<true, RPW, VPL, WHOLE> xr;
    xr.issue(p.x, M, K, K, wave, GX_WAVES, lane);
    if constexpr (NORM) xr.issue_gamma(p.gamma, K, lane);
    asm volatile("" ::: "memory");  // request order: token rows, epilogue operands, the weight stream
    load_epi();
    asm volatile("" ::: "memory");
    wload(lbeg, wa);
    if constexpr (LOOP) wload(lbeg + LINES, wb);
    asm volatile("" ::: "memory");
    if constexpr (!FP8) {
      xr.template finish<NORM>(M, M, K, xs, pitch, sx_lds, wave, GX_WAVES, lane, p.eps);
    } else {
      float amax = 0.0f;
#pragma unroll
      for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
          float f[8];
          RowIn<true>::unpack(xr.c[j][i], f);  // rows >= M and vectors past K were loaded as zeros
          amax = fmaxf(amax, vec_amax<8>(f));
        }
      if constexpr (TILED) {  // and of the other tiles
        const uint4* const src = static_cast<const uint4*>(all_x);
        const int nv = all_rows * (K / 8);
        for (int v = tid; v < nv; v += 8 * GX_WAVES * 64) {
          uint4 t[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) t[u] = src[v + u * GX_WAVES * 64 < nv ? v + u * GX_WAVES * 64 : v];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            float f[8];
            RowIn<true>::unpack(t[u], f);
            amax = fmaxf(amax, vec_amax<8>(f));
          }
        }
      }
      amax = wave_max(amax);
      if (lane == 0) sx_lds[wave] = amax;
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();  // no memory fence: the weight loads stay in flight
      asm volatile("" ::: "memory");
      float all = 0.0f;
#pragma unroll
      for (int w = 0; w < GX_WAVES; ++w) all = fmaxf(all, sx_lds[w]);
      float sc = __fdiv_rn(all, 448.0f);
      if (all == 0.0f) sc = 1.0f;
      sxv = sc;
      const float rsc = __fdiv_rn(1.0f, sc);
      const bool lean_ok = sc >= 5.421010862427522e-20f && sc <= 1.8446744073709552e19f;  // [2^-64, 2^64]
      const int nvec = K / 8;
      auto cast = [&](const uint4& c, bool lean) {
        float f[8];
        RowIn<true>::unpack(c, f);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // x / s as in the stand-alone cast: one correction with the correctly rounded reciprocal
          float q;
          if (lean) {
            q = f[e] * rsc;
            q = __builtin_fmaf(__builtin_fmaf(-sc, q, f[e]), rsc, q);
          } else {
            q = __fdiv_rn(f[e], sc);
          }
          f[e] = fminf(fmaxf(q, -448.0f), 448.0f);
        }
        int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
        int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
        return make_uint2((uint32_t)w0, (uint32_t)w1);
      };
#pragma unroll
      for (int j = 0; j < RPW; ++j) {
        const int m = wave + j * GX_WAVES;
        if (m >= M) continue;  // uniform
        auto store = [&](int i, uint2 code) {
          if (i * 64 + lane < nvec) *reinterpret_cast<uint2*>(xs + m * pitch + (i * 64 + lane) * 8) = code;
        };
        if constexpr (WHOLE) {
          uint2 code[VPL];
          auto stretch = [&](auto from, auto to) {
            constexpr int I0 = decltype(from)::value, I1 = decltype(to)::value;
            if (__builtin_expect(lean_ok, 1)) {
#pragma unroll
              for (int i = I0; i < I1; ++i) code[i] = cast(xr.c[j][i], true);
            } else {
#pragma unroll
              for (int i = I0; i < I1; ++i) code[i] = cast(xr.c[j][i], false);
            }
#pragma unroll
            for (int i = I0; i < I1; ++i) store(i, code[i]);
          };
          // Long rows in two stretches, of which rows that fill up to 5/8 of the kernel's vectors skip the second: with one, 5 to 8 rows
          // took longer than with a branch around each vector (K up to 2560 4 %, 4097..5120 6 %; so 3 % and 5 % less than that).
          constexpr int HEAD = VPL < 8 ? VPL : VPL * 5 / 8;
          stretch(std::integral_constant<int, 0>{}, std::integral_constant<int, HEAD>{});
          if constexpr (HEAD < VPL)
            if (nvec > HEAD * 64) stretch(std::integral_constant<int, HEAD>{}, std::integral_constant<int, VPL>{});
        } else {
#pragma unroll
          for (int i = 0; i < VPL; ++i)
            if (i * 64 + lane < nvec) store(i, __builtin_expect(lean_ok, 1) ? cast(xr.c[j][i], true) : cast(xr.c[j][i], false));
        }
      }
    }
  } else {
    // fp32 rows are twice as long in registers: one row of the wavefront at a time
    {
      RowsToLds<false, 1, VPL> xr;
      xr.issue(p.x, M, K, K, wave, GX_WAVES, lane);
      asm volatile("" ::: "memory");
      load_epi();
      asm volatile("" ::: "memory");
      wload(lbeg, wa);
      if constexpr (LOOP) wload(lbeg + LINES, wb);
      asm volatile("" ::: "memory");
      xr.template finish<false>(M, M, K, xs, pitch, sx_lds, wave, GX_WAVES, lane);
    }
    if (wave + GX_WAVES < M) {
      RowsToLds<false, 1, VPL> xr;
      xr.issue(p.x, M, K, K, wave + GX_WAVES, GX_WAVES, lane);
      xr.template finish<false>(M, M, K, xs, pitch, sx_lds, wave + GX_WAVES, GX_WAVES, lane);
    }
  }
  // the rest of a last, partly filled line: products with the zeros the weight loads answer there
  for (int m = wave; m < M; m += GX_WAVES)
    if (lane * 16 < pitch - 16 - K) *reinterpret_cast<uint4*>(xs + m * pitch + K + lane * 16) = make_uint4(0, 0, 0, 0);
  GV_STAMP(3);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();  // no memory fence: the weight loads stay in flight
  asm volatile("" ::: "memory");
  GV_STAMP(4);
  float sxo[OPT];
#pragma unroll
  for (int i = 0; i < OPT; ++i) {
    const int m = (tid + i * GX_WAVES * 64) / OUT;
    sxo[i] = FP8 ? sxv : sx_lds[m < M ? m : 0];
  }

  using accv = std::conditional_t<FP8, v4f, v4i>;
  accv accs[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) accs[i] = accv{0, 0, 0, 0};
  const uint8_t* xl = xs + (tok < M ? tok : 0) * pitch + (lane >> 4) * 32;
  constexpr int ROR8 = 0x128;  // DPP row_ror:8
  constexpr int STEP = LINES < 4 ? LINES : 4;
  auto consume = [&](int line0, const uint4* wc) {
#pragma unroll
    for (int t0 = 0; t0 < LINES; t0 += STEP) {
      v4i x[2 * STEP];
#pragma unroll
      for (int t = 0; t < STEP; ++t) {
        const int ln = (line0 + t0 + t) < lend ? (line0 + t0 + t) : 0;  // lines past the end multiply zero weights
        x[2 * t] = *reinterpret_cast<const v4i*>(xl + ln * 128);
        x[2 * t + 1] = *reinterpret_cast<const v4i*>(xl + ln * 128 + 16);
      }
#pragma unroll
      for (int t = 0; t < STEP; ++t) {
        const uint4 lo = wc[(t0 + t) * HALVES];
        v4i w0, w1;
        if constexpr (HALVES == 2) {
          const uint4 hi = wc[(t0 + t) * HALVES + 1];
          // lanes 8..15 of each row take hi from lane l - 8 (w0), lanes 0..7 take lo from lane l + 8 (w1)
          w0 = v4i{__builtin_amdgcn_update_dpp((int)lo.x, (int)hi.x, ROR8, 0xf, 0xc, false),
                   __builtin_amdgcn_update_dpp((int)lo.y, (int)hi.y, ROR8, 0xf, 0xc, false),
                   __builtin_amdgcn_update_dpp((int)lo.z, (int)hi.z, ROR8, 0xf, 0xc, false),
                   __builtin_amdgcn_update_dpp((int)lo.w, (int)hi.w, ROR8, 0xf, 0xc, false)};
          w1 = v4i{__builtin_amdgcn_update_dpp((int)hi.x, (int)lo.x, ROR8, 0xf, 0x3, false),
                   __builtin_amdgcn_update_dpp((int)hi.y, (int)lo.y, ROR8, 0xf, 0x3, false),
                   __builtin_amdgcn_update_dpp((int)hi.z, (int)lo.z, ROR8, 0xf, 0x3, false),
                   __builtin_amdgcn_update_dpp((int)hi.w, (int)lo.w, ROR8, 0xf, 0x3, false)};
        } else {
          // the operand's rows 8..15 repeat other pieces of rows 0..7: their products are never stored
          w0 = v4i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w};
          w1 = v4i{__builtin_amdgcn_update_dpp(0, (int)lo.x, ROR8, 0xf, 0xf, false),
                   __builtin_amdgcn_update_dpp(0, (int)lo.y, ROR8, 0xf, 0xf, false),
                   __builtin_amdgcn_update_dpp(0, (int)lo.z, ROR8, 0xf, 0xf, false),
                   __builtin_amdgcn_update_dpp(0, (int)lo.w, ROR8, 0xf, 0xf, false)};
        }
        if constexpr (!FP8) {
          accs[(2 * t) & 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, x[2 * t], accs[(2 * t) & 3], 0, 0, 0);
          accs[(2 * t + 1) & 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, x[2 * t + 1], accs[(2 * t + 1) & 3], 0, 0, 0);
        } else {
          const v8i wl = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
          const v4i xa = x[2 * t], xb = x[2 * t + 1];
          const v8i xl8 = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
          accs[t & 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wl, xl8, accs[t & 3], 0, 0, 0, 0, 0, 0);
        }
      }
    }
  };
  if constexpr (!LOOP) {
    consume(lbeg, wa);
  } else {
    for (int l0 = lbeg; l0 < lend; l0 += 2 * LINES) {
      consume(l0, wa);
      if (l0 + 2 * LINES < lend) wload(l0 + 2 * LINES, wa);
      if (l0 + LINES < lend) consume(l0 + LINES, wb);
      if (l0 + 3 * LINES < lend) wload(l0 + 3 * LINES, wb);
    }
  }
  const accv acc = (accs[0] + accs[1]) + (accs[2] + accs[3]);
  GV_STAMP(5);
  // the K parts' sums meet in LDS: [K part][token][row of the workgroup]
  __syncthreads();  // everyone is done reading the token codes: the buffer is reused
  using acct = std::conditional_t<FP8, float, int>;
  acct* const part = reinterpret_cast<acct*>(xs);
  if (R == 16 || lane < 32)
    *reinterpret_cast<accv*>(part + (kh * 16 + tok) * (GR * R) + grp * R + (lane >> 4) * 4) = acc;  // lane: 4 rows of a token
  __syncthreads();
#pragma unroll
  for (int i = 0; i < OPT; ++i) {
    const int t = tid + i * GX_WAVES * 64;
    const int m = t / OUT, n = b0 + t % OUT;
    if (m >= M || n >= FH) continue;
    const acct* const mine = part + m * (GR * R) + t % OUT;
    acct sum = mine[0];
#pragma unroll
    for (int k = 1; k < KS; ++k) sum += mine[k * 16 * GR * R];  // fp32: a fixed order
    float y = __fmul_rn(__fmul_rn((float)sum, sxo[i]), swv[i]);
    if (p.bias) y = __fadd_rn(y, bv[i]);
    if constexpr (SWI) {
      acct gsum = mine[OUT];
#pragma unroll
      for (int k = 1; k < KS; ++k) gsum += mine[k * 16 * GR * R + OUT];
      float g = __fmul_rn(__fmul_rn((float)gsum, sxo[i]), swg[i]);
      if (p.bias) g = __fadd_rn(g, bg[i]);
      if (p.y_dtype == AQ_BF16) {  // as the two projections would be stored
        y = bf16_bits_to_f32(f32_to_bf16_bits(y));
        g = bf16_bits_to_f32(f32_to_bf16_bits(g));
      }
      y = swiglu_repro(y, g);
    } else if (p.res) y = p.y_dtype == AQ_BF16 ? add_residual_bf16(y, rv[i]) : __fadd_rn(y, __uint_as_float(rv[i]));
    const int64_t o = (int64_t)m * FH + n;
    if (p.y_dtype == AQ_BF16)
      reinterpret_cast<uint16_t*>(p.y)[o] = (uint16_t)f32_to_bf16_bits(y);
    else
      reinterpret_cast<float*>(p.y)[o] = y;
  }
  GV_STAMP(6);
}

static size_t gemv_rows_lds(int64_t M, int64_t K, int ks, int rows_per_wg) {
  const size_t codes = (size_t)M * (((K + 127) / 128) * 128 + 16) + 16 * sizeof(float);
  const size_t sums = (size_t)ks * 16 * rows_per_wg * 4;  // come to lie over the codes
  return codes < sums ? sums : codes;
}

// Weight rows per workgroup: the fewest rounds of workgroups over the compute units x what a workgroup takes.  Rows of more
// than 2048 take 130 to 240 registers: one workgroup to a unit, every round begins with the latency of its rows and rounds them
// again, 8 M + 4 r + 64 quarters of a weight row (`alone`: rows with the norm, too).  Shorter rows as they are, of SwiGLU as well, take
// 50 to 90: two or three workgroups share a unit, a round starts under the one before, 5 M + 4 r + 12.  Fitted to 10 600 random sizes
// (N 512..11264, K 512..8192, 1 to 16 rows, attention rows too).  us, with 7 M + 4 r for all -> so: fp32 2 x 2592 -> 8352 23.2 -> 11.0,
// 1 x 6864 -> 4352 18.7 -> 14.1; FP8 1 x 4576 -> 9696 27.0 -> 16.7, 2 x 4816 -> 4560 17.1 -> 11.6, 1 x 512 -> 4848 4.08 -> 3.62; int8 3 x 3328 ->
// 10720 11.4 -> 9.8; norm 3 x 1408 -> 9408 6.7 -> 6.0; norm and SwiGLU 14 x 2048 -> 2 x 8416 18.5 -> 17.0.  With the larger cost for short
// rows 3 x 864 -> 10832 4.55 -> 5.08, SwiGLU without the norm 13 x 1536 -> 2 x 8272 9.7 -> 13.2 (959 sizes of it: up to 33 % from the
// better of its two, so 3 %).
static int rows_per_workgroup(int64_t M, int64_t N, bool alone, int least, int most) {
  const int64_t cus = device_cus(), fixed = alone ? 8 * M + 64 : 5 * M + 12;
  int best = most;
  int64_t cost = INT64_MAX;
  for (int r = least; r <= most; r *= 2) {
    const int64_t c = ((N + r - 1) / r + cus - 1) / cus * (fixed + 4 * r);
    if (c < cost) cost = c, best = r;
  }
  return best;
}

using rows_kernel_t = void (*)(GemvArgs);

static int launch_rows(rows_kernel_t fn, LdsOptIn& opted, const GemvArgs& a, int ks, int rows_per_wg, int64_t outputs, int outputs_per_wg,
                       hipStream_t st) {
  const size_t lds = gemv_rows_lds(a.tile_rows ? a.tile_rows : a.M, a.K, ks, rows_per_wg);
  if (lds > 64 * 1024) {
    const int e = opted.ensure(reinterpret_cast<const void*>(fn));
    if (e) return e;
  }
  const unsigned grid = (unsigned)((outputs + outputs_per_wg - 1) / outputs_per_wg);
  const unsigned tiles = a.tile_rows ? (unsigned)((a.M + a.tile_rows - 1) / a.tile_rows) : 1u;
  aq::queue_kernel(fn, dim3(grid, tiles), dim3(GX_WAVES * 64), lds, st, a);
  return (int)hipGetLastError();
}

// the row length class: vectors per lane of a row, rounded up to what kernels are built for
static int length_class(int64_t vectors) { return vectors <= 128 ? 0 : vectors <= 256 ? 1 : vectors <= 512 ? 2 : 3; }

template <int KS, int R, bool TILED>
static int launch_shape(const GemvArgs& a, RowsKind kind, hipStream_t st) {
#define AQ_GX(BF16, RPW, VPL, NORM, FP8) gemv_rows_kernel<KS, R, BF16, RPW, VPL, NORM, FP8, false, 0, TILED>
  static const rows_kernel_t i8[2][4] = {
      {AQ_GX(true, 1, 2, false, false), AQ_GX(true, 1, 4, false, false), AQ_GX(true, 1, 8, false, false),
       TILED ? nullptr : gemv_rows_kernel<KS, R, true, 1, 16, false, false>},
      {AQ_GX(true, 2, 2, false, false), AQ_GX(true, 2, 4, false, false), AQ_GX(true, 2, 8, false, false),
       TILED ? nullptr : gemv_rows_kernel<KS, R, true, 2, 16, false, false>}};  // (tiles: up to 4096)
  // (16 rows of more than 4096 cannot stay in registers between the tensor's maximum and the cast: gemv_rows_ok; tiles: up to 2048)
  static const rows_kernel_t f8[2][4] = {
      {AQ_GX(true, 1, 2, false, true), AQ_GX(true, 1, 4, false, true), TILED ? nullptr : gemv_rows_kernel<KS, R, true, 1, 8, false, true>,
       TILED ? nullptr : gemv_rows_kernel<KS, R, true, 1, 16, false, true>},
      {AQ_GX(true, 2, 2, false, true), AQ_GX(true, 2, 4, false, true), TILED ? nullptr : gemv_rows_kernel<KS, R, true, 2, 8, false, true>, nullptr}};
  static const rows_kernel_t norm[2][2] = {{AQ_GX(true, 1, 2, true, false), AQ_GX(true, 1, 4, true, false)},
                                           {AQ_GX(true, 2, 2, true, false), AQ_GX(true, 2, 4, true, false)}};
  static const rows_kernel_t f32[3] = {AQ_GX(false, 1, 4, false, false), AQ_GX(false, 1, 8, false, false), AQ_GX(false, 1, 32, false, false)};
#undef AQ_GX
  static LdsOptIn opted[2][4][4];
  const int two = (TILED ? a.tile_rows : a.M) > 8, len = length_class(a.K / (kind == ROWS_I8_F32 ? 4 : 8));
  const int flen = a.K <= 1024 ? 0 : a.K <= 2048 ? 1 : 2;
  const rows_kernel_t fn = kind == ROWS_I8_F32    ? f32[flen]
                           : kind == ROWS_I8_NORM ? norm[two][len]
                           : kind == ROWS_FP8     ? f8[two][len]
                                                  : i8[two][len];
  return launch_rows(fn, opted[two][kind][kind == ROWS_I8_F32 ? flen : len], a, KS, GX_WAVES / KS * R, a.N, GX_WAVES / KS * R, st);
}

bool gemv_rows_ok(RowsKind kind, int64_t M, int64_t K) {
  if (M < 1 || M > 16 || K > GX_MAX_K) return false;
  if (kind == ROWS_I8_NORM) return K <= 2048;      // the gain's vectors stay in registers next to the rows'
  if (kind == ROWS_FP8) return M <= 8 || K <= 4096;
  return true;
}

// Rows of up to 2048 and so many outputs that the rounds run into each other: 32 weight rows, 0 to 0.5 % from the best of the four
// (2900 sizes up to 64 K outputs; by cost the last round decides, up to 38 % wrong).  Not 9 and more rows with the norm, whose
// workgroups are alone, nor 1 to 4 fp32 rows (4 x 1536 -> 20184 8.9 with 16, 10.3 with 32).  us, by cost -> so: 15 x 1472 -> 38250 21.8
// -> 16.7, norm 3 x 1392 -> 35618 17.4 -> 13.9.
static bool rounds_merge(const GemvArgs& a, bool norm) {
  return a.K <= 2048 && a.N > (a.K > 1024 ? 64 : 128) * device_cus() && !(a.M > 8 && (norm || a.K <= 1024));
}

// More than 16 rows: tiles of 9..16 or of up to 8 rows, each with its own workgroups over the weight rows.  Every tile reads the
// weights and every workgroup rounds its tile's rows again, so it is the faster form while tiles x outputs x row length is small:
// one launch then stands for the quantiser's and the GEMM's (FP8: the maximum's, the cast's and the GEMM's), 3.3 to 5 us of which are
// launches and first requests.  Both ways as fitted to 4093 random sizes of 17 to 200 rows, us (K in units of 1024; `length`: the row
// length class, whose vectors are requested whether the row has them or not):
//   tiles      start + rounds over the compute units x (row x tile rows x length + weight x weight rows x K + all x M x K)
//   launches   two[0] + two[1] K + two[2] M N K / 10^6 + (more than one tile of 32 x 32 per unit: two[3]) + two[4] N K / 10^4, FP8 + 1.5 M K / 65536
// us from a graph, launches -> tiles, weights in the last-level cache | from HBM: bf16 32 x 2048 -> 2048 5.7 -> 4.8 | 6.7 -> 5.1, 64 x 1024 -> 3072 6.1 -> 4.7 |
// 6.9 -> 5.0, 32 x 512 -> 8192 5.5 -> 4.6 | 6.4 -> 4.8, fp32 64 x 512 -> 2048 5.2 -> 4.2 | 5.8 -> 4.6.
//
// A call on its own pays 2.4 us of the host's time for a launch, 8 us in all for two: tiles of less than that (7.5) are taken up to 5 %
// behind (TILED_ALONE): fp32 64 x 2048 -> 2048 8.1 -> 7.1, int8 181 x 1360 -> 416 8.4 -> 6.0, FP8 19 x 720 -> 6000 8.9 -> 6.7.  In a graph, or
// among a block's launches, the host's time is not what counts, and there the tiles have to be ahead by 5 %, fp32 rows, whose cost the fit
// misses by most, by 8 % (TILED).  1380 sizes drawn from 17..200 rows, both ways from a graph, slower by more than 3 % with the tiles, cache and
// HBM together: by the line for a call on its own int8 rows at 4 of 220 (at worst 1.25 | 1.26: 125 x 1216 -> 1824), with the norm 3 of 220 (1.33 |
// 1.21), fp32 rows 16 of 720 (1.25 | 1.19; 64 x 2048 -> 2048 6.4 -> 6.9 | 8.1 -> 7.8); by these none, none and one (1.05).  FP8 at none of 220 (at
// worst 1.05 | 1.03), and so its line, on which the order of its sums depends, is one for all calls.
struct TiledCost {
  double start, row, weight, all, two[5];
};
static const TiledCost& tiled_cost(RowsKind kind) {
  static const TiledCost i8 = {3.07, 0.038, 0.038, 0, {5.27, 0.27, 4.1, 0.47, 0.79}}, norm = {3.24, 0.083, 0.033, 0, {5.49, 0.44, 4.78, 0.35, 1.38}},
                         f32 = {3.26, 0.041, 0.042, 0, {4.74, 0.79, 4.33, 0.47, 0.92}}, f8 = {3.81, 0.054, 0.047, 0.018, {5.35, 0.23, 4.11, 0.4, 1.14}};
  return kind == ROWS_I8 ? i8 : kind == ROWS_I8_NORM ? norm : kind == ROWS_I8_F32 ? f32 : f8;
}
struct Tiled {
  int tile_rows, weight_rows;
  double us;
};
static Tiled tiled_best(RowsKind kind, int64_t M, int64_t N, int64_t K) {
  const TiledCost& c = tiled_cost(kind);
  const double k = (double)K / 1024, length = K <= 1024 ? 1 : K <= 2048 ? 2 : kind == ROWS_I8_F32 ? 11.2 : 4;
  const int64_t cus = device_cus();
  Tiled best = {0, 0, 1e30};
  for (int most = 8; most <= 16; most += 8) {
    const int64_t tiles = (M + most - 1) / most, rows = (M + tiles - 1) / tiles;
    for (int r = 16; r <= 64; r *= 2) {
      const double us = c.start + (double)(((N + r - 1) / r * tiles + cus - 1) / cus) * (c.row * rows * length + c.weight * r * k + c.all * M * k);
      if (us < best.us) best = {(int)rows, r, us};
    }
  }
  return best;
}
Tiling gemv_rows_tiled(RowsKind kind, int64_t M, int64_t N, int64_t K) {
  // Tiles of more outputs than 80 to a compute unit never gained (64 x 512 -> 8192: 6.3 | 6.6), nor longer bf16 rows than 4096 (FP8: 2048).
  const int64_t most = kind == ROWS_I8_NORM || kind == ROWS_FP8 ? 2048 : kind == ROWS_I8_F32 ? GX_MAX_K : 4096;
  if (M <= 16 || (M + 15) / 16 * N > 80 * device_cus() || K > most) return TILED_NOT;
  const double* two = tiled_cost(kind).two;
  const double k = (double)K / 1024, nk = (double)N * k;
  const bool rounds = (M + 31) / 32 * ((N + 31) / 32) > device_cus();
  const double cast = kind == ROWS_FP8 ? 1.5 * (double)(M * K < 98304 ? M * K : 98304) / 65536 : 0;  // by the tensor's size, up to where it takes two launches
  const double us = tiled_best(kind, M, N, K).us, by_two = two[0] + cast + two[1] * k + two[2] * M * nk / 1e6 + (rounds ? two[3] : 0) + two[4] * nk / 1e4;
  const double ahead = kind == ROWS_FP8 ? (us < 7.5 ? 1.05 : 0.95) : kind == ROWS_I8_F32 ? 0.92 : 0.95;
  return us < ahead * by_two ? TILED : us < (us < 7.5 ? 1.05 : 0.95) * by_two ? TILED_ALONE : TILED_NOT;
}

// Two exceptions, 2200 sizes with weights from HBM:
// * 1 to 4 bf16 rows of 3073 to 4096, where 64-row workgroups would be a round of which at most 5/8 of the units have one: five rounds
//   of 8-row workgroups overlap enough.  us, 64 -> 8: FP8 2 x 3824 -> 8896 14.6 -> 12.7, 1 x 3440 -> 8864 13.4 -> 12.0, int8 1 x 3440 -> 10128 12.9
//   -> 11.4; not 1 x 2864 -> 10160 (11.2 | 11.5), nor with six rounds (FP8 3 x 3504 -> 11000 13.1 | 14.0).
// * 1 to 4 fp32 rows of 1025 to 2048, whose rounds overlap the less the larger they are: 16 at most, 1 x 1424 -> 4128 4.7 -> 4.2 (in the
//   mean 1.6 % from the best of the four, so 0.8 %).
int launch_gemv_rows(const GemvArgs& a, RowsKind kind, hipStream_t st) {
  const bool few = a.M <= 4, f32 = kind == ROWS_I8_F32, norm = kind == ROWS_I8_NORM;
  if (a.M > 16) {
    const Tiled best = tiled_best(kind, a.M, a.N, a.K);
    GemvArgs t = a;
    t.tile_rows = best.tile_rows;
    switch (best.weight_rows) {
      case 16: return launch_shape<8, 16, true>(t, kind, st);
      case 32: return launch_shape<4, 16, true>(t, kind, st);
      default: return launch_shape<2, 16, true>(t, kind, st);
    }
  }
  int rows = 32;
  if (!rounds_merge(a, norm) || (f32 && (few || a.K <= 1024))) {
    rows = rows_per_workgroup(a.M, a.N, norm || a.K > 2048, 8, few && f32 && a.K > 1024 && a.K <= 2048 ? 16 : 64);
    if (rows == 64 && few && !f32 && a.K > 3072 && a.K <= 4096 && a.N <= 5 * 8 * device_cus()) rows = 8;
  }
  switch (rows) {
    case 8: return launch_shape<8, 8, false>(a, kind, st);
    case 16: return launch_shape<8, 16, false>(a, kind, st);
    case 32: return launch_shape<4, 16, false>(a, kind, st);
    default: return launch_shape<2, 16, false>(a, kind, st);
  }
}

// a.N = 2 F; K <= 2048
int launch_gemv_rows_swiglu(const GemvArgs& a, hipStream_t st) {
#define AQ_GX(KS, RPW, NORM) \
  {gemv_rows_kernel<KS, 16, true, RPW, 2, NORM, false, true>, gemv_rows_kernel<KS, 16, true, RPW, 4, NORM, false, true>}
#define AQ_GX2(KS) {{AQ_GX(KS, 1, false), AQ_GX(KS, 1, true)}, {AQ_GX(KS, 2, false), AQ_GX(KS, 2, true)}}
  static const rows_kernel_t table[2][2][2][2] = {AQ_GX2(4), AQ_GX2(2)};
#undef AQ_GX2
#undef AQ_GX
  static LdsOptIn unused;  // rows of at most 2048: never more than 64 KiB
  const bool norm = a.gamma != nullptr;
  const int r = a.K > 1024 && rounds_merge(a, norm) ? 32 : rows_per_workgroup(a.M, a.N, norm, 32, 64);
  return launch_rows(table[r == 64][a.M > 8][a.gamma != nullptr][a.K > 1024], unused, a, r == 64 ? 2 : 4, r, a.N / 2, r / 2, st);
}

// Rows from a.parts: M <= 8, K <= 2048.
int launch_gemv_rows_attn(const GemvArgs& a, hipStream_t st) {
#define AQ_GX(KS, R)                                                                                                             \
  {gemv_rows_kernel<KS, R, true, 1, 4, false, false, false, 8>, gemv_rows_kernel<KS, R, true, 1, 4, false, false, false, 4>,     \
   gemv_rows_kernel<KS, R, true, 1, 4, false, false, false, 2>, gemv_rows_kernel<KS, R, true, 1, 4, false, false, false, 1>}
  static const rows_kernel_t table[4][4] = {AQ_GX(8, 8), AQ_GX(8, 16), AQ_GX(4, 16), AQ_GX(2, 16)};
#undef AQ_GX
  static LdsOptIn unused;  // 8 rows of at most 2048: never more than 64 KiB
  // 3 or 4 rows of up to 1024 in 2 or 3 slices: 16 weight rows at least, us with 8 -> 16: 3 x 704 -> 704 4.10 -> 3.65, 4 x 256 -> 1056
  // 4.05 -> 3.64, 3 x 960 -> 544 4.10 -> 4.23 (level at 4 slices; 2 and 5 to 8 rows 2 % slower with 16)
  const bool few_bytes = (a.M == 3 || a.M == 4) && a.K <= 1024 && a.parts_ns < 4;
  const int rows = rows_per_workgroup(a.M, a.N, false, few_bytes ? 16 : 8, 64);
  const int shape = rows == 8 ? 0 : rows == 16 ? 1 : rows == 32 ? 2 : 3;
  const int wpr = a.M <= 1 ? 0 : a.M <= 2 ? 1 : a.M <= 4 ? 2 : 3;
  return launch_rows(table[shape][wpr], unused, a, shape < 2 ? 8 : shape == 2 ? 4 : 2, rows, a.N, rows, st);
}

}  // namespace aq

#ifdef AQ_LAB
// Lab build only (see aq_lab.h).
extern "C" int aq_lab_set_gemv_timeline(long long* buf) {
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(aq::gv_timeline), &buf, sizeof(buf));
}
extern "C" int aq_lab_set_gemv_skip_weights(int on) {
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(aq::gv_skip_weights), &on, sizeof(on));
}
#endif
