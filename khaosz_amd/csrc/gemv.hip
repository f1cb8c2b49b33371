// Decode path (M <= 16 tokens): a weight-streaming int8 GEMV.  The weight
// matrix is read exactly once with 16-byte loads, one wavefront reading 1 KiB
// contiguous of a row per instruction; the few activation rows come as codes
// (the caller's, or the row-wise kernel's in the caller's workspace), pulled into
// LDS once per workgroup by direct global->LDS loads and reused by every row of W,
// or are quantised by the workgroup itself (FUSED: up to 4 bf16 rows; more rows,
// fp32 and FP8 ones take gemv_rows.hip, see gemv_dispatch_fused).
// Products are v_dot4_i32_i8 (no MFMA tiles, no LDS staging of W); a wavefront
// reduces its 4 x MT partial sums with a transposed butterfly so that each
// lane ends up owning one output, then applies the same dequantising epilogue
// as the MFMA GEMM.  The int32 sums are exact, so the result is bit-identical
// to quantise + GEMM.
//
// Every byte the kernel will need is requested before anything is waited for:
// a wavefront first issues its share of the activation copy, then the weight
// loads of its first two K chunks, and only then waits for the activations.
#include <type_traits>

#include "aq_common.h"
#include "aq_gemm.h"
#include "aq_gemv.h"
#include "aq_rows.h"

namespace aq {

#ifndef AQ_GV_ROWS
#define AQ_GV_ROWS 4
#endif
#ifndef AQ_GV_WAVES
#define AQ_GV_WAVES 8
#endif
constexpr int GV_ROWS = AQ_GV_ROWS;    // weight rows per wavefront pass
constexpr int GV_WAVES = AQ_GV_WAVES;  // wavefronts per workgroup
constexpr int GV_THREADS = GV_WAVES * 64;
constexpr int GV_CHUNK = 64 * 16;  // K bytes one wavefront covers per load
constexpr int GV_DEPTH = 2;        // weight chunks in flight per wavefront

typedef __attribute__((address_space(3))) void gv_lds_void;
typedef unsigned gv_u2 __attribute__((ext_vector_type(2)));

// Reduce V values per lane across the 64 lanes so that afterwards v[0] of lane
// l holds the full sum of value index l >> (6 - log2 V) (for V <= 64).
// Lane-bit 5 and 4 stages use the gfx950 half/row swaps: one swap exchanges the
// two halves a pair of values needs, one add finishes it.  The remaining
// stages (at most 15 live values for V = 64) add across a row by DPP: lanes
// l ^ 8, then 7 - l of a half row, which differs from l in bit 2 and reaches
// the same 8 lanes together with l ^ 2 and l ^ 1 (as shuffles through LDS, four
// round trips one after the other, 1 x 2048 -> 8192 took 4.81 us; 4.65).
template <int CUR, int OFF>
struct Butterfly {
  static constexpr int DPP = OFF == 8 ? 0x128 : OFF == 4 ? 0x141 : OFF == 2 ? 0x4E : 0xB1;  // row_ror:8, row_half_mirror, quad_perm x 2
  template <int V>
  __device__ static __forceinline__ void run(int (&v)[V], int lane) {
    if constexpr (CUR > 1) {
      constexpr int H = CUR / 2;
      if constexpr (OFF == 32 || OFF == 16) {
#pragma unroll
        for (int i = 0; i < H; ++i) {
          const gv_u2 r = OFF == 32 ? __builtin_amdgcn_permlane32_swap((unsigned)v[i], (unsigned)v[i + H], false, false)
                                    : __builtin_amdgcn_permlane16_swap((unsigned)v[i], (unsigned)v[i + H], false, false);
          v[i] = (int)(r.x + r.y);
        }
      } else {
        const bool up = (lane & OFF) != 0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
          const int lo = v[i], hi = v[i + H];
          const int send = up ? lo : hi;
          const int keep = up ? hi : lo;
          v[i] = keep + __builtin_amdgcn_update_dpp(0, send, DPP, 0xf, 0xf, false);
        }
      }
      if constexpr (OFF > 1) Butterfly<H, OFF / 2>::run(v, lane);
    } else {
      if constexpr (OFF >= 16) {
        const gv_u2 r = OFF == 32 ? __builtin_amdgcn_permlane32_swap((unsigned)v[0], (unsigned)v[0], false, false)
                                  : __builtin_amdgcn_permlane16_swap((unsigned)v[0], (unsigned)v[0], false, false);
        v[0] = (int)(r.x + r.y);
      } else {
        v[0] += __builtin_amdgcn_update_dpp(0, v[0], DPP, 0xf, 0xf, false);
      }
      if constexpr (OFF > 1) Butterfly<1, OFF / 2>::run(v, lane);
    }
  }
};

constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v / 2); }

// FUSED: the kernel quantises the bf16 activation rows itself (VPL 16-byte vectors
// per lane per row) instead of copying codes a separate launch produced.
// Wavefronts per workgroup: GV_WAVES for the fused kernels (they split the row
// quantisation among them: with fewer, each would round several rows one after
// the other before any product can start), taken from the launch otherwise.  A
// workgroup covers GV_ROWS * wavefronts weight rows; the launcher shrinks it
// when N is too small for 8-wavefront workgroups to reach every compute unit.
// NORM (with FUSED): the rows are RMS-normalised with the gain p.gamma before they are quantised.
// FW: wavefronts per workgroup of a FUSED kernel (8, or 4 for short matrices).
// FK: K parts of a FUSED kernel (1; 4 for a short matrix with long rows, an MLP's down projection: every wavefront
// still rounds a row, then FK wavefronts share a group of weight rows, so that the launch has a workgroup for
// every compute unit where whole rows per wavefront would leave most of them without loads in flight).
template <int MT, bool FUSED, int VPL, bool NORM = false, int FW = GV_WAVES, int FK = 1>
__global__ __launch_bounds__(GV_THREADS) void gemv_w8a8_kernel(GemvArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [MT][K] activation codes, then [MT] scales
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = p.K, N = p.N, M = p.M;
  // wavefront-uniform first row, kept scalar so the buffer descriptor lives in SGPRs
  constexpr int WAVES = FUSED ? FW : GV_WAVES;
  const int nwaves = FUSED ? WAVES : (int)(blockDim.x >> 6);
  // K parts: ksplit wavefronts share a group of GV_ROWS rows, wavefront kpart taking chunks kpart,
  // kpart + ksplit, ...; their sums meet in LDS (exact int32).  For short N and long K, where whole rows per
  // wavefront would leave most of the device without loads in flight.
  const int ksplit = FUSED ? FK : p.ksplit;
  const int kpart = wave % ksplit;
  const int n0 = __builtin_amdgcn_readfirstlane((blockIdx.x * (nwaves / ksplit) + wave / ksplit) * GV_ROWS);

  // 0. After the reduction lane l owns output (row n0 + idx / MT, token idx % MT)
  // with idx = l >> (6 - log2(rows * MT)).  Its scales and bias are requested
  // ahead of the weight stream, so the epilogue never waits on memory, but behind
  // the activation rows (step 1): loads return in request order, and these lines,
  // which no other workgroup shares, come from HBM while the rows come from cache.
  constexpr int V = GV_ROWS * MT;
  constexpr int SH = 6 - ilog2(V);
  static_assert(V <= 64, "one output per lane at most");
  const int oidx = lane >> SH;
  const int om = oidx % MT, on = n0 + oidx / MT;
  const bool out_lane = (lane & ((1 << SH) - 1)) == 0 && om < M && on < N;
  float* sx_lds = reinterpret_cast<float*>(xs + MT * K);
  const EpiOperands epi(p, true, !FUSED, true);
  float sxv = 0.0f, swv, bv;
  uint32_t rv;  // residual element, raw bits
  auto load_epi = [&]() {
    sxv = epi.load_sx(om, out_lane);
    swv = epi.load_sw(on, out_lane);
    bv = epi.load_bias(on, out_lane);
    rv = epi.load_res(om, on, out_lane, (int)p.ldr);
  };
  // (the copy of ready-made codes goes straight to LDS and is waited for by counting the requests behind it:
  // there the operands stay in front)
  if constexpr (!FUSED) load_epi();

  // 1. activation codes -> LDS.  Either copied, 16 bytes per lane, straight from
  // global memory (rows m >= M lie outside the descriptor and arrive as zeros),
  // or produced here: each wavefront requests its rows of the bf16 activation now
  // and quantises them while the weight loads queued behind are in flight.
  constexpr int RPW = FUSED ? (MT + WAVES - 1) / WAVES : 1;
  RowsToLds<true, RPW, VPL> xrows;
  if constexpr (FUSED) {
    xrows.issue(p.x, M, K, K, wave, WAVES, lane);
    if constexpr (NORM) xrows.issue_gamma(p.gamma, K, lane);
  } else {
    const __amdgpu_buffer_rsrc_t Xr = make_rsrc(p.xq, (uint32_t)M * (uint32_t)K);
    const int xbytes = MT * K;
    const int xrounds = (xbytes + nwaves * 1024 - 1) / (nwaves * 1024);
    for (int r = 0; r < xrounds; ++r) {
      const int base = (r * nwaves + wave) * 1024;  // this wavefront's 1 KiB of the copy
      if (base < xbytes)  // uniform; xbytes is a multiple of 16 but not always of 1024:
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            Xr, (gv_lds_void*)(xs + base), 16,
            (base + lane * 16) < xbytes ? (uint32_t)(base + lane * 16) : OOB_OFFSET, 0, 0, 0);
    }
  }

  asm volatile("" ::: "memory");  // request order: activation rows, epilogue operands, the weight stream
  if constexpr (FUSED) load_epi();
  asm volatile("" ::: "memory");

  // 2. the first GV_DEPTH weight chunks of this wavefront's rows.  The
  // descriptor spans these rows only; rows past N and bytes past K fall
  // outside it and read as zero.
  const int nchunk_all = (K + GV_CHUNK - 1) / GV_CHUNK;
  const int nchunk = (nchunk_all - kpart + ksplit - 1) / ksplit;  // this wavefront's chunks (0 is possible)
  const int rows = n0 < N ? ((N - n0) < GV_ROWS ? (N - n0) : GV_ROWS) : 0;
  const __amdgpu_buffer_rsrc_t Wr =
      make_rsrc(p.wq + (int64_t)(n0 < N ? n0 : 0) * K, (uint32_t)rows * (uint32_t)K);
  auto wload = [&](int c, uint4 (&dst)[GV_ROWS]) {
    const int kb = (kpart + c * ksplit) * GV_CHUNK + lane * 16;
    const bool ok = kb < K;  // past K the offset would alias the next row
#pragma unroll
    for (int r = 0; r < GV_ROWS; ++r)
      dst[r] = GV_WLOAD(Wr, ok ? (uint32_t)r * (uint32_t)K + (uint32_t)kb : OOB_OFFSET);
  };
  uint4 w[GV_DEPTH][GV_ROWS];
#pragma unroll
  for (int d = 0; d < GV_DEPTH; ++d) wload(d, w[d]);  // chunks past the end read zeros

  // 3. the activation requests are older than the weight loads: wait until at
  // most those are outstanding (the fused path's own use of the rows makes the
  // compiler place that wait), then make every wavefront's part visible through
  // a barrier that does not drain the weight loads.
  if constexpr (FUSED) {
    xrows.template finish<NORM>(M, MT, K, xs, K, sx_lds, wave, WAVES, lane, p.eps);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's LDS writes are done
  } else {
    GV_WAIT_VMCNT(GV_DEPTH * GV_ROWS);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (FUSED) {
    if (out_lane) sxv = sx_lds[om];
  }

  int acc[GV_ROWS * MT];
#pragma unroll
  for (int i = 0; i < GV_ROWS * MT; ++i) acc[i] = 0;

  auto consume = [&](int c, const uint4 (&wc)[GV_ROWS]) {
    const int kb = (kpart + c * ksplit) * GV_CHUNK + lane * 16;
    const int kx = kb < K ? kb : 0;  // lanes past the end multiply zeros; keep the LDS read in range
    // activation rows in blocks of 4: four LDS reads in flight cover the 64 dot
    // products of the previous block without holding all MT rows in registers
    constexpr int MB = MT < 4 ? MT : 4;
#pragma unroll
    for (int m0 = 0; m0 < MT; m0 += MB) {
      uint4 x[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) x[i] = *reinterpret_cast<const uint4*>(xs + (m0 + i) * K + kx);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
#pragma unroll
        for (int r = 0; r < GV_ROWS; ++r) {
          int a = acc[r * MT + m0 + i];
          a = __builtin_amdgcn_sdot4((int)wc[r].x, (int)x[i].x, a, false);
          a = __builtin_amdgcn_sdot4((int)wc[r].y, (int)x[i].y, a, false);
          a = __builtin_amdgcn_sdot4((int)wc[r].z, (int)x[i].z, a, false);
          a = __builtin_amdgcn_sdot4((int)wc[r].w, (int)x[i].w, a, false);
          acc[r * MT + m0 + i] = a;
        }
      }
      if constexpr (MT > 8) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // K loop.  Rows of up to 2 KiB (the common decode shapes) are two chunks that
  // are already in flight: no loop.  Longer rows rotate two register buffers.
  static_assert(GV_DEPTH == 2, "the K loop below rotates exactly two buffers");
  consume(0, w[0]);
  if (nchunk > 2) wload(2, w[0]);
  __builtin_amdgcn_sched_barrier(0);
  if (nchunk > 1) consume(1, w[1]);
  for (int c = 2; c < nchunk; c += 2) {
    if (c + 1 < nchunk) wload(c + 1, w[1]);
    __builtin_amdgcn_sched_barrier(0);
    consume(c, w[0]);
    if (c + 2 < nchunk) wload(c + 2, w[0]);
    __builtin_amdgcn_sched_barrier(0);
    if (c + 1 < nchunk) consume(c + 1, w[1]);
  }

  Butterfly<V, 32>::run(acc, lane);
  if (ksplit > 1) {  // uniform over the workgroup
    int* part = reinterpret_cast<int*>(sx_lds + MT);  // [wavefront][lane]
    if (kpart != 0) part[wave * 64 + lane] = acc[0];
    __syncthreads();
    if (kpart != 0) return;
    for (int k = 1; k < ksplit; ++k) acc[0] += part[(wave + k) * 64 + lane];
  }
  if (!out_lane) return;
  float y = __fmul_rn(__fmul_rn((float)acc[0], sxv), swv);
  if (p.bias) y = __fadd_rn(y, bv);
  if (p.res) y = p.y_dtype == AQ_BF16 ? add_residual_bf16(y, rv) : __fadd_rn(y, __uint_as_float(rv));
  const int64_t o = (int64_t)om * N + on;
  if (p.y_dtype == AQ_BF16)
    reinterpret_cast<uint16_t*>(p.y)[o] = (uint16_t)f32_to_bf16_bits(y);
  else
    reinterpret_cast<float*>(p.y)[o] = y;
}

// Shape of a launch for N weight rows of K bytes.  Whole rows per wavefront, 8 wavefronts per workgroup,
// halved (down to 2) while the launch would have fewer workgroups than the device has compute units.  Rows
// of four or more chunks on a launch that still has fewer than 1024 wavefronts are cut into 2 or 4 K parts
// (more loads in flight; a wavefront keeps at least one chunk).
struct GemvShape {
  int waves, ksplit;
};

static GemvShape gemv_shape(int N, int K, bool fused, int mt) {
  GemvShape sh{GV_WAVES, 1};
  if (fused) return sh;
  const int cus = device_cus();
  const int groups = (N + GV_ROWS - 1) / GV_ROWS, nchunk = (K + GV_CHUNK - 1) / GV_CHUNK;
  // K parts until the device holds 4 wavefronts per compute unit -- 8 for up to 4 tokens, where the extra loads in
  // flight pay (N = K = 4096, 1 token: 6.25 -> 5.5 us) and the token codes every workgroup copies are few; with 8
  // tokens the same change costs 0.4 us
  const int waves_per_cu = mt <= 4 ? 8 : 4;
  while (nchunk >= 4 && sh.ksplit < 4 && groups * sh.ksplit < waves_per_cu * cus && nchunk >= 2 * sh.ksplit) sh.ksplit *= 2;
  int per_wg = GV_WAVES / sh.ksplit;  // row groups per workgroup
  while (per_wg > 1 && (groups + per_wg - 1) / per_wg < cus) per_wg >>= 1;
  if (sh.ksplit == 1 && per_wg < 2) per_wg = 2;
  sh.waves = per_wg * sh.ksplit;
  return sh;
}

template <int MT, bool FUSED, int VPL, bool NORM, int FW, int FK = 1>
static int launch_gemv_fw(GemvArgs a, hipStream_t st) {
  GemvShape sh = gemv_shape(a.N, a.K, FUSED, MT);
  if (FUSED) {
    sh.waves = FW;
    sh.ksplit = FK;
  }
  a.ksplit = sh.ksplit;
  const int rows_per_wg = GV_ROWS * (sh.waves / sh.ksplit);
  const unsigned grid = (unsigned)((a.N + rows_per_wg - 1) / rows_per_wg);
  const size_t lds = (size_t)MT * a.K + MT * sizeof(float) + (sh.ksplit > 1 ? (size_t)sh.waves * 64 * sizeof(int) : 0);
  if (lds > 64 * 1024) {  // beyond the default dynamic-LDS limit: opt this kernel in, once per device
    static LdsOptIn opted;
    const int e = opted.ensure(reinterpret_cast<const void*>(&gemv_w8a8_kernel<MT, FUSED, VPL, NORM, FW, FK>));
    if (e) return e;
  }
  aq::queue_kernel((gemv_w8a8_kernel<MT, FUSED, VPL, NORM, FW, FK>), dim3(grid), dim3(sh.waves * 64), lds, st, a);
  return (int)hipGetLastError();
}

// Fused kernels on a short matrix (N / 32 workgroups would leave most compute units without one) run with 4
// wavefronts per workgroup instead of 8: twice the workgroups, each quantising the rows again but reaching a
// compute unit of its own (q/k/v 3072 x 2048 at M = 8: 5.6 -> 5.2 us; 1536 x 1536 at M = 4: 3.8 -> 3.5 us).
// Only where the rows are short.
template <int MT, bool FUSED, int VPL, bool NORM = false>
static int launch_gemv(GemvArgs a, hipStream_t st) {
  if constexpr (FUSED && VPL <= 4) {
    if (a.N <= 4096) return launch_gemv_fw<MT, FUSED, VPL, NORM, 4>(a, st);
  }
  return launch_gemv_fw<MT, FUSED, VPL, NORM, GV_WAVES>(a, st);
}

#ifndef AQ_GV_MFMA_MIN_M
#define AQ_GV_MFMA_MIN_M 8
#endif
constexpr int GV_MFMA_MIN_M = AQ_GV_MFMA_MIN_M;  // more tokens than this take the matrix-core variant

// ---------------------------------------------------------------------------
// Streaming variant for 5..16 tokens.  With that many tokens the 16 dot
// products every weight dword needs make the vector ALU, not HBM, the limit
// of the kernel above.  This one keeps its structure -- every weight byte goes
// HBM -> registers exactly once, no LDS staging or macro-tiling of W -- but
// hands the products to the matrix core: a wavefront owns 16 weight rows, loads
// them 16 bytes per lane directly in the v_mfma_i32_16x16x64_i8 operand order
// (lane l: row l%16, K bytes 64j + 16*(l/16) .. +16 of step j, so the four
// lanes of a row cover 64 contiguous bytes and two consecutive steps consume
// whole 128-byte lines), and multiplies against the token codes held in LDS.
// The 16 x 16 result has rows = weight rows and columns = tokens, so a lane
// ends up with 4 consecutive outputs of one token: no cross-lane reduction.
// ksplit wavefronts share a row group, each taking a part of K; the parts are
// summed through LDS (exact int32).  A workgroup holds `groups` row groups:
// 2 x 2 wavefronts when N fills the device that way, fewer rows per workgroup
// and more K parts when it does not.
constexpr int GM_ROWS = 16;    // weight rows per wavefront
constexpr int GM_MAX_WAVES = 8;
constexpr int GM_BATCH = 8;    // MFMA steps (64 K bytes each) per register batch

// KS, GR: K parts and row groups per workgroup fixed at compile time (the common 2 x 2 shape), or 0: taken
// from the arguments.  RES: a residual is added (a compile-time switch: a conditional early load makes the
// compiler drain the weight loads at the join, 0.4 us of a 6.5 us launch).
// XR: rounds of token-code vectors (8 per thread each) requested ahead of the weight stream; rows too long for
// XR rounds copy the rest afterwards, which waits for the weight loads in flight.
template <int KS, int GR, bool RES, int XR>
__global__ __launch_bounds__(GM_MAX_WAVES * 64) void gemv_mfma_kernel(GemvArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [16][K + 16] token codes, [16] scales, 16 spare bytes; later the partial sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ksplit = KS ? KS : p.ksplit, groups = GR ? GR : p.groups;
  const int nthreads = ksplit * groups * 64;
  const int grp = wave / ksplit, kh = wave % ksplit;
  const int K = p.K, N = p.N, M = p.M;
  // first weight row of this wavefront's group
  const int n0 = __builtin_amdgcn_readfirstlane((blockIdx.x * groups + grp) * GM_ROWS);
  const int pitch = K + 16;  // 16 token rows then start 4 banks apart: conflict-free 16-byte reads
  const int khalf = K / ksplit;  // a multiple of 128 (checked by the launcher)
  const int nline = khalf / 128;  // 128-byte lines of a row's K part: two MFMA steps each

  // epilogue operands first: lane l -> token l%16, rows (l/16)*4 .. +3 of the group
  const int tok = lane & 15;
  const int rbase = n0 + (lane >> 4) * 4;
  float swv[4], bv[4];
  uint32_t rv[4];  // residual elements, raw bits
  // only the first K part's wavefront writes outputs: the others get empty descriptors.  Requested (load_epi)
  // between the token rows and the weight stream.  Loads return in request order: behind the weights the
  // epilogue would wait for the whole stream to drain (0.2 us), and in front of the tokens these few lines, which
  // no other workgroup shares and which therefore come from HBM, hold back the token rows that every workgroup
  // reads and the caches serve (M = 16, N = 8192: 7.45 -> 7.2 us with the rows quantised here, 5.85 -> 5.65 us on
  // codes).
  const EpiOperands epi(p, kh == 0, true, RES);
  float sxv = 0.0f;
  auto load_epi = [&]() {
    sxv = epi.load_sx(tok, tok < M);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = rbase + r;
      swv[r] = epi.load_sw(n, n < N);
      bv[r] = epi.load_bias(n, n < N);
      rv[r] = RES ? epi.load_res(tok, n, tok < M && n < N, (int)p.ldr) : 0u;
    }
  };

  // weight stream: descriptor over this wavefront's 16 rows; rows past N read as zero
  const int rows = n0 < N ? ((N - n0) < GM_ROWS ? (N - n0) : GM_ROWS) : 0;
  const __amdgpu_buffer_rsrc_t Wr =
      make_rsrc(p.wq + (int64_t)(n0 < N ? n0 : 0) * K, (uint32_t)rows * (uint32_t)K);
  // Whole 128-byte lines per load: an instruction covers one line of 8 rows (lane l: row l % 8, 16-byte piece
  // l / 8), two instructions (rows 0..7 and 8..15) per line index.  In the MFMA's own operand order (lane l: row
  // l % 16, piece l / 16 of a 64-byte step) an instruction would cover 16 half lines, and a one-shot read of
  // the weight in that pattern measures 0.35 us slower (4.65 against 4.30 us for 16 MiB).  The operands are put
  // together from a line's two registers by one row rotation per dword (see consume).
  const uint32_t woff = (uint32_t)(lane & 7) * (uint32_t)K + (uint32_t)(kh * khalf + (lane >> 3) * 16);
  const uint32_t woff8 = 8u * (uint32_t)K;
  constexpr int GM_LINES = GM_BATCH / 2;  // lines per register batch
  uint4 wa[GM_BATCH], wb[GM_BATCH];       // [2 t]: rows 0..7 of line t, [2 t + 1]: rows 8..15
  auto wload = [&](int line0, uint4 (&dst)[GM_BATCH]) {
#pragma unroll
    for (int t = 0; t < GM_LINES; ++t) {
      const bool ok = (line0 + t) < nline;
      const uint32_t o = woff + (uint32_t)(line0 + t) * 128u;
      dst[2 * t] = GV_WLOAD(Wr, ok ? o : OOB_OFFSET);
      dst[2 * t + 1] = GV_WLOAD(Wr, ok ? o + woff8 : OOB_OFFSET);
    }
  };

  // token codes -> LDS (padded rows; tokens >= M are zero).  Their loads are
  // issued before the weight loads, so they return first and the LDS fill
  // overlaps the weight stream's flight time.
  const __amdgpu_buffer_rsrc_t Xr = make_rsrc(p.xq, (uint32_t)M * (uint32_t)K);
  const int nvec_row = K / 16;
  const int nvec = 16 * nvec_row;
  constexpr int XV = 8;  // vectors per thread per round: 16 x 2048 codes in one round of 256 threads
  uint4 xvr[XR][XV];
  auto xload = [&](int v0, uint4 (&xv)[XV]) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int v = v0 + i * nthreads + tid;
      xv[i] = buffer_load_16(Xr, v < nvec ? (uint32_t)v * 16u : OOB_OFFSET);
    }
  };
  // Stores without a branch: vectors past the end go to the spare slot behind the scales.  (With the
  // store under `if (v < nvec)` the compiler sank a vector's load into that branch, behind the weight
  // loads, and then waited for every load of the wavefront before the first LDS store: the matrix
  // products started only after the whole weight stream had landed.)
  uint8_t* const spare = xs + 16 * pitch + 16 * sizeof(float);
  auto xstore = [&](int v0, const uint4 (&xv)[XV]) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int v = v0 + i * nthreads + tid;
      const int m = v / nvec_row, c = v - m * nvec_row;
      *reinterpret_cast<uint4*>(v < nvec ? xs + m * pitch + c * 16 : spare) = xv[i];
    }
  };
#pragma unroll
  for (int r = 0; r < XR; ++r) xload(r * XV * nthreads, xvr[r]);
  asm volatile("" ::: "memory");  // request order: token codes, epilogue operands, the weight stream
  load_epi();
  asm volatile("" ::: "memory");
  wload(0, wa);
  wload(GM_LINES, wb);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int r = 0; r < XR; ++r) xstore(r * XV * nthreads, xvr[r]);  // waits for the token codes only: the oldest requests
  for (int v0 = XR * XV * nthreads; v0 < nvec; v0 += XV * nthreads) {  // still longer rows
    xload(v0, xvr[0]);
    xstore(v0, xvr[0]);
  }
  // LDS writes done, then a barrier without a memory fence: the weight loads stay in flight
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // Four independent accumulators (summed at the end: int32, exact in any order) and a batch's token
  // fragments read from LDS up front: one chain of 16 dependent read -> MFMA steps took 0.6 us after the
  // token codes had landed, which is all on the kernel's critical path.
  v4i accs[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) accs[i] = v4i{0, 0, 0, 0};
  // MFMA step (t, e) of line t takes, for weight row r = lane % 16 and token lane % 16, the line's piece
  // 2 (lane / 16) + e: K bytes t 128 + (2 q + e) 16 of the wavefront's part.  (Any assignment of K bytes to the
  // steps' k slots is a valid product as long as both operands use the same one.)  Lane l holds piece l / 8 of
  // row l % 8 (register lo) and of row 8 + l % 8 (register hi), so lanes 0..7 of each row of 16 lanes have
  // their operand of step e = 0 in lo, and lanes 8..15 find theirs in hi of lane l - 8; for e = 1 it is lo of
  // lane l + 8 and the own hi: one rotation by 8 within the row of 16 lanes, written into half of the lanes.
  const uint8_t* xl = xs + tok * pitch + kh * khalf + (lane >> 4) * 32;
  auto consume = [&](int line0, const uint4 (&wc)[GM_BATCH]) {
    v4i x[GM_BATCH];
#pragma unroll
    for (int t = 0; t < GM_LINES; ++t) {
      const int ln = (line0 + t) < nline ? (line0 + t) : 0;  // lines past the end multiply zero weights
      x[2 * t] = *reinterpret_cast<const v4i*>(xl + ln * 128);
      x[2 * t + 1] = *reinterpret_cast<const v4i*>(xl + ln * 128 + 16);
    }
#pragma unroll
    for (int t = 0; t < GM_LINES; ++t) {
      const uint4 lo = wc[2 * t], hi = wc[2 * t + 1];
      constexpr int ROR8 = 0x128;  // DPP row_ror:8
      // e = 0: lanes 8..15 of each row (banks 2, 3) take hi from lane l - 8, the others keep lo
      const v4i w0 = {__builtin_amdgcn_update_dpp((int)lo.x, (int)hi.x, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.y, (int)hi.y, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.z, (int)hi.z, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.w, (int)hi.w, ROR8, 0xf, 0xc, false)};
      // e = 1: lanes 0..7 of each row (banks 0, 1) take lo from lane l + 8, the others keep hi
      const v4i w1 = {__builtin_amdgcn_update_dpp((int)hi.x, (int)lo.x, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.y, (int)lo.y, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.z, (int)lo.z, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.w, (int)lo.w, ROR8, 0xf, 0x3, false)};
      accs[(2 * t) & 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, x[2 * t], accs[(2 * t) & 3], 0, 0, 0);
      accs[(2 * t + 1) & 3] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, x[2 * t + 1], accs[(2 * t + 1) & 3], 0, 0, 0);
    }
  };
  for (int l0 = 0; l0 < nline; l0 += 2 * GM_LINES) {
    consume(l0, wa);
    if (l0 + 2 * GM_LINES < nline) wload(l0 + 2 * GM_LINES, wa);
    if (l0 + GM_LINES < nline) consume(l0 + GM_LINES, wb);
    if (l0 + 3 * GM_LINES < nline) wload(l0 + 3 * GM_LINES, wb);
  }

  v4i acc = (accs[0] + accs[1]) + (accs[2] + accs[3]);
  // sum the K parts: all but the first wavefront of each group park their 4 sums in LDS
  __syncthreads();  // everyone is done reading the token codes: the buffer is reused
  int* part = reinterpret_cast<int*>(xs) + grp * (ksplit - 1) * 256;
  if (kh != 0) {
    *reinterpret_cast<v4i*>(part + (kh - 1) * 256 + lane * 4) = acc;
  }
  __syncthreads();
  if (kh != 0) return;
  for (int k = 0; k < ksplit - 1; ++k) acc += *reinterpret_cast<const v4i*>(part + k * 256 + lane * 4);

  if (tok >= M) return;
  float y[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[r] = __fmul_rn(__fmul_rn((float)acc[r], sxv), swv[r]);
    if (p.bias) y[r] = __fadd_rn(y[r], bv[r]);
    if constexpr (RES) y[r] = p.y_dtype == AQ_BF16 ? add_residual_bf16(y[r], rv[r]) : __fadd_rn(y[r], __uint_as_float(rv[r]));
  }
  const int64_t o = (int64_t)tok * N + rbase;
  if (p.y_dtype == AQ_BF16) {
    uint16_t* dst = reinterpret_cast<uint16_t*>(p.y) + o;
    if ((N & 3) == 0 && rbase + 3 < N) {  // 8-byte aligned and fully inside
      uint2 pk;
      pk.x = pack_bf16x2(y[0], y[1]);
      pk.y = pack_bf16x2(y[2], y[3]);
      *reinterpret_cast<uint2*>(dst) = pk;
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rbase + r < N) dst[r] = (uint16_t)f32_to_bf16_bits(y[r]);
    }
  } else {
    float* dst = reinterpret_cast<float*>(p.y) + o;
    if ((N & 3) == 0 && rbase + 3 < N) {
      *reinterpret_cast<float4*>(dst) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rbase + r < N) dst[r] = y[r];
    }
  }
}

// the streaming MFMA variant needs K in whole 256-byte steps (two K parts of whole 128-byte lines)
// and its padded codes to fit LDS
static bool gemv_mfma_ok(int64_t M, int64_t K) {
  return M > GV_MFMA_MIN_M && (K % 256) == 0 && 16 * (K + 16) + 64 + 16 <= GV_MAX_LDS;
}

static int launch_gemv_mfma(GemvArgs a, hipStream_t st) {
  // 2 row groups x 2 K parts per workgroup by default; with too few rows for that to give every
  // compute unit a workgroup, one row group per workgroup and up to 8 K parts
  a.ksplit = 2;
  a.groups = 2;
  const int cus = device_cus();
  if ((a.N + 31) / 32 < cus) {
    a.groups = 1;
    while (a.ksplit < GM_MAX_WAVES && (a.N + 15) / 16 * (a.ksplit / 2) < cus && a.K % (256 * a.ksplit) == 0 &&
           a.K / (2 * a.ksplit) >= 512)
      a.ksplit *= 2;
  }
  const unsigned grid = (unsigned)((a.N + GM_ROWS * a.groups - 1) / (GM_ROWS * a.groups));
  const size_t lds = (size_t)16 * (a.K + 16) + 16 * sizeof(float) + 16;
  const bool fixed = a.ksplit == 2 && a.groups == 2, res = a.res != nullptr;
  // one round of token-code loads ahead of the weights covers 8 vectors per thread; longer rows take three
  const bool long_rows = (int64_t)16 * (a.K / 16) > (int64_t)8 * a.ksplit * a.groups * 64;
  using kern_t = void (*)(GemvArgs);
  static const kern_t table[2][2][2] = {
      {{gemv_mfma_kernel<0, 0, false, 1>, gemv_mfma_kernel<0, 0, false, 3>}, {gemv_mfma_kernel<0, 0, true, 1>, gemv_mfma_kernel<0, 0, true, 3>}},
      {{gemv_mfma_kernel<2, 2, false, 1>, gemv_mfma_kernel<2, 2, false, 3>}, {gemv_mfma_kernel<2, 2, true, 1>, gemv_mfma_kernel<2, 2, true, 3>}}};
  const kern_t fn = table[fixed][res][long_rows];
  if (lds > 64 * 1024) {
    static LdsOptIn opted[8];
    const int e = opted[fixed * 4 + res * 2 + long_rows].ensure(reinterpret_cast<const void*>(fn));
    if (e) return e;
  }
  aq::queue_kernel(fn, dim3(grid), dim3(a.ksplit * a.groups * 64), lds, st, a);
  return (int)hipGetLastError();
}

// up/gate + SwiGLU in one launch (gemv_rows.hip): bf16 rows of K <= 2048 in whole 512-byte steps, F a multiple of 16.
static bool gemv_swiglu_ok(int64_t M, int64_t F, int64_t K) {
  return M >= 1 && M <= 16 && F > 0 && (F % 16) == 0 && K <= 2048 && (K % 512) == 0;
}

// ---------------------------------------------------------------------------
// 17..32 tokens on codes: the same weight stream (every weight byte HBM -> registers once, operands assembled by
// one DPP rotation per dword) with TG = 2 groups of 16 tokens multiplied against each weight fragment: a bandwidth-bound
// launch for matrices of more than 48 outputs to a compute unit, where the GEMM whose wavefronts share K would take a second
// round of tiles (at one tile per compute unit it is the faster one).  From 33
// tokens on, with a third and fourth token group, it was the slower one (48 rows: 6.1 us, 64 rows: 7.6 us with the weights
// in the last-level cache, where a 128 x 32 tile took 5.8 us).  Same integer sums, same epilogue: the bits of the tiled GEMM.
// K is walked in chunks of 1024 bytes per wavefront (KS wavefronts per row group: 1024- or 2048-byte chunks
// per workgroup), the token codes of one chunk at a time in LDS, so that rows of any length are taken (an MLP's
// down projection) and the LDS of a compute unit holds several workgroups.  A chunk's codes are requested into
// registers while the chunk before is multiplied and stored between two barriers; the weight stream runs through
// the chunk boundaries untouched (two register batches, each reloaded as soon as it has been consumed).  GRP row
// groups of 16 rows per workgroup (every workgroup copies all token codes from L2); rows must be whole 128-byte lines
// (K % 128 == 0).
// FP8: e4m3 codes with one scale per tensor, v_mfma_f32_16x16x128_f8f6f4 and fp32 accumulation (chunks and K parts
// summed in a fixed order).
template <int TG, int KS, bool RES, int GRP = 2, bool FP8 = false>
__global__ __launch_bounds__(KS * GRP * 64) void gemv_mfma_tokens_kernel(GemvArgs p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t xs[];  // [16 TG][KC + 16] codes of one chunk; later the partial sums
  constexpr int MTOK = 16 * TG, NTHREADS = KS * GRP * 64;
  constexpr int KC = 1024 * KS;            // K bytes of a chunk
  constexpr int PITCH = KC + 16;
  constexpr int XV = MTOK * (KC / 16) / NTHREADS;  // 16-byte vectors of a chunk's codes per thread: 16 / GRP per token group
  static_assert(XV * NTHREADS == MTOK * (KC / 16) && MTOK * PITCH <= 150 * 1024 && KS * GRP <= GM_MAX_WAVES,
                "a chunk's codes: whole vectors per thread, within LDS");
  static_assert(GRP * (KS - 1) * TG * 1024 <= MTOK * PITCH, "the partial sums reuse the codes' LDS");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave / KS, kh = wave % KS;
  const int K = p.K, N = p.N, M = p.M;
  const int n0 = __builtin_amdgcn_readfirstlane((blockIdx.x * GRP + grp) * GM_ROWS);
  const int nchunk = (K + KC - 1) / KC;

  const int tok = lane & 15;
  const int rbase = n0 + (lane >> 4) * 4;
  float swv[4], bv[4], sxv[TG];
  uint32_t rv[TG][4];
  const EpiOperands epi(p, kh == 0, true, RES);

  const int rows = n0 < N ? ((N - n0) < GM_ROWS ? (N - n0) : GM_ROWS) : 0;
  const __amdgpu_buffer_rsrc_t Wr = make_rsrc(p.wq + (int64_t)(n0 < N ? n0 : 0) * K, (uint32_t)rows * (uint32_t)K);
  const uint32_t woff = (uint32_t)(lane & 7) * (uint32_t)K + (uint32_t)((lane >> 3) * 16);
  const uint32_t woff8 = 8u * (uint32_t)K;
  constexpr int GM_LINES = GM_BATCH / 2;
  uint4 wa[GM_BATCH], wb[GM_BATCH];
  // lines line0 .. line0+3 of this wavefront's 1024 bytes of chunk c (columns past K read zeros: an offset there
  // would alias the next row, so it is pushed outside the descriptor)
  auto wload = [&](int c, int line0, uint4 (&dst)[GM_BATCH]) {
#pragma unroll
    for (int t = 0; t < GM_LINES; ++t) {
      const int col = c * KC + kh * 1024 + (line0 + t) * 128;
      const bool ok = col < K;
      const uint32_t o = woff + (uint32_t)col;
      dst[2 * t] = GV_WLOAD(Wr, ok ? o : OOB_OFFSET);
      dst[2 * t + 1] = GV_WLOAD(Wr, ok ? o + woff8 : OOB_OFFSET);
    }
  };
  const __amdgpu_buffer_rsrc_t Xr = make_rsrc(p.xq, (uint32_t)M * (uint32_t)K);
  uint4 xvr[XV];
  auto xload = [&](int c) {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int v = i * NTHREADS + tid;
      const int m = v / (KC / 16), cc = v - m * (KC / 16);
      const int col = c * KC + cc * 16;
      xvr[i] = buffer_load_16(Xr, (m < M && col < K) ? (uint32_t)m * (uint32_t)K + (uint32_t)col : OOB_OFFSET);
    }
  };
  auto xstore = [&]() {
#pragma unroll
    for (int i = 0; i < XV; ++i) {
      const int v = i * NTHREADS + tid;
      const int m = v / (KC / 16), cc = v - m * (KC / 16);
      *reinterpret_cast<uint4*>(xs + m * PITCH + cc * 16) = xvr[i];
    }
  };

  xload(0);
  asm volatile("" ::: "memory");  // request order: token codes, epilogue operands, the weight stream
#pragma unroll
  for (int g = 0; g < TG; ++g) sxv[g] = epi.load_sx(FP8 ? 0 : tok + 16 * g, FP8 || tok + 16 * g < M);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = rbase + r;
    swv[r] = epi.load_sw(FP8 ? 0 : n, FP8 || n < N);
    bv[r] = epi.load_bias(n, n < N);
#pragma unroll
    for (int g = 0; g < TG; ++g) rv[g][r] = RES ? epi.load_res(tok + 16 * g, n, tok + 16 * g < M && n < N, (int)p.ldr) : 0u;
  }
  asm volatile("" ::: "memory");
  wload(0, 0, wa);
  wload(0, GM_LINES, wb);
  asm volatile("" ::: "memory");

  using accv = std::conditional_t<FP8, v4f, v4i>;
  accv accs[TG][2];
#pragma unroll
  for (int g = 0; g < TG; ++g) accs[g][0] = accs[g][1] = accv{0, 0, 0, 0};
  const uint8_t* xl = xs + tok * PITCH + kh * 1024 + (lane >> 4) * 32;
  auto consume = [&](int line0, const uint4 (&wc)[GM_BATCH]) {
#pragma unroll
    for (int t = 0; t < GM_LINES; ++t) {
      v4i x0[TG], x1[TG];
#pragma unroll
      for (int g = 0; g < TG; ++g) {
        x0[g] = *reinterpret_cast<const v4i*>(xl + g * 16 * PITCH + (line0 + t) * 128);
        x1[g] = *reinterpret_cast<const v4i*>(xl + g * 16 * PITCH + (line0 + t) * 128 + 16);
      }
      const uint4 lo = wc[2 * t], hi = wc[2 * t + 1];
      constexpr int ROR8 = 0x128;  // DPP row_ror:8 (see gemv_mfma_kernel)
      const v4i w0 = {__builtin_amdgcn_update_dpp((int)lo.x, (int)hi.x, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.y, (int)hi.y, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.z, (int)hi.z, ROR8, 0xf, 0xc, false),
                      __builtin_amdgcn_update_dpp((int)lo.w, (int)hi.w, ROR8, 0xf, 0xc, false)};
      const v4i w1 = {__builtin_amdgcn_update_dpp((int)hi.x, (int)lo.x, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.y, (int)lo.y, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.z, (int)lo.z, ROR8, 0xf, 0x3, false),
                      __builtin_amdgcn_update_dpp((int)hi.w, (int)lo.w, ROR8, 0xf, 0x3, false)};
#pragma unroll
      for (int g = 0; g < TG; ++g) {
        if constexpr (!FP8) {
          accs[g][0] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, x0[g], accs[g][0], 0, 0, 0);
          accs[g][1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, x1[g], accs[g][1], 0, 0, 0);
        } else {  // the line's two pieces are the 32 K bytes a lane feeds one 16x16x128 product
          const v8i wl = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
          const v8i xl8 = {x0[g].x, x0[g].y, x0[g].z, x0[g].w, x1[g].x, x1[g].y, x1[g].z, x1[g].w};
          accs[g][t & 1] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wl, xl8, accs[g][t & 1], 0, 0, 0, 0, 0, 0);
        }
      }
    }
  };
  // barriers without a memory fence (LDS traffic only has to be complete): the weight loads stay in flight
  auto lds_barrier = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  for (int c = 0; c < nchunk; ++c) {
    if (c > 0) lds_barrier();  // every wavefront is done with the codes of the chunk before
    xstore();                  // waits for this chunk's codes only: they are older than the weight loads in flight
    lds_barrier();
    if (c + 1 < nchunk) xload(c + 1);
    consume(0, wa);
    if (c + 1 < nchunk) wload(c + 1, 0, wa);
    consume(GM_LINES, wb);
    if (c + 1 < nchunk) wload(c + 1, GM_LINES, wb);
  }

  // sum the K parts through LDS (int32: exact; fp32: in a fixed order)
  __syncthreads();
  int* part = reinterpret_cast<int*>(xs) + (grp * (KS - 1)) * TG * 256;
  accv acc[TG];
#pragma unroll
  for (int g = 0; g < TG; ++g) acc[g] = accs[g][0] + accs[g][1];
  if (kh != 0) {
#pragma unroll
    for (int g = 0; g < TG; ++g) *reinterpret_cast<accv*>(part + ((kh - 1) * TG + g) * 256 + lane * 4) = acc[g];
  }
  __syncthreads();
  if (kh != 0) return;
  for (int k = 0; k < KS - 1; ++k)
#pragma unroll
    for (int g = 0; g < TG; ++g) acc[g] += *reinterpret_cast<const accv*>(part + (k * TG + g) * 256 + lane * 4);

#pragma unroll
  for (int g = 0; g < TG; ++g) {
    const int tk = tok + 16 * g;
    if (tk >= M) continue;
    float y[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      y[r] = __fmul_rn(__fmul_rn((float)acc[g][r], sxv[g]), swv[r]);
      if (p.bias) y[r] = __fadd_rn(y[r], bv[r]);
      if constexpr (RES) y[r] = p.y_dtype == AQ_BF16 ? add_residual_bf16(y[r], rv[g][r]) : __fadd_rn(y[r], __uint_as_float(rv[g][r]));
    }
    const int64_t o = (int64_t)tk * N + rbase;
    if (p.y_dtype == AQ_BF16) {
      uint16_t* dst = reinterpret_cast<uint16_t*>(p.y) + o;
      if ((N & 3) == 0 && rbase + 3 < N) {
        uint2 pk;
        pk.x = pack_bf16x2(y[0], y[1]);
        pk.y = pack_bf16x2(y[2], y[3]);
        *reinterpret_cast<uint2*>(dst) = pk;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (rbase + r < N) dst[r] = (uint16_t)f32_to_bf16_bits(y[r]);
      }
    } else {
      float* dst = reinterpret_cast<float*>(p.y) + o;
      if ((N & 3) == 0 && rbase + 3 < N) {
        *reinterpret_cast<float4*>(dst) = make_float4(y[0], y[1], y[2], y[3]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (rbase + r < N) dst[r] = y[r];
      }
    }
  }
}

// A launch of the token-group kernel: 64 weight rows per workgroup, half the copies of the token codes (32 x 16384 x 2048: 7.0 us
// against 7.4 us with 32), in chunks no longer than the rows, 1024 or 2048 bytes.
template <int KS>
static int launch_gemv_tokens_shape(const GemvArgs& a, hipStream_t st, bool fp8) {
  constexpr int TG = 2, GRP = 4;
  const unsigned grid = (unsigned)((a.N + GRP * GM_ROWS - 1) / (GRP * GM_ROWS));
  const size_t lds = (size_t)16 * TG * (1024 * KS + 16) + 16;
  using kern_t = void (*)(GemvArgs);
  const kern_t fn = fp8 ? (a.res ? gemv_mfma_tokens_kernel<TG, KS, true, GRP, true> : gemv_mfma_tokens_kernel<TG, KS, false, GRP, true>)
                        : (a.res ? gemv_mfma_tokens_kernel<TG, KS, true, GRP> : gemv_mfma_tokens_kernel<TG, KS, false, GRP>);
  static LdsOptIn opted[4];
  const int e = opted[(fp8 ? 2 : 0) + (a.res ? 1 : 0)].ensure(reinterpret_cast<const void*>(fn));
  if (e) return e;
  aq::queue_kernel(fn, dim3(grid), dim3(KS * GRP * 64), lds, st, a);
  return (int)hipGetLastError();
}

// (not static: the tiled GEMM's entry points in gemm_mfma.hip hand over what streams_weights says)
int gemv_tokens_launch(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw, const void* bias,
                       int bias_dtype, const void* residual, void* y, int y_dtype, int64_t M, int64_t N, int64_t K,
                       hipStream_t st, bool fp8) {
  GemvArgs a{};
  a.xq = xq;
  a.sx = sx;
  a.wq = wq;
  a.sw = sw;
  a.bias = bias;
  a.res = residual;
  a.ldr = N;
  a.y = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = y_dtype;
  return K <= 1024 ? launch_gemv_tokens_shape<1>(a, st, fp8) : launch_gemv_tokens_shape<2>(a, st, fp8);
}

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace aq

extern "C" size_t aq_gemv_w8a8_workspace_bytes(int64_t M, int64_t K) {
  if (M < 0 || K < 0) return 0;
  return aq::align256((size_t)(M * K)) + aq::align256((size_t)M * sizeof(float));
}

// *mt_out: the token-count bucket of the GEMV kernels, or -1 when the activation codes of that bucket do
// not fit the LDS of a compute unit (rows longer than 10 096 bytes at 9..16 tokens, 20 208 at 5..8, ...):
// such a call is served by the tiled MFMA GEMM, which takes any M (same integer sums, same epilogue: same bits).
static int gemv_bucket(int64_t M, int64_t K) {
  const int mt = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : 16;
  return (int64_t)mt * K + 64 + 2048 > aq::GV_MAX_LDS ? -1 : mt;  // codes, scales, K-part sums
}

static int gemv_check(const int8_t* wq, const float* sw, const void* bias, int bias_dtype, const void* residual,
                      const void* y, int y_dtype, int64_t M, int64_t N, int64_t K, int* mt_out) {
  if (y_dtype != AQ_F32 && y_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (bias && bias_dtype != AQ_F32 && bias_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (M < 0 || M > 16 || N < 0 || K <= 0 || (K % 16) != 0) return AQ_E_SHAPE;
  if (M == 0 || N == 0) return AQ_OK;
  if (!wq || !sw || !y) return AQ_E_NULL;
  // matrices on 16 bytes (vector loads and stores), scale and bias vectors on their element size
  if (aq::check_ptr16(wq) || aq::check_ptr16(y) || aq::check_ptr16(residual)) return AQ_E_ALIGN;
  if (aq::check_ptr(sw, 4) || aq::check_ptr(bias, bias_dtype == AQ_BF16 ? 2 : 4)) return AQ_E_ALIGN;
  if (N > (1 << 25) || K > (1 << 22)) return AQ_E_RANGE;  // 16 rows of N outputs are indexed in 32 bits
  *mt_out = gemv_bucket(M, K);
  return AQ_OK;
}

static int gemv_dispatch(const aq::GemvArgs& a, int mt, hipStream_t st) {
  // 9..16 rows go to the matrix-core variant, except on a short matrix with long rows (an MLP's down projection):
  // its 16-row wavefronts make N / 16 workgroups, half the device or less, where the dot-product kernel's 4-row
  // wavefronts still reach every compute unit (N = 2048, K = 5632: 7.6-8.0 against 8.5 us; N = 1536, K = 6912:
  // 11.0 against 12.9 us; at K = 2048 or from N = 3072 on the matrix core wins, 4.7 against 5.6 us).
  const bool short_long = (a.N + 15) / 16 * 2 <= aq::device_cus() && a.K >= 4096;
  if (aq::gemv_mfma_ok(a.M, a.K) && !short_long) return aq::launch_gemv_mfma(a, st);
  switch (mt) {
    case 1: return aq::launch_gemv<1, false, 4>(a, st);
    case 2: return aq::launch_gemv<2, false, 4>(a, st);
    case 4: return aq::launch_gemv<4, false, 4>(a, st);
    case 8: return aq::launch_gemv<8, false, 4>(a, st);
    default: return aq::launch_gemv<16, false, 4>(a, st);
  }
}

// One launch where a kernel quantises (and normalises) the rows itself; -1 when the shape takes two.
// Up to 4 bf16 rows have two kernels.  The dot-product kernel: one wavefront rounds a row, the others start on their weights, and
// the few products per weight dword are no load on the vector ALU; it keeps its place with many weights per row.  gemv_rows.hip
// for everything else: more rows; fp32 rows; rows of up to 1024 (3 and 4 of them, or of many weight rows); rows of 2049 to 4096,
// which the dot-product kernel holds in registers for 8192 and, on short matrices, does not cut into K parts (but 1 and 2 of
// them where 64-row workgroups are left a last round that is nearly empty: 1 x 3632 -> 10517 13.3 us, 12.0 by dot products, 1 x 3728 ->
// 38113 39.9, 31.8); longer ones of 2049 to 4096 weight rows, too many for those parts.
// Timed on both at 7433 random sizes, 1 to 4 rows, N 512..11264, K 512..8192, with the norm up to 2048: what this picks is 0.4 % from
// the faster one in the mean, 3.4 % for one in twenty.  us, this | the other: 1 x 3168 -> 1472 4.0 | 5.6, 4 x 3008 -> 1488 4.0 | 5.7, 1 x 6016
// -> 3440 6.7 | 7.8, 1 x 896 -> 9536 4.5 | 5.0, 4 x 1616 -> 1504 3.4 | 3.6; dot products 1 x 1968 -> 5648 4.5 | 5.5, 1 x 6880 -> 1585 4.8 | 5.9, 1 x
// 7088 -> 9312 18.0 | 21.6, 4 x 5024 -> 9600 15.0 | 15.9; with the norm 4 x 800 -> 10032 4.9 | 5.9, dot products 1 x 1744 -> 5839 4.4 | 5.1.
// (Where the two are within 4 % alone, the norm in front of a short matrix and 3 or 4 long rows to one, rows follow what wrote them:
// the 24-layer step of 4 with 6912 -> 1536 here 648 us, by dot products 657.)
static bool dot_kernel_better(int64_t M, int64_t N, int64_t K, bool norm) {
  if (M > 4) return false;
  if (norm) return K > 1024 && N > 4096 && (M < 3 || N <= 8192);
  if (K <= 1024) return M < 3 && N <= 8192;
  if (K <= 2048) return M < 3 || N > 2048;
  if (K <= 4096) return N > 4096 && (N <= 8192 || (M < 3 && N > (K > 3072 ? 10240 : 16384)));
  return N > 4096 || (M < 3 && N <= 2048);
}

enum FusedRoute { FUSED_NONE, FUSED_DOT, FUSED_ROWS };
static aq::RowsKind fused_kind(bool norm, bool bf16) { return norm ? aq::ROWS_I8_NORM : bf16 ? aq::ROWS_I8 : aq::ROWS_I8_F32; }
static FusedRoute fused_route(int x_dtype, bool norm, int mt, int64_t M, int64_t N, int64_t K) {
  const bool bf16 = x_dtype == AQ_BF16;
  const int64_t vpl = (K / 8 + 63) / 64;  // 16-byte vectors per lane per bf16 row
  const bool dot = bf16 && M <= 4 && mt > 0 && vpl <= (norm ? 4 : 16);
  if ((bf16 || !norm) && aq::gemv_rows_ok(fused_kind(norm, bf16), M, K) && !(dot && dot_kernel_better(M, N, K, norm))) return FUSED_ROWS;
  return dot ? FUSED_DOT : FUSED_NONE;
}

static int gemv_dispatch_fused(const aq::GemvArgs& a, int x_dtype, int mt, hipStream_t st) {
  const bool norm = a.gamma != nullptr;
  const int64_t vpl = (a.K / 8 + 63) / 64;
  const FusedRoute route = fused_route(x_dtype, norm, mt, a.M, a.N, a.K);
  if (route == FUSED_ROWS) return aq::launch_gemv_rows(a, fused_kind(norm, x_dtype == AQ_BF16), st);
  if (route == FUSED_NONE) return -1;
  // A short matrix with long rows (an MLP's down projection): with whole rows per wavefront its N / 32 workgroups
  // would leave most compute units without loads in flight.  4 K parts -- 8 weight rows per workgroup, every wavefront
  // rounding one token row first: 7.0 -> 4.8 us for one row of 5632 against 2048 weight rows (2 parts: 8.0, 8 parts:
  // 12.1 us for 8 rows).
  if (!norm && (a.N + 31) / 32 * 4 <= aq::device_cus() && a.K > 4096) {
    switch (mt) {
      case 1: return aq::launch_gemv_fw<1, true, 16, false, aq::GV_WAVES, 4>(a, st);
      case 2: return aq::launch_gemv_fw<2, true, 16, false, aq::GV_WAVES, 4>(a, st);
      default: return aq::launch_gemv_fw<4, true, 16, false, aq::GV_WAVES, 4>(a, st);
    }
  }
  const bool small = vpl <= 4;
  if (norm) {
    switch (mt) {
      case 1: return aq::launch_gemv<1, true, 4, true>(a, st);
      case 2: return aq::launch_gemv<2, true, 4, true>(a, st);
      default: return aq::launch_gemv<4, true, 4, true>(a, st);
    }
  }
  switch (mt) {
    case 1: return small ? aq::launch_gemv<1, true, 4>(a, st) : aq::launch_gemv<1, true, 16>(a, st);
    case 2: return small ? aq::launch_gemv<2, true, 4>(a, st) : aq::launch_gemv<2, true, 16>(a, st);
    default: return small ? aq::launch_gemv<4, true, 4>(a, st) : aq::launch_gemv<4, true, 16>(a, st);
  }
}

extern "C" int aq_gemv_w8a8_decode_one_launch(int x_dtype, int norm, int64_t M, int64_t N, int64_t K) {
  if ((x_dtype != AQ_F32 && x_dtype != AQ_BF16) || M < 1 || M > 16 || N < 1 || K < 1 || K % 16 || K > (1 << 22)) return 0;
  return fused_route(x_dtype, norm != 0, gemv_bucket(M, K), M, N, K) != FUSED_NONE ? 1 : 0;
}

extern "C" int aq_gemv_w8a8_codes_residual(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                                           const void* bias, int bias_dtype, const void* residual,
                                           void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
  int mt = 0;
  int rc = gemv_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, &mt);
  if (rc || M == 0 || N == 0) return rc;
  if (!xq || !sx) return AQ_E_NULL;
  if (aq::check_ptr16(xq) || aq::check_ptr(sx, 4)) return AQ_E_ALIGN;
  if (mt < 0) return aq_linear_w8a8_residual(xq, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
  aq::GemvArgs a{};
  a.xq = xq;
  a.sx = sx;
  a.wq = wq;
  a.sw = sw;
  a.bias = bias;
  a.res = residual;
  a.ldr = N;
  a.y = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = y_dtype;
  return gemv_dispatch(a, mt, static_cast<hipStream_t>(stream));
}

extern "C" int aq_gemv_w8a8_codes(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                                  const void* bias, int bias_dtype, void* y, int y_dtype, int64_t M,
                                  int64_t N, int64_t K, void* stream) {
  return aq_gemv_w8a8_codes_residual(xq, sx, wq, sw, bias, bias_dtype, nullptr, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_gemv_w8a8_decode_residual(const void* x, int x_dtype, const int8_t* wq, const float* sw,
                                            const void* bias, int bias_dtype, const void* residual,
                                            void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* ws,
                                            size_t ws_bytes, void* stream) {
  if (x_dtype != AQ_F32 && x_dtype != AQ_BF16) return AQ_E_DTYPE;
  int mt = 0;
  int rc = gemv_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, &mt);
  if (rc || M == 0 || N == 0) return rc;
  if (!x || !ws) return AQ_E_NULL;
  if (aq::check_ptr16(x) || aq::check_ptr16(ws)) return AQ_E_ALIGN;
  if (ws_bytes < aq_gemv_w8a8_workspace_bytes(M, K)) return AQ_E_WORKSPACE;
  {  // one launch where the GEMV kernel quantises the rows itself
    aq::GemvArgs a{};
    a.x = x;
    a.wq = wq;
    a.sw = sw;
    a.bias = bias;
    a.res = residual;
    a.ldr = N;
    a.y = y;
    a.M = (int)M;
    a.N = (int)N;
    a.K = (int)K;
    a.bias_dtype = bias_dtype;
    a.y_dtype = y_dtype;
    const int frc = gemv_dispatch_fused(a, x_dtype, mt, static_cast<hipStream_t>(stream));
    if (frc >= 0) return frc;
  }
  int8_t* xq = static_cast<int8_t*>(ws);
  float* sx = reinterpret_cast<float*>(static_cast<char*>(ws) + aq::align256((size_t)(M * K)));
  rc = aq_quant_rowwise_i8(x, x_dtype, M, K, K, xq, sx, stream);
  if (rc) return rc;
  return aq_gemv_w8a8_codes_residual(xq, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

// ---------------------------------------------------------------------------
// FP8 decode: rows that gemv_rows.hip casts itself, or codes and tiles whose K is cut among wavefronts (gemm_slices.hip).
extern "C" size_t aq_gemv_fp8_workspace_bytes(int64_t M, int64_t K) {
  if (M < 0 || K < 0) return 0;
  return aq::align256((size_t)(M * K)) + 256 + AQ_FP8_AMAX_WS_BYTES;  // codes, the scale, the quantiser's partial maxima
}

extern "C" int aq_gemv_fp8_decode_one_launch(int x_dtype, int64_t M, int64_t K) {
  return x_dtype == AQ_BF16 && M >= 1 && M <= 16 && aq::gemv_rows_ok(aq::ROWS_FP8, M, K) ? 1 : 0;
}

static int gemv_fp8_check(const uint8_t* wq, const float* sw, const void* bias, int bias_dtype, const void* residual,
                          const void* y, int y_dtype, int64_t M, int64_t N, int64_t K) {
  if (y_dtype != AQ_F32 && y_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (bias && bias_dtype != AQ_F32 && bias_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (M < 0 || M > 16 || N < 0 || K <= 0 || (K % 16) != 0) return AQ_E_SHAPE;
  if (M == 0 || N == 0) return AQ_OK;
  if (!wq || !sw || !y) return AQ_E_NULL;
  if (aq::check_ptr16(wq) || aq::check_ptr16(y) || aq::check_ptr16(residual)) return AQ_E_ALIGN;
  if (aq::check_ptr(sw, 4) || aq::check_ptr(bias, bias_dtype == AQ_BF16 ? 2 : 4)) return AQ_E_ALIGN;
  if (N > (1 << 25) || K > (1 << 22)) return AQ_E_RANGE;
  return AQ_OK;
}

static aq::GemvArgs gemv_fp8_args(const uint8_t* wq, const float* sw, const void* bias, int bias_dtype,
                                  const void* residual, void* y, int y_dtype, int64_t M, int64_t N, int64_t K) {
  aq::GemvArgs a{};
  a.wq = reinterpret_cast<const int8_t*>(wq);
  a.sw = sw;
  a.bias = bias;
  a.res = residual;
  a.ldr = N;
  a.y = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = y_dtype;
  return a;
}

extern "C" int aq_gemv_fp8_codes_residual(const uint8_t* xq, const float* sx, const uint8_t* wq, const float* sw,
                                          const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                          int64_t M, int64_t N, int64_t K, void* stream) {
  int rc = gemv_fp8_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K);
  if (rc || M == 0 || N == 0) return rc;
  if (!xq || !sx) return AQ_E_NULL;
  if (aq::check_ptr16(xq) || aq::check_ptr(sx, 4)) return AQ_E_ALIGN;
  if (N <= (1 << 20)) return aq_linear_fp8_residual(xq, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
  aq::GemmArgs a{};  // more outputs than its other tiles index
  a.A = xq;
  a.B = wq;
  a.C = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = a.lda = (int)K;
  a.sx = sx;
  a.sw = sw;
  a.bias = bias;
  a.bias_dtype = bias_dtype;
  a.res = residual;
  const int tile = aq::gemm_slices_tile(M, N, K, aq::device_cus());
  return y_dtype == AQ_BF16 ? aq::gemm_slices_launch<true, aq::OUT_BF16>(a, tile, static_cast<hipStream_t>(stream))
                            : aq::gemm_slices_launch<true, aq::OUT_F32>(a, tile, static_cast<hipStream_t>(stream));
}

extern "C" int aq_gemv_fp8_decode_residual(const void* x, int x_dtype, const uint8_t* wq, const float* sw,
                                           const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                           int64_t M, int64_t N, int64_t K, void* ws, size_t ws_bytes, void* stream) {
  if (x_dtype != AQ_F32 && x_dtype != AQ_BF16) return AQ_E_DTYPE;
  int rc = gemv_fp8_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K);
  if (rc || M == 0 || N == 0) return rc;
  if (!x || !ws) return AQ_E_NULL;
  if (aq::check_ptr16(x) || aq::check_ptr16(ws)) return AQ_E_ALIGN;
  if (ws_bytes < aq_gemv_fp8_workspace_bytes(M, K)) return AQ_E_WORKSPACE;
  if (aq_gemv_fp8_decode_one_launch(x_dtype, M, K)) {  // one launch: the kernel casts the rows itself
    aq::GemvArgs a = gemv_fp8_args(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K);
    a.x = x;
    return aq::launch_gemv_rows(a, aq::ROWS_FP8, static_cast<hipStream_t>(stream));
  }
  uint8_t* xq = static_cast<uint8_t*>(ws);
  float* sx = reinterpret_cast<float*>(static_cast<char*>(ws) + aq::align256((size_t)(M * K)));
  uint32_t* amax_ws = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(sx) + 256);
  rc = aq_quant_tensor_fp8(x, x_dtype, M * K, xq, sx, amax_ws, AQ_FP8_AMAX_WS_BYTES, stream);
  if (rc) return rc;
  return aq_gemv_fp8_codes_residual(xq, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

// ---------------------------------------------------------------------------
// The decode entry point for callers that cannot allocate (code under HIP graph capture, serving loops and
// harnesses that forbid hipMalloc): the workspace of aq_gemv_w8a8_decode_residual -- the activation codes and
// scales that the row quantiser hands to the GEMV when the rows are not quantised inside the GEMV kernel --
// lives in device memory that the library itself owns, one copy per GPU, for the life of the process.
namespace aq {

constexpr size_t NOALLOC_SCRATCH_BYTES = AQ_GEMV_NOALLOC_MAX_MK + 256;  // codes [M, K] then scales [M]
static_assert(AQ_GEMV_NOALLOC_MAX_MK % 256 == 0, "the scales start 256-byte aligned");
static __device__ __align__(256) uint8_t scratch[NOALLOC_SCRATCH_BYTES];

// In host code `scratch` is only a handle: the array's device address is asked of the runtime, once per
// device (each GPU holds its own copy at its own address) with that device current, and kept.  Two threads
// that come first at the same time both store the same address.
static int scratch_of_current_device(void** out) {
  static void* ptrs[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= 64) return AQ_E_RANGE;
  void* p = __atomic_load_n(&ptrs[dev], __ATOMIC_ACQUIRE);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return AQ_E_NULL;
    __atomic_store_n(&ptrs[dev], p, __ATOMIC_RELEASE);
  }
  *out = p;
  return AQ_OK;
}

}  // namespace aq

extern "C" int aq_gemv_w8a8_decode_noalloc(const void* x, int x_dtype, const int8_t* wq, const float* sw,
                                           const void* bias, int bias_dtype, const void* residual, void* y,
                                           int y_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
  // sizes beyond the scratch are rejected before anything else is looked at: AQ_E_RANGE, "size beyond ..."
  if (M > 0 && K > 0 && (M > 16 || M * K > (int64_t)AQ_GEMV_NOALLOC_MAX_MK)) return M > 16 ? AQ_E_SHAPE : AQ_E_RANGE;
  void* ws = nullptr;
  const int rc = aq::scratch_of_current_device(&ws);
  if (rc) return rc;
  // The scratch keeps the previous call's contents; nothing in it has to start at zero: the quantiser
  // writes all M rows of codes and all M scales before the GEMV reads exactly those.
  return aq_gemv_w8a8_decode_residual(x, x_dtype, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, ws,
                                      aq::NOALLOC_SCRATCH_BYTES, stream);
}

extern "C" int aq_gemv_w8a8_decode_attn(const float* partials, int64_t n_slices, int64_t head_dim, const int8_t* wq,
                                        const float* sw, const void* bias, int bias_dtype, const void* residual,
                                        void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
  int mt = 0;
  int rc = gemv_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, &mt);
  if (rc) return rc;
  if ((head_dim != 64 && head_dim != 128) || (K % head_dim) != 0 || n_slices <= 0) return AQ_E_SHAPE;
  // the in-kernel merge keeps every slice of a lane's vectors in registers
  if (M > 8 || K > AQ_GEMV_ATTN_MAX_K || n_slices > AQ_GEMV_ATTN_MAX_SLICES) return AQ_E_RANGE;
  if (M == 0 || N == 0) return AQ_OK;
  if (!partials) return AQ_E_NULL;
  if (aq::check_ptr16(partials)) return AQ_E_ALIGN;
  aq::GemvArgs a{};
  a.parts = partials;
  a.parts_ns = (int)n_slices;
  a.parts_d = (int)head_dim;
  a.wq = wq;
  a.sw = sw;
  a.bias = bias;
  a.res = residual;
  a.ldr = N;
  a.y = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = y_dtype;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return aq::launch_gemv_rows_attn(a, st);
}

extern "C" int aq_gemv_w8a8_decode_rmsnorm(const void* x, int x_dtype, const void* gamma, float eps, const int8_t* wq,
                                           const float* sw, const void* bias, int bias_dtype, const void* residual,
                                           void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* ws,
                                           size_t ws_bytes, void* stream) {
  if (x_dtype != AQ_F32 && x_dtype != AQ_BF16) return AQ_E_DTYPE;
  int mt = 0;
  int rc = gemv_check(wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, &mt);
  if (rc || M == 0 || N == 0) return rc;
  if (!x || !gamma || !ws) return AQ_E_NULL;
  if (aq::check_ptr16(x) || aq::check_ptr16(gamma) || aq::check_ptr16(ws)) return AQ_E_ALIGN;
  if (ws_bytes < aq_gemv_w8a8_workspace_bytes(M, K)) return AQ_E_WORKSPACE;
  {  // one launch where the GEMV kernel normalises and quantises the rows itself
    aq::GemvArgs a{};
    a.x = x;
    a.gamma = gamma;
    a.eps = eps;
    a.wq = wq;
    a.sw = sw;
    a.bias = bias;
    a.res = residual;
    a.ldr = N;
    a.y = y;
    a.M = (int)M;
    a.N = (int)N;
    a.K = (int)K;
    a.bias_dtype = bias_dtype;
    a.y_dtype = y_dtype;
    const int frc = gemv_dispatch_fused(a, x_dtype, mt, static_cast<hipStream_t>(stream));
    if (frc >= 0) return frc;
  }
  int8_t* xq = static_cast<int8_t*>(ws);
  float* sx = reinterpret_cast<float*>(static_cast<char*>(ws) + aq::align256((size_t)(M * K)));
  rc = aq_rmsnorm_quant_rowwise_i8(x, x_dtype, gamma, x_dtype, eps, M, K, K, xq, sx, stream);
  if (rc) return rc;
  return aq_gemv_w8a8_codes_residual(xq, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_gemv_w8a8_decode_swiglu_ok(int x_dtype, int64_t M, int64_t F, int64_t K) {
  return x_dtype == AQ_BF16 && aq::gemv_swiglu_ok(M, F, K) ? 1 : 0;
}

extern "C" int aq_gemv_w8a8_decode_swiglu(const void* x, int x_dtype, const void* gamma, float eps, const int8_t* wq,
                                          const float* sw, const void* bias, int bias_dtype, void* h, int h_dtype,
                                          int64_t M, int64_t F, int64_t K, void* stream) {
  if (x_dtype != AQ_F32 && x_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (F < 0 || F > (1 << 24)) return F < 0 ? AQ_E_SHAPE : AQ_E_RANGE;
  int mt = 0;
  int rc = gemv_check(wq, sw, bias, bias_dtype, nullptr, h, h_dtype, M, 2 * F, K, &mt);
  if (rc || M == 0 || F == 0) return rc;
  if (!x) return AQ_E_NULL;
  if (aq::check_ptr16(x) || aq::check_ptr16(gamma)) return AQ_E_ALIGN;
  if (!aq_gemv_w8a8_decode_swiglu_ok(x_dtype, M, F, K)) return AQ_E_RANGE;  // the caller takes the separate launches
  aq::GemvArgs a{};
  a.x = x;
  a.gamma = gamma;
  a.eps = eps;
  a.wq = wq;
  a.sw = sw;
  a.bias = bias;
  a.y = h;
  a.M = (int)M;
  a.N = (int)(2 * F);
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = h_dtype;
  return aq::launch_gemv_rows_swiglu(a, static_cast<hipStream_t>(stream));
}

extern "C" int aq_gemv_w8a8_decode(const void* x, int x_dtype, const int8_t* wq, const float* sw,
                                   const void* bias, int bias_dtype, void* y, int y_dtype, int64_t M,
                                   int64_t N, int64_t K, void* ws, size_t ws_bytes, void* stream) {
  return aq_gemv_w8a8_decode_residual(x, x_dtype, wq, sw, bias, bias_dtype, nullptr, y, y_dtype, M, N, K, ws, ws_bytes,
                                      stream);
}

// ---------------------------------------------------------------------------
// 17 rows and more, quantised in the launch that multiplies them: the decode kernel on tiles of up to 16 rows (gemv_rows.hip).
static aq::Tiling few_rows(int x_dtype, int norm, int fp8, int64_t M, int64_t N, int64_t K) {
  if ((x_dtype != AQ_F32 && x_dtype != AQ_BF16) || M <= 16 || N < 1 || K < 1 || K % 16) return aq::TILED_NOT;
  if ((fp8 || norm) && (x_dtype != AQ_BF16 || (fp8 && norm))) return aq::TILED_NOT;
  return aq::gemv_rows_tiled(fp8 ? aq::ROWS_FP8 : fused_kind(norm != 0, x_dtype == AQ_BF16), M, N, K);
}

extern "C" int aq_linear_few_rows_ok(int x_dtype, int norm, int fp8, int64_t M, int64_t N, int64_t K) {
  return few_rows(x_dtype, norm, fp8, M, N, K) != aq::TILED_NOT;
}

extern "C" int aq_linear_few_rows_queued_ok(int x_dtype, int norm, int fp8, int64_t M, int64_t N, int64_t K) {
  return few_rows(x_dtype, norm, fp8, M, N, K) == aq::TILED;
}

extern "C" int aq_linear_few_rows(const void* x, int x_dtype, const void* gamma, float eps, const void* wq, int fp8, const float* sw,
                                  const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype, int64_t M, int64_t N,
                                  int64_t K, void* stream) {
  if ((x_dtype != AQ_F32 && x_dtype != AQ_BF16) || (y_dtype != AQ_F32 && y_dtype != AQ_BF16)) return AQ_E_DTYPE;
  if (bias && bias_dtype != AQ_F32 && bias_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (M < 0 || N < 0 || K <= 0 || K % 16 || (gamma && !(eps >= 0.0f))) return AQ_E_SHAPE;
  if (M == 0 || N == 0) return AQ_OK;
  if (!x || !wq || !sw || !y) return AQ_E_NULL;
  if (aq::check_ptr16(x) || aq::check_ptr16(gamma) || aq::check_ptr16(wq) || aq::check_ptr16(y) || aq::check_ptr(residual, 4) ||
      aq::check_ptr(sw, 4) || aq::check_ptr(bias, bias_dtype == AQ_BF16 ? 2 : 4))
    return AQ_E_ALIGN;
  if (!aq_linear_few_rows_ok(x_dtype, gamma != nullptr, fp8, M, N, K)) return AQ_E_RANGE;
  aq::GemvArgs a{};
  a.x = x;
  a.gamma = gamma;
  a.eps = eps;
  a.wq = static_cast<const int8_t*>(wq);
  a.sw = sw;
  a.bias = bias;
  a.res = residual;
  a.ldr = N;
  a.y = y;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.bias_dtype = bias_dtype;
  a.y_dtype = y_dtype;
  return aq::launch_gemv_rows(a, fp8 ? aq::ROWS_FP8 : fused_kind(gamma != nullptr, x_dtype == AQ_BF16), static_cast<hipStream_t>(stream));
}
