// Prefill GEMMs on the CDNA4 matrix cores: int8 x int8 -> int32
// (v_mfma_i32_32x32x32_i8) and FP8 e4m3 x e4m3 -> fp32
// (v_mfma_scale_f32_32x32x64_f8f6f4 with unit scales), one kernel template.
//
//   C[m, n] = sum_k A[m, k] * B[n, k]     A = activation codes [M, K]
//                                         B = weight codes     [N, K]
// Both operands are K-contiguous, which is exactly the MFMA operand order
// (each lane feeds 16 or 32 consecutive k of one row), so no transpose is ever
// materialised.  A workgroup of 8 wavefronts (two per SIMD) owns a 256 x 128
// tile of C; each wavefront a 64 x 64 sub-tile held as 2 x 2 MFMA 32x32
// accumulators.  (When that gives too few tiles to occupy the device, the
// tile is 128 x 128, 128 x 64, 128 x 32, 64 x 64 or 64 x 32 instead, on four or
// two wavefronts.)  K is walked in 128-byte steps through three to six LDS
// stages that are filled by direct global->LDS loads (no register staging), with an XOR
// permutation of 16-byte pieces that makes the fragment reads bank-conflict
// free; the loop is software-pipelined so that LDS reads and global loads of
// later sub-steps are issued between the MFMAs of the current one, with one
// workgroup barrier per K step.  The epilogue is fused and runs straight from
// the accumulator registers: int32 store, or dequantise (+bias) and cast.
// Two other kernels take calls from here: gemm_walk.hip the 256 x 128 and
// 256 x 192 tiles of K from 512 (even N), gemm_slices.hip up to a few hundred
// rows.
#include "aq_gemm.h"

namespace aq {

// Shape of a workgroup: WM x WN x WK wavefronts, each accumulating a (32 TM) x (32 TN) sub-tile
// (TM x TN MFMA 32x32 accumulators); K walked in BK-byte steps through NSTAGE LDS stages.
//   <4, 2, 2, 2, 1, 128, 3>  256 x 128 tile, 8 wavefronts (two per SIMD) of 64 x 64, 3 stages of 48 KiB;
//   <2, 2, 2, 2, 1, 128, 3>  128 x 128 tile, 4 wavefronts (one per SIMD) of 64 x 64, 3 stages of 32 KiB (4 fit
//                            and were 1-5 % slower on this tile's shapes);
//   <2, 2, 2, 1, 1, 128, 4>  128 x 64 tile, 4 wavefronts of 64 x 32,
//   <4, 1, 1, 1, 1, 128, 4>  128 x 32 tile, 4 wavefronts of 32 x 32,
//   <2, 2, 1, 1, 1, 128, 4>  64 x 64 tile, 4 wavefronts of 32 x 32, and
//   <2, 1, 1, 1, 1, 128, 6>  64 x 32 tile, 2 wavefronts of 32 x 32 (six stages of 12 KiB: 2-20 % faster than four,
//                            while the other three were fastest with four of the 3..8 that fit, three costing
//                            them 5-25 %: their K loop runs at the latency of its loads): for a few
//                            hundred rows, where wider tiles leave most compute units without one.  A
//                            workgroup's time is the matrix-core time of its whole tile, rows past M included
//                            (128 x 128 x 2048: 16 K steps of 16 MFMAs, 3.9 us per compute unit), so with tiles
//                            to spare the smaller tile is the faster launch (128 x 2048 x 2048, weights from
//                            HBM: 12.4 us on 16 tiles of 128 x 128, 8.7 us on 64 of 128 x 32, 6.9 us on 128 of
//                            64 x 32);
// The same five tiles on twice the wavefronts, the two that share a sub-tile each taking half of every K step
// and exchanging half of their accumulators through LDS at the end (WK = 2, so that each finishes and stores
// half of the sub-tile), were measured against these in one process over 48..512 rows and four weight shapes:
// 2-6 % slower every time (128 x 128 at 512 x 8192 x 2048: 15.0 against 14.1 us; 64 x 64 at 128 x 8192 x 2048:
// 8.8 against 8.4 us).  The lab build keeps the 128 x 128 one (<2, 2, 2, 2, 2, 128, 3>) so that the K-split
// code stays compiled and tested.
// Shapes that (but for the first one on FP8) only the lab build instantiates.  Measured, none faster on int8 with
// real operand data: under a matrix-core load with toggling operands this part runs against its power limit, and
// fewer LDS reads per MFMA buy clock, not rate (8192^3: 2.31-2.42 POP/s for every shape below and for the
// 256 x 128 tile alike, while the clock moves between 1.47 and 1.65 GHz).  FP8, which is throttled less, gains 5 %
// from the first one at 8192^3 (417 against 438 us: its K loop runs at 84 % of the matrix cores' own time with 6 %
// of it waited at the stage barriers, where the 256 x 128 tile waits 40 %; a 64 x 64 sub-tile reads 32 bytes of
// fragments per wavefront and cycle, 128 per compute unit, which is all the LDS delivers, before the fills'
// writes; the 128 x 128 sub-tile needs half); the product takes it for FP8 launches of at least two rounds of
// 256 x 256 tiles.
//   <2, 2, 4, 4, 1, 64, 4>   256 x 256 tile, 4 wavefronts (one per SIMD) of 128 x 128: 256 accumulator
//                            registers per lane (the AGPR half of the register file), 8 fragment reads per
//                            16 MFMAs instead of 16, half the LDS fill per MFMA; 4 stages of 32 KiB; whole K
//                            steps, whole 256-row multiples, even N, no residual (one K-loop and one epilogue
//                            variant: with all three epilogues and both K loops the kernel was 45 000 lines of
//                            machine code whose spilled values came back from scratch one memory round trip at a
//                            time, 45 k cycles of epilogue per tile; now 12-16 k);
//   <4, 2, 2, 4, 1, 64, 4>   256 x 256 tile, 8 wavefronts of 64 x 128: 6 fragment reads per 8 MFMAs;
//   <2, 2, 4, 2, 1, 128, 3>  256 x 128 tile, 4 wavefronts of 128 x 64.
// Two independent 4-wavefront workgroups per compute unit (256 x 128 or 128 x 128 tiles with 64-byte stages, so
// that one's epilogue overlaps the other's loop) were measured too: 8192^3 in 459 and 556 us against 310 us with
// all-zero operands.
template <int WM_, int WN_, int TM_, int TN_, int WK_, int BK_, int NSTAGE_>
struct Shape {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, WK = WK_, BK = BK_, NSTAGE = NSTAGE_;
  static constexpr int NWAVES = WM * WN * WK, NTHREADS = NWAVES * 64;
  static constexpr int WAVE_M = 32 * TM, WAVE_N = 32 * TN;
  static constexpr int BM = WM * WAVE_M, BN = WN * WAVE_N;
  static constexpr int STAGE = (BM + BN) * BK;
  // Sub-tiles of 16 accumulators (128 x 128 per wavefront): the 256 accumulator registers leave no room to hold a
  // lane's 64 per-row scales through the K loop, so the tile's BM scales wait in LDS behind the stages instead;
  // such shapes also compile one K-loop variant (whole K steps) and one epilogue variant only (see gemm_kernel).
  static constexpr bool BIG = TM * TN >= 16;
  static constexpr int SX_BYTES = BIG ? BM * 4 : 0;
  static constexpr int LDS_BYTES = NSTAGE * STAGE + SX_BYTES;
  static constexpr int LDS_LINES = NSTAGE * STAGE + BN * BK;  // with a stage more of B (see gemm_tile)
  static_assert(BK == 64 || BK == 128, "K bytes per stage");
  static_assert(NWAVES % 2 == 0, "the piece permutation assumes a wavefront's row groups share parity");
  static_assert((BM * BK / 1024) % NWAVES == 0 && (BN * BK / 1024) % NWAVES == 0, "whole 1 KiB loads per wavefront");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of one compute unit");
  static_assert((NSTAGE - 1) * ((BM + BN) * BK / 16 / NTHREADS) <= 63, "the loads in flight fit the 6-bit counter");
};
using ShapeLarge = Shape<4, 2, 2, 2, 1, 128, 3>;
using ShapeSmall = Shape<2, 2, 2, 2, 1, 128, 3>;
using ShapeN64 = Shape<2, 2, 2, 1, 1, 128, 4>;
using ShapeN32 = Shape<4, 1, 1, 1, 1, 128, 4>;
using ShapeM64N64 = Shape<2, 2, 1, 1, 1, 128, 4>;
using ShapeM64N32 = Shape<2, 1, 1, 1, 1, 128, 6>;
using ShapeHuge = Shape<2, 2, 4, 4, 1, 64, 4>;  // product: large FP8 launches of odd 64-byte K steps (see huge_fp8_ok)
#ifdef AQ_LAB
using ShapeTall = Shape<2, 2, 4, 2, 1, 128, 3>;
using ShapeHuge8 = Shape<4, 2, 2, 4, 1, 64, 4>;
using ShapePair = Shape<2, 2, 2, 2, 2, 128, 3>;
#endif
// Issue order of one pipeline slot, as scheduling groups: GROUPS times
// [1 MFMA, NDS LDS reads, this group's share of the NLD global loads].
// (0x008 = MFMA, 0x100 = LDS read, 0x020 = vector-memory read.)
template <int G, int GROUPS, int NDS, int NLD>
__device__ __forceinline__ void sched_pattern() {
  if constexpr (G < GROUPS) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, NDS, 0);
    constexpr int nl = ((G + 1) * NLD) / GROUPS - (G * NLD) / GROUPS;
    if constexpr (nl > 0) __builtin_amdgcn_sched_group_barrier(0x020, nl, 0);
    sched_pattern<G + 1, GROUPS, NDS, NLD>();
  }
}

#ifdef AQ_LAB
__device__ long long aq_lab_clock[16];
#endif
// How the rows of A and B lie in 128-byte lines, K and the distance between A's rows being given:
//   EXACT  K is a whole number of BK-byte steps and rows are K apart: every 16-byte piece of every step lies inside its row and the
//          global->LDS loads need no per-lane range logic: a loop-invariant lane offset per row group and the K step as a scalar offset, no
//          vector ALU work per load.
//   ANY    K may end inside a step, and each load checks it.
//   LINES  the same, and the loads of B are whole lines, wherever its rows begin (see `phase`); for long K.
enum Rows { EXACT_ROWS, ANY_ROWS, LINE_ROWS };
template <bool FP8, int OUT, class S, Rows ROWS>
__device__ __forceinline__ void gemm_tile(const GemmArgs& p, uint8_t* smem, int pid) {
  constexpr bool EXACT = ROWS == EXACT_ROWS, LINES = ROWS == LINE_ROWS;
  constexpr int WM = S::WM, WN = S::WN, TM = S::TM, TN = S::TN, WK = S::WK, BK = S::BK, NSTAGE = S::NSTAGE;
  constexpr int NWAVES = S::NWAVES, NTHREADS = S::NTHREADS, WAVE_M = S::WAVE_M, WAVE_N = S::WAVE_N;
  constexpr int BM = S::BM, BN = S::BN, STAGE = S::STAGE;
  constexpr bool BIG = S::BIG;
  static_assert(TM % WK == 0, "the K-split pair divides the sub-tile's row blocks");
  static_assert(!BIG || (EXACT && WK == 1), "big sub-tiles: whole K steps, no K-split pair");
  constexpr int TME = TM / WK;  // row blocks a wavefront finishes and stores
  constexpr int A_LOADS = BM * BK / 16 / NTHREADS;  // 16-byte vectors per thread per K step
  constexpr int B_LOADS = BN * BK / 16 / NTHREADS;
  // NSTAGE stages of [A tile BM x BK bytes][B tile BN x BK bytes], rows unpadded.
  // Global->LDS loads land 64 lanes x 16 B contiguously (1 KiB: RPG = 8 rows of
  // 128 B or 16 rows of 64 B), so the bank-conflict-free layout is obtained by
  // permuting which 16-byte piece of its row each lane fetches: piece c of row r
  // is stored at slot c ^ ((r / RPL) % PPR), with PPR = BK / 16 pieces per row and
  // RPL = 256 / BK rows per bank line.  LDS has 64 banks here (256 bytes per bank
  // line) and a 16-byte-per-lane read is served 16 lanes at a time, so 16
  // consecutive rows reading the same piece must land on 16 distinct slots:
  // r % RPL picks the part of the bank line, the permuted piece the slot in it.
  constexpr int PPR = BK / 16, RPL = 256 / BK, RPG = 1024 / BK;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_k = WK == 1 ? 0 : wave / (WM * WN), wave_mn = WK == 1 ? wave : wave % (WM * WN);
  const int wave_m = wave_mn / WN, wave_n = wave_mn % WN;

  int tile_m, tile_n;
  tile_of_block(pid, p.tiles_m, p.tiles_n, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int M = p.M, N = p.N, K = p.K;

  // Tile-local buffer descriptors: rows past the M / N edge fall outside and read as zero.
  const int rows_a = (M - m0) < BM ? (M - m0) : BM;
  const int rows_b = (N - n0) < BN ? (N - n0) : BN;
  const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A + (int64_t)m0 * p.lda, (uint32_t)rows_a * (uint32_t)p.lda);
  const __amdgpu_buffer_rsrc_t Br = make_rsrc(p.B + (int64_t)n0 * K, (uint32_t)rows_b * (uint32_t)K);

  const int col = lane & 31;
  const int rq = (lane >> 5) * 4;  // row offset of this lane's half inside each group of 8 rows
  // first row of the part of the sub-tile this wavefront finishes (wavefront-uniform: kept scalar)
  const int mw = __builtin_amdgcn_readfirstlane(m0 + wave_m * WAVE_M + wave_k * (32 * TME));

  // One load instruction of a wavefront fills 1 KiB = RPG tile rows.  Wavefront w
  // owns the row groups w, w+NWAVES, w+2*NWAVES, ... of A and of B.
  // Row of lane l in group j: RPG j + l / PPR; (row / RPL) % PPR is the same for every
  // group of a wavefront because RPG NWAVES / RPL is a multiple of PPR.
  static_assert((RPG * NWAVES / RPL) % PPR == 0, "the piece permutation is the same for all row groups of a wavefront");
  const int ld_row = wave * RPG + lane / PPR;  // + RPG*NWAVES*i
  const int ld_piece = ((lane % PPR) ^ ((ld_row / RPL) % PPR)) * 16;  // piece this lane fetches
  const uint32_t ld_off = (uint32_t)ld_row * (uint32_t)K + ld_piece;
  const uint32_t row32 = (uint32_t)(RPG * NWAVES) * (uint32_t)K;  // byte distance between a wavefront's row groups
  constexpr int NLOADS = A_LOADS + B_LOADS;
  const int nk = (K + BK - 1) / BK;
  // Two accumulator columns per wavefront, bf16 outputs and an even N: a lane's two are neighbours of the output, which the order of
  // B's rows in a stage makes them (column 2 c + j behind accumulator j of lane c), so that a row's 32 lanes store a whole
  // 128-byte line (fp32 and int32 outputs fill one with a column each).
  constexpr bool ADJ = TN == 2 && OUT == OUT_BF16;
  const bool pair_ok = (N & 1) == 0;  // uniform: bf16 rows start dword-aligned, pairs never straddle N
  uint32_t ld_vo[A_LOADS > B_LOADS ? A_LOADS : B_LOADS];  // lane offset of row group i; EXACT: A and B alike
  uint32_t ld_vb[ADJ || !EXACT ? B_LOADS : 1];             // ... of B, where its rows have an order or a distance of their own
  // row of the tile of B that row r of a stage holds
  auto b_row = [&](int r) { return ADJ && pair_ok ? (r & ~63) + 2 * (r & 31) + ((r >> 5) & 1) : r; };
  // LINES: rows of B begin anywhere in a line, `phase` bytes behind its beginning (A's rows the caller lays out: lda).  A stage of B holds a
  // line of every row: line t has bytes BK t - phase .. + BK of the row, piece q of a step (of the row's own bytes) in piece q's place of line
  // s, or of line s + 1 where 16 q + phase is past the line's end.  Step s takes pieces of both, so one stage more of B is kept, and a load
  // brings one line of each row where a step of the row's own bytes would touch two.
  auto phase = [&](int row) { return (int)((reinterpret_cast<uintptr_t>(p.B) + (uint64_t)(uint32_t)(n0 + row) * (uint32_t)K) & (BK - 1)); };
  // Byte of the row that this lane's piece of line 0 begins at.  Rows 8 apart have one phase, so it is the same for every row group (ADJ: for
  // every other one).
  constexpr int NKB = ADJ ? 2 : 1;
  int ld_kb[LINES ? NKB : 1];
  if constexpr (EXACT) {
#pragma unroll
    for (int i = 0; i < (A_LOADS > B_LOADS ? A_LOADS : B_LOADS); ++i) ld_vo[i] = ld_off + (uint32_t)i * row32;
    if constexpr (ADJ) {
#pragma unroll
      for (int i = 0; i < B_LOADS; ++i) ld_vb[i] = (uint32_t)b_row(ld_row + i * RPG * NWAVES) * (uint32_t)K + ld_piece;
    }
  } else {
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) ld_vo[i] = (uint32_t)(ld_row + i * RPG * NWAVES) * (uint32_t)p.lda + ld_piece;
    if constexpr (LINES) {
#pragma unroll
      for (int i = 0; i < NKB; ++i) {
        const int ph = phase(b_row(ld_row + i * RPG * NWAVES));
        ld_kb[i] = ld_piece + ph < BK ? ld_piece : ld_piece - BK;
      }
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i)
      ld_vb[i] = (uint32_t)b_row(ld_row + i * RPG * NWAVES) * (uint32_t)K + (uint32_t)(LINES ? ld_kb[LINES ? i % NKB : 0] + BK : ld_piece);
  }
  auto b_off = [&](int i) { return ADJ || !EXACT ? ld_vb[ADJ || !EXACT ? i : 0] : ld_vo[i]; };
  constexpr int A_STAGE = LINES ? BM * BK : STAGE;                                  // bytes between stages of A
  constexpr int B_FIRST = NSTAGE * A_STAGE, B_LAST = B_FIRST + NSTAGE * (BN * BK);  // LINES: B's have a ring of their own, of NSTAGE + 1
  auto behind = [](int at) { return at == B_LAST ? B_FIRST : at + BN * BK; };
  int b_ld = B_FIRST;  // LINES: where the line of B goes that issue_load requests
  // load number `idx` (0..NLOADS-1) of K step kt into stage buffer `buf`; LINES: of A, and of line kt + 1 of B
  auto issue_load = [&](int kt, int buf, int idx, auto kind) {
    if constexpr (EXACT) {
      // steps past the last one request the last step again (into a stage nobody reads): in range by construction
      const int k0s = (decltype(kind)::value == 2 || kt < nk ? kt : nk - 1) * BK;  // wavefront-uniform: a scalar offset
      uint8_t* st = smem + buf * STAGE + wave * 1024;
      if (idx < A_LOADS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Ar, (lds_void*)(st + idx * (1024 * NWAVES)), 16, ld_vo[idx], k0s, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Br, (lds_void*)(st + BM * BK + (idx - A_LOADS) * (1024 * NWAVES)), 16,
                                                 b_off(idx - A_LOADS), k0s, 0, 0);
      return;
    }
    // K is a multiple of 16: a piece is all in or all out.  Pieces past K would alias the next row, so they are pushed outside the
    // descriptor (-> zeros); so are all of the steps past the last one.
    uint8_t* sta = smem + buf * A_STAGE + wave * 1024;
    uint8_t* stb = (LINES ? smem + b_ld : smem + buf * STAGE + BM * BK) + wave * 1024;
    if constexpr (!LINES) {
      const int k0 = kt * BK;
      const bool in = k0 + ld_piece < K;
      if (idx < A_LOADS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Ar, (lds_void*)(sta + idx * (1024 * NWAVES)), 16, in ? ld_vo[idx] + (uint32_t)k0 : OOB_OFFSET, 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Br, (lds_void*)(stb + (idx - A_LOADS) * (1024 * NWAVES)), 16,
                                                 in ? b_off(idx - A_LOADS) + (uint32_t)k0 : OOB_OFFSET, 0, 0, 0);
    } else {
      // most steps need no check (a compare and a select in each load are 10 % of an int8 launch of 64 x 64 tiles)
      constexpr bool WHOLE = decltype(kind)::value == 2;      // nothing of the step or of the line is past K
      const int k0s = (WHOLE || kt < nk ? kt : nk - 1) * BK;  // less than the bytes behind the descriptor
      const int i = idx - A_LOADS;
      if (idx < A_LOADS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Ar, (lds_void*)(sta + idx * (1024 * NWAVES)), 16,
                                                 WHOLE || kt * BK + ld_piece < K ? ld_vo[idx] : OOB_OFFSET, k0s, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Br, (lds_void*)(stb + i * (1024 * NWAVES)), 16,
                                                 WHOLE || kt * BK + BK + ld_kb[LINES ? i % NKB : 0] < K ? b_off(i) : OOB_OFFSET, k0s, 0, 0);
    }
  };

#ifdef AQ_LAB_STALL
  const long long tl_start = clock64();
#endif
  using acc_t = typename Acc<FP8>::type;
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // Fragment reads: lane -> tile row lane%32; its K pieces within a row
  // are (ks*2 + lane/32) for int8 (16 B per MFMA) and (ks*4 + (lane/32)*2 + {0,1})
  // for FP8 (32 B per MFMA); slot = piece ^ ((row / RPL) % PPR), which depends on lane%32 only
  // (sub-tile rows start at multiples of 32).
  const int fr_a = (wave_m * WAVE_M + (lane & 31)) * BK;
  const int fr_b = BM * BK + (wave_n * WAVE_N + (lane & 31)) * BK;
  const int fsw = ((lane & 31) / RPL) % PPR;
  constexpr int KSUB = FP8 ? 64 : 32;  // K per MFMA
  constexpr int NKS = BK / KSUB / WK;  // MFMA sub-steps per stage and wavefront: 4 or 2 (int8), 2 or 1 (FP8)
  // this wavefront's sub-steps of a stage start at piece wave_k * NKS * KSUB / 16; NKS is a power
  // of two, so adding the sub-step number to that base is an XOR and folds into the permutation
  const int swz = (FP8 ? ((((lane >> 5) * 2) ^ fsw) << 4) : (((lane >> 5) ^ fsw) << 4)) ^ (wave_k * NKS * KSUB);
  using frag_t = typename Frag<FP8>::type;
  // LINES: pieces of a step from this byte on lie in the line behind, by accumulator column where those are rows of two phases (ADJ)
  constexpr int PP = FP8 ? 2 : 1, NJ = ADJ ? TN : 1;  // 16-byte pieces of a lane's fragment
  int fb_end[LINES ? NJ : 1];
  if constexpr (LINES) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      fb_end[j] = BK - phase(b_row(wave_n * WAVE_N + j * 32 + (lane & 31))) - wave_k * NKS * KSUB - (lane >> 5) * PP * 16;
  }
  int line_cur = 0;  // LINES: offset of the line of B that belongs to the stage whose fragments are read, and of the one behind
  int line_next = 0;
  auto read_b = [&](int ks, int j) -> frag_t {
    auto piece = [&](int pp) {
      const int o = ((ks * 2 * PP) << 4 ^ swz ^ pp << 4) + fr_b - BM * BK + j * 32 * BK;
      return *reinterpret_cast<const v4i*>(smem + o + (ks * KSUB + pp * 16 >= fb_end[ADJ && LINES ? j : 0] ? line_next : line_cur));
    };
    if constexpr (!FP8) {
      return piece(0);
    } else {
      const v4i lo = piece(0), hi = piece(1);
      return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    }
  };
  auto load_frags = [&](const uint8_t* st, int ks, frag_t (&a)[TM], frag_t (&b)[TN]) {
    if constexpr (LINES) {
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j] = read_b(ks, j);
    }
    if constexpr (!FP8) {
      const int o = ((ks * 2) << 4) ^ swz;
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const v4i*>(st + fr_a + i * 32 * BK + o);
      if constexpr (!LINES) {
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = *reinterpret_cast<const v4i*>(st + fr_b + j * 32 * BK + o);
      }
    } else {
      const int o0 = ((ks * 4) << 4) ^ swz, o1 = o0 ^ 16;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(st + fr_a + i * 32 * BK + o0);
        const v4i hi = *reinterpret_cast<const v4i*>(st + fr_a + i * 32 * BK + o1);
        a[i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
      if constexpr (!LINES) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const v4i lo = *reinterpret_cast<const v4i*>(st + fr_b + j * 32 * BK + o0);
          const v4i hi = *reinterpret_cast<const v4i*>(st + fr_b + j * 32 * BK + o1);
          b[j] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
      }
    }
  };

  // One pipeline slot = the TM*TN MFMAs of one sub-step, with the LDS reads of
  // the next sub-step's fragments and (LOADS) a share of the global->LDS loads
  // of a later stage interleaved between them, so that a wavefront (the only
  // one on its SIMD) never queues a burst of memory instructions in front of
  // the matrix core.
  frag_t af[2][TM], bf[2][TN];
  // fragment number f of a sub-step, in the order the next sub-step's MFMAs need them: A0, B0 .. B(TN-1), A1 ..
  auto load_frag = [&](const uint8_t* st, int ks, int f, frag_t (&a)[TM], frag_t (&b)[TN]) {
    const bool is_a = f == 0 || f > TN;
    const int idx = f == 0 ? 0 : f <= TN ? f - 1 : f - TN;
    if (LINES && !is_a) {
      b[idx] = read_b(ks, idx);
      return;
    }
    const uint8_t* base = st + (is_a ? fr_a : fr_b) + idx * 32 * BK;
    if constexpr (!FP8) {
      const v4i v = *reinterpret_cast<const v4i*>(base + (((ks * 2) << 4) ^ swz));
      if (is_a) a[idx] = v; else b[idx] = v;
    } else {
      const int o0 = ((ks * 4) << 4) ^ swz;
      const v4i lo = *reinterpret_cast<const v4i*>(base + o0);
      const v4i hi = *reinterpret_cast<const v4i*>(base + (o0 ^ 16));
      const v8i v = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if (is_a) a[idx] = v; else b[idx] = v;
    }
  };
  // slot number Q (0 = slot A .. NKS-1) issues loads [Q*NLOADS/NKS, (Q+1)*NLOADS/NKS) of its stage.
  // The order is written out and fenced: MFMA, then the fragment read(s) and at most a global load that
  // it covers, so that every memory instruction is issued in the shadow of a running MFMA and no fragment is
  // read right in front of its first use (left to itself the scheduler bunches the reads before the MFMAs
  // that need them).  The last MFMAs of a slot carry no reads: the fragments have landed when the next slot starts.
  auto slot = [&](auto cur_c, const uint8_t* st_next, int ks_next, auto loads_c, int kt_ld, int buf_ld,
                  auto q_c) {
    constexpr int CUR = decltype(cur_c)::value;
    constexpr bool LOADS = decltype(loads_c)::value != 0;
    constexpr int Q = decltype(q_c)::value;
    constexpr int LD0 = (Q * NLOADS) / NKS, LPS = LOADS ? ((Q + 1) * NLOADS) / NKS - LD0 : 0;
    constexpr int NMMA = TM * TN, NFR = TM + TN;
    constexpr int GROUPS = NMMA > 4 ? NMMA - 2 : NMMA;  // MFMAs that carry memory instructions
    if constexpr (NMMA >= 8) {
      // Large sub-tiles (one wavefront per SIMD, or few fragment reads per MFMA): the fragment reads go out in
      // pairs behind every STRIDE-th MFMA and the global loads behind the MFMA after it.  Measured on a loop of
      // independent MFMAs with one wavefront per SIMD: two reads behind every fourth MFMA cost nothing (512.3
      // cycles per 16 MFMAs against 512.4 without reads), one behind every second 24 cycles, all eight first 40.
      constexpr int NPAIR = (NFR + 1) / 2, STRIDE = NMMA / NPAIR;
#pragma unroll
      for (int m = 0; m < NMMA; ++m) {
        acc[m / TN][m % TN] = mma<FP8>(af[CUR][m / TN], bf[CUR][m % TN], acc[m / TN][m % TN]);
        if (m % STRIDE == 0 && m / STRIDE < NPAIR) {
          load_frag(st_next, ks_next, 2 * (m / STRIDE), af[CUR ^ 1], bf[CUR ^ 1]);
          if (2 * (m / STRIDE) + 1 < NFR) load_frag(st_next, ks_next, 2 * (m / STRIDE) + 1, af[CUR ^ 1], bf[CUR ^ 1]);
        } else if (m % STRIDE == 1 && m / STRIDE < NPAIR) {
#pragma unroll
          for (int q = ((m / STRIDE) * LPS) / NPAIR; q < ((m / STRIDE + 1) * LPS) / NPAIR; ++q) issue_load(kt_ld, buf_ld, LD0 + q, loads_c);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
#pragma unroll
    for (int m = 0; m < NMMA; ++m) {
      acc[m / TN][m % TN] = mma<FP8>(af[CUR][m / TN], bf[CUR][m % TN], acc[m / TN][m % TN]);
      if (m < GROUPS) {
#pragma unroll
        for (int f = (m * NFR) / GROUPS; f < ((m + 1) * NFR) / GROUPS; ++f) load_frag(st_next, ks_next, f, af[CUR ^ 1], bf[CUR ^ 1]);
#pragma unroll
        for (int q = (m * LPS) / GROUPS; q < ((m + 1) * LPS) / GROUPS; ++q) issue_load(kt_ld, buf_ld, LD0 + q, loads_c);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using std::integral_constant;
  using k0 = integral_constant<int, 0>;
  using k1 = integral_constant<int, 1>;
  using q0 = integral_constant<int, 0>;
  using q1 = integral_constant<int, 1>;
  using q2 = integral_constant<int, 2>;
  using q3 = integral_constant<int, 3>;
  using no = integral_constant<int, 0>;
  using yes = integral_constant<int, 1>;
  using whole = integral_constant<int, 2>;

  // Rotated software pipeline over K steps ("stages" s = 0 .. nk-1):
  //   iteration s:  slots    MFMAs of (s, 0 .. NKS-2)       | read fragments (s, 1 .. NKS-1)
  //                 wait for this wavefront's loads of stage s+1, barrier
  //                 slot A   MFMAs of (s, last sub-step)    | read fragments (s+1, 0)
  // with the loads of stage s+NSTAGE spread from slot A of s over the slots of s+1.
  // At the barrier every wavefront holds the last fragments of stage s in
  // registers, so stage s's LDS buffer is free for the loads of stage s+NSTAGE right
  // after it, and stage s+1 is complete and visible for slot A's fragment reads.
  // Loads past the last K step are still issued (outside the descriptors they
  // write zeros into a stage nobody reads) so that the count of outstanding
  // loads per wavefront is the same at every wait.
  // Epilogue operands, requested right behind stage 0 so that their latency is
  // hidden behind the whole K loop and they never delay the first tile: per-row
  // activation scales as float4 per lane (accumulator register r of lane l
  // belongs to row (r/4)*8 + (l/32)*4 + r%4), per-column weight scale and bias
  // as one scalar per 32x32 tile column.  Nothing is done with the values until
  // the epilogue (bias stays a raw bit pattern), so no wait is placed here.
  float sx1 = 1.0f, sw1 = 1.0f;
  float sxr[BIG ? 1 : TME][4][4];  // [i][g][q]: row mw + i*32 + g*8 + rq + q (big sub-tiles: in LDS instead)
  float* const sx_lds = reinterpret_cast<float*>(smem + NSTAGE * STAGE);  // [BM], big sub-tiles only
  float swn[TN];
  uint32_t bias_raw[TN];
  const bool has_bias = OUT != OUT_I32 && p.bias != nullptr;
  const bool bias_bf16 = p.bias_dtype == AQ_BF16;
  auto column = [&](int j) { return ADJ && pair_ok ? 2 * col + j : j * 32 + col; };  // inside the wavefront's
  auto load_epilogue_operands = [&]() {
    if constexpr (FP8) {
      sx1 = *p.sx;
      sw1 = *p.sw;
      const __amdgpu_buffer_rsrc_t Bsr =
          make_rsrc(has_bias ? p.bias : (const void*)p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const uint32_t n = (uint32_t)(n0 + wave_n * WAVE_N + column(j));  // past N, or no bias: outside -> 0
        bias_raw[j] = bias_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(Bsr, n * 2u, 0, 0)
                                : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Bsr, n * 4u, 0, 0);
      }
    } else if constexpr (OUT != OUT_I32) {
      // rows past M fall outside the descriptor and read as zero (their outputs are never stored)
      const int rows_left = __builtin_amdgcn_readfirstlane((M - mw) > 0 ? (M - mw) : 0);
      const __amdgpu_buffer_rsrc_t Sr =
          make_rsrc(p.sx + (rows_left ? mw : 0), (uint32_t)(rows_left < 32 * TME ? rows_left : 32 * TME) * 4u);
      if constexpr (BIG) {
        // the tile's BM scales straight into LDS, 64 per load instruction; rows past M read as zero
        const __amdgpu_buffer_rsrc_t Tr = make_rsrc(p.sx + m0, (uint32_t)rows_a * 4u);
#pragma unroll
        for (int r = 0; r < BM / 64 / NWAVES; ++r)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(Tr, (lds_void*)(sx_lds + (r * NWAVES + wave) * 64), 4,
                                                   (uint32_t)((r * NWAVES + wave) * 64 + lane) * 4u, 0, 0, 0);
      } else if ((M & 3) == 0) {  // uniform: the 4 rows of a float4 are all in or all out, and 16-byte aligned
#pragma unroll
        for (int i = 0; i < TME; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const uint4 t = buffer_load_16(Sr, (uint32_t)(i * 32 + g * 8 + rq) * 4u);
            sxr[i][g][0] = __uint_as_float(t.x);
            sxr[i][g][1] = __uint_as_float(t.y);
            sxr[i][g][2] = __uint_as_float(t.z);
            sxr[i][g][3] = __uint_as_float(t.w);
          }
      } else {
#pragma unroll
        for (int i = 0; i < TME; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              sxr[i][g][q] = __uint_as_float(
                  (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Sr, (i * 32 + g * 8 + rq + q) * 4, 0, 0));
      }
      const __amdgpu_buffer_rsrc_t Wsr = make_rsrc(p.sw, (uint32_t)N * 4u);
      const __amdgpu_buffer_rsrc_t Bsr =
          make_rsrc(has_bias ? p.bias : p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const uint32_t n = (uint32_t)(n0 + wave_n * WAVE_N + column(j));  // past N: outside -> 0
        swn[j] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Wsr, n * 4u, 0, 0));
        bias_raw[j] = bias_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(Bsr, n * 2u, 0, 0)
                                : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Bsr, n * 4u, 0, 0);
      }
    }
  };
  if constexpr (LINES) {
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i)  // line 0: bytes before the row are never read
      __builtin_amdgcn_raw_ptr_buffer_load_lds(Br, (lds_void*)(smem + b_ld + wave * 1024 + i * (1024 * NWAVES)), 16,
                                               (uint32_t)ld_kb[LINES ? i % NKB : 0] < (uint32_t)K ? b_off(i) - BK : OOB_OFFSET, 0, 0, 0);
    b_ld = behind(b_ld);
  }
#pragma unroll
  for (int q = 0; q < NLOADS; ++q) issue_load(0, 0, q, yes{});
  asm volatile("" ::: "memory");  // keep the request order: stage 0, epilogue operands, the other stages
  load_epilogue_operands();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int st = 1; st < NSTAGE; ++st) {
    b_ld = behind(b_ld);
#pragma unroll
    for (int q = 0; q < NLOADS; ++q) issue_load(st, st, q, yes{});
  }

  // sub-steps 0 .. NKS-2 of a stage whose first fragments sit in af[C0]
  auto middle_slots = [&](auto c0_c, const uint8_t* stc, auto loads_c, int kt_ld, int buf_ld) {
    constexpr int C0 = decltype(c0_c)::value;
    using c0 = integral_constant<int, C0>;
    using c1 = integral_constant<int, C0 ^ 1>;
    if constexpr (NKS == 4) {
      slot(c0{}, stc, 1, loads_c, kt_ld, buf_ld, q1{});
      slot(c1{}, stc, 2, loads_c, kt_ld, buf_ld, q2{});
      slot(c0{}, stc, 3, loads_c, kt_ld, buf_ld, q3{});
    } else if constexpr (NKS == 2) {
      slot(c0{}, stc, 1, loads_c, kt_ld, buf_ld, q1{});
    }
  };
  // the fragment buffer the last sub-step of such a stage computes from
  auto last_of = [](auto c0_c) { return integral_constant<int, (NKS % 2 == 0) ? (decltype(c0_c)::value ^ 1) : decltype(c0_c)::value>{}; };

  AQ_WAIT_VMCNT((NSTAGE - 1) * NLOADS);  // all but the younger stages: stage 0 (and the operands) have landed
  AQ_BARRIER();
#ifdef AQ_LAB_STALL
  const long long tl_stage0 = clock64();
#endif
  b_ld = line_cur = B_FIRST;  // the loop's loads of B go where the line was that the step before took first
  line_next = behind(line_cur);
  auto next_lines = [&] {
    if constexpr (LINES) b_ld = line_cur, line_cur = line_next, line_next = behind(line_next);
  };
  load_frags(smem, 0, af[0], bf[0]);
  middle_slots(k0{}, smem, no{}, 0, 0);  // no loads to issue yet: every stage buffer is in flight
  __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0): the last fragments of stage 0 are in registers
  AQ_WAIT_VMCNT((NSTAGE - 2) * NLOADS);  // stage 1 has landed
  AQ_BARRIER();
  // slot A of stage 0: its buffer (0) is free now and takes stage NSTAGE
  next_lines();
  slot(last_of(k0{}), smem + A_STAGE, 0, yes{}, NSTAGE, 0, q0{});
  int b_prev = 0;  // buffer of stage s-1
#ifdef AQ_LAB_STALL
  long long st_t0 = 0, st_t1 = 0, st_sum = 0;
  const long long st_begin = clock64();
#endif
  auto stage_in = [&](int s, auto c0_c, auto loads_c, int b_prev, int b_cur, int b_next) {
    // sub-steps 0 .. NKS-2 of stage s; the rest of stage s-1+NSTAGE's loads go into stage s-1's buffer
    middle_slots(c0_c, smem + b_cur * A_STAGE, loads_c, s - 1 + NSTAGE, b_prev);
#ifdef AQ_LAB_STALL
    const long long st_now = clock64();
#endif
    __builtin_amdgcn_s_waitcnt(0xc07f);        // lgkmcnt(0): the last fragments of stage s are in registers
    AQ_WAIT_VMCNT((NSTAGE - 2) * NLOADS);  // stage s+1 has landed (later ones may still be in flight)
    AQ_BARRIER();
#ifdef AQ_LAB_STALL
    st_sum += st_t1 - st_t0;  // the previous step's wait: both of its clock reads have returned by now
    st_t0 = st_now;
    st_t1 = clock64();
#endif
    // slot A: last sub-step of stage s | first fragments of stage s+1 | first loads of stage s+NSTAGE
    next_lines();
    slot(last_of(c0_c), smem + b_next * A_STAGE, 0, loads_c, s + NSTAGE, b_cur, q0{});
  };
  auto stage = [&](int s, auto c0_c, auto loads_c) {
    const int b_cur = b_prev == NSTAGE - 1 ? 0 : b_prev + 1;
    const int b_next = b_cur == NSTAGE - 1 ? 0 : b_cur + 1;
    stage_in(s, c0_c, loads_c, b_prev, b_cur, b_next);
    b_prev = b_cur;
  };
  int s = 1;
  // Long K: a turn of the loop is NSTAGE steps, whose buffers are then constants -- LDS addresses become offsets of the reads, and what is
  // left beside products, reads and loads is the load's m0 (27 instructions a step instead of 56 with 64 x 64 tiles, 62 instead of 92 with
  // 128 x 128).  us, step by step -> so: 128 x 128, 2048 x 2048 x 8192 34.6 -> 33.7, FP8 31.0 -> 29.9, 2048 x 1536 x 6912 27.0 -> 26.0, x 8192 29.5 -> 28.0;
  // 64 x 64, 512 x 2048 x 6912 13.3 -> 13.2, FP8 13.2 -> 12.9; 64 x 32, 200 x 2048 x 6912 11.1 -> 10.6, FP8 11.3 -> 10.3.  Shorter K: level in the mean,
  // between 1000 x 4096 x 2048 13.8 -> 14.8 and 2048 x 1536 x 4096 17.3 -> 16.7; two wavefronts per SIMD (256 x 128): 4096 x 3071 x 6912 104 -> 106.
  if constexpr (EXACT && NKS % 2 == 0 && NWAVES <= 4 && !BIG) {
    if (nk >= 48) {  // uniform
      for (; s + 2 * NSTAGE <= nk; s += NSTAGE) {
#pragma unroll
        for (int u = 0; u < NSTAGE; ++u) stage_in(s + u, k0{}, whole{}, u, (u + 1) % NSTAGE, (u + 2) % NSTAGE);
      }
    }
  }
  if constexpr (NKS % 2 == 0) {
    if constexpr (LINES)
      for (const int end = K / BK - 1 - NSTAGE; s < end; ++s) stage(s, k0{}, whole{});  // line s + NSTAGE + 1 ends before K
    for (; s < nk; ++s) stage(s, k0{}, yes{});
  } else {  // one sub-step per stage: the fragment buffers alternate per stage
    auto pairs = [&](int end, auto loads_c) {
      for (; s + 1 < end; s += 2) {
        stage(s, k1{}, loads_c);
        stage(s + 1, k0{}, loads_c);
      }
    };
    if constexpr (LINES) pairs(K / BK - 1 - NSTAGE, whole{});
    pairs(nk, yes{});
    if (s < nk) stage(s, k1{}, yes{});
  }
  AQ_WAIT_VMCNT(0);  // drain the padding loads before the workgroup's LDS can be released or reused
#ifdef AQ_LAB_STALL
  const long long tl_loop_end = clock64();
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    aq_lab_clock[2] = st_sum + (st_t1 - st_t0);
    aq_lab_clock[3] = tl_loop_end - st_begin;
    aq_lab_clock[4] = tl_stage0 - tl_start;   // tile start -> first stage landed and visible
    aq_lab_clock[5] = st_begin - tl_stage0;   // first K step without loads
  }
#endif

  if constexpr (WK == 2) {
    // The two wavefronts of a sub-tile hold the sums over their halves of every K step.  Each
    // keeps half of the row blocks (the first wavefront the upper ones) and parks the other half
    // in LDS for its partner (over the stage buffers, which nobody reads any more once every
    // wavefront is past the barrier); then both add what the partner left for them and run the
    // epilogue on their half.  int32 sums are exact in any order; FP8 partial sums are fp32,
    // inside the stated tolerance.
    __syncthreads();
    using part_t = std::conditional_t<FP8, v4f, v4i>;
    constexpr int SLOT = TME * TN * 4 * 64;  // part_t elements one wavefront parks
    part_t* mine = reinterpret_cast<part_t*>(smem) + (wave_mn * 2 + wave_k) * SLOT + lane;
    part_t* theirs = reinterpret_cast<part_t*>(smem) + (wave_mn * 2 + (wave_k ^ 1)) * SLOT + lane;
    static_assert(NWAVES * SLOT * 16 <= NSTAGE * STAGE, "the parked accumulators fit the stage buffers");
    if (wave_k == 0) {  // uniform
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            mine[((i * TN + j) * 4 + g) * 64] = part_t{acc[TME + i][j][g * 4], acc[TME + i][j][g * 4 + 1],
                                                       acc[TME + i][j][g * 4 + 2], acc[TME + i][j][g * 4 + 3]};
    } else {
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
          for (int g = 0; g < 4; ++g)
            mine[((i * TN + j) * 4 + g) * 64] =
                part_t{acc[i][j][g * 4], acc[i][j][g * 4 + 1], acc[i][j][g * 4 + 2], acc[i][j][g * 4 + 3]};
          acc[i][j] = acc[TME + i][j];  // the lower row blocks move to the front: the epilogue indexes from 0
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TME; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const part_t t = theirs[((i * TN + j) * 4 + g) * 64];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[i][j][g * 4 + q] += t[q];
        }
  }

  // ---- epilogue, straight from the accumulator registers (no LDS, no barrier).
  // A lane owns one output column per 32x32 tile and 64 of the wavefront's 128
  // rows.  Stores go through a buffer descriptor based at the wavefront's first
  // output: the lane part of the address (its column, its half of the 8-row
  // group) is one VGPR computed once, the row part is a scalar offset, so no
  // vector ALU work is spent on addresses.  Lanes whose column is past N carry
  // an out-of-range offset and their stores are dropped by the hardware.
  // bf16 outputs are paired across neighbouring lanes: each lane converts its
  // two rows (2h, 2h+1) into one packed dword, swaps it with its neighbour
  // (DPP quad_perm [1,0,3,2]) and byte-permutes the two into "my row, both
  // columns": even lanes write row 2h, odd lanes row 2h+1, 4 bytes per lane,
  // 64 contiguous bytes per row segment.
  constexpr int ESZ = (OUT == OUT_BF16) ? 2 : 4;
  const int nw = __builtin_amdgcn_readfirstlane(n0 + wave_n * WAVE_N);  // first column of this wavefront
  const __amdgpu_buffer_rsrc_t Cr =
      make_rsrc(reinterpret_cast<uint8_t*>(p.C) + ((int64_t)mw * N + nw) * ESZ, 0x40000000u);
  // Residual: the same window over the tensor that is added to the rounded output; each lane
  // reads exactly the elements it then writes, so the residual may be the output itself.
  const bool has_res = !BIG && OUT != OUT_I32 && p.res != nullptr;  // uniform (big sub-tiles are not launched with a residual)
  const __amdgpu_buffer_rsrc_t Rr = make_rsrc(
      reinterpret_cast<const uint8_t*>(has_res ? p.res : p.C) + ((int64_t)mw * N + nw) * ESZ, has_res ? 0x40000000u : 0u);
  const bool odd = lane & 1;
  const uint32_t perm_sel = odd ? 0x03020706u : 0x05040100u;
  const uint32_t rowb = (uint32_t)N * ESZ;
  const bool rows_inside = mw + 32 * TME <= M;  // uniform
  // CHECK_M: some rows of this wavefront are past M.  PAIR: the bf16 dword path.
  auto store_all = [&](auto check_c, auto pair_c) {
    constexpr bool CHECK_M = decltype(check_c)::value;
    constexpr bool PAIR = (OUT == OUT_BF16) && decltype(pair_c)::value;
    // lane part of the byte offset of column j; the pairing path stores at the even column of the pair
    auto lane_offset = [&](int j) -> uint32_t {
      const int cj = j * 32 + col;  // column inside the wavefront's 64
      return nw + cj < N ? (uint32_t)rq * rowb + (uint32_t)(PAIR ? (cj & ~1) : cj) * ESZ + (PAIR && odd ? rowb : 0u)
                         : OOB_OFFSET;
    };
    // The residual elements a lane will add, requested ahead of the arithmetic: all columns at once on
    // the paired bf16 path (32 registers; the stores of one column would otherwise sit between the
    // loads of the next and their use), column by column on the others.
    constexpr int RLD = PAIR ? 2 : 4;  // loads per 4-row group: packed row pairs, or single elements
    constexpr bool HOIST = PAIR && TN * TME <= 4;
    uint32_t rr[HOIST ? TN : 1][TME][4][RLD];
    auto load_residual = [&](int j) {
      const uint32_t vbase = lane_offset(j);
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int q = 0; q < RLD; ++q) {
            const int r0 = i * 32 + g * 8;
            const int rowq = PAIR ? 2 * q : q;
            uint32_t vo = vbase;
            if (CHECK_M && mw + r0 + rq + rowq + (PAIR && odd ? 1 : 0) >= M) vo = OOB_OFFSET;
            if constexpr (OUT == OUT_F32 || PAIR)
              rr[HOIST ? j : 0][i][g][q] = __builtin_amdgcn_raw_buffer_load_b32(Rr, vo, (r0 + rowq) * rowb, 0);
            else
              rr[HOIST ? j : 0][i][g][q] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(Rr, vo, (r0 + rowq) * rowb, 0);
          }
    };
    if constexpr (OUT != OUT_I32 && HOIST) {
      if (has_res) {
#pragma unroll
        for (int j = 0; j < TN; ++j) load_residual(j);
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float bn = 0.0f;
      if constexpr (OUT != OUT_I32)
        bn = !has_bias ? 0.0f : bias_bf16 ? bf16_bits_to_f32(bias_raw[j]) : __uint_as_float(bias_raw[j]);
      const uint32_t vbase = lane_offset(j);
      if constexpr (OUT != OUT_I32 && !HOIST) {
        if (has_res) load_residual(j);
      }
#pragma unroll
      for (int i = 0; i < TME; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int r0 = i * 32 + g * 8;  // + rq + q : row inside the wavefront's 128
          if constexpr (OUT == OUT_I32) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              uint32_t vo = vbase;
              if (CHECK_M && mw + r0 + rq + q >= M) vo = OOB_OFFSET;
              __builtin_amdgcn_raw_buffer_store_b32((uint32_t)acc[i][j][g * 4 + q], Cr, vo, (r0 + q) * rowb, STORE_WT);
            }
          } else {
            float y[4];
            v4f sxq = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (BIG && !FP8)
              sxq = *reinterpret_cast<const v4f*>(sx_lds + (mw - m0) + r0 + rq);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if constexpr (FP8) {
                // without a bias bn is +0: it changes no bit unless the product is -0, whose sign a bf16 or
                // fp32 consumer of a Linear output never sees as a different value
                y[q] = __fadd_rn(__fmul_rn(__fmul_rn(acc[i][j][g * 4 + q], sx1), sw1), bn);
              } else {
                // three separately rounded fp32 operations, never contracted.  Without a bias
                // bn is +0: the product of an integer and two positive scales is never -0,
                // so adding it changes no bit.
                y[q] = __fadd_rn(__fmul_rn(__fmul_rn((float)acc[i][j][g * 4 + q], BIG ? sxq[q] : sxr[BIG ? 0 : i][g][q]), swn[j]), bn);
              }
            }
            if constexpr (OUT == OUT_F32) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                uint32_t vo = vbase;
                if (CHECK_M && mw + r0 + rq + q >= M) vo = OOB_OFFSET;
                if (has_res) y[q] = __fadd_rn(y[q], __uint_as_float(rr[HOIST ? j : 0][i][g][q]));
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[q]), Cr, vo, (r0 + q) * rowb, STORE_WT);
              }
            } else if constexpr (PAIR) {
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const uint32_t mine = pack_bf16x2(y[2 * h], y[2 * h + 1]);  // lo: row 2h, hi: row 2h+1
                const uint32_t other =
                    (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xB1 /* quad_perm [1,0,3,2] */, 0xf, 0xf, true);
                // even lane: {mine.lo, other.lo} = row 2h, columns (c, c+1)
                // odd lane:  {other.hi, mine.hi} = row 2h+1, columns (c-1, c)
                uint32_t pk = __builtin_amdgcn_perm(other, mine, perm_sel);
                if (has_res) {  // rounded output + residual, rounded again: what a separate add gives
                  const uint32_t r = rr[HOIST ? j : 0][i][g][h];
                  pk = pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(r << 16)),
                                   __fadd_rn(__uint_as_float(pk & 0xffff0000u), __uint_as_float(r & 0xffff0000u)));
                }
                uint32_t vo = vbase;
                if (CHECK_M && mw + r0 + rq + 2 * h + (odd ? 1 : 0) >= M) vo = OOB_OFFSET;
                __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, vo, (r0 + 2 * h) * rowb, STORE_WT);
              }
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                uint32_t vo = vbase;
                if (CHECK_M && mw + r0 + rq + q >= M) vo = OOB_OFFSET;
                uint32_t ob = f32_to_bf16_bits(y[q]);
                if (has_res) ob = f32_to_bf16_bits(__fadd_rn(__uint_as_float(ob << 16), __uint_as_float(rr[HOIST ? j : 0][i][g][q] << 16)));
                __builtin_amdgcn_raw_buffer_store_b16((uint16_t)ob, Cr, vo, (r0 + q) * rowb, STORE_WT);
              }
            }
          }
        }
      }
    }
  };
  // Neighbouring columns in a lane: a dword of output per row, 32 lanes a line.  us, half a line by pairs of lanes -> so:
  // 2048 x 1536 x 1536 + residual 10.8 -> 10.4, 512 x 8192 x 1024 8.3 -> 7.8, 500 x 10992 x 1024 10.4 -> 9.1, 2000 x 5040 x 256
  // 13.1 -> 11.9 (on other cards the halves cost up to half of such a launch, see gemm_walk.hip).
  auto store_lines = [&](auto check_c) {
    constexpr bool CHECK_M = decltype(check_c)::value;
    const uint32_t at0 = nw + 2 * col < N ? (uint32_t)rq * rowb + (uint32_t)(2 * col) * ESZ : OOB_OFFSET;
    auto at = [&](int r) { return CHECK_M && mw + r + rq >= M ? OOB_OFFSET : at0; };
    uint32_t rr[TME][16];  // all of the residual, requested before any of it is used
    if (has_res) {
#pragma unroll
      for (int i = 0; i < TME; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = i * 32 + e / 4 * 8 + e % 4;
          rr[i][e] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, at(r), r * rowb, 0);
        }
    }
    float bn[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bn[j] = !has_bias ? 0.0f : bias_bf16 ? bf16_bits_to_f32(bias_raw[j]) : __uint_as_float(bias_raw[j]);
#pragma unroll
    for (int i = 0; i < TME; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int r = i * 32 + e / 4 * 8 + e % 4;
        float y[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if constexpr (FP8)
            y[j] = __fadd_rn(__fmul_rn(__fmul_rn(acc[i][j][e], sx1), sw1), bn[j]);
          else
            y[j] = __fadd_rn(__fmul_rn(__fmul_rn((float)acc[i][j][e], sxr[i][e / 4][e % 4]), swn[j]), bn[j]);
        }
        uint32_t pk = pack_bf16x2(y[0], y[1]);
        if (has_res)  // rounded output + residual, rounded again: what a separate add gives
          pk = pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(rr[i][e] << 16)),
                           __fadd_rn(__uint_as_float(pk & 0xffff0000u), __uint_as_float(rr[i][e] & 0xffff0000u)));
        __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, at(r), r * rowb, STORE_WT);
      }
  };
  if constexpr (ADJ) {
    if (pair_ok && rows_inside)
      store_lines(no{});
    else if (pair_ok)
      store_lines(yes{});
    else
      store_all(yes{}, no{});
  } else if constexpr (BIG) {
    store_all(no{}, yes{});  // one variant (256 outputs per lane): the launcher sends ragged M and odd N to another shape
  } else {
    if (rows_inside && pair_ok)
      store_all(no{}, yes{});   // interior tiles: straight-line, no per-row checks
    else if (pair_ok)
      store_all(yes{}, yes{});
    else
      store_all(yes{}, no{});
  }
#ifdef AQ_LAB_STALL
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    aq_lab_clock[6] = clock64() - tl_loop_end;  // accumulator exchange (split K steps) + epilogue issue
    aq_lab_clock[7] = clock64() - tl_start;     // the whole tile as wavefront 0 sees it
  }
#endif
}

// A workgroup walks tiles pid, pid + gridDim.x, ...: with more tiles than compute units the launch is one
// resident workgroup per compute unit instead of a queue of short-lived ones (the LDS stages allow one at a time).
template <bool FP8, int OUT, class S, Rows ROWS>
__global__ __launch_bounds__(S::NTHREADS) void gemm_kernel(GemmArgs p) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[ROWS == LINE_ROWS ? S::LDS_LINES : S::LDS_BYTES];
  const int nt = p.tiles_m * p.tiles_n;
#ifdef AQ_LAB
  struct Clk {
    long long c0, w0;
    __device__ Clk() : c0(clock64()), w0(wall_clock64()) {}
    __device__ ~Clk() {
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        aq_lab_clock[0] = clock64() - c0;
        aq_lab_clock[1] = wall_clock64() - w0;
      }
    }
  } clk;
#endif
  for (int pid = blockIdx.x; pid < nt; pid += gridDim.x) {
    gemm_tile<FP8, OUT, S, ROWS>(p, smem, pid);
    if (pid + (int)gridDim.x < nt) __syncthreads();  // every wavefront is done with the stages before they are refilled
  }
}

// Tile shape by the number of rounds over the compute units a launch needs: a workgroup per compute unit at a
// time, so the cost of a launch is its number of rounds times the cost of a round of that shape (us at K = 2048
// with the weights streamed from HBM, on top of 4 us of launch and pipeline fill; every term scales with K alike):
//   256 x 128: 15.0   128 x 128: 10.8   128 x 64: 7.0   128 x 32: 5.0   64 x 64: 4.6   64 x 32: 3.5
// After a full round, a last round of the two wide shapes that fills only part of the device costs about half a
// round plus half its fill (384 large tiles, 1.5 rounds, take 1.74 times as long as 256); a first round runs at the
// latency of its K loop whatever the fill (128 x 128: 64 tiles 12.3-14.8 us, 256 tiles 14.5 us), and so does every
// round of the small shapes (64 x 32: 64 tiles 6.9 us, 256 tiles 7.0 us, 352 tiles 12.0 us), whose rounds count
// whole.  Fitted on
// 33..2048 rows against N = 1024..16384 and K = 1024..5632, where the rule picks the fastest shape or one within
// 6 % of it.  The small tiles are for launches of a few rounds only.
enum TileKind {
  TILE_AUTO = 0, TILE_STREAMS = 31 /* no tile: gemv.hip's */, TILE_N32 = 32, TILE_M64N32 = 33, TILE_N64 = 64, TILE_M64N64 = 65, TILE_SMALL = 128,
  TILE_PAIR = 129, TILE_WIDE = 192,
  TILE_LARGE = 256, TILE_TALL = 257, TILE_HUGE = 512, TILE_HUGE8 = 513, TILE_WALK = 258  // and SlicesTile's
};
#ifdef AQ_LAB
static int g_forced_tile = 0;  // lab build only: TILE_AUTO = by shape, otherwise forced (tuning and tests)
#endif

// Where gemm_walk_kernel can take the call, its tiles stand for the 256 x 128 one: that at the same cost of a round but less of a
// last one (0.7 + 0.1 of its fill; 0.55 where its tiles are cut in two), and 256 x 192 at 1.45 of a round (last 0.7 + 0.2): with
// five fragments read and 56 KiB brought in for three columns of products, where 256 x 128 has four and 48 for two, it is the
// faster one, by up to a third, where it saves a round or most of one.  Measured over 470 random sizes of 300..8192 rows, N
// 512..11264, K 512..8192, int8 and FP8, on several cards: what this picks is 0.2 % from the faster of the two in the mean, 7 % at
// most but for one size in a hundred (256 x 128 alone: 5 %, 43 %).  us, gemm_kernel's tiles -> 256 x 192 (256 x 128 of the walk):
// 4096 x 3072 x 2048 31.5 -> 25.2 (30.2), FP8 27.6 -> 22.8 (27.5), 1476 x 6480 x 4448 72.5 -> 49.2 (69), 6263 x 1456 x 3696 63 -> 42.8
// (59), 6952 x 1232 x 992 with a residual 30.2 -> 17.7 (26), FP8 2954 x 11104 x 4000 172 -> 142 (172); not 4096 x 11264 x 2048 (95, 109).
// With a residual, 256 x 192 takes 1.6 of a round: both types hold 48 bytes of it per lane beside 96 accumulators, and ask for a third
// (int8) or all of it (FP8) only when the products are done.  At 1.45, of 600 random sizes with a residual it was 6 % slower than the
// faster of the two for one in twenty, up to 19 %; now 0.25 % in the mean, 3 % for one in twenty (us, 256 x 192 | 256 x 128: FP8 3668 x 4864 x 512
// 24.8 | 21.2, int8 4780 x 9200 x 3840 192 | 169, FP8 6678 x 10632 x 6032 472 | 509).
static int choose_tile_for(int64_t M, int64_t N, int64_t cus, bool walk = false, bool res = false) {
  auto rounds = [cus](int64_t tiles, double last, double fill) {
    const int64_t full = tiles / cus, rest = tiles % cus;
    if (full == 0) return 1.0;
    return (double)full + (rest ? last + fill * (double)rest / cus : 0.0);
  };
  struct Cand {
    int kind, bm, bn;
    double round_us;
    bool small;
    double last, fill;  // of a round, for a last one behind others
  };
  const Cand cands[] = {{TILE_LARGE, 256, 128, 15.0, false, 0.5, 0.5}, {TILE_SMALL, 128, 128, 10.8, false, 0.5, 0.5},
                        {TILE_N64, 128, 64, 7.0, true, 0, 0},          {TILE_N32, 128, 32, 5.0, true, 0, 0},
                        {TILE_M64N64, 64, 64, 4.6, true, 0, 0},        {TILE_M64N32, 64, 32, 3.5, true, 0, 0},
                        {TILE_WIDE, 256, 192, res ? 24.0 : 21.75, false, 0.7, 0.2}};
  int best = TILE_LARGE;
  double cost = 0.0;
  for (const Cand& c : cands) {
    if (c.kind == TILE_WIDE && !walk) continue;
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
    if (c.small && tiles > 4 * cus) continue;
    double last = c.last, fill = c.fill;
    if (c.kind == TILE_LARGE && walk) {
      const bool halves = gemm_walk_halves(tiles, cus);
      last = halves ? 0.55 : 0.7, fill = halves ? 0.0 : 0.1;
    }
    const double us = c.round_us * (c.small ? (double)((tiles + cus - 1) / cus) : rounds(tiles, last, fill));
    if (c.kind == TILE_LARGE || us < cost) {
      cost = us;
      best = c.kind;
    }
  }
  return best;
}

template <bool FP8, int OUT, class S>
static int launch_shape(GemmArgs& a, hipStream_t st) {
  a.tiles_m = (a.M + S::BM - 1) / S::BM;
  a.tiles_n = (a.N + S::BN - 1) / S::BN;
  // one resident workgroup per compute unit walks the tiles (a workgroup's LDS stages fill a compute unit):
  // 3-5 % faster than queueing a workgroup per tile once there are more tiles than compute units
  const int64_t ntiles = (int64_t)a.tiles_m * a.tiles_n, cus = device_cus();
  const unsigned grid = (unsigned)(ntiles < cus ? ntiles : cus);
  if constexpr (!S::BIG) {  // (big sub-tiles are launched for whole K steps only)
    if (a.K % S::BK != 0 || a.lda != a.K) {
      // Lines from 11 of them on: the extra line and the longer prologue cost 0.2..0.3 us.  us, ANY -> LINES at K 1008, 1520, 3056, 4592 (rows of A on
      // lines): 64 x 64 tiles, 333 x 1536 5.08 -> 5.47, 6.17 -> 6.15, 8.81 -> 8.25, 11.01 -> 10.14; 128 x 64, 798 x 1648 7.26 -> 7.27, 8.61 -> 8.45, 12.2 ->
      // 11.5, 15.9 -> 14.7; 128 x 128, 2048 x 1536 8.89 -> 8.73, 10.9 -> 10.7, 16.8 -> 15.6, 22.7 -> 21.0, FP8 8.34 -> 8.17, 10.3 -> 9.8, 15.9 -> 14.2, 21.4 ->
      // 18.5.  Not with 32 outputs in a tile, where a wavefront's select serves one product: 64 x 32 tiles 6.57 -> 7.02 at K 2032, 10.3 -> 10.6 at 4592.
      if constexpr (S::BN > 32) {
        if (a.K >= 11 * S::BK) {
          aq::queue_kernel((gemm_kernel<FP8, OUT, S, LINE_ROWS>), dim3(grid), dim3(S::NTHREADS), 0, st, a);
          return (int)hipGetLastError();
        }
      }
      aq::queue_kernel((gemm_kernel<FP8, OUT, S, ANY_ROWS>), dim3(grid), dim3(S::NTHREADS), 0, st, a);
      return (int)hipGetLastError();
    }
  }
  aq::queue_kernel((gemm_kernel<FP8, OUT, S, EXACT_ROWS>), dim3(grid), dim3(S::NTHREADS), 0, st, a);
  return (int)hipGetLastError();
}

// FP8 launches the 256 x 256 tile serves and gains on: whole 256-row multiples, even N, no residual (the tile's one K-loop and
// epilogue variant), and, against the walked tiles at 3491 random sizes:
// * K of an odd number of 64-byte steps: rows then begin in the middle of a line, which 128-byte steps bring in as two halves of
//   lines and 64-byte steps do not.  K of whole lines never gains: 256 x 256 / the walked tiles, K 2049..2560 1.18, up to 4096 1.10, up
//   to 8192 1.06, up to 16384 1.02 (us 5376 x 7278 x 2816 121 | 93, 4096 x 10688 x 3584 140 | 127, 8192^3 432 | 429, 4096 x 8192 x 4096 112 | 110).
// * K above 3072: its loop stops between tiles, gemm_walk_kernel's does not: K 1024..2048 1.10, up to 2560 1.00, up to 3072 0.99,
//   up to 4096 0.96, up to 5120 0.94, up to 8192 0.90 (us 4864 x 8640 x 3264 126 | 131, 7424 x 6440 x 5312 212 | 244, 7424 x 5760 x 8000 294 | 327).
//   K below 512, which is not walked: 1.25 of gemm_kernel's other tiles with bf16 outputs, 1.04 with fp32 ones (120 sizes).
// * two rounds at least, and the last one more than half full: with less 1.04 to 1.14 at any K.
// In all 6 % faster than the walk where it is taken, and the choice 2 % from the best tile in the mean (taken for any K above 2048
// and any last round, 11 %).
static bool huge_fp8_ok(const GemmArgs& a, int64_t cus) {
  if (a.lda != a.K || a.K <= 3072 || a.K % (2 * ShapeHuge::BK) != ShapeHuge::BK || (a.N % 2) != 0 || (a.M % ShapeHuge::BM) != 0 || a.res != nullptr) return false;
  const int64_t tiles = (int64_t)(a.M / ShapeHuge::BM) * ((a.N + ShapeHuge::BN - 1) / ShapeHuge::BN);
  return tiles >= 2 * cus && (tiles % cus == 0 || 2 * (tiles % cus) > cus);
}

// The tile that takes a call on a device of `cus` compute units.  TILE_WALK and TILE_WIDE: of gemm_walk_kernel, a SlicesTile: of
// gemm_slices_kernel.
static int choose_tile(const GemmArgs& a, bool fp8, int out, int64_t cus) {
  if (fp8 && out != OUT_I32 && huge_fp8_ok(a, cus)) return TILE_HUGE;
  const bool walk = out != OUT_I32 && gemm_walk_ok(a, out);
  const int tile = choose_tile_for(a.M, a.N, cus, walk, a.res != nullptr);
  if (walk && tile == TILE_LARGE) return TILE_WALK;
  if (tile == TILE_WIDE || out == OUT_I32) return tile;
  const int slices = gemm_slices_tile(a.M, a.N, a.K, cus);
  return slices ? slices : tile;
}

template <bool FP8, int OUT>
static int launch(GemmArgs& a, hipStream_t st) {
  int tile = choose_tile(a, FP8, OUT, device_cus());
#ifdef AQ_LAB
  if (g_forced_tile) {
    tile = g_forced_tile;
    if ((tile == TILE_WALK || tile == TILE_WIDE) && (OUT == OUT_I32 || !gemm_walk_ok(a, OUT))) tile = TILE_LARGE;
    if (tile == TILE_HUGE && (a.K % ShapeHuge::BK != 0 || a.N % 2 != 0 || a.M % ShapeHuge::BM != 0 || a.res != nullptr)) tile = TILE_LARGE;
  }
#endif
  if constexpr (OUT != OUT_I32) {
    switch (tile) {
      case TILE_WALK: return gemm_walk_launch<FP8, OUT>(a, st, 128);
      case TILE_WIDE: return gemm_walk_launch<FP8, OUT>(a, st, 192);
    }
    if (tile >= SLICES_FIRST && tile <= SLICES_LAST) return gemm_slices_launch<FP8, OUT>(a, tile, st);
    if constexpr (FP8)
      if (tile == TILE_HUGE) return launch_shape<FP8, OUT, ShapeHuge>(a, st);
  }
  switch (tile) {
    case TILE_SMALL: return launch_shape<FP8, OUT, ShapeSmall>(a, st);
    case TILE_N64: return launch_shape<FP8, OUT, ShapeN64>(a, st);
    case TILE_N32: return launch_shape<FP8, OUT, ShapeN32>(a, st);
    case TILE_M64N64: return launch_shape<FP8, OUT, ShapeM64N64>(a, st);
    case TILE_M64N32: return launch_shape<FP8, OUT, ShapeM64N32>(a, st);
#ifdef AQ_LAB
    case TILE_TALL: return launch_shape<FP8, OUT, ShapeTall>(a, st);
    case TILE_HUGE: return launch_shape<FP8, OUT, ShapeHuge>(a, st);
    case TILE_HUGE8: return launch_shape<FP8, OUT, ShapeHuge8>(a, st);
    case TILE_PAIR: return launch_shape<FP8, OUT, ShapePair>(a, st);
#endif
    default: return launch_shape<FP8, OUT, ShapeLarge>(a, st);
  }
}

static int check_gemm(const void* A, const void* B, const void* C, int64_t M, int64_t N, int64_t K) {
  if (M < 0 || N < 0 || K <= 0 || (K % 16) != 0) return AQ_E_SHAPE;
  if (M == 0 || N == 0) return AQ_OK;
  if (!A || !B || !C) return AQ_E_NULL;
  if (check_ptr16(A) || check_ptr16(B) || check_ptr16(C)) return AQ_E_ALIGN;
  // 32-bit tile-relative offsets: 256 rows * K bytes of an operand and 256 rows * N * 4 bytes of the
  // output window of a workgroup must fit 31 bits
  if (K > (1 << 22) || M > (1 << 30) || N > (1 << 20)) return AQ_E_RANGE;
  if (((M + 127) / 128) * ((N + 127) / 128) > (int64_t)0x7fffffff) return AQ_E_RANGE;
  return AQ_OK;
}

// 17..32 rows, in whole lines, of more outputs than tiles cut among wavefronts serve: the weight-streaming kernel takes them.  Not 16 rows
// and fewer, however long: us, weights in the last-level cache | from HBM, the weight-streaming kernel -> tiles of 16 x 64 or 16 x 32: 16 x
// 11008 -> 8200 29.5 -> 20.6 | 29.2 -> 26.5, -> 12288 35.0 -> 26.6 | 34.8 -> 35.6, -> 20000 62.8 -> 36.8 | 63.3 -> 49.5, -> 32000 73.4 -> 65.9 |
// 74.7 -> 67.8; 8 x 20480 -> 8200 50.6 -> 29.1 | 49.7 -> 42.6; of 119 sizes the slowest 16 x 14336 -> 32000 74.3 -> 79.6 and, from HBM, 9 x
// 16384 -> 16384 49.7 -> 53.7.
static bool streams_weights(int64_t M, int64_t N, int64_t K, int64_t cus) {
  return M > 16 && M <= 32 && K % 128 == 0 && !gemm_slices_tile(M, N, K, cus);
}

static GemmArgs make_args(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K) {
  GemmArgs a{};
  a.A = static_cast<const uint8_t*>(A);
  a.B = static_cast<const uint8_t*>(B);
  a.C = C;
  a.M = (int)M;
  a.N = (int)N;
  a.K = a.lda = (int)K;
  return a;
}

}  // namespace aq

#ifdef AQ_LAB
extern "C" int aq_lab_read_clock(long long* host2) {
  return (int)hipMemcpyFromSymbol(host2, HIP_SYMBOL(aq::aq_lab_clock), 64);
}
extern "C" int aq_lab_set_gemm_tile(int rows) {
  if (rows != 192 && rows != 258 && (rows < aq::SLICES_FIRST || rows > aq::SLICES_LAST) && rows != 0 && rows != 129 && rows != 33 && rows != 65 && rows != 64 && rows != 32 && rows != 128 && rows != 256 && rows != 257 && rows != 512 && rows != 513) return AQ_E_SHAPE;
  aq::g_forced_tile = rows;
  return AQ_OK;
}
extern "C" int aq_lab_choose_gemm_tile(int64_t M, int64_t N, int64_t K, int fp8, int y_dtype, int residual, int compute_units) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 16 || M > (1 << 30) || N > (1 << 20) || K > (1 << 22) || compute_units <= 0) return AQ_E_SHAPE;
  if ((fp8 && y_dtype < 0) || (y_dtype >= 0 && y_dtype != AQ_F32 && y_dtype != AQ_BF16) || (y_dtype < 0 && residual)) return AQ_E_DTYPE;
  if (y_dtype >= 0 && aq::streams_weights(M, N, K, compute_units)) return aq::TILE_STREAMS;
  static const char some = 0;
  aq::GemmArgs a = aq::make_args(nullptr, nullptr, nullptr, M, N, K);
  a.res = residual ? &some : nullptr;  // only whether there is one
  return aq::choose_tile(a, fp8 != 0, y_dtype < 0 ? aq::OUT_I32 : y_dtype == AQ_BF16 ? aq::OUT_BF16 : aq::OUT_F32, compute_units);
}
#endif

extern "C" int aq_gemm_i8_i32(const int8_t* xq, const int8_t* wq, int32_t* acc, int64_t M, int64_t N,
                              int64_t K, void* stream) {
  int rc = aq::check_gemm(xq, wq, acc, M, N, K);
  if (rc || M == 0 || N == 0) return rc;
  aq::GemmArgs a = aq::make_args(xq, wq, acc, M, N, K);
  return aq::launch<false, aq::OUT_I32>(a, static_cast<hipStream_t>(stream));
}

extern "C" int aq_linear_w8a8(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                              const void* bias, int bias_dtype, void* y, int y_dtype, int64_t M,
                              int64_t N, int64_t K, void* stream) {
  return aq_linear_w8a8_residual(xq, sx, wq, sw, bias, bias_dtype, nullptr, y, y_dtype, M, N, K, stream);
}

namespace aq {
// gemv.hip: the weight-streaming kernel for 17..32 rows (same sums, same epilogue: same bits)
int gemv_tokens_launch(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw, const void* bias,
                       int bias_dtype, const void* residual, void* y, int y_dtype, int64_t M, int64_t N, int64_t K,
                       hipStream_t st, bool fp8);

}  // namespace aq

namespace aq {
// y = codes [M, K], rows ldx bytes apart, times weights [N, K], scaled
static int linear_codes(bool fp8, const void* xq, int64_t ldx, const float* sx, const void* wq, const float* sw, const void* bias, int bias_dtype,
                        const void* residual, void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
  if (y_dtype != AQ_F32 && y_dtype != AQ_BF16) return AQ_E_DTYPE;
  if (bias && bias_dtype != AQ_F32 && bias_dtype != AQ_BF16) return AQ_E_DTYPE;
  int rc = check_gemm(xq, wq, y, M, N, K);
  if (!rc && (ldx < K || ldx % 16 || ldx > (1 << 22))) return ldx < K ? AQ_E_SHAPE : ldx % 16 ? AQ_E_ALIGN : AQ_E_RANGE;
  if (rc || M == 0 || N == 0) return rc;
  if (!sx || !sw) return AQ_E_NULL;
  if (check_ptr(sx, 4) || check_ptr(sw, 4) || check_ptr(bias, bias_dtype == AQ_BF16 ? 2 : 4) || check_ptr(residual, 4)) return AQ_E_ALIGN;
  hipStream_t st = static_cast<hipStream_t>(stream);
  bool streams = ldx == K && streams_weights(M, N, K, device_cus()) && check_ptr16(residual) == 0;
#ifdef AQ_LAB
  streams = streams && !g_forced_tile;
#endif
  if (streams)
    return gemv_tokens_launch(static_cast<const int8_t*>(xq), sx, static_cast<const int8_t*>(wq), sw, bias, bias_dtype, residual, y, y_dtype, M, N, K,
                              st, fp8);
  GemmArgs a = make_args(xq, wq, y, M, N, K);
  a.lda = (int)ldx;
  a.sx = sx;
  a.sw = sw;
  a.bias = bias;
  a.bias_dtype = bias_dtype;
  a.res = residual;
  if (fp8) return y_dtype == AQ_BF16 ? launch<true, OUT_BF16>(a, st) : launch<true, OUT_F32>(a, st);
  return y_dtype == AQ_BF16 ? launch<false, OUT_BF16>(a, st) : launch<false, OUT_F32>(a, st);
}
}  // namespace aq

extern "C" int aq_linear_w8a8_residual(const int8_t* xq, const float* sx, const int8_t* wq, const float* sw,
                                       const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                       int64_t M, int64_t N, int64_t K, void* stream) {
  return aq::linear_codes(false, xq, K, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_linear_fp8(const uint8_t* xq, const float* sx, const uint8_t* wq, const float* sw,
                             void* y, int y_dtype, int64_t M, int64_t N, int64_t K, void* stream) {
  return aq_linear_fp8_residual(xq, sx, wq, sw, nullptr, AQ_F32, nullptr, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_linear_fp8_residual(const uint8_t* xq, const float* sx, const uint8_t* wq, const float* sw,
                                      const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                      int64_t M, int64_t N, int64_t K, void* stream) {
  return aq::linear_codes(true, xq, K, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_linear_w8a8_strided(const int8_t* xq, int64_t ldx, const float* sx, const int8_t* wq, const float* sw,
                                      const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                      int64_t M, int64_t N, int64_t K, void* stream) {
  return aq::linear_codes(false, xq, ldx, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

extern "C" int aq_linear_fp8_strided(const uint8_t* xq, int64_t ldx, const float* sx, const uint8_t* wq, const float* sw,
                                     const void* bias, int bias_dtype, const void* residual, void* y, int y_dtype,
                                     int64_t M, int64_t N, int64_t K, void* stream) {
  return aq::linear_codes(true, xq, ldx, sx, wq, sw, bias, bias_dtype, residual, y, y_dtype, M, N, K, stream);
}

// Rows of K bytes that are no whole number of 128-byte lines begin in the middle of one, all but every eighth, and each 128-byte step of such
// a row is two halves of lines: twice the requests, of which a compute unit has so many in flight.  The weights are the caller's; the codes
// of the activations are written here, to rows that begin on lines.  us, K apart -> whole lines (all rows on lines, weights too): 798 x 4704 -> 1648 19.4 -> 16.2
// (13.9), 333 x 6896 -> 1536 18.5 -> 14.9 (12.6), 2048 x 6896 -> 1536 35.3 -> 30.0 (25.0), 4096 x 2032 -> 11264 108 -> 92.5 (89.4), 7601 x 4272 -> 1096 47.7 ->
// 44.9 (40.5), FP8 4958 x 1264 -> 6288 51.2 -> 43.2, 952 x 3392 -> 1392 13.2 -> 11.8 (10.8); level with few rows (64 x 2032 -> 2048 4.2).  Not where the
// 256 x 256 FP8 tile serves, whose 64-byte steps halve no line (with a residual it does not: 4864 x 3264 -> 8640 148.7 -> 132.8, 8192 x 8128 -> 8192 583 -> 486),
// nor the weight-streaming kernel, which takes rows as they are.  Nor what the quantisers do not write in rows: more than 2^31 vectors of 16 bytes,
// of which fp32 rows have K / 4.  Nor where the gaps alone take the codes past the 31-bit offsets of the kernel that walks tiles.
// Nor short rows of that kernel: in some processes, on most cards, it reads codes that have just been written at a half to three quarters of its
// rate if they begin on lines, with no more requests, misses or bytes than in others.  us of quantiser and GEMM, K apart -> whole lines, where
// that happens | where it does not: 6181 x 720 -> 1096 18.8 -> 22.9 | 18.8 -> 17.9, 6020 x 880 -> 4400 47 -> 62 | 45 -> 40.5, 7182 x 1088 -> 4192
// 52 -> 74.  1018 sizes of it by K, in the mean (slowest): 512 to 1151 0.999 (1.40) | 0.955 (1.09), to 1663 0.961 (1.16) | 0.928, to 2047 0.957 (1.20) |
// 0.916, from 2048 on 0.901 (1.02) | 0.897.  The other tiles gain where it happens too (132 sizes, 0.947, slowest 1.01).
extern "C" int64_t aq_linear_codes_pitch(int fp8, int residual, int64_t M, int64_t N, int64_t K) {
  if (M <= 16 || N < 1 || K < 1 || K % 16 || K % 128 == 0 || K > (1 << 22) - 128 || M > (1 << 30) || M * K / 4 > (int64_t)0x7fffffff) return K;
  const int64_t pitch = (K + 127) / 128 * 128, reach = aq::OOB_OFFSET;
  if (aq::streams_weights(M, N, K, aq::device_cus()) || (M * pitch > reach && M * K <= reach)) return K;
  static const char some = 0;
  aq::GemmArgs a = aq::make_args(nullptr, nullptr, nullptr, M, N, K);
  a.res = residual ? &some : nullptr;  // only whether there is one
  const int tile = aq::choose_tile(a, fp8 != 0, aq::OUT_BF16, aq::device_cus());
  return tile == aq::TILE_HUGE || ((tile == aq::TILE_WALK || tile == aq::TILE_WIDE) && K < 2048) ? K : pitch;
}
