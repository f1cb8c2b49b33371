// The tiled GEMM of gemm_mfma.hip for tiles of 256 x 128 and 256 x 192: at most one resident workgroup per compute unit walks tiles,
// and its K loop does not stop between them.
//
// What bounds it: a tile of K = 1536 or 2048 is 12 to 16 K steps of 1024 matrix-core cycles (256 x 128), and the separate tiles of
// gemm_kernel put a drain of the stores, the latency of the first stages, a step without loads and the epilogue around
// them: 22 k cycles a tile for 13 k of K loop.  Here the last two steps of a tile already request the next tile's first
// two stages, so its first fragments are in registers when the epilogue ends, and the epilogue's stores drain under the
// next tile's first step.  (gemm_kernel also requests three stages past the last one for the sake of an even count, a
// quarter of all fills at K = 1536.)  Row scales wait in LDS and the output's end is the descriptors' (one epilogue, no row checks): an
// int8 tile takes 160 registers, with a residual 206, where gemm_kernel takes 227 (FP8 194 and 231, where it takes 164; 256 x 192
// tiles 192 to 256).  One round of tiles is faster too, 4096 x 2048 x 2048 19.1 us in gemm_kernel, 18.2 here, 1234 x 4576 x 2528 22.7 -> 21.2.
//
// 256 x 192: 4096 x 3072 is 16 x 24 tiles of 256 x 128, one and a half rounds in the time of two, and 16 x 16 of these.  Three stages of 56 KiB do not fit LDS: two, and a stage is requested whole as soon as its place is free.  (Half
// steps through five 28 KiB stages, four times the barriers: 10 to 15 % slower.  256 x 256 on the same two buffers: level with
// 256 x 128 at 4096 x 11264 x 2048, slower elsewhere; four wavefronts of 128 x 96: 30 % slower.)
//
// And the last round of 256 x 128: nt tiles on `cus` compute units take ceil(nt / cus) rounds, the last of them nearly empty in the
// worst case (864 tiles: 3.4 rounds in the time of 4).  When at most half the compute units would have a tile in it, its
// tiles are cut in two, 128 x 128 each -- behind three rounds or more: the halves run code that no instruction cache
// holds yet, which costs what they save after a single round (384 tiles of K = 2048: 38.5 us against 32.7 with whole ones).
//
// Measured in one process, gemm_kernel's 256 x 128 tile -> the walk's, us: int8 2048 x 13824 x 1536 53 -> 45.6 on one device, 65 -> 48
// on another; 4096 x 11264 x 2048 105 -> 97; 8192 x 8192 x 2048 138 -> 129, 144 -> 134; FP8 8192 x 4096 x 2048 63.8 -> 60.8.  The
// rest is the K loop at the clock the power limit leaves.  (A ninth wavefront that touches the lines six steps ahead took 38 us
// for 4096 x 4096 x 2048 where memory was slow, 2 to 10 % more elsewhere: not kept.)
//
// Int8: whole-number sums, one epilogue for all tiles: the bits of gemm_kernel.  FP8: the same order of sums.
#include "aq_gemm.h"

namespace aq {

typedef int v2i_t __attribute__((ext_vector_type(2)));

struct WalkArgs {
  GemmArgs g;
  int full;    // tiles that are walked whole; the ones behind them are cut in two
  int halves;  // 128 x 128 tiles
};

// Tile `idx` of `count`: workgroup ids are dealt round-robin to the XCDs; a contiguous run of ids per XCD, as tile_of_block
__device__ __forceinline__ int xcd_run(int pid, int count) {
  const int per = count / NUM_XCD, rem = count % NUM_XCD, xcd = pid % NUM_XCD, idx = pid / NUM_XCD;
  return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// A walk over tiles of 128 TM x 64 TN on 4 x 2 wavefronts of (32 TM) x (32 TN).  HALF: ids number the halves of the cut tiles.
// RES: a residual is added to the rounded outputs.
template <bool FP8, int OUT, int TM, int TN, int NSTAGE, bool HALF, bool RES>
__device__ __forceinline__ void walk(const WalkArgs& w, uint8_t* smem, int pid, int count) {
  const GemmArgs& p = w.g;
  static_assert(OUT == OUT_BF16 || (OUT == OUT_F32 && !RES), "outputs");
  constexpr int BM = 128 * TM, BN = 64 * TN, BK = 128, NTHREADS = 512;
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int A_LOADS = BM * BK / 16 / NTHREADS, B_LOADS = BN * BK / 16 / NTHREADS, NLOADS = A_LOADS + B_LOADS;
  constexpr int KSUB = FP8 ? 64 : 32, NKS = BK / KSUB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave / 2, wave_n = wave % 2;
  const int M = p.M, N = p.N, K = p.K, nk = (K + BK - 1) / BK;
  const int col = lane & 31, rq = (lane >> 5) * 4;
  const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A, (uint32_t)M * (uint32_t)p.lda), Br = make_rsrc(p.B, (uint32_t)N * (uint32_t)K);

  // A load instruction of a wavefront fills 1 KiB = 8 tile rows; wavefront w owns the row groups w, w + 8, ... of A and B.
  // The 16-byte pieces of a row are permuted as in gemm_kernel: piece c of row r at slot c ^ (r / 2 % 8).
  const int ld_row = wave * 8 + lane / 8;
  const int ld_piece = ((lane % 8) ^ (ld_row / 2 % 8)) * 16;
  uint32_t vo[NLOADS];  // this lane's byte offsets of the tile whose stages are being requested
  // Column of the tile behind accumulator column j of a lane with `col` c, in wavefronts wn: j = 0 and 1 are neighbours, so that a lane
  // holds a dword of bf16 output and a row's 32 lanes a whole line of 128 bytes.  (As 64 bytes a row, paired across lanes, the
  // stores were what bounded short K: us, then -> so: 3000 x 2416 x 1024 15.7 -> 11.1, 2816 x 9472 x 896 50.8 -> 31.1, 7000 x 5056 x
  // 768 52.6 -> 34.5, 4096 x 11264 x 2048 97.6 -> 95.0, fp32 4096 x 4096 x 1024 41.9 -> 24.4.  Written back instead of through, the
  // halves meet in L2: 17.4, 33.6, 38.5, 98.4, 34.1.)  The third column of
  // 192-wide tiles fills 64 bytes of the line between, each wavefront its half.  The order is made where rows of B are requested.
  auto column_of = [&](int wn, int j, int c) { return j == 2 ? 64 + wn * 32 + c : wn * (TN == 3 ? 128 : 64) + 2 * c + j; };
  struct Where {
    int m0, n0;
  };
  auto where = [&](int id) {
    int t = xcd_run(id, count), sub = 0;
    if constexpr (HALF) sub = t % 2, t = w.full + t / 2;
    const int group_sz = GROUP_M * p.tiles_n, group = t / group_sz, first_m = group * GROUP_M;
    const int gm = p.tiles_m - first_m < GROUP_M ? p.tiles_m - first_m : GROUP_M, in_group = t - group * group_sz;
    Where at;
    at.m0 = (first_m + in_group % gm) * 256 + sub * 128;
    at.n0 = in_group / gm * BN;
    return at;
  };
  auto aim = [&](const Where& at) {  // rows past the edge: the last row again, their outputs are not stored
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
      const int r = at.m0 + ld_row + 64 * i;
      vo[i] = (uint32_t)(r < M ? r : M - 1) * (uint32_t)p.lda + (uint32_t)ld_piece;
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int r = at.n0 + column_of((ld_row + 64 * i) / (32 * TN), (ld_row + 64 * i) / 32 % TN, (ld_row + 64 * i) % 32);
      vo[A_LOADS + i] = (uint32_t)(r < N ? r : N - 1) * (uint32_t)K + (uint32_t)ld_piece;
    }
  };
  auto issue_load = [&](int k0, int buf, int idx) {  // pieces past K: outside the descriptor, zeros in LDS
    uint8_t* st = smem + buf * STAGE + wave * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(idx < A_LOADS ? Ar : Br,
                                             (lds_void*)(st + (idx < A_LOADS ? idx * 8192 : BM * BK + (idx - A_LOADS) * 8192)), 16,
                                             k0 + ld_piece < K ? vo[idx] : OOB_OFFSET, k0, 0, 0);
  };

  float* const sx_lds = reinterpret_cast<float*>(smem + NSTAGE * STAGE) + wave * 64;

  using acc_t = typename Acc<FP8>::type;
  using frag_t = typename Frag<FP8>::type;
  acc_t acc[TM][TN];
  frag_t af[2][TM], bf[2][TN];
  const int fr_a = (wave_m * 32 * TM + col) * BK, fr_b = BM * BK + (wave_n * 32 * TN + col) * BK;
  const int fsw = col / 2 % 8;
  const int swz = FP8 ? (((lane >> 5) * 2) ^ fsw) << 4 : ((lane >> 5) ^ fsw) << 4;
  auto load_frag = [&](const uint8_t* st, int ks, int f, frag_t (&a)[TM], frag_t (&b)[TN]) {
    const bool is_a = f == 0 || f > TN;  // in the order the products need them: A0, B0, B1, A1
    const int idx = f == 0 ? 0 : f <= TN ? f - 1 : f - TN;
    const uint8_t* base = st + (is_a ? fr_a : fr_b) + idx * 32 * BK;
    if constexpr (!FP8) {
      const v4i v = *reinterpret_cast<const v4i*>(base + (((ks * 2) << 4) ^ swz));
      if (is_a) a[idx] = v; else b[idx] = v;
    } else {
      const int o0 = ((ks * 4) << 4) ^ swz;
      const v4i lo = *reinterpret_cast<const v4i*>(base + o0), hi = *reinterpret_cast<const v4i*>(base + (o0 ^ 16));
      const v8i v = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      if (is_a) a[idx] = v; else b[idx] = v;
    }
  };
  // One sub-step: its products, the next sub-step's fragment reads and the loads [LD0, LD1) of the requested stage written between
  // them (see gemm_kernel)
  auto slot = [&](auto cur_c, const uint8_t* st_next, int ks_next, int k_ld, int b_ld, auto lo_c, auto hi_c) {
    constexpr int CUR = decltype(cur_c)::value, LD0 = decltype(lo_c)::value, NLD = decltype(hi_c)::value - LD0;
    constexpr int NMMA = TM * TN, NFR = TM + TN;
#pragma unroll
    for (int m = 0; m < NMMA; ++m) {
      acc[m / TN][m % TN] = mma<FP8>(af[CUR][m / TN], bf[CUR][m % TN], acc[m / TN][m % TN]);
#pragma unroll
      for (int f = (m * NFR) / NMMA; f < ((m + 1) * NFR) / NMMA; ++f) load_frag(st_next, ks_next, f, af[CUR ^ 1], bf[CUR ^ 1]);
#pragma unroll
      for (int q = (m * NLD) / NMMA; q < ((m + 1) * NLD) / NMMA; ++q) issue_load(k_ld, b_ld, LD0 + q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using c0 = std::integral_constant<int, 0>;
  using c1 = std::integral_constant<int, 1>;
  using all = std::integral_constant<int, NLOADS>;
  int b_cur = 0;  // buffer of the current stage
  // A K step: its first fragments are in af[0].  Requests the stage two steps on (k_ld, by vo): with three buffers spread over the
  // step, into the one that the step before left; with two behind the step's barrier, all at once, into the step's own (spread
  // over the step that follows, its last loads had a quarter of that to arrive in: 1476 x 6480 x 4448 53.8 us, 50.9 so).
  // BEHIND: vector memory operations that may still be in flight behind the next stage's loads, besides this step's own loads.
  auto step = [&](int k_ld, auto behind_c) {
    constexpr int BEHIND = (NSTAGE == 3 ? NLOADS : 0) + decltype(behind_c)::value;
    const int b_next = b_cur == NSTAGE - 1 ? 0 : b_cur + 1, b_prev = b_cur == 0 ? NSTAGE - 1 : b_cur - 1;
    const uint8_t *st = smem + b_cur * STAGE, *st_next = smem + b_next * STAGE;
    using spread = std::integral_constant<int, NSTAGE == 3 ? NLOADS : 0>;
    if constexpr (NKS == 4) {
      using l1 = std::integral_constant<int, spread::value / 3>;
      using l2 = std::integral_constant<int, spread::value * 2 / 3>;
      slot(c0{}, st, 1, k_ld, b_prev, c0{}, l1{});
      slot(c1{}, st, 2, k_ld, b_prev, l1{}, l2{});
      slot(c0{}, st, 3, k_ld, b_prev, l2{}, spread{});
    } else {
      slot(c0{}, st, 1, k_ld, b_prev, c0{}, spread{});
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the last fragments of the stage are in registers
    AQ_WAIT_VMCNT(BEHIND < 63 ? BEHIND : 63);  // the next stage has landed
    AQ_BARRIER();
    slot(c1{}, st_next, 0, k_ld, b_cur, spread{}, all{});
    b_cur = b_next;
  };

  Where now = where(pid);
  aim(now);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int q = 0; q < NLOADS; ++q) issue_load(s * BK, s, q);
  AQ_WAIT_VMCNT(NLOADS);  // stage 0 has landed
  AQ_BARRIER();
#pragma unroll
  for (int f = 0; f < TM + TN; ++f) load_frag(smem, 0, f, af[0], bf[0]);

  constexpr int STORES = TM * (TN == 2 ? 16 : OUT == OUT_BF16 ? 24 : 32);  // per lane and tile
  for (bool first = true;; first = false) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    int k0 = 2 * BK;
    if (first)
      step(k0, c0{});
    else
      step(k0, std::integral_constant<int, STORES>{});  // the stores of the tile before
    for (int s = 1; s < nk - 2; ++s) step(k0 += BK, c0{});
    // the epilogue's operands, then the next tile's first two stages
    const int mw = now.m0 + wave_m * 32 * TM, nt = now.n0;  // wavefront-uniform
    auto my_column = [&](int j) { return nt + column_of(wave_n, j, col); };
    float sx1 = 1.0f, sw1 = 1.0f, swn[TN], bn[TN];
    uint32_t braw[TN];
    const bool has_bias = p.bias != nullptr, bias_bf16 = p.bias_dtype == AQ_BF16;
    const __amdgpu_buffer_rsrc_t Bsr = make_rsrc(has_bias ? p.bias : (const void*)p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
    if constexpr (FP8) {
      sx1 = *p.sx;
      sw1 = *p.sw;
    } else {
      const __amdgpu_buffer_rsrc_t Sr = make_rsrc(p.sx, (uint32_t)M * 4u), Wr = make_rsrc(p.sw, (uint32_t)N * 4u);
      // the wavefront's 32 TM row scales wait in LDS, in a place of its own: as registers they are what makes wide tiles spill
      if constexpr (TM == 2)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Sr, (lds_void*)sx_lds, 4, (uint32_t)(mw + lane) * 4u, 0, 0, 0);
      else if (lane < 32)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(Sr, (lds_void*)sx_lds, 4, (uint32_t)(mw + lane) * 4u, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        swn[j] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Wr, my_column(j) * 4, 0, 0));
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
      braw[j] = bias_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(Bsr, my_column(j) * 2, 0, 0)
                          : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Bsr, my_column(j) * 4, 0, 0);
    const bool odd = lane & 1;
    constexpr int ESZ = OUT == OUT_BF16 ? 2 : 4;
    const uint32_t rowb = (uint32_t)N * ESZ;
    // byte offsets, from the tile's first column of the wavefront's first row, of what this lane stores of its pair of columns and (bf16:
    // paired with the neighbouring lane's, the even lane the first row of two, the odd lane the second) of its third column
    const uint32_t pair_at = my_column(0) < N ? (uint32_t)rq * rowb + (uint32_t)(my_column(0) - nt) * ESZ : OOB_OFFSET;
    uint32_t third_at = OOB_OFFSET;
    if constexpr (TN == 3)
      if (my_column(2) < N) {
        const uint32_t c = (uint32_t)(my_column(2) - nt);
        third_at = (uint32_t)rq * rowb + (OUT == OUT_BF16 ? (c & ~1u) * 2 + (odd ? rowb : 0u) : c * 4);
      }
    // The wavefront's window of the outputs, from the tile's first column to the end of its last row: rows past M fall outside.  (Their
    // offset is the lane's alone: the range check takes a scalar offset off the window's size first, which may be smaller.)
    const int rows = M - mw < 32 * TM ? M - mw : 32 * TM;
    const uint32_t window = rows > 0 ? (uint32_t)rows * rowb - (uint32_t)nt * ESZ : 0u;
    const int64_t first_out = rows > 0 ? ((int64_t)mw * N + nt) * ESZ : 0;
    // Each lane reads what it then writes (the residual may be the output): as many columns as the registers have room for two
    // steps before they are needed, the others in front of the epilogue.  192-wide FP8 tiles have room for half of them there, the
    // rows of one accumulator row, and ask for the other half behind the first one's stores: 244 registers; all at once spilled 12 of
    // 256, median of 150 sizes 1.067 x this time (K up to 1024 1.12, above 4096 1.04).
    constexpr int EARLY = !RES ? 0 : TN == 2 || !FP8 ? 2 : 0;
    uint32_t rr[RES ? TM : 1][16], rt[RES ? TM : 1][8];
    const __amdgpu_buffer_rsrc_t Rr = make_rsrc(reinterpret_cast<const uint8_t*>(RES ? p.res : p.C) + first_out, window);
    auto load_residual = [&](int i0, int i1, auto pairs_c, auto third_c) {
#pragma unroll
      for (int i = i0; i < i1; ++i) {
        if constexpr (decltype(pairs_c)::value) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            rr[i][r] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, pair_at + (i * 32 + r / 4 * 8 + r % 4) * rowb, 0, 0);
        }
        if constexpr (decltype(third_c)::value) {
#pragma unroll
          for (int h = 0; h < 8; ++h)
            rt[i][h] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Rr, third_at + (i * 32 + h / 2 * 8 + h % 2 * 2) * rowb, 0, 0);
        }
      }
    };
    using early = std::integral_constant<bool, EARLY != 0>;
    using late = std::integral_constant<bool, RES && EARLY == 0>;
    using third = std::integral_constant<bool, RES && TN == 3>;
    load_residual(0, TM, early{}, std::false_type{});
    asm volatile("" ::: "memory");
    const bool last = pid + (int)gridDim.x >= count;
    pid += gridDim.x;
    if (!last) {
      now = where(pid);
      aim(now);
    } else {  // nothing: loads outside the descriptors touch no memory
#pragma unroll
      for (int i = 0; i < NLOADS; ++i) vo[i] = OOB_OFFSET;
    }
    step(0, std::integral_constant<int, EARLY * TM * 8>{});  // the residual may still be on its way
    step(BK, c0{});
    load_residual(0, late::value ? 1 : TM, late{}, third{});
    asm volatile("" ::: "memory");

    // ---- epilogue, as in gemm_kernel: three rounded operations, rows of neighbouring columns paired across lanes
    const __amdgpu_buffer_rsrc_t Cr = make_rsrc(reinterpret_cast<uint8_t*>(p.C) + first_out, window);
#pragma unroll
    for (int j = 0; j < TN; ++j) bn[j] = !has_bias ? 0.0f : bias_bf16 ? bf16_bits_to_f32(braw[j]) : __uint_as_float(braw[j]);
    // rounded output + residual, rounded again: what a separate add gives
    auto add_residual = [](uint32_t pk, uint32_t r) {
      return pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(r << 16)),
                         __fadd_rn(__uint_as_float(pk & 0xffff0000u), __uint_as_float(r & 0xffff0000u)));
    };
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (late::value && i > 0) load_residual(i, i + 1, late{}, third{});
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int r0 = i * 32 + g * 8;
        v4f sxq = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (!FP8) sxq = *reinterpret_cast<const v4f*>(sx_lds + r0 + rq);
        float y[TN][4];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if constexpr (FP8)
              y[j][q] = __fadd_rn(__fmul_rn(__fmul_rn(acc[i][j][g * 4 + q], sx1), sw1), bn[j]);
            else
              y[j][q] = __fadd_rn(__fmul_rn(__fmul_rn((float)acc[i][j][g * 4 + q], sxq[q]), swn[j]), bn[j]);
          }
        if constexpr (OUT == OUT_F32) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const v2i_t o = {__float_as_int(y[0][q]), __float_as_int(y[1][q])};
            __builtin_amdgcn_raw_buffer_store_b64(o, Cr, pair_at + (r0 + q) * rowb, 0, STORE_WT);
            if constexpr (TN == 3) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y[2][q]), Cr, third_at + (r0 + q) * rowb, 0, STORE_WT);
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            uint32_t pk = pack_bf16x2(y[0][q], y[1][q]);
            if constexpr (RES) pk = add_residual(pk, rr[i][g * 4 + q]);
            __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, pair_at + (r0 + q) * rowb, 0, STORE_WT);
          }
          if constexpr (TN == 3) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {  // rows 2h, 2h + 1 of two lanes -> two columns of one row (see gemm_kernel)
              const uint32_t mine = pack_bf16x2(y[2][2 * h], y[2][2 * h + 1]);
              const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xB1 /* quad_perm [1,0,3,2] */, 0xf, 0xf, true);
              uint32_t pk = __builtin_amdgcn_perm(other, mine, odd ? 0x03020706u : 0x05040100u);
              if constexpr (RES) pk = add_residual(pk, rt[i][g * 2 + h]);
              __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, third_at + (r0 + 2 * h) * rowb, 0, STORE_WT);
            }
          }
        }
      }
    }
    if (last) break;
  }
  AQ_WAIT_VMCNT(0);  // nothing lands in LDS behind the walk
  AQ_BARRIER();
}

template <bool FP8, int OUT, int TN, int NSTAGE, bool RES>
__global__ __launch_bounds__(512) void gemm_walk_kernel(WalkArgs w) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[NSTAGE * (256 + 64 * TN) * 128 + 8 * 64 * 4];
  walk<FP8, OUT, 2, TN, NSTAGE, false, RES>(w, smem, blockIdx.x, w.full);  // the grid is no larger than w.full
  if constexpr (TN == 2)
    if ((int)blockIdx.x < w.halves) walk<FP8, OUT, 1, 2, NSTAGE, true, RES>(w, smem, blockIdx.x, w.halves);
}

// Four K steps at least (one to begin a tile's loop, two that request the next tile's stages), pairs of columns, operands within
// a 32-bit offset.  (Which tile, and whether this kernel at all: choose_tile_for.)
bool gemm_walk_ok(const GemmArgs& a, int out) {
  if (a.K < 512 || a.N % 2 || (int64_t)a.M * a.lda > (int64_t)OOB_OFFSET || (int64_t)a.N * a.K > (int64_t)OOB_OFFSET) return false;
  return out == OUT_BF16 || !a.res;
}

template <bool FP8, int OUT, int TN, int NSTAGE, bool RES>
static int walk_launch(const GemmArgs& a, hipStream_t st) {
  WalkArgs w{};
  w.g = a;
  w.g.tiles_m = (a.M + 255) / 256;
  w.g.tiles_n = (a.N + 64 * TN - 1) / (64 * TN);
  const int cus = device_cus(), nt = w.g.tiles_m * w.g.tiles_n, rest = nt % cus;
  w.halves = TN == 2 && gemm_walk_halves(nt, cus) ? 2 * rest : 0;
  w.full = nt - w.halves / 2;
  queue_kernel(gemm_walk_kernel<FP8, OUT, TN, NSTAGE, RES>, dim3((unsigned)(w.full < cus ? w.full : cus)), dim3(512), 0, st, w);
  return (int)hipGetLastError();
}
template <bool FP8, int OUT>
int gemm_walk_launch(const GemmArgs& a, hipStream_t st, int width) {
  if constexpr (OUT == OUT_BF16)
    if (a.res)
      return width == 192 ? walk_launch<FP8, OUT, 3, 2, true>(a, st) : walk_launch<FP8, OUT, 2, 3, true>(a, st);
  return width == 192 ? walk_launch<FP8, OUT, 3, 2, false>(a, st) : walk_launch<FP8, OUT, 2, 3, false>(a, st);
}
template int gemm_walk_launch<false, OUT_BF16>(const GemmArgs&, hipStream_t, int);
template int gemm_walk_launch<false, OUT_F32>(const GemmArgs&, hipStream_t, int);
template int gemm_walk_launch<true, OUT_BF16>(const GemmArgs&, hipStream_t, int);
template int gemm_walk_launch<true, OUT_F32>(const GemmArgs&, hipStream_t, int);

}  // namespace aq
