// The tiled GEMM of gemm_mfma.hip for more 256 x 128 tiles than compute units, or with a residual: at most one resident
// workgroup per compute unit walks tiles, and its K loop does not stop between them.
//
// What bounds it: a tile of K = 1536 or 2048 is 12 to 16 K steps of 1024 matrix-core cycles, and the separate tiles of
// gemm_kernel put a drain of the stores, the latency of the first stages, a step without loads and the epilogue around
// them: 22 k cycles a tile for 13 k of K loop.  Here the last two steps of a tile already request the next tile's first
// two stages, so its first fragments are in registers when the epilogue ends, and the epilogue's stores drain under the
// next tile's first step.  (gemm_kernel also requests three stages past the last one for the sake of an even count, a
// quarter of all fills at K = 1536.)
//
// And the last round: nt tiles on `cus` compute units take ceil(nt / cus) rounds, the last of them nearly empty in the
// worst case (864 tiles: 3.4 rounds in the time of 4).  When at most half the compute units would have a tile in it, its
// tiles are cut in two, 128 x 128 each -- behind three rounds or more: the halves run code that no instruction cache
// holds yet, which costs what they save after a single round (384 tiles of K = 2048: 38.5 us against 32.7 with whole ones).
//
// Measured in one process, gemm_kernel's 256 x 128 tile -> this one, us: int8 2048 x 13824 x 1536 50.2 -> 46.1 on one
// device, 61.7 -> 49.4 on another; 4096 x 11264 x 2048 98.4 -> 90.9, 105 -> 93; 4096 x 4096 x 2048 35.2 -> 33.4, 46.8 -> 43.9;
// 8192 x 8192 x 2048 138 -> 129, 144 -> 134; FP8 2048 x 13824 x 1536 45.3 -> 41.4, 50 -> 43.  The rest is the K loop at the
// clock the power limit leaves.  (A ninth wavefront that touches the lines six steps ahead took 38 us for 4096 x 4096
// x 2048 where memory was slow, 2 to 10 % more elsewhere: not kept.)
//
// Int8: whole-number sums, one epilogue for all tiles: the bits of gemm_kernel.  FP8: the same order of sums.
#include "aq_gemm.h"

namespace aq {

struct WalkArgs {
  GemmArgs g;
  int full;    // 256 x 128 tiles that are walked whole; the ones behind them are cut in two
  int halves;  // 128 x 128 tiles
};

// Tile `idx` of `count`: workgroup ids are dealt round-robin to the XCDs; a contiguous run of ids per XCD, as tile_of_block
__device__ __forceinline__ int xcd_run(int pid, int count) {
  const int per = count / NUM_XCD, rem = count % NUM_XCD, xcd = pid % NUM_XCD, idx = pid / NUM_XCD;
  return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// A walk over tiles of 128 TM x 128 on 4 x 2 wavefronts of (32 TM) x 64.  HALF: ids number the halves of the cut tiles.
// RES: a residual is added to the rounded outputs.
template <bool FP8, int TM, bool HALF, bool RES>
__device__ __forceinline__ void walk(const WalkArgs& w, uint8_t* smem, int pid, int count) {
  const GemmArgs& p = w.g;
  constexpr int TN = 2, BM = 128 * TM, BN = 128, BK = 128, NSTAGE = 3, NWAVES = 8, NTHREADS = 512;
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int A_LOADS = BM * BK / 16 / NTHREADS, B_LOADS = BN * BK / 16 / NTHREADS, NLOADS = A_LOADS + B_LOADS;
  constexpr int KSUB = FP8 ? 64 : 32, NKS = BK / KSUB;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave / 2, wave_n = wave % 2;
  const int M = p.M, N = p.N, K = p.K, nk = K / BK;
  const int col = lane & 31, rq = (lane >> 5) * 4;
  const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A, (uint32_t)M * (uint32_t)K), Br = make_rsrc(p.B, (uint32_t)N * (uint32_t)K);

  // A load instruction of a wavefront fills 1 KiB = 8 tile rows; wavefront w owns the row groups w, w + 8, ... of A and B.
  // The 16-byte pieces of a row are permuted as in gemm_kernel: piece c of row r at slot c ^ (r / 2 % 8).
  const int ld_row = wave * 8 + lane / 8;
  const uint32_t ld_piece = (uint32_t)((lane % 8) ^ (ld_row / 2 % 8)) * 16;
  uint32_t vo[NLOADS];  // this lane's byte offsets of the tile whose stages are being requested
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
      vo[i] = (uint32_t)(r < M ? r : M - 1) * (uint32_t)K + ld_piece;
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
      const int r = at.n0 + ld_row + 64 * i;
      vo[A_LOADS + i] = (uint32_t)(r < N ? r : N - 1) * (uint32_t)K + ld_piece;
    }
  };
  auto issue_load = [&](int k0, int buf, int idx) {
    uint8_t* st = smem + buf * STAGE + wave * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(idx < A_LOADS ? Ar : Br,
                                             (lds_void*)(st + (idx < A_LOADS ? idx * 8192 : BM * BK + (idx - A_LOADS) * 8192)), 16,
                                             vo[idx], k0, 0, 0);
  };

  using acc_t = typename Acc<FP8>::type;
  using frag_t = typename Frag<FP8>::type;
  acc_t acc[TM][TN];
  frag_t af[2][TM], bf[2][TN];
  const int fr_a = (wave_m * 32 * TM + col) * BK, fr_b = BM * BK + (wave_n * 64 + col) * BK;
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
  // One sub-step: its products, the next sub-step's fragment reads and a share [LD0, LD1) of the requested stage's loads
  // written between them (see gemm_kernel)
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
  int b_prev = 2;  // buffer of the stage before the current one: free, takes the stage after next
  // K step s of the tile: its first fragments are in af[0]; requests the stage two steps on (k_ld, by vo); BEHIND: vector
  // memory operations that may still be in flight behind the next stage's loads, besides this step's own loads
  auto step = [&](int k_ld, auto behind_c) {
    constexpr int BEHIND = decltype(behind_c)::value;
    const int b_cur = b_prev == NSTAGE - 1 ? 0 : b_prev + 1, b_next = b_cur == NSTAGE - 1 ? 0 : b_cur + 1;
    const uint8_t *st = smem + b_cur * STAGE, *st_next = smem + b_next * STAGE;
    if constexpr (NKS == 4) {
      using l1 = std::integral_constant<int, NLOADS / 3>;
      using l2 = std::integral_constant<int, NLOADS * 2 / 3>;
      slot(c0{}, st, 1, k_ld, b_prev, c0{}, l1{});
      slot(c1{}, st, 2, k_ld, b_prev, l1{}, l2{});
      slot(c0{}, st, 3, k_ld, b_prev, l2{}, all{});
    } else {
      slot(c0{}, st, 1, k_ld, b_prev, c0{}, all{});
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the last fragments of the stage are in registers
    AQ_WAIT_VMCNT(NLOADS + BEHIND < 63 ? NLOADS + BEHIND : 63);  // the next stage has landed
    AQ_BARRIER();
    slot(c1{}, st_next, 0, 0, 0, c0{}, c0{});
    b_prev = b_cur;
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

  constexpr int STORES = TM * TN * 8;  // per lane and tile
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
    const int mw = now.m0 + wave_m * 32 * TM, nw = now.n0 + wave_n * 64;  // wavefront-uniform
    float sx1 = 1.0f, sw1 = 1.0f, sxr[TM][4][4], swn[TN], bn[TN];
    uint32_t braw[TN];
    const bool has_bias = p.bias != nullptr, bias_bf16 = p.bias_dtype == AQ_BF16;
    const __amdgpu_buffer_rsrc_t Bsr = make_rsrc(has_bias ? p.bias : (const void*)p.sw, has_bias ? (uint32_t)N * (bias_bf16 ? 2u : 4u) : 0u);
    if constexpr (FP8) {
      sx1 = *p.sx;
      sw1 = *p.sw;
    } else {
      const __amdgpu_buffer_rsrc_t Sr = make_rsrc(p.sx, (uint32_t)M * 4u), Wr = make_rsrc(p.sw, (uint32_t)N * 4u);
      if ((M & 3) == 0) {  // uniform: the 4 rows are all in or all out
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const uint4 t = buffer_load_16(Sr, (uint32_t)(mw + i * 32 + g * 8 + rq) * 4u);
            sxr[i][g][0] = __uint_as_float(t.x), sxr[i][g][1] = __uint_as_float(t.y);
            sxr[i][g][2] = __uint_as_float(t.z), sxr[i][g][3] = __uint_as_float(t.w);
          }
      } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              sxr[i][g][q] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Sr, (mw + i * 32 + g * 8 + rq + q) * 4, 0, 0));
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
        swn[j] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Wr, (nw + j * 32 + col) * 4, 0, 0));
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
      braw[j] = bias_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(Bsr, (nw + j * 32 + col) * 2, 0, 0)
                          : (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(Bsr, (nw + j * 32 + col) * 4, 0, 0);
    const bool odd = lane & 1;
    const uint32_t rowb = (uint32_t)N * 2;
    uint32_t vbase[TN];  // byte offset of the first pair that this lane stores of column j, from the wavefront's first output
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int cj = j * 32 + col;
      vbase[j] = nw + cj < N ? (uint32_t)rq * rowb + (uint32_t)(cj & ~1) * 2 + (odd ? rowb : 0u) : OOB_OFFSET;
    }
    // Each lane reads the pairs that it then writes (the residual may be the output), two steps before they are needed.
    uint32_t rr[RES ? TN : 1][TM][4][2];
    if constexpr (RES) {
      const __amdgpu_buffer_rsrc_t Rr = make_rsrc(reinterpret_cast<const uint8_t*>(p.res) + ((int64_t)mw * N + nw) * 2, 0x40000000u);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int r0 = i * 32 + g * 8 + 2 * h;
              rr[j][i][g][h] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                  Rr, mw + r0 + rq + (odd ? 1 : 0) < M ? vbase[j] : OOB_OFFSET, r0 * rowb, 0);
            }
    }
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
    step(0, std::integral_constant<int, RES ? STORES : 0>{});  // the residual may still be on its way
    step(BK, c0{});

    // ---- epilogue, as in gemm_kernel: three rounded operations, rows of neighbouring columns paired across lanes
    const __amdgpu_buffer_rsrc_t Cr = make_rsrc(reinterpret_cast<uint8_t*>(p.C) + ((int64_t)mw * N + nw) * 2, 0x40000000u);
    const uint32_t perm_sel = odd ? 0x03020706u : 0x05040100u;
    auto store_all = [&](auto check_c) {
      constexpr bool CHECK_M = decltype(check_c)::value;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        bn[j] = !has_bias ? 0.0f : bias_bf16 ? bf16_bits_to_f32(braw[j]) : __uint_as_float(braw[j]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int r0 = i * 32 + g * 8;
            float y[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if constexpr (FP8)
                y[q] = __fadd_rn(__fmul_rn(__fmul_rn(acc[i][j][g * 4 + q], sx1), sw1), bn[j]);
              else
                y[q] = __fadd_rn(__fmul_rn(__fmul_rn((float)acc[i][j][g * 4 + q], sxr[i][g][q]), swn[j]), bn[j]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const uint32_t mine = pack_bf16x2(y[2 * h], y[2 * h + 1]);
              const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xB1 /* quad_perm [1,0,3,2] */, 0xf, 0xf, true);
              uint32_t pk = __builtin_amdgcn_perm(other, mine, perm_sel);
              if constexpr (RES)  // rounded output + residual, rounded again: what a separate add gives
                pk = pack_bf16x2(__fadd_rn(__uint_as_float(pk << 16), __uint_as_float(rr[j][i][g][h] << 16)),
                                 __fadd_rn(__uint_as_float(pk & 0xffff0000u), __uint_as_float(rr[j][i][g][h] & 0xffff0000u)));
              uint32_t at = vbase[j];
              if (CHECK_M && mw + r0 + rq + 2 * h + (odd ? 1 : 0) >= M) at = OOB_OFFSET;
              __builtin_amdgcn_raw_buffer_store_b32(pk, Cr, at, (r0 + 2 * h) * rowb, STORE_WT);
            }
          }
      }
    };
    if (mw + 32 * TM <= M)
      store_all(std::integral_constant<bool, false>{});
    else
      store_all(std::integral_constant<bool, true>{});
    if (last) break;
  }
  AQ_WAIT_VMCNT(0);  // nothing lands in LDS behind the walk
  AQ_BARRIER();
}

template <bool FP8, bool RES>
__global__ __launch_bounds__(512) void gemm_walk_kernel(WalkArgs w) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[3 * (256 + 128) * 128];
  walk<FP8, 2, false, RES>(w, smem, blockIdx.x, w.full);  // the grid is no larger than w.full
  if ((int)blockIdx.x < w.halves) walk<FP8, 1, true, RES>(w, smem, blockIdx.x, w.halves);
}

// bf16 outputs, whole K steps, four of them at least (two to begin a tile's loop, two that request the next tile's stages),
// pairs of columns, operands within a 32-bit offset.  Up to one tile per compute unit there is nothing to walk to, and it is the
// residual, requested two steps ahead, that pays: us, gemm_kernel -> here: 4096 x 2048 x 2048 21.9 -> 19.7, x 5632 45.2 -> 43.3,
// 3000 x 2048 x 1024 12.9 -> 11.8 (several rounds: 4096 x 4096 x 2048 41.5 -> 37.8, 2048 x 13824 x 1536 59.9 -> 50.6).  Without
// one, one round of tiles goes from 4 % faster to 1.5 % slower with the card's clocks: gemm_kernel keeps it.
bool gemm_walk_ok(const GemmArgs& a) {
  if (a.K % 128 || a.K < 512 || a.N % 2 || (int64_t)a.M * a.K > (int64_t)OOB_OFFSET || (int64_t)a.N * a.K > (int64_t)OOB_OFFSET)
    return false;
  return a.res || (int64_t)((a.M + 255) / 256) * ((a.N + 127) / 128) > device_cus();
}

template <bool FP8>
int gemm_walk_launch(const GemmArgs& a, hipStream_t st) {
  WalkArgs w{};
  w.g = a;
  w.g.tiles_m = (a.M + 255) / 256;
  w.g.tiles_n = (a.N + 127) / 128;
  const int cus = device_cus(), nt = w.g.tiles_m * w.g.tiles_n, rest = nt % cus;
  w.halves = rest <= cus / 2 && nt >= 3 * cus ? 2 * rest : 0;
  w.full = nt - w.halves / 2;
  queue_kernel(a.res ? gemm_walk_kernel<FP8, true> : gemm_walk_kernel<FP8, false>, dim3((unsigned)(w.full < cus ? w.full : cus)),
               dim3(512), 0, st, w);
  return (int)hipGetLastError();
}
template int gemm_walk_launch<false>(const GemmArgs&, hipStream_t);
template int gemm_walk_launch<true>(const GemmArgs&, hipStream_t);

}  // namespace aq
