// Causal self-attention over a prompt or a chunk of one (prefill): what the
// reference computes with repeat_kv + scaled_dot_product_attention
// (astrai/model/components/attention.py:15-23, 93-100).  Grouped-query attention
// without repeating heads, bf16 tensors, fp32 softmax statistics and
// accumulation, head dimension 64 or 128.  Keys and values come from the new
// tokens' own rows, or from the paged cache (a chunk on top of cached tokens).
//
// Workgroup = (32 QW query positions, one query head, one sequence), QW x KW
// wavefronts.  A block of 64 keys against 32 queries is one serial chain of products,
// softmax and products, about 0.85 us at head dimension 64 whatever else the device
// does, and a query's blocks follow one another: a prompt of a few hundred tokens or a
// short chunk on a long context leaves most of the chip idle while that chain runs.
// KW > 1 shortens it: the KW wavefronts of a query row take KW blocks' scores and
// probabilities side by side and leave them in LDS, then each adds all KW blocks, in
// order, to its share of the head dimension.  Sums, running maxima and roundings are
// those of KW = 1: same bits.
//
// Everything is computed transposed so that no register ever has to change lanes:
//
//   S^T[key, q] = K Q^T    v_mfma_f32_32x32x16_bf16 with A = K (rows of the LDS
//                          tile, 16-byte reads), B = Q^T (the wavefront's query
//                          rows, held in registers for the whole kernel).  A
//                          lane ends up with the scores of ONE query (column
//                          l % 32) against 16 keys per 32-key tile.
//   softmax                per query = per lane: running maximum and denominator
//                          need one exchange with lane l ^ 32 per block, the
//                          rescale of the output accumulator is lane-wise.
//   O^T[d, q] += V^T P^T   B = P^T: the probabilities a lane already holds are,
//                          packed to bf16 in register order, exactly its operand
//                          (the matrix core does not care which key sits in which
//                          k slot as long as A agrees); A = V^T through the
//                          transposing LDS read (ds_read_b64_tr_b16: 4 keys of one
//                          dimension per lane from 4 rows of 16 dimensions).
//
// K and V rows go from memory straight into LDS (16 bytes per lane, no registers)
// as they are, one block ahead of the products, into the other of two buffers: one
// barrier per block.  A row's 16-byte pieces are permuted (row_key) so that both
// the row reads of K and the transposing reads of V spread over all banks.
#include "aq_common.h"
#include "aq_rope.h"

namespace aq {

struct PrefillAttnArgs {
  const uint16_t* q;   // element (b, s, h, d) at q + (b*S + s)*q_stride + h*D + d
  const uint16_t* k;   // likewise with KV heads
  const uint16_t* v;
  uint16_t* out;       // [B, S, Hq, D]
  int64_t q_stride, k_stride, v_stride;  // elements between consecutive tokens
  float scale_log2e;
  int S, Hq, Hkv, B;
  // PAGED kernels: keys and values of positions 0 .. start + S - 1 are read through the page table from
  // caches [n_pages, page, Hkv, D]; query s sits at position start + s
  const uint16_t* kc;
  const uint16_t* vc;
  const int64_t* table;  // [B, P] physical page ids, < 0: unmapped (zero keys and values)
  int64_t P, page, n_pages;
  int start, page_shift;
  // ROT kernels:
  const float* freqs;    // [S, D/2, 2] (cos, sin) per sequence; sequences freqs_stride floats apart (0: shared)
  int64_t freqs_stride;
  const uint16_t* q_gain;
  float eps;
  int table_lds;  // entries of the page table that are copied into LDS first (all a launch needs, or 0: read from memory)
  int paired;     // != 0: the second half of the workgroups takes the query blocks lightest first
  int wgs;        // workgroups that attend; the ones behind them read ahead
  unsigned ahead_wgs;
  Ahead ahead;
};

typedef __bf16 pa_bf16x8 __attribute__((ext_vector_type(8)));
typedef short pa_s16x4 __attribute__((ext_vector_type(4)));
typedef float pa_f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void pa_lds_void;
typedef __attribute__((address_space(3))) pa_s16x4 pa_lds_s16x4;

__device__ const uint4 pa_zero_row[16] = {};  // what a row of an unmapped page reads as

// 16 bytes per lane from memory to LDS, 1 KiB in lane order from byte `at` (wavefront-uniform).  Written out because the compiler,
// given the builtin, waits for every such load in flight before the next LDS read of any kind -- here the other buffer's,
// requested a moment earlier.  The kernel waits itself, before the barrier that hands a buffer over.
__device__ __forceinline__ void load_row_lds(const uint16_t* src, uint32_t at) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "{m0}"(at) : "memory");  // m0 needs a wait state
}

// The 16-byte piece of row r that sits in slot s of the row is s ^ row_key(r): the low bits of r, reversed.  16 rows
// reading the same piece (K) fall on all slots of the bank lines; the 8 neighbouring rows x 64 bytes of a transposing
// read (V) are told apart by their lowest bits, which reversed move a row's pieces by 64 bytes and more.
template <int D>
__device__ __forceinline__ int row_key(int row) {
  if constexpr (D == 64)  // 128-byte rows: two to a bank line
    return (int)(__builtin_bitreverse32((uint32_t)(row >> 1) & 7u) >> 29);
  else
    return (int)(__builtin_bitreverse32((uint32_t)row & 15u) >> 28);
}

// PAGED: a chunk of S new tokens on top of `start` cached ones -- K and V of all start + S positions come from the
// paged cache (the new tokens' rows have been written there already), causality is by position.
// ROT: q holds heads as the projection left them; they are rotated (and, with q_gain, RMS-normalised) as they are read.
template <int D, int QW, int KW, bool PAGED, bool ROT>
__global__ __launch_bounds__(QW* KW * 64) __attribute__((amdgpu_waves_per_eu(2))) void prefill_attn_kernel(PrefillAttnArgs p) {
  if ((int)blockIdx.x >= p.wgs) return read_ahead(p.ahead, (int)blockIdx.x - p.wgs, QW * KW * 64);
  constexpr int QB = 32 * QW;                       // query rows of the workgroup
  constexpr int KB = 64;                            // keys of a block
  constexpr int NT = KB / 32;                       // 32-key tiles of a block
  constexpr int DSTEPS = D / 16;                    // matrix-core steps over the head dimension
  constexpr int DT = D / 32;                        // 32-row tiles of the transposed output
  constexpr int ROWB = 2 * D;                       // bytes of a K or V row
  constexpr int RPI = 1024 / ROWB, LPR = 64 / RPI;  // rows of a 1 KiB load, lanes of a row
  constexpr int TILE = KB * ROWB;                   // bytes of a block's K (or V)
  constexpr int LOADS = TILE / 1024 / QW;           // 1 KiB loads of K (and of V) per wavefront and block
  constexpr int BUF = KW * 2 * TILE;
  static_assert(LOADS >= 1 && TILE % (1024 * QW) == 0, "whole loads per wavefront");
  __shared__ float maxima[KW][QW][32], psums[KW][QW][64];  // (KW > 1)
  extern __shared__ __align__(1024) uint8_t pa_lds[];  // 2 buffers of KW [K block | V block]; page table (PAGED)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = wave % QW, kw = wave / QW;
  const int col = lane & 31, g = lane >> 5;
  const int S = p.S;
  // Workgroups are numbered heaviest first: a query block attends to every key block up to its own, so the
  // last block of a sequence has the most work.  All (head, sequence) pairs of the last query block come
  // first, then the block before it, ... -- the long workgroups start at once and the short ones fill in
  // behind them (in launch order the light blocks of head 0 would start first and the heavy ones of the last
  // heads would run alone at the end: 34 -> 28 us at 8 x 512, 339 -> 219 us at 4 x 2048 x 32 heads).
  // When the whole launch is resident at once, the second half of the numbering runs lightest first instead: the
  // workgroup that joins a heavy one on its compute unit is then a light one.
  const int nqb = (S + QB - 1) / QB, per = p.Hq * p.B;
  const int rank = (int)blockIdx.x / per, hrank = (nqb + 1) / 2;
  const int qblk = (p.paired && rank >= hrank) ? rank - hrank : nqb - 1 - rank;
  const int q0 = qblk * QB, h = ((int)blockIdx.x % per) % p.Hq, b = ((int)blockIdx.x % per) / p.Hq;
  const int kvh = h / (p.Hq / p.Hkv);
  const int qw0 = q0 + qw * 32;            // first query row of this wavefront
  const int qpos = qw0 + col;              // this lane's query
  const int64_t tok0 = (int64_t)b * S;
  const int off = PAGED ? p.start : 0;     // position of query 0
  const int T = off + S;                   // key positions
  const int qw0p = qw0 + off, qposp = qpos + off;  // positions of the wavefront's first / this lane's query
  const int last_q = (q0 + QB < S ? q0 + QB : S) - 1 + off;  // position of the workgroup's last query
  const int last_w = last_q < qw0p + 31 ? last_q : qw0p + 31;  // ... and of the wavefront's
  const int nblk = last_q / KB + 1;                          // blocks that hold a key some query of the workgroup may see
  const int nit = (nblk + KW - 1) / KW;

  // the page table of this sequence, ids checked, where blocks straddle pages: rows of unmapped pages read zeros
  int* const table = reinterpret_cast<int*>(pa_lds + 2 * BUF);
  auto phys_of = [&](int lp) -> int {
    const int64_t t = p.table[(int64_t)b * p.P + lp];
    return t >= 0 && t < p.n_pages ? (int)t : -1;
  };
  if constexpr (PAGED) {
    if (p.table_lds) {
      for (int i = tid; i < p.table_lds; i += QW * KW * 64) table[i] = phys_of(i);
      __syncthreads();
    }
  }
  // this lane's piece of the rows that the wavefront's loads bring: elements into the row
  const int chunk0 = qw * LOADS;
  int pc[LOADS];
#pragma unroll
  for (int c = 0; c < LOADS; ++c) pc[c] = ((lane % LPR) ^ row_key<D>((chunk0 + c) * RPI + lane / LPR)) * 8;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(pa_lds_void*)pa_lds;
  const uint16_t* const kbase = p.k + tok0 * p.k_stride + (int64_t)kvh * D;
  const uint16_t* const vbase = p.v + tok0 * p.v_stride + (int64_t)kvh * D;
  auto issue = [&](int it, int buf) __attribute__((always_inline)) {
    const int j = it * KW + kw;
    if (j >= nblk) return;  // wavefront-uniform
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + buf * BUF + kw * 2 * TILE + chunk0 * 1024);
    const int rows = T - j * KB;  // rows past the last position: any row that is there, masked by causality
    if (!PAGED || p.page % KB == 0) {
      // the block's rows are equally spaced: contiguous tensors, or the whole block in one page (an unmapped one: a row
      // of zeros again and again)
      const uint16_t *ks, *vs;
      int kstep, vstep;
      if constexpr (PAGED) {
        const int lp = __builtin_amdgcn_readfirstlane(p.page_shift >= 0 ? (j * KB) >> p.page_shift : j * KB / (int)p.page);
        const int64_t phys = p.table[(int64_t)b * p.P + lp];
        const int64_t first = ((phys * p.page + (j * KB - lp * (int)p.page)) * p.Hkv + kvh) * D;
        const bool mapped = phys >= 0 && phys < p.n_pages;
        ks = mapped ? p.kc + first : reinterpret_cast<const uint16_t*>(pa_zero_row);
        vs = mapped ? p.vc + first : reinterpret_cast<const uint16_t*>(pa_zero_row);
        kstep = vstep = mapped ? p.Hkv * D : 0;
      } else {
        kstep = (int)p.k_stride, vstep = (int)p.v_stride;
        ks = kbase + (uint32_t)(j * KB * kstep);
        vs = vbase + (uint32_t)(j * KB * vstep);
      }
#pragma unroll
      for (int c = 0; c < LOADS; ++c) {
        int r = (chunk0 + c) * RPI + lane / LPR;
        r = r < rows ? r : rows - 1;
        load_row_lds(ks + (uint32_t)(r * kstep + pc[c]), dst + c * 1024);
        load_row_lds(vs + (uint32_t)(r * vstep + pc[c]), dst + TILE + c * 1024);
      }
      return;
    }
    // pages that blocks straddle.  Every address first, then the loads: a load is a fence to the compiler, and a page
    // lookup behind each one would wait for LDS once per row
    int64_t row[LOADS];
#pragma unroll
    for (int c = 0; c < LOADS; ++c) {
      int key = (chunk0 + c) * RPI + lane / LPR;
      key = j * KB + (key < rows ? key : rows - 1);
      const int lp = key / (int)p.page, in_page = key - lp * (int)p.page;
      const int phys = p.table_lds ? table[lp] : phys_of(lp);
      row[c] = phys < 0 ? -1 : (((int64_t)phys * p.page + in_page) * p.Hkv + kvh) * D + pc[c];
    }
#pragma unroll
    for (int c = 0; c < LOADS; ++c) {
      const uint16_t* zero = reinterpret_cast<const uint16_t*>(pa_zero_row);
      load_row_lds(row[c] < 0 ? zero : p.kc + row[c], dst + c * 1024);
      load_row_lds(row[c] < 0 ? zero : p.vc + row[c], dst + TILE + c * 1024);
    }
  };
  issue(0, 0);

  // Q^T operand: lane = (query col, dimensions 16 step + 8 g .. + 8); rows past S read row S - 1
  uint4 qf[DSTEPS];
  if constexpr (!ROT) {
    const int qr = qpos < S ? qpos : S - 1;
    const uint16_t* src = p.q + (tok0 + qr) * p.q_stride + (int64_t)h * D + g * 8;
#pragma unroll
    for (int st = 0; st < DSTEPS; ++st) qf[st] = *reinterpret_cast<const uint4*>(src + st * 16);
  } else {
    // whole rows at a time, through the second buffer (nothing is requested into it before the first barrier) to the lanes that
    // take them.  (A lane reading its own query's pieces touches a line with every piece, of the rotary table too: 3.5 us of 25
    // at 8 x 512 x 16 heads of 128.)  Same bits as rope_kv_write_kernel's.
    constexpr int NQ = 32 / RPI;
    static_assert(QW * KW * 32 * ROWB <= BUF, "the queries fit a buffer");
    const int piece = lane % LPR;
    uint4 x[NQ];
    float4 fa[NQ], fb[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int r = qw0 + i * RPI + lane / LPR, qr = r < S ? r : S - 1;
      const float* cs = p.freqs + (int64_t)b * p.freqs_stride + (int64_t)qr * D + piece * 8;
      x[i] = *reinterpret_cast<const uint4*>(p.q + (tok0 + qr) * p.q_stride + (int64_t)h * D + piece * 8);
      fa[i] = *reinterpret_cast<const float4*>(cs);
      fb[i] = *reinterpret_cast<const float4*>(cs + 4);
    }
    uint8_t* const mine = pa_lds + BUF + wave * 32 * ROWB;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int row = i * RPI + lane / LPR;
      x[i] = rope8(x[i], fa[i], fb[i]);
      if (p.q_gain)  // uniform
        x[i] = chunk_normed(x[i], rms_scale(head_sumsq<D>(x[i]), (float)D, p.eps), *reinterpret_cast<const uint4*>(p.q_gain + piece * 8));
      *reinterpret_cast<uint4*>(mine + row * ROWB + ((piece ^ row_key<D>(row)) << 4)) = x[i];
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): other lanes' pieces are read next (the rows are this wavefront's own: no barrier)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int st = 0; st < DSTEPS; ++st)
      qf[st] = *reinterpret_cast<const uint4*>(mine + col * ROWB + (((2 * st + g) ^ row_key<D>(col)) << 4));
  }
  // fragment addresses inside a block: K row `col`, piece 2 step + g; V rows 4 g + i / 4 (and 8 further), i = lane % 16,
  // dimensions 16 (lane / 16 % 2) + 4 (i % 4) of a 32-dimension tile
  const int kfr = col * ROWB + ((g ^ row_key<D>(col)) << 4);  // ^ (2 step) << 4
  const int vrow = 4 * g + (lane & 15) / 4, vpiece = ((lane >> 4) & 1) * 2 + (lane & 3) / 2;
  const int vfr0 = vrow * ROWB + ((vpiece ^ row_key<D>(vrow)) << 4) + (lane & 1) * 8;  // ^ dt << 6
  const int vfr1 = (vrow + 8) * ROWB + ((vpiece ^ row_key<D>(vrow + 8)) << 4) + (lane & 1) * 8;

  // dimension tiles whose sums this wavefront keeps: all, or with KW > 1 its share (with fewer tiles than wavefronts the
  // last ones keep none)
  constexpr int DTW = DT > KW ? DT / KW : 1;
  const int dt0 = KW == 1 ? 0 : kw * DTW;
  const bool sums = KW == 1 || dt0 < DT;
  pa_f32x16 o[DTW];
#pragma unroll
  for (int dt = 0; dt < DTW; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
  float m = -INFINITY, l = 0.0f;  // running maximum of this lane's query; this lane's half of its denominator

  for (int it = 0; it < nit; ++it) {
    // block `it` has landed and everyone is done with the one before
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();
    if (it + 1 < nit) issue(it + 1, (it + 1) & 1);
    const int kb0 = (it * KW + kw) * KB;
    const bool ahead = kb0 > last_w;  // wavefront-uniform: every key of the block is ahead of every query here
    if (KW == 1 && ahead) continue;
    uint8_t* const buf = pa_lds + (it & 1) * BUF;
    const uint8_t* ks = buf + kw * 2 * TILE;
    pa_f32x16 s[NT];
    float bm = -INFINITY;
    if (!ahead) {
      // ---- scores, transposed: NT tiles of 32 keys
      // The K fragments are read two dimension steps ahead of the products that take them, and the tiles' accumulation
      // chains alternate: left to itself the compiler put every LDS read right in front of its MFMA (one LDS round trip
      // per product) and ran one tile's chain after the other's.
      {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
        constexpr int GRP = 4 / NT, NG = DSTEPS / GRP;
        uint4 fa[2][GRP][NT];
        auto ldk = [&](int buf, int st0) __attribute__((always_inline)) {
#pragma unroll
          for (int i = 0; i < GRP; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              fa[buf][i][t] = *reinterpret_cast<const uint4*>(ks + t * 32 * ROWB + (kfr ^ ((2 * (st0 + i)) << 4)));
        };
        ldk(0, 0);
        if (NG > 1) ldk(1, GRP);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
#pragma unroll
          for (int i = 0; i < GRP; ++i) {
            const pa_bf16x8 qv = __builtin_bit_cast(pa_bf16x8, qf[gi * GRP + i]);
#pragma unroll
            for (int t = 0; t < NT; ++t)
              s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(pa_bf16x8, fa[gi & 1][i][t]), qv, s[t], 0, 0, 0);
          }
          if (gi + 2 < NG) ldk(gi & 1, (gi + 2) * GRP);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      // ---- online softmax for this lane's query; register r of tile kt is key kb0 + 32 kt + 8 (r / 4) + 4 g + r % 4.
      // Scores stay unscaled; the scale (> 0) is applied to the maximum and inside the exponent's fma.
      const bool diag = kb0 + KB - 1 > qw0p;  // wavefront-uniform: some key of the block is ahead of some query
      if (diag) {  // a branch, not a compare and select per score in every block: most blocks lie wholly behind the queries
#pragma unroll
        for (int kt = 0; kt < NT; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (kb0 + kt * 32 + 8 * (r / 4) + 4 * g + (r % 4) > qposp) s[kt][r] = -INFINITY;
      }
#pragma unroll
      for (int kt = 0; kt < NT; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) bm = fmaxf(bm, s[kt][r]);
      const LanePair b2 = lanes32_pair(bm);
      bm = fmaxf(b2.x, b2.y) * p.scale_log2e;
    }
    // The running maximum only has to bound the exponents, not equal the true maximum: it is raised (and the
    // accumulators rescaled) only when some query of the wavefront would otherwise see an exponent above 2^8;
    // with probabilities up to 256 nothing overflows and bf16 keeps its relative precision.  After the first
    // block this is rare, and the rescale of the accumulators is skipped.
    float alpha[KW], mk = m;  // factor of the sums in front of each block, the maximum this wavefront's block works with
    bool raise[KW];           // wavefront-uniform
    if constexpr (KW > 1) {
      if (g == 0) maxima[kw][qw][col] = bm;
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      const float b = KW == 1 ? bm : maxima[k][qw][col];
      raise[k] = __builtin_amdgcn_ballot_w64(b > m + 8.0f) != 0;  // m = -inf in block 0: raised there
      alpha[k] = 1.0f;
      if (raise[k]) {
        const float mn = fmaxf(m, b);  // finite from block 0 on: key 0 is visible to every query
        alpha[k] = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
      }
      if (k == kw || KW == 1) mk = m;
    }
    uint4 pf[NT][2];  // P^T operands: tile kt, keys 16 s2 .. + 16
    float ps = 0.0f;
    if (!ahead) {
#pragma unroll
      for (int kt = 0; kt < NT; ++kt) {
        float pv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][r], p.scale_log2e, -mk));
          ps += pv[r];
        }
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
          pf[kt][s2] = make_uint4(pack_bf16x2(pv[8 * s2 + 0], pv[8 * s2 + 1]), pack_bf16x2(pv[8 * s2 + 2], pv[8 * s2 + 3]),
                                  pack_bf16x2(pv[8 * s2 + 4], pv[8 * s2 + 5]), pack_bf16x2(pv[8 * s2 + 6], pv[8 * s2 + 7]));
      }
      if constexpr (KW > 1) {  // over the block's keys, which everyone has read
        static_assert(QW * NT * 2048 <= TILE, "the probabilities fit the keys' place");
        uint4* dst = reinterpret_cast<uint4*>(buf + kw * 2 * TILE + qw * NT * 2048) + lane;
#pragma unroll
        for (int kt = 0; kt < NT; ++kt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) dst[(2 * kt + s2) * 64] = pf[kt][s2];
        psums[kw][qw][lane] = ps;
      }
    }
    if constexpr (KW > 1) __syncthreads();
    // ---- output, transposed: O^T[d, q] = alpha O^T + V^T P^T, block by block
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      if (KW > 1 && ((it * KW + k) * KB > last_w || !sums)) break;  // wavefront-uniform
      const uint8_t* vs = buf + k * 2 * TILE + TILE;
      if (raise[k]) {  // one branch for all tiles (a branch per tile kept the tiles' products apart)
        l *= alpha[k];
#pragma unroll
        for (int dt = 0; dt < DTW; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha[k];
      }
      if constexpr (KW > 1) {
        const uint4* src = reinterpret_cast<const uint4*>(buf + k * 2 * TILE + qw * NT * 2048) + lane;
#pragma unroll
        for (int kt = 0; kt < NT; ++kt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) pf[kt][s2] = src[(2 * kt + s2) * 64];
        ps = psums[k][qw][lane];
      }
      l += ps;
      // V^T fragments of all tiles, read before the products, whose chains alternate.  k slots of this lane group:
      // keys 32 kt + 16 s2 + {4 g .. + 4, 8 + 4 g .. + 4}, kk = 2 kt + s2.
      constexpr int KK = 2 * NT;
      pa_bf16x8 fv[DTW][KK];
#pragma unroll
      for (int dt = 0; dt < DTW; ++dt)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const uint8_t* at = vs + kk * 16 * ROWB;
          const pa_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)(at + (vfr0 ^ ((dt0 + dt) << 6))));
          const pa_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)(at + (vfr1 ^ ((dt0 + dt) << 6))));
          fv[dt][kk] = __builtin_bit_cast(pa_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d0 = 0; d0 < DTW; d0 += 2)
#pragma unroll
        for (int kk = 0; kk < KK; ++kk)
#pragma unroll
          for (int dt = d0; dt < (d0 + 2 < DTW ? d0 + 2 : DTW); ++dt)
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fv[dt][kk], __builtin_bit_cast(pa_bf16x8, pf[kk >> 1][kk & 1]), o[dt], 0, 0, 0);
    }
  }
  const LanePair l2 = lanes32_pair(l);
  l = l2.x + l2.y;
  // ---- normalise and store: register r of tile dt is dimension 32 dt + 8 (r / 4) + 4 g + r % 4 of query col
  if (qpos < S && sums) {
    const float inv = 1.0f / l;
    uint16_t* dst = p.out + ((tok0 + qpos) * p.Hq + h) * D + dt0 * 32 + 4 * g;
#pragma unroll
    for (int dt = 0; dt < DTW; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        uint2 w;
        w.x = pack_bf16x2(o[dt][4 * a + 0] * inv, o[dt][4 * a + 1] * inv);
        w.y = pack_bf16x2(o[dt][4 * a + 2] * inv, o[dt][4 * a + 3] * inv);
        *reinterpret_cast<uint2*>(dst + dt * 32 + 8 * a) = w;
      }
  }
}

constexpr int PA_TABLE_MAX = 2048;                         // page-table entries kept in LDS
constexpr int LDS_BYTES = 160 * 1024, STATIC_LDS = 1536;  // of a compute unit; of a workgroup beside its buffers, at most

template <int D, int QW, int KW, bool PAGED, bool ROT>
static int launch_prefill_attn(PrefillAttnArgs& a, hipStream_t st) {
  const int64_t wgs = ((int64_t)(a.S + 32 * QW - 1) / (32 * QW)) * a.Hq * a.B;
  a.wgs = (int)wgs;
  constexpr int KB = 64, BUFS = 2 * KW * 2 * KB * 2 * D;
  size_t lds = BUFS;
  if constexpr (PAGED) {
    const int64_t entries = ((int64_t)a.start + a.S + a.page - 1) / a.page;
    a.table_lds = a.page % KB != 0 && entries <= PA_TABLE_MAX ? (int)entries : 0;
    lds += (size_t)a.table_lds * sizeof(int);
  }
  constexpr auto kernel = prefill_attn_kernel<D, QW, KW, PAGED, ROT>;
  // Workgroups that the device holds at once.  Registers decide at head dimension 64 with one wavefront per query row (124
  // and 128 of them: four, where the buffers would allow five), the buffers elsewhere; a page table in LDS may cost another.
  // Launches of four to five workgroups per compute unit, numbered as if resident -> heaviest first, us: 4 x 1408 x 24 heads
  // 42.8 -> 41.2, 4 x 1536 46.0 -> 44.3, 1 x 6400 186 -> 164, 10 x 600 27.8 -> 26.3, 10 x 512 x 32 26.8 -> 25.9; 12 x 512 x 24
  // and 9 x 512 x 32 the other way, 23.7 -> 24.8 and 23.4 -> 24.6.
  static int cached[64] = {};
  int per_cu = per_device(cached, 1, [&](int* v, int) { return hipOccupancyMaxActiveBlocksPerMultiprocessor(v, kernel, QW * KW * 64, BUFS); });
  if (lds > BUFS && per_cu > LDS_BYTES / (int)(lds + STATIC_LDS)) per_cu = LDS_BYTES / (int)(lds + STATIC_LDS);
  const int64_t room = (int64_t)per_cu * device_cus();
  a.paired = wgs <= room;
  // No reading ahead without room beside the workgroups that attend: it would run behind them.  24-layer model, 1536 wide, ms,
  // room for two workgroups per compute unit in all kernels -> for as many as fit: 8 x 512 tokens 6.37 -> 6.10, 6 x 512
  // 5.23 -> 4.97, 5 x 512 4.64 -> 4.30, 9 x 384 5.49 -> 5.31; and no longer beside one that fills its compute unit: 1 x 300
  // 1.70 -> 1.67, 300 on 700 cached 1.83 -> 1.81, 2 x 128 1.53 -> 1.55.
  if (wgs + AHEAD_WGS > room) a.ahead_wgs = 0;
  aq::queue_kernel(kernel, dim3((unsigned)(wgs + a.ahead_wgs)), dim3(QW * KW * 64), lds, st, a);
  return (int)hipGetLastError();
}

// How many wavefronts take a query row's blocks side by side.  One (128 queries per workgroup) moves the fewest K and V
// bytes per query and is the faster form once the chip is full of such workgroups; with fewer, a launch lasts as long as
// its longest chain of blocks, which two or four wavefronts shorten, 64 or 32 queries per workgroup.  The buffers of two
// take 64 KiB at head dimension 64 (two workgroups per compute unit), 128 KiB at 128, those of four 128 KiB: they pay
// while the launch is resident at once, and up to twice that where the chain is long.  us, head dimension 64, 24 heads
// (1 | 2 | 4 wavefronts): 1 x 300 new tokens 7.3 | 6.8 | 6.0, 4 x 512 12.1 | 13.5 | 26, 1 x 2048 32 | 28 | 57, 64 on 1500
// cached 29 | 22 | 16, 500 on 1500 36 | 27 | 32; head dimension 128, 16 heads (1 | 2): 1 x 1000 23 | 18, 4 x 300
// 10.2 | 11.0, 64 on 1500 38 | 28.  Before, with keys staged through registers, one wavefront per query row and a page
// lookup per row: 7.7, 12.4, 34, 48, 61; 27.5, 11.8, 76.
template <int D, bool PAGED, bool ROT>
static int launch_prefill_attn(PrefillAttnArgs& a, hipStream_t st) {
  const int64_t heads = (int64_t)a.Hq * a.B, cus = device_cus(), T = (PAGED ? a.start : 0) + (int64_t)a.S;
  const int64_t q32 = (a.S + 31) / 32 * heads, q64 = (a.S + 63) / 64 * heads;
  if constexpr (D == 64) {
    if (q32 <= cus) return launch_prefill_attn<D, 1, 4, PAGED, ROT>(a, st);
  }
  if (T > 128 && q64 <= (D == 128 ? 1 : T < 1024 ? 2 : 4) * cus) return launch_prefill_attn<D, 2, 2, PAGED, ROT>(a, st);
  return launch_prefill_attn<D, 4, 1, PAGED, ROT>(a, st);
}

template <bool PAGED>
static int launch_prefill_attn(PrefillAttnArgs& a, int64_t D, hipStream_t st) {
  if (a.freqs) return D == 128 ? launch_prefill_attn<128, PAGED, true>(a, st) : launch_prefill_attn<64, PAGED, true>(a, st);
  return D == 128 ? launch_prefill_attn<128, PAGED, false>(a, st) : launch_prefill_attn<64, PAGED, false>(a, st);
}

}  // namespace aq

namespace {
struct Rotation {  // of the query heads as they are read; freqs null: they are rotated already
  const float* freqs = nullptr;
  int64_t freqs_stride = 0;
  const void* q_gain = nullptr;
  float eps = 0.0f;
};
int check_rotation(const Rotation& r, int64_t S, int64_t D) {
  if ((r.freqs_stride != 0 && r.freqs_stride < S * D) || (r.q_gain && !(r.eps >= 0.0f))) return AQ_E_SHAPE;
  return aq::check_ptr16(r.freqs) || (r.freqs_stride & 3) || aq::check_ptr16(r.q_gain) ? AQ_E_ALIGN : AQ_OK;
}
void set_rotation(aq::PrefillAttnArgs& a, const Rotation& r) {
  a.freqs = r.freqs;
  a.freqs_stride = r.freqs_stride;
  a.q_gain = static_cast<const uint16_t*>(r.q_gain);
  a.eps = r.eps;
}
}  // namespace

static int prefill_attn_causal(const void* q, int64_t q_stride, const Rotation& rot, const void* k, int64_t k_stride, const void* v,
                               int64_t v_stride, void* out, float scale, int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t D,
                               const aq_span* ahead, int n_ahead, void* stream) {
  if (D != 64 && D != 128) return AQ_E_SHAPE;
  if (B < 0 || S < 0 || Hq <= 0 || Hkv <= 0 || (Hq % Hkv) != 0 || !(scale > 0.0f)) return AQ_E_SHAPE;
  if (q_stride < Hq * D || k_stride < Hkv * D || v_stride < Hkv * D) return AQ_E_SHAPE;
  if (B == 0 || S == 0) return AQ_OK;
  if (!q || !k || !v || !out) return AQ_E_NULL;
  if (aq::check_ptr16(q) || aq::check_ptr16(k) || aq::check_ptr16(v) || aq::check_ptr16(out) || (q_stride & 7) ||
      (k_stride & 7) || (v_stride & 7))
    return AQ_E_ALIGN;
  if (S > (1 << 30) || Hq > 65535 || B > 65535 || ((S + 31) / 32) * Hq * B > (int64_t)0x7fffffff)
    return AQ_E_RANGE;
  // 32-bit byte offsets inside one sequence's K and V (a key block past the end included)
  if ((S + 64) * k_stride * 2 > (int64_t)0x7fffffff || (S + 64) * v_stride * 2 > (int64_t)0x7fffffff)
    return AQ_E_RANGE;
  if (const int rc = aq::check_spans(ahead, n_ahead)) return rc;
  if (const int rc = check_rotation(rot, S, D)) return rc;
  aq::PrefillAttnArgs a{};
  set_rotation(a, rot);
  a.ahead_wgs = aq::set_ahead(a.ahead, ahead, n_ahead);
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.out = static_cast<uint16_t*>(out);
  a.q_stride = q_stride;
  a.k_stride = k_stride;
  a.v_stride = v_stride;
  a.scale_log2e = scale * 1.44269504088896341f;
  a.S = (int)S;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.B = (int)B;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return aq::launch_prefill_attn<false>(a, D, st);
}

extern "C" int aq_prefill_attn_causal_ahead(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                            int64_t v_stride, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                            int64_t Hkv, int64_t D, const aq_span* ahead, int n_ahead, void* stream) {
  return prefill_attn_causal(q, q_stride, Rotation{}, k, k_stride, v, v_stride, out, scale, B, S, Hq, Hkv, D, ahead, n_ahead, stream);
}

extern "C" int aq_rope_prefill_attn_causal_ahead(const void* q, int64_t q_stride, const float* freqs, int64_t freqs_stride,
                                                 const void* q_gain, float eps, const void* k, int64_t k_stride, const void* v,
                                                 int64_t v_stride, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                                 int64_t Hkv, int64_t D, const aq_span* ahead, int n_ahead, void* stream) {
  if (!freqs && B > 0 && S > 0) return AQ_E_NULL;
  return prefill_attn_causal(q, q_stride, Rotation{freqs, freqs_stride, q_gain, eps}, k, k_stride, v, v_stride, out, scale, B, S, Hq,
                             Hkv, D, ahead, n_ahead, stream);
}

extern "C" int aq_prefill_attn_causal(const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v,
                                      int64_t v_stride, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                      int64_t Hkv, int64_t D, void* stream) {
  return aq_prefill_attn_causal_ahead(q, q_stride, k, k_stride, v, v_stride, out, scale, B, S, Hq, Hkv, D, nullptr, 0, stream);
}

static int prefill_attn_paged(const void* q, int64_t q_stride, const Rotation& rot, const void* k_cache, const void* v_cache,
                                     const int64_t* page_table, int64_t P, int64_t start, int64_t page_size,
                                     int64_t n_pages, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                     int64_t Hkv, int64_t D, const aq_span* ahead, int n_ahead, void* stream) {
  if (D != 64 && D != 128) return AQ_E_SHAPE;
  if (B < 0 || S < 0 || start < 0 || Hq <= 0 || Hkv <= 0 || (Hq % Hkv) != 0 || P <= 0 || page_size <= 0 ||
      n_pages <= 0 || !(scale > 0.0f) || q_stride < Hq * D)
    return AQ_E_SHAPE;
  if (start + S > P * page_size) return AQ_E_SHAPE;  // positions the page table does not cover
  if (B == 0 || S == 0) return AQ_OK;
  if (!q || !k_cache || !v_cache || !page_table || !out) return AQ_E_NULL;
  if (aq::check_ptr16(q) || aq::check_ptr16(k_cache) || aq::check_ptr16(v_cache) || aq::check_ptr16(out) ||
      (q_stride & 7))
    return AQ_E_ALIGN;
  if (start + S > (1 << 30) || Hq > 65535 || B > 65535 ||
      ((S + 31) / 32) * Hq * B > (int64_t)0x7fffffff)
    return AQ_E_RANGE;
  if (const int rc = aq::check_spans(ahead, n_ahead)) return rc;
  if (const int rc = check_rotation(rot, S, D)) return rc;
  aq::PrefillAttnArgs a{};
  set_rotation(a, rot);
  a.ahead_wgs = aq::set_ahead(a.ahead, ahead, n_ahead);
  a.q = static_cast<const uint16_t*>(q);
  a.out = static_cast<uint16_t*>(out);
  a.q_stride = q_stride;
  a.kc = static_cast<const uint16_t*>(k_cache);
  a.vc = static_cast<const uint16_t*>(v_cache);
  a.table = page_table;
  a.P = P;
  a.page = page_size;
  a.n_pages = n_pages;
  a.start = (int)start;
  a.page_shift = -1;
  for (int sh = 0; sh < 31; ++sh)
    if (page_size == ((int64_t)1 << sh)) a.page_shift = sh;
  a.scale_log2e = scale * 1.44269504088896341f;
  a.S = (int)S;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.B = (int)B;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return aq::launch_prefill_attn<true>(a, D, st);
}

extern "C" int aq_prefill_attn_paged_ahead(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                                           const int64_t* page_table, int64_t P, int64_t start, int64_t page_size,
                                           int64_t n_pages, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                           int64_t Hkv, int64_t D, const aq_span* ahead, int n_ahead, void* stream) {
  return prefill_attn_paged(q, q_stride, Rotation{}, k_cache, v_cache, page_table, P, start, page_size, n_pages, out, scale, B, S, Hq,
                            Hkv, D, ahead, n_ahead, stream);
}

extern "C" int aq_rope_prefill_attn_paged_ahead(const void* q, int64_t q_stride, const float* freqs, int64_t freqs_stride,
                                                const void* q_gain, float eps, const void* k_cache, const void* v_cache,
                                                const int64_t* page_table, int64_t P, int64_t start, int64_t page_size,
                                                int64_t n_pages, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                                int64_t Hkv, int64_t D, const aq_span* ahead, int n_ahead, void* stream) {
  if (!freqs && B > 0 && S > 0) return AQ_E_NULL;
  return prefill_attn_paged(q, q_stride, Rotation{freqs, freqs_stride, q_gain, eps}, k_cache, v_cache, page_table, P, start, page_size,
                            n_pages, out, scale, B, S, Hq, Hkv, D, ahead, n_ahead, stream);
}

extern "C" int aq_prefill_attn_paged(const void* q, int64_t q_stride, const void* k_cache, const void* v_cache,
                                     const int64_t* page_table, int64_t P, int64_t start, int64_t page_size,
                                     int64_t n_pages, void* out, float scale, int64_t B, int64_t S, int64_t Hq,
                                     int64_t Hkv, int64_t D, void* stream) {
  return aq_prefill_attn_paged_ahead(q, q_stride, k_cache, v_cache, page_table, P, start, page_size, n_pages, out, scale, B, S, Hq,
                                     Hkv, D, nullptr, 0, stream);
}
