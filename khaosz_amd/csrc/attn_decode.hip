// Attention around the quantized projections, on the paged KV cache in place:
// the reference rotates q and k with complex multiplies, writes k/v page by
// page, gathers every page into a contiguous [B, T, Hkv, D] copy, repeats the
// KV heads and calls a generic attention, per layer and per step
// (astrai/model/components/attention.py:83-103,
// astrai/inference/core/cache.py:216-274).  Kernels here:
//
//   rope_kv_write   rotates q and k of the new tokens (interleaved pairs, fp32,
//                   rope.py:26-33), stores q, and writes k and v into their page
//                   slots (cache.py:216-252) -- one token per sequence at decode,
//                   the whole prompt at prefill;
//   paged_attn      softmax(q K^T / sqrt(D)) V for one query token per sequence
//                   over the pages of that sequence, all query heads of a KV
//                   head in one workgroup (grouped-query attention without
//                   materialising the repeated heads, attention.py:15-23);
//                   optionally doing rope_kv_write's work for that token itself.
//
// bf16 tensors, head dimension 64 or 128, fp32 arithmetic.  Unmapped pages
// (table entry < 0 or out of range) are skipped on write and read as zero keys
// and values, as the reference's gather does.
#include "aq_common.h"
#include "aq_rope.h"
#include "aq_rows.h"

namespace aq {

struct RopeArgs {
  const uint16_t* qkv;   // [B, S, (Hq + 2 Hkv) * D]
  const float* freqs;    // [S, D/2, 2] (cos, sin) per sequence; sequences freqs_stride floats apart (0: shared)
  int64_t freqs_stride;
  const int64_t* table;  // [B, P]
  uint16_t* kc;          // [n_pages, page, Hkv, D]
  uint16_t* vc;
  uint16_t* q_out;       // [B, S, Hq, D], or null: the query heads are left alone
  uint16_t* k_out;       // [B, S, Hkv, D] rotated keys, or null
  int64_t P, pos, page, n_pages, S;
  int B, Hq, Hkv, D;
  const uint16_t* q_gain;  // [D] RMSNorm gains of the rotated q / k heads, or null: no qk-norm
  const uint16_t* k_gain;
  float eps;
};

// One thread per 16-byte chunk (8 elements) of a head vector of a token.  Without q_out the query heads are left to whoever reads
// them (the prefill attention rotates its own): 4096 tokens of 16 + 2 x 4 heads of 128 move 21 MB instead of 50, and the launch, at
// the rate of a copy either way, takes 6.2 us instead of 11.3 (attention 0.2 to 0.8 more; 2048 tokens of 24 + 2 x 4 heads of 64:
// 4.6 -> 2.8, attention 0.8 more).
__global__ __launch_bounds__(256) void rope_kv_write_kernel(RopeArgs p) {
  const int h0 = p.q_out ? 0 : p.Hq;
  const int64_t heads = p.Hq + 2 * p.Hkv - h0;
  const int cph = p.D / 8;  // chunks per head vector
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= (int64_t)p.B * p.S * heads * cph) return;
  const int ch = (int)(c % cph);
  const int64_t hv = c / cph, tokn = hv / heads;
  const int h = (int)(hv % heads) + h0;
  const int64_t b = tokn / p.S, s = tokn % p.S;
  uint4 x = *reinterpret_cast<const uint4*>(p.qkv + (tokn * (p.Hq + 2 * p.Hkv) + h) * p.D + ch * 8);
  if (h < p.Hq + p.Hkv) x = rope8(x, p.freqs + b * p.freqs_stride + s * p.D + ch * 8);  // v heads do not rotate
  if (p.q_gain) {  // uniform: qk-norm
    const float ss = p.D == 128 ? head_sumsq<128>(x) : head_sumsq<64>(x);
    if (h < p.Hq + p.Hkv) {
      const uint16_t* gain = h < p.Hq ? p.q_gain : p.k_gain;
      x = chunk_normed(x, rms_scale(ss, (float)p.D, p.eps), *reinterpret_cast<const uint4*>(gain + ch * 8));
    }
  }
  if (h < p.Hq) {
    *reinterpret_cast<uint4*>(p.q_out + (tokn * p.Hq + h) * p.D + ch * 8) = x;
    return;
  }
  const bool is_k = h < p.Hq + p.Hkv;
  const int kvh = is_k ? h - p.Hq : h - p.Hq - p.Hkv;
  if (is_k && p.k_out) *reinterpret_cast<uint4*>(p.k_out + (tokn * p.Hkv + kvh) * p.D + ch * 8) = x;
  const int64_t pos = p.pos + s, lp = pos / p.page;
  const int64_t phys = lp < p.P ? p.table[b * p.P + lp] : -1;
  if (phys < 0 || phys >= p.n_pages) return;  // unmapped: the token is dropped, as in the reference
  uint16_t* dst = (is_k ? p.kc : p.vc) + ((phys * p.page + pos % p.page) * p.Hkv + kvh) * p.D + ch * 8;
  *reinterpret_cast<uint4*>(dst) = x;
}

struct AttnArgs {
  const uint16_t* q;     // [B, Hq, D]
  const uint16_t* kc;    // [n_pages, page, Hkv, D]
  const uint16_t* vc;
  const int64_t* table;  // [B, P]
  const int64_t* lens;   // [B] positions each sequence may attend to (its own length), or null: all T
  uint16_t* out;         // [B, Hq, D]
  float* ws;             // partial results [B, Hq, NS, D + 4] when NS > 1
  const uint16_t* qkv;   // ROPE kernels: [B, (Hq + 2 Hkv) * D] projections of the new token (position T - 1)
  const float* freqs;    // ROPE kernels: its rotary table, as in RopeArgs
  uint16_t* kc_w;        // ROPE kernels: the caches again, writable
  uint16_t* vc_w;
  int64_t freqs_stride;
  int64_t P, T, page, n_pages;
  float scale_log2e;     // softmax scale times log2(e): scores live in the exp2 domain
  int B, Hq, Hkv, NS;
  const uint16_t* q_gain;  // QKN kernels: [D] RMSNorm gains of the rotated q / k heads
  const uint16_t* k_gain;
  float eps;
  int page_shift;  // log2 of a page of 64, 128, 256 .. positions, otherwise 62
  const int64_t* lens_at;  // lens, or without them anything of B numbers (the table): read without asking, beside the table
  UDiv by_hkv, by_ns, by_page;  // by_page: pages of other sizes, of launches whose positions it takes (mul 0: a division)
};

constexpr int ATT_WAVES = 4;
constexpr int ATT_KPW = 64;                  // positions per wavefront
constexpr int ATT_KPG = ATT_WAVES * ATT_KPW; // positions per workgroup
constexpr int ATT_MAX_D = 128;
constexpr float ATT_MASKED = -1.0e30f;  // score (exp2 domain) of a cached position the sequence may not attend to

// maximum / sum over each row of 16 consecutive lanes, result in all of them
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false)));   // quad_perm [1,0,3,2]
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false)));   // quad_perm [2,3,0,1]
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false)));  // row_half_mirror
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false)));  // row_mirror
  return v;
}
__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));
  return v;
}

typedef __bf16 attn_bf16x8 __attribute__((ext_vector_type(8)));
typedef float attn_f32x4 __attribute__((ext_vector_type(4)));

// Workgroup = one (sequence, KV head, slice of the cached positions): the G
// query heads of the KV head share every K and V byte.  A wavefront owns 64
// consecutive positions, a workgroup 256; the NS slices of a sequence run as
// separate workgroups so that a decode batch of a few sequences still spreads
// over the device.  Every K and V load of a wavefront, 16 bytes per lane, is
// requested before anything is computed.
//   scores   on the matrix core: S[key, head] = K Q^T as v_mfma_f32_16x16x32_bf16
//            tiles, the G <= 8 query heads padded to 16 columns, four tiles of 16
//            keys, D / 32 steps each.  K rows are loaded straight in operand
//            order (lane l: key l % 16 of the tile, dimensions 8 (l / 16) .. + 8
//            of the step), queries likewise; a lane ends up with the scores of
//            one head for 4 keys per tile;
//   softmax  maximum and denominator over a lane's 16 keys in registers and over
//            the 4 lanes of a head by row swaps (with heads in registers and keys
//            in lanes, as one or two heads are, every head takes four DPP steps,
//            twice); probabilities to LDS;
//   values   V rows are loaded CPR = D / 8 lanes to a row (a load covers 4 or 8
//            whole rows); a lane accumulates p * V over the keys it loaded (8
//            dimensions x G heads), the key groups are summed by swaps.
// A launch of few sequences is one wavefront's chain of latencies, most of it
// between the lookup of its pages and its sums (8 x 544 positions, 16/4 heads of
// 128: 6.9 us from a graph, 4 x 576, 24/4 heads of 64: 5.3; 8.1 and 6.3 with a
// row lookup per load, heads in registers and all sums by fused multiply-add).
// The wavefronts' (maximum, denominator, numerator) are merged through LDS and
// either normalised into the output (NS == 1) or left in the workspace for
// attn_merge_kernel.
// ROPE: the kernel also does rope_kv_write_kernel's work for the new token at
// position T - 1 -- every workgroup rotates its own queries from the raw
// projection, and the one wavefront whose positions include T - 1 rotates the
// new key, stores it and the new value into their page slot and uses them from
// registers instead of what it read from the cache.  Same roundings, so caches
// and outputs are the bits the two separate launches give.
// QKN (with ROPE): the rotated queries and the rotated new key are RMS-normalised over the head dimension (see
// chunk_sumsq) before they are used and stored: what rope_kv_write_kernel does with gains, same bits.  A head
// vector's chunk c = 4 ks + kq sits in register ks of the lane with that kq.
// WHOLE: pages of 64, 128, 256 .. positions: a wavefront's rows lie in one page.
template <int G, int D, bool WHOLE, bool ROPE, bool QKN = false>
__global__ __launch_bounds__(ATT_WAVES * 64) void paged_attn_decode_kernel(AttnArgs p) {
  static_assert(!QKN || ROPE, "qk-norm belongs to the kernels that rotate");
  constexpr int CPR = D / 8;     // 16-byte chunks per row: 16 or 8
  constexpr int RPL = 64 / CPR;  // rows per load instruction: 4 or 8
  constexpr int NL = 64 / RPL;   // loads per wavefront (= CPR)
  constexpr int KPW = ATT_KPW, KPG = ATT_KPG;
  constexpr int ATT_THREADS = ATT_WAVES * 64;
  constexpr int PART = D + 4;    // numerator[D], maximum, denominator, 2 floats of padding
  static_assert(D == 64 || D == 128, "head dimension");
  constexpr int NM = (G + 1) / 4, GV = G > 4 * NM ? G - 4 * NM : 0;  // groups of 4 heads on the matrix core; heads past them (1, 2)
  constexpr bool FEW = G <= 2;
  constexpr int GP = 4 * NM + GV, PS = KPW + 16;                    // (rows of 80: 4 heads x 16 keys in 64 banks, both ways)
  __shared__ __align__(16) float p_s[ATT_WAVES][GP][PS];
  __shared__ float m_s[ATT_WAVES][G], l_s[ATT_WAVES][G];
  __shared__ __align__(16) float acc_s[ATT_WAVES][G][D];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = lane / CPR, ch = lane % CPR;  // key within a load, 16-byte chunk of the row
  // the KV heads of one slice are neighbours in the launch order: together they read whole
  // [position][Hkv][D] stretches of the pages at about the same time
  const int bs = p.by_hkv(blockIdx.x), kvh = blockIdx.x - bs * p.Hkv;
  const int b = p.by_ns(bs), split = bs - b * p.NS;
  const int64_t T = p.T;
  const int64_t t0 = (int64_t)split * KPG + wave * KPW;  // first position of this wavefront
  // Where the rows are.  WHOLE: one lookup, and every load's address is that plus the lane's own offset.  The table's entry
  // (otherwise its first, not used) and the sequence's length are requested before anything else and first used behind the
  // queries' requests (8 x 544 positions, 16/4 heads of 128: 9.46 us; 9.60 with divisions by the numbers of heads and slices, a
  // wait for the length and the lookup behind them).  Other pages: lane L looks up the page of position t0 + L, as early.  Kernels
  // of their own: with both ways in one, their loads became one stretch behind the addresses of all of them (pages of 64 and more,
  // 16/4 heads of 128 and 24/4 of 64: 4 % longer; pages of 16: 10 x 786 positions of 16/4 9.37 us, 8.91 so, 14 x 647 of 24/4 8.48, 7.93).
  const int64_t lp0 = WHOLE ? t0 >> p.page_shift : 0;
  int64_t entry = 0, phys = -1, in_page = 0, len = p.lens_at[b];
  if constexpr (WHOLE) {
    entry = p.table[(int64_t)b * p.P + (lp0 < p.P ? lp0 : p.P - 1)];
    asm volatile("" ::"s"(p.T), "s"(p.page), "s"(p.n_pages), "s"(p.lens), "s"(p.kc), "s"(p.vc));  // arguments: one request for all
  } else if (t0 + lane < T) {
    const int64_t t = t0 + lane, lp = p.by_page.mul ? (int64_t)p.by_page((uint32_t)t) : t / p.page;
    in_page = t - lp * p.page;
    if (lp < p.P) phys = p.table[(int64_t)b * p.P + lp];
  }
  __builtin_amdgcn_sched_barrier(0);

  constexpr int KS = D / 32;                  // matrix-core steps over the head dimension
  const int col = lane & 15, kq = lane >> 4;  // operand row / column, group of 8 dimensions inside a step
  // The queries (and their rotary table values) do not depend on the page table: requested first, used after
  // the K and V loads have been issued, so that the wavefront waits for one memory round trip less.  (Wavefronts past T request
  // them too: a branch here would end the stretch in which the scalar requests go out together.)
  uint4 qraw[KS];
  float4 fa[KS], fb[KS];
  const int hq = col < G ? col : 0;  // heads past G: zero rows of the operand (their loads read head 0)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 32 + kq * 8;
    if constexpr (ROPE) {
      qraw[ks] = *reinterpret_cast<const uint4*>(p.qkv + ((int64_t)b * (p.Hq + 2 * p.Hkv) + kvh * G + hq) * D + d0);
      const float* cs = p.freqs + (int64_t)b * p.freqs_stride + d0;
      fa[ks] = *reinterpret_cast<const float4*>(cs);
      fb[ks] = *reinterpret_cast<const float4*>(cs + 4);
    } else {
      qraw[ks] = *reinterpret_cast<const uint4*>(p.q + ((int64_t)b * p.Hq + kvh * G + hq) * D + d0);
    }
  }
  // RMSNorm of a rotated head vector held as KS chunks per lane (chunk 4 ks + kq), gains requested by the caller
  auto head_norm = [&](uint4 (&v)[KS], const uint4 (&gain)[KS]) {
    float ss[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ss[ks] = chunk_sumsq(v[ks]);
      const LanePair c1 = lanes16_pair(ss[ks]);                  // c ^ 1
      const LanePair c2 = lanes32_pair(__fadd_rn(c1.x, c1.y));  // c ^ 2
      ss[ks] = __fadd_rn(c2.x, c2.y);
    }
    float tot = __fadd_rn(ss[0], ss[1]);                            // c ^ 4
    if constexpr (KS == 4) tot = __fadd_rn(tot, __fadd_rn(ss[2], ss[3]));  // c ^ 8
    const float r = rms_scale(tot, (float)D, p.eps);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) v[ks] = chunk_normed(v[ks], r, gain[ks]);
  };
  uint4 qgain[KS], kgain[KS];
  if constexpr (QKN) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      qgain[ks] = *reinterpret_cast<const uint4*>(p.q_gain + ks * 32 + kq * 8);
      kgain[ks] = *reinterpret_cast<const uint4*>(p.k_gain + ks * 32 + kq * 8);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (WHOLE) asm volatile("" : "+s"(entry), "+s"(len));  // not requested later than above
  // (element offsets, -1: unmapped or past T; row: of lane L, of position t0 + L)
  const int rstep = p.Hkv * D;  // elements between consecutive positions of a page
  int64_t first = -1, row = -1;
  if constexpr (WHOLE) {
    if (t0 < T && lp0 < p.P && entry >= 0 && entry < p.n_pages)
      first = (((entry << p.page_shift) + (t0 - (lp0 << p.page_shift))) * p.Hkv + kvh) * D;
  } else if (phys >= 0 && phys < p.n_pages) {
    row = ((phys * p.page + in_page) * p.Hkv + kvh) * D;
  }
  // A sequence shorter than T (a decode batch of sequences at different positions): positions from its own
  // length on are masked, as the additive mask of the reference's forward does.  The mask value is finite, so
  // a wavefront or slice whose positions are all masked leaves a partial result that later merges weigh with 0.
  const int64_t vis = p.lens && len < T ? (len > 0 ? len : 0) : T;
  // Positions that are all masked weigh nothing in the merges: their keys and values are not read (model step of 11 sequences
  // spread over 1400 positions: 941 -> 922 us).  Not so where every position is masked, and the new token's wavefront
  // has it to store.  Asked only here, so that nothing above waits for the length.
  const bool masked = t0 >= vis && vis > 0 && !(ROPE && T - 1 < t0 + KPW);
  if (t0 < T && !masked) {  // wavefront-uniform
    auto row_of = [&](int src) -> int64_t {
      const int lo = __shfl((int)(uint32_t)row, src, 64), hi = __shfl((int)(row >> 32), src, 64);
      return ((int64_t)hi << 32) | (uint32_t)lo;
    };
    const bool has_new = ROPE && T - 1 >= t0 && T - 1 < t0 + KPW;  // wavefront-uniform
    // ---- operands of the scores
    // keys: tile t holds positions t0 + 16 t .. + 16; lane = (key col, dimensions ks * 32 + kq * 8 .. + 8).
    // values: lane = (key sub of a load, 16-byte chunk ch of the row).  Rows that are unmapped or past T read
    // row 0 of the cache and are zeroed afterwards.  Every load is issued before any loaded value is touched
    // (the fix-ups below are selects on data, kept out of the issue loops: with them inside, the compiler
    // waited for each load before issuing the next).
    uint4 kb[4][KS], vv[NL];
    uint64_t there;  // bit per position: its row is there
    if constexpr (WHOLE) {
      // (20 lookups by shuffle, with 64-bit arithmetic each, took 0.3 us of the launch at head dimension 64, and 0.1 to 0.2 at 128, where
      // 32 loads of 1 KiB wait for each other to be taken)
      const uint16_t *ks0 = p.kc + (first >= 0 ? first : 0) + (uint32_t)(col * rstep + kq * 8);
      const uint16_t *vs0 = p.vc + (first >= 0 ? first : 0) + (uint32_t)(sub * rstep + ch * 8);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kb[t][ks] = *reinterpret_cast<const uint4*>(ks0 + t * 16 * rstep + ks * 32);
#pragma unroll
      for (int i = 0; i < NL; ++i) vv[i] = *reinterpret_cast<const uint4*>(vs0 + i * RPL * rstep);
      there = first < 0 ? 0 : ~0ull >> (t0 + KPW > T ? (int)(t0 + KPW - T) : 0);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int64_t r = row_of(t * 16 + col);
        const uint16_t* src = p.kc + (r >= 0 ? r : 0) + kq * 8;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) kb[t][ks] = *reinterpret_cast<const uint4*>(src + ks * 32);
      }
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int64_t r = row_of(i * RPL + sub);
        vv[i] = *reinterpret_cast<const uint4*>(p.vc + (r >= 0 ? r : 0) + ch * 8);
      }
      there = __builtin_amdgcn_ballot_w64(row >= 0);
    }
    __builtin_amdgcn_sched_barrier(0);  // nothing that waits for a load may move above the last load's issue
    if (there != ~0ull) {  // wavefront-uniform; rare: a hole, or the wavefront that holds T - 1
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          if (!(there >> (t * 16 + col) & 1)) kb[t][ks] = make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < NL; ++i)
        if (!(there >> (i * RPL + sub) & 1)) vv[i] = make_uint4(0, 0, 0, 0);
    }
    if (ROPE && has_new) {  // wavefront-uniform: this wavefront owns position T - 1
      // the new key and value: rotated here, stored into their page slot, and used from registers in place
      // of what was just read from that slot
      const uint16_t* tok = p.qkv + (int64_t)b * (p.Hq + 2 * p.Hkv) * D;
      // the same in every lane; -1: its page is unmapped
      const int64_t rn = !WHOLE ? row_of((int)(T - 1 - t0)) : first < 0 ? -1 : first + (T - 1 - t0) * rstep;
      if (rn >= 0) {
        const int tn = (int)(T - 1 - t0) >> 4, cn = (int)(T - 1 - t0) & 15;  // tile and column of the new key
        uint4 kn[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          kn[ks] = rope8(*reinterpret_cast<const uint4*>(tok + (int64_t)(p.Hq + kvh) * D + ks * 32 + kq * 8), fa[ks], fb[ks]);
        if constexpr (QKN) head_norm(kn, kgain);  // (every column holds the same new key: all lanes take part)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int d0 = ks * 32 + kq * 8;
          if (col == cn) *reinterpret_cast<uint4*>(p.kc_w + rn + d0) = kn[ks];
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (t == tn && col == cn) kb[t][ks] = kn[ks];
        }
        const uint4 vn = *reinterpret_cast<const uint4*>(tok + (int64_t)(p.Hq + p.Hkv + kvh) * D + ch * 8);
        const int in = (int)(T - 1 - t0) / RPL, sn = (int)(T - 1 - t0) % RPL;  // load and key group of the new value
        if (sub == sn) *reinterpret_cast<uint4*>(p.vc_w + rn + ch * 8) = vn;
#pragma unroll
        for (int i = 0; i < NL; ++i)
          if (i == in && sub == sn) vv[i] = vn;
      }
    }
    // queries: lane = (head col, dimensions ks * 32 + kq * 8 .. + 8)
    uint4 qa[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (ROPE)
        qa[ks] = rope8(qraw[ks], fa[ks], fb[ks]);
      else
        qa[ks] = qraw[ks];
    }
    if constexpr (QKN) head_norm(qa, qgain);  // (columns past G normalise a copy of head 0 and are zeroed below)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (col >= G) qa[ks] = make_uint4(0, 0, 0, 0);
    }
    // ---- scores and softmax over the wavefront's 64 positions.  One or two heads: S[head][key] per tile, this lane gets key col,
    // heads 4 kq .. + 4 (kq = 0 holds the heads there are): 4 exponentials per head, where a lane with a head of its own takes 16
    // (11 x 479 positions, 8/8 heads of 64: 7.26 us, 6.90 so; 1 x 356, 4/2 of 128: 7.85, 7.58; with three heads level).
    attn_f32x4 sc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      attn_f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const attn_bf16x8 k8 = __builtin_bit_cast(attn_bf16x8, kb[t][ks]), q8 = __builtin_bit_cast(attn_bf16x8, qa[ks]);
        c = FEW ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(q8, k8, c, 0, 0, 0) : __builtin_amdgcn_mfma_f32_16x16x32_bf16(k8, q8, c, 0, 0, 0);
      }
      sc[t] = c;
    }
    const int n_all = T - t0 < KPW ? (int)(T - t0) : KPW, n_vis = vis - t0 < n_all ? (vis > t0 ? (int)(vis - t0) : 0) : n_all;
    if constexpr (FEW) {
#pragma unroll
      for (int r = 0; r < G; ++r) {
        float pv[4], mx = -INFINITY, sum = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int key = t * 16 + col;
          pv[t] = key < n_vis ? sc[t][r] * p.scale_log2e : key < n_all ? ATT_MASKED : -INFINITY;
          mx = fmaxf(mx, pv[t]);
        }
        mx = row16_max(mx);  // finite: position t0 is valid
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          pv[t] = __builtin_amdgcn_exp2f(pv[t] - mx);  // 0 for positions past T
          sum += pv[t];
          if (kq == 0) p_s[wave][r][t * 16 + col] = pv[t];
        }
        sum = row16_sum(sum);
        if (lane == 0) {
          m_s[wave][r] = mx;
          l_s[wave][r] = sum;
        }
      }
    } else {
      // S[key][head]: this lane gets head col, keys 4 kq .. + 4 of the tile: 16 positions of it, the others 16 and 32 lanes away
      float pv[4][4], mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) pv[t][r] = sc[t][r] * p.scale_log2e;
      if (n_vis < KPW) {  // wavefront-uniform
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = t * 16 + 4 * kq + r;
            pv[t][r] = key < n_vis ? pv[t][r] : key < n_all ? ATT_MASKED : -INFINITY;
          }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, pv[t][r]);
      const LanePair m16 = lanes16_pair(mx);
      const LanePair m32 = lanes32_pair(fmaxf(m16.x, m16.y));
      mx = fmaxf(m32.x, m32.y);  // finite: position t0 is valid
      float part[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        part[r] = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          pv[t][r] = __builtin_amdgcn_exp2f(pv[t][r] - mx);  // 0 for positions past T
          part[r] += pv[t][r];
        }
      }
      const LanePair s16 = lanes16_pair((part[0] + part[1]) + (part[2] + part[3]));
      const LanePair s32 = lanes32_pair(s16.x + s16.y);
      const float sum = s32.x + s32.y;
      if (col < GP) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          *reinterpret_cast<float4*>(&p_s[wave][col][t * 16 + 4 * kq]) = make_float4(pv[t][0], pv[t][1], pv[t][2], pv[t][3]);
        if (kq == 0 && col < G) {
          m_s[wave][col] = mx;
          l_s[wave][col] = sum;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // this wavefront's LDS writes are done (wavefront-private region)
    asm volatile("" ::: "memory");
    // ---- numerator (unmapped rows and positions past T contribute zeros)
    // Four heads at a time as outer products on the matrix core, 16 of 4 heads x 4 lanes: a lane's element of V times its key's
    // probability of each head, added to the lane's own four sums with one rounding: the bits of the fused multiply-add that the
    // heads past them take (also for infinities and denormals), in the same order.  A product took 10 clocks where four
    // fused multiply-adds take 16 (launch of 8 x 544 positions at head dimension 128, 4 heads: 9.97 -> 9.55 us; 4 x 576, 64, 6 heads:
    // 7.13 -> 6.97), and one register holds the probabilities of PER loads, each broadcast to the lanes of its keys.
    constexpr int PER = CPR / 4, CB = PER == 4 ? 2 : 1;               // blocks of 4 lanes that share a key
    attn_f32x4 accm[NM > 0 ? NM : 1][8];
    float acc[GV > 0 ? GV : 1][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
      for (int m = 0; m < NM; ++m) accm[m][e] = attn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int g = 0; g < GV; ++g) acc[g][e] = 0.0f;
    }
    float pm[NM > 0 ? NM : 1][NL / PER];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int i = 0; i < NL / PER; ++i)
        pm[m][i] = p_s[wave][4 * m + (lane & 3)][(i * PER + ((lane >> 2) & (PER - 1))) * RPL + sub];
    auto outer = [&](float pj, float v, attn_f32x4 c, int step) {  // the block is an immediate
      switch (step) {
        case 0: return __builtin_amdgcn_mfma_f32_4x4x1f32(pj, v, c, CB, 0, 0);
        case 1: return __builtin_amdgcn_mfma_f32_4x4x1f32(pj, v, c, CB, 1, 0);
        case 2: return __builtin_amdgcn_mfma_f32_4x4x1f32(pj, v, c, CB, 2, 0);
        default: return __builtin_amdgcn_mfma_f32_4x4x1f32(pj, v, c, CB, 3, 0);
      }
    };
    auto widened = [&](int i, int e) {  // element e of load i
      const uint32_t w = e < 2 ? vv[i].x : e < 4 ? vv[i].y : e < 6 ? vv[i].z : vv[i].w;
      return __uint_as_float(e & 1 ? w & 0xffff0000u : w << 16);
    };
    // The next load's values are widened before this one's products, which stay together: a product waits two slots for a
    // register written just before it, and 11 clocks after any other vector instruction (products and widening in turn: 9.84 us).
    float v8[2][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v8[0][e] = widened(0, e);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      float pg[GV > 0 ? GV : 1];
#pragma unroll
      for (int g = 0; g < GV; ++g) pg[g] = p_s[wave][4 * NM + g][i * RPL + sub];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (i + 1 < NL) v8[(i + 1) & 1][e] = widened(i + 1, e);
#pragma unroll
        for (int g = 0; g < GV; ++g) acc[g][e] = __builtin_fmaf(pg[g], v8[i & 1][e], acc[g][e]);
      }
      if constexpr (NM > 0) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e) accm[m][e] = outer(pm[m][i / PER], v8[i & 1][e], accm[m][e], i % PER);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // Sum over the RPL key groups (lanes CPR apart) with a transposed butterfly: at each stage a lane keeps
    // one half of its values and trades the other half with its partner, so the 8 G values per lane cost
    // 8 G (1 - 1 / RPL) exchanges instead of 8 G log2(RPL), and a lane ends up with 8 G / RPL finished sums.
    {
      constexpr int NV = 8 * G;
      float a[NV];
#pragma unroll
      for (int j = 0; j < NV; ++j) a[j] = j / 8 < 4 * NM ? accm[j / 32][j % 8][j / 8 % 4] : acc[j / 8 - 4 * NM][j % 8];
      int base = 0;  // first original index of the values this lane still holds
#pragma unroll
      for (int st = 0; (CPR << st) < 64; ++st) {
        const int off = CPR << st, h = NV >> (st + 1);
        const bool up = (lane & off) != 0;
#pragma unroll
        for (int i = 0; i < h; ++i) {
          if (off == 32 || off == 16) {
            // half / row swaps: lanes without the bit receive the partner's a[i], lanes with it the partner's
            // a[i + h], next to their own; one add finishes the exchange
            typedef unsigned att_u2 __attribute__((ext_vector_type(2)));
            const att_u2 r = off == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a[i]), __float_as_uint(a[i + h]), false, false)
                                       : __builtin_amdgcn_permlane16_swap(__float_as_uint(a[i]), __float_as_uint(a[i + h]), false, false);
            a[i] = __uint_as_float(r.x) + __uint_as_float(r.y);
          } else {
            // 8 lanes away inside rows of 16 (head dimension 64): both halves' sums, then this lane's one
            const float lo = a[i] + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a[i]), 0x128, 0xf, 0xf, false));
            const float hi = a[i + h] + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a[i + h]), 0x128, 0xf, 0xf, false));
            a[i] = up ? hi : lo;
          }
        }
        base += up ? h : 0;
      }
      asm volatile("" : "+v"(base));  // one address computation below, not a code path per value of base
      float* dst = &acc_s[wave][0][ch * 8];
#pragma unroll
      for (int i = 0; i < NV / RPL; ++i) {
        const int j = base + i;
        dst[(j >> 3) * D + (j & 7)] = a[i];
      }
    }
  } else {  // a wavefront past T, or all masked: nothing to add
    if (lane < G) {
      m_s[wave][lane] = -INFINITY;
      l_s[wave][lane] = 0.0f;
    }
    for (int i = lane; i < G * D; i += 64) acc_s[wave][i / D][i % D] = 0.0f;
  }
  // ---- merge the wavefronts' partial results
  __syncthreads();
  for (int i = tid; i < G * D / 2; i += ATT_THREADS) {
    const int g = i / (D / 2), d = (i % (D / 2)) * 2;  // dimensions d, d + 1
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < ATT_WAVES; ++w) mm = fmaxf(mm, m_s[w][g]);
    float n0 = 0.0f, n1 = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < ATT_WAVES; ++w) {
      const float a = m_s[w][g] == -INFINITY ? 0.0f : exp2f(m_s[w][g] - mm);  // wavefronts past T
      n0 = __builtin_fmaf(acc_s[w][g][d], a, n0);
      n1 = __builtin_fmaf(acc_s[w][g][d + 1], a, n1);
      den = __builtin_fmaf(l_s[w][g], a, den);
    }
    const int64_t head = (int64_t)b * p.Hq + kvh * G + g;
    if (p.NS == 1 && p.out != nullptr) {  // out == nullptr: the caller wants the partial results whatever NS is
      const float r = attn_inv_denominator(den);
      store_wt(reinterpret_cast<uint32_t*>(p.out + head * D + d), pack_bf16x2(__fmul_rn(n0, r), __fmul_rn(n1, r)));
    } else {
      float* part = p.ws + (head * p.NS + split) * PART;
      store_wt(reinterpret_cast<uint2*>(part + d), make_uint2(__float_as_uint(n0), __float_as_uint(n1)));
      if (d == 0) store_wt(reinterpret_cast<uint2*>(part + D), make_uint2(__float_as_uint(mm), __float_as_uint(den)));
    }
  }
}

// Combines the NS slices of one (sequence, query head): thread = dimension pair (D / 2 threads).
__global__ __launch_bounds__(ATT_MAX_D / 2) void attn_merge_kernel(const float* ws, uint16_t* out, int NS, int D) {
  const int d = threadIdx.x * 2, part_sz = D + 4;
  const float* part = ws + (int64_t)blockIdx.x * NS * part_sz;
  // Slices are taken eight at a time, all loads of a group requested before any is used: with one slice per
  // loop turn every load waited for the one before it (32 slices: two passes of 32 round trips).  The sums
  // still run in slice order.
  constexpr int GRP = 8;
  float mm = -INFINITY;
  float n0 = 0.0f, n1 = 0.0f, den = 0.0f;
  if (NS <= GRP) {
    // The usual case (up to 2048 positions): (maximum, denominator) and the numerators of every slice are
    // requested together, so the launch is one memory round trip instead of two (maxima first, then values).
    float2 md[GRP], v[GRP];
#pragma unroll
    for (int i = 0; i < GRP; ++i) {
      const bool ok = i < NS;  // uniform
      md[i] = ok ? *reinterpret_cast<const float2*>(part + i * part_sz + D) : make_float2(-INFINITY, 0.0f);
      v[i] = ok ? *reinterpret_cast<const float2*>(part + i * part_sz + d) : make_float2(0.0f, 0.0f);
    }
#pragma unroll
    for (int i = 0; i < GRP; ++i) mm = fmaxf(mm, md[i].x);
#pragma unroll
    for (int i = 0; i < GRP; ++i) {
      if (i < NS) {
        const float a = attn_slice_weight(md[i].x, mm);
        n0 = __builtin_fmaf(v[i].x, a, n0);
        n1 = __builtin_fmaf(v[i].y, a, n1);
        den = __builtin_fmaf(md[i].y, a, den);
      }
    }
  } else {
    for (int s0 = 0; s0 < NS; s0 += GRP) {  // slice 0 always holds a position
      float mv[GRP];
#pragma unroll
      for (int i = 0; i < GRP; ++i) mv[i] = s0 + i < NS ? part[(s0 + i) * part_sz + D] : -INFINITY;
#pragma unroll
      for (int i = 0; i < GRP; ++i) mm = fmaxf(mm, mv[i]);
    }
    for (int s0 = 0; s0 < NS; s0 += GRP) {
      float2 md[GRP], v[GRP];
#pragma unroll
      for (int i = 0; i < GRP; ++i) {
        const bool ok = s0 + i < NS;  // uniform
        md[i] = ok ? *reinterpret_cast<const float2*>(part + (s0 + i) * part_sz + D) : make_float2(0.0f, 0.0f);
        v[i] = ok ? *reinterpret_cast<const float2*>(part + (s0 + i) * part_sz + d) : make_float2(0.0f, 0.0f);
      }
#pragma unroll
      for (int i = 0; i < GRP; ++i) {
        if (s0 + i < NS) {
          const float a = attn_slice_weight(md[i].x, mm);
          n0 = __builtin_fmaf(v[i].x, a, n0);
          n1 = __builtin_fmaf(v[i].y, a, n1);
          den = __builtin_fmaf(md[i].y, a, den);
        }
      }
    }
  }
  const float r = attn_inv_denominator(den);
  store_wt(reinterpret_cast<uint32_t*>(out + (int64_t)blockIdx.x * D + d), pack_bf16x2(__fmul_rn(n0, r), __fmul_rn(n1, r)));
}

inline int64_t attn_slices(int64_t T) { return (T + ATT_KPG - 1) / ATT_KPG; }
// sized for the larger head dimension, so that the size does not depend on D
inline int64_t attn_workspace_bytes(int64_t B, int64_t Hq, int64_t ns) {
  return B * Hq * ns * (ATT_MAX_D + 4) * (int64_t)sizeof(float);
}

}  // namespace aq

// q_gain == nullptr: no qk-norm (then k_gain and eps are not looked at).  keys_only: q_out is not written.
static int rope_kv_write(const void* qkv, const float* freqs, int64_t freqs_stride, const int64_t* page_table,
                         int64_t P, int64_t pos, int64_t S, int64_t page_size, void* k_cache, void* v_cache,
                         int64_t n_pages, void* q_out, void* k_out, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                         const void* q_gain, const void* k_gain, float eps, void* stream, bool keys_only = false) {
  if (D != 64 && D != 128) return AQ_E_SHAPE;
  if (q_gain && (!k_gain || !(eps >= 0.0f))) return k_gain ? AQ_E_SHAPE : AQ_E_NULL;
  if (aq::check_ptr16(q_gain) || (q_gain && aq::check_ptr16(k_gain))) return AQ_E_ALIGN;
  if (B < 0 || S < 0 || Hq <= 0 || Hkv <= 0 || P <= 0 || pos < 0 || page_size <= 0 || n_pages <= 0) return AQ_E_SHAPE;
  if (freqs_stride != 0 && freqs_stride < S * D) return AQ_E_SHAPE;
  if (B == 0 || S == 0) return AQ_OK;
  if (!qkv || !freqs || !page_table || !k_cache || !v_cache || (!q_out && !keys_only)) return AQ_E_NULL;
  if (aq::check_ptr16(qkv) || aq::check_ptr16(k_cache) || aq::check_ptr16(v_cache) || aq::check_ptr16(q_out) ||
      aq::check_ptr16(freqs) || (freqs_stride & 3) || (k_out && aq::check_ptr16(k_out)))
    return AQ_E_ALIGN;
  const int64_t chunks = B * S * ((keys_only ? 0 : Hq) + 2 * Hkv) * (D / 8);
  if (chunks > (int64_t)0x7fffffff * 256) return AQ_E_RANGE;
  aq::RopeArgs a{};
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.freqs = freqs;
  a.freqs_stride = freqs_stride;
  a.table = page_table;
  a.kc = static_cast<uint16_t*>(k_cache);
  a.vc = static_cast<uint16_t*>(v_cache);
  a.q_out = static_cast<uint16_t*>(q_out);
  a.k_out = static_cast<uint16_t*>(k_out);
  a.P = P;
  a.pos = pos;
  a.page = page_size;
  a.n_pages = n_pages;
  a.S = S;
  a.B = (int)B;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.D = (int)D;
  a.q_gain = static_cast<const uint16_t*>(q_gain);
  a.k_gain = static_cast<const uint16_t*>(k_gain);
  a.eps = eps;
  aq::queue_kernel(aq::rope_kv_write_kernel, dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  return (int)hipGetLastError();
}

extern "C" int aq_rope_kv_write(const void* qkv, const float* freqs, int64_t freqs_stride, const int64_t* page_table,
                                int64_t P, int64_t pos, int64_t S, int64_t page_size, void* k_cache, void* v_cache,
                                int64_t n_pages, void* q_out, void* k_out, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                void* stream) {
  return rope_kv_write(qkv, freqs, freqs_stride, page_table, P, pos, S, page_size, k_cache, v_cache, n_pages, q_out, k_out,
                       B, Hq, Hkv, D, nullptr, nullptr, 0.0f, stream);
}

extern "C" int aq_rope_kv_write_qknorm(const void* qkv, const float* freqs, int64_t freqs_stride,
                                       const int64_t* page_table, int64_t P, int64_t pos, int64_t S, int64_t page_size,
                                       void* k_cache, void* v_cache, int64_t n_pages, void* q_out, void* k_out, int64_t B,
                                       int64_t Hq, int64_t Hkv, int64_t D, const void* q_gain, const void* k_gain,
                                       float eps, void* stream) {
  if (!q_gain || !k_gain) return AQ_E_NULL;
  return rope_kv_write(qkv, freqs, freqs_stride, page_table, P, pos, S, page_size, k_cache, v_cache, n_pages, q_out, k_out,
                       B, Hq, Hkv, D, q_gain, k_gain, eps, stream);
}

extern "C" int aq_rope_kv_cache_write(const void* qkv, const float* freqs, int64_t freqs_stride, const int64_t* page_table,
                                      int64_t P, int64_t pos, int64_t S, int64_t page_size, void* k_cache, void* v_cache,
                                      int64_t n_pages, void* k_out, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                      const void* k_gain, float eps, void* stream) {
  return rope_kv_write(qkv, freqs, freqs_stride, page_table, P, pos, S, page_size, k_cache, v_cache, n_pages, nullptr, k_out, B,
                       Hq, Hkv, D, k_gain, k_gain, eps, stream, true);
}

extern "C" int64_t aq_paged_attn_decode_workspace_bytes(int64_t B, int64_t Hq, int64_t Hkv, int64_t total_len) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || total_len <= 0) return 0;
  const int64_t ns = aq::attn_slices(total_len);
  return ns == 1 ? 0 : aq::attn_workspace_bytes(B, Hq, ns);
}

template <int G, int D, bool WHOLE>
static void attn_launch(bool rope, dim3 grid, dim3 block, hipStream_t st, const aq::AttnArgs& a) {
  if (rope && a.q_gain)
    aq::queue_kernel((aq::paged_attn_decode_kernel<G, D, WHOLE, true, true>), grid, block, 0, st, a);
  else if (rope)
    aq::queue_kernel((aq::paged_attn_decode_kernel<G, D, WHOLE, true>), grid, block, 0, st, a);
  else
    aq::queue_kernel((aq::paged_attn_decode_kernel<G, D, WHOLE, false>), grid, block, 0, st, a);
}

// q == nullptr: the fused form, queries and the new token come from qkv / freqs.
// partials: stop after the slices' partial results (no merge launch, `out` unused).
static int attn_decode(const void* q, const void* qkv, const float* freqs, int64_t freqs_stride, void* k_cache,
                       void* v_cache, const int64_t* page_table, int64_t P, int64_t total_len,
                       const int64_t* seq_lens, int64_t page_size,
                       int64_t n_pages, float scale, void* out, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                       void* workspace, int64_t workspace_bytes, void* stream, bool partials = false,
                       const void* q_gain = nullptr, const void* k_gain = nullptr, float eps = 0.0f) {
  const bool rope = q == nullptr;
  if (D != 64 && D != 128) return AQ_E_SHAPE;
  if (q_gain && (!rope || !k_gain)) return AQ_E_NULL;  // qk-norm belongs to the forms that rotate
  if (q_gain && !(eps >= 0.0f)) return AQ_E_SHAPE;
  if (aq::check_ptr16(q_gain) || (q_gain && aq::check_ptr16(k_gain))) return AQ_E_ALIGN;
  if (B < 0 || Hq <= 0 || Hkv <= 0 || (Hq % Hkv) != 0 || P <= 0 || total_len <= 0 || page_size <= 0 ||
      n_pages <= 0 || !(scale > 0.0f))
    return AQ_E_SHAPE;
  const int64_t G = Hq / Hkv;
  if (G != 1 && G != 2 && G != 3 && G != 4 && G != 6 && G != 8) return AQ_E_SHAPE;  // query heads per KV head
  if (rope && freqs_stride != 0 && freqs_stride < D) return AQ_E_SHAPE;
  if (B == 0) return AQ_OK;
  if (!(rope ? (qkv != nullptr && freqs != nullptr) : (q != nullptr)) || !k_cache || !v_cache || !page_table ||
      (!out && !partials))
    return AQ_E_NULL;
  if (aq::check_ptr16(rope ? qkv : q) || aq::check_ptr16(k_cache) || aq::check_ptr16(v_cache) ||
      (!partials && aq::check_ptr16(out)))
    return AQ_E_ALIGN;
  if (rope && (aq::check_ptr16(freqs) || (freqs_stride & 3))) return AQ_E_ALIGN;
  const int64_t ns = aq::attn_slices(total_len);
  if (B * Hkv * ns > (int64_t)0x7fffffff || B * Hq > (int64_t)0x7fffffff) return AQ_E_RANGE;
  if (ns > 1 || partials) {
    if (!workspace) return AQ_E_NULL;
    if (aq::check_ptr16(workspace)) return AQ_E_ALIGN;
    if (workspace_bytes < aq::attn_workspace_bytes(B, Hq, ns)) return AQ_E_WORKSPACE;
  }
  aq::AttnArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.qkv = static_cast<const uint16_t*>(qkv);
  a.freqs = freqs;
  a.freqs_stride = freqs_stride;
  a.kc = static_cast<const uint16_t*>(k_cache);
  a.vc = static_cast<const uint16_t*>(v_cache);
  a.kc_w = static_cast<uint16_t*>(k_cache);
  a.vc_w = static_cast<uint16_t*>(v_cache);
  a.table = page_table;
  a.lens = seq_lens;
  a.out = partials ? nullptr : static_cast<uint16_t*>(out);
  a.ws = static_cast<float*>(workspace);
  a.P = P;
  a.T = total_len;
  a.page = page_size;
  a.n_pages = n_pages;
  a.scale_log2e = scale * 1.44269504088896341f;
  a.B = (int)B;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.NS = (int)ns;
  a.q_gain = static_cast<const uint16_t*>(q_gain);
  a.k_gain = static_cast<const uint16_t*>(k_gain);
  a.eps = eps;
  a.lens_at = seq_lens ? seq_lens : page_table;
  a.by_hkv = aq::UDiv::of((uint32_t)Hkv);
  a.by_ns = aq::UDiv::of((uint32_t)ns);
  if (total_len <= ((int64_t)1 << 31) && page_size <= ((int64_t)1 << 31)) a.by_page = aq::UDiv::of((uint32_t)page_size);
  a.page_shift = 62;
  for (int sh = 6; sh < 62; ++sh)
    if (page_size == ((int64_t)1 << sh)) a.page_shift = sh;
  const dim3 grid((unsigned)(B * Hkv * ns)), block(aq::ATT_WAVES * 64);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool whole = a.page_shift < 62;
#define AQ_ATTN_CASE(G_)                                                                                                          \
  case G_:                                                                                                                        \
    if (D == 128) (whole ? attn_launch<G_, 128, true> : attn_launch<G_, 128, false>)(rope, grid, block, st, a);                   \
    else (whole ? attn_launch<G_, 64, true> : attn_launch<G_, 64, false>)(rope, grid, block, st, a);                              \
    break;
  switch (G) {
    AQ_ATTN_CASE(1)
    AQ_ATTN_CASE(2)
    AQ_ATTN_CASE(3)
    AQ_ATTN_CASE(4)
    AQ_ATTN_CASE(6)
    AQ_ATTN_CASE(8)
  }
#undef AQ_ATTN_CASE
  int rc = (int)hipGetLastError();
  if (rc != 0 || ns == 1 || partials) return rc;
  aq::queue_kernel(aq::attn_merge_kernel, dim3((unsigned)(B * Hq)), dim3((unsigned)(D / 2)), 0, st, a.ws, a.out, a.NS,
                     (int)D);
  return (int)hipGetLastError();
}

extern "C" int aq_paged_attn_decode(const void* q, const void* k_cache, const void* v_cache,
                                    const int64_t* page_table, int64_t P, int64_t total_len,
                                    const int64_t* seq_lens, int64_t page_size,
                                    int64_t n_pages, float scale, void* out, int64_t B, int64_t Hq, int64_t Hkv,
                                    int64_t D, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!q && B > 0) return AQ_E_NULL;
  return attn_decode(q, nullptr, nullptr, 0, const_cast<void*>(k_cache), const_cast<void*>(v_cache), page_table, P,
                     total_len, seq_lens, page_size, n_pages, scale, out, B, Hq, Hkv, D, workspace, workspace_bytes, stream);
}

extern "C" int aq_rope_paged_attn_decode(const void* qkv, const float* freqs, int64_t freqs_stride,
                                         const int64_t* page_table, int64_t P, int64_t total_len,
                                         const int64_t* seq_lens, int64_t page_size,
                                         void* k_cache, void* v_cache, int64_t n_pages, float scale, void* out,
                                         int64_t B, int64_t Hq, int64_t Hkv, int64_t D, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  if ((!qkv || !freqs) && B > 0) return AQ_E_NULL;
  return attn_decode(nullptr, qkv, freqs, freqs_stride, k_cache, v_cache, page_table, P, total_len, seq_lens, page_size, n_pages,
                     scale, out, B, Hq, Hkv, D, workspace, workspace_bytes, stream);
}

extern "C" int64_t aq_paged_attn_decode_slices(int64_t total_len) { return total_len <= 0 ? 0 : aq::attn_slices(total_len); }

extern "C" int64_t aq_paged_attn_decode_partials_bytes(int64_t B, int64_t Hq, int64_t total_len) {
  if (B <= 0 || Hq <= 0 || total_len <= 0) return 0;
  return aq::attn_workspace_bytes(B, Hq, aq::attn_slices(total_len));
}

extern "C" int aq_paged_attn_decode_partials(const void* q, const void* k_cache, const void* v_cache,
                                             const int64_t* page_table, int64_t P, int64_t total_len,
                                             const int64_t* seq_lens,
                                             int64_t page_size, int64_t n_pages, float scale, int64_t B, int64_t Hq,
                                             int64_t Hkv, int64_t D, void* partials, int64_t partials_bytes,
                                             void* stream) {
  if (!q && B > 0) return AQ_E_NULL;
  return attn_decode(q, nullptr, nullptr, 0, const_cast<void*>(k_cache), const_cast<void*>(v_cache), page_table, P,
                     total_len, seq_lens, page_size, n_pages, scale, nullptr, B, Hq, Hkv, D, partials, partials_bytes, stream,
                     true);
}

extern "C" int aq_rope_paged_attn_decode_partials(const void* qkv, const float* freqs, int64_t freqs_stride,
                                                  const int64_t* page_table, int64_t P, int64_t total_len,
                                                  const int64_t* seq_lens,
                                                  int64_t page_size, void* k_cache, void* v_cache, int64_t n_pages,
                                                  float scale, int64_t B, int64_t Hq, int64_t Hkv, int64_t D,
                                                  void* partials, int64_t partials_bytes, void* stream) {
  if ((!qkv || !freqs) && B > 0) return AQ_E_NULL;
  return attn_decode(nullptr, qkv, freqs, freqs_stride, k_cache, v_cache, page_table, P, total_len, seq_lens, page_size, n_pages,
                     scale, nullptr, B, Hq, Hkv, D, partials, partials_bytes, stream, true);
}

extern "C" int aq_rope_paged_attn_decode_qknorm(const void* qkv, const float* freqs, int64_t freqs_stride,
                                                const int64_t* page_table, int64_t P, int64_t total_len,
                                                const int64_t* seq_lens, int64_t page_size, void* k_cache, void* v_cache,
                                                int64_t n_pages, float scale, void* out, int64_t B, int64_t Hq,
                                                int64_t Hkv, int64_t D, const void* q_gain, const void* k_gain, float eps,
                                                void* workspace, int64_t workspace_bytes, void* stream) {
  if ((!qkv || !freqs) && B > 0) return AQ_E_NULL;
  if (!q_gain || !k_gain) return AQ_E_NULL;
  return attn_decode(nullptr, qkv, freqs, freqs_stride, k_cache, v_cache, page_table, P, total_len, seq_lens, page_size, n_pages,
                     scale, out, B, Hq, Hkv, D, workspace, workspace_bytes, stream, false, q_gain, k_gain, eps);
}

extern "C" int aq_rope_paged_attn_decode_partials_qknorm(const void* qkv, const float* freqs, int64_t freqs_stride,
                                                         const int64_t* page_table, int64_t P, int64_t total_len,
                                                         const int64_t* seq_lens, int64_t page_size, void* k_cache,
                                                         void* v_cache, int64_t n_pages, float scale, int64_t B,
                                                         int64_t Hq, int64_t Hkv, int64_t D, const void* q_gain,
                                                         const void* k_gain, float eps, void* partials,
                                                         int64_t partials_bytes, void* stream) {
  if ((!qkv || !freqs) && B > 0) return AQ_E_NULL;
  if (!q_gain || !k_gain) return AQ_E_NULL;
  return attn_decode(nullptr, qkv, freqs, freqs_stride, k_cache, v_cache, page_table, P, total_len, seq_lens, page_size, n_pages,
                     scale, nullptr, B, Hq, Hkv, D, partials, partials_bytes, stream, true, q_gain, k_gain, eps);
}
