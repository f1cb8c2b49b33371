// The rotation of query and key heads and the RMSNorm behind it, a 16-byte chunk at a time: what the kernels that rotate share,
// so that all of them give the same bits.
#ifndef AQ_ROPE_H
#define AQ_ROPE_H

#include "aq_common.h"
#include "aq_rows.h"

namespace aq {

// Rotates 8 consecutive elements (4 interleaved pairs): (x0 + i x1)(c + i s) with four rounded
// products, one rounded difference and one rounded sum per pair.  a, b: 4 (cos, sin) pairs.
__device__ __forceinline__ uint4 rope8(uint4 x, float4 a, float4 b) {
  const float c[4] = {a.x, a.z, b.x, b.z}, sn[4] = {a.y, a.w, b.y, b.w};
  const uint32_t in[4] = {x.x, x.y, x.z, x.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x0 = __uint_as_float(in[i] << 16), x1 = __uint_as_float(in[i] & 0xffff0000u);
    const float r0 = __fsub_rn(__fmul_rn(x0, c[i]), __fmul_rn(x1, sn[i]));
    const float r1 = __fadd_rn(__fmul_rn(x0, sn[i]), __fmul_rn(x1, c[i]));
    o[i] = pack_bf16x2(r0, r1);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}
__device__ __forceinline__ uint4 rope8(uint4 x, const float* cs) {
  return rope8(x, *reinterpret_cast<const float4*>(cs), *reinterpret_cast<const float4*>(cs + 4));
}

// RMSNorm over the head dimension of a rotated query or key (attention.py:62-64, 86-89: after the rotation, before
// the key goes into the cache).  The rotated values are taken as they are stored, rounded to bf16.  Sum of squares
// in a fixed order that does not depend on which kernel holds the vector how: per 8-element chunk the rounded
// squares are added in memory order, then the D / 8 chunk sums are combined by a butterfly over the chunk index
// (chunk c with c ^ 1, then ^ 2, ^ 4, ^ 8; fl(a + b) is the same whichever partner computes it).  Then
// r = 1 / sqrt(ss / D + eps) (every operation correctly rounded) and y = bf16((x * r) * gain).
__device__ __forceinline__ float chunk_sumsq(uint4 x) {
  const uint32_t in[4] = {x.x, x.y, x.z, x.w};
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x0 = __uint_as_float(in[i] << 16), x1 = __uint_as_float(in[i] & 0xffff0000u);
    s = __fadd_rn(s, __fmul_rn(x0, x0));
    s = __fadd_rn(s, __fmul_rn(x1, x1));
  }
  return s;
}
// the sum over a head vector whose D / 8 chunks sit in neighbouring lanes of one DPP row, in all of them
template <int D>
__device__ __forceinline__ float head_sumsq(uint4 x) {
  float ss = chunk_sumsq(x);
  ss = __fadd_rn(ss, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0xB1, 0xf, 0xf, false)));   // c ^ 1
  ss = __fadd_rn(ss, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x4E, 0xf, 0xf, false)));   // c ^ 2
  ss = __fadd_rn(ss, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x141, 0xf, 0xf, false)));  // the other quad of the half row: c ^ 4
  if constexpr (D == 128)
    ss = __fadd_rn(ss, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x140, 0xf, 0xf, false)));  // the other half row: c ^ 8
  return ss;
}
__device__ __forceinline__ uint4 chunk_normed(uint4 x, float r, uint4 gain) {
  const uint32_t in[4] = {x.x, x.y, x.z, x.w}, gn[4] = {gain.x, gain.y, gain.z, gain.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x0 = __uint_as_float(in[i] << 16), x1 = __uint_as_float(in[i] & 0xffff0000u);
    const float g0 = __uint_as_float(gn[i] << 16), g1 = __uint_as_float(gn[i] & 0xffff0000u);
    o[i] = pack_bf16x2(__fmul_rn(__fmul_rn(x0, r), g0), __fmul_rn(__fmul_rn(x1, r), g1));
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

}  // namespace aq

#endif  // AQ_ROPE_H
