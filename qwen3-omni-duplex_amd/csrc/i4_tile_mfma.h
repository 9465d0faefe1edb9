// Device helpers of the kernels that multiply I4_LAYOUT_TILE weights on MFMA
// (i4_moe_mfma.hip, i4_tile_gemm.hip): activation staging, operand decode, weight loads.
// The operand layout and the numerics are described at the top of i4_moe_mfma.hip.
#pragma once

#include "i4_moe_launch.h"

namespace i4 {

// Staged activations: token m's 16 words of a superchunk are one 256-byte row, word w
// at slot w ^ (m & 15) (xs_at).  An MFMA operand load (lanes = 16 tokens x 4
// words) and a staging store (16 lanes = 4 tokens x 4 words) each touch every bank
// once per 16 lanes; measured on gfx950, the swizzled rows read at 4.4 cycles per
// wave-wide 16-byte load against 8.1 with a one-word pad per row.
static constexpr int MF_TSTRIDE = 16;  // uint4 per staged token row
__device__ inline int xs_at(int m, int w) { return m * MF_TSTRIDE + (w ^ (m & 15)); }

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ inline u32x4 bload16(rsrc_t r, u32 voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
// the same past the L1 (sc1): sees what other CUs of the launch wrote through
__device__ inline u32x4 bload16_coherent(rsrc_t r, u32 voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, kCoherent);
}
__device__ inline u32 bload4(rsrc_t r, u32 voff, int soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
template <int ST> __device__ inline u32 bload_scale(rsrc_t r, u32 voff, int soff) {
  if constexpr (ST == I4_F32) return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
  else return (u32)__builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
}

template <int XT> __device__ inline f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (XT == I4_F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// 8 exact halves M + q of one tile word (nibble slots (p, p + 4) -> half pair p),
// columns 8m .. 8m + 7 in order
template <int XT> __device__ inline u32x4 decode8(u32 w, u32 mg) {
  constexpr u32 MK = 0x000F000Fu;
  return u32x4{(w & MK) | mg, ((w >> 4) & MK) | mg, ((w >> 8) & MK) | mg, ((w >> 12) & MK) | mg};
}

// fp16 pair (M + q0, M + q1) + nz, nz = (-(M + z), -(M + z)): exactly (q0 - z, q1 - z)
__device__ inline u32 sub_zero(u32 p, u32 nz) {
  return __builtin_bit_cast(u32, __builtin_bit_cast(f16x2, p) + __builtin_bit_cast(f16x2, nz));
}

// -(M + z) twice, fp16, for the zero point of group g held in zero word zw
__device__ inline u32 neg_zero2(u32 zw, int g) {
  return (0xE400u | ((zw >> (4 * (g & 7))) & 15u)) * 0x00010001u;
}

// B operand of one MFMA step (nz: neg_zero2 of the step's group, fp16 only;
// mg: magic_v<XT>())
template <int XT> __device__ inline u32x4 b_operand(u32 word, u32 nz, u32 mg) {
  u32x4 b = decode8<XT>(word, mg);
  if constexpr (XT == I4_F16) {
    b.x = sub_zero(b.x, nz);
    b.y = sub_zero(b.y, nz);
    b.z = sub_zero(b.z, nz);
    b.w = sub_zero(b.w, nz);
  }
  return b;
}

// the group scale as two fp16 copies (rounded to fp16 when stored wider)
template <int ST> __device__ inline u32 scale_h2(u32 raw) {
  if constexpr (ST == I4_F16) {
    return (raw & 0xFFFFu) * 0x00010001u;
  } else {
    const u32 h = __builtin_bit_cast(uint16_t, (_Float16)scale_from_raw<ST>(raw));
    return h * 0x00010001u;
  }
}

// fp16 pairs a * s (one v_pk_mul_f16)
__device__ inline u32 mul_h2(u32 a, u32 s) {
  return __builtin_bit_cast(u32, __builtin_bit_cast(f16x2, a) * __builtin_bit_cast(f16x2, s));
}

// fp16 B operand times the group scale: (q - z) s, one rounding per element.
// The components go through scalars: a bit cast applied directly to a vector
// component expression (b.y) reads component 0 with this compiler.
__device__ inline u32x4 scale_b(u32x4 b, u32 s2) {
  const u32 b0 = b.x, b1 = b.y, b2 = b.z, b3 = b.w;
  return u32x4{mul_h2(b0, s2), mul_h2(b1, s2), mul_h2(b2, s2), mul_h2(b3, s2)};
}

// first row block of n-block nb of wave `wave` (of WN along the rows) in column tile `tile`
template <bool GATEUP, int NB, int WN = 4>
__device__ inline int nblock(int tile, int wave, int nb, int I) {
  if constexpr (GATEUP)
    return tile * (WN * NB / 2) + (NB / 2) * wave + (nb % (NB / 2)) + (nb >= NB / 2 ? (I >> 4) : 0);
  else
    return tile * (WN * NB) + NB * wave + nb;
}

// the weight operands of one wave: NB n-blocks of expert e, lane (r, j).
// Lane offsets live in VGPRs; the n-block offsets are wave-uniform and go in
// the scalar offset of each load, with the superchunk / group offset.
template <int ST, int NB> struct WBuf {
  rsrc_t p, s, z;
  u32 lw, ls, lz;              // per-lane byte offsets
  int bw[NB], bs[NB], bz[NB];  // per-n-block byte offsets (wave-uniform)
  u32 zor;                     // 0x88888888 when the weight has no zero points
  int gshift;
};

template <int ST, int NB>
__device__ inline WBuf<ST, NB> wbuf(const TW& w, int e, const int (&blk)[NB], int r, int j) {
  constexpr int SB = ST == I4_F32 ? 4 : 2;
  const int SC = w.K >> 7;
  const int NG = (w.K + (32 << w.gshift) - 1) >> (w.gshift + 5), NZW = (NG + 7) >> 3;
  WBuf<ST, NB> b;
  b.p = rsrc(w.packed + e * w.pes, (u32)w.N * (u32)(w.K >> 1));
  b.s = rsrc((const char*)w.scale + e * w.ses * SB, (u32)w.N * NG * SB);
  if (w.zeros) {
    b.z = rsrc(w.zeros + e * w.zes, (u32)w.N * NZW * 4u);
    b.zor = 0u;
  } else {
    b.z = rsrc(w.packed, 0u);
    b.zor = 0x88888888u;
  }
  b.lw = (u32)r * 64u + (u32)j * 16u;
  b.ls = (u32)r * SB;
  b.lz = (u32)r * 4u;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    b.bw[nb] = blk[nb] * SC * 1024;
    b.bs[nb] = blk[nb] * NG * 16 * SB;
    b.bz[nb] = blk[nb] * NZW * 64;
  }
  b.gshift = w.gshift;
  return b;
}

// superchunk sc of every n-block: the 16-byte tile word, the raw scale(s) and
// the zero word (one zero word covers the superchunk's groups).  Nothing here
// touches the loaded values, so issuing never waits for a load.
template <int ST, bool GB, int NB>
__device__ inline void wissue(const WBuf<ST, NB>& b, int sc, TSlot<GB> (&o)[NB]) {
  constexpr int SB = ST == I4_F32 ? 4 : 2;
  const int g0 = (4 * sc) >> b.gshift;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    o[nb].w = bload16(b.p, b.lw, b.bw[nb] + sc * 1024);
    if constexpr (GB) {
      o[nb].s[0] = bload_scale<ST>(b.s, b.ls, b.bs[nb] + g0 * 16 * SB);
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        o[nb].s[t] = bload_scale<ST>(b.s, b.ls, b.bs[nb] + ((4 * sc + t) >> b.gshift) * 16 * SB);
    }
    o[nb].z = bload4(b.z, b.lz, b.bz[nb] + (g0 >> 3) * 64);  // | zor where it is used
  }
}

// end of a group: the scale of the lane's column times its sums
template <int ST> __device__ inline void add_group(f32x4& res, const f32x4& d, u32 sraw) {
  const float sv = scale_from_raw<ST>(sraw);
#pragma unroll
  for (int i = 0; i < 4; ++i) res[i] = fmaf(sv, d[i], res[i]);
}

}  // namespace i4
