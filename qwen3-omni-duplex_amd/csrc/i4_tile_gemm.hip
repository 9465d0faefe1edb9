// Projections of many rows: 128 tokens x 256 weight rows per workgroup of eight waves.
//
// The operand layout and numerics are those of i4_moe_mfma.hip: fp16 entries of more than
// 16 tokens fold the scale into B, everything else is exact.  There a workgroup multiplies
// 64 tokens with 128 rows, so every byte staged in LDS or decoded feeds half to a quarter
// of the MFMAs it feeds here.  Wave v owns two n-blocks of 16 weight rows (GATEUP: a gate
// block and its up block), decodes them itself and multiplies them with every token of the
// entry; the 128 activation rows of a superchunk are staged once for all eight waves, double
// buffered, loaded one superchunk ahead.  One workgroup fills a CU (up to 256 VGPRs).
//
// Bound: issue.  A superchunk takes 2.9 us with groups of 32 (5.9 vector instructions per
// MFMA, 4 of them FMAs that apply the scales: MFMA busy 29 %, VALU 51 %, LDS 41 % of the
// cycles, the two waves of a SIMD overlapping little) and 2.3 us with folded scales (2.6;
// MFMA 37 %), the same on an idle card.  Measured: bf16 2048 -> 5120, 1500 rows 109 -> 50 us
// (630 TFLOP/s); the 3001-token MoE block, with its router and combine, 942 -> 523 us.
// Slower: waves in a 2 x 4 arrangement of 64 x 64 (54 us), 128 x 128 tiles of four waves, two
// workgroups per CU (62 us), MFMA and FMA groups interleaved by hand (58-62 us), a branch
// around the last step of an odd superchunk count, whose products alone are skipped (245 us).
// The zero points' presence is a template argument for bf16: chosen at run time, the
// compiler multiplied and selected in every group (72 us).
#include "i4_tile_mfma.h"

namespace i4 {

// One entry of <= TG_TOK tokens x one column tile of 32 NW weight rows.  GB: groups of 128
// or more columns; SYM: bf16 without zero points; LIN: a dense linear layer over M rows
// (entry y is rows TG_TOK y ..), bias and output type as in k_tile_mfma.  An entry may be
// empty.
template <int XT, int ST, bool GB, bool SYM, bool GATEUP, bool LIN, int NW>
__global__ __launch_bounds__(64 * NW) void k_tile_gemm(
    const uint16_t* __restrict__ src, u32 src_bytes, int topk, const int4* __restrict__ entries,
    const int* __restrict__ n_entries, const int32_t* __restrict__ perm, TW w, int I,
    uint16_t* __restrict__ act, void* __restrict__ ys, int M, const void* __restrict__ bias,
    int ot, int n_cols) {
  constexpr bool F16 = XT == I4_F16;
  constexpr int NB = 2, NT = 64 * NW, TPT = NT / TG_TOK, WPT = 16 / TPT;
  __shared__ u32x4 xs[2][TG_TOK * MF_TSTRIDE];
  __shared__ __align__(16) float xsum[2][F16 ? 4 : 4 * TG_TOK];
  // XCD-aware order: blocks go round-robin over the 8 XCDs, so block b takes tile
  // (b & 7) * per + (b >> 3): each XCD walks a contiguous run of (entry, column) tiles,
  // whose activations stay in its L2 for all of an entry's column tiles
  const int nl = LIN ? (M + TG_TOK - 1) / TG_TOK : *n_entries;
  const int total = nl * n_cols, per = (total + 7) >> 3;
  const int xi = (int)blockIdx.x >> 3, id = ((int)blockIdx.x & 7) * per + xi;
  if (xi >= per || id >= total) return;
  const int by = id / n_cols, bx = id - by * n_cols;
  const u32 mg = magic_v<XT>();
  const int4 en = LIN ? int4{0, by * TG_TOK, min(TG_TOK, M - by * TG_TOK), 0} : entries[by];
  const int e = en.x, pos0 = en.y, cnt = en.z;
  if (cnt <= 0) return;
  const int K = w.K, SC = K >> 7;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, ln = lane & 15, kb = lane >> 4;
  const bool ev = (unsigned)e < (unsigned)w.E;
  const int nmb = (cnt + 15) >> 4;
  int blk[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
    blk[nb] = nblock<GATEUP, NB, NW>(bx, wave, nb, I);
  const WBuf<ST, NB> wb = wbuf<ST, NB>(w, ev ? e : 0, blk, ln, kb);
  const int tk = (int)threadIdx.x / TPT, kw = WPT * ((int)threadIdx.x % TPT);
  const int p0 = pos0 + min(tk, cnt - 1);
  const int row = GATEUP ? perm[p0] / topk : p0;
  const rsrc_t xr = rsrc(src, src_bytes);
  const u32 vx = ((u32)row * (u32)K + 8u * (u32)kw) * 2u;
  const float xscale = SYM ? -(Half<XT>::MAGIC + 8.f) : -1.f;
  u32x4 xd[WPT];
  auto load_x = [&](int sc) {
    sc = min(sc, SC - 1);
#pragma unroll
    for (int q = 0; q < WPT; ++q) xd[q] = bload16(xr, vx + 16u * q, sc * 256);
  };
  auto commit = [&](int buf, const u32x4 (&x)[WPT]) {
#pragma unroll
    for (int q = 0; q < WPT; ++q) xs[buf][xs_at(tk, kw + q)] = x[q];
    if constexpr (!F16) {
      constexpr u32 ONE2 = 0x3F803F80u;
#pragma unroll
      for (int c = 0; c < WPT / 4; ++c) {
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int q = 4 * c; q < 4 * c + 4; ++q) {
          s0 = Half<XT>::dot2(x[q].x, ONE2, s0);
          s1 = Half<XT>::dot2(x[q].y, ONE2, s1);
          s0 = Half<XT>::dot2(x[q].z, ONE2, s0);
          s1 = Half<XT>::dot2(x[q].w, ONE2, s1);
        }
        xsum[buf][TG_TOK * ((kw >> 2) + c) + tk] = xscale * (s0 + s1);
      }
    }
  };
  f32x4 res[8][NB];
#pragma unroll
  for (int mb = 0; mb < 8; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) res[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto compute_nm = [&]<int NM>(int sc, const TSlot<GB>* sl, int buf) {
    constexpr bool FOLD = F16 && NM > 1;
    const int g0 = (4 * sc) >> w.gshift;
    u32 zw[NB], nz[NB], s2[NB];
    float mz[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      zw[nb] = sl[nb].z | wb.zor;
      nz[nb] = F16 && GB ? neg_zero2(zw[nb], g0) : 0u;
      s2[nb] = FOLD && GB ? scale_h2<ST>(sl[nb].s[0]) : 0u;
      mz[nb] = Half<XT>::MAGIC + zero_of(zw[nb], g0);
    }
    f32x4 d[NM][NB];
    auto sums = [&](int mb, int t) {
      return *(const f32x4*)&xsum[buf][TG_TOK * t + 16 * mb + 4 * kb];
    };
    if constexpr (!FOLD && GB) {
#pragma unroll
      for (int mb = 0; mb < NM; ++mb) {
        f32x4 sm = {0.f, 0.f, 0.f, 0.f};
        if constexpr (!F16) sm = (sums(mb, 0) + sums(mb, 1)) + (sums(mb, 2) + sums(mb, 3));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) d[mb][nb] = F16 || SYM ? sm : sm * mz[nb];
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int g = (4 * sc + t) >> w.gshift;
      u32x4 b[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const u32 z2 = GB ? nz[nb] : F16 ? neg_zero2(zw[nb], g) : 0u;
        b[nb] = b_operand<XT>(word_t(sl[nb].w, t), z2, mg);
        if constexpr (FOLD) b[nb] = scale_b(b[nb], GB ? s2[nb] : scale_h2<ST>(sl[nb].s[t]));
        if constexpr (!GB && !F16) mz[nb] = Half<XT>::MAGIC + zero_of(zw[nb], g);
      }
#pragma unroll
      for (int mb = 0; mb < NM; ++mb) {
        const u32x4 a = xs[buf][xs_at(16 * mb + ln, 4 * t + kb)];
        if constexpr (FOLD) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) res[mb][nb] = mfma16<XT>(a, b[nb], res[mb][nb]);
        } else {
          if constexpr (!GB) {
            f32x4 sm = {0.f, 0.f, 0.f, 0.f};
            if constexpr (!F16) sm = sums(mb, t);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) d[mb][nb] = F16 || SYM ? sm : sm * mz[nb];
          }
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) d[mb][nb] = mfma16<XT>(a, b[nb], d[mb][nb]);
        }
      }
      if constexpr (!FOLD && !GB) {
#pragma unroll
        for (int mb = 0; mb < NM; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) add_group<ST>(res[mb][nb], d[mb][nb], sl[nb].s[t]);
      }
    }
    if constexpr (!FOLD && GB) {
#pragma unroll
      for (int mb = 0; mb < NM; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) add_group<ST>(res[mb][nb], d[mb][nb], sl[nb].s[0]);
    }
  };
  auto run = [&]<int NM>() {
    TSlot<GB> w0[NB], w1[NB];
    auto step = [&](int sc, const TSlot<GB> (&cur)[NB], TSlot<GB> (&next)[NB]) {
      const int buf = sc & 1;
      commit(buf, xd);
      __syncthreads();
      load_x(sc + 1);
      wissue<ST, GB, NB>(wb, min(sc + 1, SC - 1), next);
      __builtin_amdgcn_sched_barrier(0);
      if (sc < SC) compute_nm.template operator()<NM>(sc, cur, buf);
    };
    load_x(0);
    wissue<ST, GB, NB>(wb, 0, w0);
    for (int sc = 0; sc < SC; sc += 2) {
      step(sc, w0, w1);
      step(sc + 1, w1, w0);
    }
  };
  if (nmb > 4) run.template operator()<8>();
  else if (nmb > 2) run.template operator()<4>();
  else if (nmb > 1) run.template operator()<2>();
  else run.template operator()<1>();
#pragma unroll
  for (int mb = 0; mb < 8; ++mb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 16 * mb + 4 * kb + i;
      if (m >= cnt) continue;
      if constexpr (GATEUP) {
        const int n = (bx * NW + wave) * 16 + ln;
        const float v = ev ? silu(res[mb][0][i]) * res[mb][1][i] : __builtin_nanf("");
        act[(int64_t)(pos0 + m) * I + n] = Half<XT>::from_f32(v);
      } else if constexpr (LIN) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int n = 16 * ((bx * NW + wave) * NB + nb) + ln;
          const int64_t o = (int64_t)(pos0 + m) * w.N + n;
          float v = res[mb][nb][i];
          if (ot == I4_F32) {
            if (bias) v += ((const float*)bias)[n];
            store_out<I4_F32>(ys, o, v);
          } else if (ot == I4_F16) {
            if (bias) v += Half<I4_F16>::to_f32(((const uint16_t*)bias)[n]);
            store_out<I4_F16>(ys, o, v);
          } else {
            if (bias) v += Half<I4_BF16>::to_f32(((const uint16_t*)bias)[n]);
            store_out<I4_BF16>(ys, o, v);
          }
        }
      } else {
        const int64_t o = (int64_t)perm[pos0 + m] * w.N + 16 * (bx * NW + wave) * NB + ln;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          ((uint16_t*)ys)[o + 16 * nb] =
              Half<XT>::from_f32(ev ? res[mb][nb][i] : __builtin_nanf(""));
      }
    }
  }
}

// ---------------------------------------------------------------------------
namespace {

template <int XT, int ST, bool GATEUP, bool LIN>
int tile_gemm_t(int max_entries, const void* src, int src_rows, int topk, const int4* ent,
                const int* nent, const int32_t* perm, const TW& w, int I, void* out,
                const void* bias, int ot, hipStream_t s) {
  const int64_t src_bytes = (int64_t)src_rows * w.K * 2;
  // buffer offsets are 32-bit: the activation rows and one expert's weights must fit
  if (src_bytes >= ((int64_t)1 << 31) || (int64_t)w.N * w.K / 2 >= ((int64_t)1 << 31))
    return I4_ERR_SHAPE;
  const int n_cols = (GATEUP ? 2 * I : w.N) / (32 * TG_NW);
  const dim3 grid(8u * (unsigned)(((int64_t)max_entries * n_cols + 7) / 8));
  uint16_t* act = GATEUP ? (uint16_t*)out : nullptr;
  void* ys = GATEUP ? nullptr : out;
#define I4_TG(GB_, SYM_)                                                                        \
  hipLaunchKernelGGL((k_tile_gemm<XT, ST, GB_, SYM_, GATEUP, LIN, TG_NW>), grid,                \
                     dim3(64 * TG_NW), 0, s, (const uint16_t*)src, (u32)src_bytes, topk, ent,   \
                     nent, perm, w, I, act, ys, src_rows, bias, ot, n_cols)
  const bool sym = XT == I4_BF16 && !w.zeros, gb = w.gshift >= 2;
  if (gb && sym) I4_TG(true, (XT == I4_BF16));
  else if (gb) I4_TG(true, false);
  else if (sym) I4_TG(false, (XT == I4_BF16));
  else I4_TG(false, false);
#undef I4_TG
  return hipGetLastError() == hipSuccess ? I4_OK : I4_ERR_LAUNCH;
}

}  // namespace

template <int XT, int ST>
int launch_tile_gemm_linear(const void* x, int M, const TW& w, const void* bias, void* y, int ot,
                            hipStream_t s) {
  return tile_gemm_t<XT, ST, false, true>((M + TG_TOK - 1) / TG_TOK, x, M, 0, nullptr, nullptr,
                                          nullptr, w, 0, y, bias, ot, s);
}

template <int XT, int ST>
int launch_tile_gemm_moe(bool gate_up, int max_entries, const void* src, int src_rows, int topk,
                         const int4* ent, const int* nent, const int32_t* perm, const TW& w,
                         int I, void* out, hipStream_t s) {
  if (gate_up)
    return tile_gemm_t<XT, ST, true, false>(max_entries, src, src_rows, topk, ent, nent, perm, w,
                                            I, out, nullptr, 0, s);
  return tile_gemm_t<XT, ST, false, false>(max_entries, src, src_rows, topk, ent, nent, perm, w,
                                           0, out, nullptr, 0, s);
}

#define I4_INST(XT_, ST_)                                                                        \
  template int launch_tile_gemm_linear<XT_, ST_>(const void*, int, const TW&, const void*, void*, \
                                                 int, hipStream_t);                              \
  template int launch_tile_gemm_moe<XT_, ST_>(bool, int, const void*, int, int, const int4*,     \
                                              const int*, const int32_t*, const TW&, int, void*, \
                                              hipStream_t);
I4_INST(I4_F16, I4_F32) I4_INST(I4_F16, I4_F16) I4_INST(I4_F16, I4_BF16)
I4_INST(I4_BF16, I4_F32) I4_INST(I4_BF16, I4_F16) I4_INST(I4_BF16, I4_BF16)
#undef I4_INST

}  // namespace i4
