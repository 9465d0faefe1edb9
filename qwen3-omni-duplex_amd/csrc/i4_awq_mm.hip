// AutoAWQ weights in place times several rows of x, on MFMA.
//
// The AWQ layout is K-major: word (k, c) holds columns 8c .. 8c + 7 of row k.  A B operand
// of v_mfma_f32_16x16x32 wants 8 consecutive k of one column per lane, so lane (r, j) takes
// column word c = 16 strip + r of the 8 rows 32 s + 8 j .. + 7: eight words, a 64-byte run
// per row and 16 lanes, and from them the operands of its word's eight columns (row pairs
// merged byte-wise with v_perm_b32, as in the AWQ GEMVs).  Step s then is eight MFMAs, one
// per nibble slot, each over 16 columns eight apart: a wave covers 128 columns x 16 MB rows
// x 32 k.  A operands come straight from x.
//   fp16: B = q - z exactly.  bf16: B = 16 + q exactly (a nibble in the mantissa's upper
//   bits) and an MFMA with ones gives S_m, the sum of row m's activations, in the
//   accumulator's own layout: s (D - (16 + z) S_m).  The difference cancels and leaves the
//   rounding of the two terms, which grows with the bias: 24 rows, 4096 -> 2048, groups of
//   128, relative 2-norm of the fp32 result against float64: 5.5e-7 with 128 + q (one
//   operation per nibble pair less), 1.0e-7 with 16 + q; the GEMV 2.2e-7.
// Every group's sums are scaled in fp32, as in the GEMVs: the same precision.
//
// The GEMVs above stream the weight once per row of x (24 rows of 4096 -> 2048: 97 us, 105
// us profiled); here the 4 waves of a workgroup take consecutive k ranges, summed in LDS,
// and the launch is split along K into fp32 partials until the chip is filled.  Two
// neighbouring strips share every 128-byte line of a row and run on one XCD.
//
// Bound: latency (one step or two per wave, the hand-over to the summing launch).  Both
// launches, back to back in a graph, GEMV -> here: 4096 -> 2048 8 rows 14.0 -> 7.6, 24 rows
// 96 -> 9.5, 256 rows 1000 -> 18 us; 2048 -> 512 24 rows 15.3 -> 7.7 us.
#include "i4_launch.h"
#include "i4_tile_mfma.h"

namespace i4 {

// columns of the nibble slots: 0, 2, 4, 6, 1, 3, 5, 7
__device__ inline constexpr int mm_col(int slot) { return (slot & 3) * 2 + (slot >> 2); }

template <int XT, int ST, int MB>
__global__ __launch_bounds__(256) void k_awq_mm(
    const uint16_t* __restrict__ x, u32 x_bytes, int M, const int32_t* __restrict__ qw,
    const void* __restrict__ scales, const int32_t* __restrict__ qz, int N, int K, int gshift,
    int ksplit, float* __restrict__ part, void* __restrict__ y, int ot,
    const void* __restrict__ bias) {
  constexpr bool F16 = XT == I4_F16;
  constexpr int SB = ST == I4_F32 ? 4 : 2;
  __shared__ f32x4 red[4][8][64];
  const int NW = N >> 3, strips = (NW + 15) >> 4;
  // block b: strip pair and K range u, the pair's two strips eight blocks apart (one XCD)
  const int b = blockIdx.x, u = (b >> 4) * 8 + (b & 7);
  const int pr = u / ksplit, kz = u - pr * ksplit, strip = 2 * pr + ((b >> 3) & 1);
  if (strip >= strips) return;
  const int m0 = 16 * MB * (int)blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, ln = lane & 15, kb = lane >> 4;
  const int cw = strip * 16 + ln, c = min(cw, NW - 1);
  // steps of this workgroup, then of this wave
  const int S = K >> 5, a0 = kz * S / ksplit, na = (kz + 1) * S / ksplit - a0;
  const int s_lo = a0 + na * wave / 4, s_hi = a0 + na * (wave + 1) / 4;
  const u32 mg = F16 ? magic_v<XT>() : vgpr_const(0x41804180u);  // bf16: 16 twice
  constexpr u32 ONE2 = 0x3F803F80u;
  const u32x4 ones = {ONE2, ONE2, ONE2, ONE2};
  // the expert's weight and a row block of x are below 2^31 bytes (checked on the host)
  const rsrc_t rw = rsrc(qw, (u32)K * (u32)NW * 4u), rx = rsrc(x, x_bytes);
  const u32 vw = ((u32)(8 * kb) * (u32)NW + (u32)c) * 4u;
  u32 vx[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    vx[mb] = ((u32)min(m0 + 16 * mb + ln, M - 1) * (u32)K + 8u * (u32)kb) * 2u;
  struct Slot {
    u32 w[8];
    u32x4 a[MB];
  };
  auto load = [&](int s, Slot& o) {
    s = min(s, S - 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) o.w[i] = bload4(rw, vw, (32 * s + i) * NW * 4);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) o.a[mb] = bload16(rx, vx[mb], s * 64);
  };
  f32x4 tot[MB][8], d[MB][8], ds[MB];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    ds[mb] = zero;
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) tot[mb][sl] = d[mb][sl] = zero;
  }
  u32 zw = 0, nz[8];
  u32 sr[8];
  // scales and zero points of step s's group
  auto load_group = [&](int s) {
    const int64_t g = s >> gshift;
    zw = qz ? (u32)qz[g * NW + c] : 0x88888888u;
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) {
      if constexpr (F16) nz[sl] = neg_zero2(zw, sl);
      sr[sl] = load_scale_raw<ST>(scales, g * N + 8 * c + mm_col(sl));
    }
  };
  auto step = [&](int s, const Slot& o) {
    u32x4 bo[8];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32 sel = 0x0C000C00u | (u32)q | ((u32)(4 + q) << 16);
        const u32 t = __builtin_amdgcn_perm(o.w[2 * p + 1], o.w[2 * p], sel);
        u32 lo, hi;
        if constexpr (F16) {
          lo = sub_zero((t & 0x000F000Fu) | mg, nz[2 * q]);
          hi = sub_zero(((t >> 4) & 0x000F000Fu) | mg, nz[2 * q + 1]);
        } else {
          lo = ((t << 3) & 0x00780078u) | mg;
          hi = ((t >> 1) & 0x00780078u) | mg;
        }
        bo[2 * q][p] = lo;
        bo[2 * q + 1][p] = hi;
      }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if constexpr (!F16) ds[mb] = mfma16<XT>(o.a[mb], ones, ds[mb]);
#pragma unroll
      for (int sl = 0; sl < 8; ++sl) d[mb][sl] = mfma16<XT>(o.a[mb], bo[sl], d[mb][sl]);
    }
  };
  auto end_group = [&]() {
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) {
      const float sv = scale_from_raw<ST>(sr[sl]);
      const float mz = 16.f + (float)((zw >> (4 * sl)) & 15u);  // bf16
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          tot[mb][sl][i] += sv * (F16 ? d[mb][sl][i] : d[mb][sl][i] - mz * ds[mb][i]);
        d[mb][sl] = zero;
      }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) ds[mb] = zero;
  };
  if (s_lo < s_hi) {
    Slot cur, next;
    load(s_lo, cur);
    load_group(s_lo);
    for (int s = s_lo; s < s_hi; ++s) {
      load(s + 1, next);
      step(s, cur);
      if (s + 1 == s_hi || (s + 1) >> gshift != s >> gshift) {
        end_group();
        if (s + 1 < s_hi) load_group(s + 1);
      }
      cur = next;
    }
  }
  // the four waves' sums in order, then out (or to this K range's partials)
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    if (mb) __syncthreads();
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) red[wave][sl][lane] = tot[mb][sl];
    __syncthreads();
    // thread t: rows 4 kb .. + 3, two adjacent columns 8 cw + 2 wave, + 1 (slots wave, wave + 4)
    const f32x4 v0 = (red[0][wave][lane] + red[1][wave][lane]) +
                     (red[2][wave][lane] + red[3][wave][lane]);
    const f32x4 v1 = (red[0][wave + 4][lane] + red[1][wave + 4][lane]) +
                     (red[2][wave + 4][lane] + red[3][wave + 4][lane]);
    if (cw < NW) {
      const int n = 8 * cw + 2 * wave;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + 16 * mb + 4 * kb + i;
        if (m >= M) continue;
        const int64_t o = (int64_t)m * N + n;
        float a = v0[i], e = v1[i];
        if (ksplit > 1) {
          *(float2*)(part + (int64_t)kz * M * N + o) = float2{a, e};
        } else if (ot == I4_F32) {
          if (bias) a += ((const float*)bias)[n], e += ((const float*)bias)[n + 1];
          store_out<I4_F32>(y, o, a);
          store_out<I4_F32>(y, o + 1, e);
        } else if (ot == I4_F16) {
          const uint16_t* bh = (const uint16_t*)bias;
          if (bh) a += Half<I4_F16>::to_f32(bh[n]), e += Half<I4_F16>::to_f32(bh[n + 1]);
          store_out<I4_F16>(y, o, a);
          store_out<I4_F16>(y, o + 1, e);
        } else {
          const uint16_t* bh = (const uint16_t*)bias;
          if (bh) a += Half<I4_BF16>::to_f32(bh[n]), e += Half<I4_BF16>::to_f32(bh[n + 1]);
          store_out<I4_BF16>(y, o, a);
          store_out<I4_BF16>(y, o + 1, e);
        }
      }
    }
  }
}

// K ranges: about 256 workgroups (512: 13 against 9.6 us at 32 rows, 2048 -> 4096, for the
// partials), each wave at least one step of 32
int awq_mm_ksplit(int M, int N, int K) {
  const int64_t tiles = (int64_t)((N + 127) / 128) * ((M + 31) / 32);
  int64_t ks = (256 + tiles - 1) / tiles;
  const int most = K / 128;
  if (ks > most) ks = most;
  return ks < 1 ? 1 : (int)ks;
}

bool awq_mm_fits(int M, int N, int K) {
  // buffer offsets are 32-bit
  return (int64_t)M * K * 2 < ((int64_t)1 << 31) && (int64_t)N * K / 2 < ((int64_t)1 << 31);
}

template <int XT, int ST>
int launch_awq_mm(const void* x, int M, const i4_qweight& w, const void* bias, void* y, int ot,
                  float* part, hipStream_t s) {
  const int ks = awq_mm_ksplit(M, w.N, w.K);
  const int pairs = ((w.N + 127) / 128 + 1) / 2;
  const int MB = M > 16 ? 2 : 1;
  const dim3 grid(16 * ((pairs * ks + 7) / 8), (M + 16 * MB - 1) / (16 * MB));
  const int gshift = i4_group_shift(w.group);
#define I4_MM(MB_)                                                                              \
  hipLaunchKernelGGL((k_awq_mm<XT, ST, MB_>), grid, dim3(256), 0, s, (const uint16_t*)x,        \
                     (u32)((int64_t)M * w.K * 2), M, w.packed, w.scale, w.zeros, w.N, w.K,      \
                     gshift, ks, part, y, ot, bias)
  if (MB == 2) I4_MM(2);
  else I4_MM(1);
#undef I4_MM
  if (hipGetLastError() != hipSuccess) return I4_ERR_LAUNCH;
  return ks > 1 ? launch_linear_finish(part, ks, M, w.N, bias, y, ot, s) : I4_OK;
}

#define I4_INST(XT_, ST_)                                                                    \
  template int launch_awq_mm<XT_, ST_>(const void*, int, const i4_qweight&, const void*,     \
                                       void*, int, float*, hipStream_t);
I4_INST(I4_F16, I4_F32) I4_INST(I4_F16, I4_F16) I4_INST(I4_F16, I4_BF16)
I4_INST(I4_BF16, I4_F32) I4_INST(I4_BF16, I4_F16) I4_INST(I4_BF16, I4_BF16)
#undef I4_INST

}  // namespace i4
