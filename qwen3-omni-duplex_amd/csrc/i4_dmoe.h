// Shared device code of the Talker block's kernels (i4_dmoe.hip, i4_dmoe_group.hip):
// stacked 16-bit / int8 weights, their row dot products and the activation staging.
#pragma once

#include "i4_common.h"

namespace i4 {

static constexpr int DWG = 256;   // threads per workgroup
static constexpr int DMAXC = 8;   // 16-byte chunks of one weight row held per lane
// polls of a single-launch down workgroup before it gives up (a launch whose
// workgroups are dispatched in block order never reaches it)
static constexpr int kHandPolls = 1 << 20;

struct DW {                // one stacked weight [E][N][K]
  const void* data;        // 16-bit values, or int8 when scale != NULL
  const uint16_t* scale;   // [E][N] in the activation dtype, or NULL
  int64_t es;              // elements per expert (N * K)
  int N, K;
};

template <int XT> __device__ inline float round_to(float v) {
  return Half<XT>::to_f32(Half<XT>::from_f32(v));
}

// 16 bytes at chunk c of row n of expert e (bpe bytes per element)
__device__ inline u32x4 drow16(const DW& w, int e, int n, int c, int bpe) {
  const char* row = (const char*)w.data + ((int64_t)e * w.es + (int64_t)n * w.K) * bpe;
  return ldg16(row + 16 * (int64_t)c);
}

template <int XT> __device__ inline float dot16(u32x4 w, u32x4 x, float a) {
  a = Half<XT>::dot2(w.x, x.x, a);
  a = Half<XT>::dot2(w.y, x.y, a);
  a = Half<XT>::dot2(w.z, x.z, a);
  return Half<XT>::dot2(w.w, x.w, a);
}

// byte B of w as a float (v_cvt_f32_ubyteB)
template <int B> __device__ inline float ubyte(u32 w) { return (float)((w >> (8 * B)) & 0xFFu); }

// 16 int8 weights against xf[0..3] (the chunk's 16 activations), xsum their sum
__device__ inline float dot_i8(u32x4 w, const f32x4* xf, float xsum, float a) {
  const u32 v[4] = {w.x ^ 0x80808080u, w.y ^ 0x80808080u, w.z ^ 0x80808080u,
                    w.w ^ 0x80808080u};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 x = xf[i];
    a += ubyte<0>(v[i]) * x.x;
    a += ubyte<1>(v[i]) * x.y;
    a += ubyte<2>(v[i]) * x.z;
    a += ubyte<3>(v[i]) * x.w;
  }
  return a - 128.f * xsum;
}

// Activation staging in LDS, K values of a row (K % 16 == 0):
//   xs   [K / 8]  u32x4  the raw halves (16-bit weights)
//   xf   [K / 4]  f32x4  the values in fp32 (int8 weights only, F32)
//   xsum [K / 16] float  the sum of each 16 values (F32)
// One 8-value unit u per call; the lanes holding units u and u ^ 1 must run
// the call together (the chunk sum pairs them with a lane swizzle).
template <int XT, bool F32>
__device__ inline void commit_unit(int u, u32x4 d, u32x4* xs, f32x4* xf, float* xsum) {
  xs[u] = d;
  if constexpr (F32) {
    const u32 w[4] = {d.x, d.y, d.z, d.w};
    float f[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = Half<XT>::to_f32((uint16_t)(w[i] & 0xFFFFu));
      f[2 * i + 1] = Half<XT>::to_f32((uint16_t)(w[i] >> 16));
    }
    xf[2 * u] = f32x4{f[0], f[1], f[2], f[3]};
    xf[2 * u + 1] = f32x4{f[4], f[5], f[6], f[7]};
    const float s = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
    const float o = __builtin_bit_cast(
        float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, s), 0x041F));  // lane ^ 1
    if ((u & 1) == 0) xsum[u >> 1] = s + o;
  }
}

// byte offsets of the staging arrays for K staged values, and their total
__host__ __device__ inline size_t stage_xf_off(int K) { return (size_t)K * 2; }
__host__ __device__ inline size_t stage_xsum_off(int K) { return (size_t)K * 6; }
__host__ __device__ inline size_t stage_bytes(int K, bool f32) {
  return f32 ? (size_t)K * 6 + (size_t)K / 4 : (size_t)K * 2;
}

// sigmoid(g_s . x) of token row xr (H values), the dot product and the sigmoid
// each rounded to the activation dtype as the reference's 16-bit Linear and
// sigmoid round them (fused_moe.py:139); 1 without a gate.  Every thread of
// the workgroup calls it and receives the value.
template <int XT>
__device__ inline float shared_gate_value(const uint16_t* sgate_w, const uint16_t* xr, int H) {
  __shared__ float s_d[DWG / 64];
  if (!sgate_w) return 1.f;
  float d = 0.f;
  for (int k = threadIdx.x; k < H; k += DWG)
    d += Half<XT>::to_f32(sgate_w[k]) * Half<XT>::to_f32(xr[k]);
  d = group_sum<64>(d);
  if ((threadIdx.x & 63) == 0) s_d[threadIdx.x >> 6] = d;
  __syncthreads();
  const float z = round_to<XT>((s_d[0] + s_d[1]) + (s_d[2] + s_d[3]));
  return round_to<XT>(1.f / (1.f + expf(-z)));
}

}  // namespace i4
