// The Talker block (i4_dmoe.hip) for many tokens: the tokens of one expert share one
// read of its rows.
//
// k_d_gate_up / k_d_down stream a routed expert's rows once per token, so a call of T
// tokens moves T x 19 MB through the caches (bf16, T = 700: 983 + 848 us).  Here
// k_dg_group sorts the (token, slot) pairs by expert and cuts them into entries of at
// most DG_TOK tokens, and a workgroup holds its rows of one expert in registers while
// the entry's tokens pass by in LDS: each weight byte is read once per entry.  The
// shared expert is one more expert that every token selects.
//
// Results are those of the per-token kernels bit for bit, so a token's output does not
// depend on the call it is part of.  That fixes the arithmetic: a row's dot product is
// split over L lanes (64, or 32 for down and int8 rows), lane l accumulating chunks l,
// l + L, ... in order, and the lanes are then added as a butterfly adds them (lane l
// with l ^ 1, then ^ 2, ^ 4 ...).  A matrix instruction adds in another order, so the
// products run on v_dot2 (int8: fp32 FMA on converted bytes, each conversion shared by
// four tokens).  What the per-token kernels spend most on beside the loads is that
// butterfly: 6 adds in every lane for one finished value.  With eight rows and several
// tokens per wave a halving butterfly does it: each step adds the same pairs but keeps
// half of the values in each lane, so the 64 values of 8 rows x 8 tokens cost 2.8
// instructions each and end one per lane.
//
// Bounds: up to about 150 tokens the weights (302 MB of bf16 experts at the Talker's
// size, all 128 hit), beyond that the dot2 rate.
#include "i4_dmoe_group.h"
#include "i4_halve.h"

namespace i4 {

// ---------------------------------------------------------------- grouping
// One workgroup: the (token, slot) pairs sorted by expert (perm) and cut into entries
// {expert, first position, tokens} of at most DG_TOK tokens.  The order of an expert's
// pairs is whatever the LDS counters give: every pair's result is its own.
__global__ __launch_bounds__(1024) void k_dg_group(const int32_t* __restrict__ sel, int pairs,
                                                   int E, int32_t* __restrict__ perm,
                                                   int4* __restrict__ entries,
                                                   int* __restrict__ n_entries,
                                                   int32_t* __restrict__ status) {
  __shared__ int s_cnt[512], s_next[512], s_wc[8], s_we[8];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (tid < 512) s_cnt[tid] = 0;
  if (status && tid == 0) *status = I4_OK;  // nothing in this path waits
  __syncthreads();
  for (int s0 = 0; s0 < pairs; s0 += 4096) {
    int e[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) e[u] = sel[min(s0 + 1024 * u + tid, pairs - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + 1024 * u + tid < pairs) atomicAdd(&s_cnt[e[u]], 1);
  }
  __syncthreads();
  int c = 0, ne = 0, ic = 0, ie = 0;
  if (wave < 8) {  // thread e < 512 owns expert e
    c = tid < E ? s_cnt[tid] : 0;
    ne = (c + DG_TOK - 1) / DG_TOK;
    ic = wave_incl_scan(c);
    ie = wave_incl_scan(ne);
    if (lane == 63) {
      s_wc[wave] = ic;
      s_we[wave] = ie;
    }
  }
  __syncthreads();
  if (wave < 8) {
    int bc = 0, be = 0;
    for (int w = 0; w < wave; ++w) {
      bc += s_wc[w];
      be += s_we[w];
    }
    const int off = bc + ic - c, eoff = be + ie - ne;
    s_next[tid] = off;
    for (int q = 0; q < ne; ++q)
      entries[eoff + q] = int4{tid, off + q * DG_TOK, min(DG_TOK, c - q * DG_TOK), 0};
    if (tid == 511) *n_entries = be + ie;
  }
  __syncthreads();
  for (int s0 = 0; s0 < pairs; s0 += 4096) {
    int e[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) e[u] = sel[min(s0 + 1024 * u + tid, pairs - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 1024 * u + tid;
      if (s < pairs) perm[atomicAdd(&s_next[e[u]], 1)] = s;
    }
  }
}

// ---------------------------------------------------------------- expert rows x tokens
struct DGArgs {
  const uint16_t* src;    // routed rows: x [T][H] (gate_up: pair p reads row p / topk) or
                          // act [pairs][I] (down: pair p reads row p)
  const uint16_t* src_s;  // shared rows [T][..]
  int topk, T;
  DW w, ws;               // routed and shared weights (ws.data NULL: no shared expert)
  const int32_t* perm;
  const int4* entries;
  const int* n_entries;
  void* dst;              // gate_up: act [pairs][I]; down: ys [pairs][H] fp32
  void* dst_s;            // gate_up: act_s [T][Is]; down: ys_s [T][H] fp32
  int tiles, tiles_s;     // row tiles of a routed / the shared expert
  int n_shared;           // blocks of the shared expert (first in the grid)
};

// tokens staged at a time (at most 35 KB of LDS)
constexpr int dg_stage(bool i8, bool gate_up, int nr) {
  return i8 ? (nr > 2 ? 4 : 8) : gate_up ? 8 : 16;
}

// geometry of one form: L lanes per row, 64 / L rows side by side in a wave, 8 rows per
// lane; TB tokens finish together
template <bool I8, bool GATEUP> struct DGForm {
  static constexpr int L = (I8 || !GATEUP) ? 32 : 64;
  static constexpr int HALVES = 64 / L;
  static constexpr int TB = L / 8;
  static constexpr int ROWS = 4 * 8 * HALVES / (GATEUP ? 2 : 1);  // rows (row pairs) per tile
};

// One entry (cnt tokens of expert e, pair ids or tokens through `id`) x one row tile.
// NR: chunks per lane.  id(s): pair id (token for the shared expert) of entry position s;
// row(id): its source row.
template <int XT, bool I8, bool GATEUP, int NR, class Id, class Row>
__device__ inline void dg_body(const DW& w, int e, int tile, int cnt, Id id, Row row,
                               const uint16_t* __restrict__ src, void* __restrict__ dst,
                               unsigned char* lds) {
  using F = DGForm<I8, GATEUP>;
  constexpr int L = F::L, TB = F::TB, STG = dg_stage(I8, GATEUP, NR);
  constexpr int CPT = L * NR;                         // chunks per token
  constexpr int WPC = I8 ? 2 : 1;                     // staged 16-byte words per chunk
  constexpr int WPTK = CPT * WPC;                     // words per token
  constexpr int NW = STG * WPTK / 256;                // words per thread and stage
  static_assert(STG * WPTK % 256 == 0 && STG % TB == 0, "whole words per thread");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cl = lane & (L - 1), half = L == 64 ? 0 : lane >> 5;
  const int K = w.K, CH = K / (I8 ? 16 : 8);
  const int NO = GATEUP ? w.N >> 1 : w.N;             // output columns
  // the rows of this lane: r = 2 q + (up) of pair q, or row r
  const int n0 = tile * F::ROWS + (wave * F::HALVES + half) * (GATEUP ? 4 : 8);
  auto row_of = [&](int r) {
    if constexpr (GATEUP) return (r & 1) * NO + min(n0 + (r >> 1), NO - 1);
    else return min(n0 + r, NO - 1);
  };
  __shared__ int s_id[DG_TOK];
  if ((int)threadIdx.x < DG_TOK) s_id[threadIdx.x] = id(min((int)threadIdx.x, cnt - 1));
  u32x4 wv[8][NR];
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int i = 0; i < NR; ++i)
      wv[r][i] = drow16(w, e, row_of(r), min(cl + i * L, CH - 1), I8 ? 1 : 2);
  float sc = 1.f;  // the scale of the row this lane finishes
  if constexpr (I8) sc = Half<XT>::to_f32(w.scale[(int64_t)e * w.N + row_of(lane & 7)]);
  __syncthreads();
  // staging: word q = tid + 256 u of the stage is word q % WPTK of token q / WPTK
  const int units = K >> 3;
  u32x4 xd[NW];
  auto load_x = [&](int s0) {
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const int q = (int)threadIdx.x + 256 * u, t = q / WPTK, m = q - t * WPTK;
      const int s = min(s0 + t, cnt - 1);
      xd[u] = ldg16(src + (int64_t)row(s_id[s]) * K + 8 * min(m, units - 1));
      if (m >= units) xd[u] = u32x4{0u, 0u, 0u, 0u};
    }
  };
  u32x4* xs = (u32x4*)lds;            // 16-bit: [STG][CPT] words
  f32x4* xf = (f32x4*)lds;            // int8: [STG][4][CPT], values 4 j .. of chunk c
  float* xsum = (float*)(lds + (size_t)STG * CPT * 64);  // int8: [STG][CPT]
  auto commit_x = [&]() {
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const int q = (int)threadIdx.x + 256 * u;
      if constexpr (!I8) {
        xs[q] = xd[u];
      } else {
        const int t = q / WPTK, m = q - t * WPTK, c = m >> 1;
        const u32 d[4] = {xd[u].x, xd[u].y, xd[u].z, xd[u].w};
        float f[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f[2 * i] = Half<XT>::to_f32((uint16_t)(d[i] & 0xFFFFu));
          f[2 * i + 1] = Half<XT>::to_f32((uint16_t)(d[i] >> 16));
        }
        f32x4* o = xf + (int64_t)(t * 4 + 2 * (m & 1)) * CPT + c;
        o[0] = f32x4{f[0], f[1], f[2], f[3]};
        o[CPT] = f32x4{f[4], f[5], f[6], f[7]};
        // the chunk sum in commit_unit's order (i4_dmoe.h)
        const float s = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
        const float s1 = s + dpp_mov<0xB1>(s);
        if ((m & 1) == 0) xsum[t * CPT + c] = s1;
      }
    }
  };
  if (CH < CPT) {  // lanes past the row's end multiply zeros
#pragma unroll
    for (int i = 0; i < NR; ++i)
      if (cl + i * L >= CH) {
#pragma unroll
        for (int r = 0; r < 8; ++r) wv[r][i] = u32x4{0u, 0u, 0u, 0u};
      }
  }
  if constexpr (I8) {  // q + 128 as an unsigned byte (past the end: 128 x 0)
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int i = 0; i < NR; ++i) wv[r][i] ^= u32x4{0x80808080u, 0x80808080u, 0x80808080u,
                                                     0x80808080u};
  }
  load_x(0);
  for (int s0 = 0; s0 < cnt; s0 += STG) {
    commit_x();
    __syncthreads();
    if (s0 + STG < cnt) load_x(s0 + STG);
#pragma unroll 1
    for (int b = 0; b < STG && s0 + b < cnt; b += TB) {
      float pv[TB];  // per token: row lane & 7 summed over lane bits 0..2
      if constexpr (!I8) {
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          pv[t] = 0.f;
          if (s0 + b + t < cnt) {
            float acc[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) acc[r] = 0.f;
#pragma unroll
            for (int i = 0; i < NR; ++i) {
              const u32x4 x = xs[(b + t) * CPT + cl + i * L];
#pragma unroll
              for (int r = 0; r < 8; ++r) acc[r] = dot16<XT>(wv[r][i], x, acc[r]);
            }
            pv[t] = halve_rows(acc, lane);
          }
        }
      } else {
        float acc[TB][8];
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
          for (int r = 0; r < 8; ++r) acc[t][r] = 0.f;
        // the bytes stay bytes: converted once for the whole loop they would take four
        // times the registers
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
          for (int i = 0; i < NR; ++i) asm volatile("" : "+v"(wv[r][i]));
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const int c = cl + i * L;
#pragma unroll
          for (int h = 0; h < 2; ++h) {  // 8 of the chunk's 16 values at a time
            f32x4 x[TB][2];
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
              for (int j = 0; j < 2; ++j) x[t][j] = xf[((b + t) * 4 + 2 * h + j) * CPT + c];
#pragma unroll
            for (int r = 0; r < 8; ++r) {
              const u32 w2[2] = {h ? wv[r][i].z : wv[r][i].x, h ? wv[r][i].w : wv[r][i].y};
              float f[8];
#pragma unroll
              for (int k = 0; k < 2; ++k) {
                f[4 * k] = ubyte<0>(w2[k]);
                f[4 * k + 1] = ubyte<1>(w2[k]);
                f[4 * k + 2] = ubyte<2>(w2[k]);
                f[4 * k + 3] = ubyte<3>(w2[k]);
              }
#pragma unroll
              for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                  acc[t][r] += f[4 * k] * x[t][k].x;
                  acc[t][r] += f[4 * k + 1] * x[t][k].y;
                  acc[t][r] += f[4 * k + 2] * x[t][k].z;
                  acc[t][r] += f[4 * k + 3] * x[t][k].w;
                }
            }
          }
#pragma unroll
          for (int t = 0; t < TB; ++t) {
            const float s = xsum[(b + t) * CPT + c];
#pragma unroll
            for (int r = 0; r < 8; ++r) acc[t][r] -= 128.f * s;
          }
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) pv[t] = halve_rows(acc[t], lane);
      }
      // tokens over the remaining lane bits
      float v;
      if constexpr (TB == 8) {
        v = halve_tokens(pv, lane);
      } else {
        v = halve<4>(halve<3>(pv[0], pv[1], lane), halve<3>(pv[2], pv[3], lane), lane);
      }
      if constexpr (I8) v *= sc;
      const int s = s0 + b + ((lane >> 3) & (TB - 1));
      if constexpr (GATEUP) {
        const float u = dpp_mov<0xB1>(v);  // the pair's up row sits one lane on
        const int n = n0 + ((lane >> 1) & 3);
        if ((lane & 1) == 0 && s < cnt && n < NO)
          ((uint16_t*)dst)[(int64_t)s_id[s] * NO + n] = Half<XT>::from_f32(silu(v) * u);
      } else {
        const int n = n0 + (lane & 7);
        if (s < cnt && n < NO) ((float*)dst)[(int64_t)s_id[s] * NO + n] = v;
      }
    }
    __syncthreads();
  }
}

// Blocks [0, n_shared): the shared expert (row tile b % tiles_s of tokens DG_TOK (b /
// tiles_s) ..), then the routed entries (sized for the worst case; past *n_entries they
// exit).  The shared expert's full entries go first: they are the longest workgroups.
template <int XT, bool RI8, bool SI8, bool GATEUP, int NRR, int NRS>
__global__ __launch_bounds__(256) void k_dg(DGArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  int b = blockIdx.x;
  if (b < a.n_shared) {
    const int t0 = b / a.tiles_s * DG_TOK;
    dg_body<XT, SI8, GATEUP, NRS>(a.ws, 0, b % a.tiles_s, min(DG_TOK, a.T - t0),
                                  [&](int s) { return t0 + s; }, [](int p) { return p; },
                                  a.src_s, a.dst_s, lds);
    return;
  }
  b -= a.n_shared;
  const int en = b / a.tiles;
  if (en >= *a.n_entries) return;
  const int4 q = a.entries[en];
  const int topk = a.topk;
  dg_body<XT, RI8, GATEUP, NRR>(
      a.w, q.x, b % a.tiles, q.z, [&](int s) { return a.perm[q.y + s]; },
      [&](int p) { return GATEUP ? p / topk : p; }, a.src, a.dst, lds);
}

// out[t] = sum_j w_j ys[t][j] + sg ys_s[t] (+ residual), k_d_down's order and arithmetic;
// one token per workgroup, which also makes the token's shared gate.
template <int XT>
__global__ __launch_bounds__(DWG) void k_dg_combine(const float* __restrict__ ys,
                                                    const float* __restrict__ ys_s,
                                                    const float* __restrict__ wts, int topk,
                                                    int H, const uint16_t* __restrict__ x,
                                                    const uint16_t* __restrict__ sgate_w,
                                                    const uint16_t* __restrict__ residual,
                                                    uint16_t* __restrict__ out) {
  const int64_t t = blockIdx.x;
  float sg = 0.f;
  if (ys_s) sg = shared_gate_value<XT>(sgate_w, x + t * H, H);
  float wj[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) wj[j] = wts[t * topk + min(j, topk - 1)];
  for (int n = 4 * (int)threadIdx.x; n < H; n += 4 * DWG) {
    f32x4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = *(const f32x4*)(ys + (t * topk + min(j, topk - 1)) * (int64_t)H + n);
    f32x4 vs = {0.f, 0.f, 0.f, 0.f};
    if (ys_s) vs = *(const f32x4*)(ys_s + t * H + n);
    u32x2 rr = {0u, 0u};
    if (residual) rr = *(const u32x2*)(residual + t * H + n);
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (j < topk) s += wj[j] * v[j][i];
      if (ys_s) s += sg * vs[i];
      const u32 rw = i < 2 ? rr.x : rr.y;
      if (residual) s += Half<XT>::to_f32((uint16_t)(rw >> (16 * (i & 1))));
      o[i] = Half<XT>::from_f32(s);
    }
    *(u32x2*)(out + t * H + n) =
        u32x2{(u32)o[0] | ((u32)o[1] << 16), (u32)o[2] | ((u32)o[3] << 16)};
  }
}

// ---------------------------------------------------------------- host
namespace {

// chunks per lane of a K-value row (at most 4: the caller's shape limits)
int dg_rounds(int K, bool i8, bool gate_up) {
  const int L = (i8 || !gate_up) ? 32 : 64, ch = K / (i8 ? 16 : 8);
  return (ch + L - 1) / L;
}

size_t dg_lds(int nr, bool i8, bool gate_up) {
  const int L = (i8 || !gate_up) ? 32 : 64;
  return (size_t)dg_stage(i8, gate_up, nr) * L * nr * (i8 ? 64 + 4 : 16);
}

// the template's step for nr rounds of the routed / the shared rows; gate_up rows are H
// values in both formats, so they have the same rounds (H / 512)
int dg_step(int nr) { return nr <= 1 ? 1 : nr <= 2 ? 2 : 4; }
int dg_step_s(int nr, bool gate_up) { return gate_up ? dg_step(nr) : nr <= 3 ? 3 : 4; }

template <int XT, bool RI8, bool SI8, bool GATEUP>
int dg_launch(DGArgs a, int max_entries, hipStream_t s) {
  using FR = DGForm<RI8, GATEUP>;
  using FS = DGForm<SI8, GATEUP>;
  const int nrr = dg_step(dg_rounds(a.w.K, RI8, GATEUP));
  int nrs = dg_step_s(0, GATEUP);
  if (GATEUP) nrs = nrr;
  a.tiles = ((GATEUP ? a.w.N >> 1 : a.w.N) + FR::ROWS - 1) / FR::ROWS;
  a.tiles_s = 1;
  a.n_shared = 0;
  size_t lds = dg_lds(nrr, RI8, GATEUP);
  if (a.ws.data) {
    nrs = dg_step_s(dg_rounds(a.ws.K, SI8, GATEUP), GATEUP);
    a.tiles_s = ((GATEUP ? a.ws.N >> 1 : a.ws.N) + FS::ROWS - 1) / FS::ROWS;
    a.n_shared = a.tiles_s * ((a.T + DG_TOK - 1) / DG_TOK);
    lds = max(lds, dg_lds(nrs, SI8, GATEUP));
  }
  const unsigned grid = (unsigned)a.n_shared + (unsigned)a.tiles * (unsigned)max_entries;
#define I4_DG(R_, S_)                                                                            if (nrr == R_ && nrs == S_) {                                                                    hipLaunchKernelGGL((k_dg<XT, RI8, SI8, GATEUP, R_, S_>), dim3(grid), dim3(256), lds, s, a);     return hipGetLastError() == hipSuccess ? I4_OK : I4_ERR_LAUNCH;                              }
  if constexpr (GATEUP) {
    I4_DG(1, 1) I4_DG(2, 2) I4_DG(4, 4)
  } else {
    I4_DG(1, 3) I4_DG(2, 3) I4_DG(4, 3) I4_DG(1, 4) I4_DG(2, 4) I4_DG(4, 4)
  }
#undef I4_DG
  return I4_ERR_SHAPE;
}

}  // namespace

int i4_launch_dg(const DGCall& c, int xt, hipStream_t s) {
  const int pairs = c.T * c.topk;
  hipLaunchKernelGGL(k_dg_group, dim3(1), dim3(1024), 0, s, c.sel, pairs, c.E, c.perm,
                     c.entries, c.n_entries, c.status);
  if (hipGetLastError() != hipSuccess) return I4_ERR_LAUNCH;
  const int max_entries = (int)dg_max_entries(c.T, c.E, c.topk);
  DGArgs g;
  g.src = g.src_s = c.x;
  g.topk = c.topk;
  g.T = c.T;
  g.w = c.gu;
  g.ws = c.sgu;
  g.perm = c.perm;
  g.entries = c.entries;
  g.n_entries = c.n_entries;
  g.dst = c.act;
  g.dst_s = c.act_s;
  DGArgs d = g;
  d.src = c.act;
  d.src_s = c.act_s;
  d.w = c.dn;
  d.ws = c.sdn;
  d.dst = c.ys;
  d.dst_s = c.ys_s;
  const bool ri8 = c.gu.scale != nullptr, si8 = c.sgu.data && c.sgu.scale;
  int rc = I4_ERR_DTYPE;
#define I4_DG_CASE(XT_, R_, S_)                                                     \
  if (xt == XT_ && ri8 == R_ && si8 == S_) {                                        \
    rc = dg_launch<XT_, R_, S_, true>(g, max_entries, s);                           \
    if (rc == I4_OK) rc = dg_launch<XT_, R_, S_, false>(d, max_entries, s);         \
  }
  I4_DG_CASE(I4_F16, false, false)
  I4_DG_CASE(I4_F16, true, false)
  I4_DG_CASE(I4_F16, true, true)
  I4_DG_CASE(I4_BF16, false, false)
  I4_DG_CASE(I4_BF16, true, false)
  I4_DG_CASE(I4_BF16, true, true)
#undef I4_DG_CASE
  if (rc != I4_OK) return rc;
  const int H = c.dn.N;
  const float* ys_s = c.sgu.data ? c.ys_s : nullptr;
  if (xt == I4_F16)
    hipLaunchKernelGGL(k_dg_combine<I4_F16>, dim3(c.T), dim3(DWG), 0, s, c.ys, ys_s, c.wts,
                       c.topk, H, c.x, c.sgate_w, c.residual, c.out);
  else
    hipLaunchKernelGGL(k_dg_combine<I4_BF16>, dim3(c.T), dim3(DWG), 0, s, c.ys, ys_s, c.wts,
                       c.topk, H, c.x, c.sgate_w, c.residual, c.out);
  return hipGetLastError() == hipSuccess ? I4_OK : I4_ERR_LAUNCH;
}

}  // namespace i4
