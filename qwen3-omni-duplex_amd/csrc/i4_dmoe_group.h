// Launch interface of the Talker block's grouped path (i4_dmoe_group.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "i4_dmoe.h"

namespace i4 {

static constexpr int DG_TOK = 64;     // tokens per entry
static constexpr int DG_CHUNK = 1024;  // tokens per pass: bounds the workspace (ys)

// entries of T tokens: sum over experts of ceil(n_e / DG_TOK)
inline size_t dg_max_entries(int T, int E, int topk) {
  const size_t p = (size_t)T * topk;
  return (p < (size_t)E ? p : (size_t)E) + p / DG_TOK;
}

struct DGCall {
  const uint16_t* x;  // [T][H], T <= DG_CHUNK
  int T, topk, E;
  const int32_t* sel;  // [T][topk]
  const float* wts;
  DW gu, dn, sgu, sdn;      // sgu.data NULL: no shared expert
  const uint16_t* sgate_w;  // [H] or NULL (gate 1)
  const uint16_t* residual;
  uint16_t* out;
  // workspace
  int32_t* perm;   // [T topk]
  int4* entries;   // [dg_max_entries]
  int* n_entries;
  uint16_t* act;   // [T topk][I]
  uint16_t* act_s; // [T][Is]
  float* ys;       // [T topk][H]
  float* ys_s;     // [T][H]
  int32_t* status;  // set to I4_OK (nullable)
};

// Whether the grouped kernels serve these weight formats (the int8 shared expert of a
// 16-bit block keeps the per-token kernels: no module builds one).
inline bool dg_formats(bool ri8, bool si8) { return ri8 || !si8; }

int i4_launch_dg(const DGCall& c, int xt, hipStream_t s);

}  // namespace i4
