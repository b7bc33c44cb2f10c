// The bf16 chunk update's backward pass and state write (update_mm.hip); fp32 masters.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace uttt {

struct UpdateBackArgs {
  int B, C, D, F, ntb, tok_pad;  // ntb token blocks of 64, tok_pad = 64 ntb
  const void* k;                 // bf16 (B, C, D), token stride D
  int64_t k_rs;
  const float* w_down;  // (B, F, D)
  const float* u;       // fp32 (B, tok_pad, F): the K path's products
  const float* g;
  const void* h;   // bf16 (B, tok_pad, F)
  const void* dz;  // bf16 (B, tok_pad, D), rows past C zero
  void* du;        // bf16 (B, tok_pad, F)
  void* dg;
  float* nrm;  // (B, F / 64): squared gradient norm of each F tile, one token block only
};
void launch_update_back(const UpdateBackArgs& a, hipStream_t st);

struct UpdateWriteArgs {
  int B, C, D, F, ntb, tok_pad;
  const void* k;
  int64_t k_rs;
  const void* h;
  const void* dz;
  const void* du;
  const void* dg;
  const float* w[3];
  const float* s[3];
  float* w_out[3];
  float* s_out[3];
  float beta;
  // several token blocks: the row scalars (B, 4) = clip factor, decay, active flag, and the norm
  // form's output, (B, 3 (D / 64) (F / 64)) squared norms of the gradient tiles
  const float* scalars;
  float* nrm;
  // one token block: what the write forms the row scalars from (scalars null)
  const float* tile_nrm;  // (B, F / 64), k_update_back's
  const void* alpha;      // bf16 (B, C)
  int64_t alpha_rs;
  const float* mask;  // (B, C) or null
  int64_t mask_rs;
  const float* loss;  // (B, 64)
  float max_norm, min_row_surprise;
  float* surprise;
  float* row_loss;  // (B, 2) or null
};
// The squared norm of every gradient tile (more than one token block), and the state write.
void launch_update_norm(const UpdateWriteArgs& a, hipStream_t st);
void launch_update_write(const UpdateWriteArgs& a, hipStream_t st);

}  // namespace uttt
