// The matrix products of the frozen readout over more than one 64-token block (readout_mm.hip):
// H = SiLU(X W_gate) * (X W_up) and Z partials = H W_down, bf16 activations, W in bf16 or fp32
// (rounded to bf16 on the way into the matrix units), fp32 accumulation.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace uttt {

struct ReadoutMmArgs {
  int B, T, D, F;
  int tok_pad;  // rows per batch row of H and of the partials (a multiple of 64, >= T)
  const void* x;  // bf16 (B, T, D), token stride D
  int64_t x_rs;
  const void* w_up;  // (B | 1, D, F)
  const void* w_gate;
  const void* w_down;  // (B | 1, F, D)
  int64_t w_rs;        // 0: shared
  bool w_fp32;
  void* h;     // bf16 (B, tok_pad, F)
  float* zp;   // fp32 (readout_mm_splits(..), B, tok_pad, D)
};

// How many partials the down product leaves for the LayerNorm to sum.
int readout_mm_splits(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32);

void launch_readout_mm(const ReadoutMmArgs& a, hipStream_t st);

}  // namespace uttt
