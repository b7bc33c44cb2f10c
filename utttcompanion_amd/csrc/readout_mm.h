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
  float* zp;   // fp32 (splits, B, tok_pad, D)
};

// The forward products of a chunk update (K rows through the cursor weights, Q rows through the read
// weights): the same products with two row sets.  Where both sets read the same weights they form
// one matrix of 2 tok_pad rows per batch row, so that a weight tile is read once for both.
struct UpdateMmArgs {
  int B, T, D, F;
  int tok_pad;
  const void* x[2];  // bf16 (B, T, D), token stride D: K, Q
  int64_t x_rs[2];
  const float* w_up[2];
  const float* w_gate[2];
  const float* w_down[2];
  int64_t w_rs[2];
  void* h[2];      // bf16 (B, tok_pad, F)
  float* u_store;  // fp32 (B, tok_pad, F): K rows' products
  float* g_store;
  float* zp;  // fp32 (2, splits, B, tok_pad, D)
  int splits;
};

// Splits of the update's down product, at most `most`.
int update_mm_splits(int64_t B, int64_t T, int64_t D, int64_t F, bool joint, int most);

void launch_update_up(const UpdateMmArgs& a, bool joint, hipStream_t st);
void launch_update_down(const UpdateMmArgs& a, bool joint, hipStream_t st);

// The two products of the readout.  The down product leaves readout_mm_splits partials for the LayerNorm
// to sum; where readout_mm_down is false, k_down_partial is the better one.
bool readout_mm_down(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32);
int readout_mm_splits(int64_t B, int64_t T, int64_t D, int64_t F, bool w_fp32);
void launch_readout_up(const ReadoutMmArgs& a, hipStream_t st);
void launch_readout_down(const ReadoutMmArgs& a, hipStream_t st);

}  // namespace uttt
