// Sliding-window prefill attention for bf16 operands (swa_prefill.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/uttt_amd.h"

namespace uttt {

// An upper bound of the key splits a bf16 call makes, from the sizes that do not depend on how
// the heads share their keys.
int swa_prefill_mm_max_splits(int64_t batch, int64_t n_heads, int64_t q_len, int64_t kv_len, int64_t window);

// The splits of this call (1: the output is written; more: fp32 partials, part[b][h][split][q][2 +
// head_dim] with q_pad queries per split: row max, row sum, unnormalised output).
int swa_prefill_mm_splits(const uttt_swa_prefill_args& a);

void launch_swa_prefill_mm(const uttt_swa_prefill_args& a, float* part, int q_pad, hipStream_t st);

}  // namespace uttt
