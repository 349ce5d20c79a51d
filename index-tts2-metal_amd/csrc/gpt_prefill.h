// gpt_prefill.h -- row kernels of the GPT decoder's prefill (gpt_prefill.hip):
// the prefix rows go through each layer together, as split f16 pairs on the
// matrix cores (launch_gemm_rows) between these LayerNorm and attention
// kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.h"

namespace mit2hip {

// y = LayerNorm(x) of M rows of kGptW floats, written as a split f16 pair
// (y, its lo half at y + y_lo).  Sets *overflow when a row does not fit (see
// kSplitMax, kSplitFull).  Clears `sets` counts of each row, small[set * stride +
// row] (count_small), for the kernels behind it.
hipError_t launch_gpt_ln_rows(const float* x, const float* g, const float* b, int M, half_t* y, size_t y_lo,
                              int* overflow, hipStream_t s, uint32_t* small = nullptr, int sets = 0, int stride = 0);

// Causal attention of M query rows q [M][kGptW] at cache rows kv0 .. kv0 + M - 1
// over the head-major caches [heads][cap][64], which already hold those rows:
// row m sees keys 0 .. kv0 + m.  The output is a split f16 pair as above; the
// heads' parts of a row that are all small are counted at small[m].
hipError_t launch_gpt_attn_rows(const float* q, const float* kc, const float* vc, int cap, int kv0, int M,
                                half_t* y, size_t y_lo, int* overflow, uint32_t* small, hipStream_t s);

}  // namespace mit2hip
