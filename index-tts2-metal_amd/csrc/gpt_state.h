// gpt_state.h -- what the GPT decoder's kernels share (gpt.hip, gpt_token.hip):
// the device-side decode state and the model's fixed sizes.
#pragma once

#include <stdint.h>

#include "device_common.h"
#include "gemm.h"
#include "gpt.h"

namespace mit2hip {

constexpr int kW = kGptW, kQKV = 3840, kMLP = 5120, kHeads = 20, kHD = 64;
constexpr int kVocab = GptDecoder::kVocab, kPos = GptDecoder::kPositions;

// Device-side decode state.
struct GptState {
  int32_t kv;         // rows in the key/value caches
  int32_t step;       // decode steps taken
  int32_t n_pred;     // predicted tokens written
  int32_t n_in;       // input tokens written (the start token included)
  int32_t stopped;    // 1 once the stop token was predicted
  int32_t stop_step;  // step of the first stop token, else -1
  int32_t cur_token;  // the last input token
  int32_t hf;         // position rule: step s > 0 uses position s + 1
  int32_t argmax;     // argmax of the last head launch
  int32_t max_pred;   // capacity of the predicted array (inputs: + 1)
  int32_t cap;        // rows of each key/value cache
  int32_t rows;       // rows of the prefix buffer
  int32_t overflow;   // 1: a value of the row-product prefill did not fit a split f16 pair
  int32_t top_k;      // sampling (sample_kernel): top-k (0: off)
  float temperature;  //   temperature, top-p, repetition penalty
  float top_p;
  float penalty;
  int32_t n_hist;     //   repetition-history prefix tokens
  uint64_t rng;       //   splitmix64 state, advanced once per sampled step
  int32_t hist_given; //   1: the history starts with the caller's prefix (even an
                      //   empty one), 0: with the start token
  uint32_t epoch;     // tag epoch of step 0 (gpt_token.hip): step s uses epoch + s
  int32_t unfit;      // 1: a value of the resident step kernel did not fit one
  int32_t aborted;    // 1: a wait of the resident step kernel ran out
  int32_t pend;       // prefix rows the plain prefill's chunks cover (rows 0..pend-1)
  int32_t yield_signs;  // of other work on the GPU lately (gpt.hip, yield_gpu)
  uint32_t owed;        // and the ticks owed to it
  int32_t pad[5];

  // The logits are worthless: no token is picked from them.
  __host__ __device__ bool failed() const { return (overflow | unfit | aborted) != 0; }
};
static_assert(sizeof(GptState) == 128, "GptState layout");

}  // namespace mit2hip
