// gpt_token.h -- one GPT decode step as a single resident kernel (gpt_token.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "gpt_state.h"

namespace mit2hip {

constexpr int kTokWG = 256;     // workgroups, one per CU, all resident at once
constexpr int kTokSplits = 4;   // workgroups that share a head's keys
constexpr int kTokHeadRows = (kVocab + kTokWG - 1) / kTokWG;  // mel_head rows per workgroup

// The words the workgroups hand each other (see gpt_token.hip).
constexpr int kTokAttRow = 80;  // words of a head's part: 64 sums, max, exp-sum, unused
// The slots of two workgroups share no 64-byte line: a line that several
// workgroups write while all poll it goes back and forth between the caches.
constexpr int kTokXSlot = 8;    // words of a workgroup's residual-stream slot (5 used)
constexpr int kTokFSlot = 24;   // ... of its c_fc slot (20 used)
struct TokenMail {
  alignas(128) uint64_t xa[kTokWG * kTokXSlot];  // the residual stream after a layer
  alignas(128) uint64_t xb[kTokWG * kTokXSlot];  // ... after its attention
  alignas(128) uint64_t qkv[kQKV];
  alignas(128) uint64_t att[kTokSplits * kHeads * kTokAttRow];
  alignas(128) uint64_t fc[kTokWG * kTokFSlot];
};

struct TokenArgs {
  // layer 0's arrays; layer l's are l * stride bytes further
  const char *ln1_w, *ln1_b, *attn_w, *attn_b, *proj_w, *proj_b, *ln2_w, *ln2_b, *fc_w, *fc_b, *mp_w, *mp_b;
  size_t stride;
  int L;
  const float *lnf_w, *lnf_b, *fn_w, *fn_b, *head_b, *mel_emb, *pos_emb;
  const half_t* head_w;
  GptState* st;
  float *kc, *vc;  // [L][heads][cap][64]
  int cap;
  TokenMail* mail;
  float* logits;
  float* blk_val;  // [kTokWG] first maximum of each workgroup's logits and its row
  int* blk_idx;
  uint32_t* start;  // [kTokWG] when each workgroup started (device_ticks)
  uint32_t spin_limit;  // polls a wait may take (0.2 us each)
};

// The device's constant clock: ticks of 10 ns.
__device__ __forceinline__ uint32_t device_ticks() {
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint32_t)__builtin_amdgcn_s_memrealtime();
#else
  return 0;
#endif
}

// Whether every workgroup of the kernel fits the device at once.
bool gpt_token_fits(int device);

// Embeds the state's current token, runs the layers and the head; appends the
// token's key and value rows to the caches and advances st->kv.  The caller
// keeps any two launches on a device from overlapping.
hipError_t launch_gpt_token(const TokenArgs& a, hipStream_t s);

}  // namespace mit2hip
