// gpt_prefill.hip -- LayerNorm and causal attention over the prefix rows of
// the GPT decoder (see gpt_prefill.h).  run_gpt_kv_prefill_cpu
// (runtime/impl/gpt.cpp:1796) pushes the rows through one at a time; here a
// layer takes up to kPrefillRows rows per launch.
#include "gpt_prefill.h"

#include "gemm.h"

namespace mit2hip {

namespace {

constexpr int kHeads = 20, kHD = 64;

// Four values as a split pair; reports one that is too large for it (or NaN).
// Returns their largest magnitude.
__device__ __forceinline__ float store_split4(half_t* dst, size_t lo, float4 v, int* overflow) {
  if (!(fabsf(v.x) <= kSplitMax && fabsf(v.y) <= kSplitMax && fabsf(v.z) <= kSplitMax && fabsf(v.w) <= kSplitMax))
    *overflow = 1;
  half_t h[4], l[4];
  split_f16(v.x, h[0], l[0]);
  split_f16(v.y, h[1], l[1]);
  split_f16(v.z, h[2], l[2]);
  split_f16(v.w, h[3], l[3]);
  *reinterpret_cast<half4*>(dst) = half4{h[0], h[1], h[2], h[3]};
  *reinterpret_cast<half4*>(dst + lo) = half4{l[0], l[1], l[2], l[3]};
  return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}

// cpu_layernorm (tokenizer_tests.cpp:2992-3010), one wave per row, the row in
// registers: two passes over them, eps 1e-5.
constexpr int kLnRows = 4;  // rows (waves) per block
__global__ __launch_bounds__(kLnRows * 64) void ln_rows_kernel(const float* x, const float* g, const float* b, int M,
                                                               half_t* y, size_t y_lo, int* overflow,
                                                               uint32_t* small, int sets, int stride) {
  constexpr int CH = kGptW / 256;  // float4 chunks per lane
  const int m = blockIdx.x * kLnRows + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (m >= M) return;
  float4 v[CH], gv[CH], bv[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) v[c] = reinterpret_cast<const float4*>(x + (size_t)m * kGptW)[lane + 64 * c];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    gv[c] = reinterpret_cast<const float4*>(g)[lane + 64 * c];
    bv[c] = reinterpret_cast<const float4*>(b)[lane + 64 * c];
  }
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) s += (v[c].x + v[c].y) + (v[c].z + v[c].w);
  const float mean = warp_sum(s) * (1.0f / kGptW);
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    v[c].x -= mean; v[c].y -= mean; v[c].z -= mean; v[c].w -= mean;
    q += (v[c].x * v[c].x + v[c].y * v[c].y) + (v[c].z * v[c].z + v[c].w * v[c].w);
  }
  const float inv = 1.0f / sqrtf(warp_sum(q) * (1.0f / kGptW) + 1e-5f);
  float big = 0.f;
#pragma unroll
  for (int c = 0; c < CH; ++c)
    big = fmaxf(big, store_split4(y + (size_t)m * kGptW + 4 * (lane + 64 * c), y_lo,
                                  make_float4(v[c].x * inv * gv[c].x + bv[c].x, v[c].y * inv * gv[c].y + bv[c].y,
                                              v[c].z * inv * gv[c].z + bv[c].z, v[c].w * inv * gv[c].w + bv[c].w),
                                  overflow));
  if (!__any(big >= kSplitFull) && __any(big > 0.f)) *overflow = 1;
  for (int i = lane; i < sets; i += 64) small[(size_t)i * stride + m] = 0u;  // (last: nothing waits for it)
}

// Block (head, 16 queries); its four waves take alternate 16-key tiles with a
// running softmax and merge at the end.  fp32 throughout, on the fp32 matrix
// instruction (16x16x4), which multiplies fp32 exactly as the vector units do:
//   S^T = K Q^T   16 steps; slot j = lane / 16 of step t is dim 16 j + t, so a
//                 lane's K and Q operands are 16 consecutive floats
//   O^T += V^T P  4 steps per 16 dims; slot j of step s is key 4 j + s, the
//                 key whose probability the lane already holds from S^T
// so the probabilities never cross lanes; only the running max does.  The
// arithmetic is small (116 MFLOP a layer at 213 rows); the time, 12 us, is the
// latency of the key tiles a wave walks in turn, hence four waves on 16
// queries and the longest rows first.
constexpr int kAttnWaves = 4;
constexpr int kOStride = kHD + 4;  // LDS row of a query's output (floats)
__global__ __launch_bounds__(kAttnWaves * 64) void attn_rows_kernel(const float* q, const float* kc, const float* vc,
                                                                    int cap, int kv0, int M, half_t* y, size_t y_lo,
                                                                    int* overflow, uint32_t* small) {
  __shared__ float sO[kAttnWaves][16][kOStride];
  __shared__ float sM[kAttnWaves][16], sL[kAttnWaves][16];
  const int h = blockIdx.x;
  const int q0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * 16;  // the longest rows first
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, j = lane >> 4;
  const float* kh = kc + (size_t)h * cap * kHD;
  const float* vh = vc + (size_t)h * cap * kHD;
  const int last = kv0 + min(q0 + 15, M - 1);  // the block's last visible key
  const int qpos = kv0 + q0 + lr;              // this lane's query sees keys <= qpos

  float qv[16];
  {
    const float4* src =
        reinterpret_cast<const float4*>(q + (size_t)min(q0 + lr, M - 1) * kGptW + h * kHD + 16 * j);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float4 t = src[u];
      qv[4 * u] = t.x * 0.125f;  // 1 / sqrt(64), exact
      qv[4 * u + 1] = t.y * 0.125f;
      qv[4 * u + 2] = t.z * 0.125f;
      qv[4 * u + 3] = t.w * 0.125f;
    }
  }
  float mx = -INFINITY, l = 0.f;
  floatx4 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = 16 * wave; k0 <= last; k0 += 16 * kAttnWaves) {
    float kv[16], vv[4][4];
    const float4* ks = reinterpret_cast<const float4*>(kh + (size_t)min(k0 + lr, last) * kHD + 16 * j);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float4 t = ks[u];
      kv[4 * u] = t.x; kv[4 * u + 1] = t.y; kv[4 * u + 2] = t.z; kv[4 * u + 3] = t.w;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int d = 0; d < 4; ++d) vv[s][d] = vh[(size_t)min(k0 + 4 * j + s, last) * kHD + 16 * d + lr];
    floatx4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 16; ++t) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[t], qv[t], sc, 0, 0, 0);
    float tm = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (k0 + 4 * j + r > qpos) sc[r] = -INFINITY;
      tm = fmaxf(tm, sc[r]);
    }
    tm = fmaxf(tm, __shfl_xor(tm, 16, kWave));
    tm = fmaxf(tm, __shfl_xor(tm, 32, kWave));
    const float mn = fmaxf(mx, tm);
    const float ms = mn == -INFINITY ? 0.f : mn;  // no visible key yet: every probability is 0
    const float alpha = expf(mx - ms);
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = expf(sc[r] - ms);
    l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));  // this lane's keys; summed over j below
    mx = mn;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      o[d] *= alpha;
#pragma unroll
      for (int s = 0; s < 4; ++s) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[s][d], p[s], o[d], 0, 0, 0);
    }
  }
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
  if (j == 0) {
    sM[wave][lr] = mx;
    sL[wave][lr] = l;
  }
#pragma unroll
  for (int d = 0; d < 4; ++d)  // O^T: dims 16 d + 4 j + r of query lr
    *reinterpret_cast<float4*>(&sO[wave][lr][16 * d + 4 * j]) = make_float4(o[d][0], o[d][1], o[d][2], o[d][3]);
  __syncthreads();
  // merge: thread -> query tid / 16, dims 4 (tid % 16) ..
  const int qi = threadIdx.x >> 4, d4 = (threadIdx.x & 15) * 4;
  if (q0 + qi >= M) return;
  float mm = sM[0][qi];
#pragma unroll
  for (int w = 1; w < kAttnWaves; ++w) mm = fmaxf(mm, sM[w][qi]);
  float L = 0.f;
  float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int w = 0; w < kAttnWaves; ++w) {
    const float f = expf(sM[w][qi] - mm);  // a wave without keys: m = -inf, factor 0
    const float4 ow = *reinterpret_cast<const float4*>(&sO[w][qi][d4]);
    L += f * sL[w][qi];
    O.x += f * ow.x; O.y += f * ow.y; O.z += f * ow.z; O.w += f * ow.w;
  }
  const float big = store_split4(y + (size_t)(q0 + qi) * kGptW + h * kHD + d4, y_lo,
                                 make_float4(O.x / L, O.y / L, O.z / L, O.w / L), overflow);
  // (16 lanes a query: one head's part of its row)
  const uint64_t full = __ballot(big >= kSplitFull) >> (lane & 48);
  if ((full & 0xffffu) == 0) {
    const uint64_t some = __ballot(big > 0.f) >> (lane & 48);
    if (lr == 0) count_small(small + q0 + qi, kHeads, (some & 0xffffu) != 0, overflow);
  }
}

}  // namespace

hipError_t launch_gpt_ln_rows(const float* x, const float* g, const float* b, int M, half_t* y, size_t y_lo,
                              int* overflow, hipStream_t s, uint32_t* small, int sets, int stride) {
  if (M <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(ln_rows_kernel, dim3((M + kLnRows - 1) / kLnRows), dim3(kLnRows * 64), 0, s, x, g, b, M, y, y_lo,
                     overflow, small, sets, stride);
  return hipGetLastError();
}

hipError_t launch_gpt_attn_rows(const float* q, const float* kc, const float* vc, int cap, int kv0, int M,
                                half_t* y, size_t y_lo, int* overflow, uint32_t* small, hipStream_t s) {
  if (M <= 0 || kv0 < 0 || kv0 + M > cap) return hipErrorInvalidValue;
  hipLaunchKernelGGL(attn_rows_kernel, dim3(kHeads, (M + 15) / 16), dim3(kAttnWaves * 64), 0, s, q, kc, vc, cap, kv0,
                     M, y, y_lo, overflow, small);
  return hipGetLastError();
}

}  // namespace mit2hip
