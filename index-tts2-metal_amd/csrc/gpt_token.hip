// gpt_token.hip -- one GPT decode step as a single resident kernel.
//
// A step is 24 layers of five dependent phases (qkv, attention, projection,
// c_fc, mlp projection), each a few MB of weights.  As separate launches each
// phase pays for its launch, the ramp of its loads and their drain, and HBM
// idles meanwhile.  Here 256 workgroups, one per CU, stay for the whole step:
// each owns fixed rows of every matrix (15, 5, 20 and 5 a layer), and its
// waves load a phase's rows of the *next* layer into the registers that the
// phase has just used, so about a layer's weights (39 MB over the chip) are
// always in flight and no phase waits for HBM.
//
// What bounds it: the hand-overs, five a layer.  A code takes 0.38 ms at 150
// cached rows and 0.43 at 700 (15 us a layer), where the separate launches take
// 0.65 and 0.71; 0.965 GB of weights at 4.8 TB/s would be 0.20.  Without the
// weight loads it takes 0.33 at either, so HBM is nearly hidden; a hand-over to
// all 256 workgroups takes 0.9 us at best (of one word between two of them: 0.5).
//
// Hand-over between workgroups.  A value that another workgroup needs is
// stored as one 64-bit word, its tag (step and layer) above its bits, with a
// relaxed agent-scope atomic store; readers poll the words themselves until
// the tags match.  The word carries its own proof of being new, so nothing
// depends on the order of two different words and no fence, counter or
// second round trip is needed (a release fence writes back the whole L2; a
// counter costs two more trips to the coherence point).  A word is reused a
// layer later: its owner gets there only after reading values that every
// workgroup made after it had read the word's last value.
//
// Waits are bounded: a wave that polls spin_limit times without success sets
// st->aborted and stops waiting, as does every wave that sees the flag, so the
// kernel always ends; the host then decodes with the separate launches.
//
// Workgroup: 16 waves of three kinds, each with its own loop over the layers
// (so that one kind's waits do not bind another's), meeting at LDS barriers:
//   waves 0-9    products.  Wave w takes the K slice [K w / 10, K (w + 1) / 10)
//                of all the workgroup's rows; the partial sums meet in LDS and
//                wave 0 finishes them
//   waves 10-14  poll the phase's input vector into LDS (the residual stream four
//                of them, with the LayerNorm statistics of each wave's 320
//                values); four do the attention's arithmetic (80 workgroups: 20
//                heads in 4 parts)
//   wave 15      brings the LayerNorm weights and biases, the products' biases and
//                the keys and values of the workgroup's part of a head into LDS a
//                layer ahead
#include "gpt_token.h"

#include <type_traits>

namespace mit2hip {

namespace {

constexpr int kCW = 10, kPW = 5, kKW = 1;  // product, poll and key waves
constexpr int kThreads = 64 * (kCW + kPW + kKW);
constexpr int kRQ = kQKV / kTokWG, kRP = kW / kTokWG, kRF = kMLP / kTokWG;  // rows per workgroup
static_assert(kRQ == 15 && kRP == 5 && kRF == 20, "the matrix-core blocks below");
constexpr int kXW = 4;                          // poll waves of the residual stream, a workgroup's slot a lane third
constexpr int kPoll = kW / kXW;                 // their values
static_assert(kXW * 64 == kTokWG, "64 slots a wave");
constexpr int kAttnWG = kHeads * kTokSplits;
constexpr int kLdsKeys = 208;                   // keys of a split held in LDS
constexpr int kAW = 4;                          // poll waves that walk the keys
constexpr int kAU = 4;                          // key groups a wave reads together
// K steps of 32 and how a product's rows fill the 16 rows of a block:
//  block of 16 (c_attn's 15 rows, c_fc's and the head's first ones): kStepsW
//  steps, kSW a wave
//  5 rows x 3 ranges of K (the projections): range r's rows are rows 5 r .. of
//  the block, the ranges kR3W / kR3F wide (past K: zeros), kS3W / kS3F a wave
//  4 rows x 4 ranges (c_fc's last rows): ranges of kR4, one step a wave
constexpr int kSW = kW / 32 / kCW, kR3W = 448, kS3W = 2, kR3F = 1728, kS3F = 6, kR4 = kW / 4;
static_assert(kSW * kCW * 32 == kW && kR4 == 32 * kCW, "whole steps per wave");
static_assert(3 * kR3W >= kW && kS3W * kCW * 32 >= kR3W && 3 * kR3F >= kMLP && kS3F * kCW * 32 >= kR3F, "ranges");
static_assert(kTokHeadRows <= 36, "the head's rows use the blocks of c_attn and c_fc");
// Clocks / 64 that a phase's poll waits before its first look: about as long as
// its words take at best (poll says why).  ms a code at 20 / 150 / 400 / 700 /
// 1,500 cached rows, all of them
//   not at all       0.461 0.467 0.482 0.508 0.605
//   x 0.5            0.404 0.412 0.432 0.450 0.547
//   x 0.75           0.384 0.389 0.418 0.434 0.531
//   as here          0.376 0.377 0.412 0.431 0.525
//   x 1.25           0.382 0.382 0.408 0.430 0.523
//   x 1.5            0.395 0.395 0.409 0.435 0.530
//   the attention's (which takes longer with the rows) x 1.5, the others as here
//                    0.386 0.385 0.404 0.432 0.526
constexpr int kSleepXa = 56, kSleepQ = 4, kSleepAtt = 32, kSleepXb = 32, kSleepFc = 40;
constexpr int kSleepIdle = 96;  // ... the attention's, more where a workgroup has no part in it

struct Lds {  // (the small arrays first: LDS instructions hold 64 KB offsets)
  alignas(16) half_t x[2][3 * kR3W];   // the phase's input vector as a split pair (hi, lo), zeros past kW
  half_t xf[2][3 * kR3F];  // ... the mlp projection's, zeros past kMLP
  float ln[2][2][kW];      // ln_1 / ln_2 (ln_f / final_norm): weight, bias
  float part[kCW][3][16];  // a wave's products: block, row
  float bias[2][4][64];    // by layer parity: the workgroup's rows of the four products' (or the head's) bias
  float q[3 * kHD];        // this head's q, and the new key and value
  float xr[8];             // the residual stream at the workgroup's rows
  float o[4 * kAW][kHD];
  float ml[4 * kAW][2];
  float stat[2][kXW][2];  // (mean, sum of squared deviations) of equal parts of x
  int holds[4][kPW];      // what each poll wave's part of a phase's input holds
  alignas(1024) float k[kLdsKeys * kHD];
  float v[kLdsKeys * kHD];
};
// (a larger one would not launch, and every step would silently be plain)
static_assert(sizeof(Lds) <= 160 * 1024, "the LDS of a CU");

// LDS barrier: orders this wave's LDS accesses only (a full fence would also
// wait for the weights in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The key waves' barrier: their only LDS accesses are loads straight into it,
// which they wait for where it matters (a fence would wait at every barrier).
__device__ __forceinline__ void bare_barrier() {
  __asm__ volatile("" : : : "memory");
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" : : : "memory");
}

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// Sum over a lane's 16-lane row, in every lane (row rotations).
__device__ __forceinline__ float sum16(float v) {
  v = dpp_add<0x128>(v);
  v = dpp_add<0x124>(v);
  v = dpp_add<0x122>(v);
  return dpp_add<0x121>(v);
}
__device__ __forceinline__ float max16(float v) {
  auto step = [](float x, auto c) {
    return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(c)::value, 0xf, 0xf, false)));
  };
  v = step(v, std::integral_constant<int, 0x128>{});
  v = step(v, std::integral_constant<int, 0x124>{});
  v = step(v, std::integral_constant<int, 0x122>{});
  return step(v, std::integral_constant<int, 0x121>{});
}
__device__ __forceinline__ float lane_of(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// Sum over the wave (uniform): the rows' sums, rows 0 and 2 into 1 and 3, then 1 into 3.
__device__ __forceinline__ float sum64(float v) {
  v = sum16(v);
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xa, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xc, 0xf, false));
  return lane_of(v, 63);
}

__device__ __forceinline__ uint64_t word(float v, uint32_t tag) {
  return ((uint64_t)tag << 32) | (uint32_t)__float_as_int(v);
}
__device__ __forceinline__ void put(uint64_t* p, float v, uint32_t tag) {
  __hip_atomic_store(p, word(v, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Two neighbouring words (each is read whole; which of the two is older does
// not matter), past the CU's own cache, as an agent-scope load is.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 get2(buffer_rsrc_t r, int byte) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_raw_buffer_load_b128(r, byte, 0, 16);  // 16: sc1
#else
  return u32x4{};
#endif
}

// Reads the word pairs at byte offsets off(i), i < N, of `base` until all carry
// `tag`.  A poll ahead of the data costs more than it gains: it brings the
// line into every XCD's L2, from where the store that follows has to recall
// it, so the wave first sleeps kSleep x 64 clocks, about as long as the words
// take at best.  `dead` (uniform): a wait has run out, nothing is waited for.
template <int N, int kSleep, typename F>
__device__ __forceinline__ void poll(const uint64_t* base, int bytes, F off, uint32_t tag, float (&v)[2 * N],
                                     bool& dead, const TokenArgs& a) {
  const buffer_rsrc_t rs = make_buffer_rsrc(base, bytes);
  __builtin_amdgcn_s_sleep(kSleep);
  u32x4 r[N];
  auto look = [&]() {
    __asm__ volatile("" : : : "memory");  // new loads each time
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = get2(rs, off(i));
    __asm__ volatile("" : : : "memory");
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && r[i][1] == tag && r[i][3] == tag;
    return __all(ok) || dead;
  };
  uint32_t spins = 0;
  while (!look()) {
    ++spins;
    if (spins >= a.spin_limit) {
      __hip_atomic_store(&a.st->aborted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dead = true;
    } else if ((spins & 1023u) == 0) {
      dead = __builtin_amdgcn_readfirstlane(
                 __hip_atomic_load(&a.st->aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    v[2 * i] = __int_as_float((int)r[i][0]);
    v[2 * i + 1] = __int_as_float((int)r[i][2]);
  }
}

// (mean, sum of squared deviations) of the wave's kPoll values v[i] with ok(i);
// two passes.
template <int N, typename G>
__device__ __forceinline__ void put_stats(Lds& s, int set, int part, const float (&v)[N], G ok, int lane) {
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) t += ok(i) ? v[i] : 0.f;
  const float mean = sum64(t) * (1.0f / kPoll);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) q += ok(i) ? (v[i] - mean) * (v[i] - mean) : 0.f;
  q = sum64(q);
  if (lane == 0) *reinterpret_cast<float2*>(s.stat[set][part]) = make_float2(mean, q);
}
// LayerNorm statistics of the whole vector from its equal parts' (the squared
// deviations about the parts' own means, plus the means' about the mean).
__device__ __forceinline__ void all_stats(const Lds& s, int set, float& mean, float& inv) {
  float m[kXW], q = 0.f, t = 0.f;
#pragma unroll
  for (int i = 0; i < kXW; ++i) {
    const float2 f = *reinterpret_cast<const float2*>(s.stat[set][i]);
    m[i] = f.x;
    t += f.x;
    q += f.y;
  }
  mean = t * (1.0f / kXW);
  float d = 0.f;
#pragma unroll
  for (int i = 0; i < kXW; ++i) d += (m[i] - mean) * (m[i] - mean);
  const float var = (q + d * (float)kPoll) * (1.0f / kW);
  inv = 1.0f / sqrtf(var + 1e-5f);
}
// What a wave's part of a phase's input vector holds (big: a lane's largest
// magnitude): 1 a nonzero value, 2 one of at least kSplitFull as well; uniform.
__device__ __forceinline__ int holds(float big) {
  return (__any(big > 0.f) ? 1 : 0) | (__any(big >= kSplitFull) ? 2 : 0);
}
// v[0], v[1], ... as split pairs at positions i, i + 1, i + step, i + step + 1, ...;
// reports values that are too large (or a NaN).  Returns the largest magnitude.
template <int N>
__device__ __forceinline__ float put_split(half_t* hi, half_t* lo, int i, int step, const float (&v)[N], GptState* st) {
  float big = 0.f;
  bool nan = false;
#pragma unroll
  for (int e = 0; e < N; e += 2) {
    big = fmaxf(big, fmaxf(fabsf(v[e]), fabsf(v[e + 1])));
    nan = nan || !(v[e] == v[e]) || !(v[e + 1] == v[e + 1]);
    half_t h0, l0, h1, l1;
    split_f16(v[e], h0, l0);
    split_f16(v[e + 1], h1, l1);
    *reinterpret_cast<half2v*>(hi + i + (e / 2) * step) = half2v{h0, h1};
    *reinterpret_cast<half2v*>(lo + i + (e / 2) * step) = half2v{l0, l1};
  }
  if (nan || big > kSplitMax) st->unfit = 1;
  return big;
}

template <typename T>
__device__ __forceinline__ const T* at(const char* base, size_t off) {
  return reinterpret_cast<const T*>(base + off);
}

// The running softmax of one 16-lane row of a wave: lane's 4 dims.
struct Soft {
  float m, l;
  float4 o;
};
// Adds U keys a lane group (scores from the group's 16 lanes x 4 dims).
template <int U>
__device__ __forceinline__ void soft_step(Soft& t, float4 q4, const float4 (&k4)[U], const float4 (&v4)[U],
                                          const bool (&ok)[U]) {
  float sc[U], mx = t.m;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float d = sum16((q4.x * k4[u].x + q4.y * k4[u].y) + (q4.z * k4[u].z + q4.w * k4[u].w));
    sc[u] = ok[u] ? d * 0.125f : -INFINITY;  // 1 / sqrt(64)
    mx = fmaxf(mx, sc[u]);
  }
  const float ms = mx == -INFINITY ? 0.f : mx;
  const float f = expf(t.m - ms);
  t.l *= f;
  t.o.x *= f; t.o.y *= f; t.o.z *= f; t.o.w *= f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float p = ok[u] ? expf(sc[u] - ms) : 0.f;
    t.l += p;
    t.o.x += p * v4[u].x; t.o.y += p * v4[u].y; t.o.z += p * v4[u].z; t.o.w += p * v4[u].w;
  }
  t.m = mx;
}

// Attention of s.q over this workgroup's part of head h in layer l: cached
// rows kTokSplits i + sp, and the new row for the part it falls to.  Wave w of
// kAW; its result (max, exp-sum, sums) goes to s.ml and s.o.
__device__ __forceinline__ void attend(const TokenArgs& a, Lds& s, int l, int h, int sp, int kv, int w, int lane) {
  const int ks = lane & 15, rg = lane >> 4;
  const int n = kv > sp ? (kv - sp + kTokSplits - 1) / kTokSplits : 0;
  const int nl = min(n, kLdsKeys);
  const float4 q4 = *reinterpret_cast<const float4*>(s.q + 4 * ks);
  Soft t = {-INFINITY, 0.f, make_float4(0.f, 0.f, 0.f, 0.f)};
  for (int g0 = w; 4 * g0 < nl; g0 += kAW * kAU) {
    float4 k4[kAU], v4[kAU];
    bool ok[kAU];
#pragma unroll
    for (int u = 0; u < kAU; ++u) {
      const int i = 4 * (g0 + kAW * u) + rg;
      ok[u] = i < nl;
      const int ic = min(i, nl - 1);
      k4[u] = *reinterpret_cast<const float4*>(s.k + ic * kHD + 4 * ks);
      v4[u] = *reinterpret_cast<const float4*>(s.v + ic * kHD + 4 * ks);
    }
    soft_step<kAU>(t, q4, k4, v4, ok);
  }
  const float* kh = a.kc + ((size_t)(l * kHeads + h) * a.cap) * kHD + 4 * ks;
  const float* vh = a.vc + ((size_t)(l * kHeads + h) * a.cap) * kHD + 4 * ks;
  for (int i0 = kLdsKeys + 4 * w; i0 < n; i0 += 4 * kAW * kAU) {  // past the LDS: from memory
    float4 k4[kAU], v4[kAU];
    bool ok[kAU];
#pragma unroll
    for (int u = 0; u < kAU; ++u) {
      const int i = i0 + 4 * kAW * u + rg;
      ok[u] = i < n;
      const size_t r = (size_t)(kTokSplits * min(i, n - 1) + sp) * kHD;
      k4[u] = *reinterpret_cast<const float4*>(kh + r);
      v4[u] = *reinterpret_cast<const float4*>(vh + r);
    }
    soft_step<kAU>(t, q4, k4, v4, ok);
  }
  if (w == 0 && kv % kTokSplits == sp) {  // the new row, in lane group 0
    const bool ok[1] = {rg == 0};
    const float4 k4[1] = {*reinterpret_cast<const float4*>(s.q + kHD + 4 * ks)};
    const float4 v4[1] = {*reinterpret_cast<const float4*>(s.q + 2 * kHD + 4 * ks)};
    soft_step<1>(t, q4, k4, v4, ok);
  }
  *reinterpret_cast<float4*>(&s.o[4 * w + rg][4 * ks]) = t.o;
  if (ks == 0) *reinterpret_cast<float2*>(s.ml[4 * w + rg]) = make_float2(t.m, t.l);
}
// The lane groups' results merged and handed over (one wave).
__device__ __forceinline__ void put_attention(const TokenArgs& a, Lds& s, int h, int sp, int lane, uint32_t tag) {
  constexpr int P = 4 * kAW;
  static_assert(P == 16, "one result per lane of a row");
  const float2 ml = *reinterpret_cast<const float2*>(s.ml[lane & 15]);
  float ov[P];
#pragma unroll
  for (int i = 0; i < P; ++i) ov[i] = s.o[i][lane];
  const float M = max16(ml.x);
  const float f = ml.x == -INFINITY ? 0.f : expf(ml.x - M);
  const float L = sum16(f * ml.y);
  float o = 0.f;
#pragma unroll
  for (int i = 0; i < P; ++i) o += lane_of(f, i) * ov[i];
  uint64_t* dst = a.mail->att + (sp * kHeads + h) * kTokAttRow;
  put(dst + lane, o, tag);
  if (lane < 2) put(dst + kHD + lane, lane == 0 ? M : L, tag);
}

// ------------------------------------------------------------ product waves
// A product is D = A B on the matrix cores: A's rows are weight rows (exact in
// f16), B's columns 2 r and 2 r + 1 the hi and lo halves of the input over K
// range r, so a row's value is D[row][2 r] + D[row][2 r + 1] / 2048.  (As dot
// products on the vector units, with their conversions and lane sums, a code
// took 0.53 ms where it took 0.47 so, before the polls slept.)
constexpr int kOob = 1 << 30;  // a byte offset past every buffer: reads zeros, without a memory access

__device__ __forceinline__ half8 buffer_load8(buffer_rsrc_t r, int voffset) {
#if defined(__HIP_DEVICE_COMPILE__)
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voffset, 0, 0);
  return __builtin_bit_cast(half8, v);
#else
  return half8{};
#endif
}

__device__ __forceinline__ void product_waves(const TokenArgs& a, Lds& s, int wg, int w, int lane, uint32_t tag0) {
  const int rr = lane & 15, g = lane >> 4;  // block row (A) or column (B); 8-wide K group
  half8 wq[kSW], wp[kS3W], wf[kSW + 1], wm[kS3F];
  // byte offsets of this lane's row and K group within the workgroup's rows of a matrix
  const int r3 = rr / 5, j3 = rr % 5, r4 = rr >> 2, j4 = rr & 3;
  const int v16 = rr * (2 * kW) + 16 * g + 64 * kSW * w;
  const int v4 = j4 * (2 * kW) + r4 * (2 * kR4) + 16 * g + 64 * w;
  int v3w[kS3W], v3f[kS3F];
#pragma unroll
  for (int i = 0; i < kS3W; ++i) {
    const int st = kS3W * w + i, k = r3 * kR3W + 32 * st + 8 * g;
    v3w[i] = rr < 15 && 32 * st < kR3W && k < kW ? j3 * (2 * kW) + 2 * k : kOob;
  }
#pragma unroll
  for (int i = 0; i < kS3F; ++i) {
    const int st = kS3F * w + i, k = r3 * kR3F + 32 * st + 8 * g;
    v3f[i] = rr < 15 && 32 * st < kR3F && k < kMLP ? j3 * (2 * kMLP) + 2 * k : kOob;
  }
  // B operands: this lane's column (range, half) and K group
  const int bc = min(rr >> 1, 2), hl = rr & 1;
  const half_t* b16 = s.x[hl] + 32 * kSW * w + 8 * g;
  const half_t* b4 = s.x[hl] + min(rr >> 1, 3) * kR4 + 32 * w + 8 * g;
  const half_t* b3w = s.x[hl] + min(bc * kR3W + 32 * kS3W * w + 8 * g, 3 * kR3W - 32 * (kS3W - 1) - 8);
  const half_t* b3f = s.xf[hl] + min(bc * kR3F + 32 * kS3F * w + 8 * g, 3 * kR3F - 32 * (kS3F - 1) - 8);

  // The weights' loads, layer l (l = a.L: the head's rows in c_attn's and
  // c_fc's registers).  Unconditional, or the loop would copy their registers
  // at its end.
  auto rows_of = [&](const void* base, int row0, int rows, int k) {
    return make_buffer_rsrc(static_cast<const half_t*>(base) + (size_t)row0 * k, max(rows - row0, 0) * k * 2);
  };
  auto next_qkv = [&](int l, size_t off) {
    const bool head = l == a.L;
    const buffer_rsrc_t r = head ? rows_of(a.head_w, wg * kTokHeadRows, kVocab, kW)
                                 : rows_of(a.attn_w + off, wg * kRQ, (wg + 1) * kRQ, kW);
#pragma unroll
    for (int i = 0; i < kSW; ++i) wq[i] = buffer_load8(r, v16 + 64 * i);
  };
  auto next_fc = [&](int l, size_t off) {
    const bool head = l == a.L;
    const buffer_rsrc_t r = head ? rows_of(a.head_w, wg * kTokHeadRows + 16, kVocab, kW)
                                 : rows_of(a.fc_w + off, wg * kRF, (wg + 1) * kRF, kW);
#pragma unroll
    for (int i = 0; i < kSW; ++i) wf[i] = buffer_load8(r, v16 + 64 * i);
    wf[kSW] = buffer_load8(r, v4 + 16 * 2 * kW);
  };
  auto next_proj = [&](size_t off) {
    const buffer_rsrc_t r = rows_of(a.proj_w + off, wg * kRP, (wg + 1) * kRP, kW);
#pragma unroll
    for (int i = 0; i < kS3W; ++i) wp[i] = buffer_load8(r, v3w[i]);
  };
  auto next_mp = [&](size_t off) {
    const buffer_rsrc_t r = rows_of(a.mp_w + off, wg * kRP, (wg + 1) * kRP, kMLP);
#pragma unroll
    for (int i = 0; i < kS3F; ++i) wm[i] = buffer_load8(r, v3f[i]);
  };
  auto product = [&](const half8* wv, const half_t* b, auto cnt) {
    floatx4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < decltype(cnt)::value; ++i)
      d = mfma16x16x32(wv[i], *reinterpret_cast<const half8*>(b + 32 * i), d);
    // the lo half's column is the next lane's
#pragma unroll
    for (int r = 0; r < 4; ++r)
      d[r] += kSplitInv * __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d[r]), 0xb1, 0xf, 0xf, false));
    return d;
  };
  auto put_part = [&](int blk, const floatx4& d) {
    *reinterpret_cast<float4*>(&s.part[w][blk][4 * g]) = make_float4(d[0], d[1], d[2], d[3]);
  };
  // sums over the waves of block blk's row (lane & 15)
  auto waves_sum = [&](int blk) {
    float v[kCW];
#pragma unroll
    for (int i = 0; i < kCW; ++i) v[i] = s.part[i][blk][rr];
    float t = (v[0] + v[1]) + (v[2] + v[3]);
    t += (v[4] + v[5]) + (v[6] + v[7]);
    return t + (v[8] + v[9]);
  };
  // ... of the projections' rows: the three ranges' rows j, 5 + j, 10 + j
  auto ranges_sum = [&]() {
    const float t = waves_sum(min(r3, 2));
    return t + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(t), 0x105, 0xf, 0xf, false)) +
           __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(t), 0x10a, 0xf, 0xf, false));
  };
  using CW = std::integral_constant<int, kSW>;
  using C1 = std::integral_constant<int, 1>;

  next_qkv(0, 0);
  next_proj(0);
  next_fc(0, 0);
  next_mp(0);
  __builtin_amdgcn_sched_barrier(0);

  lds_barrier();  // the key wave's first loads
  float xres = 0.f;  // wave 0, lanes < kRP: the residual stream at the workgroup's rows
#pragma clang loop unroll(disable)
  for (int l = 0; l < a.L; ++l) {
    const uint32_t tag = tag0 + l;
    // (with no next layer, the last layer's projections are read again)
    const size_t noff = a.stride * (size_t)min(l + 1, a.L - 1);
    // c_attn
    lds_barrier();
    lds_barrier();
    {
      const floatx4 d = product(wq, b16, CW{});
      if (rr == 0) put_part(0, d);
    }
    lds_barrier();
    if (w == 0) {
      xres = s.xr[lane & 7];
      const float v = waves_sum(0) + s.bias[l & 1][0][lane];
      if (lane < kRQ) put(a.mail->qkv + wg * kRQ + lane, v, tag);
    }
    next_qkv(l + 1, noff);
    __builtin_amdgcn_sched_barrier(0);

    if (wg < kAttnWG) {  // the poll waves' attention
      lds_barrier();
      lds_barrier();
    }

    // attention projection + residual
    lds_barrier();
    {
      const floatx4 d = product(wp, b3w, std::integral_constant<int, kS3W>{});
      if (rr < 6 && hl == 0) put_part(rr >> 1, d);
    }
    lds_barrier();
    if (w == 0) {
      xres = xres + (ranges_sum() + s.bias[l & 1][1][lane]);
      if (lane < kTokXSlot) put(a.mail->xb + wg * kTokXSlot + lane, xres, tag);  // (a whole line)
    }
    next_proj(noff);
    __builtin_amdgcn_sched_barrier(0);

    // c_fc + gelu
    lds_barrier();
    lds_barrier();
    {
      const floatx4 d = product(wf, b16, CW{});
      const floatx4 e = product(wf + kSW, b4, C1{});
      if (rr == 0) put_part(0, d);
      if (rr == 2 * g) put_part(1, e);  // rows 4 g .. of the block: range g
    }
    lds_barrier();
    if (w == 0) {
      float v = waves_sum(g & 1);
      float u = dpp_add<0x128>(v);  // block 1: the four ranges
      u = dpp_add<0x124>(u);
      v = gelu_new((lane < 16 ? v : u) + s.bias[l & 1][2][lane]);
      if (lane < kTokFSlot) put(a.mail->fc + wg * kTokFSlot + lane, v, tag);
    }
    next_fc(l + 1, noff);
    __builtin_amdgcn_sched_barrier(0);

    // mlp projection + residual
    lds_barrier();
    {
      const floatx4 d = product(wm, b3f, std::integral_constant<int, kS3F>{});
      if (rr < 6 && hl == 0) put_part(rr >> 1, d);
    }
    lds_barrier();
    if (w == 0) {
      const float v = xres + (ranges_sum() + s.bias[l & 1][3][lane]);
      if (lane < kTokXSlot) put(a.mail->xa + wg * kTokXSlot + lane, v, tag);
    }
    next_mp(noff);
    __builtin_amdgcn_sched_barrier(0);
  }

  // head
  lds_barrier();
  lds_barrier();
  lds_barrier();
  {
    const floatx4 d = product(wq, b16, CW{});
    const floatx4 e = product(wf, b16, CW{});
    const floatx4 f = product(wf + kSW, b4, C1{});
    if (rr == 0) put_part(0, d);
    if (rr == 0) put_part(1, e);
    if (rr == 2 * g) put_part(2, f);
  }
  lds_barrier();
  if (w == 0) {
    const int row = wg * kTokHeadRows + lane;
    float v = waves_sum(min(g, 2));
    float u = dpp_add<0x128>(v);
    u = dpp_add<0x124>(u);
    const bool live = lane < kTokHeadRows && row < kVocab;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    if (live) {
      bv = (lane < 32 ? v : u) + s.bias[a.L & 1][0][lane];
      bi = row;
      a.logits[row] = bv;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {  // the first maximum
      const float ov = __shfl_xor(bv, off, kWave);
      const int oi = __shfl_xor(bi, off, kWave);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (lane == 0) {
      a.blk_val[wg] = bv;
      a.blk_idx[wg] = bi;
      if (wg == 0) a.st->kv += 1;
    }
  }
}

// --------------------------------------------------------------- poll waves
__device__ __forceinline__ void poll_waves(const TokenArgs& a, Lds& s, int wg, int pw, int lane, int kv,
                                           uint32_t tag0) {
  // The residual stream (waves pw < kXW): 64 slots a wave, three word pairs a
  // slot, of which this lane holds lane + 64 i: values pos(i), pos(i) + 1 (the
  // third pair's second word is none).
  constexpr int NP = 3, N = 2 * NP, NF = kMLP / (64 * kPW);
  static_assert(kRP == 5 && NF == 16 && kAW <= kPW && kXW <= kPW, "three pairs a slot; whole pairs");
  bool dead = false;
  float v[N];
  int slot[NP], third[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    slot[i] = 64 * pw + (lane + 64 * i) / 3;
    third[i] = (lane + 64 * i) % 3;
  }
  const bool xw = pw < kXW;
  auto pos = [&](int i) { return kRP * slot[i] + 2 * third[i]; };
  auto ok = [&](int i) { return (i & 1) == 0 || third[i / 2] < 2; };
  auto pairs = [&](int i) { return 8 * (kTokXSlot * slot[i] + 2 * third[i]); };
  if (xw) {
    GptState* st = a.st;
    const int tok = min(max(st->cur_token, 0), kVocab - 1);
    const int at = min((st->hf && st->step > 0) ? st->step + 1 : st->step, kPos - 1);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = pos(i / 2) + (ok(i) ? i & 1 : 0);
      v[i] = a.mel_emb[(size_t)tok * kW + e] + a.pos_emb[(size_t)at * kW + e];
    }
  }
  auto norm = [&](int which) {  // v: LayerNorm, with the other waves of the stream
    float gv[N], bv[N];
    if (xw) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        gv[i] = s.ln[which][0][pos(i / 2) + (ok(i) ? i & 1 : 0)];
        bv[i] = s.ln[which][1][pos(i / 2) + (ok(i) ? i & 1 : 0)];
      }
      put_stats(s, which, pw, v, ok, lane);
    }
    lds_barrier();
    if (xw) {
      float mean, inv;
      all_stats(s, which, mean, inv);
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = (v[i] - mean) * inv * gv[i] + bv[i];
    }
  };
  // The four phases' input vectors a layer, each in parts of a wave.  While the
  // products run, between the phase's two barriers, every wave notes what its part
  // holds, and after them wave 0 reports a vector that is all below kSplitFull
  // (but not all 0).
  float big = 0.f;
  auto input_done = [&](int phase) {
    lds_barrier();
    const int h = holds(big);
    if (lane == 0) s.holds[phase][pw] = h;
    lds_barrier();
    if (pw == 0) {
      const int hp = lane < kPW ? s.holds[phase][lane] : 0;
      if (__any(hp != 0) && !__any((hp & 2) != 0)) a.st->unfit = 1;
    }
  };
  auto put_x = [&]() {
    big = 0.f;
    if (!xw) return;
    bool nan = false;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (!ok(i)) continue;
      nan = nan || !(v[i] == v[i]);
      big = fmaxf(big, fabsf(v[i]));
      half_t h, l;
      split_f16(v[i], h, l);
      s.x[0][pos(i / 2) + (i & 1)] = h;
      s.x[1][pos(i / 2) + (i & 1)] = l;
    }
    if (nan || big > kSplitMax) a.st->unfit = 1;
  };
  for (int i = lane + 64 * pw; i < 3 * kR3W - kW; i += 64 * kPW) s.x[0][kW + i] = s.x[1][kW + i] = (half_t)0.f;
  for (int i = lane + 64 * pw; i < 3 * kR3F - kMLP; i += 64 * kPW) s.xf[0][kMLP + i] = s.xf[1][kMLP + i] = (half_t)0.f;
  lds_barrier();  // the key wave's first loads
#pragma clang loop unroll(disable)
  for (int l = 0; l < a.L; ++l) {
    const uint32_t tag = tag0 + l;
    // (opaque, so that no address is formed ahead of the loop and held in a register)
    __asm__ volatile("" : "+v"(lane), "+v"(slot[0]), "+v"(slot[1]), "+v"(slot[2]), "+v"(third[0]), "+v"(third[1]),
                     "+v"(third[2]));
    // c_attn's input
    if (l > 0 && xw) poll<NP, kSleepXa>(a.mail->xa, sizeof a.mail->xa, pairs, tag - 1, v, dead, a);
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (xw && slot[i / 2] == wg && ok(i)) s.xr[2 * third[i / 2] + (i & 1)] = v[i];
    norm(0);
    put_x();
    input_done(0);
    // the head's query, and the new key and value: waves 0 (q, k) and 1 (v)
    if (wg < kAttnWG) {
      const int h = wg % kHeads, sp = wg / kHeads;
      if (pw < 2) {
        float t[2];
        const int part = min(2 * pw + (lane >> 5), 2), d = 2 * (lane & 31);
        poll<1, kSleepQ>(a.mail->qkv, sizeof a.mail->qkv, [&](int) { return 8 * (part * kW + h * kHD + d); }, tag, t,
                         dead, a);
        *reinterpret_cast<float2*>(s.q + part * kHD + d) = make_float2(t[0], t[1]);
        if (part > 0 && kv % kTokSplits == sp)
          *reinterpret_cast<float2*>((part == 1 ? a.kc : a.vc) + ((size_t)(l * kHeads + h) * a.cap + kv) * kHD + d) =
              make_float2(t[0], t[1]);
      }
      lds_barrier();
      if (pw < kAW) attend(a, s, l, h, sp, kv, pw, lane);
      lds_barrier();
      if (pw == 0) put_attention(a, s, h, sp, lane, tag);
    } else {
      __builtin_amdgcn_s_sleep(kSleepIdle);
    }
    // the attention's parts: heads 4 pw ..; this lane's dims 2 (lane % 32) and
    // the next of heads 2 (lane / 32), 2 (lane / 32) + 1, all parts; lanes
    // 4 i + sp also part sp's max and exp-sum of head i
    {
      constexpr int kRow = kTokAttRow, NO = 2 * kTokSplits;
      static_assert(kTokSplits == 4 && kPW * 4 == kHeads, "one quad of lanes per head, four heads a wave");
      const int hb = 4 * pw, hh = 2 * (lane >> 5), d = 2 * (lane & 31);
      float o[2 * (NO + 1)];
      poll<NO + 1, kSleepAtt>(
          a.mail->att, sizeof a.mail->att,
          [&](int i) {
            return i < NO ? 8 * (((i & 3) * kHeads + hb + hh + (i >> 2)) * kRow + d)
                          : 8 * (((lane & 3) * kHeads + hb + ((lane >> 2) & 3)) * kRow + kHD);
          },
          tag, o, dead, a);
      float M = o[2 * NO];
      M = fmaxf(M, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(M), 0xb1, 0xf, 0xf, false)));
      M = fmaxf(M, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(M), 0x4e, 0xf, 0xf, false)));
      const float f = o[2 * NO] == -INFINITY ? 0.f : expf(o[2 * NO] - M);
      float L = f * o[2 * NO + 1];
      L = dpp_add<0xb1>(L);
      L = dpp_add<0x4e>(L);
      const float sc = f / L;
      float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < NO; ++i) {
        const float lo = lane_of(sc, i), hi = lane_of(sc, 8 + i);  // heads 0, 1 | 2, 3
        const float c = hh == 0 ? lo : hi;
        t[2 * (i >> 2)] += c * o[2 * i];
        t[2 * (i >> 2) + 1] += c * o[2 * i + 1];
      }
      big = put_split(s.x[0], s.x[1], (hb + hh) * kHD + d, kHD, t, a.st);
    }
    input_done(1);
    // c_fc's input
    if (xw) poll<NP, kSleepXb>(a.mail->xb, sizeof a.mail->xb, pairs, tag, v, dead, a);
    norm(1);
    put_x();
    input_done(2);
    // the mlp projection's input
    {
      const int p0 = pw * 32 * NF + lane, f0 = 2 * p0;  // pairs p0 + 64 i, ten a slot
      float f[NF];
      poll<NF / 2, kSleepFc>(
          a.mail->fc, sizeof a.mail->fc,
          [&](int i) {
            const int p = p0 + 64 * i, sl = p / (kRF / 2);
            return 8 * (kTokFSlot * sl + 2 * (p - sl * (kRF / 2)));
          },
          tag, f, dead, a);
      big = put_split(s.xf[0], s.xf[1], f0, 128, f, a.st);
    }
    input_done(3);
  }
  if (xw) poll<NP, kSleepXa>(a.mail->xa, sizeof a.mail->xa, pairs, tag0 + a.L - 1, v, dead, a);
  norm(0);
  norm(1);
  put_x();
  input_done(2);
}

// ----------------------------------------------------------------- key wave
__device__ __forceinline__ void key_wave(const TokenArgs& a, Lds& s, int wg, int lane, int kv) {
  const bool attn = wg < kAttnWG;
  const int h = wg % kHeads, sp = wg / kHeads;
  const int n = kv > sp ? min((kv - sp + kTokSplits - 1) / kTokSplits, kLdsKeys) : 0;
  // local keys 4 g + lane / 16, four to a 1 KB load
  auto fetch = [&](int l) {
    const float* kh = a.kc + ((size_t)(l * kHeads + h) * a.cap) * kHD + 4 * (lane & 15);
    const float* vh = a.vc + ((size_t)(l * kHeads + h) * a.cap) * kHD + 4 * (lane & 15);
    for (int g = 0; 4 * g < n; ++g) {
      const size_t r = (size_t)(kTokSplits * min(4 * g + (lane >> 4), n - 1) + sp) * kHD;
      __builtin_amdgcn_global_load_lds((const void*)(kh + r), (lds_ptr_t*)(s.k + 4 * g * kHD), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(vh + r), (lds_ptr_t*)(s.v + 4 * g * kHD), 16, 0, 0);
    }
  };
  // a norm's weight and bias: five 1 KB loads each
  auto fetch_ln = [&](int which, const float* g, const float* b) {
#pragma unroll
    for (int i = 0; i < kW / 256; ++i) {
      __builtin_amdgcn_global_load_lds((const void*)(g + 4 * lane + 256 * i), (lds_ptr_t*)(s.ln[which][0] + 256 * i), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(b + 4 * lane + 256 * i), (lds_ptr_t*)(s.ln[which][1] + 256 * i), 16, 0, 0);
    }
  };
  // the biases of layer l (l = L: the head's) at this workgroup's rows, a row a lane
  auto fetch_bias = [&](int l, size_t off) {
    auto one = [&](int which, const float* src, int r0, int rows, int rmax) {
      __builtin_amdgcn_global_load_lds((const void*)(src + min(r0 + min(lane, rows - 1), rmax)),
                                       (lds_ptr_t*)s.bias[l & 1][which], 4, 0, 0);
    };
    if (l == a.L) {
      one(0, a.head_b, wg * kTokHeadRows, kTokHeadRows, kVocab - 1);
    } else {
      one(0, at<float>(a.attn_b, off), wg * kRQ, kRQ, kQKV - 1);
      one(1, at<float>(a.proj_b, off), wg * kRP, kRP, kW - 1);
      one(2, at<float>(a.fc_b, off), wg * kRF, kRF, kMLP - 1);
      one(3, at<float>(a.mp_b, off), wg * kRP, kRP, kW - 1);
    }
  };
  // all but the last `left` loads have landed (vmcnt)
  auto landed = [&](auto left) {
    constexpr int n = decltype(left)::value;
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
  };
  using All = std::integral_constant<int, 0>;
  using ButNorm = std::integral_constant<int, 2 * (kW / 256)>;
  static_assert(kW % 256 == 0 && kLdsKeys % 4 == 0, "whole 1 KB loads");
  fetch_ln(0, at<float>(a.ln1_w, 0), at<float>(a.ln1_b, 0));
  fetch_ln(1, at<float>(a.ln2_w, 0), at<float>(a.ln2_b, 0));
  fetch_bias(0, 0);
  if (attn) fetch(0);
  landed(All{});
  bare_barrier();
#pragma clang loop unroll(disable)
  for (int l = 0; l < a.L; ++l) {
    const bool last = l + 1 == a.L;
    const size_t noff = a.stride * (size_t)(l + 1);
    landed(All{});
    bare_barrier();  // c_attn
    bare_barrier();
    bare_barrier();
    fetch_ln(0, last ? a.lnf_w : at<float>(a.ln1_w, noff), last ? a.lnf_b : at<float>(a.ln1_b, noff));
    fetch_bias(l + 1, noff);
    if (attn) {
      bare_barrier();
      bare_barrier();
      if (!last) fetch(l + 1);
    }
    bare_barrier();  // projection
    bare_barrier();
    bare_barrier();  // c_fc
    bare_barrier();
    bare_barrier();
    fetch_ln(1, last ? a.fn_w : at<float>(a.ln2_w, noff), last ? a.fn_b : at<float>(a.ln2_b, noff));
    landed(ButNorm{});  // the next layer's first norm is read ahead of its first barrier
    bare_barrier();     // mlp projection
    bare_barrier();
  }
  landed(All{});
#pragma unroll
  for (int i = 0; i < 4; ++i) bare_barrier();
}

__global__ __launch_bounds__(kThreads) void token_kernel(TokenArgs a) {
  __shared__ __attribute__((aligned(1024))) Lds s;
  if (a.st->stopped) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wg = blockIdx.x;
  if (threadIdx.x == kThreads - 1) a.start[wg] = device_ticks();
  const int kv = __builtin_amdgcn_readfirstlane(a.st->kv);
  const uint32_t tag0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)((a.st->epoch + (uint32_t)a.st->step) << 6));
  if (wave < kCW)
    product_waves(a, s, wg, wave, lane, tag0);
  else if (wave < kCW + kPW)
    poll_waves(a, s, wg, wave - kCW, lane, kv, tag0);
  else
    key_wave(a, s, wg, lane, kv);
}

}  // namespace

bool gpt_token_fits(int device) {
  int cus = 0, per_cu = 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return false;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(token_kernel), kThreads, 0) !=
      hipSuccess)
    return false;
  return (long)cus * per_cu >= kTokWG;
}

hipError_t launch_gpt_token(const TokenArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(token_kernel, dim3(kTokWG), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace mit2hip
