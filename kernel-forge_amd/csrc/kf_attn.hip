// Attention of one decode token over the KV cache, one launch (gfx950).
//
//   out[h] = softmax(mask[h] + q[h] . K[kv] / sqrt(d)) . V[kv],  kv = h / (heads / kv_heads)
//
// q fp16 [heads, d]; cache_k fp16 [kv_heads, d, max_seq] (K transposed); cache_v fp16
// [kv_heads, max_seq, d]; mask fp16 rows of max_seq additive values; out fp16 [heads, d].  Scores,
// softmax and the weighted sum stay in fp32; the output is rounded once.  Error against 64 bits (32 heads on 4, d =
// 64, max_seq 96 .. 288, q of 1, 2 and 4 times unit variance, 120 draws): 2.08e-4 of the result, what rounding the exact
// result to fp16 gives, with __expf as with expf (0.3 us slower); the library's three launches, which round scores
// and probabilities to fp16, 4.7e-4 to 9.1e-4.  Whole models of 4 to 22 layers are 0.983x as far from 64 bits as with
// those (0.93x to 1.06x by seed); the two differ by 3e-3 of the logits, each being about that far off.
//
// What bounds it: latency.  The work of a TinyLlama layer at max_seq = 160 is 40 KiB of K and V per KV
// head; as three library launches (a batched product, a softmax over fp16 scores, a batched product)
// it took 14 us of a 31 us layer, nearly all of it launch and tail.  So: one launch, a workgroup of
// eight wavefronts per query head (K and V of a KV head come from L2 for the heads that share it), and
// as few dependent steps as possible:
//   * the wavefronts split the keys, 32 consecutive ones each per pass, and meet once, at the end: each
//     keeps the running maximum, sum and V sums of its own keys;
//   * q, the mask, the first keys and the first V rows are all loaded before the first wait;
//   * scores: 16 lanes own key pairs (K is stored transposed: 64-byte runs), four slices of lanes split d;
//   * V: 16-byte pieces, d / 8 lanes per key, kAttnV steps loaded together; the lanes' sums are added by
//     shuffles where d / 8 is a power of two, then the wavefronts' through LDS in fixed order
//     (deterministic).
// MI355X, d = 64, max_seq 96 / 160 / 288 / 512 / 1024: 4.5 / 4.9 / 5.8 / 6.6 / 9.6 us per launch in a graph;
// the three library launches take 12.1 / 14.0 / 14.0 / 13.5 / 18.2.  Before, with the wavefronts splitting
// d and meeting at five barriers: 5.1 / 5.1 / 6.7 / 7.1 / 10.3; before that, with four wavefronts and V
// rows and last sums one dependent load at a time: 5.7 / 7.0 / 9.4 / 12.1 / 21.0.  One workgroup per head
// is the wrong split for long caches: from about 131072 / d keys on the library's launches are faster
// (d = 64, 2048 / 4096 keys: 15.5 against 27.5, 29.0 against 25.9; d = 128, 1024 / 2048: 15.1 against 17.0,
// 26.2 against 26.0), and the decoder keeps them there.
#include "kf_device.h"
#include "kf_launch.h"

namespace kf {
namespace {

constexpr int kAttnThreads = 512, kAttnWaves = kAttnThreads / 64;
constexpr int kAttnSlices = 4;     // of d, 16 lanes each
constexpr int kAttnK = 16;         // K rows of a slice loaded together
constexpr int kAttnV = 4;          // V steps loaded together; the first ones before the scores
constexpr int kAttnSums = 4096;    // floats: 8 wavefronts x (64 / (d / 8)) keys x d

__device__ __forceinline__ float dpp_f(float v, const int ctrl_index) {
  const int i = bit_cast<int>(v);
  switch (ctrl_index) {
    case 0: return bit_cast<float>(__builtin_amdgcn_mov_dpp(i, 0xB1, 0xF, 0xF, true));   // quad_perm 1,0,3,2
    case 1: return bit_cast<float>(__builtin_amdgcn_mov_dpp(i, 0x4E, 0xF, 0xF, true));   // quad_perm 2,3,0,1
    case 2: return bit_cast<float>(__builtin_amdgcn_mov_dpp(i, 0x141, 0xF, 0xF, true));  // row_half_mirror
    default: return bit_cast<float>(__builtin_amdgcn_mov_dpp(i, 0x140, 0xF, 0xF, true)); // row_mirror
  }
}
__device__ __forceinline__ float lane_f(float v, int lane) {
  return bit_cast<float>(__builtin_amdgcn_readlane(bit_cast<int>(v), lane));
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v = fmaxf(v, dpp_f(v, i));
  return fmaxf(fmaxf(lane_f(v, 0), lane_f(v, 16)), fmaxf(lane_f(v, 32), lane_f(v, 48)));
}
__device__ __forceinline__ float wave_add(float v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v += dpp_f(v, i);
  return (lane_f(v, 0) + lane_f(v, 16)) + (lane_f(v, 32) + lane_f(v, 48));
}

// Orders a wavefront's own LDS writes before its reads (no other wavefront touches the region).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// VEC: max_seq is even and cache_k 4-byte aligned, keys are read in pairs.
template <bool VEC>
__global__ __launch_bounds__(kAttnThreads) void decode_attention_kernel(const half_t* __restrict__ q,
                                                                        const half_t* __restrict__ cache_k,
                                                                        const half_t* __restrict__ cache_v,
                                                                        const half_t* __restrict__ mask,
                                                                        half_t* __restrict__ out, int rep, int d,
                                                                        int max_seq, int mask_stride, float scale) {
  constexpr int KPL = VEC ? 2 : 1;                // keys per lane
  constexpr int KPW = 16 * KPL;                   // keys per wavefront and pass
  constexpr int BLOCK = KPW * kAttnWaves;
  extern __shared__ __attribute__((aligned(16))) float attn_lds[];
  float* const stat = attn_lds;                   // max [8], sum [8]
  float* const sums = attn_lds + 16;
  const int h = blockIdx.x, kv = h / rep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* const ps = sums + kAttnSums + 32 * wave;                          // this pass's probabilities
  float* const qs = sums + kAttnSums + 32 * kAttnWaves + wave * d;
  const half_t* const kb = cache_k + (size_t)kv * d * max_seq;
  const half_t* const vb = cache_v + (size_t)kv * max_seq * d;
  const half_t* const mrow = mask + (size_t)h * mask_stride;

  // K rows i .. i + kAttnK - 1 of this lane's slice and keys; rows past the slice re-read its last one.
  const int slice = lane >> 4, dn = d / kAttnSlices, d0 = slice * dn;      // d % 8 == 0
  const int key0 = KPW * wave + KPL * (lane & 15);
  auto load_k = [&](half2_t (&k)[kAttnK], int i, int s) {
    const int sc = min(s, max_seq - KPL);
#pragma unroll
    for (int j = 0; j < kAttnK; ++j) {
      const uint32_t at = (uint32_t)((d0 + min(i + j, dn - 1)) * max_seq + sc);
      if constexpr (VEC) k[j] = *reinterpret_cast<const half2_t*>(kb + at);
      else k[j] = half2_t{kb[at], (half_t)0};
    }
  };
  // V steps i .. i + kAttnV - 1 of this lane in the pass at `base`; keys past the end re-read the last one.
  const int lpk = d >> 3;                                // lanes per key
  const int kps = 64 / lpk;                              // keys per step
  const int vk = lane / lpk, vc = lane - vk * lpk;       // vk == kps where d / 8 does not divide 64: idle
  auto load_v = [&](u32x4 (&v)[kAttnV], int i, int base) {
#pragma unroll
    for (int j = 0; j < kAttnV; ++j)
      v[j] = load_u32x4(vb + (uint32_t)(min(base + vk + (i + j) * kps, max_seq - 1) * d + 8 * vc));
  };
  auto load_mask = [&](int s) { return (float)mrow[min(s, max_seq - 1)]; };

  half2_t k[kAttnK];
  u32x4 v[kAttnV];
  for (int i = lane; i < d; i += 64) qs[i] = (float)q[(size_t)h * d + i];
  load_k(k, 0, key0);
  float mask0 = load_mask(key0), mask1 = VEC ? load_mask(key0 + 1) : 0.0f;
  load_v(v, 0, KPW * wave);
  wave_lds_sync();

  float m = -__builtin_inff(), sum = 0.0f;  // sum: this lane's keys
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (int base = KPW * wave; base < max_seq; base += BLOCK) {
    const int s = base + KPL * (lane & 15);
    if (base >= BLOCK) {
      load_k(k, 0, s);
      mask0 = load_mask(s);
      if constexpr (VEC) mask1 = load_mask(s + 1);
      load_v(v, 0, base);
    }
    float a0 = 0.0f, a1 = 0.0f;
    for (int i = 0; i < dn; i += kAttnK) {
      if (i > 0) load_k(k, i, s);
#pragma unroll
      for (int j = 0; j < kAttnK; ++j)
        if (i + j < dn) {  // uniform
          const float qj = qs[d0 + i + j];
          a0 = fmaf(qj, (float)k[j][0], a0);
          if constexpr (VEC) a1 = fmaf(qj, (float)k[j][1], a1);
        }
    }
    // The four slices' sums, in every lane; lanes 0 .. 15 count for the row's sum.
    a0 += __shfl_xor(a0, 16);
    a0 += __shfl_xor(a0, 32);
    const float t0 = s < max_seq ? fmaf(a0, scale, mask0) : -__builtin_inff();
    float t1 = -__builtin_inff();
    if constexpr (VEC) {
      a1 += __shfl_xor(a1, 16);
      a1 += __shfl_xor(a1, 32);
      t1 = s < max_seq ? fmaf(a1, scale, mask1) : -__builtin_inff();
    }
    // Running maximum.  While every key is masked it is -inf and the exponentials are taken against 0,
    // so they are 0; a NaN score drops out of the maximum and makes its exponential NaN.
    const float mn = fmaxf(m, wave_max(fmaxf(t0, t1)));
    const float ref = mn == -__builtin_inff() ? 0.0f : mn;
    const float p0 = __expf(t0 - ref), p1 = VEC ? __expf(t1 - ref) : 0.0f;
    if (base >= BLOCK) {
      const float f = __expf(m - ref);
      sum *= f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] *= f;
    }
    m = mn;
    if (lane < 16) {
      sum += p0 + p1;
      ps[KPL * lane] = p0;
      if constexpr (VEC) ps[KPL * lane + 1] = p1;
    }
    wave_lds_sync();
    // Weighted sum of V: this lane's 8 dims over the pass's keys vk, vk + kps, ...
    for (int i = 0; i * kps < KPW; i += kAttnV) {
      if (i > 0) load_v(v, i, base);
#pragma unroll
      for (int j = 0; j < kAttnV; ++j) {
        const int key = vk + (i + j) * kps;
        if (key < KPW && base + key < max_seq && vk < kps) {
          const float p = ps[key];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const half2_t h2 = bit_cast<half2_t>(v[j][e]);
            acc[2 * e] = fmaf(p, (float)h2[0], acc[2 * e]);
            acc[2 * e + 1] = fmaf(p, (float)h2[1], acc[2 * e + 1]);
          }
        }
      }
    }
    wave_lds_sync();  // the probabilities have been read
  }
  sum = wave_add(sum);

  // Lanes of a wavefront that hold the same dims are lpk apart.
  const bool pow2 = (lpk & (lpk - 1)) == 0;  // lpk <= 32
  if (pow2) {
    for (int off = lpk; off < 64; off <<= 1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off);
    }
  }
  const int rows = pow2 ? 1 : kps, row = wave * rows + (pow2 ? 0 : vk);
  if (pow2 ? lane < lpk : vk < kps) {
#pragma unroll
    for (int e = 0; e < 8; ++e) sums[row * d + 8 * vc + e] = acc[e];
  }
  if (lane == 0) {
    stat[wave] = m;
    stat[kAttnWaves + wave] = sum;
  }
  __syncthreads();
  if (tid < d) {
    float top = stat[0];
#pragma unroll
    for (int i = 1; i < kAttnWaves; ++i) top = fmaxf(top, stat[i]);
    float total = 0.0f, o = 0.0f;
#pragma unroll
    for (int i = 0; i < kAttnWaves; ++i) {
      const float f = __expf(stat[i] - top);  // all keys masked: -inf - -inf, NaN
      total = fmaf(f, stat[kAttnWaves + i], total);
      float r = sums[i * rows * d + tid];
      for (int j = 1; j < rows; ++j) r += sums[(i * rows + j) * d + tid];
      o = fmaf(f, r, o);
    }
    out[(size_t)h * d + tid] = (half_t)(o / total);
  }
}

}  // namespace

hipError_t decode_attention_launch(const void* q, const void* cache_k, const void* cache_v, const void* mask, void* out,
                                   int heads, int kv_heads, int head_dim, int max_seq, int mask_stride, float scale,
                                   hipStream_t stream) {
  const size_t lds = sizeof(float) * (16 + kAttnSums + kAttnWaves * (32 + head_dim));  // at most 26 KiB
  const auto fn = max_seq % 2 == 0 && (reinterpret_cast<uintptr_t>(cache_k) & 3) == 0 ? decode_attention_kernel<true>
                                                                                      : decode_attention_kernel<false>;
  hipLaunchKernelGGL(fn, dim3(heads), dim3(kAttnThreads), lds, stream, static_cast<const half_t*>(q),
                     static_cast<const half_t*>(cache_k), static_cast<const half_t*>(cache_v),
                     static_cast<const half_t*>(mask), static_cast<half_t*>(out), heads / kv_heads, head_dim, max_seq,
                     mask_stride, scale);
  return hipGetLastError();
}

}  // namespace kf
