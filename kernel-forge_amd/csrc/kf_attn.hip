// Attention of one decode token over the KV cache, one launch (gfx950).
//
//   out[h] = softmax(mask[h] + q[h] . K[kv] / sqrt(d)) . V[kv],  kv = h / (heads / kv_heads)
//
// q fp16 [heads, d]; cache_k fp16 [kv_heads, d, max_seq] (K transposed); cache_v fp16
// [kv_heads, max_seq, d]; mask fp16 rows of max_seq additive values; out fp16 [heads, d].  Scores,
// softmax and the weighted sum stay in fp32; the output is rounded once.
//
// What bounds it: latency.  The work of a TinyLlama layer at max_seq = 160 is 40 KiB of K and V per KV
// head; as three library launches (a batched product, a softmax over fp16 scores, a batched product)
// it took 14 us of a 31 us layer, nearly all of it launch and tail.  So: one launch, a workgroup of
// eight wavefronts per query head (K and V of a KV head come from L2 for the heads that share it), and
// as few dependent steps as possible:
//   * q, the mask, the first keys and the first V rows are all loaded before the first wait;
//   * scores: lanes own consecutive keys (K is stored transposed, so a wavefront reads whole lines),
//     four slices of wavefronts split d, two halves split the keys; the four partial sums meet in LDS;
//   * the sum of the exponentials is only needed at the end, so it shares a barrier with them;
//   * V: 16-byte pieces, d / 8 lanes per key, 4096 / d keys per step, kAttnV steps loaded together; the
//     lanes' sums are added by shuffles within a wavefront where d / 8 is a power of two, then in fixed
//     order through LDS (deterministic).
// MI355X, d = 64, max_seq 96 / 160 / 288 / 512 / 1024: 5.1 / 5.1 / 6.7 / 7.1 / 10.3 us per
// launch in a graph; the three library launches take 12.1 / 14.0 / 14.0 / 13.7 / 18.2.  A first version
// (four wavefronts, nothing of K loaded ahead, V rows past the first six steps and the last sum one
// dependent load at a time) took 5.7 / 7.0 / 9.4 / 12.1 / 21.0.  One workgroup per head is the wrong
// split for long caches: from about 131072 / d keys on the library's launches are faster (d = 64, 2048
// / 4096 keys: 16.8 against 27.5, 31.4 against 25.8; d = 128, 1024 / 2048: 15.9 against 16.2, 27.9
// against 25.6), and the decoder keeps them there.
#include <algorithm>

#include "kf_device.h"
#include "kf_launch.h"

namespace kf {
namespace {

constexpr int kAttnThreads = 512, kAttnWaves = kAttnThreads / 64;
constexpr int kAttnSlices = 4;   // of d
constexpr int kAttnK = 16;       // K rows of a slice loaded together
constexpr int kAttnV = 4;        // V steps loaded together; the first ones before the softmax

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

// LDS floats: q [d], the wavefronts' max and sum [16], partial scores [4][max_seq] (then row 0 holds the
// exponentials), and the V sums (up to 4096) over rows 1..3 of the scores when they fit, else after
// them.
__host__ __device__ inline int attn_sum_off(int max_seq, int d) {
  return d + 16 + (3 * max_seq >= 4096 ? max_seq : kAttnSlices * max_seq);
}

// VEC: max_seq is even and cache_k 4-byte aligned, keys are read in pairs.
template <bool VEC>
__global__ __launch_bounds__(kAttnThreads) void decode_attention_kernel(const half_t* __restrict__ q,
                                                                        const half_t* __restrict__ cache_k,
                                                                        const half_t* __restrict__ cache_v,
                                                                        const half_t* __restrict__ mask,
                                                                        half_t* __restrict__ out, int rep, int d,
                                                                        int max_seq, int mask_stride, float scale) {
  constexpr int KPL = VEC ? 2 : 1;                                        // keys per lane
  constexpr int BLOCK = KPL * 64 * kAttnWaves / kAttnSlices;              // keys per pass
  extern __shared__ __attribute__((aligned(16))) float attn_lds[];
  float* const qs = attn_lds;
  float* const stat = attn_lds + d;
  float* const part = stat + 16;
  float* const sums = attn_lds + attn_sum_off(max_seq, d);
  const int h = blockIdx.x, kv = h / rep;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const half_t* const kb = cache_k + (size_t)kv * d * max_seq;
  const half_t* const vb = cache_v + (size_t)kv * max_seq * d;
  const half_t* const mrow = mask + (size_t)h * mask_stride;

  // K rows i .. i + kAttnK - 1 of this lane's keys; rows past the slice re-read its last one.
  const int slice = wave & (kAttnSlices - 1), dn = d / kAttnSlices, d0 = slice * dn;  // d % 8 == 0
  const int key0 = KPL * (64 * (wave / kAttnSlices) + lane);
  auto load_k = [&](half2_t (&k)[kAttnK], int i, int s) {
    const int sc = min(s, max_seq - KPL);
#pragma unroll
    for (int j = 0; j < kAttnK; ++j) {
      const uint32_t at = (uint32_t)((d0 + min(i + j, dn - 1)) * max_seq + sc);
      if constexpr (VEC) k[j] = *reinterpret_cast<const half2_t*>(kb + at);
      else k[j] = half2_t{kb[at], (half_t)0};
    }
  };
  // V steps i .. i + kAttnV - 1 of this lane; keys past the end re-read the last one.
  const int lpk = d >> 3;                                // lanes per key
  const int kps = kAttnThreads / lpk;                    // keys per step
  const int vk = tid / lpk, vc = tid - vk * lpk;         // vk == kps where d / 8 does not divide 512: idle
  auto load_v = [&](u32x4 (&v)[kAttnV], int i) {
#pragma unroll
    for (int j = 0; j < kAttnV; ++j)
      v[j] = load_u32x4(vb + (uint32_t)(min(vk + (i + j) * kps, max_seq - 1) * d + 8 * vc));
  };

  half2_t k[kAttnK];
  u32x4 v[kAttnV];
  const float q0 = tid < d ? (float)q[(size_t)h * d + tid] : 0.0f;  // d <= 256
  load_k(k, 0, key0);
  const float mask0 = tid < max_seq ? (float)mrow[tid] : 0.0f;
  load_v(v, 0);
  if (tid < d) qs[tid] = q0;
  __syncthreads();

  // Partial scores of this wavefront's slice of d.
  for (int base = 0; base < max_seq; base += BLOCK) {
    const int s = base + key0;
    float a0 = 0.0f, a1 = 0.0f;
    for (int i = 0; i < dn; i += kAttnK) {
      if (base + i > 0) load_k(k, i, s);
#pragma unroll
      for (int j = 0; j < kAttnK; ++j)
        if (i + j < dn) {  // uniform
          const float qj = qs[d0 + i + j];
          a0 = fmaf(qj, (float)k[j][0], a0);
          if constexpr (VEC) a1 = fmaf(qj, (float)k[j][1], a1);
        }
    }
    if (s < max_seq) {
      part[slice * max_seq + s] = a0;
      if constexpr (VEC) part[slice * max_seq + s + 1] = a1;
    }
  }
  __syncthreads();

  // Scores and their maximum, then the exponentials and their sum.  A NaN score drops out of the
  // maximum and makes its exponential, and so the row, NaN, as softmax does.
  float m = -__builtin_inff();
  for (int s = tid; s < max_seq; s += kAttnThreads) {
    const float sc = ((part[s] + part[max_seq + s]) + part[2 * max_seq + s]) + part[3 * max_seq + s];
    const float t = fmaf(sc, scale, s == tid ? mask0 : (float)mrow[s]);
    part[s] = t;
    m = fmaxf(m, t);
  }
  m = wave_max(m);
  if (lane == 0) stat[wave] = m;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kAttnWaves; ++i) m = fmaxf(m, stat[i]);
  float sum = 0.0f;
  for (int s = tid; s < max_seq; s += kAttnThreads) {
    const float e = __expf(part[s] - m);  // all keys masked: -inf - -inf, NaN
    part[s] = e;
    sum += e;
  }
  sum = wave_add(sum);
  if (lane == 0) stat[8 + wave] = sum;
  __syncthreads();

  // Weighted sum of V: this thread's 8 dims over keys vk, vk + kps, ...
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
  for (int i = 0; i * kps < max_seq; i += kAttnV) {
    if (i > 0) load_v(v, i);
#pragma unroll
    for (int j = 0; j < kAttnV; ++j) {
      const int s = vk + (i + j) * kps;
      if (s < max_seq && vk < kps) {
        const float p = part[s];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const half2_t h2 = bit_cast<half2_t>(v[j][e]);
          acc[2 * e] = fmaf(p, (float)h2[0], acc[2 * e]);
          acc[2 * e + 1] = fmaf(p, (float)h2[1], acc[2 * e + 1]);
        }
      }
    }
  }
  // Lanes of a wavefront that hold the same dims are lpk apart.
  const bool pow2 = (lpk & (lpk - 1)) == 0;  // lpk <= 32
  if (pow2) {
    for (int off = lpk; off < 64; off <<= 1) {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off);
    }
  }
  const int rows = pow2 ? kAttnWaves : kps, row = pow2 ? wave : vk;
  if (pow2 ? lane < lpk : vk < kps) {
#pragma unroll
    for (int e = 0; e < 8; ++e) sums[row * d + 8 * vc + e] = acc[e];
  }
  __syncthreads();
  if (tid < d) {
    float total = 0.0f, o = 0.0f;
#pragma unroll
    for (int i = 0; i < kAttnWaves; ++i) total += stat[8 + i];
#pragma unroll 8
    for (int r = 0; r < rows; ++r) o += sums[r * d + tid];
    out[(size_t)h * d + tid] = (half_t)(o / total);
  }
}

}  // namespace

hipError_t decode_attention_launch(const void* q, const void* cache_k, const void* cache_v, const void* mask, void* out,
                                   int heads, int kv_heads, int head_dim, int max_seq, int mask_stride, float scale,
                                   hipStream_t stream) {
  const size_t lds =
      sizeof(float) * std::max(attn_sum_off(max_seq, head_dim) + 4096, head_dim + 16 + kAttnSlices * max_seq);
  const auto fn = max_seq % 2 == 0 && (reinterpret_cast<uintptr_t>(cache_k) & 3) == 0 ? decode_attention_kernel<true>
                                                                                      : decode_attention_kernel<false>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLdsPerCu);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(fn, dim3(heads), dim3(kAttnThreads), lds, stream, static_cast<const half_t*>(q),
                     static_cast<const half_t*>(cache_k), static_cast<const half_t*>(cache_v),
                     static_cast<const half_t*>(mask), static_cast<half_t*>(out), heads / kv_heads, head_dim, max_seq,
                     mask_stride, scale);
  return hipGetLastError();
}

}  // namespace kf
