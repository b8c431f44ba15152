// INT4 dequant GEMM on the CDNA4 matrix cores (v_mfma_f32_16x16x32_f16).
//
// y[M, N] = x[M, K] @ W_hat^T with W_hat = fp16_rne(q * s) exactly as the reference's
// tensor-core path dequantizes (dequant_gemm_tc_kernel.cuh:100-112), fp32 accumulation,
// fp16 RNE output.  Optional split-K writes fp32 partials that kf::splitk_reduce sums in
// fixed split order (deterministic), the behaviour of the reference's splitk_reduce
// (dequant_gemm_tc_kernel.cuh:156-162).
//
// Kernel families (gemm_plan picks one, its tile and a split-K factor with a fitted cost model):
//   * streaming tiles (kf_stream.hip), 8 x 16 up to 64 x 64: small and medium M;
//   * gemm_dma4_kernel<TM, TN, NS>: (16 TM) x (32 TN) tiles fed by LDS-DMA, 8 wavefronts as 4 k-groups x
//     2 column halves, 128-k stages, for grids of up to about one tile per CU;
//   * gemm_dma2_kernel: 128 x 128 tiles fed by LDS-DMA, 4 wavefronts, for grids of several tiles per CU;
//   * gemm_wide_kernel: 192 x 256 tiles fed by LDS-DMA, 8 wavefronts, one workgroup per CU, for
//     grids of about one tile per CU (half the L2 -> LDS bytes per output of the 128 x 128 tiles).
//
// Common to the DMA tiles (gfx950: 4 SIMDs per CU, ~2 VALU ops hide under one 16x16x32 MFMA, LDS
// reads ~150-200 B/clk per CU):
//   * Every byte of a stage goes global -> LDS through LDS-DMA; the weights stay PACKED in LDS (4
//     bits per weight: 4x less LDS traffic than an fp16 W_hat tile) and each wavefront dequantizes
//     its own columns' words.
//   * LDS layouts are XOR-swizzled: sixteen consecutive lanes of a fragment read touch all 64 banks
//     (SQ_LDS_BANK_CONFLICT is 14-19% of SQ_LDS_IDX_ACTIVE in the four-k-group tiles).
//   * MFMA operands: lane l serves row / column l % 16 and k-group g = l / 16.
//   * Tiles are ordered in bands of group_m M-tiles (all N-tiles of a band before the next
//     band); the (split, tile) jobs of a launch, split-major, are dealt to the 8 XCDs in
//     contiguous runs of equal length, so the x rows an XCD uses stay in its L2, each weight
//     tile is fetched once per band, and no XCD holds more jobs than another (a 1-D grid: the
//     hardware deals workgroup i to XCD i % 8).
#include <algorithm>
#include <type_traits>

#include "kf_device.h"
#include "kf_launch.h"

namespace kf {
namespace {

constexpr int kXcds = 8;

// Job of this workgroup in a 1-D grid of ceil(jobs / 8) * 8 workgroups: XCD x (= blockIdx.x % 8)
// takes jobs x * per_xcd .. + per_xcd - 1.  Job j = split * tiles + tile.  False: no job.
__device__ __forceinline__ bool gemm_job(int tiles, int splits, int& split, int& tile) {
  const uint32_t jobs = tiles * splits;
  const uint32_t per_xcd = (jobs + kXcds - 1) / kXcds;
  const uint32_t j = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  if (j >= jobs) return false;
  split = splits > 1 ? j / (uint32_t)tiles : 0;
  tile = j - split * tiles;
  return true;
}

// ---- gemm_dma2_kernel: 128 x 128 tile, 2 k-groups (4 wavefronts), 64-k stages ---------------
//
// Every byte of a stage goes global -> LDS through the gfx950 LDS-DMA loads
// (global_load_lds_dwordx4 / _ushort: lane l's data lands at M0 + 16 l, or M0 + 4 l for
// 16-bit loads, zero-extended), so staging costs no registers and no VALU/LDS-write
// instructions, and the 128 accumulators per lane of a 128 x 64 wave tile fit with two
// wavefronts per SIMD.  A 128 x 64 wave tile makes one dequantized weight fragment feed 8
// MFMAs (the VALU work stays under the MFMA shadow) and one x fragment feed 4 (LDS reads
// stay well under the LDS bandwidth).
//
// Wavefront (kw, wn): column half wn (64 columns) and k-group kw, which takes k 32 kw ..
// 32 kw + 31 of every 64-k stage; the k-groups' accumulators are summed in fixed order through LDS
// at the end (in-block split-K).  Four wave tasks per 128 x 128 tile spread evenly over the 1024
// SIMDs when the grid has several tiles per CU.
//
// The DMA loads are issued from inline assembly with a "memory" clobber: the compiler
// neither tracks them nor moves LDS accesses across them, and the loop contains no
// compiler-tracked global loads, so its own waits never cover the prefetches.  Each
// wavefront issues exactly kDmaPerStage loads per stage (stage indices are clamped, never
// skipped), so "s_waitcnt vmcnt(kDmaPerStage)" means: the older stage has landed, the
// newer one may still be in flight.
//
// LDS stage layout (bytes): x rows of A_ROW = 2 BK bytes with 16-byte chunk c at slot
// c ^ a_swz(row); packed rows of BK / 2 bytes with 16-byte chunk h at h ^ b_swz(row).  Sixteen
// consecutive lanes of a fragment read touch all banks.  Three stages rotate.  Scales:
// a stage lies inside one group (G >= 64 = BK), so they live in their own ring of three slabs of
// 4-byte slots, one slab per group, fetched by the k-group 0 wavefronts with the first stage of the
// group (that stage costs those two wavefronts one more DMA, and their wait count for it is one
// higher).
struct DmaCfg {
  static constexpr int KW = 2, BM = 128, BN = 128, BK = 32 * KW, NS = 3, WAVES = 2 * KW, THREADS = 64 * WAVES;
  static constexpr int TM = 8, TN = 4;
  static constexpr int A_ROW = BK * 2;               // bytes of x per row and stage (128 / 256)
  static constexpr int A_CH = BK / 8;                // 16-byte chunks per x row (8 / 16)
  static constexpr int A_RSH = A_ROW >= 256 ? 0 : 1; // rows per 256-byte bank window: 1 or 2
  static constexpr int A_BYTES = BM * A_ROW;
  static constexpr int B_OFF = A_BYTES;
  static constexpr int B_ROW = BK / 2;               // bytes of packed weights per row and stage
  static constexpr int B_CH = BK / 32;               // 16-byte chunks per packed row (2 / 4)
  static constexpr int B_BYTES = BN * B_ROW;
  static constexpr int STAGE = B_OFF + B_BYTES;
  static constexpr int S_SLAB = BN * 4;              // [BN] 4-byte scale slots
  static constexpr int S_RING = NS * STAGE;          // per-group ring: [NS][BN]
  static constexpr int RING_END = S_RING + NS * S_SLAB;
  static constexpr int OUT_ROW = BN * 2 + 16;        // epilogue fp16 tile row stride (bytes), padded
  static constexpr int WAVE_TILE = TM * TN * 256 * 4;  // fp32 partial tile of one wavefront
  static constexpr int RED_BYTES = (KW / 2) * 2 * WAVE_TILE;  // k-group partials staged at once
  static constexpr int SMEM = RING_END > RED_BYTES ? (RING_END > BM * OUT_ROW ? RING_END : BM * OUT_ROW)
                                                   : (RED_BYTES > BM * OUT_ROW ? RED_BYTES : BM * OUT_ROW);
  static constexpr int kDmaPerStage = 5;             // per wavefront: 4 x, 1 packed (+1 scales, see below)
  static_assert(A_BYTES == 4 * 1024 * WAVES && B_BYTES == 1024 * WAVES, "4 x and 1 packed DMA per wavefront");
  static_assert(SMEM <= 160 * 1024, "LDS");
};

__device__ __forceinline__ void dma_16B(uint32_t lds, const void* src) {
  asm volatile("global_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ void dma_u16(uint32_t lds, const void* src) {
  asm volatile("global_load_lds_ushort %1, off" ::"{m0}"(lds), "v"(src) : "memory");
}

__global__ __launch_bounds__(DmaCfg::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_dma2_kernel(const half_t* __restrict__ x, const uint32_t* __restrict__ packed,
                     const half_t* __restrict__ scales, half_t* __restrict__ y, float* __restrict__ ws, int M, int N,
                     int K, int log2_group, int stages_per_split, int splits, int tiles_m, int tiles_n,
                     int group_m) {
  using C = DmaCfg;
  constexpr int BM = C::BM, BN = C::BN, BK = C::BK, NS = C::NS, THREADS = C::THREADS, TM = C::TM, TN = C::TN;
  constexpr int A_ROW = C::A_ROW, B_ROW = C::B_ROW, B_OFF = C::B_OFF, STAGE = C::STAGE, OUT_ROW = C::OUT_ROW;
  constexpr int kDmaPerStage = C::kDmaPerStage;
  __shared__ __attribute__((aligned(16))) unsigned char smem[C::SMEM];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1;
  const int kw = wave >> 1;
  const int g = lane >> 4;
  const int l16 = lane & 15;

  int split, t;
  if (!gemm_job(tiles_m * tiles_n, splits, split, t)) return;
  const int band = group_m * tiles_n;
  const int bi = t / band;
  const int tb = t - bi * band;
  const int gm = min(group_m, tiles_m - bi * group_m);
  const int m0 = (bi * group_m + tb % gm) * BM;
  const int n0 = (tb / gm) * BN;

  const int nst = K / BK;
  const int st_begin = split * stages_per_split;
  const int last = min(nst, st_begin + stages_per_split) - 1;
  const int ns = last + 1 - st_begin;

  // XOR swizzles: x chunk c of row r at slot c ^ a_swz(r); packed chunk h of row r at h ^ b_swz(r).
  auto a_swz = [](int row) { return (row >> C::A_RSH) & (C::A_CH - 1); };
  auto b_swz = [](int row) { return (row / (16 / C::B_CH)) & (C::B_CH - 1); };

  // Per-lane DMA sources at k = 0 (advanced by the stage's k offset).  x: this wave's 4
  // instructions of 1 KiB cover 1024 / A_ROW rows each; packed: one instruction of 1 KiB.
  constexpr int A_RPI = 1024 / A_ROW, A_LPR = A_ROW / 16;  // rows per instruction, lanes per row
  constexpr int B_RPI = 1024 / B_ROW, B_LPR = B_ROW / 16;
  const half_t* a_src[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int row = A_RPI * (4 * wave + q) + lane / A_LPR;
    a_src[q] = x + (size_t)min(m0 + row, M - 1) * K + 8 * ((lane % A_LPR) ^ a_swz(row));
  }
  const int brow = B_RPI * wave + lane / B_LPR;
  const uint32_t* b_src =
      packed + (size_t)min(n0 + brow, N - 1) * (K >> 3) + 4 * ((lane % B_LPR) ^ b_swz(brow));
  const int groups = K >> log2_group;
  const half_t* s_src = scales + (size_t)min(n0 + 64 * wn + lane, N - 1) * groups;
  const uint32_t smem_base = (uint32_t)(uintptr_t)smem;

  // Per-group scale ring: split-local stage i (clamped) starts a scale group when
  // i == 0 or its k0 is a multiple of G; groups are numbered from the split's first stage.
  // The clamped repeats of the last stage past the split's end never start one.
  const int log2_spg = log2_group - 6;  // log2(stages per group)
  auto starts_group = [&](int i) {
    const int st = st_begin + i;
    return i == 0 || (st <= last && (st & ((1 << log2_spg) - 1)) == 0);
  };
  auto group_of = [&](int i) {  // split-local group index of split-local stage i (i <= ns - 1)
    return ((st_begin + i) >> log2_spg) - (st_begin >> log2_spg);
  };
  // DMA of split-local stage i (clamped) into buffer i % NS, plus scales.  Returns whether
  // this wavefront issued a scale load (one more outstanding load).
  auto issue = [&](int i, int buf) {  // buf == i % NS
    const int st = min(st_begin + i, last);
    const int k0 = st * BK;
    const uint32_t base = __builtin_amdgcn_readfirstlane(smem_base + (uint32_t)(buf * STAGE));
#pragma unroll
    for (int q = 0; q < 4; ++q) dma_16B(base + 1024 * (4 * wave + q), a_src[q] + k0);
    dma_16B(base + B_OFF + 1024 * wave, b_src + (k0 >> 3));
    const bool sc = kw == 0 && starts_group(i);
    if (sc) {
      const uint32_t sbase = __builtin_amdgcn_readfirstlane(
          smem_base + (uint32_t)(C::S_RING + (group_of(i) % NS) * C::S_SLAB + 256 * wn));
      dma_u16(sbase, s_src + (k0 >> log2_group));
    }
    return sc;
  };
  auto wait_older = [&](bool newer_has_scales) {  // all but the newest stage's loads landed
    if (newer_has_scales)
      wait_vmcnt<kDmaPerStage + 1>();
    else
      wait_vmcnt<kDmaPerStage>();
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // Lane-dependent LDS offsets inside a stage.  x: row l16 (+16 per block), chunk 4 kw + g.
  // packed: row 64 wn + 16 j + l16, dword 4 kw + g.  scales: column 64 wn + 16 j + l16.
  const int a_off = l16 * A_ROW + 16 * ((4 * kw + g) ^ a_swz(l16));
  const int b_off = B_OFF + (64 * wn + l16) * B_ROW + 16 * (kw ^ b_swz(l16)) + 4 * g;
  const int s_off = 4 * (64 * wn + l16);

  const UnpackConsts uc = unpack_consts();
  half8_t a[TM];
  uint32_t w[TN];
  half2_t s2[TN];
  auto read_frags = [&](int i, int buf) {  // buf == i % NS, a compile-time constant at the call
    const unsigned char* st = smem + buf * STAGE;
    const unsigned char* slab = smem + C::S_RING + (group_of(i) % NS) * C::S_SLAB;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      w[j] = *reinterpret_cast<const uint32_t*>(st + b_off + 16 * B_ROW * j);
      const half_t sc = *reinterpret_cast<const half_t*>(slab + s_off + 64 * j);
      s2[j] = half2_t{sc, sc};
    }
#pragma unroll
    for (int q = 0; q < TM; ++q) a[q] = *reinterpret_cast<const half8_t*>(st + a_off + 16 * A_ROW * q);
  };

  // Stage i: DMA issued at iteration i - 2 into buffer i % NS; at iteration i - 1 each
  // wavefront waits for its own loads of it and the barrier publishes it; at iteration i
  // its fragments are read and its MFMAs run.  The DMA of stage i + 2 (iteration i)
  // overwrites the buffer of stage i - 1, whose reads completed before the barrier of
  // iteration i - 1 (lgkmcnt(0) precedes every barrier).  Likewise the scale slab
  // of group q is fetched with q's first stage i (iteration i - 2) into the slab of group
  // q - 3, last read at a stage <= i - 3 (groups span >= 1 stage), before that barrier.
  // The loop is unrolled by NS so every buffer offset is a compile-time immediate.
  issue(0, 0);
  wait_older(issue(1, 1));
  __syncthreads();
  auto step = [&](auto buf_c, int s) {  // stage s, held in buffer CUR == s % NS
    constexpr int CUR = decltype(buf_c)::value;
    read_frags(s, CUR);
    wait_older(issue(s + 2, (CUR + 2) % NS));  // stage s + 1 landed
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const half8_t b = dequant8(w[j], s2[j], uc);
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a[i], acc[i][j], 0, 0, 0);
    }
  };
  static_assert(NS == 3, "the unrolled loop below assumes three stages");
  for (int s = 0; s < ns; s += NS) {
    step(std::integral_constant<int, 0>(), s);
    if (s + 1 >= ns) break;
    step(std::integral_constant<int, 1>(), s + 1);
    if (s + 2 >= ns) break;
    step(std::integral_constant<int, 2>(), s + 2);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped tail loads, before LDS is reused
  __syncthreads();

  // The k-groups' partial tiles are added in fixed order (a0 + a1) through LDS.
  float* red = reinterpret_cast<float*>(smem) + wn * TM * TN * 256 + 4 * lane;
  if (kw == 1) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) *reinterpret_cast<float4_t*>(red + (i * TN + j) * 256) = acc[i][j];
  }
  __syncthreads();
  if (kw == 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += *reinterpret_cast<const float4_t*>(red + (i * TN + j) * 256);
  }

  // The MFMAs take the weights as their first operand, so each 16 x 16 block comes out
  // transposed: lane l, element r holds y row l%16, column 4*(l/16)+r (four consecutive columns:
  // one 8-byte LDS write per block in the epilogue; same products, same order, same bits).
  if (ws) {
    if (kw == 0) {
      float* part = ws + (size_t)split * M * N;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = m0 + 16 * i + l16, col = n0 + 64 * wn + 16 * j + 4 * g;
          if (row < M && col < N) *reinterpret_cast<float4_t*>(part + (size_t)row * N + col) = acc[i][j];
        }
    }
    return;
  }
  // fp16 tile through LDS, then 16-byte row-major stores by all wavefronts.
  __syncthreads();  // the partial tiles have been read
  if (kw == 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const half2_t lo = {(half_t)acc[i][j][0], (half_t)acc[i][j][1]};
        const half2_t hi = {(half_t)acc[i][j][2], (half_t)acc[i][j][3]};
        *reinterpret_cast<u32x2*>(smem + (16 * i + l16) * OUT_ROW + 2 * (64 * wn + 16 * j + 4 * g)) =
            u32x2{bit_cast<uint32_t>(lo), bit_cast<uint32_t>(hi)};
      }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < BM * BN / 8 / THREADS; ++q) {
    const int c = tid + THREADS * q;
    const int row = c >> 4, chunk = c & 15;
    const int gr = m0 + row, gc = n0 + 8 * chunk;
    if (gr < M && gc < N)
      *reinterpret_cast<u32x4*>(y + (size_t)gr * N + gc) = *reinterpret_cast<const u32x4*>(smem + row * OUT_ROW + 16 * chunk);
  }
}

// ---- gemm_dma4_kernel: (16 TM) x (32 TN) tile, 4 k-groups (8 wavefronts), 128-k stages ------------
//
// The tile for grids of up to about one workgroup per CU: eight wavefronts as 2 column halves x 4
// k-groups, so a small tile still keeps two wavefronts on every SIMD, and TM row blocks per
// dequantized word.  The row count is the point of the template: the tile height is chosen so that M
// pads little and the grid fills the CUs (M = 517 in 112-row tiles is 560 rows, in 128-row tiles 640;
// M = 200 in 80-row tiles is three tiles).  Stages rotate through NS buffers, NS - 1 of them in
// flight, and the loop is rolled (buffer offsets in registers): each wavefront issues the same
// number of copies per stage, so one counted wait serves the whole loop.  Copies past a tile's last
// instruction repeat that instruction (same bytes to the same place).
// MI355X, against the 64 x 128 register-staged and 128 x 128 tiles chosen before: N x K = 2048 x 5632 at
// M = 517 / 768: 42.8 / 43.9 -> 24.8 / 29.0 us; 4096 x 4096 at M = 517: 34.4 -> 26.5; 1536 x 8960 at
// M = 517 / 1024: 45.8 / 55.4 -> 27.4 / 42.7; 128 x 128 itself (2048 x 5632 at M = 2048): 52.1 -> 47.9.
template <int TM_, int TN_, int NS_>
struct Dma4Cfg {
  static constexpr int TM = TM_, TN = TN_, NS = NS_;
  static constexpr int BM = 16 * TM, BN = 32 * TN, BK = 128, WAVES = 8, THREADS = 64 * WAVES;
  static constexpr int A_ROW = 2 * BK;                         // bytes of x per row and stage
  static constexpr int A_INST = BM * A_ROW / 1024;             // copies of 4 rows
  static constexpr int A_PW = (A_INST + WAVES - 1) / WAVES;    // ... per wavefront
  static constexpr int B_ROW = BK / 2;                         // bytes of packed weights per row and stage
  static constexpr int B_OFF = BM * A_ROW;
  static constexpr int B_INST = BN * B_ROW / 1024;             // copies of 16 rows
  static constexpr int B_PW = (B_INST + WAVES - 1) / WAVES;
  static constexpr int S_OFF = B_OFF + BN * B_ROW;             // 4-byte scale slots [BN][2]: one per 64 k
  static constexpr int S_INST = BN / 32;                       // copies of 32 columns
  static constexpr int S_PW = (S_INST + WAVES - 1) / WAVES;
  static constexpr int STAGE = S_OFF + BN * 8;
  static constexpr int kDmaPerStage = A_PW + B_PW + S_PW;
  static constexpr int OUT_ROW = BN * 2 + 16;
  static constexpr int RED = 4 * TM * TN * 1024;               // two k-groups' partial tiles
  static constexpr int OUT = BM * OUT_ROW;
  static constexpr int SMEM = NS * STAGE > RED ? (NS * STAGE > OUT ? NS * STAGE : OUT) : (RED > OUT ? RED : OUT);
  static_assert(BN % 64 == 0 && SMEM <= 160 * 1024, "tile");
};

template <class C>
__device__ __forceinline__ void dma4_tile(const half_t* x, const uint32_t* packed, const half_t* scales, half_t* y,
                                          float* part, int M, int N, int K, int log2_group, int m0, int n0,
                                          int st_begin, int ns) {
  constexpr int BM = C::BM, BN = C::BN, BK = C::BK, NS = C::NS, TM = C::TM, TN = C::TN, WAVES = C::WAVES;
  constexpr int A_ROW = C::A_ROW, B_ROW = C::B_ROW, OUT_ROW = C::OUT_ROW;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[C::SMEM];  // static: no attribute call above 64 KiB

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1;
  const int kw = wave >> 1;
  const int g = lane >> 4;
  const int l16 = lane & 15;

  // x chunk c (16 bytes) of row r at slot c ^ (r & 15); packed chunk h at h ^ ((r >> 2) & 3).
  const half_t* a_src[C::A_PW];
  uint32_t a_dst[C::A_PW];
#pragma unroll
  for (int q = 0; q < C::A_PW; ++q) {
    const int i = min(q * WAVES + wave, C::A_INST - 1);
    const int row = 4 * i + (lane >> 4);
    a_src[q] = x + (size_t)min(m0 + row, M - 1) * K + (size_t)st_begin * BK + 8 * ((lane & 15) ^ (row & 15));
    a_dst[q] = 1024 * i;
  }
  const uint32_t* b_src[C::B_PW];
  uint32_t b_dst[C::B_PW];
#pragma unroll
  for (int q = 0; q < C::B_PW; ++q) {
    const int i = min(q * WAVES + wave, C::B_INST - 1);
    const int row = 16 * i + (lane >> 2);
    b_src[q] = packed + (size_t)min(n0 + row, N - 1) * (K >> 3) + (size_t)st_begin * (BK / 8) +
               4 * ((lane & 3) ^ ((row >> 2) & 3));
    b_dst[q] = C::B_OFF + 1024 * i;
  }
  const half_t* s_src[C::S_PW];
  uint32_t s_dst[C::S_PW];
#pragma unroll
  for (int q = 0; q < C::S_PW; ++q) {
    const int i = min(q * WAVES + wave, C::S_INST - 1);
    s_src[q] = scales + (size_t)min(n0 + 32 * i + (lane >> 1), N - 1) * (K >> log2_group);
    s_dst[q] = C::S_OFF + 256 * i;
  }
  const uint32_t smem_base = (uint32_t)(uintptr_t)smem;
  auto issue = [&](int i, uint32_t slot) {  // split-local stage i (clamped) into the buffer at `slot`
    const size_t st = min(i, ns - 1);
    const uint32_t base = smem_base + slot;
    const int group = ((st_begin + (int)st) * BK + 64 * (lane & 1)) >> log2_group;
#pragma unroll
    for (int q = 0; q < C::A_PW; ++q) dma_16B(__builtin_amdgcn_readfirstlane(base + a_dst[q]), a_src[q] + st * BK);
#pragma unroll
    for (int q = 0; q < C::B_PW; ++q)
      dma_16B(__builtin_amdgcn_readfirstlane(base + b_dst[q]), b_src[q] + st * (BK / 8));
#pragma unroll
    for (int q = 0; q < C::S_PW; ++q)
      dma_u16(__builtin_amdgcn_readfirstlane(base + s_dst[q]), s_src[q] + group);
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // Lane offsets inside a stage: x row l16, chunk 4 kw + g; packed row of column 16 TN wn + l16, dword
  // 4 kw + g; its scale for this k-group's 64 k.
  const int a_off = l16 * A_ROW + 16 * ((4 * kw + g) ^ l16);
  const int b_off = C::B_OFF + (16 * TN * wn + l16) * B_ROW + 16 * (kw ^ ((l16 >> 2) & 3)) + 4 * g;
  const int s_off = C::S_OFF + 8 * (16 * TN * wn + l16) + 4 * (kw >> 1);
  const UnpackConsts uc = unpack_consts();

  // Stage s is copied NS - 1 iterations ahead.  At iteration s every wavefront reads its fragments
  // of stage s, issues stage s + NS - 1 into the buffer of stage s - 1 (whose reads completed before
  // the barrier of iteration s - 1), waits until its own copies of stage s + 1 have landed, and the
  // barrier publishes them.
  constexpr int kInFlight = (NS - 2) * C::kDmaPerStage;
  static_assert(kInFlight <= 63, "vmcnt is six bits");
#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue(i, i * C::STAGE);
  wait_vmcnt<kInFlight>();
  __syncthreads();
  uint32_t slot = 0, next = (NS - 1) * C::STAGE;
#pragma unroll 1
  for (int s = 0; s < ns; ++s) {
    half8_t a[TM];
    uint32_t w[TN];
    half2_t s2[TN];
    const unsigned char* st = smem + slot;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      w[j] = *reinterpret_cast<const uint32_t*>(st + b_off + 16 * B_ROW * j);
      const half_t sc = *reinterpret_cast<const half_t*>(st + s_off + 128 * j);
      s2[j] = half2_t{sc, sc};
    }
#pragma unroll
    for (int q = 0; q < TM; ++q) a[q] = *reinterpret_cast<const half8_t*>(st + a_off + 16 * A_ROW * q);
    issue(s + NS - 1, next);
    next = slot;
    slot = slot + C::STAGE == NS * C::STAGE ? 0 : slot + C::STAGE;
    wait_vmcnt<kInFlight>();
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const half8_t b = dequant8(w[j], s2[j], uc);
#pragma unroll
      for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a[i], acc[i][j], 0, 0, 0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped tail copies, before LDS is reused
  __syncthreads();

  // The k-groups' partial tiles are added in fixed order through LDS: (a0 + a2) + (a1 + a3).  Round
  // r hands k-group giver's tile to k-group taker through slot h (one 2 x wave-tile region per
  // slot); straight-line code keeps acc in registers.
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const bool give = r ? kw == 1 : kw >= 2;
    const bool take = r ? kw == 0 : kw < 2;
    const int h = r ? 0 : (kw & 1);
    float* base = red + ((h * 2 + wn) * TM * TN) * 256 + 4 * lane;
    if (r > 0) __syncthreads();  // the first round's tiles have been read
    if (give) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *reinterpret_cast<float4_t*>(base + (i * TN + j) * 256) = acc[i][j];
    }
    __syncthreads();
    if (take) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += *reinterpret_cast<const float4_t*>(base + (i * TN + j) * 256);
    }
  }

  if (part) {
    if (kw == 0) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = m0 + 16 * i + l16, col = n0 + 16 * TN * wn + 16 * j + 4 * g;
          if (row < M && col < N) *reinterpret_cast<float4_t*>(part + (size_t)row * N + col) = acc[i][j];
        }
    }
    return;
  }
  // fp16 tile through LDS, then 16-byte row-major stores by all wavefronts.
  __syncthreads();  // the partial tiles have been read
  if (kw == 0) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const half2_t lo = {(half_t)acc[i][j][0], (half_t)acc[i][j][1]};
        const half2_t hi = {(half_t)acc[i][j][2], (half_t)acc[i][j][3]};
        *reinterpret_cast<u32x2*>(smem + (16 * i + l16) * OUT_ROW + 2 * (16 * TN * wn + 16 * j + 4 * g)) =
            u32x2{bit_cast<uint32_t>(lo), bit_cast<uint32_t>(hi)};
      }
  }
  __syncthreads();
  for (int c = tid; c < BM * BN / 8; c += C::THREADS) {
    const int row = c / (BN / 8), chunk = c % (BN / 8);
    const int gr = m0 + row, gc = n0 + 8 * chunk;
    if (gr < M && gc < N)
      *reinterpret_cast<u32x4*>(y + (size_t)gr * N + gc) = *reinterpret_cast<const u32x4*>(smem + row * OUT_ROW + 16 * chunk);
  }
}

// Rows and columns of job t's tile: bands of group_m row tiles, all column tiles of a band before the next.
__device__ __forceinline__ void band_tile(int t, int tiles_m, int tiles_n, int group_m, int& mt, int& nt) {
  const uint32_t band = group_m * tiles_n, bi = (uint32_t)t / band, tb = t - bi * band;
  const uint32_t gm = min(group_m, tiles_m - (int)bi * group_m);
  nt = gm > 1 ? tb / gm : tb;
  mt = bi * group_m + (tb - nt * gm);
}

// The arguments fit the 14 dwords that arrive in registers, as those of stream_kernel do; the tile counts
// come from M and N.  Tiles of up to 80 rows gain 1.5-3% of their time by that: 28672 x 4096 at M = 32 21.6 -> 21.1 us,
// 4096 x 4096 at M = 517 26.5 -> 26.0.  The non-temporal hint on weights that one row tile reads, which helps the
// streaming tiles, costs 5-15% here (21.1 -> 23.7): a stage takes half of each 128-byte line.
template <class C>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_dma4_kernel(const half_t* __restrict__ x, const uint32_t* __restrict__ packed,
                      const half_t* __restrict__ scales, half_t* __restrict__ y, float* __restrict__ ws, int M, int N,
                      int K, uint32_t stages_splits_group) {
  const int stages_per_split = stages_splits_group >> 8, splits = (stages_splits_group >> 4) & 15;
  const int log2_group = stages_splits_group & 15;
  const int tiles_m = ((uint32_t)M + C::BM - 1) / C::BM, tiles_n = ((uint32_t)N + C::BN - 1) / C::BN;
  int split, t, mt, nt;
  if (!gemm_job(tiles_m * tiles_n, splits, split, t)) return;
  band_tile(t, tiles_m, tiles_n, max(1, tiles_m / kXcds), mt, nt);
  const int st_begin = split * stages_per_split;
  const int ns = min(K / C::BK - st_begin, stages_per_split);  // >= 1: no split is empty
  dma4_tile<C>(x, packed, scales, y, ws ? ws + (size_t)split * M * N : nullptr, M, N, K, log2_group, mt * C::BM,
               nt * C::BN, st_begin, ns);
}

// Several problems of one M, K and group size in one launch (see stream_grouped_kernel): the tiles of
// siblings fill the last round of workgroups together.
template <class C>
__global__ __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_dma4_grouped_kernel(int count, int M, int K, int log2_group, int tiles_m, int tiles_n, int group_m,
                              const GroupTable table) {
  int split, t, mt, nt;
  if (!gemm_job(tiles_m * tiles_n, 1, split, t)) return;
  band_tile(t, tiles_m, tiles_n, group_m, mt, nt);
  const GroupEntry e = group_entry(table, count, nt);
  dma4_tile<C>(e.x, e.packed, e.scales, e.y, nullptr, M, e.N, K, log2_group, mt * C::BM, (nt - e.tile0) * C::BN, 0,
               K / C::BK);
}

// Wide DMA-fed tile: 192 x 256 per workgroup, 8 wavefronts as 2 x 4 wave tiles of 96 x 64, every
// wavefront over the whole 64-k stage (no k split, no partial-tile reduction), one workgroup per
// CU (99 KiB of stages and scale ring).  Per 64-k stage a CU moves 32 KiB from L2 into LDS for
// 192 x 256 outputs, against 40 KiB for the two 128 x 128 tiles of gemm_dma2_kernel (half the
// outputs): x, fp16 and the larger operand, is re-read from L2 once per 256 columns instead of
// once per 128.  Stage pipeline, swizzles, scale ring and counted waits are those of
// gemm_dma2_kernel.  MI355X, M = 2048, N = 5632, K = 2048 (242 tiles, one per CU): 52 us = 906
// TFLOPS against 56 us for the 128 x 128 tiles.  A tile alone on its CU takes 44 us (K = 2048), so
// the tile pays only where its count fills whole rounds of 256; gemm_plan weighs that.
struct WideCfg {
  static constexpr int BM = 192, BN = 256, BK = 64, NS = 3, WM = 2, WN = 4, WAVES = WM * WN, THREADS = 64 * WAVES;
  static constexpr int TM = 6, TN = 4;               // 16 x 16 blocks per wavefront
  static constexpr int A_ROW = BK * 2;               // 128 bytes of x per row and stage
  static constexpr int A_CH = BK / 8;                // 8 chunks of 16 bytes
  static constexpr int A_BYTES = BM * A_ROW;         // 24 KiB
  static constexpr int B_OFF = A_BYTES;
  static constexpr int B_ROW = BK / 2;               // 32 bytes of packed weights per row and stage
  static constexpr int B_CH = BK / 32;               // 2 chunks
  static constexpr int B_BYTES = BN * B_ROW;         // 8 KiB
  static constexpr int STAGE = B_OFF + B_BYTES;
  static constexpr int S_SLAB = BN * 4;              // [BN] 4-byte slots
  static constexpr int S_RING = NS * STAGE;
  static constexpr int RING_END = S_RING + NS * S_SLAB;
  static constexpr int OUT_ROW = BN * 2 + 16;
  static constexpr int SMEM = RING_END > BM * OUT_ROW ? RING_END : BM * OUT_ROW;
  static constexpr int A_DMA = A_BYTES / 1024 / WAVES;  // 3 x instructions per wavefront and stage
  static constexpr int kDmaPerStage = A_DMA + 1;        // + 1 packed
  static_assert(A_DMA * 1024 * WAVES == A_BYTES && B_BYTES == 1024 * WAVES, "DMA split");
  static_assert(SMEM <= 160 * 1024, "LDS");
};

__global__ __launch_bounds__(WideCfg::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemm_wide_kernel(const half_t* __restrict__ x, const uint32_t* __restrict__ packed,
                      const half_t* __restrict__ scales, half_t* __restrict__ y, float* __restrict__ ws, int M, int N,
                      int K, int log2_group, int stages_per_split, int splits, int tiles_m, int tiles_n,
                      int group_m) {
  using C = WideCfg;
  constexpr int BM = C::BM, BN = C::BN, BK = C::BK, NS = C::NS, THREADS = C::THREADS, TM = C::TM, TN = C::TN;
  constexpr int A_ROW = C::A_ROW, B_ROW = C::B_ROW, B_OFF = C::B_OFF, STAGE = C::STAGE, OUT_ROW = C::OUT_ROW;
  constexpr int kDmaPerStage = C::kDmaPerStage, A_DMA = C::A_DMA;
  __shared__ __attribute__((aligned(16))) unsigned char smem[C::SMEM];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3;
  const int wm = wave >> 2;
  const int g = lane >> 4;
  const int l16 = lane & 15;

  int split, t;
  if (!gemm_job(tiles_m * tiles_n, splits, split, t)) return;
  const int band = group_m * tiles_n;
  const int bi = t / band;
  const int tb = t - bi * band;
  const int gm = min(group_m, tiles_m - bi * group_m);
  const int m0 = (bi * group_m + tb % gm) * BM;
  const int n0 = (tb / gm) * BN;

  const int nst = K / BK;
  const int st_begin = split * stages_per_split;
  const int last = min(nst, st_begin + stages_per_split) - 1;
  const int ns = last + 1 - st_begin;

  // XOR swizzles: x chunk c of row r at slot c ^ a_swz(r); packed chunk h of row r at h ^ b_swz(r).
  auto a_swz = [](int row) { return (row >> 1) & (C::A_CH - 1); };
  auto b_swz = [](int row) { return (row >> 3) & (C::B_CH - 1); };

  // DMA sources at k = 0.  x: A_DMA instructions of 1 KiB (8 rows) per wavefront; packed: one
  // of 1 KiB (32 rows).
  const half_t* a_src[A_DMA];
#pragma unroll
  for (int q = 0; q < A_DMA; ++q) {
    const int row = 8 * (A_DMA * wave + q) + (lane >> 3);
    a_src[q] = x + (size_t)min(m0 + row, M - 1) * K + 8 * ((lane & 7) ^ a_swz(row));
  }
  const int brow = 32 * wave + (lane >> 1);
  const uint32_t* b_src = packed + (size_t)min(n0 + brow, N - 1) * (K >> 3) + 4 * ((lane & 1) ^ b_swz(brow));
  const int groups = K >> log2_group;
  const half_t* s_src = scales + (size_t)min(n0 + 64 * wn + lane, N - 1) * groups;
  const uint32_t smem_base = (uint32_t)(uintptr_t)smem;

  const int log2_spg = log2_group - 6;  // log2(stages per group)
  auto starts_group = [&](int i) {
    const int st = st_begin + i;
    return i == 0 || (st <= last && (st & ((1 << log2_spg) - 1)) == 0);
  };
  auto group_of = [&](int i) { return ((st_begin + i) >> log2_spg) - (st_begin >> log2_spg); };
  auto issue = [&](int i, int buf) {
    const int st = min(st_begin + i, last);
    const int k0 = st * BK;
    const uint32_t base = __builtin_amdgcn_readfirstlane(smem_base + (uint32_t)(buf * STAGE));
#pragma unroll
    for (int q = 0; q < A_DMA; ++q) dma_16B(base + 1024 * (A_DMA * wave + q), a_src[q] + k0);
    dma_16B(base + B_OFF + 1024 * wave, b_src + (k0 >> 3));
    const bool sc = wm == 0 && starts_group(i);
    if (sc) {
      const uint32_t sbase = __builtin_amdgcn_readfirstlane(
          smem_base + (uint32_t)(C::S_RING + (group_of(i) % NS) * C::S_SLAB + 256 * wn));
      dma_u16(sbase, s_src + (k0 >> log2_group));
    }
    return sc;
  };
  auto wait_older = [&](bool newer_has_scales) {
    if (newer_has_scales)
      wait_vmcnt<kDmaPerStage + 1>();
    else
      wait_vmcnt<kDmaPerStage>();
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // Lane offsets: x row 96 wm + l16 (+16 per block), chunk 4 kk + g; packed row 64 wn + 16 j + l16,
  // chunk kk, dword g; scales column 64 wn + 16 j + l16.
  const int a_row0 = 96 * wm + l16;
  const int a_off0 = a_row0 * A_ROW + 16 * ((0 + g) ^ a_swz(a_row0));
  const int a_off1 = a_row0 * A_ROW + 16 * ((4 + g) ^ a_swz(a_row0));
  const int b_row0 = 64 * wn + l16;
  const int b_off0 = B_OFF + b_row0 * B_ROW + 16 * (0 ^ b_swz(b_row0)) + 4 * g;
  const int b_off1 = B_OFF + b_row0 * B_ROW + 16 * (1 ^ b_swz(b_row0)) + 4 * g;
  const int s_off = 4 * (64 * wn + l16);

  const UnpackConsts uc = unpack_consts();
  half8_t a[2][TM];
  uint32_t w[2][TN];
  half2_t s2[TN];
  auto read_frags = [&](int i, int buf) {
    const unsigned char* st = smem + buf * STAGE;
    const unsigned char* slab = smem + C::S_RING + (group_of(i) % NS) * C::S_SLAB;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      w[0][j] = *reinterpret_cast<const uint32_t*>(st + b_off0 + 16 * B_ROW * j);
      w[1][j] = *reinterpret_cast<const uint32_t*>(st + b_off1 + 16 * B_ROW * j);
      const half_t sc = *reinterpret_cast<const half_t*>(slab + s_off + 64 * j);
      s2[j] = half2_t{sc, sc};
    }
#pragma unroll
    for (int q = 0; q < TM; ++q) {
      a[0][q] = *reinterpret_cast<const half8_t*>(st + a_off0 + 16 * A_ROW * q);
      a[1][q] = *reinterpret_cast<const half8_t*>(st + a_off1 + 16 * A_ROW * q);
    }
  };

  issue(0, 0);
  wait_older(issue(1, 1));
  __syncthreads();
  // Stage pipeline of gemm_dma2_kernel: stage i's fragments (both 32-k steps) are read at
  // iteration i, before the barrier after which stage i + 2's DMA may overwrite stage i - 1's
  // buffer; the scheduling barrier keeps the next stage's reads out of this stage's MFMAs.
  auto step = [&](auto buf_c, int s) {
    constexpr int CUR = decltype(buf_c)::value;
    __builtin_amdgcn_sched_barrier(0);
    read_frags(s, CUR);
    wait_older(issue(s + 2, (CUR + 2) % NS));
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const half8_t b = dequant8(w[kk][j], s2[j], uc);
#pragma unroll
        for (int i = 0; i < TM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a[kk][i], acc[i][j], 0, 0, 0);
      }
  };
  // Whole rounds of NS stages, then the remaining one or two: an exit in the middle of the
  // unrolled round made the compiler copy the accumulators between its copies of the round and
  // spill (256 VGPRs + 111 spilled against 236 without).
  static_assert(NS == 3, "the unrolled loop below assumes three stages");
  int s = 0;
  for (; s + NS <= ns; s += NS) {
    step(std::integral_constant<int, 0>(), s);
    step(std::integral_constant<int, 1>(), s + 1);
    step(std::integral_constant<int, 2>(), s + 2);
  }
  if (s < ns) step(std::integral_constant<int, 0>(), s);
  if (s + 1 < ns) step(std::integral_constant<int, 1>(), s + 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  // fp16 tile through LDS, then 16-byte row-major stores by all wavefronts (no split-K: ws unused).
  // The MFMAs take the weights as their first operand, so block (i, j) comes out transposed: lane
  // (g, l16) holds y[row 16 i + l16][columns 16 j + 4 g .. + 3], four consecutive fp16 that go to
  // LDS in one 8-byte write (a quarter of the writes of the row-per-element layout; the sums are
  // the same products added in the same order: bit-identical, 51.8 -> 50.6 us at M = 2048,
  // N = 5632, K = 2048).  Storing those 8 bytes straight to y instead measured 54.6 us.
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const half2_t lo = {(half_t)acc[i][j][0], (half_t)acc[i][j][1]};
      const half2_t hi = {(half_t)acc[i][j][2], (half_t)acc[i][j][3]};
      *reinterpret_cast<u32x2*>(smem + (96 * wm + 16 * i + l16) * OUT_ROW + 2 * (64 * wn + 16 * j + 4 * g)) =
          u32x2{bit_cast<uint32_t>(lo), bit_cast<uint32_t>(hi)};
    }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < BM * BN / 8 / THREADS; ++q) {
    const int c = tid + THREADS * q;
    const int row = c >> 5, chunk = c & 31;
    const int gr = m0 + row, gc = n0 + 8 * chunk;
    if (gr < M && gc < N)
      *reinterpret_cast<u32x4*>(y + (size_t)gr * N + gc) = *reinterpret_cast<const u32x4*>(smem + row * OUT_ROW + 16 * chunk);
  }
}

// y = fp16(sum over the splits of their fp32 partials, in split order), four outputs per thread; the
// partials of four splits are loaded together (one at a time, 4 bytes each, it took 2.4-5 us at
// M N = 131,072 .. 409,600 and 5-8 splits; now 2.2-2.9).
__global__ __launch_bounds__(256) void splitk_reduce(const float4_t* __restrict__ ws, u32x2* __restrict__ y, size_t mn4,
                                                      int splits) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < mn4; i += (size_t)gridDim.x * 256) {
    float4_t s = ws[i];
    int z = 1;
    for (; z + 3 < splits; z += 4) {
      const float4_t p0 = ws[z * mn4 + i], p1 = ws[(z + 1) * mn4 + i], p2 = ws[(z + 2) * mn4 + i],
                     p3 = ws[(z + 3) * mn4 + i];
      s += p0;
      s += p1;
      s += p2;
      s += p3;
    }
    for (; z < splits; ++z) s += ws[z * mn4 + i];
    const half2_t lo = {(half_t)s[0], (half_t)s[1]}, hi = {(half_t)s[2], (half_t)s[3]};
    y[i] = u32x2{bit_cast<uint32_t>(lo), bit_cast<uint32_t>(hi)};
  }
}

typedef void (*GemmFn)(const half_t*, const uint32_t*, const half_t*, half_t*, float*, int, int, int, int, int, int,
                       int, int, int);

typedef void (*GemmDma4Fn)(const half_t*, const uint32_t*, const half_t*, half_t*, float*, int, int, int, uint32_t);
typedef void (*GemmGroupedFn)(int, int, int, int, int, int, int, const GroupTable);

// A tile of a DMA kernel: its size, k per stage and workgroup.
struct DmaEntry {
  int bm, bn, bk, threads;
  GemmFn fn;
  GemmDma4Fn dma4;        // four k-groups, in place of fn
  GemmGroupedFn grouped;  // ... only
};
template <int TM, int TN, int NS>
constexpr DmaEntry dma4_entry() {
  using C = Dma4Cfg<TM, TN, NS>;
  return DmaEntry{C::BM, C::BN, C::BK, C::THREADS, nullptr, gemm_dma4_kernel<C>, gemm_dma4_grouped_kernel<C>};
}
const DmaEntry kDma[] = {
    dma4_entry<2, 4, 4>(), dma4_entry<3, 4, 4>(), dma4_entry<4, 4, 3>(),
    dma4_entry<5, 4, 3>(), dma4_entry<7, 4, 3>(), dma4_entry<8, 4, 3>(),
    DmaEntry{128, 128, DmaCfg::BK, DmaCfg::THREADS, gemm_dma2_kernel, nullptr, nullptr},
    DmaEntry{192, 256, WideCfg::BK, WideCfg::THREADS, gemm_wide_kernel, nullptr, nullptr},
};
constexpr int kNumDma = sizeof(kDma) / sizeof(kDma[0]);

}  // namespace

int gemm_num_configs() { return stream_num_configs() + kNumDma; }

// Whether a configuration runs this K: the DMA tiles take whole stages (the 192 x 256 tile, pairs of them).
static bool config_takes_k(int cfg, int K) {
  if (cfg < stream_num_configs()) return true;
  return K % kDma[cfg - stream_num_configs()].bk == 0 && (cfg != gemm_num_configs() - 1 || K % 128 == 0);
}

// Plan with an explicit configuration (streaming tiles first, then kDma) that takes K, and split count.
GemmPlan gemm_plan_with(int cfg, int splits, int K) {
  GemmPlan p = {};
  p.cfg = cfg;
  if (cfg < stream_num_configs()) {
    const StreamTile t = stream_tile_of(cfg);
    p.block_m = t.bm;
    p.block_n = t.bn;
    p.threads = 64 * t.ks;
    p.splits = splits;  // the kernel balances the 64-k pieces over them
    return p;
  }
  const DmaEntry& e = kDma[cfg - stream_num_configs()];
  p.block_m = e.bm;
  p.block_n = e.bn;
  p.threads = e.threads;
  const int nst = K / e.bk;
  p.kt_per_split = ceil_div(nst, splits);
  p.splits = ceil_div(nst, p.kt_per_split);  // no empty splits
  return p;
}

namespace {

// Cost of a configuration, in microseconds (see gemm_plan): workgroups resident per CU, and the
// coefficients of 1, w, w k, k, r k and the weight's size, where w = workgroups of the busiest CU, r =
// rounds of resident workgroups, k = thousands of K per split.  Weighted least squares (relative error, no
// negative terms, a timing weighing as the fourth power of its nearness to the size's best) over
// graph-replayed timings of every configuration and split count on 1571 (M, N, K) points: the TinyLlama,
// Qwen2.5 and hidden-4096 layer shapes, deep and narrow layers and random sizes, N = 64 .. 28672, K = 384 ..
// 65536, M = 5 .. 2300, weights rotated through more than the MALL, on MI355X; then small random changes kept
// where the time of the chosen configurations, or of the shared launches of 721 sets of siblings, fell.  The rms
// error is 6.6%; over those points the plan takes 1.004x the time of the best configuration measured, 2.7% of
// them more than 1.05x and the worst 1.18x.  Fitted without 339 of them, 1.005x on those.
struct CostTerms {
  int resident;
  double c[6];
};
const CostTerms kCost[] = {
    {2, {1.984, 0.4153, 0.2482, 0, 0.2089, 0.03732}},  // 8 x 16, 8 wavefronts
    {2, {1.845, 0.4258, 0.3692, 0, 0.2073, 0.03661}},  // 16 x 16, 8 wavefronts
    {1, {0.886, 1.644, 0.8801, 0.01794, 0, 0.04079}},  // 16 x 32, 8 wavefronts
    {1, {0.579, 2.181, 1.31, 0.2099, 0, 0.04975}},  // 16 x 64, 8 wavefronts
    {1, {1.117, 1.392, 0.6625, 0, 0, 0.05753}},  // 24 x 16, 8 wavefronts
    {1, {1.136, 1.264, 0.7326, 0, 0, 0.05531}},  // 32 x 16, 8 wavefronts
    {1, {0.8871, 1.904, 1.01, 0.06335, 0, 0.06971}},  // 32 x 32, 8 wavefronts
    {1, {1.019, 2.211, 1.189, 0.06349, 0, 0.06941}},  // 32 x 48, 8 wavefronts
    {1, {1.04, 1.797, 0.8525, 0, 0, 0.06783}},  // 48 x 16, 8 wavefronts
    {1, {1.259, 1.727, 1.253, 0, 0, 0.06864}},  // 48 x 32, 8 wavefronts
    {1, {1.29, 2.13, 1.649, 0.007682, 0, 0.06996}},  // 48 x 48, 8 wavefronts
    {3, {2.001, 0.3777, 0.6995, 0.1152, 0.6246, 0.06622}},  // 32 x 32, 4 wavefronts
    {2, {2.182, 0.8556, 1.111, 0.09628, 0.7392, 0.06249}},  // 48 x 48, 4 wavefronts
    {2, {1.973, 0.8494, 0.969, 0, 1.071, 0.05605}},  // 64 x 32, 4 wavefronts
    {1, {1.268, 2.544, 2.267, 0, 0, 0.05075}},  // 64 x 48, 4 wavefronts
    {1, {1.407, 3.238, 2.549, 0, 0, 0.05075}},  // 64 x 64, 4 wavefronts
    {4, {1.961, 0.2121, 0.2981, 0.01678, 0.3614, 0.0314}},  // 8 x 16, 4 wavefronts
    {3, {1.708, 0.1784, 0.2774, 0, 0.7866, 0.04328}},  // 16 x 16, 4 wavefronts
    {2, {2.592, 0.7188, 2.733, 0, 0.565, 0.05338}},  // 32 x 128, 8 wavefronts
    {1, {1.143, 2.937, 3.828, 0, 0, 0.04331}},  // 48 x 128, 8 wavefronts
    {2, {3.103, 1.157, 3.993, 0, 0.3402, 0.04573}},  // 64 x 128, 8 wavefronts
    {1, {0.8987, 4.095, 4.752, 0, 0, 0.04338}},  // 80 x 128, 8 wavefronts
    {1, {1.188, 3.945, 6.805, 0, 0, 0.02955}},  // 112 x 128, 8 wavefronts
    {1, {0.5004, 5.407, 6.61, 0, 0, 0.03066}},  // 128 x 128, 8 wavefronts
    {2, {3.71, 1.076, 4.24, 0, 4.835, 0.01889}},  // 128 x 128, 4 wavefronts
    {1, {2.347, 5.555, 19.64, 0, 0, 0.0132}},  // 192 x 256, 8 wavefronts
};
// Split-K costs one more launch plus the fp32 partials (same fit), and is taken only when the
// model predicts it at least 2% faster.  One margin for all sizes: asking for a workspace at fixed rows of deep
// layers made 2048 x 5632 at M = 64 / 900 take 9.6 / 34.0 us split where 7.6 / 30.2 unsplit are possible, and
// 2048 x 12416 at M = 1773 107 where 93 are.
constexpr double kSplitUs = 2.268, kSplitUsPerMElem = 1.372, kSplitMargin = 1.02;
constexpr double kSiblingUs = 0.5;   // see gemm_plan_within
constexpr int kMaxSplits = 8;        // the largest split count the fit was measured on
constexpr int kMinSplitK = 512;      // k per split

}  // namespace

// Modelled time of `tiles` workgroups of a configuration per split.  Each XCD runs its share of the
// workgroups, spread over its CUs.
static double plan_cost(int cfg, long tiles, int splits, int M, double n, int K, int cus) {
  const CostTerms& t = kCost[cfg];
  const int cus_per_xcd = std::max(1, cus / kXcds);
  const long per_cu = (((tiles * splits + kXcds - 1) / kXcds) + cus_per_xcd - 1) / cus_per_xcd;
  const long rounds = (per_cu + t.resident - 1) / t.resident;
  const double k = K * 1e-3 / splits;
  const double cost =
      t.c[0] + (t.c[1] + t.c[2] * k) * per_cu + (t.c[3] + t.c[4] * rounds) * k + t.c[5] * n * K * 1e-6;
  return splits == 1 ? cost : (cost + kSplitUs + kSplitUsPerMElem * 1e-6 * splits * (double)M * n) * kSplitMargin;
}

// At M <= 16 the K split over wavefronts depends on M and K alone (see gemm_plan).  Four wavefronts
// leave room for more workgroups per CU, which wide layers want; eight shorten a long K.  Best tile
// with 4 / 8 (us): 17920 x 1536 at M = 6 / 16: 7.5 / 8.5 and 8.4 / 10.6; 11264 x 2048: 5.5 / 6.1 and
// 6.1 / 6.6; 2560 x 2048: 3.5 / 3.4 and 4.5 / 3.7; 28672 x 4096: 15.9 / 18.0 and 22.9 / 21.5; 4096 x
// 4096: 5.1 / 4.6 and 6.5 / 5.2; 4096 x 14336: 11.2 / 9.4 and 17.0 / 12.3.
static int small_m_waves(int M, int K) { return K < 2048 || (M <= 8 && K <= 4096) ? 4 : 8; }

// Kernel choice: the configuration and split-K factor with the smallest modelled time.
//   * M <= 16: streaming tiles of small_m_waves(M, K) wavefronts without split-K only, so the K split
//     (and with it every bit of a column) does not depend on N and concatenated q|k|v or gate|up rows
//     give the separate layers' results.
//   * Narrow layers (k and v) get kSiblingUs off where they sum in the order of the K x K layer's plan (q),
//     so that they can share its launch: that saves a call with its siblings 2-4 us, and costs a call by itself
//     at most the half (q|k|v of 1024 + 2 x 128 columns, K = 1024, M = 27: 3.5 us together, 6.4 where q and k, v
//     take different wavefront counts).  Over 779 measured sets q|k|v takes 0.947x the time without it, over 273
//     narrow layers a call by itself 1.003x.
//   * Partials take max_partials bytes at most; splits of 1 take none, so there is a plan for any limit.
GemmPlan gemm_plan_within(int M, int N, int K, int cu_count, size_t max_partials) {
  static_assert(sizeof(kCost) / sizeof(kCost[0]) == kNumStreamConfigs + kNumDma, "one cost entry per configuration");
  const int cus = cu_count > 0 ? cu_count : 256;
  const int num_stream = stream_num_configs();
  const bool narrow = M > 16 && N <= 1024 && 4 * N <= K;
  const GemmPlan square = narrow ? gemm_plan(M, K, K, cu_count) : GemmPlan{};
  int best_cfg = -1, best_splits = 1;
  double best = 1e300;
  for (int cfg = 0; cfg < gemm_num_configs(); ++cfg) {
    int bm, bn, threads;
    if (cfg < num_stream) {
      const StreamTile t = stream_tile_of(cfg);
      bm = t.bm, bn = t.bn, threads = 64 * t.ks;
      if (M <= 16 && t.ks != small_m_waves(M, K)) continue;
    } else {
      const DmaEntry& e = kDma[cfg - num_stream];
      bm = e.bm, bn = e.bn, threads = e.threads;
      if (M <= 16 || !config_takes_k(cfg, K)) continue;
    }
    const long tiles = (long)ceil_div(M, bm) * ceil_div(N, bn);
    if ((tiles + kXcds) * threads > 0x7FFFFFFFL) continue;
    // The 192 x 256 tile writes no partials; more splits than two rounds of workgroups never pay.
    const bool can_split = M > 16 && tiles < 2 * cus && cfg != gemm_num_configs() - 1;
    const int max_splits = can_split ? std::min(kMaxSplits, std::max(1, K / kMinSplitK)) : 1;
    for (int s = 1; s <= max_splits; ++s) {
      if (s > 1 && (size_t)s * M * N * sizeof(float) > max_partials) break;
      double cost = plan_cost(cfg, tiles, s, M, N, K, cus);
      if (narrow && s == 1 && gemm_same_sums(square, gemm_plan_with(cfg, 1, K))) cost -= kSiblingUs;
      if (cost < best) {
        best = cost;
        best_cfg = cfg;
        best_splits = s;
      }
    }
  }
  if (best_cfg < 0) best_cfg = 0;  // past every grid limit, and past this one's; the caller's check refuses it
  return gemm_plan_with(best_cfg, best_splits, K);
}

// The plan is a function of its arguments; each thread keeps the last ones it asked for (the workspace
// query and the launch of a call, and a model's few shapes), which is 0.6 us of an eager call's host time.
GemmPlan gemm_plan(int M, int N, int K, int cu_count) {
  struct Entry {
    int M, N, K, cus;
    GemmPlan plan;
  };
  constexpr uint32_t kEntries = 64;
  static thread_local Entry entries[kEntries];  // M = 0: empty
  Entry& e = entries[((uint32_t)M * 0x9E3779B1u ^ (uint32_t)N * 0x85EBCA6Bu ^ (uint32_t)K * 0xC2B2AE35u) >> 26];
  if (e.M != M || e.N != N || e.K != K || e.cus != cu_count) 
    e = Entry{M, N, K, cu_count, gemm_plan_within(M, N, K, cu_count, SIZE_MAX)};
  return e.plan;
}

size_t gemm_workspace_bytes(const GemmPlan& p, int M, int N) {
  return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

bool gemm_same_sums(const GemmPlan& a, const GemmPlan& b) {
  if (a.splits != 1 || b.splits != 1) return false;
  const int ns = stream_num_configs();
  if (a.cfg < ns || b.cfg < ns)
    return a.cfg < ns && b.cfg < ns && stream_tile_of(a.cfg).ks == stream_tile_of(b.cfg).ks;
  return kDma[a.cfg - ns].grouped && kDma[b.cfg - ns].grouped;
}

// Streaming tiles sum an element in an order that depends on K and their wavefronts only, the DMA tiles
// of four k-groups in one that depends on K only, so any tile of the same kind gives a sibling the bits
// of its own plan.  All plans have to be of one kind (gemm_same_sums); the tile is the one with the
// smallest modelled time for all columns together, taken where that is less than the sum of the
// separate launches.  Separate / grouped, us: q|k|v of 2048 + 2 x 256 columns, K = 2048, at M = 16 / 64 /
// 200: 10.2 / 4.1, 10.8 / 5.6, 13.0 / 9.5; gate|up of 2 x 5632: 9.5 / 7.0, 12.6 / 11.8, 24.8 / 18.4; 2 x 14336, K =
// 4096, at M = 64 / 128 / 517: 33.7 / 32.0, 52.1 / 40.5, 167 / 165.  The worst of 279 sets: 2 x 15360, K = 3968, at M =
// 27 31.7 / 32.7.
int gemm_group_config(const GemmPlan* plans, const int* N, int count, int M, int K, int cu_count) {
  const int cus = cu_count > 0 ? cu_count : 256;
  double best = 0.0, columns = 0.0;
  for (int i = 0; i < count; ++i) {
    if (!gemm_same_sums(plans[0], plans[i])) return -1;
    best += plan_cost(plans[i].cfg, (long)ceil_div(M, plans[i].block_m) * ceil_div(N[i], plans[i].block_n), 1, M, N[i],
                      K, cus);
    columns += N[i];
  }
  int best_cfg = -1;
  for (int cfg = 0; cfg < gemm_num_configs(); ++cfg) {
    if (!config_takes_k(cfg, K)) continue;
    const GemmPlan p = gemm_plan_with(cfg, 1, K);
    if (!gemm_same_sums(plans[0], p)) continue;
    long tiles = 0;
    for (int i = 0; i < count; ++i) tiles += ceil_div(N[i], p.block_n);
    tiles *= ceil_div(M, p.block_m);
    if ((tiles + kXcds) * p.threads > 0x7FFFFFFFL) continue;
    const double cost = plan_cost(cfg, tiles, 1, M, columns, K, cus);
    if (cost < best) {
      best = cost;
      best_cfg = cfg;
    }
  }
  return best_cfg;
}

hipError_t gemm_grouped_launch(int cfg, const GemvProblem* problems, int count, int M, int K, int group_size,
                               hipStream_t stream) {
  if (cfg < stream_num_configs()) return stream_grouped_launch(cfg, problems, count, M, K, group_size, stream);
  const DmaEntry& e = kDma[cfg - stream_num_configs()];
  GroupTable table = {};
  const int tiles_m = ceil_div(M, e.bm), tiles_n = group_table(problems, count, e.bn, table);
  const int grid = ceil_div(tiles_m * tiles_n, kXcds) * kXcds;
  hipLaunchKernelGGL(e.grouped, dim3(grid), dim3(e.threads), 0, stream, count, M, K, group_size == 128 ? 7 : 6,
                     tiles_m, tiles_n, std::max(1, tiles_m / kXcds), table);
  return hipGetLastError();
}

hipError_t gemm_launch(const GemmPlan& p, const void* x, const void* packed, const void* scales, void* y,
                       void* ws, int M, int N, int K, int group_size, hipStream_t stream) {
  float* part = p.splits > 1 ? static_cast<float*>(ws) : nullptr;
  hipError_t err;
  if (p.cfg < stream_num_configs()) {
    err = stream_launch(p.cfg, p.splits, x, packed, scales, y, part, M, N, K, group_size, stream);
  } else {
    const DmaEntry& e = kDma[p.cfg - stream_num_configs()];
    const int log2_group = group_size == 128 ? 7 : 6;
    const int tiles_m = ceil_div(M, e.bm);
    const int tiles_n = ceil_div(N, e.bn);
    const int grid_x = ceil_div(tiles_m * tiles_n * p.splits, kXcds) * kXcds;
    const half_t* xh = static_cast<const half_t*>(x);
    const uint32_t* w = static_cast<const uint32_t*>(packed);
    const half_t* sc = static_cast<const half_t*>(scales);
    half_t* yh = static_cast<half_t*>(y);
    if (e.dma4) {
      hipLaunchKernelGGL(e.dma4, dim3(grid_x), dim3(e.threads), 0, stream, xh, w, sc, yh, part, M, N, K,
                         (uint32_t)p.kt_per_split << 8 | p.splits << 4 | log2_group);
    } else {
      // Bands of M-tiles: one band per XCD when the M-tiles divide evenly, else single rows.
      hipLaunchKernelGGL(e.fn, dim3(grid_x), dim3(e.threads), 0, stream, xh, w, sc, yh, part, M, N, K, log2_group,
                         p.kt_per_split, p.splits, tiles_m, tiles_n, std::max(1, tiles_m / kXcds));
    }
    err = hipGetLastError();
  }
  if (err != hipSuccess || p.splits == 1) return err;
  const size_t mn4 = (size_t)M * N / 4;  // N % 64 == 0
  size_t blocks = (mn4 + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(splitk_reduce, dim3((unsigned)blocks), dim3(256), 0, stream, static_cast<const float4_t*>(ws),
                     static_cast<u32x2*>(y), mn4, p.splits);
  return hipGetLastError();
}

}  // namespace kf
