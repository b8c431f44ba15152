// Streaming INT4 GEMM for small and medium M on gfx950: every wavefront is its own pipeline.
//
// y[M, N] = x[M, K] @ W_hat^T with W_hat = fp16_rne(q * s) (the operand the reference's tensor-core
// kernel uses, dequant_gemm_tc_kernel.cuh:100-112), fp32 accumulation, fp16 RNE output.
//
// What bounds it.  At these M the matrix cores need under 2 us; the time goes into moving x and the
// weights from L2 / HBM into the CUs.  A CU's vector-memory path takes one 64-byte request per
// clock only when the lanes of a request are neighbours in memory: on MI355X a wavefront load of
// 64 x 16 bytes runs at 110-140 B/ns per CU when each run of 8 lanes covers one 128-byte line, at
// 80-95 with 4 lanes (64 B), 42-55 with 2 and 18-40 when neighbouring lanes read different rows -
// which is what MFMA fragments (lane l = row l % 16) do when they are loaded from memory directly.
// So nothing here is loaded in fragment order: x and the packed weights go to LDS with LDS-DMA in
// 128-byte row pieces, and the fragments are read from LDS.
//
//   * A workgroup owns an (8 XG) x (16 TN) tile of y; its KS wavefronts split the K range, each
//     taking a contiguous run of 64-k "pieces" of the whole tile.  A wavefront's x and weight
//     buffers are its own part of LDS, so the main loop has no barrier: it waits for its own
//     copies with counted waits.  The KS partial tiles are summed in fixed wavefront order through
//     LDS at the end (deterministic), or written as fp32 partials when K is also split over
//     workgroups (splits > 1, summed by splitk_reduce in fixed order).
//   * x: one LDS-DMA instruction copies 8 rows x 128 bytes (one piece).  XG instructions per
//     piece; PP pieces per iteration.  One buffer: a wavefront reads its fragments into registers
//     and starts the next copy into the same buffer before its MFMAs, so the copy runs under them
//     (two or four buffers in LDS measured no faster: the other wavefronts of the CU hide the
//     rest, and the LDS holds more workgroups instead).
//   * Weights: one instruction copies 8 rows x 128 bytes, a "step" of WP = 4 pieces, into one of WS
//     slots.  Copies complete in order and an iteration waits for its x, so only a step issued right
//     after that x stays in flight over an iteration; the others have landed one iteration after their
//     issue.  Scales: 2 bytes per column and 64-k piece, copied with the step into 4-byte slots.
//   * MFMA operands: lane l serves row / column l % 16 and k-group g = l / 16.  In sub-step t (0, 1)
//     of a piece it supplies k = 16 g + 8 t .. + 7 for both operands: x chunk 2 g + t of its row,
//     packed word 2 g + t of its column.  16-byte chunks are XOR-swizzled within their row (by
//     the row's position in the 256-byte bank window), which permutes lanes inside one line of the
//     copy and spreads sixteen consecutive lanes of a fragment read over all banks (counted all the same:
//     SQ_LDS_BANK_CONFLICT is 34-47% of SQ_LDS_IDX_ACTIVE).
//   * The MFMAs take the weights as their first operand, so each 16 x 16 block comes out
//     transposed: lane l, element r holds row l % 16, column 4 (l / 16) + r (8-byte stores of y).
//   * The loop is rolled on purpose.  The kernels live for 3-20 us; a version with the steps
//     unrolled and the LDS reads of the next piece issued before the MFMAs of this one ran 5-20%
//     slower everywhere, from instruction fetch and from scheduling around its extra waits.
//
// Measured on MI355X (graph replays, weights rotated through HBM), against the kernels this one
// replaced (a skinny kernel loading fragments from memory, register-staged 16 x 64 .. 64 x 128
// tiles): N x K = 5632 x 2048 at M = 16 / 64 / 128: 6.1 / 8.9 / 12.3 -> 4.8 / 6.4 / 8.3 us;
// 2048 x 2048: 4.6 / 7.2 / 7.7 -> 3.6 / 4.2 / 5.1; 256 x 2048 at M = 64: 6.8 -> 3.0; 2048 x 5632 at
// M = 16 / 64: 8.8 / 12.1 -> 6.1 / 7.6; 28672 x 4096 at M = 8: 33.5 -> 17.
#include <algorithm>

#include "kf_device.h"
#include "kf_launch.h"

namespace kf {
namespace {

constexpr int kXcds = 8;

// One tile configuration (see the header comment).  A wavefront's LDS: PP pieces of x, then WS
// steps of [packed words, scales]; the partial tile reuses it.
template <int XG_, int TN_, int KS_, int PP_, int WS_>
struct StreamCfg {
  static constexpr int XG = XG_, TN = TN_, KS = KS_, PP = PP_, WS = WS_;
  static constexpr int WP = 4;                                  // pieces per weight step: a 128-byte line of a packed row
  static constexpr int TM = (XG + 1) / 2;                       // 16-row blocks
  static constexpr int IPS = WP / PP;                           // iterations per weight step
  static constexpr int X_PIECE = XG * 1024, X_BYTES = PP * X_PIECE;
  static constexpr int W_ROW = 32 * WP, W_CH = 2 * WP;          // bytes and 16-byte chunks of a packed row per step
  static constexpr int W_RPI = 32 / WP;                         // rows per copy instruction
  static constexpr int WIN = 2 * TN;                            // copy instructions of a step's words
  static constexpr int SIN = TN;                                // ... and of its scales
  static constexpr int S_OFF = WIN * 1024, W_SLOT = S_OFF + SIN * 256;
  static constexpr int RING = X_BYTES + WS * W_SLOT;
  static constexpr int PART = TM * TN * 1024;                   // fp32 partial tile
  static constexpr int WAVE = RING > PART ? RING : PART;
  static constexpr int LDS = KS * WAVE;
  static_assert(WP % PP == 0 && WS >= 2, "a step holds whole iterations, and the next steps are in flight");
  static_assert(LDS <= 160 * 1024, "LDS");
};

__device__ __forceinline__ void dma_16B(uint32_t lds, const void* src) {
  asm volatile("global_load_lds_dwordx4 %1, off" ::"{m0}"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ void dma_16B_stream(uint32_t lds, const void* src) {
  asm volatile("global_load_lds_dwordx4 %1, off nt" ::"{m0}"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ void dma_u16(uint32_t lds, const void* src) {
  asm volatile("global_load_lds_ushort %1, off" ::"{m0}"(lds), "v"(src) : "memory");
}

// Rows m0 .. m0 + 8 XG - 1, columns n0 .. n0 + 16 TN - 1 over the 64-k pieces [k_begin, k_end).
// part: fp32 [M, N] partials to write instead of y, or nullptr.  once: no other workgroup reads these
// weights (see issue_w).
template <class C>
__device__ __forceinline__ void stream_tile(const half_t* x, const uint32_t* packed, const half_t* scales, half_t* y,
                                            float* part, int M, int N, int K, int log2_group, int m0, int n0,
                                            int k_begin, int k_end, bool once) {
  constexpr int XG = C::XG, TN = C::TN, KS = C::KS, PP = C::PP, WS = C::WS, WP = C::WP, TM = C::TM;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS];  // static: no attribute call above 64 KiB
  const int lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;

  // This wavefront's pieces [p0, p0 + np).
  const uint32_t pieces = k_end - k_begin;
  const int p0 = k_begin + (int)(wave * pieces / KS);
  const int np = k_begin + (int)((wave + 1) * pieces / KS) - p0;
  const int nit = (np + PP - 1) / PP, nq = (np + WP - 1) / WP;

  unsigned char* const my = smem + wave * C::WAVE;
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)my);
  const uint32_t wbase = base + C::X_BYTES;

  // Copy sources at the wavefront's first piece.  Rows past M or N re-read the last one (their
  // results are not stored); chunk positions carry the swizzle.
  auto x_swz = [](int r) { return (r >> 1) & 7; };
  auto w_swz = [](int r) { return ((r & 15) / (8 / WP)) & (C::W_CH - 1); };
  const half_t* xs[XG];
#pragma unroll
  for (int i = 0; i < XG; ++i) {
    const int r = 8 * i + (lane >> 3);
    xs[i] = x + (size_t)min(m0 + r, M - 1) * K + (size_t)64 * p0 + 8 * ((lane & 7) ^ x_swz(r));
  }
  const uint32_t* ws[C::WIN];
#pragma unroll
  for (int i = 0; i < C::WIN; ++i)
    ws[i] = packed + (size_t)min(n0 + C::W_RPI * i + lane / C::W_CH, N - 1) * (K >> 3);
  const half_t* ss[C::SIN];
#pragma unroll
  for (int i = 0; i < C::SIN; ++i)
    ss[i] = scales + (size_t)min(n0 + (64 / WP) * i + lane / WP, N - 1) * (K >> log2_group);

  auto issue_x = [&](int it) {  // XG * PP copies; pieces past the range re-read its last one
#pragma unroll
    for (int pp = 0; pp < PP; ++pp) {
      const size_t p = PP == 1 ? it : min(PP * it + pp, np - 1);
#pragma unroll
      for (int i = 0; i < XG; ++i) dma_16B(base + pp * C::X_PIECE + 1024 * i, xs[i] + 64 * p);
    }
  };
  // WIN + SIN copies; chunks past K re-read its last one.  The non-temporal hint keeps weights that
  // are read once from displacing x in the caches (28672 x 4096 at M = 8: 19.7 -> 18.9 us), but costs
  // a second fetch where another row tile reads a line again (11264 x 2048, M = 200 in four tiles:
  // 21.4 with plain copies, 23.9 with the hint).
  auto issue_w = [&](int q, uint32_t slot) {
    const int first = p0 + WP * q;
#pragma unroll
    for (int i = 0; i < C::WIN; ++i) {
      const int c = min(2 * first + ((lane % C::W_CH) ^ w_swz(C::W_RPI * i + lane / C::W_CH)), (K >> 5) - 1);
      if (once)  // uniform
        dma_16B_stream(wbase + slot + 1024 * i, ws[i] + 4 * (size_t)c);
      else
        dma_16B(wbase + slot + 1024 * i, ws[i] + 4 * (size_t)c);
    }
    const int group = min(first + lane % WP, (K >> 6) - 1) >> (log2_group - 6);
#pragma unroll
    for (int i = 0; i < C::SIN; ++i) dma_u16(wbase + slot + C::S_OFF + 256 * i, ss[i] + group);
  };

  float4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  const UnpackConsts uc = unpack_consts();
  const int xo0 = l16 * 128 + 16 * ((2 * g) ^ x_swz(l16)), xo1 = l16 * 128 + 16 * ((2 * g + 1) ^ x_swz(l16));

  // Order of the copies: weight steps 0 .. WS - 2, x of iteration 0, weight step WS - 1; then per
  // iteration, once its fragments are in registers, x of the next one and, after a step's last
  // iteration, the weight step that takes its slot.  An iteration needs its x and everything
  // older; only a weight step issued right after that x may still be in flight (w_last).
#pragma unroll
  for (int q = 0; q < WS - 1; ++q)
    if (q < nq) issue_w(q, q * C::W_SLOT);
  if (nit > 0) issue_x(0);
  bool w_last = WS - 1 < nq;
  if (w_last) issue_w(WS - 1, (WS - 1) * C::W_SLOT);
  uint32_t wslot = 0;
  int phase = 0, q = 0;
#pragma unroll 1
  for (int it = 0; it < nit; ++it) {
    if (w_last)
      wait_vmcnt<C::WIN + C::SIN>();
    else
      wait_vmcnt<0>();
    half8_t a[PP][TM][2];
    u32x2 w[PP][TN];
    half_t sc[PP][TN];
    const unsigned char* wp = my + C::X_BYTES + wslot;
#pragma unroll
    for (int pp = 0; pp < PP; ++pp) {
      const int ps = (PP == WP ? 0 : PP * phase) + pp;  // piece within the step
      const int wo = l16 * C::W_ROW + 16 * ((2 * ps + (g >> 1)) ^ w_swz(l16)) + 8 * (g & 1);
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        w[pp][j] = *reinterpret_cast<const u32x2*>(wp + 16 * C::W_ROW * j + wo);
        sc[pp][j] = *reinterpret_cast<const half_t*>(wp + C::S_OFF + 4 * (WP * (16 * j + l16) + ps));
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        // With an odd XG the last block has 8 rows; its other lanes read them again.
        const int wrap = (XG & 1) && i == TM - 1 ? 1023 : -1;
        const unsigned char* xp = my + pp * C::X_PIECE + 2048 * i;
        a[pp][i][0] = *reinterpret_cast<const half8_t*>(xp + (xo0 & wrap));
        a[pp][i][1] = *reinterpret_cast<const half8_t*>(xp + (xo1 & wrap));
      }
    }
    // The fragments are in registers before the buffers they came from are written again.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (it + 1 < nit) issue_x(it + 1);
    w_last = false;
    if (++phase == C::IPS) {
      phase = 0;
      w_last = q + WS < nq;
      if (w_last) issue_w(q + WS, wslot);
      ++q;
      wslot = wslot + C::W_SLOT == WS * C::W_SLOT ? 0 : wslot + C::W_SLOT;
    }
#pragma unroll
    for (int pp = 0; pp < PP; ++pp) {
      if (PP > 1 && pp > 0 && PP * it + pp >= np) break;  // uniform
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const half8_t b = dequant8(w[pp][j][t], half2_t{sc[pp][j], sc[pp][j]}, uc);
#pragma unroll
          for (int i = 0; i < TM; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a[pp][i][t], acc[i][j], 0, 0, 0);
        }
    }
  }

  // Every copy this wavefront issued has landed (the last iteration waited for all of them), so
  // its buffers take its partial tile without a barrier.
  float* mine = reinterpret_cast<float*>(my) + 4 * lane;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) *reinterpret_cast<float4_t*>(mine + (i * TN + j) * 256) = acc[i][j];
  __syncthreads();
  const int rows = min(M, m0 + 8 * XG);
  for (int e = threadIdx.x; e < TM * TN * 64; e += 64 * KS) {
    float4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int z = 0; z < KS; ++z) v += *reinterpret_cast<const float4_t*>(smem + z * C::WAVE + 16 * e);
    const int b = e >> 6, l = e & 63;
    const int i = b / TN, j = b - i * TN;
    const int row = m0 + 16 * i + (l & 15), c = n0 + 16 * j + 4 * (l >> 4);
    if (row < rows && c < N) {  // N % 64 == 0: the four columns are all inside or all past it
      if (part) {
        *reinterpret_cast<float4_t*>(part + (size_t)row * N + c) = v;
      } else {
        const half2_t lo = {(half_t)v[0], (half_t)v[1]}, hi = {(half_t)v[2], (half_t)v[3]};
        *reinterpret_cast<u32x2*>(y + (size_t)row * N + c) = u32x2{bit_cast<uint32_t>(lo), bit_cast<uint32_t>(hi)};
      }
    }
  }
}

// Workgroups are dealt to the 8 XCDs in contiguous runs of jobs (the hardware deals workgroup b to
// XCD b % 8), split-major.  -1: no job.
__device__ __forceinline__ int stream_job(uint32_t jobs) {
  const uint32_t per_xcd = (jobs + kXcds - 1) / kXcds;
  const uint32_t j = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
  return blockIdx.x / kXcds < per_xcd && j < jobs ? (int)j : -1;
}
// Row and column tile of tile t, row tiles or column tiles as neighbours.
__device__ __forceinline__ void stream_tile_at(uint32_t t, uint32_t tiles_m, uint32_t tiles_n, bool rows_first, int& mt,
                                               int& nt) {
  if (tiles_m == 1) {
    mt = 0;
    nt = t;
    return;
  }
  const uint32_t d = rows_first ? tiles_m : tiles_n, q = t / d, r = t - q * d;
  mt = rows_first ? r : q;
  nt = rows_first ? q : r;
}

// The kernels of small layers live for 3-5 us, so what a workgroup does before its first copy counts:
// the arguments fit the 14 dwords that arrive in registers (one more costs a scalar load from memory
// first), the tile counts come from M and N, the divisions are unsigned and left out where one tile row or
// one split makes them trivial (signed 64-bit ones were most of the time to the first copy).  N x K = 256 x
// 2048 at M = 9 / 64: 3.8 / 3.5 -> 3.15 / 3.0 us; 2048 x 2048 at M = 6: 4.0 -> 3.4; 17920 x 1536 at M = 5: 8.2 ->
// 7.3; 4096 x 14336 at M = 32: 18.1 -> 17.4.
template <class C>
__global__ __launch_bounds__(64 * C::KS) void stream_kernel(const half_t* __restrict__ x,
                                                            const uint32_t* __restrict__ packed,
                                                            const half_t* __restrict__ scales, half_t* __restrict__ y,
                                                            float* __restrict__ part, int M, int N, int K,
                                                            int splits_group) {
  constexpr uint32_t BM = 8 * C::XG, BN = 16 * C::TN;
  const uint32_t splits = (uint32_t)splits_group >> 8;
  const int log2_group = splits_group & 255;
  const uint32_t tiles_m = ((uint32_t)M + BM - 1) / BM, tiles_n = ((uint32_t)N + BN - 1) / BN;
  const uint32_t tiles = tiles_m * tiles_n;
  const int job = stream_job(tiles * splits);
  if (job < 0) return;
  const uint32_t pieces = (uint32_t)K >> 6;
  uint32_t split = 0, k0 = 0, k1 = pieces;
  if (splits > 1) {  // splits <= 8, K < 2^31: the products fit
    split = (uint32_t)job / tiles;
    k0 = split * pieces / splits;
    k1 = (split + 1) * pieces / splits;
  }
  // The larger operand is read by one XCD only as far as its L2 can serve it: with more bytes of
  // weights than of x, the row tiles of a column tile are neighbours, else the column tiles of a row
  // tile (256 x 2048 at M = 2048: 12.4 -> 6.9 us).
  int mt, nt;
  stream_tile_at(job - split * tiles, tiles_m, tiles_n, M <= N / 4, mt, nt);
  stream_tile<C>(x, packed, scales, y, part ? part + (size_t)split * M * N : nullptr, M, N, K, log2_group, mt * (int)BM,
                 nt * (int)BN, k0, k1, tiles_m == 1);
}

// Several problems of one M, K and group size in one launch: column tiles are numbered through the
// problems, problem p owning tiles slot[p].tile0 up to the next problem's.  Each output has the bits of
// its own stream_kernel launch at the same KS: the K split does not depend on N or on the tile.  A
// launch of its own costs a small layer about 2 us of start and tail, more than its work.
template <class C>
__global__ __launch_bounds__(64 * C::KS) void stream_grouped_kernel(int count, int M, int K, int log2_group,
                                                                    int tiles_m, int tiles_n, int rows_first,
                                                                    const GroupTable table) {
  const int job = stream_job(tiles_m * tiles_n);
  if (job < 0) return;
  int mt, nt;
  stream_tile_at(job, tiles_m, tiles_n, rows_first, mt, nt);
  const GroupEntry e = group_entry(table, count, nt);
  stream_tile<C>(e.x, e.packed, e.scales, e.y, nullptr, M, e.N, K, log2_group, mt * 8 * C::XG,
                 (nt - e.tile0) * 16 * C::TN, 0, K >> 6, tiles_m == 1);
}

typedef void (*StreamFn)(const half_t*, const uint32_t*, const half_t*, half_t*, float*, int, int, int, int);
typedef void (*StreamGroupedFn)(int, int, int, int, int, int, int, const GroupTable);

struct StreamEntry {
  int xg, tn, ks, lds;
  StreamFn fn;
  StreamGroupedFn grouped;
};
template <int XG, int TN, int KS, int PP, int WS>
constexpr StreamEntry stream_entry() {
  using C = StreamCfg<XG, TN, KS, PP, WS>;
  return StreamEntry{XG, TN, KS, C::LDS, stream_kernel<C>, stream_grouped_kernel<C>};
}

const StreamEntry kStream[] = {
    stream_entry<1, 1, 8, 4, 2>(), stream_entry<2, 1, 8, 2, 2>(), stream_entry<2, 2, 8, 2, 2>(),
    stream_entry<2, 4, 8, 1, 2>(), stream_entry<3, 1, 8, 2, 4>(), stream_entry<4, 1, 8, 1, 4>(),
    stream_entry<4, 2, 8, 1, 2>(), stream_entry<4, 3, 8, 1, 2>(), stream_entry<6, 1, 8, 1, 4>(),
    stream_entry<6, 2, 8, 1, 3>(), stream_entry<6, 3, 8, 1, 2>(), stream_entry<4, 2, 4, 1, 2>(),
    stream_entry<6, 3, 4, 1, 2>(), stream_entry<8, 2, 4, 1, 2>(), stream_entry<8, 3, 4, 1, 2>(),
    stream_entry<8, 4, 4, 1, 2>(), stream_entry<1, 1, 4, 4, 2>(), stream_entry<2, 1, 4, 1, 4>(),
};
static_assert(sizeof(kStream) / sizeof(kStream[0]) == kNumStreamConfigs, "configuration count");

}  // namespace

StreamTile stream_tile_of(int cfg) {
  const StreamEntry& e = kStream[cfg];
  return StreamTile{8 * e.xg, 16 * e.tn, e.ks, e.lds};
}

hipError_t stream_launch(int cfg, int splits, const void* x, const void* packed, const void* scales, void* y,
                         float* part, int M, int N, int K, int group_size, hipStream_t stream) {
  const StreamEntry& e = kStream[cfg];
  const int tiles_m = ceil_div(M, 8 * e.xg), tiles_n = ceil_div(N, 16 * e.tn);
  const int grid = ceil_div(tiles_m * tiles_n * splits, kXcds) * kXcds;
  hipLaunchKernelGGL(e.fn, dim3(grid), dim3(64 * e.ks), 0, stream, static_cast<const half_t*>(x),
                     static_cast<const uint32_t*>(packed), static_cast<const half_t*>(scales),
                     static_cast<half_t*>(y), splits > 1 ? part : nullptr, M, N, K,
                     splits << 8 | (group_size == 128 ? 7 : 6));
  return hipGetLastError();
}

int group_table(const GemvProblem* problems, int count, int bn, GroupTable& table) {
  int tiles_n = 0;
  for (int i = 0; i < count; ++i) {
    const GemvProblem& q = problems[i];
    table.slot[i] = GroupSlot{q.x, q.packed, q.scales, q.y, q.N, tiles_n};
    tiles_n += ceil_div(q.N, bn);
  }
  return tiles_n;
}

hipError_t stream_grouped_launch(int cfg, const GemvProblem* problems, int count, int M, int K, int group_size,
                                 hipStream_t stream) {
  const StreamEntry& e = kStream[cfg];
  GroupTable table = {};
  const int tiles_m = ceil_div(M, 8 * e.xg), tiles_n = group_table(problems, count, 16 * e.tn, table);
  const int grid = ceil_div(tiles_m * tiles_n, kXcds) * kXcds;
  hipLaunchKernelGGL(e.grouped, dim3(grid), dim3(64 * e.ks), 0, stream, count, M, K, group_size == 128 ? 7 : 6,
                     tiles_m, tiles_n, 4L * M <= 16L * e.tn * tiles_n ? 1 : 0, table);
  return hipGetLastError();
}

}  // namespace kf
