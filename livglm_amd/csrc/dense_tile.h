// Dense GEMM tiles of the resident linears and the shared expert (see
// dense_gemm.hip): y = x W^T or the SwiGLU of two such products, W row-major in
// MXFP8, MXFP4 or bf16.
#pragma once

#include "lds_stage.h"
#include "mfma_tile.h"

namespace glm {

constexpr int kDenseWF = 4;  // waves along the weight rows
constexpr int kDenseXcds = 8;

struct DenseArgs {
  const uint16_t *x;  // bf16 [T][K]
  const uint8_t *w[2], *s[2];
  uint16_t *out;  // bf16 [T][N]
  int T, N, K;
  int row_tiles, tok_tiles;
  int rows_outer;  // consecutive items walk the tokens of one row tile, else the reverse
  float limit;     // bf16-rounded SwiGLU limit (gate/up)
};

// A format's staged weights: kRow bytes of a row per K chunk, and one lane's
// share of a 16-row block.
template <int FMT>
struct DenseRaw;
template <>
struct DenseRaw<FMT_MXFP8> {
  static constexpr int kChunk = 128, kRow = 128;
  glm_u32x4 c[2];
  __device__ static int swz(int row) { return row & 7; }
  __device__ __forceinline__ void read(const uint8_t *row, int r, int q) {
    c[0] = *reinterpret_cast<const glm_u32x4 *>(row + 16 * ((2 * q) ^ swz(r)));
    c[1] = *reinterpret_cast<const glm_u32x4 *>(row + 16 * ((2 * q + 1) ^ swz(r)));
  }
  __device__ __forceinline__ glm_bf16x8 frag(int i, float sc) const {
    return mxfp8_words_to_bf16x8(c[i >> 1][2 * (i & 1)], c[i >> 1][2 * (i & 1) + 1], sc);
  }
};
template <>
struct DenseRaw<FMT_MXFP4> {
  static constexpr int kChunk = 128, kRow = 64;
  glm_u32x4 c;
  __device__ static int swz(int row) { return (row >> 2) & 3; }
  __device__ __forceinline__ void read(const uint8_t *row, int r, int q) {
    c = *reinterpret_cast<const glm_u32x4 *>(row + 16 * (q ^ swz(r)));
  }
  __device__ __forceinline__ glm_bf16x8 frag(int i, float sc) const {
    return mxfp4_word_to_bf16x8(c[i], sc);
  }
};
template <>
struct DenseRaw<FMT_BF16> {
  static constexpr int kChunk = 64, kRow = 128;
  glm_u32x4 c[2];
  __device__ static int swz(int row) { return row & 7; }
  __device__ __forceinline__ void read(const uint8_t *row, int r, int q) {
    c[0] = *reinterpret_cast<const glm_u32x4 *>(row + 16 * (q ^ swz(r)));
    c[1] = *reinterpret_cast<const glm_u32x4 *>(row + 16 * ((4 + q) ^ swz(r)));
  }
  __device__ __forceinline__ glm_bf16x8 frag(int i, float) const {
    return __builtin_bit_cast(glm_bf16x8, c[i]);
  }
};

// One stage of the ring: [16 TB WT tokens][kChunk bf16], then
// [64 BR weight rows][kRow], then (MX) [64 BR] dwords of E8M0 bytes.  WT waves
// along the tokens; as many stages (2 to 8) as fit KB: a small tile's chunk
// takes the memory latency over the chunks in flight.
template <int FMT, int BR, int TB, int WT, int KB>
struct DenseLds {
  using Raw = DenseRaw<FMT>;
  static constexpr bool kMx = FMT != FMT_BF16;
  static constexpr int kWaves = kDenseWF * WT;
  static constexpr int kTok = 16 * TB * WT, kRows = 16 * BR * kDenseWF;
  static constexpr int kXRow = Raw::kChunk * 2, kXPieces = kXRow / 16;
  static constexpr int kWPieces = Raw::kRow / 16;
  static constexpr int kX = kTok * kXRow, kW = kRows * Raw::kRow, kS = kMx ? kRows * 4 : 0;
  static constexpr int kStage = kX + kW + kS;
  // direct loads per wave and stage (the first kRows / 64 waves add one of scales)
  static constexpr int kXLoads = kX / (1024 * kWaves), kWLoads = kW / (1024 * kWaves);
  static constexpr int kLoads = kXLoads + kWLoads;
  static_assert(kX % (1024 * kWaves) == 0 && kW % (1024 * kWaves) == 0, "staging");
  static constexpr int kStages = KB * 1024 / kStage < 8 ? KB * 1024 / kStage : 8;
  static constexpr int kBytes = kStages * kStage;
  static_assert(kStages >= 2, "LDS ring exceeds its share");
  __device__ static int xswz(int row) { return row & (kXPieces - 1); }
};

// Waits until at most `ahead` (0 .. MAX, uniform) chunks of LOADS loads are
// outstanding.
template <int MAX, int LOADS>
__device__ __forceinline__ void wait_chunks_ahead(int ahead) {
  static_assert(MAX * LOADS < 64, "the wait counter's range");
  if (ahead >= MAX) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(MAX * LOADS));
  } else if constexpr (MAX > 0) {
    wait_chunks_ahead<MAX - 1, LOADS>(ahead);
  }
}

// One workgroup's work item; lin is its workgroup's index among the launch's
// dense ones, congruent to blockIdx.x modulo the XCDs.
template <int FMT, int NPROJ, int BR, int TB, int WT, int KB>
__device__ __forceinline__ void dense_item(const DenseArgs &a, int lin) {
  using L = DenseLds<FMT, BR, TB, WT, KB>;
  constexpr int kWaves = L::kWaves;
  using Raw = DenseRaw<FMT>;
  constexpr int kI = Raw::kChunk / 32;        // MFMAs along a chunk
  constexpr int kFeat = L::kRows / NPROJ;     // features per workgroup
  constexpr int HB = BR / NPROJ;              // 16-row blocks per projection of a wave
  constexpr int kS = L::kStages;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  // XCD-aware: workgroups are dealt to the 8 XCDs round-robin by linear id, so
  // XCD x takes the x-th contiguous eighth of the items
  const int items = a.row_tiles * a.tok_tiles;
  const int per_xcd = (items + kDenseXcds - 1) / kDenseXcds;
  const int on_xcd = lin / kDenseXcds;
  const int item = (lin % kDenseXcds) * per_xcd + on_xcd;
  if (on_xcd >= per_xcd || item >= items) return;
  const int rt = a.rows_outer ? item / a.tok_tiles : item % a.row_tiles;
  const int tt = a.rows_outer ? item % a.tok_tiles : item / a.row_tiles;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int wf = wave % kDenseWF, wt = wave / kDenseWF;
  const int K = a.K, N = a.N;
  const int nchunks = K / Raw::kChunk;
  const int f0 = rt * kFeat, t0 = tt * L::kTok;

  // ---- load assignment, fixed over the K loop: load j of wave w fills the
  // (kWaves j + w)-th 1 KB of the tokens, then of the weight rows.  Tokens past the
  // last one and rows past the last feature re-read the last (their MFMA rows
  // and columns are independent of the others and not stored).
  uint32_t xoff[L::kXLoads], woff[L::kWLoads];
#pragma unroll
  for (int j = 0; j < L::kXLoads; ++j) {
    const int slot = (j * kWaves + wave) * 64 + lane;
    const int row = slot / L::kXPieces, piece = (slot % L::kXPieces) ^ L::xswz(row);
    xoff[j] = (uint32_t)min(t0 + row, a.T - 1) * (uint32_t)(2 * K) + 16 * piece;
  }
#pragma unroll
  for (int j = 0; j < L::kWLoads; ++j) {
    const int slot = (j * kWaves + wave) * 64 + lane;
    const int row = slot / L::kWPieces, piece = (slot % L::kWPieces) ^ Raw::swz(row);
    woff[j] = (uint32_t)min(f0 + row % kFeat, N - 1) * (uint32_t)row_bytes(FMT, K) + 16 * piece;
  }
  const int srow = (wave * 64 + lane) % L::kRows;  // (waves past the rows load none)
  const uint32_t soff = (uint32_t)min(f0 + srow % kFeat, N - 1) * (uint32_t)(K >> 5);
  const uint32_t wbytes = (uint32_t)N * (uint32_t)row_bytes(FMT, K), sbytes = (uint32_t)N * (uint32_t)(K >> 5);
  const __amdgpu_buffer_rsrc_t xres = make_rsrc(a.x, (uint32_t)a.T * (uint32_t)(2 * K));
  const __amdgpu_buffer_rsrc_t wres[2] = {make_rsrc(a.w[0], wbytes), make_rsrc(a.w[NPROJ - 1], wbytes)};
  const __amdgpu_buffer_rsrc_t sres[2] = {make_rsrc(a.s[0], sbytes), make_rsrc(a.s[NPROJ - 1], sbytes)};
  auto issue = [&](int c, int stage) {
    uint8_t *base = smem + stage * L::kStage;
    if (L::kMx && wave * 64 < L::kRows) {  // (whole waves lie in one projection: kFeat % 64 == 0)
      const bool up = NPROJ == 2 && wave * 64 >= kFeat;
      buf4_to_lds(up ? sres[1] : sres[0], base + L::kX + L::kW + wave * 256, soff, (uint32_t)c * 4);
    }
#pragma unroll
    for (int j = 0; j < L::kXLoads; ++j)
      buf16_to_lds(xres, base + (j * kWaves + wave) * 1024, xoff[j], (uint32_t)c * L::kXRow);
#pragma unroll
    for (int j = 0; j < L::kWLoads; ++j) {
      // a 1 KB block of rows lies in one projection
      const bool up = NPROJ == 2 && (j * kWaves + wave) * (1024 / Raw::kRow) >= kFeat;
      buf16_to_lds(up ? wres[1] : wres[0], base + L::kX + (j * kWaves + wave) * 1024, woff[j],
                   (uint32_t)c * Raw::kRow);
    }
  };

  glm_f32x4 acc[BR][TB];
#pragma unroll
  for (int b = 0; b < BR; ++b)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[b][t] = glm_f32x4{0.f, 0.f, 0.f, 0.f};

  // staged row of this lane in the wave's block b
  auto wrow = [&](int b) { return (b / HB) * kFeat + wf * HB * 16 + (b % HB) * 16 + r; };
  auto compute = [&](int stage) {
    const uint8_t *base = smem + stage * L::kStage;
    const uint8_t *sx = base + (wt * TB * 16 + r) * L::kXRow;
    Raw w[BR];
    float sc[BR];
#pragma unroll
    for (int b = 0; b < BR; ++b) {
      w[b].read(base + L::kX + wrow(b) * Raw::kRow, r, q);
      sc[b] = L::kMx ? e8m0_to_f32(base[L::kX + L::kW + wrow(b) * 4 + q]) : 1.0f;
    }
#pragma unroll
    for (int i = 0; i < kI; ++i) {
      const int piece = (L::kMx ? 4 * q + i : 4 * i + q) ^ L::xswz(r);
      glm_bf16x8 af[BR];
#pragma unroll
      for (int b = 0; b < BR; ++b) af[b] = w[b].frag(i, sc[b]);
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        const glm_bf16x8 xb = *reinterpret_cast<const glm_bf16x8 *>(sx + t * 16 * L::kXRow + 16 * piece);
#pragma unroll
        for (int b = 0; b < BR; ++b)
          acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[b], xb, acc[b][t], 0, 0, 0);
      }
    }
  };
  // Ring: the loads of the next kS - 1 chunks are in flight while one is
  // multiplied.  The barrier of chunk c also says that every wave is done with
  // chunk c - 1, whose stage the loads of chunk c + kS - 1 overwrite.
#pragma unroll
  for (int c = 0; c < kS - 1; ++c)
    if (c < nchunks) issue(c, c);
  int stage = 0;
  for (int c = 0; c < nchunks; ++c) {
    // (waves that load scales too have more in flight and wait for a little more)
    wait_chunks_ahead<kS - 2, L::kLoads>(min(kS - 2, nchunks - 1 - c));
    ring_barrier();
    if (c + kS - 1 < nchunks) issue(c + kS - 1, stage == 0 ? kS - 1 : stage - 1);
    compute(stage);
    stage = stage + 1 == kS ? 0 : stage + 1;
  }

  // ---- epilogue: each 16-token block of the wave's features through its own
  // LDS area, so that a token's features leave as one contiguous piece
  ring_barrier();
  constexpr int kSegs = 2 * HB;  // 16-byte pieces of a token's features
  constexpr int kStride = 16 * kSegs + 16;
  static_assert(kWaves * 16 * kStride <= L::kBytes, "output staging");
  uint8_t *yst = smem + wave * 16 * kStride;
  const int fw = f0 + wf * HB * 16, tw = t0 + wt * TB * 16;
#pragma unroll
  for (int t = 0; t < TB; ++t) {
    if (tw + 16 * t >= a.T) break;
#pragma unroll
    for (int b = 0; b < HB; ++b) {
      uint32_t o[4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
        o[m] = NPROJ == 2 ? f32_to_bf16(limited_swiglu(bf16_round(acc[b][t][m]),
                                                       bf16_round(acc[BR - HB + b][t][m]), a.limit))
                          : f32_to_bf16(acc[b][t][m]);
      *reinterpret_cast<uint2 *>(yst + r * kStride + (b * 16 + 4 * q) * 2) =
          uint2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int p = 0; p < 16 * kSegs; p += 64) {
      const int tok = (p + lane) / kSegs, seg = (p + lane) % kSegs;
      if (tok < 16 && tw + 16 * t + tok < a.T && fw + 8 * seg < N)
        *reinterpret_cast<glm_u32x4 *>(a.out + (size_t)(tw + 16 * t + tok) * N + fw + 8 * seg) =
            *reinterpret_cast<const glm_u32x4 *>(yst + tok * kStride + 16 * seg);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

}  // namespace glm
