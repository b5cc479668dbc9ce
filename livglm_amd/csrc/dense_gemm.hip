// Dense many-token GEMMs of the resident linears and the MX shared expert on
// gfx950 MFMA (DeferredLinear.__call__, layers.py:38-70, and DenseMLP,
// layers.py:160-171, over a prompt's tokens):
//   NPROJ = 1: y[t][n] = bf16(x[t] . W[n])
//   NPROJ = 2: y[t][n] = limited_swiglu(bf16(x[t] . Wg[n]), bf16(x[t] . Wu[n]))
// with W row-major in MXFP8, MXFP4 or bf16.
//
// Split of the work.  A workgroup is eight waves, four along the weight rows x
// two along the tokens; a wave owns 16 BR weight rows (gate/up: half of them
// from each projection) x 16 TB tokens.  Both operands are staged in LDS by
// direct global->LDS loads whose consecutive lanes walk consecutive memory:
// the resident weights are row-major, and a wave that fetched its MFMA
// operands itself would touch a different row with every lane (64 L1 accesses
// a load; that form was bound by them at 1.55 us a 128-wide chunk whatever the
// tile).  The weights stay in their stored format in LDS and are converted to
// bf16 (exact, the scaled converts) on their way into the MFMA, so a chunk of
// them costs a quarter (MXFP4) or half (MXFP8) of its bf16 bytes in LDS space
// and reads.  16-byte pieces are XOR-swizzled by row so that operand reads hit
// distinct banks.
//
// Measured at 1500 tokens x 4096 x 4096 (the streaming tiles of mx_gemv.hip,
// which go over the weights once per 64 tokens, in brackets): MXFP8 55-62 us
// (415), MXFP4 52 (390), bf16 68 (433), i.e. 0.8-0.95 PFLOP/s; 4096 tokens
// MXFP8 145 us (1121).  What bounds it: a chunk's fixed part (barrier, operand
// reads and conversions before the first MFMAs) does not overlap its MFMAs.
//
// K of MFMA i, slot s of lane (r, q), r = lane & 15, q = lane >> 4:
//   MX formats  128 c + 32 q + 8 i + s   (lane q's 32 weights are one E8M0 group)
//   bf16         64 c + 32 i + 8 q + s
// Output lane (r, q) holds rows 4q..4q+3 of a 16-row block for token column r.
#include "dense_tile.h"

namespace glm {

constexpr int kDenseWT = 2;  // waves along the tokens
constexpr int kDenseThreads = 64 * kDenseWF * kDenseWT;
constexpr int kDenseCUs = 256;
constexpr int kDenseKB = 156;  // LDS of a workgroup, one a CU

template <int FMT, int BR, int TB>
using DenseTileLds = DenseLds<FMT, BR, TB, kDenseWT, kDenseKB>;

template <int FMT, int NPROJ, int BR, int TB>
__global__ __launch_bounds__(kDenseThreads) void dense_gemm_kernel(DenseArgs a) {
  dense_item<FMT, NPROJ, BR, TB, kDenseWT, kDenseKB>(a, blockIdx.x);
}

}  // namespace glm

using namespace glm;

template <int FMT, int NPROJ, int BR, int TB>
static void launch_dense_tile(hipStream_t stream, DenseArgs a) {
  using L = DenseTileLds<FMT, BR, TB>;
  constexpr int feat = L::kRows / NPROJ;
  a.row_tiles = (a.N + feat - 1) / feat;
  a.tok_tiles = (a.T + L::kTok - 1) / L::kTok;
  a.rows_outer = (long long)NPROJ * row_bytes(FMT, a.N) >= 2LL * a.T;
  const long long items = (long long)a.row_tiles * a.tok_tiles;
  const dim3 grid((unsigned)((items + kDenseXcds - 1) / kDenseXcds * kDenseXcds));
  hipLaunchKernelGGL((dense_gemm_kernel<FMT, NPROJ, BR, TB>), grid, dim3(kDenseThreads),
                     (size_t)L::kBytes, stream, a);
}

struct DenseTile {
  int br, tb;
};

// bf16 stages hold 64 of K: token tiles are pairs of blocks a wave there, so
// that a stage is whole rounds of loads, and MXFP4's need 128 weight rows for
// that; gate/up tiles hold both projections.
// 64-row tiles (br 1) are for few tokens.
template <int FMT, int NPROJ>
constexpr bool dense_takes(int br, int tb) {
  return (FMT != FMT_BF16 || tb % 2 == 0) &&
         (br > 1 || (FMT != FMT_MXFP4 && NPROJ == 1 && tb <= 2));
}

// The tile that takes the fewest rounds of the CUs, each priced by its size.
// A workgroup alone on its CU took, in us per 128 of K (MXFP8, K 4096):
// 0.81 + 0.055 br tb with 256-row tiles (tb 1 / 2 / 3 / 4: 1.04 / 1.23 / 1.46 /
// 1.68), 0.48 + 0.08 br tb with 128-row ones (0.65 / 0.78 / 0.93 / 1.15); the
// weights below are these in one unit, used for the other formats and for
// gate/up as well.  64-row tiles (tb 1 / 2: 0.43 / 0.52)
// where those would leave most of the chip idle: 100 tokens at N = K = 4096
// 15.8 us in MXFP8 and 20.1 in bf16, where 128-row tiles take 20.5 and 26.3.
// Picked against measured best at
// N 4096, K 4096: T 1500 (4, 3) 62 us, where (4, 4) takes 70, (2, 3) 68,
// (4, 2) 93; T 333, N 2048, K 2048: (2, 1) 12 us, (4, 4) 29.
template <int FMT, int NPROJ>
static DenseTile dense_tile(int T, int N) {
  DenseTile best{0, 0};
  long long best_cost = 0;
  for (int br = 4; br >= 1; br /= 2)
    for (int tb = 4; tb >= 1; --tb) {
      if (!dense_takes<FMT, NPROJ>(br, tb)) continue;
      const int feat = 64 * br / NPROJ;
      const long long items = (long long)((N + feat - 1) / feat) * ((T + 32 * tb - 1) / (32 * tb));
      const long long rounds = (items + kDenseCUs - 1) / kDenseCUs;
      const long long cost =
          rounds * (br == 4 ? 30 + 2 * br * tb : br == 2 ? 18 + 3 * br * tb : 14 + 4 * tb);
      if (!best.br || cost < best_cost) {
        best = DenseTile{br, tb};
        best_cost = cost;
      }
    }
  return best;
}

template <int FMT, int NPROJ, int BR, int TB = 4>
static void launch_dense_rows(hipStream_t stream, const DenseArgs &a, int tb) {
  if constexpr (dense_takes<FMT, NPROJ>(BR, TB)) {
    if (tb == TB) return launch_dense_tile<FMT, NPROJ, BR, TB>(stream, a);
  }
  if constexpr (TB > 1) launch_dense_rows<FMT, NPROJ, BR, TB - 1>(stream, a, tb);
}

template <int FMT, int NPROJ>
static int launch_dense(hipStream_t stream, const DenseArgs &a) {
  const DenseTile tile = dense_tile<FMT, NPROJ>(a.T, a.N);
  if (tile.br == 4)
    launch_dense_rows<FMT, NPROJ, 4>(stream, a, tile.tb);
  else if (tile.br == 2)
    launch_dense_rows<FMT, NPROJ, 2>(stream, a, tile.tb);
  else
    launch_dense_rows<FMT, NPROJ, 1>(stream, a, tile.tb);
  GLM_LAUNCH_CHECK("dense_gemm_kernel");
  return GLM_OK;
}

// K in whole chunks, N in whole 16-row blocks, x and W within the reach of
// 32-bit offsets, and scales that can be read four at a time (s0, s1: of the
// two projections, or null).
bool glm_dense_gemm_supported(int T, int K, int N, int fmt, const uint8_t *s0, const uint8_t *s1) {
  return (((uintptr_t)s0 | (uintptr_t)s1) & 3u) == 0 && T >= 1 && N >= 16 && N % 16 == 0 && K % (fmt == GLM_FMT_BF16 ? 64 : 128) == 0 &&
         2LL * T * K < (1LL << 32) && 2LL * N * K < (1LL << 32);
}

// nproj 1: out = x W^T; 2: the SwiGLU of two projections (w1/s1 the up one).
int glm_dense_gemm_launch(hipStream_t stream, int nproj, const uint16_t *x, int T, int K,
                          const void *w0, const uint8_t *s0, const void *w1, const uint8_t *s1,
                          int fmt, int N, float limit, uint16_t *out) {
  DenseArgs a{};
  a.x = x;
  a.w[0] = static_cast<const uint8_t *>(w0);
  a.w[1] = static_cast<const uint8_t *>(w1);
  a.s[0] = s0;
  a.s[1] = s1;
  a.out = out;
  a.T = T;
  a.N = N;
  a.K = K;
  a.limit = glm_limit_bf16(limit);
  if (nproj == 2) {
    switch (fmt) {
      case GLM_FMT_MXFP8: return launch_dense<FMT_MXFP8, 2>(stream, a);
      case GLM_FMT_MXFP4: return launch_dense<FMT_MXFP4, 2>(stream, a);
      default: return launch_dense<FMT_BF16, 2>(stream, a);
    }
  }
  switch (fmt) {
    case GLM_FMT_MXFP8: return launch_dense<FMT_MXFP8, 1>(stream, a);
    case GLM_FMT_MXFP4: return launch_dense<FMT_MXFP4, 1>(stream, a);
    default: return launch_dense<FMT_BF16, 1>(stream, a);
  }
}
