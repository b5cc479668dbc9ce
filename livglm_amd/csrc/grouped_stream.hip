// Block-scaled grouped GEMMs for few rows per expert, where the experts'
// weights are what a launch waits for (the layer's routed projections,
// native_expert_ssd.py:726-743, as grouped_gemm.hip's wide forms).
//
// A workgroup is four waves over a row tile of up to 64 rows x 256 weight rows
// (gate/up: 128 features of each projection), a wave 64 weight rows x all of
// the tile's rows.  A wave's weights are its own, so they go from the
// tile-major bank straight into registers in the MFMA's operand order, two
// chunks of 4 KB ahead; only the activations, which all four waves read, and
// the scales pass through LDS (a ring of three stages, filled by direct loads
// in the same order).  That leaves room for two workgroups a CU, whose loads
// overlap each other's barriers, first loads and epilogues; the wide forms
// have one workgroup a CU with a 32 KB chunk of weights in flight and nothing
// beside its start and end.
//
// Two kinds of activations.  BF: bf16 as they are, the weights converted to
// bf16 (exact) on their way into the MFMA, which the wait for the weights
// covers; their loads are non-temporal (about one row tile an expert).  Else
// the wide forms' FP8 hi/lo split, twice the rows per MFMA time, in their
// order of sums, so that the results are theirs bit for bit.
//
// Layers of uniform routing, the wide forms in brackets: d 2048, E 128, k 8,
// I 768, 333 tokens 111 us (157); d 4096, E 288, k 8, I 2048, 66 tokens 586 us
// (793), 200 tokens 703 us (912), 1023 tokens 890 us (1128).  In split form
// without non-temporal loads 333 tokens took 123 us, with them 114; four stages
// measured 1 % slower, two stages 1 to 3 %.
//
// The shared expert's dense tiles (dense_tile.h) ride in the same launches, so
// that its MFMAs run beside the experts' weight stream: at 333 tokens (d 2048,
// split form) 123 us where its two products as launches of their own made it
// 152, at 1500 (E 120, d 1536) 138 and 163.
#include <algorithm>
#include <cmath>

#include "act_split.h"
#include "dense_tile.h"
#include "lds_stage.h"
#include "mfma_tile.h"
#include "topk_select.h"  // wave_lds_sync

namespace glm {

constexpr int kStreamRows = 64;          // rows of a row tile
constexpr int kStreamRing = 3;           // chunks in flight or in use

struct StreamLds {
  static constexpr int kRows = kStreamRows;
  static constexpr int kXS = kRows * 256;              // [2 terms][16 NB] scale dwords, whole waves
  static constexpr int kXSSlots = (2 * kRows + 63) / 64 * 64;
  static constexpr int kWS = kXS + kXSSlots * 4;       // [256 weight rows] scale dwords
  static constexpr int kStage = kWS + 256 * 4;
  static constexpr int kBytes = kStreamRing * kStage;
  static constexpr int kYRow = 144;  // bytes per row of the down epilogue's staging (128 + 16)
  static_assert(4 * 16 * kYRow <= kBytes, "the down epilogue's staging fits the ring");
};

constexpr int kStreamThreads = 256;
constexpr int kStreamCUs = 256;
constexpr int kStreamTileW = 256;  // weight rows per workgroup

template <int N>
struct StreamStage {
  static constexpr int value = N;
};
typedef int glm_i32x8 __attribute__((ext_vector_type(8)));

// A weight load; NT: non-temporal.
template <bool NT>
__device__ __forceinline__ glm_u32x4 buf16_load(__amdgpu_buffer_rsrc_t rs, uint32_t voff,
                                                uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, NT ? 2 : 0);
}

template <int NPROJ, bool BF, int NB>
__device__ __forceinline__ void stream_body(const SplitArgs &a, long long e, int pos0, int rows,
                                            int ftile) {
  using L = StreamLds;
  constexpr int RING = kStreamRing;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = a.K;
  const int nchunks = K / 128;
  constexpr int kHalf = kStreamTileW / 2;
  const int f0 = ftile * (kStreamTileW / NPROJ);
  auto act_row = [&](int row) -> uint32_t {
    const int pos = pos0 + (row < rows ? row : 0);  // past the end: re-read row 0
    return (uint32_t)(a.act_index != nullptr ? a.act_index[pos] : pos);
  };

  // ---- load assignment, fixed over the K loop; every wave issues the same
  // count per chunk: NB loads of 4 activation rows, one of 64 activation scale
  // slots, one of 64 weight rows' scales, then its four weight blocks
  // (BF has no activation scales)
  constexpr int kLoads = NB + (BF ? 1 : 2) + 4;
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(a.xhi, a.split_bytes);
  const uint32_t lo_off = (uint32_t)(a.xlo - a.xhi);
  uint32_t xoff[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int row = (j * 4 + wv) * 4 + (lane >> 4);
    const int piece = (lane & 15) ^ (row & 15);
    xoff[j] = BF ? act_row(row) * (uint32_t)(2 * K) + piece * 16
                 : act_row(row) * (uint32_t)K + (piece < 8 ? 0u : lo_off) + (piece & 7) * 16;
  }
  // scale slot s = term * 16 NB + row; slots past the last one (and the waves
  // past them) repeat earlier ones
  constexpr int kXSUsed = (2 * 16 * NB + 63) / 64 * 64;
  const int xs0 = (wv * 64) % kXSUsed;
  uint32_t xsoff = 0;
  if constexpr (!BF) {
    const int s = xs0 + lane < 2 * 16 * NB ? xs0 + lane : 0;
    xsoff = (uint32_t)((s >= 16 * NB ? a.xslo : a.xshi) - a.xhi) +
            act_row(s % (16 * NB)) * (uint32_t)(K / 32);
  }
  const bool up = NPROJ == 2 && wv >= 2;  // whose scales this wave loads
  const __amdgpu_buffer_rsrc_t wsrs =
      make_rsrc(a.s[up ? NPROJ - 1 : 0] + e * a.s_stride, (uint32_t)a.N * (uint32_t)(K / 32));
  const uint32_t wsoff =
      (uint32_t)(f0 + (NPROJ == 2 ? wv * 64 % kHalf : wv * 64) + lane) * (uint32_t)(K / 32);
  // the wave's four 16-row blocks: gate/up two of each projection (32
  // features), down 64 consecutive features
  const uint32_t wbytes = (uint32_t)a.N * (uint32_t)(K / 2);
  const __amdgpu_buffer_rsrc_t wrs[2] = {make_rsrc(a.w[0] + e * a.w_stride, wbytes),
                                         make_rsrc(a.w[NPROJ - 1] + e * a.w_stride, wbytes)};
  uint32_t wuni[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
    wuni[b] = (uint32_t)((f0 + (NPROJ == 2 ? wv * 32 + (b % 2) * 16 : wv * 64 + b * 16)) / 16) *
              (uint32_t)(K / 128) * 1024u;

  glm_u32x4 w[RING][4];
  // the loads of chunk c into stage st; chunks past the last one read nothing
  // (an offset past the buffer; in a split above 2 GiB another place of it),
  // so that every step issues the same count
  auto issue = [&](int c, int st) {
    const bool in = c < nchunks;
    const uint32_t far = in ? 0u : 0x80000000u;
    const uint32_t cx = (in ? (uint32_t)c * (BF ? 256u : 128u) : 0u) + far, cs = (in ? (uint32_t)c * 4u : 0u) + far;
    uint8_t *base = smem + st * L::kStage;
#pragma unroll
    for (int j = 0; j < NB; ++j) buf16_to_lds(xrs, base + (j * 4 + wv) * 1024, xoff[j] + cx, 0);
    if constexpr (!BF) buf4_to_lds(xrs, base + L::kXS + xs0 * 4, xsoff + cs, 0);
    buf4_to_lds(wsrs, base + L::kWS + wv * 256, wsoff + cs, 0);
    const uint32_t wl = 16u * lane + (in ? (uint32_t)c * 1024u : 0u) + far;
#pragma unroll
    for (int b = 0; b < 4; ++b) w[st][b] = buf16_load<BF>(wrs[NPROJ == 2 ? b / 2 : 0], wl, wuni[b]);
    __builtin_amdgcn_sched_barrier(0);
  };

  glm_f32x4 acc[4][NB];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int t = 0; t < NB; ++t) acc[b][t] = glm_f32x4{0.f, 0.f, 0.f, 0.f};

  // activation row 16 m + r, piece p at row * 256 + 16 (p ^ r); term t's
  // operand is pieces 8 t + q and 8 t + 4 + q
  const uint32_t xl = (uint32_t)(r * 256 + 16 * (q ^ r));
  const uint32_t xsl = (uint32_t)(L::kXS + 4 * r + q);
  const uint32_t wsl = (uint32_t)(L::kWS + 4 * ((NPROJ == 2 ? wv * 32 : wv * 64) + r) + q);
  auto compute = [&](int st) {
    const uint8_t *base = smem + st * L::kStage;
    int wsc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
      wsc[b] = base[wsl + 4 * (NPROJ == 2 ? (b / 2) * kHalf + (b % 2) * 16 : b * 16)];
    if constexpr (BF) {
      // MFMA i takes K = 32 q + 8 i + s in lane (r, q): piece 4 q + i
      float sc[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) sc[b] = e8m0_to_f32((uint32_t)wsc[b]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        glm_bf16x8 af[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) af[b] = mxfp4_word_to_bf16x8(w[st][b][i], sc[b]);
#pragma unroll
        for (int ct = 0; ct < NB; ++ct) {
          const glm_bf16x8 xb = *reinterpret_cast<const glm_bf16x8 *>(
              base + r * 256 + 16 * ((4 * q + i) ^ r) + ct * 4096);
#pragma unroll
          for (int b = 0; b < 4; ++b)
            acc[b][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[b], xb, acc[b][ct], 0, 0, 0);
        }
      }
    } else {
    glm_i32x8 wa[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const glm_u32x4 v = w[st][b];
      wa[b] = glm_i32x8{(int)v[0], (int)v[1], (int)v[2], (int)v[3], 0, 0, 0, 0};
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ct = 0; ct < NB; ++ct) {
        const glm_u32x4 b0 =
            *reinterpret_cast<const glm_u32x4 *>(base + (xl ^ (128u * t)) + ct * 4096);
        const glm_u32x4 b1 =
            *reinterpret_cast<const glm_u32x4 *>(base + (xl ^ (128u * t + 64u)) + ct * 4096);
        const glm_i32x8 xb = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3],
                              (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
        const int xsc = base[xsl + 4 * (t * 16 * NB + ct * 16)];
#pragma unroll
        for (int b = 0; b < 4; ++b)
          acc[b][ct] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wa[b], xb, acc[b][ct], 4, 0,
                                                                        0, wsc[b], 0, xsc);
      }
    }
  };

  // Chunk c: wait for its loads (those of the RING - 2 chunks after it stay in
  // flight), meet the other waves -- their loads of it have landed too, and
  // none reads chunk c - 1 any more, whose stage takes chunk c + RING - 1.
  // The loop takes RING chunks a turn, so that a chunk's stage is static; what
  // is left over starts at stage 0 again and needs no more loads.
#pragma unroll
  for (int c = 0; c < RING - 1; ++c) issue(c, c);
  int c0 = 0;
  for (; c0 + RING <= nchunks; c0 += RING) {
#pragma unroll
    for (int u = 0; u < RING; ++u) {
      // (fences: MFMAs moved across the barrier keep two chunks' operands alive)
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((RING - 2) * kLoads));
      ring_barrier();
      __builtin_amdgcn_sched_barrier(0);
      issue(c0 + u + RING - 1, (u + RING - 1) % RING);
      compute(u);
    }
  }
  auto left = [&](auto ut) {
    constexpr int U = decltype(ut)::value;
    if (U < RING - 1 && c0 + U < nchunks) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((U < RING - 1 ? RING - 2 - U : 0) * kLoads));
      ring_barrier();
      compute(U);
    }
  };
  left(StreamStage<0>{});
  left(StreamStage<1>{});
  left(StreamStage<2>{});
  static_assert(RING <= 4, "at most three chunks are left over");
  // no load may land in LDS that this workgroup reuses or leaves
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));

  // ---- epilogue: lane (r, q) of block (b, ct) holds weight rows 4q..4q+3 of
  // the block for token column r
  if constexpr (NPROJ == 2 && BF) {
#pragma unroll
    for (int ct = 0; ct < NB; ++ct) {
      const int row = ct * 16 + r;
      if (row >= rows) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint32_t o[4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
          o[m] = f32_to_bf16(limited_swiglu(bf16_round(acc[i][ct][m]), bf16_round(acc[2 + i][ct][m]),
                                            a.limit));
        store_rows4(a.out + (size_t)(pos0 + row) * a.N + f0 + wv * 32 + i * 16 + 4 * q, o);
      }
    }
  } else if constexpr (NPROJ == 2) {
    // h's FP8 hi/lo split, as the wide forms write it: the wave's 32 features
    // of a token are one scale group, 8 per lane in lanes (r, q = 0..3)
    const float lim = a.limit > 0.0f ? a.limit : __builtin_inff();
    const SplitLayout S(a.out_rows, a.N);
    const int g0 = f0 + wv * 32;
#pragma unroll
    for (int ct = 0; ct < NB; ++ct) {
      const int row = ct * 16 + r;
      float v[8];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int m = 0; m < 4; m += 2) {
          float ga = acc[i][ct][m], gb = acc[i][ct][m + 1];
          float ua = acc[2 + i][ct][m], ub = acc[2 + i][ct][m + 1];
          bf16_round2(ga, gb);
          bf16_round2(ua, ub);
          limited_swiglu2_fast(ga, gb, ua, ub, lim, v[4 * i + m], v[4 * i + m + 1]);
        }
      uint32_t ch[2], cl[2];
      int bh, bl;
      split_group_part(v, ch, cl, &bh, &bl);
      if (row < rows) {
        const size_t prow = (size_t)(pos0 + row);
        uint8_t *hi = a.out_split + prow * a.N + g0;
        uint8_t *lo = a.out_split + S.lo + prow * a.N + g0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          *reinterpret_cast<uint32_t *>(hi + i * 16 + 4 * q) = ch[i];
          *reinterpret_cast<uint32_t *>(lo + i * 16 + 4 * q) = cl[i];
        }
        if (q == 0) {
          a.out_split[S.shi + prow * (a.N / 32) + g0 / 32] = (uint8_t)bh;
          a.out_split[S.slo + prow * (a.N / 32) + g0 / 32] = (uint8_t)bl;
        }
      }
    }
  } else {
    // y through LDS so that every store writes whole 128-byte lines; the
    // wave's area lies in stages that every wave is done with
    ring_barrier();
    uint8_t *yst = smem + wv * (16 * L::kYRow);
    const int rr = lane >> 3, seg = lane & 7;
#pragma unroll
    for (int ct = 0; ct < NB; ++ct) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        uint32_t o[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) o[m] = f32_to_bf16(acc[b][ct][m]);
        *reinterpret_cast<uint2 *>(yst + r * L::kYRow + (b * 16 + 4 * q) * 2) =
            uint2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
      }
      wave_lds_sync();
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = ct * 16 + 8 * h + rr;
        const glm_u32x4 v = *reinterpret_cast<const glm_u32x4 *>(yst + (8 * h + rr) * L::kYRow + 16 * seg);
        if (row < rows)
          *reinterpret_cast<glm_u32x4 *>(a.out + (size_t)(pos0 + row) * a.N + f0 + wv * 64 + 8 * seg) = v;
      }
      wave_lds_sync();
    }
  }
}

// The riding product's tile: 128 weight rows (gate/up: 64 features of each
// projection) x 64 tokens, on four waves.
constexpr int kRideKB = 78;  // LDS of a workgroup, two a CU
template <int FMT>
using RideLds = DenseLds<FMT, 2, 4, 1, kRideKB>;

// Work items and their order as in the wide forms (a tile of more than
// kStreamRows rows is cut there).  FMT >= 0: the riding product's workgroups
// lie between the routed ones in groups of one per XCD, the first of every
// `period` + 1 groups until there are no more of them.
template <int NPROJ, bool BF, int FMT>
__global__ __launch_bounds__(kStreamThreads) __attribute__((amdgpu_waves_per_eu(2)))
void grouped_stream_kernel(SplitArgs a, DenseArgs ride, int ride_groups, int period) {
  int group = blockIdx.x / kXcds;
  const int xcd = blockIdx.x % kXcds;
  if constexpr (FMT >= 0) {
    if (group < ride_groups * (period + 1)) {
      const int before = group / (period + 1);
      if (group % (period + 1) == 0)
        return dense_item<FMT, NPROJ, 2, 4, 1, kRideKB>(ride, before * kXcds + xcd);
      group -= before + 1;
    } else {
      group -= ride_groups;
    }
  }
  const int nft = a.feature_tiles;
  const int ntiles = max(0, min(*a.num_tiles, a.max_tiles));
  const int items = ntiles * nft;
  const int per_xcd = (items + kXcds - 1) / kXcds;
  const int item = xcd * per_xcd + group;
  if (group >= per_xcd || item >= items) return;
  const int4 tile = a.tiles[item / nft];
  if (tile.z <= 0 || tile.x < 0 || tile.y < 0) return;
  const int rows = min(tile.z, kStreamRows);
  const int ftile = item % nft;
  const int nb = __builtin_amdgcn_readfirstlane((rows + 15) >> 4);
  if (nb == 4) return stream_body<NPROJ, BF, 4>(a, tile.x, tile.y, rows, ftile);
  if (nb == 3) return stream_body<NPROJ, BF, 3>(a, tile.x, tile.y, rows, ftile);
  if (nb == 2) return stream_body<NPROJ, BF, 2>(a, tile.x, tile.y, rows, ftile);
  stream_body<NPROJ, BF, 1>(a, tile.x, tile.y, rows, ftile);
}

}  // namespace glm

using namespace glm;

int glm_grouped_tile_rows();

int glm_grouped_stream_rows() { return kStreamRows; }

// Whether the streaming form takes bf16 activations or their split: up to 48
// rows an expert (d 4096, E 288: 600 / 1023 tokens, 17 / 28 rows, 801 / 890
// against 845 / 918 us; E 128, 44 rows 150 and 149; E 120, 75 rows 141 and 139).
bool glm_grouped_stream_bf16(long long pairs, int E) { return pairs <= 48LL * E; }

// How well the wide forms' items fill the CUs: the share of whole rounds of them,
// with half the weight on how full the tiles' rows are (an item's time is its K
// loop before it is its rows).  The rows of an expert are taken a tenth above the
// average, since a tile more on some experts starts a round.
static double wide_fill(long long pairs, int E, int d, int I) {
  const int tile_rows = glm_grouped_tile_rows();
  const double tiles = E * std::ceil(1.1 * pairs / E / tile_rows);
  const double gate_up = tiles * ((I + 255) / 256), down = tiles * d / 512;
  auto rounds = [](double items) { return std::ceil(items / kStreamCUs); };
  const double full = (gate_up * d + down * I) / kStreamCUs / (rounds(gate_up) * d + rounds(down) * I);
  return full * (0.5 + 0.5 * pairs / (tiles * tile_rows));
}

// Rows per tile of the layer's grouped GEMMs, the streaming form's or the wide
// forms' (256 features by at most glm_grouped_tile_rows rows).  Layer times, wide
// against streaming.
//
// Up to 88 rows an expert the streaming form (75 rows, d 1536, E 120, I 640: 159 :
// 140 us; at 94, d 2048, E 128, I 768: 211 : 216), but not above 60 rows at long K
// where the wide forms fill at least two rounds (d 4096, E 288, I 2048, MXFP8 shared
// expert: 58 rows 1395 : 1383 us, 64 rows 1435 : 1570; d 5120, E 128, I 1536: 56 rows
// 636 : 634, 75 rows 698 : 782; rounds 0.78 full, E 160, I 1280: 70 rows 612 : 605).
//
// Above, the streaming form while the wide forms' items are fewer than the CUs and
// fill them badly (bf16 shared expert; d 1024, E 16, k 2, I 512: 256 rows, fill 0.23, 91 :
// 70 us, 512 rows, 0.45, 99 : 97, 1024 rows, 0.9, 131 : 152; d 1024, E 8, k 2, I 256: 1024
// rows, 0.27, 89 : 78, 4096 rows, 0.85, 165 : 189; d 2048, E 24, k 8, I 768: 333 rows, 0.61,
// 150 : 130; d 2048, E 64, k 8, I 512: 175 rows, 0.77, 155 : 135; d 4096, where K is
// longer: E 16, k 4, I 1024: 350 rows, 0.65, 258 : 247, 500 rows, 0.89, 310 : 334; E 8, k 2,
// I 2048: 400 rows, 0.69, 289 : 317).
int glm_grouped_layer_tile_rows(long long pairs, int E, int d, int I) {
  const int wide = glm_grouped_tile_rows();
  const int features = (I + 255) / 256;
  const bool long_k = d >= 4096;
  bool stream;
  if (pairs <= 88LL * E)
    stream = !(long_k && pairs > 60LL * E && E * features >= 2 * kStreamCUs &&
               wide_fill(pairs, E, d, I) >= 0.65);
  else
    stream = std::max((long long)E, pairs / wide) * features < kStreamCUs &&
             wide_fill(pairs, E, d, I) < (long_k ? 0.68 : 0.8);
  return stream ? kStreamRows : wide;
}

template <int NPROJ, bool BF, int FMT>
static void launch_stream(hipStream_t stream, const SplitArgs &a, long long groups, int E,
                          const RidingGemm *ride) {
  DenseArgs d{};
  long long ride_groups = 0, period = 0;
  size_t lds = StreamLds::kBytes;
  if constexpr (FMT >= 0) {
    using L = RideLds<FMT>;
    constexpr int feat = L::kRows / NPROJ;
    d.x = ride->x;
    for (int p = 0; p < 2; ++p) {
      d.w[p] = static_cast<const uint8_t *>(ride->w[p]);
      d.s[p] = ride->s[p];
    }
    d.out = ride->out;
    d.T = ride->T;
    d.N = ride->N;
    d.K = ride->K;
    d.limit = glm_limit_bf16(ride->limit);
    d.row_tiles = (d.N + feat - 1) / feat;
    d.tok_tiles = (d.T + L::kTok - 1) / L::kTok;
    d.rows_outer = 1;
    ride_groups = ((long long)d.row_tiles * d.tok_tiles + kXcds - 1) / kXcds;
    // spread over the groups that have work if every expert has a tile, but for
    // the last two rounds of the CUs: a riding item started there would end late
    constexpr long long kRound = 2 * kStreamCUs / kXcds;
    const long long busy = std::min(groups, ((long long)E * a.feature_tiles + kXcds - 1) / kXcds);
    period = std::max(0LL, busy - 2 * kRound) / ride_groups;
    lds = std::max(lds, (size_t)L::kBytes);
  }
  const dim3 grid((unsigned)((groups + ride_groups) * kXcds));
  hipLaunchKernelGGL((grouped_stream_kernel<NPROJ, BF, FMT>), grid, dim3(kStreamThreads), lds, stream,
                     a, d, (int)ride_groups, (int)period);
}

template <int NPROJ, bool BF>
static int stream_launch(hipStream_t stream, SplitArgs a, int max_tiles, int E,
                         const RidingGemm *ride) {
  a.feature_tiles = a.N / (kStreamTileW / NPROJ);
  a.max_tiles = max_tiles;
  const long long groups = ((long long)max_tiles * a.feature_tiles + kXcds - 1) / kXcds;
  if (ride == nullptr)
    launch_stream<NPROJ, BF, -1>(stream, a, groups, E, nullptr);
  else if (ride->fmt == GLM_FMT_MXFP8)
    launch_stream<NPROJ, BF, FMT_MXFP8>(stream, a, groups, E, ride);
  else if (ride->fmt == GLM_FMT_MXFP4)
    launch_stream<NPROJ, BF, FMT_MXFP4>(stream, a, groups, E, ride);
  else
    launch_stream<NPROJ, BF, FMT_BF16>(stream, a, groups, E, ride);
  GLM_LAUNCH_CHECK("grouped_stream_kernel");
  return GLM_OK;
}

// The routed gate/up over row tiles of glm_grouped_layer_tile_rows rows: x's
// split in, h's split out; `ride` (or null) a SwiGLU of two dense products.
int glm_grouped_stream_gate_up_launch(hipStream_t stream, const void *x_split, int T,
                                      const int32_t *pair_token, const int4 *tiles,
                                      const int32_t *num_tiles, int max_tiles, int d, int I, int E,
                                      const uint8_t *gw, const uint8_t *gs, const uint8_t *uw,
                                      const uint8_t *us, float limit, void *h_split, long long P,
                                      const RidingGemm *ride) {
  SplitArgs a{};
  set_split(a, x_split, T, d, ACT_FP8X2);
  a.out_split = static_cast<uint8_t *>(h_split);
  a.out_rows = P;
  a.act_index = pair_token;
  a.tiles = tiles;
  a.num_tiles = num_tiles;
  a.w[0] = gw;
  a.w[1] = uw;
  a.s[0] = gs;
  a.s[1] = us;
  a.w_stride = (long long)I * (d / 2);
  a.s_stride = (long long)I * (d / 32);
  a.N = I;
  a.K = d;
  a.limit = glm_limit_bf16(limit);
  return stream_launch<2, false>(stream, a, max_tiles, E, ride);
}

// The routed down over the same tiles; `ride` (or null) one dense product.
int glm_grouped_stream_down_launch(hipStream_t stream, const void *h_split, long long P,
                                   const int4 *tiles, const int32_t *num_tiles, int max_tiles,
                                   int I, int d, int E, const uint8_t *dw, const uint8_t *ds,
                                   uint16_t *y, const RidingGemm *ride) {
  SplitArgs a{};
  set_split(a, h_split, P, I, ACT_FP8X2);
  a.tiles = tiles;
  a.num_tiles = num_tiles;
  a.w[0] = a.w[1] = dw;
  a.s[0] = a.s[1] = ds;
  a.w_stride = (long long)d * (I / 2);
  a.s_stride = (long long)d * (I / 32);
  a.N = d;
  a.K = I;
  a.out = y;
  return stream_launch<1, false>(stream, a, max_tiles, E, ride);
}

// The same on bf16 activations: x [T][d] in, h [P][I] out.
int glm_grouped_stream_gate_up_bf16_launch(hipStream_t stream, const uint16_t *x, int T,
                                           const int32_t *pair_token, const int4 *tiles,
                                           const int32_t *num_tiles, int max_tiles, int d, int I,
                                           int E, const uint8_t *gw, const uint8_t *gs,
                                           const uint8_t *uw, const uint8_t *us, float limit,
                                           uint16_t *h, const RidingGemm *ride) {
  SplitArgs a{};
  a.xhi = a.xlo = a.xshi = a.xslo = reinterpret_cast<const uint8_t *>(x);
  a.split_bytes = (uint32_t)((size_t)T * d * 2);
  a.act_index = pair_token;
  a.tiles = tiles;
  a.num_tiles = num_tiles;
  a.w[0] = gw;
  a.w[1] = uw;
  a.s[0] = gs;
  a.s[1] = us;
  a.w_stride = (long long)I * (d / 2);
  a.s_stride = (long long)I * (d / 32);
  a.N = I;
  a.K = d;
  a.out = h;
  a.limit = glm_limit_bf16(limit);
  return stream_launch<2, true>(stream, a, max_tiles, E, ride);
}

// h [P][I] in, y [P][d] out.
int glm_grouped_stream_down_bf16_launch(hipStream_t stream, const uint16_t *h, long long P,
                                        const int4 *tiles, const int32_t *num_tiles, int max_tiles,
                                        int I, int d, int E, const uint8_t *dw, const uint8_t *ds,
                                        uint16_t *y, const RidingGemm *ride) {
  SplitArgs a{};
  a.xhi = a.xlo = a.xshi = a.xslo = reinterpret_cast<const uint8_t *>(h);
  a.split_bytes = (uint32_t)((size_t)P * I * 2);
  a.tiles = tiles;
  a.num_tiles = num_tiles;
  a.w[0] = a.w[1] = dw;
  a.s[0] = a.s[1] = ds;
  a.w_stride = (long long)d * (I / 2);
  a.s_stride = (long long)d * (I / 32);
  a.N = d;
  a.K = I;
  a.out = y;
  return stream_launch<1, true>(stream, a, max_tiles, E, ride);
}

bool glm_gemv_splits(int d, int I);

// Whether the decode layer (16 to 64 tokens, the router's logits on MFMA) runs
// on the streaming form instead of the decode kernels (decode_kernels: they take
// the layer), which go over K in one round of loads a workgroup and run an MX
// shared expert by itself.  At d 4096, E 288, k 8, I 2048: 16 / 24 / 32 / 64 tokens
// 298 / 383 / 432 / 573 us (decode kernels 301 / 409 / 498 / 723); d 2048, E 128,
// I 768: 63.9 / 74.6 / 76.1 / 86.9 (64.3 / 75.3 / 79.8 / 91.5), with an MXFP8 shared
// expert 63.6 / 74.5 / 75.9 / 86.5 (74.2 / 87.4 / 93.9 / 110.8).
//
// A streaming workgroup takes 128 features over all of K, a decode workgroup 16
// over a quarter of it, so the streaming form needs work items for the CUs.
// Counted for uniform routing, which 16 or more tokens come close to: items of
// the gate/up launch and rows per expert reached.  Layer times, decode kernels
// against streaming form, bf16 shared expert / none (d, E, k, I: tokens, items, rows):
//   4096, 16, 4, 512:  48, 64, 12    52 : 65 us /  46 : 52
//   2048, 32, 4, 512:  48, 128, 6    36 : 43    /  34 : 34
//   2048, 24, 8, 768:  32, 144, 11   43 : 44    /  39 : 36;  64, 144, 21  55 : 47 / 49 : 39
//   1024, 64, 4, 512:  16, 165, 1.6  28 : 30    /  27 : 28;  64, 252, 4   35 : 36 / 31 : 28
//   4096, 48, 8, 512:  48, 192, 8    77 : 73    /  71 : 60
//   4096, 64, 4, 512:  32, 224, 2.3              71 : 63;  64, 252, 4   82 : 90
//   3072, 64, 6, 512:  32, 245, 3    61 : 71    /  57 : 53
//   4096, 32, 8, 1024: 16, 253, 4    80 : 90    /  77 : 63;  64, 256, 16 129 : 94 / 109 : 69
// a little more than an item per CU makes some take two:
//   2048, 64, 2, 1024: 32, 327, 1.6  50 : 56    /  49 : 53
//   4096, 24, 8, 2048: 22, 384, 7   130 : 98
// and from 400 items on the streaming form is level or better throughout.  Below
// 32 MB of weights the layer is launches either way (d 1024, E 16, k 2, I 512, 32
// tokens: 23 : 30 / 21 : 25).  An MX shared expert costs the decode kernels two
// launches more, which only few, long items outweigh (MXFP8; 4096, 16, 4, 512: 16
// tokens 54 : 58 us, 20 58 : 59, 32 61 : 60; 1024, 16, 2, 512, 16 tokens 29 : 28).
//
// Where the decode kernels do not take the layer, the other choice is the GEMV
// tiles over the work list; the streaming form is taken whatever the size where
// these have no K split (d 1024, E 8, k 2, I 1408, 32 tokens: 27.5 us, one thread per
// output 2945).
bool glm_grouped_stream_decode(int T, int d, int E, int k, int I, int Is, int shared_fmt,
                               bool decode_kernels) {
  if (T < 16 || T > kStreamRows || d % 512 != 0 || I % 128 != 0) return false;
  const bool heavy = 1.5 * std::min((long long)E, (long long)T * k) * d * I >= 32e6;
  const bool mx = Is > 0 && shared_fmt != GLM_FMT_BF16;
  if (!decode_kernels) return heavy || mx || !glm_gemv_splits(d, I);
  const double reached = E * (1.0 - std::pow(1.0 - (double)k / E, T));
  const double items = reached * (I / 128), rows = T * k / reached;
  if (mx) return T >= 24 || items >= 96 || d <= 1024;
  if (!heavy) return false;
  if (items >= 400) return true;
  if (items > kStreamCUs && rows < 4) return false;
  // (the shared expert's own items need room beside the routed ones)
  if (T >= (Is > 0 ? 32 : 24)) return items >= 115 + d / ((Is > 0 ? 7 : 30) * rows);
  return items >= 180 && items * rows >= (Is > 0 ? 1400 : 1000);
}
