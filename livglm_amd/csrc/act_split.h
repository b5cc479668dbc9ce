// Activation splits of the block-scaled MFMA GEMMs (grouped_gemm.hip,
// grouped_stream.hip): their formats, layout and the FP8 hi/lo arithmetic, and
// the arguments that the GEMMs share.
#pragma once

#include "glm_common.h"

namespace glm {

constexpr int kXcds = 8;

// Activation formats of the block-scaled GEMMs (the C ABI's act_format).
constexpr int ACT_FP8X2 = 0, ACT_FP6X2 = 1, ACT_FP4 = 2, ACT_FP8FP6 = 3;

__host__ __device__ constexpr int act_terms(int af) { return af == ACT_FP4 ? 1 : 2; }
// Stored code bytes of one term per activation row of K elements.
__host__ __device__ constexpr long long act_code_row(int K, int af) {
  return af == ACT_FP4 ? K / 2 : K;
}

// Byte offsets of an activation split of `rows` x K: hi codes, lo codes,
// hi scales, lo scales, each 256-byte aligned (ACT_FP4: codes, scales).
// Code rows: ACT_FP8X2 one byte per element; ACT_FP4 two per byte, low
// nibble first (the MXFP4 weight layout); ACT_FP6X2 per 128-element chunk
// 128 bytes: group g's 32 codes packed 6 bits each, low bits first, bytes
// 0..15 at 16 g and bytes 16..23 at 64 + 16 g (so that the FP8 operand reads
// -- 16 bytes at 16 g and at 64 + 16 g -- fetch a whole E2M3 operand; the
// other 8 bytes are zero).
struct SplitLayout {
  size_t lo, shi, slo, total;
  __host__ __device__ SplitLayout(long long rows, int K, int af = ACT_FP8X2) {
    const size_t codes = ((size_t)(rows * act_code_row(K, af)) + 255) & ~(size_t)255;
    const size_t scales = ((size_t)rows * (K / 32) + 255) & ~(size_t)255;
    const int n = act_terms(af);
    lo = codes;
    shi = n * codes;
    slo = shi + scales;  // ACT_FP4: past the end, unused
    total = n * (codes + scales);
  }
};

// E8M0 exponent byte for a group whose largest magnitude is amax: the
// smallest 2^(b - 127) with amax / 2^(b - 127) <= mmax 2^emax, the element
// format's maximum (mmax in [0.5, 1)); 127 for an all-zero group.
__device__ __forceinline__ int fit_scale_byte(float amax, float mmax, int emax) {
  if (!(amax > 0.0f)) return 127;
  int e;
  const float m = frexpf(amax, &e);  // amax = m 2^e, m in [0.5, 1)
  const int k = m <= mmax ? e - emax : e - emax + 1;
  return min(max(k + 127, 0), 254);
}
// E4M3FN: maximum 448 = 0.875 2^9
__device__ __forceinline__ int split_scale_byte(float amax) { return fit_scale_byte(amax, 0.875f, 9); }

// Four lanes per 32-element group, eight elements each: hi/lo E4M3FN codes and
// their scales.  A wave loads 1 KB of contiguous bf16 per instruction and
// stores 512 contiguous bytes of codes; the group maxima are combined over the
// lane quad with DPP.  (One lane per group loaded 64 B strides per instruction.)
__device__ __forceinline__ float quad_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true)));
  return fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xf, 0xf, true)));
}
// The FP8 hi/lo split of one 32-element scale group held 8 per lane by four
// lanes: v holds this lane's elements (hi and lo codes of v[4 j .. 4 j + 3] go
// to ch[j] / cl[j]); gmax(a) is the maximum of a over the group's four lanes.
// The scaled converts divide by (down) and multiply by (up) the f32 scale
// operand, of which only the exponent field counts: the E8M0 byte b shifted
// into that field stands for 2^(b - 127), also for b = 0.  Codes and residuals
// are those of ldexp by 127 - b and the unscaled converts (checked on the
// device for every byte class, FP8 subnormals and ties).
template <typename GroupMax>
__device__ __forceinline__ void fp8_split_lane8(float v[8], GroupMax gmax, uint32_t ch[2],
                                                uint32_t cl[2], int &bh, int &bl) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
  bh = split_scale_byte(gmax(amax));
  const float sh = __uint_as_float((uint32_t)bh << 23);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    s16x2 w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(s16x2{0, 0}, v[4 * j], v[4 * j + 1], sh, false);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(w, v[4 * j + 2], v[4 * j + 3], sh, true);
    ch[j] = __builtin_bit_cast(uint32_t, w);
    // residuals, exact in f32
    v[4 * j] -= __builtin_amdgcn_cvt_scalef32_f32_fp8(ch[j], sh, 0);
    v[4 * j + 1] -= __builtin_amdgcn_cvt_scalef32_f32_fp8(ch[j], sh, 1);
    v[4 * j + 2] -= __builtin_amdgcn_cvt_scalef32_f32_fp8(ch[j], sh, 2);
    v[4 * j + 3] -= __builtin_amdgcn_cvt_scalef32_f32_fp8(ch[j], sh, 3);
  }
  float ramax = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) ramax = fmaxf(ramax, fabsf(v[j]));
  bl = split_scale_byte(gmax(ramax));
  const float sl = __uint_as_float((uint32_t)bl << 23);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    s16x2 w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(s16x2{0, 0}, v[4 * j], v[4 * j + 1], sl, false);
    w = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(w, v[4 * j + 2], v[4 * j + 3], sl, true);
    cl[j] = __builtin_bit_cast(uint32_t, w);
  }
}

// Maximum over the four lanes l, l ^ 16, l ^ 32, l ^ 48: gfx950's row swaps
// (one VALU instruction each, no LDS round trip).
__device__ __forceinline__ float quad_row_max(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
  const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(t[0]), __uint_as_float(t[1]));
}

// The split of one 32-element scale group held 8 per lane by the four lanes
// q = 0..3 of a lane row (lanes r, r + 16, r + 32, r + 48); v holds this
// lane's elements 16 i + 4 q + m at v[4 i + m].  The arithmetic of
// act_split_kernel: ch[i] / cl[i] are the hi / lo codes of elements
// 16 i + 4 q .. + 3, bh / bl the group's scale bytes.
__device__ __forceinline__ void split_group_part(float v[8], uint32_t ch[2], uint32_t cl[2],
                                                 int *bh_out, int *bl_out) {
  fp8_split_lane8(v, [](float m) { return quad_row_max(m); }, ch, cl, *bh_out, *bl_out);
}

struct SplitArgs {
  const uint8_t *xhi, *xlo;    // activation codes (SplitLayout)
  const uint8_t *xshi, *xslo;  // activation scales [rows][K/32]
  uint32_t split_bytes;        // the split buffer starting at xhi (SplitLayout)
  const int32_t *act_index;    // sorted position -> activation row (nullptr: the position)
  const int4 *tiles;           // {expert, first sorted position, rows, 0}
  const int32_t *num_tiles;    // device-side count, read once and clamped to max_tiles
  int max_tiles;               // entries of `tiles` (the grid is sized for them)
  const uint8_t *w[2];         // stacked MXFP4 weights [E][N][K/2] per projection
  const uint8_t *s[2];         // stacked E8M0 scales [E][N][K/32]
  long long w_stride, s_stride;
  int N, K;
  int feature_tiles;
  uint16_t *out;               // bf16 [rows][N]
  float limit;
  // gate/up, ACT_FP8X2: when set, the epilogue writes the FP8 hi/lo split of
  // h (the down GEMM's input, SplitLayout(out_rows, N)) instead of h itself
  uint8_t *out_split;
  long long out_rows;
};

static inline void set_split(SplitArgs &a, const void *split, long long rows, int K, int af) {
  const SplitLayout L(rows, K, af);
  const uint8_t *base = static_cast<const uint8_t *>(split);
  a.split_bytes = (uint32_t)L.total;
  a.xhi = base;
  a.xlo = base + L.lo;
  a.xshi = base + L.shi;
  a.xslo = af == ACT_FP4 ? base + L.shi : base + L.slo;
}

}  // namespace glm
