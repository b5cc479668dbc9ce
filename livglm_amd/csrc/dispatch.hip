// Token-to-expert dispatch: histogram -> exclusive prefix sum -> stable permute.
//
// The reference materialises routes on the host once per layer (unique +
// compact remap, native_expert_ssd.py:475-525; expert_ssd.py:159-169).  Here
// the grouping stays on the device: pairs p = t*k + j are counting-sorted by
// expert id, ties kept in ascending p, so each expert's rows are contiguous
// for the expert kernels.
#include <algorithm>

#include "glm_common.h"

namespace glm {

constexpr int kDispatchThreads = 1024;

// Exclusive scan of one value per thread over a 1024-thread block.  Returns
// the exclusive prefix; *total receives the block sum.
__device__ __forceinline__ int block_exclusive_scan(int v, int *s_wave, int *total) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  if (wave == 0) {
    int w = lane < kDispatchThreads / 64 ? s_wave[lane] : 0;
    int wi = w;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(wi, off, 64);
      if (lane >= off) wi += o;
    }
    if (lane < kDispatchThreads / 64) s_wave[lane] = wi - w;  // exclusive wave base
    if (lane == kDispatchThreads / 64 - 1) s_wave[kDispatchThreads / 64] = wi;
  }
  __syncthreads();
  const int base = s_wave[wave];
  *total = s_wave[kDispatchThreads / 64];
  __syncthreads();
  return base + incl - v;
}

// Row tiles of the grouped GEMMs: an expert's c rows go to
// nt = ceil(c / tile_rows) tiles (tile_rows a multiple of 16), its 16-row
// blocks dealt out evenly, so every tile but the last is a whole number of
// blocks and none exceeds tile_rows (ceil(c / 16) <= nt * tile_rows / 16).
// Tile i is {first row within the expert, rows}.
__device__ __forceinline__ int row_tiles(int c, int tile_rows) {
  return (c + tile_rows - 1) / tile_rows;
}
__device__ __forceinline__ int2 row_tile(int c, int nt, int i) {
  const long long blocks = (c + 15) / 16;
  const int r0 = 16 * (int)(i * blocks / nt);
  const int r1 = min(16 * (int)((i + 1) * blocks / nt), c);
  return make_int2(r0, r1 - r0);
}

constexpr int kDispatchWaves = kDispatchThreads / 64;
constexpr int kMaxDispatchE = 448;
// Pairs of the single-workgroup dispatch, four to a thread.
constexpr int kSinglePairs = 4096;

// Lanes of the wave that hold this lane's key (at most E): one ballot per bit.
__device__ __forceinline__ uint64_t same_key_lanes(uint32_t key, int E) {
  const int nbits = 32 - __clz(E);
  uint64_t same = ~0ull;
  for (int bit = 0; bit < nbits; ++bit) {
    const uint64_t m = __ballot((key >> bit) & 1u);
    same &= ((key >> bit) & 1u) ? m : ~m;
  }
  return same;
}
__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Single workgroup, P <= kSinglePairs, E <= kMaxDispatchE.  A pair's place is
// its expert's offset + that expert's pairs in earlier groups of 64 pairs (one
// wave's turn each) + its rank among the lanes of its own turn (as
// dispatch_rank_kernel).  A chain of latencies: the indices, one LDS pass over
// the turns' counts by a thread an expert, one scan.  LDS: counts, then
// prefixes, [turns][E].  The layer at 2,664
// pairs and 128 experts takes 157.9 us instead of 178.5 (a chunk of 1,024
// pairs at a time through bitmaps in LDS: 29.4 us for this kernel alone).
__global__ __launch_bounds__(kDispatchThreads) void dispatch_kernel(
    const uint32_t *__restrict__ idx, int P, int k, int E, int32_t *__restrict__ counts,
    int32_t *__restrict__ offsets, int32_t *__restrict__ perm, int32_t *__restrict__ inv,
    int32_t *__restrict__ pair_token, int32_t *__restrict__ active,
    int32_t *__restrict__ num_active, int4 *__restrict__ work, int32_t *__restrict__ status,
    int tile_rows, int4 *__restrict__ tiles, int32_t *__restrict__ num_tiles) {
  extern __shared__ uint32_t smem[];
  uint16_t *turn = reinterpret_cast<uint16_t *>(smem);  // [turns][E]
  __shared__ int s_scan[kDispatchWaves + 1];
  __shared__ int32_t s_off[kMaxDispatchE];
  __shared__ int s_bad;
  constexpr int kPer = kSinglePairs / kDispatchThreads;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int turns = (P + 63) / 64;
  uint32_t key[kPer];  // E stands for "no pair" (past the end, or an index >= E, dropped)
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int p = u * kDispatchThreads + tid;
    key[u] = p < P ? idx[p] : (uint32_t)E;
  }
  for (int i = tid; i < (turns * E + 1) / 2; i += kDispatchThreads) smem[i] = 0;
  if (tid == 0) s_bad = 0;
  __syncthreads();
  int below[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (u * kDispatchThreads >= P) break;  // uniform
    if (key[u] >= (uint32_t)E) {
      if (u * kDispatchThreads + tid < P) s_bad = 1;
      key[u] = E;
    }
    const uint64_t same = same_key_lanes(key[u], E);
    below[u] = lanes_below(same);
    if (key[u] < (uint32_t)E && below[u] == 0)
      turn[(u * kDispatchWaves + wave) * E + key[u]] = (uint16_t)__popcll(same);
  }
  __syncthreads();
  // expert tid: exclusive prefix over the turns, its total
  int total = 0;
  if (tid < E) {
    for (int w0 = 0; w0 < turns; w0 += 8) {
      int n[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) n[j] = w0 + j < turns ? turn[(w0 + j) * E + tid] : 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (w0 + j < turns) turn[(w0 + j) * E + tid] = (uint16_t)total;
        total += n[j];
      }
    }
  }
  // one scan for the pairs (at most 2^12), the active experts (448) and the
  // row tiles (2^12 / 16 + 448), packed from bit 0, 13 and 22
  const int nt = tiles != nullptr && tid < E ? row_tiles(total, tile_rows) : 0;
  int all = 0;
  const uint32_t ex = (uint32_t)block_exclusive_scan(
      (int)((uint32_t)total | (total > 0 ? 1u << 13 : 0u) | (uint32_t)nt << 22), s_scan, &all);
  const int off = ex & 0x1fff, ex_a = (ex >> 13) & 0x1ff, ex_t = ex >> 22;
  const int pairs = all & 0x1fff, tot_a = ((uint32_t)all >> 13) & 0x1ff;
  if (tid < E) {
    s_off[tid] = off;
    offsets[tid] = off;
    counts[tid] = total;
    if (total > 0) {
      active[ex_a] = tid;
      work[ex_a] = make_int4(tid, off, total, 0);
    }
    for (int i = 0; i < nt; ++i) {
      const int2 t = row_tile(total, nt, i);
      tiles[ex_t + i] = make_int4(tid, off + t.x, t.y, 0);
    }
  }
  if (tid == 0) {
    offsets[E] = pairs;
    num_active[0] = tot_a;
    status[0] = s_bad;
    if (num_tiles != nullptr) num_tiles[0] = (int)((uint32_t)all >> 22);
  }
  for (int x = tot_a + tid; x < E; x += kDispatchThreads) {
    active[x] = -1;
    work[x] = make_int4(-1, 0, 0, 0);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    const int p = u * kDispatchThreads + tid;
    if (p >= P) break;
    if (key[u] < (uint32_t)E) {
      const int pos = s_off[key[u]] + turn[(u * kDispatchWaves + wave) * E + key[u]] + below[u];
      perm[pos] = p;
      inv[p] = pos;
      pair_token[pos] = p / k;
    } else {
      inv[p] = -1;
    }
  }
  // positions past the valid pairs (dropped indices >= E) hold -1
  for (int pos = pairs + tid; pos < P; pos += kDispatchThreads) {
    perm[pos] = -1;
    pair_token[pos] = -1;
  }
}

// ---------------------------------------------------------------------------
// Multi-workgroup dispatch for many pairs: the pairs are cut into chunks of
// 1024 (one workgroup each), in two kernels that run on every chunk at once.
// (1) dispatch_rank_kernel: every chunk ranks its pairs stably within the
// chunk -- lanes of a wave with the same expert are found with one ballot per
// bit of the expert id, a pair's rank is the number of such lanes below it
// plus the same expert's pairs in the chunk's earlier waves (per-wave counts
// in LDS) -- and writes its expert counts.  (2) dispatch_place_kernel: every
// chunk sums the chunk counts itself (expert totals and the counts of the
// chunks before it), scans the totals into expert offsets and places its
// pairs at offset + earlier chunks + rank; chunk 0 also writes the offsets,
// counts, work list and row tiles.  The result is identical to the
// single-workgroup dispatch.
// ---------------------------------------------------------------------------
// LDS: per-wave expert counts [kDispatchWaves][E] (E <= 448).
__global__ __launch_bounds__(kDispatchThreads) void dispatch_rank_kernel(
    const uint32_t *__restrict__ idx, int P, int E, int32_t *__restrict__ chunk_counts,
    int32_t *__restrict__ local_rank) {
  extern __shared__ int32_t wcnt[];  // [kDispatchWaves][E]
  __shared__ int s_bad;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < kDispatchWaves * E; i += kDispatchThreads) wcnt[i] = 0;
  if (tid == 0) s_bad = 0;
  const int p = blockIdx.x * kDispatchThreads + tid;
  const uint32_t e = p < P ? idx[p] : (uint32_t)E;
  // key E stands for "no pair" (past the end, or an index >= E, which is dropped)
  const uint32_t key = e < (uint32_t)E ? e : (uint32_t)E;
  __syncthreads();
  if (p < P && e >= (uint32_t)E) s_bad = 1;
  const uint64_t same = same_key_lanes(key, E);
  const int below = lanes_below(same);
  if (key < (uint32_t)E && below == 0) wcnt[wave * E + key] = __popcll(same);
  __syncthreads();
  // per expert: exclusive prefix over the waves; the chunk's count
  for (int x = tid; x < E; x += kDispatchThreads) {
    int run = 0;
#pragma unroll
    for (int w = 0; w < kDispatchWaves; ++w) {
      const int c = wcnt[w * E + x];
      wcnt[w * E + x] = run;
      run += c;
    }
    chunk_counts[(size_t)blockIdx.x * (E + 1) + x] = run;
  }
  __syncthreads();
  if (tid == 0) chunk_counts[(size_t)blockIdx.x * (E + 1) + E] = s_bad;
  if (p < P) local_rank[p] = key < (uint32_t)E ? wcnt[wave * E + key] + below : -1;
}

// rank_inv: in, the chunk-local ranks of dispatch_rank_kernel; out, inv.
// pair_token may be null (then the caller fills it from perm).
__global__ __launch_bounds__(kDispatchThreads) void dispatch_place_kernel(
    const uint32_t *__restrict__ idx, int P, int k, int E,
    const int32_t *__restrict__ chunk_counts, int nchunks, int32_t *__restrict__ rank_inv,
    int32_t *__restrict__ perm, int32_t *__restrict__ pair_token, int32_t *__restrict__ counts,
    int32_t *__restrict__ offsets, int32_t *__restrict__ active, int32_t *__restrict__ num_active,
    int4 *__restrict__ work, int32_t *__restrict__ status, int tile_rows,
    int4 *__restrict__ tiles, int32_t *__restrict__ num_tiles) {
  __shared__ int32_t base[kMaxDispatchE];
  __shared__ int s_scan[kDispatchThreads / 64 + 1];
  const int tid = threadIdx.x;
  const int chunk = blockIdx.x;
  // expert tid: its total over all chunks and its pairs in the chunks before
  // this one (16 chunks' loads issued together)
  int total = 0, before = 0;
  if (tid < E) {
    for (int c0 = 0; c0 < nchunks; c0 += 16) {
      int n[16];
#pragma unroll
      for (int j = 0; j < 16; ++j)
        n[j] = c0 + j < nchunks ? chunk_counts[(size_t)(c0 + j) * (E + 1) + tid] : 0;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        total += n[j];
        before += c0 + j < chunk ? n[j] : 0;
      }
    }
  }
  int all = 0;
  const int off = block_exclusive_scan(tid < E ? total : 0, s_scan, &all);
  if (tid < E) base[tid] = off + before;
  __syncthreads();
  const int p = chunk * kDispatchThreads + tid;
  if (p < P) {
    const uint32_t e = idx[p];
    const int r = rank_inv[p];
    if (e < (uint32_t)E && r >= 0) {
      const int pos = base[e] + r;
      perm[pos] = p;
      rank_inv[p] = pos;
      if (pair_token != nullptr) pair_token[pos] = p / k;
    } else {
      rank_inv[p] = -1;
    }
  }
  if (chunk != 0) return;
  // chunk 0: offsets, counts, the work list of active experts, row tiles
  int tot_a = 0;
  const int ex_a = block_exclusive_scan(tid < E && total > 0 ? 1 : 0, s_scan, &tot_a);
  const int nt = tiles != nullptr && tid < E ? row_tiles(total, tile_rows) : 0;
  int tot_t = 0;
  const int ex_t = block_exclusive_scan(nt, s_scan, &tot_t);
  if (tid < E) {
    offsets[tid] = off;
    counts[tid] = total;
    if (total > 0) {
      active[ex_a] = tid;
      work[ex_a] = make_int4(tid, off, total, 0);
    }
    for (int i = 0; i < nt; ++i) {
      const int2 t = row_tile(total, nt, i);
      tiles[ex_t + i] = make_int4(tid, off + t.x, t.y, 0);
    }
  }
  for (int x = tot_a + tid; x < E; x += kDispatchThreads) {
    active[x] = -1;
    work[x] = make_int4(-1, 0, 0, 0);
  }
  // positions past the valid pairs (dropped indices >= E) hold -1
  for (int pos = all + tid; pos < P; pos += kDispatchThreads) {
    perm[pos] = -1;
    if (pair_token != nullptr) pair_token[pos] = -1;
  }
  int bad = 0;
  for (int c = tid; c < nchunks; c += kDispatchThreads) bad |= chunk_counts[(size_t)c * (E + 1) + E];
  bad = __syncthreads_or(bad);
  if (tid == 0) {
    offsets[E] = all;
    num_active[0] = tot_a;
    status[0] = bad ? 1 : 0;
    if (num_tiles != nullptr) num_tiles[0] = tot_t;
  }
}

// pair_token from perm once the scatter is done (the public dispatch keeps
// the chunk counts in pair_token until then); positions past the valid pairs
// hold -1 in both.
__global__ void dispatch_tokens_kernel(const int32_t *__restrict__ offsets, int E, int P, int k,
                                       int32_t *__restrict__ perm,
                                       int32_t *__restrict__ pair_token) {
  const int total = offsets[E];
  for (int pos = blockIdx.x * blockDim.x + threadIdx.x; pos < P; pos += gridDim.x * blockDim.x) {
    if (pos < total) {
      pair_token[pos] = perm[pos] / k;
    } else {
      perm[pos] = -1;
      pair_token[pos] = -1;
    }
  }
}

// Row tiles of the grouped GEMMs from a work list (one workgroup): slot u of
// {expert, first position, rows, 0} gives row_tiles(rows, tile_rows) tiles.
__global__ __launch_bounds__(kDispatchThreads) void tiles_from_work_kernel(
    const int4 *__restrict__ work, int E, int tile_rows, int4 *__restrict__ tiles,
    int32_t *__restrict__ num_tiles) {
  __shared__ int s_scan[kDispatchThreads / 64 + 1];
  const int tid = threadIdx.x;
  int carry = 0;
  for (int u0 = 0; u0 < E; u0 += kDispatchThreads) {
    const int u = u0 + tid;
    const int4 wk = u < E ? work[u] : make_int4(-1, 0, 0, 0);
    const int n = wk.x >= 0 ? wk.z : 0;
    const int nt = row_tiles(n, tile_rows);
    int tot = 0;
    const int ex = block_exclusive_scan(nt, s_scan, &tot);
    for (int i = 0; i < nt; ++i) {
      const int2 t = row_tile(n, nt, i);
      tiles[carry + ex + i] = make_int4(wk.x, wk.y + t.x, t.y, 0);
    }
    carry += tot;
  }
  if (tid == 0) num_tiles[0] = carry;
}

}  // namespace glm

int glm_grouped_tile_rows();

extern "C" int glm_moe_tiles(void *stream, const int32_t *work, int E, int32_t *tiles,
                             int32_t *num_tiles) {
  glm::clear_error();
  GLM_REQUIRE(work && tiles && num_tiles, GLM_ERR_INVALID_ARGUMENT, "moe_tiles: null pointer");
  GLM_REQUIRE(E >= 1, GLM_ERR_INVALID_ARGUMENT, "moe_tiles: invalid E=%d", E);
  GLM_REQUIRE(glm_aligned16({work, tiles}), GLM_ERR_INVALID_ARGUMENT,
              "moe_tiles: work and tiles must be 16-byte aligned");
  hipLaunchKernelGGL(glm::tiles_from_work_kernel, dim3(1), dim3(glm::kDispatchThreads), 0,
                     (hipStream_t)stream, reinterpret_cast<const int4 *>(work), E,
                     glm_grouped_tile_rows(), reinterpret_cast<int4 *>(tiles), num_tiles);
  GLM_LAUNCH_CHECK("tiles_from_work_kernel");
  return GLM_OK;
}

// LDS of the single-workgroup dispatch: a 16-bit count per turn and expert.
static size_t dispatch_lds_bytes(int P, int E) {
  return ((size_t)((P + 63) / 64) * E + 1) / 2 * sizeof(uint32_t);
}

// Pairs above which the dispatch runs on many workgroups (it then needs
// glm_dispatch_chunk_ints(P, E) ints of scratch).
constexpr int kMultiDispatchPairs = glm::kSinglePairs;
size_t glm_dispatch_chunk_ints(long long P, int E) {
  return P > kMultiDispatchPairs
             ? (size_t)((P + glm::kDispatchThreads - 1) / glm::kDispatchThreads) * (E + 1)
             : 0;
}

// tiles/num_tiles (optional): row tiles of tile_rows rows for the grouped
// GEMMs; tiles needs room for ceil(T*k / tile_rows) + E entries.
// chunk_scratch: glm_dispatch_chunk_ints(P, E) ints for the multi-workgroup
// dispatch; without it (the public entry point) the chunk counts live in
// pair_token -- ceil(P / 1024) * (E + 1) <= P ints for E <= 448 and P > 4096
// -- and pair_token is filled from perm at the end.
int glm_dispatch_launch(hipStream_t stream, const uint32_t *indices, int T, int k, int E,
                        int32_t *counts, int32_t *offsets, int32_t *perm, int32_t *inv,
                        int32_t *pair_token, int32_t *active, int32_t *num_active, int4 *work,
                        int32_t *status, int tile_rows, int4 *tiles, int32_t *num_tiles,
                        int32_t *chunk_scratch) {
  const int P = T * k;
  if (P > kMultiDispatchPairs) {
    const int nchunks = (P + glm::kDispatchThreads - 1) / glm::kDispatchThreads;
    const bool in_place = chunk_scratch == nullptr;
    if (in_place) {
      GLM_REQUIRE((size_t)nchunks * (E + 1) <= (size_t)P, GLM_ERR_UNSUPPORTED_SHAPE,
                  "dispatch: %d chunks x %d experts do not fit in pair_token", nchunks, E + 1);
      chunk_scratch = pair_token;
    }
    // the chunk-local ranks go through inv, which the second kernel overwrites
    hipLaunchKernelGGL(glm::dispatch_rank_kernel, dim3(nchunks), dim3(glm::kDispatchThreads),
                       (size_t)glm::kDispatchWaves * E * 4, stream, indices, P, E, chunk_scratch,
                       inv);
    GLM_LAUNCH_CHECK("dispatch_rank_kernel");
    hipLaunchKernelGGL(glm::dispatch_place_kernel, dim3(nchunks), dim3(glm::kDispatchThreads), 0,
                       stream, indices, P, k, E, chunk_scratch, nchunks, inv, perm,
                       in_place ? nullptr : pair_token, counts, offsets, active, num_active, work,
                       status, tile_rows, tiles, num_tiles);
    GLM_LAUNCH_CHECK("dispatch_place_kernel");
    if (in_place) {
      const int blocks = std::min((P + 255) / 256, 1024);
      hipLaunchKernelGGL(glm::dispatch_tokens_kernel, dim3(blocks), dim3(256), 0, stream, offsets,
                         E, P, k, perm, pair_token);
      GLM_LAUNCH_CHECK("dispatch_tokens_kernel");
    }
    return GLM_OK;
  }
  hipLaunchKernelGGL(glm::dispatch_kernel, dim3(1), dim3(glm::kDispatchThreads),
                     dispatch_lds_bytes(P, E), stream, indices, P, k, E, counts, offsets, perm,
                     inv, pair_token, active, num_active, work, status, tile_rows, tiles,
                     num_tiles);
  GLM_LAUNCH_CHECK("dispatch_kernel");
  return GLM_OK;
}

extern "C" int glm_moe_dispatch(void *stream, const uint32_t *indices, int T, int top_k, int E,
                                int32_t *counts, int32_t *offsets, int32_t *perm, int32_t *inv,
                                int32_t *pair_token, int32_t *active, int32_t *num_active,
                                int32_t *work, int32_t *status) {
  glm::clear_error();
  GLM_REQUIRE(indices && counts && offsets && perm && inv && pair_token && active &&
                  num_active && work && status,
              GLM_ERR_INVALID_ARGUMENT, "dispatch: null pointer argument");
  GLM_REQUIRE(T >= 0 && top_k >= 1 && E >= 1, GLM_ERR_INVALID_ARGUMENT,
              "dispatch: invalid sizes T=%d k=%d E=%d", T, top_k, E);
  GLM_REQUIRE(E <= 448, GLM_ERR_UNSUPPORTED_SHAPE, "dispatch: E=%d exceeds 448", E);
  GLM_REQUIRE((long long)T * top_k < (1LL << 30), GLM_ERR_UNSUPPORTED_SHAPE,
              "dispatch: too many pairs");
  GLM_REQUIRE(glm_aligned16({work}), GLM_ERR_INVALID_ARGUMENT,
              "dispatch: work must be 16-byte aligned");
  return glm_dispatch_launch((hipStream_t)stream, indices, T, top_k, E, counts, offsets, perm,
                             inv, pair_token, active, num_active, (int4 *)work, status, 0,
                             nullptr, nullptr, nullptr);
}
