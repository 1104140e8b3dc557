// Block selection: equal-budget top-k per query tile, the block mask, and
// the full / partial key-tile lists the attention kernel walks.
//
// Top-k: one wave per (head, query tile). Scores become 64-bit keys
// (orderable fp32 score << 32 | ~column); lane l holds the keys of columns
// l, l + 64, .., sorts them in registers (a bitonic network over N = 16 or
// 32 keys, zeros padding the list) and keeps them in LDS in that order,
// lane-strided so every LDS access is conflict-free. k_hi rounds of a
// wave-wide max over the lanes' current heads extract the winners in
// descending order; the winning lane's next head is one LDS read. The
// rounds are what the kernel spends its time on, so the LDS holds only the
// row's columns (dynamic size, 20 KB per workgroup at 592 columns: 8
// workgroups per CU instead of the 2 a 2048-column array allows), and a
// round takes the max of the 32-bit score keys alone (about a third of the
// instructions of a max over the 64-bit keys); only when several lanes hold
// the same score does a second max pick the lowest column (48 heads x 592
// columns, k_hi 35: 112 -> 79 us; x 1,632, k_hi 48: 842 -> 750, most of it
// the sort of 32 keys).
// The order is total: higher score first, lower column first on equal
// scores.
//
// Lists: one wave per (head, row), 64 columns per step, positions from a
// ballot + popcount prefix (no sort, no atomics).

#include <type_traits>

#include "veda_common.h"

namespace veda {
namespace {

// Order key of a score: unsigned order of keys = numeric order of scores,
// with every NaN (either sign) one key above +inf, as torch.sort / topk rank
// NaN above every number (so NaNs tie among themselves and fall back to
// column order).
constexpr uint32_t kNaNKey = 0xffffffffu;
constexpr uint32_t kNegInfKey = 0x007fffffu;  // orderable(-inf)

__device__ __forceinline__ uint32_t orderable(float v) {
  if (v != v) return kNaNKey;
  if (v == 0.f) v = 0.f;  // -0 ties with +0, as in a float comparison
  uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Max over the 64 lanes of a 32-bit key, wave-uniform. Within a 16-lane row:
// DPP exchanges with lane ^ 1, lane ^ 2, the mirror inside 8 and the mirror
// inside 16 (each folds into its v_max_u32); across rows: the row 16 lanes
// away, then the lane 32 positions away (the swaps leave {own, partner} in
// their two results, in either order).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xF, 0xF, false));   // quad_perm
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0u, v, 0x4E, 0xF, 0xF, false));   // quad_perm
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0u, v, 0x141, 0xF, 0xF, false));  // half mirror
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0u, v, 0x140, 0xF, 0xF, false));  // mirror
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)max(b[0], b[1]));
}

constexpr int kMaxCols = 2048;  // columns of one block (FA4's 2048-block cap)
constexpr int kSelWaves = 4;

// Sorts N keys descending (bitonic network, indices fixed at compile time,
// so the keys stay in registers).
template <int N>
__device__ __forceinline__ void sort_desc(uint64_t (&k)[N]) {
#pragma unroll
  for (int size = 2; size <= N; size <<= 1)
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1)
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int j = i ^ stride;
        if (j > i) {
          const uint64_t a = k[i], b = k[j];
          const bool sw = (i & size) == 0 ? a < b : a > b;
          k[i] = sw ? b : a;
          k[j] = sw ? a : b;
        }
      }
}

template <int N>  // keys per lane the registers hold (>= the row's columns / 64)
__global__ void __launch_bounds__(256) select_topk_kernel(
    const float* __restrict__ scores, int64_t n_heads, int64_t n_rows, int64_t ssh,
    int64_t ssr, int64_t block_start, int n_cols, const uint8_t* __restrict__ kv_ok,
    const int64_t* __restrict__ rows, int k_lo, int k_hi, const uint8_t* __restrict__ extra,
    int64_t n_extra, int64_t* __restrict__ index, uint8_t* __restrict__ keep, int64_t osh,
    int64_t osr, int64_t col0) {
  extern __shared__ uint64_t keys[];  // [kSelWaves][per_lane * 64]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * kSelWaves + wave;
  if (item >= n_heads * n_rows) return;  // whole wave exits together
  const int64_t h = item / n_rows, r = item % n_rows;
  const int64_t tile_id = rows != nullptr ? rows[r] : r;
  const int64_t diag = tile_id - block_start;  // column of the own tile, if in block
  const float* srow = scores + h * ssh + r * ssr + block_start;
  const int per_lane = (n_cols + 63) / 64;
  uint64_t* kv = keys + wave * per_lane * 64;
  uint64_t k[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int c = j * 64 + lane;
    uint64_t key = 0;  // absent column: below every real key
    if (j < per_lane && c < n_cols) {
      float v = srow[c];
      if (!kv_ok[block_start + c]) v = -INFINITY;
      if (c == diag) v = INFINITY;
      key = ((uint64_t)orderable(v) << 32) | (uint32_t)(~(uint32_t)c);
    }
    k[j] = key;
  }
  sort_desc(k);
#pragma unroll
  for (int j = 0; j < N; ++j)
    if (j < per_lane) kv[j * 64 + lane] = k[j];
  uint32_t best = (uint32_t)(k[0] >> 32);  // score key and column of this lane's head
  uint32_t col = ~(uint32_t)k[0];
  int pos = 0;  // index of this lane's current head in its sorted list
  const bool has_extra = tile_id >= 0 && tile_id < n_extra && extra[tile_id] != 0;
  const int allowed = k_lo + (has_extra ? 1 : 0);
  int64_t* irow = index + h * osh + r * osr + col0;
  uint8_t* krow = keep + h * osh + r * osr + col0;
  for (int t = 0; t < k_hi; ++t) {
    const uint32_t top = wave_max_u32(best);
    uint64_t at = __ballot(best == top);
    if (at & (at - 1)) {  // equal scores in several lanes: the lowest column (wave-uniform branch)
      const uint32_t c = wave_max_u32(best == top ? ~col : 0u);
      at = __ballot(best == top && ~col == c);
    }
    if (lane == __builtin_ctzll(at)) {
      irow[t] = block_start + (int64_t)col;
      // kept: within the row's budget and `val > -inf` (False for NaN,
      // mask.py:251-284)
      krow[t] = (t < allowed && top > kNegInfKey && top != kNaNKey) ? 1 : 0;
      ++pos;
      const uint64_t next = pos < per_lane ? kv[pos * 64 + lane] : 0;
      best = (uint32_t)(next >> 32);
      col = ~(uint32_t)next;
    }
  }
}

constexpr int kMaxTiles = 8192;

__global__ void __launch_bounds__(256) dense_mask_kernel(
    const int64_t* __restrict__ index, const uint8_t* __restrict__ keep, int64_t n_sel,
    int64_t k_total, const uint8_t* __restrict__ kv_ok, int n_tiles, int64_t n_video,
    int64_t out_rows, uint8_t* __restrict__ mask) {
  __shared__ uint8_t row[kMaxTiles];
  const int64_t h = blockIdx.x / out_rows, r = blockIdx.x % out_rows;
  const bool video_row = r < n_sel && r < n_video;
  for (int c = threadIdx.x; c < n_tiles; c += blockDim.x)
    row[c] = (!video_row || c >= n_video) ? kv_ok[c] : 0;
  __syncthreads();
  if (video_row) {
    const int64_t base = (h * n_sel + r) * k_total;
    for (int64_t t = threadIdx.x; t < k_total; t += blockDim.x) {
      const int64_t c = index[base + t];
      if (keep[base + t] && c >= 0 && c < n_tiles) row[c] = 1;
    }
  }
  __syncthreads();
  uint8_t* out = mask + (h * out_rows + r) * n_tiles;
  for (int c = threadIdx.x; c < n_tiles; c += blockDim.x) out[c] = row[c];
}

// Index lists: one wave per (head, row). The row's classes (0 outside the
// row's members, 1 full member, 2 partial member) are first staged in LDS
// with wide independent loads; the lists are then written 64 columns at a
// time, each lane storing its column once per list (members at their rank,
// non-members after all members), so every store instruction is whole.
// Rows longer than kListCols take the two-pass form from global memory.
constexpr int kListWaves = 4;
constexpr int kListCols = 4096;

template <int VEC>
__device__ __forceinline__ void stage_classes(const uint8_t* __restrict__ m,
                                              const uint8_t* __restrict__ kv_ok,
                                              const uint8_t* __restrict__ full_tile, int n_tiles,
                                              int lane, uint8_t* cls, int& counts) {
  using Vec = typename std::conditional<VEC == 16, uint4,
              typename std::conditional<VEC == 4, uint32_t, uint8_t>::type>::type;
  int nf = 0, np = 0;
#pragma unroll 4
  for (int c = lane * VEC; c < n_tiles; c += 64 * VEC) {
    union { Vec v; uint8_t b[VEC]; } mm, kk, ff, out;
    mm.v = *reinterpret_cast<const Vec*>(m + c);
    kk.v = *reinterpret_cast<const Vec*>(kv_ok + c);
    ff.v = *reinterpret_cast<const Vec*>(full_tile + c);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const bool member = mm.b[j] && kk.b[j];
      const bool full = ff.b[j] != 0;
      out.b[j] = member ? (full ? 1 : 2) : 0;
      nf += member && full;
      np += member && !full;
    }
    *reinterpret_cast<Vec*>(cls + c) = out.v;
  }
  counts = nf | (np << 16);  // both at most 4096
}

// The lists of one row whose classes are in `cls` (this wave's LDS row), NF
// full and NP partial members.
__device__ __forceinline__ void write_lists(const uint8_t* cls, int n_tiles, int lane, int NF,
                                            int NP, int32_t* __restrict__ fi,
                                            int32_t* __restrict__ pi) {
  const uint64_t below = (1ull << lane) - 1ull;
  int nf = 0, np = 0;  // members before the chunk
  for (int c0 = 0; c0 < n_tiles; c0 += 64) {
    const int c = c0 + lane;
    const int k = c < n_tiles ? cls[c] : 0;
    const uint64_t bf = __ballot(k == 1), bp = __ballot(k == 2);
    const int rf = __popcll(bf & below), rp = __popcll(bp & below);
    if (c < n_tiles) {
      fi[k == 1 ? nf + rf : NF + (c0 - nf) + (lane - rf)] = c;
      pi[k == 2 ? np + rp : NP + (c0 - np) + (lane - rp)] = c;
    }
    nf += __popcll(bf);
    np += __popcll(bp);
  }
}

// Orders this wave's LDS accesses before it against those after it.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// index_lists of dense_block_mask(selection) without the mask: one wave per
// (head, row of all n_tiles tiles). A video row's members are its kept
// columns and the global columns, a global row's every column, each where
// kv_ok. Against the two kernels it saves writing and reading the mask and a
// launch: 25 + 32 -> 35 us at 48 heads x 592 x 592, 95 + 284 -> 224 us at
// 1,648 x 1,648 (4.7 TB/s of list entries written).
__global__ void __launch_bounds__(64 * kListWaves) selection_lists_kernel(
    const int64_t* __restrict__ index, const uint8_t* __restrict__ keep, int64_t n_items,
    int64_t k_total, const uint8_t* __restrict__ kv_ok, const uint8_t* __restrict__ full_tile,
    int n_tiles, int n_video, int32_t* __restrict__ part_cnt, int32_t* __restrict__ part_idx,
    int32_t* __restrict__ full_cnt, int32_t* __restrict__ full_idx) {
  __shared__ __align__(16) uint8_t cls_lds[kListWaves][kListCols];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * kListWaves + wave;
  if (item >= n_items) return;  // each wave uses only its own LDS row
  const int64_t h = item / n_tiles, r = item % n_tiles;
  const bool video_row = r < n_video;
  uint8_t* cls = cls_lds[wave];
  for (int c = lane; c < n_tiles; c += 64)
    cls[c] = (!video_row || c >= n_video) && kv_ok[c] ? (full_tile[c] ? 1 : 2) : 0;
  if (video_row) {
    wave_lds_sync();
    const int64_t base = (h * n_video + r) * k_total;
    for (int64_t t = lane; t < k_total; t += 64) {
      const int64_t c = index[base + t];
      if (keep[base + t] && c >= 0 && c < n_tiles && kv_ok[c]) cls[c] = full_tile[c] ? 1 : 2;
    }
  }
  wave_lds_sync();
  int NF = 0, NP = 0;
  for (int c0 = 0; c0 < n_tiles; c0 += 64) {
    const int k = c0 + lane < n_tiles ? cls[c0 + lane] : 0;
    NF += __popcll(__ballot(k == 1));
    NP += __popcll(__ballot(k == 2));
  }
  write_lists(cls, n_tiles, lane, NF, NP, full_idx + item * n_tiles, part_idx + item * n_tiles);
  if (lane == 0) {
    full_cnt[item] = NF;
    part_cnt[item] = NP;
  }
}

// Transposed lists (row = key tile, entries = its query tiles; all members
// in the full or all in the partial list, by the key tile's own fullness).
// Workgroup = (head, 64 key tiles). The mask's 64 columns come in as one
// 64-bit word per query row (a ballot over one coalesced 64-byte read), a
// chunk of rows at a time in LDS; a ballot over 64 rows' words at one
// column's bit then is that column's membership, from which every store of
// a list row is 64 consecutive entries. One launch in place of a transposed
// copy, a list kernel and four selects: at 48 heads x 592 x 592 about 195 us
// in eight launches -> 64 us.
constexpr int kTransThreads = 512;
constexpr int kTransRows = 4096;  // rows staged at a time

__global__ void __launch_bounds__(kTransThreads) index_lists_t_kernel(
    const uint8_t* __restrict__ mask, int n_rows, int n_cols, const uint8_t* __restrict__ kv_ok,
    const uint8_t* __restrict__ full_tile, int32_t* __restrict__ part_cnt,
    int32_t* __restrict__ part_idx, int32_t* __restrict__ full_cnt,
    int32_t* __restrict__ full_idx) {
  __shared__ uint64_t words[kTransRows];
  constexpr int kWaves = kTransThreads / 64, kColsPerWave = 64 / kWaves;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int groups = (n_cols + 63) / 64;
  const int64_t h = blockIdx.x / groups;
  const int c0 = (int)(blockIdx.x % groups) * 64;
  const int c = c0 + lane;
  const bool col_ok = c < n_cols && kv_ok[c];
  const uint8_t* m = mask + h * n_rows * n_cols + c;
  const int chunks = (n_rows + kTransRows - 1) / kTransRows;
  // the words of rows [r0, r0 + kTransRows) (zero past the last row)
  auto stage = [&](int r0) {
    const int end = min(n_rows - r0, kTransRows), padded = (end + 63) & ~63;
#pragma unroll 8
    for (int r = wave; r < padded; r += kWaves) {
      const bool in = r < end && col_ok && m[(int64_t)(r0 + r) * n_cols] != 0;
      const uint64_t w = __ballot(in);
      if (lane == 0) words[r] = w;
    }
    __syncthreads();
  };
  int total[kColsPerWave];
#pragma unroll
  for (int i = 0; i < kColsPerWave; ++i) total[i] = 0;
  for (int k = 0; k < chunks; ++k) {
    if (k > 0) __syncthreads();  // the previous chunk's words are read
    stage(k * kTransRows);
    for (int r = lane; r - lane < min(n_rows - k * kTransRows, kTransRows); r += 64) {
      const uint64_t w = words[r];
#pragma unroll
      for (int i = 0; i < kColsPerWave; ++i)
        total[i] += __popcll(__ballot((w >> (wave * kColsPerWave + i)) & 1));
    }
  }
  int seen[kColsPerWave];
#pragma unroll
  for (int i = 0; i < kColsPerWave; ++i) seen[i] = 0;
  const uint64_t below = (1ull << lane) - 1ull;
  for (int k = 0; k < chunks; ++k) {
    if (chunks > 1) {
      __syncthreads();
      stage(k * kTransRows);
    }
    const int r0 = k * kTransRows;
    for (int r = lane; r - lane < min(n_rows - r0, kTransRows); r += 64) {
      const uint64_t w = words[r];
      const int at = r0 + r;
#pragma unroll
      for (int i = 0; i < kColsPerWave; ++i) {
        const int col = c0 + wave * kColsPerWave + i;  // wave-uniform
        if (col >= n_cols) break;
        const bool in = (w >> (wave * kColsPerWave + i)) & 1;
        const uint64_t b = __ballot(in);
        const int64_t row = (h * n_cols + col) * n_rows;
        const bool full = full_tile[col] != 0;
        int32_t* list = (full ? full_idx : part_idx) + row;
        int32_t* other = (full ? part_idx : full_idx) + row;
        if (at < n_rows) {
          const int before = seen[i] + __popcll(b & below);  // members before this row
          list[in ? before : total[i] + at - before] = at;
          other[at] = at;
        }
        seen[i] += __popcll(b);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kColsPerWave; ++i) {
    const int col = c0 + wave * kColsPerWave + i;
    if (col < n_cols && lane == 0) {
      const bool full = full_tile[col] != 0;
      full_cnt[h * n_cols + col] = full ? total[i] : 0;
      part_cnt[h * n_cols + col] = full ? 0 : total[i];
    }
  }
}

__global__ void __launch_bounds__(64 * kListWaves) index_lists_kernel(
    const uint8_t* __restrict__ mask, int64_t n_items, int n_tiles, int vec,
    const uint8_t* __restrict__ kv_ok, const uint8_t* __restrict__ full_tile,
    int32_t* __restrict__ part_cnt, int32_t* __restrict__ part_idx,
    int32_t* __restrict__ full_cnt, int32_t* __restrict__ full_idx) {
  __shared__ __align__(16) uint8_t cls_lds[kListWaves][kListCols];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t item = (int64_t)blockIdx.x * kListWaves + wave;
  if (item >= n_items) return;  // each wave uses only its own LDS row
  const uint8_t* m = mask + item * n_tiles;
  int32_t* fi = full_idx + item * n_tiles;
  int32_t* pi = part_idx + item * n_tiles;
  const uint64_t below = (1ull << lane) - 1ull;
  if (n_tiles <= kListCols) {
    uint8_t* cls = cls_lds[wave];
    int counts;
    if (vec == 16)
      stage_classes<16>(m, kv_ok, full_tile, n_tiles, lane, cls, counts);
    else if (vec == 4)
      stage_classes<4>(m, kv_ok, full_tile, n_tiles, lane, cls, counts);
    else
      stage_classes<1>(m, kv_ok, full_tile, n_tiles, lane, cls, counts);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) counts += __shfl_xor(counts, off);
    const int NF = counts & 0xffff, NP = counts >> 16;
    wave_lds_sync();  // the lanes' LDS stores are seen by the other lanes of this wave
    write_lists(cls, n_tiles, lane, NF, NP, fi, pi);
    if (lane == 0) {
      full_cnt[item] = NF;
      part_cnt[item] = NP;
    }
    return;
  }
  int nf = 0, np = 0;
  for (int c0 = 0; c0 < n_tiles; c0 += 64) {
    const int c = c0 + lane;
    bool f = false, p = false;
    if (c < n_tiles && m[c] && kv_ok[c]) {
      f = full_tile[c] != 0;
      p = !f;
    }
    const uint64_t bf = __ballot(f), bp = __ballot(p);
    if (f) fi[nf + __popcll(bf & below)] = c;
    if (p) pi[np + __popcll(bp & below)] = c;
    nf += __popcll(bf);
    np += __popcll(bp);
  }
  // Non-members follow, ascending (the stable argsort of ~member).
  int of = nf, op = np;
  for (int c0 = 0; c0 < n_tiles; c0 += 64) {
    const int c = c0 + lane;
    bool f = false, p = false;
    if (c < n_tiles) {
      const bool member = m[c] && kv_ok[c];
      const bool full = full_tile[c] != 0;
      f = !(member && full);
      p = !(member && !full);
    }
    const uint64_t bf = __ballot(f), bp = __ballot(p);
    if (f) fi[of + __popcll(bf & below)] = c;
    if (p) pi[op + __popcll(bp & below)] = c;
    of += __popcll(bf);
    op += __popcll(bp);
  }
  if (lane == 0) {
    full_cnt[item] = nf;
    part_cnt[item] = np;
  }
}

}  // namespace
}  // namespace veda

using namespace veda;

extern "C" int veda_select_topk(const float* scores, int64_t n_heads, int64_t n_rows,
                                int64_t s_stride_h, int64_t s_stride_r, int64_t block_start,
                                int64_t n_cols, const uint8_t* kv_ok, const int64_t* rows,
                                int64_t k_lo, int64_t k_hi, const uint8_t* extra,
                                int64_t n_extra, int64_t* index, uint8_t* keep,
                                int64_t o_stride_h, int64_t o_stride_r, int64_t col0,
                                void* stream) {
  VEDA_REQUIRE(n_cols >= 1 && n_cols <= kMaxCols, "select_topk: n_cols %lld not in [1, %d]",
               (long long)n_cols, kMaxCols);
  VEDA_REQUIRE(1 <= k_lo && k_lo <= k_hi && k_hi <= n_cols,
               "select_topk: need 1 <= k_lo <= k_hi <= n_cols, got %lld %lld %lld",
               (long long)k_lo, (long long)k_hi, (long long)n_cols);
  VEDA_REQUIRE(block_start >= 0 && n_heads >= 0 && n_rows >= 0, "select_topk: negative size");
  const int64_t items = n_heads * n_rows;
  if (items == 0) return VEDA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const size_t lds = (size_t)kSelWaves * ((n_cols + 63) / 64) * 64 * sizeof(uint64_t);  // <= 64 KB
  static_assert(32 * 64 >= kMaxCols, "select_topk_kernel<32> holds kMaxCols keys per wave");
  const unsigned grid = (unsigned)((items + kSelWaves - 1) / kSelWaves);
  if (n_cols <= 16 * 64)
    select_topk_kernel<16><<<grid, 256, lds, s>>>(
        scores, n_heads, n_rows, s_stride_h, s_stride_r, block_start, (int)n_cols, kv_ok, rows,
        (int)k_lo, (int)k_hi, extra, n_extra, index, keep, o_stride_h, o_stride_r, col0);
  else
    select_topk_kernel<32><<<grid, 256, lds, s>>>(
        scores, n_heads, n_rows, s_stride_h, s_stride_r, block_start, (int)n_cols, kv_ok, rows,
        (int)k_lo, (int)k_hi, extra, n_extra, index, keep, o_stride_h, o_stride_r, col0);
  return check_launch("veda_select_topk");
}

extern "C" int veda_dense_block_mask(const int64_t* index, const uint8_t* keep, int64_t n_heads,
                                     int64_t n_sel, int64_t k_total, const uint8_t* kv_ok,
                                     int64_t n_tiles, int64_t n_video, int global_rows,
                                     uint8_t* mask, void* stream) {
  VEDA_REQUIRE(n_tiles >= 1 && n_tiles <= kMaxTiles, "dense_block_mask: n_tiles %lld > %d",
               (long long)n_tiles, kMaxTiles);
  VEDA_REQUIRE(!global_rows || n_sel == n_video,
               "dense_block_mask: global_rows needs a selection of all video rows");
  const int64_t out_rows = global_rows ? n_tiles : n_sel;
  const int64_t blocks = n_heads * out_rows;
  if (blocks == 0) return VEDA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  dense_mask_kernel<<<(unsigned)blocks, 256, 0, s>>>(index, keep, n_sel, k_total, kv_ok,
                                                     (int)n_tiles, n_video, out_rows, mask);
  return check_launch("veda_dense_block_mask");
}

extern "C" int veda_index_lists(const uint8_t* block_mask, int64_t n_heads, int64_t n_rows,
                                int64_t n_tiles, const uint8_t* kv_ok, const uint8_t* full_tile,
                                int32_t* part_cnt, int32_t* part_idx, int32_t* full_cnt,
                                int32_t* full_idx, void* stream) {
  VEDA_REQUIRE(n_tiles >= 1 && n_tiles < (1ll << 31), "index_lists: bad n_tiles");
  const int64_t items = n_heads * n_rows;
  if (items == 0) return VEDA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  // widest load every row start and both column tables allow
  auto aligned = [&](int64_t a) {
    return n_tiles % a == 0 && reinterpret_cast<uintptr_t>(block_mask) % a == 0 &&
           reinterpret_cast<uintptr_t>(kv_ok) % a == 0 &&
           reinterpret_cast<uintptr_t>(full_tile) % a == 0;
  };
  const int vec = aligned(16) ? 16 : aligned(4) ? 4 : 1;
  index_lists_kernel<<<(unsigned)((items + kListWaves - 1) / kListWaves), 64 * kListWaves, 0,
                       s>>>(block_mask, items, (int)n_tiles, vec, kv_ok, full_tile, part_cnt,
                            part_idx, full_cnt, full_idx);
  return check_launch("veda_index_lists");
}

extern "C" int veda_selection_lists(const int64_t* index, const uint8_t* keep, int64_t n_heads,
                                    int64_t n_video, int64_t k_total, const uint8_t* kv_ok,
                                    const uint8_t* full_tile, int64_t n_tiles, int32_t* part_cnt,
                                    int32_t* part_idx, int32_t* full_cnt, int32_t* full_idx,
                                    void* stream) {
  VEDA_REQUIRE(n_tiles >= 1 && n_tiles <= kListCols, "selection_lists: n_tiles %lld not in [1, %d]",
               (long long)n_tiles, kListCols);
  VEDA_REQUIRE(n_video >= 0 && n_video <= n_tiles, "selection_lists: n_video %lld outside [0, %lld]",
               (long long)n_video, (long long)n_tiles);
  VEDA_REQUIRE(n_heads >= 0 && k_total >= 0, "selection_lists: negative size");
  const int64_t items = n_heads * n_tiles;
  if (items == 0) return VEDA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  selection_lists_kernel<<<(unsigned)((items + kListWaves - 1) / kListWaves), 64 * kListWaves, 0,
                           s>>>(index, keep, items, k_total, kv_ok, full_tile, (int)n_tiles,
                                (int)n_video, part_cnt, part_idx, full_cnt, full_idx);
  return check_launch("veda_selection_lists");
}

extern "C" int veda_index_lists_t(const uint8_t* block_mask, int64_t n_heads, int64_t n_rows,
                                  int64_t n_tiles, const uint8_t* kv_ok, const uint8_t* full_tile,
                                  int32_t* part_cnt, int32_t* part_idx, int32_t* full_cnt,
                                  int32_t* full_idx, void* stream) {
  VEDA_REQUIRE(n_tiles >= 1 && n_tiles < (1ll << 31) && n_rows >= 0 && n_rows < (1ll << 31) - 64 &&
                   n_heads >= 0,
               "index_lists_t: bad sizes");
  const int64_t groups = n_heads * ((n_tiles + 63) / 64);
  VEDA_REQUIRE(groups < (1ll << 31), "index_lists_t: too many heads x key tiles for one launch");
  if (groups == 0) return VEDA_OK;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  index_lists_t_kernel<<<(unsigned)groups, kTransThreads, 0, s>>>(
      block_mask, (int)n_rows, (int)n_tiles, kv_ok, full_tile, part_cnt, part_idx, full_cnt,
      full_idx);
  return check_launch("veda_index_lists_t");
}
