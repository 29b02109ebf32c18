// Library core: errors, device init, prefix sums, map transpose, device
// sparsity builder, pattern expansion, greedy colouring and row batching.
#include <algorithm>
#include <climits>
#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"

namespace op2hip {

static thread_local char g_error[1024];

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

// ---------------------------------------------------------------------------
// small utility kernels

__global__ void fill_i32(int32_t *p, int64_t n, int32_t v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

static int fill(int32_t *p, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return OP2HIP_OK;
  const uint32_t grid = std::min<uint32_t>(ceil_div(n, 256), 16384);
  fill_i32<<<grid, 256, 0, s>>>(p, n, v);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

// ---------------------------------------------------------------------------
// exclusive scan: tiles of kScanTile items, one 256-thread block per tile.

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ int64_t block_inclusive_scan(int64_t v, int64_t *lds) {
  const int t = threadIdx.x;
  lds[t] = v;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    const int64_t add = t >= off ? lds[t - off] : 0;
    __syncthreads();
    lds[t] += add;
    __syncthreads();
  }
  return lds[t];
}

// out[i+1] = tile-local inclusive prefix; tile_sums[b] = tile total.
__global__ void scan_tiles(int64_t n, const int32_t *__restrict__ in,
                           int32_t *__restrict__ out, int64_t *__restrict__ tile_sums) {
  __shared__ int64_t lds[kScanThreads];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
  int64_t v[kScanItems];
  int64_t run = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    run += (i < n) ? in[i] : 0;
    v[k] = run;
  }
  const int64_t incl = block_inclusive_scan(run, lds);
  const int64_t excl = incl - run;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k;
    if (i < n) out[i + 1] = static_cast<int32_t>(excl + v[k]);
  }
  if (threadIdx.x == kScanThreads - 1) tile_sums[blockIdx.x] = incl;
}

// Single block: exclusive scan of tile_sums in place, total to total[0] and
// *aside (if any) beside it.
__global__ void scan_tile_sums(int64_t ntiles, int64_t *__restrict__ tile_sums,
                               int64_t *__restrict__ total, const int32_t *__restrict__ aside) {
  __shared__ int64_t lds[kScanThreads];
  int64_t carry = 0;
  for (int64_t b = 0; b < ntiles; b += kScanThreads) {
    const int64_t i = b + threadIdx.x;
    const int64_t v = i < ntiles ? tile_sums[i] : 0;
    const int64_t incl = block_inclusive_scan(v, lds);
    if (i < ntiles) tile_sums[i] = carry + incl - v;
    __syncthreads();
    carry += lds[kScanThreads - 1];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    total[0] = carry;
    total[1] = aside ? *aside : 0;
  }
}

// Every tile's offset to its prefixes.  Up to kScanFewTiles tiles each block
// sums the tiles before its own itself (kSums; tile_sums are the tiles' own
// then, and the last block leaves the total), which saves the launch of
// scan_tile_sums, 4.4 us and a gap; the sums' reads grow with the square of
// the tiles, 4 MB from cache at 1,024.
constexpr int64_t kScanFewTiles = 1024;

template <bool kSums>
__global__ void scan_add_offsets(int64_t n, int32_t *__restrict__ out,
                                 const int64_t *__restrict__ tile_sums,
                                 int64_t *__restrict__ total, const int32_t *__restrict__ aside) {
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t off;
  if constexpr (kSums) {
    __shared__ int64_t lds[kScanThreads];
    int64_t before = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kScanThreads) before += tile_sums[b];
    block_inclusive_scan(before, lds);
    off = lds[kScanThreads - 1];
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
      total[0] = off + tile_sums[blockIdx.x];
      total[1] = aside ? *aside : 0;
    }
  } else {
    off = tile_sums[blockIdx.x];
  }
  for (int k = threadIdx.x; k < kScanTile; k += kScanThreads) {
    const int64_t i = base + k;
    if (i < n) out[i + 1] = static_cast<int32_t>(out[i + 1] + off);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0;
}

static size_t scan_bytes(int64_t n) {
  const int64_t ntiles = std::max<int64_t>(1, (n + kScanTile - 1) / kScanTile);
  return (size_t)(ntiles + 2) * sizeof(int64_t);
}

// The total comes back to the host, and with it a device counter (aside).
static int scan(int64_t n, const int32_t *in, int32_t *out, int64_t *total_host,
                void *work, size_t work_bytes, hipStream_t s, const int32_t *aside = nullptr,
                int64_t *aside_host = nullptr) {
  OP2HIP_REQUIRE(n >= 0, "scan: negative length");
  if (work_bytes < scan_bytes(n)) {
    set_error("scan: workspace %zu < %zu bytes", work_bytes, scan_bytes(n));
    return OP2HIP_ERR_WORKSPACE;
  }
  const int64_t ntiles = std::max<int64_t>(1, (n + kScanTile - 1) / kScanTile);
  int64_t *tile_sums = static_cast<int64_t *>(work);
  int64_t *total = tile_sums + ntiles;
  scan_tiles<<<(uint32_t)ntiles, kScanThreads, 0, s>>>(n, in, out, tile_sums);
  OP2HIP_LAUNCHED();
  if (ntiles <= kScanFewTiles) {
    scan_add_offsets<true><<<(uint32_t)ntiles, kScanThreads, 0, s>>>(n, out, tile_sums, total, aside);
  } else {
    scan_tile_sums<<<1, kScanThreads, 0, s>>>(ntiles, tile_sums, total, aside);
    OP2HIP_LAUNCHED();
    scan_add_offsets<false><<<(uint32_t)ntiles, kScanThreads, 0, s>>>(n, out, tile_sums, total, aside);
  }
  OP2HIP_LAUNCHED();
  int64_t back[2] = {0, 0};
  OP2HIP_CHECK(hipMemcpyAsync(back, total, sizeof(back), hipMemcpyDeviceToHost, s));
  OP2HIP_CHECK(hipStreamSynchronize(s));
  const int64_t t = back[0];
  if (aside_host) *aside_host = back[1];
  if (total_host) *total_host = t;
  if (t > INT32_MAX) {
    set_error("scan: total %lld exceeds int32", (long long)t);
    return OP2HIP_ERR_OVERFLOW;
  }
  return OP2HIP_OK;
}

// ---------------------------------------------------------------------------
// map transpose

// pos (may be null): each entry's place among its row's entries, as counted.
__global__ void transpose_count(int32_t nrows, const int32_t *__restrict__ map,
                                int64_t nent, int32_t *__restrict__ counts,
                                int32_t *__restrict__ bad, int32_t *__restrict__ pos) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nent;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t r = map[i];
    if (r < 0) continue;
    if (r >= nrows) { atomicAdd(bad, 1); continue; }
    const int32_t at = atomicAdd(&counts[r], 1);
    if (pos) pos[i] = at;
  }
}

// With the places found while counting, filling needs no second round of
// atomics (48 us for the P2 24^3 cube's 829,440 entries, 9 us with them);
// without, each row's cursor hands them out.
__global__ void transpose_place(int32_t nrows, const int32_t *__restrict__ map, int64_t nent,
                                const int32_t *__restrict__ inc_ptr,
                                const int32_t *__restrict__ pos, int32_t *__restrict__ inc_ent) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nent;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t r = map[i];
    if (r >= 0 && r < nrows) inc_ent[(int64_t)inc_ptr[r] + pos[i]] = static_cast<int32_t>(i);
  }
}

__global__ void transpose_fill(int32_t nrows, const int32_t *__restrict__ map,
                               int64_t nent, int32_t *__restrict__ cursor,
                               int32_t *__restrict__ inc_ent) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < nent;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t r = map[i];
    if (r < 0 || r >= nrows) continue;
    const int32_t pos = atomicAdd(&cursor[r], 1);
    inc_ent[pos] = static_cast<int32_t>(i);
  }
}

// Sort each row's incidence list ascending.  A block takes 256 rows and stages
// their lists in LDS; every entry then finds its place by counting the smaller
// entries of its row, all entries of the block at once (one thread sorting a
// row in memory is a chain of dependent loads: 52 us for the 82,944 cells and
// 117,649 nodes of the P2 24^3 cube, 20 us this way).  Rows whose lists do not
// fit the stage together are sorted by one thread each.
constexpr int kSortRows = 256;
constexpr int kSortStage = 7168;

__global__ void __launch_bounds__(kSortRows)
transpose_sort(int32_t nrows, const int32_t *__restrict__ inc_ptr,
               int32_t *__restrict__ inc_ent) {
  __shared__ int32_t ptr[kSortRows + 1];
  __shared__ int32_t ent[kSortStage];
  for (int64_t r0 = (int64_t)blockIdx.x * kSortRows; r0 < nrows;
       r0 += (int64_t)gridDim.x * kSortRows) {
    const int32_t nr = (int32_t)min((int64_t)kSortRows, nrows - r0);
    for (int32_t k = threadIdx.x; k <= nr; k += kSortRows) ptr[k] = inc_ptr[r0 + k];
    __syncthreads();
    const int32_t base = ptr[0], n = ptr[nr] - base;
    if (n <= kSortStage) {
      for (int32_t k = threadIdx.x; k < n; k += kSortRows) ent[k] = inc_ent[(int64_t)base + k];
      __syncthreads();
      for (int32_t k = threadIdx.x; k < n; k += kSortRows) {
        int32_t a = 0, b = nr;   // the row of entry k: the last one that starts at or before it
        while (b - a > 1) {
          const int32_t mid = (a + b) >> 1;
          if (ptr[mid] - base <= k) a = mid; else b = mid;
        }
        const int32_t lo = ptr[a] - base, hi = ptr[a + 1] - base, v = ent[k];
        int32_t rank = 0;
        for (int32_t t = lo; t < hi; ++t) rank += ent[t] < v;
        inc_ent[(int64_t)base + lo + rank] = v;
      }
    } else if ((int32_t)threadIdx.x < nr) {
      const int32_t lo = ptr[threadIdx.x], hi = ptr[threadIdx.x + 1];
      for (int32_t a = lo + 1; a < hi; ++a) {
        const int32_t v = inc_ent[a];
        int32_t b = a - 1;
        while (b >= lo && inc_ent[b] > v) {
          inc_ent[b + 1] = inc_ent[b];
          --b;
        }
        inc_ent[b + 1] = v;
      }
    }
    __syncthreads();  // the next rows reuse the stage
  }
}

static int sort_incidences(int32_t nrows, const int32_t *inc_ptr, int32_t *inc_ent, hipStream_t s) {
  if (nrows <= 0) return OP2HIP_OK;
  transpose_sort<<<std::min<uint32_t>(ceil_div(nrows, kSortRows), 16384), kSortRows, 0, s>>>(
      nrows, inc_ptr, inc_ent);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

static size_t transpose_bytes(int32_t nrows) {
  // counts/cursor (nrows int32) + flag + scan workspace, 256-byte aligned parts
  size_t a = ((size_t)std::max(nrows, 1) * 4 + 255) & ~(size_t)255;
  return a + 256 + scan_bytes(nrows);
}

// ---------------------------------------------------------------------------
// sparsity rows: the sorted distinct columns of every block row

struct PairTable {
  const int32_t *cmap[OP2HIP_MAX_PAIRS];
  const int32_t *inc_ptr[OP2HIP_MAX_PAIRS];
  const int32_t *inc_ent[OP2HIP_MAX_PAIRS];
  int32_t rarity[OP2HIP_MAX_PAIRS];
  int32_t carity[OP2HIP_MAX_PAIRS];
  int32_t npairs;
};

constexpr int kRowCap = 2048;

__device__ __forceinline__ int32_t candidate(const PairTable &pt, int32_t r, int64_t k,
                                             const int32_t *lo, const int32_t *cnt,
                                             int32_t diag_col) {
  for (int p = 0; p < pt.npairs; ++p) {
    const int64_t n = (int64_t)cnt[p] * pt.carity[p];
    if (k < n) {
      const int32_t inc = lo[p] + (int32_t)(k / pt.carity[p]);
      const int32_t j = (int32_t)(k % pt.carity[p]);
      const int32_t e = pt.inc_ent[p][inc] / pt.rarity[p];
      return pt.cmap[p][(int64_t)e * pt.carity[p] + j];
    }
    k -= n;
  }
  return diag_col;  // the diagonal candidate (or -1)
}

__device__ __forceinline__ int32_t block64_sum(int32_t v, int32_t *lds) {
  // 64-thread block reduction through LDS
  lds[threadIdx.x] = v;
  __syncthreads();
  for (int off = 32; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) lds[threadIdx.x] += lds[threadIdx.x + off];
    __syncthreads();
  }
  const int32_t s = lds[0];
  __syncthreads();
  return s;
}

__device__ __forceinline__ int32_t block64_min(int32_t v, int32_t *lds) {
  lds[threadIdx.x] = v;
  __syncthreads();
  for (int off = 32; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) lds[threadIdx.x] = min(lds[threadIdx.x], lds[threadIdx.x + off]);
    __syncthreads();
  }
  const int32_t s = lds[0];
  __syncthreads();
  return s;
}

// Rows of at most kCap candidates: a group of kLanes lanes takes a row, reads
// its candidates (at most six a lane, all loads issued together) and enters
// them in the group's hash table in LDS; a lane whose entry was new holds one
// distinct column.  Counting is then the number of new entries, and filling
// ranks every distinct column among the others.  Comparing all pairs of
// candidates took 412 us (count) and 873 us (fill) for the 117,649 rows of the
// P2 24^3 cube, whose candidates (50 an edge, 240 a vertex) repeat 2 to 4
// times; a table visit per candidate takes 51 and 94 us.
template <int kLanes>
struct RowTable {
  static constexpr int kSlots = kLanes * 8;     // a power of two
  static constexpr int kRounds = 6;
  static constexpr int kCap = kLanes * kRounds; // three quarters of the slots
  static constexpr int kGroups = 256 / kLanes;
};

// LDS accesses before it are seen by those after it in every lane of the wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ int64_t row_candidates(const PairTable &pt, int32_t r, int32_t ncols,
                                                  int32_t set_diag) {
  int64_t m = set_diag && r < ncols ? 1 : 0;
  for (int p = 0; p < pt.npairs; ++p)
    m += (int64_t)(pt.inc_ptr[p][r + 1] - pt.inc_ptr[p][r]) * pt.carity[p];
  return m;
}

template <bool kFill, int kLanes>
__global__ void __launch_bounds__(256)
sparsity_rows(int32_t nrows, int32_t ncols, PairTable pt, int32_t set_diag,
              const int32_t *__restrict__ rowptr, int32_t *__restrict__ out) {
  using Tab = RowTable<kLanes>;
  constexpr int kR = Tab::kRounds;
  __shared__ int32_t tables[Tab::kGroups][Tab::kSlots];
  __shared__ __align__(16) int32_t uniques[kFill ? Tab::kGroups : 1][kFill ? Tab::kCap : 1];
  __shared__ int32_t lo[Tab::kGroups][OP2HIP_MAX_PAIRS], cnt[Tab::kGroups][OP2HIP_MAX_PAIRS];
  const int grp = threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
  const int shift = (threadIdx.x & 63) / kLanes * kLanes;   // of the group's bits in a ballot
  const uint64_t group_mask = kLanes == 64 ? ~0ull : ((1ull << (kLanes & 63)) - 1);
  int32_t *table = tables[grp];
  for (int k = lane; k < Tab::kSlots; k += kLanes) table[k] = -1;
  const int64_t step = (int64_t)gridDim.x * Tab::kGroups;
  int32_t first_inc = 0, ninc = 0;   // of the next row, one pair a lane
  auto load_range = [&](int64_t r) {
    if (lane < pt.npairs && r < nrows) {
      first_inc = pt.inc_ptr[lane][r];
      ninc = pt.inc_ptr[lane][r + 1] - first_inc;
    }
  };
  load_range((int64_t)blockIdx.x * Tab::kGroups + grp);
  for (int64_t r0 = (int64_t)blockIdx.x * Tab::kGroups + grp; r0 < nrows; r0 += step) {
    const int32_t r = (int32_t)r0;
    wave_lds_sync();   // the previous row is done with them
    if (lane < pt.npairs) {
      lo[grp][lane] = first_inc;
      cnt[grp][lane] = ninc;
    }
    wave_lds_sync();
    load_range(r0 + step);
    const int32_t base = kFill ? rowptr[r] : 0;
    const bool has_diag = set_diag && r < ncols;
    int64_t total = has_diag ? 1 : 0;
    for (int p = 0; p < pt.npairs; ++p) total += (int64_t)cnt[grp][p] * pt.carity[p];
    if (total > Tab::kCap) continue;   // sparsity_long_rows takes it
    const int m = (int)total;
    // every lane's incidences, then every lane's columns
    int32_t c[kR], slot[kR], col[kR], pair[kR];
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      if (u * kLanes >= m) break;
      uint32_t k = lane + u * kLanes;
      c[u] = pair[u] = -1;
      if (k >= (uint32_t)m) continue;
      for (int p = 0; p < pt.npairs; ++p) {
        const uint32_t ar = (uint32_t)pt.carity[p], n = (uint32_t)cnt[grp][p] * ar;
        if (k < n) {
          const uint32_t q = k / ar;
          pair[u] = p;
          col[u] = (int32_t)(k - q * ar);
          c[u] = pt.inc_ent[p][lo[grp][p] + (int32_t)q];
          break;
        }
        k -= n;
      }
      if (pair[u] < 0) c[u] = r;   // past the pairs' candidates: the diagonal
    }
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      if (u * kLanes >= m) break;
      if (pair[u] < 0) continue;
      const int p = pair[u];
      const int32_t e = (int32_t)((uint32_t)c[u] / (uint32_t)pt.rarity[p]);
      c[u] = pt.cmap[p][(int64_t)e * pt.carity[p] + col[u]];
    }
    int count = 0;
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      if (u * kLanes >= m) break;
      slot[u] = -1;
      if (c[u] >= 0) {
        uint32_t h = ((uint32_t)c[u] * 2654435761u) / (uint32_t)(0x100000000ull / Tab::kSlots);
        for (;;) {   // ends: fewer entries than slots
          const int32_t was = atomicCAS(&table[h], -1, c[u]);
          if (was == -1) slot[u] = (int32_t)h;
          if (was == -1 || was == c[u]) break;
          h = (h + 1) & (Tab::kSlots - 1);
        }
      }
      const uint64_t news = (__ballot(slot[u] >= 0) >> shift) & group_mask;
      if constexpr (kFill) {
        if (slot[u] >= 0) uniques[grp][count + __popcll(news & ((1ull << lane) - 1))] = c[u];
      }
      count += __popcll(news);
    }
    if constexpr (!kFill) {
      if (lane == 0) out[r] = count;
    } else {
      if (lane < 3 && count + lane < Tab::kCap) uniques[grp][count + lane] = INT32_MAX;
      wave_lds_sync();
      const int4 *quad = reinterpret_cast<const int4 *>(uniques[grp]);
      int32_t *row = out + base;
#pragma unroll
      for (int u = 0; u < kR; ++u) {
        if (u * kLanes >= m) break;
        if (slot[u] < 0) continue;
        int rank = 0;
        for (int t = 0; t < (count + 3) / 4; ++t) {
          const int4 q = quad[t];
          rank += (q.x < c[u]) + (q.y < c[u]) + (q.z < c[u]) + (q.w < c[u]);
        }
        row[rank] = c[u];
      }
    }
    // the slots this lane filled are emptied for the next row
#pragma unroll
    for (int u = 0; u < kR; ++u) {
      if (u * kLanes >= m) break;
      if (slot[u] >= 0) table[slot[u]] = -1;
    }
    wave_lds_sync();
  }
}

// Rows of more than `cap` candidates, a block of 64 threads for 64 rows in
// turn: all pairs of candidates up to kRowCap, repeated minimum extraction
// straight from the maps beyond.
template <bool kFill>
__global__ void __launch_bounds__(64)
sparsity_long_rows(int32_t nrows, int32_t ncols, PairTable pt, int32_t set_diag, int32_t cap,
                   const int32_t *__restrict__ rowptr, int32_t *__restrict__ out) {
  __shared__ int32_t cand[kRowCap];
  __shared__ uint8_t first[kRowCap];
  __shared__ int32_t red[64];
  __shared__ int32_t lo[OP2HIP_MAX_PAIRS], cnt[OP2HIP_MAX_PAIRS];
  const int64_t r0 = (int64_t)blockIdx.x * 64, mine_r = r0 + threadIdx.x;
  uint64_t todo = __ballot(mine_r < nrows && row_candidates(pt, (int32_t)mine_r, ncols, set_diag) > cap);
  for (; todo; todo &= todo - 1) {
    const int32_t r = (int32_t)(r0 + __ffsll((unsigned long long)todo) - 1);
    if (threadIdx.x < (unsigned)pt.npairs) {
      const int p = threadIdx.x;
      lo[p] = pt.inc_ptr[p][r];
      cnt[p] = pt.inc_ptr[p][r + 1] - lo[p];
    }
    __syncthreads();
    const bool has_diag = set_diag && r < ncols;
    const int32_t diag_col = has_diag ? r : -1;
    const int64_t m = row_candidates(pt, r, ncols, set_diag);
    const int32_t base = kFill ? rowptr[r] : 0;
    if (m <= kRowCap) {
      for (int64_t k = threadIdx.x; k < m; k += 64)
        cand[k] = candidate(pt, r, k, lo, cnt, diag_col);
      __syncthreads();
      int32_t mine = 0;
      for (int64_t k = threadIdx.x; k < m; k += 64) {
        const int32_t c = cand[k];
        bool f = c >= 0;
        for (int64_t t = 0; f && t < k; ++t) f = cand[t] != c;
        first[k] = f;
        mine += f;
      }
      __syncthreads();
      if (!kFill) {
        const int32_t total = block64_sum(mine, red);
        if (threadIdx.x == 0) out[r] = total;
      } else {
        for (int64_t k = threadIdx.x; k < m; k += 64) {
          if (!first[k]) continue;
          const int32_t c = cand[k];
          int32_t rank = 0;
          for (int64_t t = 0; t < m; ++t) rank += (first[t] && cand[t] < c);
          out[base + rank] = c;
        }
      }
      __syncthreads();
    } else {
      // longer still: repeated minimum extraction straight from the maps
      int32_t last = -1, count = 0;
      for (;;) {
        int32_t best = INT32_MAX;
        for (int64_t k = threadIdx.x; k < m; k += 64) {
          const int32_t c = candidate(pt, r, k, lo, cnt, diag_col);
          if (c > last && c < best) best = c;
        }
        best = block64_min(best, red);
        if (best == INT32_MAX) break;
        if (kFill && threadIdx.x == 0) out[base + count] = best;
        ++count;
        last = best;
      }
      if (!kFill && threadIdx.x == 0) out[r] = count;
      __syncthreads();
    }
  }
}

// Blocks of a launch over rows.  Counting: as many as the chip holds at once,
// so that a block empties its tables once and reads its next row's range ahead
// (51 us against 57 for the P2 24^3 cube); filling takes longer for the rows of
// vertices, and one row a group shares them out better (94 against 112 us).
template <bool kFill>
constexpr uint32_t kRowBlocks = kFill ? 65536 : 2048;

// Half a wave takes rows of up to 32 candidates on average (P1 triangles: 19),
// a whole wave longer ones (P2 tetrahedra: 73).
template <bool kFill>
static int launch_sparsity_rows(int32_t nrows, int32_t ncols, const op2hip_map_pair *pairs,
                                const PairTable &pt, int32_t set_diag, const int32_t *rowptr,
                                int32_t *out, hipStream_t s) {
  if (nrows <= 0) return OP2HIP_OK;
  double cands = set_diag ? nrows : 0;
  for (int p = 0; p < pt.npairs; ++p)
    cands += (double)pairs[p].iter_size * pt.rarity[p] * pt.carity[p];
  const bool half = cands <= 32.0 * nrows;
  if (half)
    sparsity_rows<kFill, 32><<<std::min<uint32_t>(ceil_div(nrows, RowTable<32>::kGroups), kRowBlocks<kFill>),
                               256, 0, s>>>(nrows, ncols, pt, set_diag, rowptr, out);
  else
    sparsity_rows<kFill, 64><<<std::min<uint32_t>(ceil_div(nrows, RowTable<64>::kGroups), kRowBlocks<kFill>),
                               256, 0, s>>>(nrows, ncols, pt, set_diag, rowptr, out);
  OP2HIP_LAUNCHED();
  sparsity_long_rows<kFill><<<ceil_div(nrows, 64), 64, 0, s>>>(
      nrows, ncols, pt, set_diag, half ? RowTable<32>::kCap : RowTable<64>::kCap, rowptr, out);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

// ---------------------------------------------------------------------------
// tiles of consecutive elements: the distinct targets of a tile, by a hash
// table in LDS, ranked among each other; one workgroup a tile.  Plan work, once
// per map: the 4,096 candidates at most keep table and list within 48 KB.

constexpr int kTargetSlots = 2 * OP2HIP_TILE_CANDIDATES;

template <bool kFill>
__global__ void __launch_bounds__(256)
tile_targets(int32_t n, int32_t tile, const int32_t *__restrict__ table, int32_t arity,
             const int32_t *__restrict__ tile_ptr, int32_t *__restrict__ out,
             uint16_t *__restrict__ local) {
  __shared__ int32_t keys[kTargetSlots];
  __shared__ __align__(16) int32_t list[OP2HIP_TILE_CANDIDATES + 4];
  __shared__ int32_t count;
  const int32_t b = blockIdx.x;
  const int64_t c0 = (int64_t)b * tile * arity;
  const int32_t m = (int32_t)(min((int64_t)n * arity, c0 + (int64_t)tile * arity) - c0);
  for (int32_t k = threadIdx.x; k < kTargetSlots; k += 256) keys[k] = -1;
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  auto home = [](int32_t c) {
    return ((uint32_t)c * 2654435761u) / (uint32_t)(0x100000000ull / kTargetSlots);
  };
  for (int32_t k = threadIdx.x; k < m; k += 256) {
    const int32_t c = table[c0 + k];
    uint32_t h = home(c);
    for (;;) {   // ends: at most half the slots are taken
      const int32_t was = atomicCAS(&keys[h], -1, c);
      if (was == -1) {
        const int32_t at = atomicAdd(&count, 1);
        if (kFill) list[at] = c;
      }
      if (was == -1 || was == c) break;
      h = (h + 1) & (kTargetSlots - 1);
    }
  }
  __syncthreads();
  const int32_t u = count;
  if constexpr (!kFill) {
    if (threadIdx.x == 0) out[b] = u;
  } else {
    if (threadIdx.x < 4) list[u + threadIdx.x] = INT32_MAX;
    __syncthreads();
    const int4 *quad = reinterpret_cast<const int4 *>(list);
    const int32_t p0 = tile_ptr[b];
    for (int32_t k = threadIdx.x; k < u; k += 256) {
      const int32_t c = list[k];
      int32_t rank = 0;
      for (int32_t t = 0; t < (u + 3) / 4; ++t) {
        const int4 q = quad[t];
        rank += (q.x < c) + (q.y < c) + (q.z < c) + (q.w < c);
      }
      out[(int64_t)p0 + rank] = c;
    }
    __syncthreads();   // out of this tile is whole (its writers are this workgroup's)
    for (int32_t k = threadIdx.x; k < m; k += 256) {
      const int32_t c = table[c0 + k];
      int32_t lo = 0, hi = u - 1;
      while (lo < hi) {
        const int32_t mid = (lo + hi) >> 1;
        if (out[(int64_t)p0 + mid] < c) lo = mid + 1; else hi = mid;
      }
      local[c0 + k] = (uint16_t)lo;
    }
  }
}

// Partial sums of every target, one thread per target and component: bound by
// its scattered 8-byte reads, so two slots and their partials are loaded at
// once and the output's value beside the range (10 us for 361,201 targets of
// four values, 13 us for the 1,753,001 entries of a P1 matrix, 11 and 14.5 us
// one at a time; the tiles before it take 24 and 11 us, where device atomics
// took 72 and 137 us).
template <typename T, typename A>
__global__ void __launch_bounds__(256)
tile_targets_add(int32_t nrows, int32_t dim, const int32_t *__restrict__ ptr,
                 const int32_t *__restrict__ slots, const A *__restrict__ partials,
                 T *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)nrows * dim) return;
  const int32_t r = dim == 1 ? (int32_t)i : (int32_t)(i / dim), j = (int32_t)(i - (int64_t)r * dim);
  constexpr int kAtOnce = 2;
  int32_t k = ptr[r];
  const int32_t end = ptr[r + 1];
  if (k == end) return;
  const T old = out[i];
  A sum = A(0);
  for (; k < end; k += kAtOnce) {
    int32_t slot[kAtOnce];
    A v[kAtOnce];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) slot[u] = slots[k + u < end ? k + u : end - 1];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) v[u] = partials[(int64_t)slot[u] * dim + j];
#pragma unroll
    for (int u = 0; u < kAtOnce; ++u) sum += k + u < end ? v[u] : A(0);
  }
  out[i] = T(A(old) + sum);
}

__global__ void mat_slots(int64_t total, const int32_t *__restrict__ rowptr,
                          const int32_t *__restrict__ colidx, const int32_t *__restrict__ rmap,
                          int32_t rarity, const int32_t *__restrict__ cmap, int32_t carity,
                          int32_t *__restrict__ slots, int32_t *__restrict__ bad) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < total;
       k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t ei = k / carity;   // element and local row
    const int32_t r = rmap[ei], c = cmap[ei / rarity * carity + k % carity];
    const int32_t at = r < 0 || c < 0 ? -1 : find_slot(colidx, rowptr[r], rowptr[r + 1], c);
    if (at < 0) atomicAdd(bad, 1);
    slots[k] = at;
  }
}

// Zero bytes from a 16-byte boundary on, bound by the stores.  Four words a
// thread; beyond the 256 MB of the last-level cache one word a thread, stored
// past the caches.  A pass with the loop that follows, against torch's fill:
// 23 MB 25.1 and 26.5 us, 52 MB 104.5 and 108, 59 MB 96 and 99; 765 MB 576 and
// 597 (four plain words a thread 599; past the caches, 52 MB would take 110).
typedef uint32_t ClearWord __attribute__((ext_vector_type(4)));
constexpr int64_t kClearCached = 256ll << 20;

template <int kWords, bool kPast>
__global__ void __launch_bounds__(256)
clear_words(ClearWord *__restrict__ p, int64_t n, uint8_t *__restrict__ rest, int32_t nrest) {
  const int64_t first = (int64_t)blockIdx.x * (256 * kWords) + threadIdx.x;
  const ClearWord zero = {0, 0, 0, 0};
#pragma unroll
  for (int u = 0; u < kWords; ++u) {
    const int64_t i = first + u * 256;
    if (i >= n) break;
    if (kPast) __builtin_nontemporal_store(zero, p + i);
    else p[i] = zero;
  }
  if (first < nrest) rest[first] = 0;
}

// Smallest and largest of n entries: a pair per workgroup, bound by one read of
// the entries.
__global__ void __launch_bounds__(256)
entry_range(int64_t n, const int32_t *__restrict__ v, int32_t *__restrict__ pairs) {
  __shared__ int32_t least[4], most[4];
  int32_t lo = INT32_MAX, hi = INT32_MIN;
#pragma unroll 4
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    lo = min(lo, v[i]);
    hi = max(hi, v[i]);
  }
  for (int d = 32; d > 0; d >>= 1) {
    lo = min(lo, __shfl_xor(lo, d));
    hi = max(hi, __shfl_xor(hi, d));
  }
  if (threadIdx.x % 64 == 0) {
    least[threadIdx.x / 64] = lo;
    most[threadIdx.x / 64] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      lo = min(lo, least[w]);
      hi = max(hi, most[w]);
    }
    pairs[2 * blockIdx.x] = lo;
    pairs[2 * blockIdx.x + 1] = hi;
  }
}

// Half the sum of squares of n values in two launches: every workgroup writes
// one partial, the second launch adds them, both in a fixed order.  One pass
// over memory, where a product, a reduction over it and a scaling were three:
// 0.8 million values (6.6 MB, from the last-level cache) 4 + 2 against 17 us.
constexpr int kHalfSquareBlocks = 1024, kHalfSquareAtOnce = 4;

__device__ __forceinline__ double sum_of_workgroup(double v) {
  __shared__ double waves[16];
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
  if (threadIdx.x % 64 == 0) waves[threadIdx.x / 64] = v;
  __syncthreads();
  v = 0.0;
  for (uint32_t w = 0; w < blockDim.x / 64; ++w) v += waves[w];
  return v;
}

__global__ void __launch_bounds__(256)
half_square_partials(int64_t n, const double *__restrict__ x, double *__restrict__ partials) {
  const int64_t stride = (int64_t)gridDim.x * 256;
  double sum = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += stride * kHalfSquareAtOnce) {
    double v[kHalfSquareAtOnce];
#pragma unroll
    for (int u = 0; u < kHalfSquareAtOnce; ++u) v[u] = i + u * stride < n ? x[i + u * stride] : 0.0;
#pragma unroll
    for (int u = 0; u < kHalfSquareAtOnce; ++u) sum += v[u] * v[u];
  }
  sum = sum_of_workgroup(sum);
  if (threadIdx.x == 0) partials[blockIdx.x] = sum;
}

__global__ void __launch_bounds__(kHalfSquareBlocks)
half_square_total(int32_t n, const double *__restrict__ partials, double *__restrict__ out) {
  const double sum = sum_of_workgroup((int32_t)threadIdx.x < n ? partials[threadIdx.x] : 0.0);
  if (threadIdx.x == 0) *out = 0.5 * sum;
}

__global__ void expand_rowptr(int32_t nrows, const int32_t *__restrict__ rowptr,
                              int32_t rdim, int32_t cdim, int32_t *__restrict__ out) {
  for (int32_t r = blockIdx.x * blockDim.x + threadIdx.x; r <= nrows;
       r += gridDim.x * blockDim.x) {
    if (r == nrows) {
      out[(int64_t)nrows * rdim] = rowptr[nrows] * rdim * cdim;
      continue;
    }
    const int32_t len = rowptr[r + 1] - rowptr[r];
    for (int ri = 0; ri < rdim; ++ri)
      out[(int64_t)r * rdim + ri] = rowptr[r] * rdim * cdim + ri * len * cdim;
  }
}

__global__ void expand_colidx(int32_t nrows, const int32_t *__restrict__ rowptr,
                              const int32_t *__restrict__ colidx, int32_t rdim,
                              int32_t cdim, const int32_t *__restrict__ rowptr_out,
                              int32_t *__restrict__ out) {
  for (int32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nrows;
       r += gridDim.x * blockDim.x) {
    const int32_t lo = rowptr[r], len = rowptr[r + 1] - lo;
    for (int ri = 0; ri < rdim; ++ri) {
      int32_t *o = out + rowptr_out[(int64_t)r * rdim + ri];
      for (int32_t s = 0; s < len; ++s)
        for (int cj = 0; cj < cdim; ++cj) o[s * cdim + cj] = colidx[lo + s] * cdim + cj;
    }
  }
}

static int make_pairs(const op2hip_map_pair *pairs, int32_t npairs,
                      const int32_t *const *inc_ptr, const int32_t *const *inc_ent,
                      PairTable *pt) {
  OP2HIP_REQUIRE(npairs >= 0 && npairs <= OP2HIP_MAX_PAIRS,
                 "sparsity: %d map pairs (max %d)", npairs, OP2HIP_MAX_PAIRS);
  std::memset(pt, 0, sizeof(*pt));
  pt->npairs = npairs;
  for (int p = 0; p < npairs; ++p) {
    OP2HIP_REQUIRE(pairs[p].rarity > 0 && pairs[p].carity > 0, "sparsity: bad arity");
    OP2HIP_REQUIRE(inc_ptr && inc_ent && inc_ptr[p] && inc_ent[p],
                   "sparsity: missing row incidences of pair %d", p);
    pt->cmap[p] = pairs[p].cmap;
    pt->inc_ptr[p] = inc_ptr[p];
    pt->inc_ent[p] = inc_ent[p];
    pt->rarity[p] = pairs[p].rarity;
    pt->carity[p] = pairs[p].carity;
  }
  return OP2HIP_OK;
}

}  // namespace op2hip

using namespace op2hip;

extern "C" {

int op2hip_abi_version(void) { return OP2HIP_ABI_VERSION; }

const char *op2hip_last_error(void) { return g_error; }

int op2hip_init(int32_t device) {
  int n = 0;
  OP2HIP_CHECK(hipGetDeviceCount(&n));
  OP2HIP_REQUIRE(device >= 0 && device < n, "device %d not present (%d devices)", device, n);
  OP2HIP_CHECK(hipSetDevice(device));
  hipDeviceProp_t prop;
  OP2HIP_CHECK(hipGetDeviceProperties(&prop, device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    set_error("device %d is %s; this library is built for gfx950 only", device,
              prop.gcnArchName);
    return OP2HIP_ERR_ARG;
  }
  // the no-allocation entry point's scratch address on this device
  void *scratch = nullptr;
  return noalloc_scratch_address(device, &scratch);
}

int op2hip_scan_workspace(int64_t n, size_t *bytes) {
  OP2HIP_REQUIRE(bytes, "scan_workspace: NULL");
  *bytes = scan_bytes(n);
  return OP2HIP_OK;
}

int op2hip_exclusive_scan(int64_t n, const int32_t *in, int32_t *out, int64_t *total_host,
                          void *work, size_t work_bytes, void *stream) {
  return scan(n, in, out, total_host, work, work_bytes, stream_of(stream));
}

int op2hip_transpose_workspace(int32_t nrows, size_t *bytes) {
  OP2HIP_REQUIRE(bytes && nrows >= 0, "transpose_workspace: bad arguments");
  *bytes = transpose_bytes(nrows);
  return OP2HIP_OK;
}

int op2hip_transpose_count_places(int32_t nrows, const int32_t *map, int32_t arity,
                                  int32_t iter_size, int32_t *inc_ptr, int64_t *total_host,
                                  int32_t *places, void *work, size_t work_bytes, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && arity > 0 && iter_size >= 0 && inc_ptr,
                 "transpose_count: bad arguments");
  OP2HIP_REQUIRE(iter_size == 0 || map, "transpose_count: NULL map");
  if (work_bytes < transpose_bytes(nrows)) {
    set_error("transpose: workspace %zu < %zu", work_bytes, transpose_bytes(nrows));
    return OP2HIP_ERR_WORKSPACE;
  }
  char *w = static_cast<char *>(work);
  const size_t a = ((size_t)std::max(nrows, 1) * 4 + 255) & ~(size_t)255;
  int32_t *counts = reinterpret_cast<int32_t *>(w);
  int32_t *bad = counts + nrows;   // cleared with the counts; within the 256 bytes after them
  void *scan_work = w + a + 256;
  int rc;
  if ((rc = fill(counts, (int64_t)nrows + 1, 0, s))) return rc;
  const int64_t nent = (int64_t)iter_size * arity;
  if (nent > 0) {
    transpose_count<<<std::min<uint32_t>(ceil_div(nent, 256), 16384), 256, 0, s>>>(
        nrows, map, nent, counts, bad, places);
    OP2HIP_LAUNCHED();
  }
  int64_t nbad = 0;
  if ((rc = scan(nrows, counts, inc_ptr, total_host, scan_work, work_bytes - a - 256, s, bad, &nbad)))
    return rc;
  if (nbad) {
    set_error("transpose: %lld map entries >= %d (target set size)", (long long)nbad, nrows);
    return OP2HIP_ERR_ARG;
  }
  return OP2HIP_OK;
}

int op2hip_transpose_count(int32_t nrows, const int32_t *map, int32_t arity,
                           int32_t iter_size, int32_t *inc_ptr, int64_t *total_host,
                           void *work, size_t work_bytes, void *stream) {
  return op2hip_transpose_count_places(nrows, map, arity, iter_size, inc_ptr, total_host, nullptr,
                                       work, work_bytes, stream);
}

int op2hip_transpose_fill_places(int32_t nrows, const int32_t *map, int32_t arity,
                                 int32_t iter_size, const int32_t *inc_ptr,
                                 const int32_t *places, int32_t *inc_ent, void *stream) {
  hipStream_t s = stream_of(stream);
  const int64_t nent = (int64_t)iter_size * arity;
  OP2HIP_REQUIRE(nrows >= 0 && arity > 0 && iter_size >= 0 && inc_ptr && (nent == 0 || places),
                 "transpose_fill_places: bad arguments");
  if (nent > 0) {
    transpose_place<<<std::min<uint32_t>(ceil_div(nent, 256), 16384), 256, 0, s>>>(
        nrows, map, nent, inc_ptr, places, inc_ent);
    OP2HIP_LAUNCHED();
  }
  return sort_incidences(nrows, inc_ptr, inc_ent, s);
}

int op2hip_transpose_fill(int32_t nrows, const int32_t *map, int32_t arity,
                          int32_t iter_size, const int32_t *inc_ptr, int32_t *inc_ent,
                          void *work, size_t work_bytes, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && arity > 0 && iter_size >= 0 && inc_ptr,
                 "transpose_fill: bad arguments");
  if (work_bytes < transpose_bytes(nrows)) {
    set_error("transpose: workspace %zu < %zu", work_bytes, transpose_bytes(nrows));
    return OP2HIP_ERR_WORKSPACE;
  }
  int32_t *cursor = static_cast<int32_t *>(work);
  if (nrows > 0)
    OP2HIP_CHECK(hipMemcpyAsync(cursor, inc_ptr, sizeof(int32_t) * nrows,
                                hipMemcpyDeviceToDevice, s));
  const int64_t nent = (int64_t)iter_size * arity;
  if (nent > 0) {
    transpose_fill<<<std::min<uint32_t>(ceil_div(nent, 256), 16384), 256, 0, s>>>(
        nrows, map, nent, cursor, inc_ent);
    OP2HIP_LAUNCHED();
  }
  return sort_incidences(nrows, inc_ptr, inc_ent, s);
}

int op2hip_sparsity_count(int32_t nrows, int32_t ncols, const op2hip_map_pair *pairs,
                          int32_t npairs, const int32_t *const *inc_ptr,
                          const int32_t *const *inc_ent, int32_t set_diag,
                          int32_t *rowptr, int64_t *nnz_host, void *work,
                          size_t work_bytes, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && ncols >= 0 && rowptr, "sparsity_count: bad arguments");
  PairTable pt;
  int rc;
  if ((rc = make_pairs(pairs, npairs, inc_ptr, inc_ent, &pt))) return rc;
  const size_t a = ((size_t)std::max(nrows, 1) * 4 + 255) & ~(size_t)255;
  if (work_bytes < a + scan_bytes(nrows)) {
    set_error("sparsity: workspace %zu < %zu", work_bytes, a + scan_bytes(nrows));
    return OP2HIP_ERR_WORKSPACE;
  }
  int32_t *counts = static_cast<int32_t *>(work);
  if ((rc = launch_sparsity_rows<false>(nrows, ncols, pairs, pt, set_diag, nullptr, counts, s)))
    return rc;
  return scan(nrows, counts, rowptr, nnz_host, static_cast<char *>(work) + a,
              work_bytes - a, s);
}

int op2hip_sparsity_fill(int32_t nrows, int32_t ncols, const op2hip_map_pair *pairs,
                         int32_t npairs, const int32_t *const *inc_ptr,
                         const int32_t *const *inc_ent, int32_t set_diag,
                         const int32_t *rowptr, int32_t *colidx, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && ncols >= 0 && rowptr, "sparsity_fill: bad arguments");
  PairTable pt;
  int rc;
  if ((rc = make_pairs(pairs, npairs, inc_ptr, inc_ent, &pt))) return rc;
  return launch_sparsity_rows<true>(nrows, ncols, pairs, pt, set_diag, rowptr, colidx, s);
}

int op2hip_tile_targets_count(int32_t n, int32_t tile, const int32_t *table, int32_t arity,
                              int32_t *counts, void *stream) {
  OP2HIP_REQUIRE(n >= 0 && tile > 0 && arity > 0 &&
                     (int64_t)tile * arity <= OP2HIP_TILE_CANDIDATES && (n == 0 || (table && counts)),
                 "tile_targets_count: bad arguments");
  if (n == 0) return OP2HIP_OK;
  tile_targets<false><<<ceil_div(n, tile), 256, 0, stream_of(stream)>>>(n, tile, table, arity, nullptr,
                                                                        counts, nullptr);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_tile_targets_fill(int32_t n, int32_t tile, const int32_t *table, int32_t arity,
                             const int32_t *tile_ptr, int32_t *nodes, uint16_t *local,
                             void *stream) {
  OP2HIP_REQUIRE(n >= 0 && tile > 0 && arity > 0 &&
                     (int64_t)tile * arity <= OP2HIP_TILE_CANDIDATES &&
                     (n == 0 || (table && tile_ptr && nodes && local)),
                 "tile_targets_fill: bad arguments");
  if (n == 0) return OP2HIP_OK;
  tile_targets<true><<<ceil_div(n, tile), 256, 0, stream_of(stream)>>>(n, tile, table, arity, tile_ptr,
                                                                       nodes, local);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_tile_targets_add(int32_t type, int32_t nrows, int32_t dim, const int32_t *ptr,
                            const int32_t *slots, const void *partials, void *out,
                            void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && dim > 0 && type >= 0 && type <= 3 &&
                     (nrows == 0 || (ptr && slots && partials && out)),
                 "tile_targets_add: bad arguments");
  if (nrows == 0) return OP2HIP_OK;
  const uint32_t grid = ceil_div((int64_t)nrows * dim, 256);
  if (type == 0)
    tile_targets_add<<<grid, 256, 0, s>>>(nrows, dim, ptr, slots, (const double *)partials, (double *)out);
  else if (type == 1)
    tile_targets_add<<<grid, 256, 0, s>>>(nrows, dim, ptr, slots, (const double *)partials, (float *)out);
  else if (type == 2)
    tile_targets_add<<<grid, 256, 0, s>>>(nrows, dim, ptr, slots, (const int32_t *)partials, (int32_t *)out);
  else
    tile_targets_add<<<grid, 256, 0, s>>>(nrows, dim, ptr, slots, (const int64_t *)partials, (int64_t *)out);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_mat_slots(int32_t n, const int32_t *rowptr, const int32_t *colidx,
                     const int32_t *rmap, int32_t rarity, const int32_t *cmap, int32_t carity,
                     int32_t *slots, int32_t *bad, void *stream) {
  OP2HIP_REQUIRE(n >= 0 && rarity > 0 && carity > 0 &&
                     (n == 0 || (rowptr && colidx && rmap && cmap && slots && bad)),
                 "mat_slots: bad arguments");
  const int64_t total = (int64_t)n * rarity * carity;
  if (total == 0) return OP2HIP_OK;
  mat_slots<<<std::min<uint32_t>(ceil_div(total, 256), 65536), 256, 0, stream_of(stream)>>>(
      total, rowptr, colidx, rmap, rarity, cmap, carity, slots, bad);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_clear(void *data, int64_t bytes, void *stream) {
  OP2HIP_REQUIRE(bytes >= 0 && (bytes == 0 || (data && reinterpret_cast<uintptr_t>(data) % 16 == 0)),
                 "clear: bad arguments");
  if (bytes == 0) return OP2HIP_OK;
  hipStream_t s = stream_of(stream);
  const int64_t n = bytes / 16;
  ClearWord *p = static_cast<ClearWord *>(data);
  uint8_t *rest = reinterpret_cast<uint8_t *>(p + n);
  const int32_t nrest = (int32_t)(bytes % 16);
  if (bytes > kClearCached)
    clear_words<1, true><<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(p, n, rest, nrest);
  else
    clear_words<4, false><<<(uint32_t)std::max<int64_t>(1, (n + 1023) / 1024), 256, 0, s>>>(p, n, rest, nrest);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_entry_range(int64_t n, const int32_t *values, int32_t npairs, int32_t *pairs,
                       void *stream) {
  OP2HIP_REQUIRE(n >= 0 && npairs > 0 && pairs && (n == 0 || values), "entry_range: bad arguments");
  entry_range<<<npairs, 256, 0, stream_of(stream)>>>(n, values, pairs);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_half_square(int64_t n, const double *x, double *partials, double *out, void *stream) {
  OP2HIP_REQUIRE(n >= 0 && partials && out && (n == 0 || x), "half_square: bad arguments");
  hipStream_t s = stream_of(stream);
  const int32_t grid = (int32_t)std::min<int64_t>((n + 255) / 256, kHalfSquareBlocks);
  static_assert(kHalfSquareBlocks == OP2HIP_HALF_SQUARE_PARTIALS);
  if (grid > 0) half_square_partials<<<grid, 256, 0, s>>>(n, x, partials);
  half_square_total<<<1, kHalfSquareBlocks, 0, s>>>(grid, partials, out);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_pattern_expand(int32_t nrows, const int32_t *rowptr, const int32_t *colidx,
                          int32_t rdim, int32_t cdim, int32_t *rowptr_out,
                          int32_t *colidx_out, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nrows >= 0 && rdim > 0 && cdim > 0, "pattern_expand: bad arguments");
  expand_rowptr<<<std::min<uint32_t>(ceil_div((int64_t)nrows + 1, 256), 16384), 256, 0, s>>>(
      nrows, rowptr, rdim, cdim, rowptr_out);
  OP2HIP_LAUNCHED();
  if (nrows > 0) {
    expand_colidx<<<std::min<uint32_t>(ceil_div(nrows, 256), 16384), 256, 0, s>>>(
        nrows, rowptr, colidx, rdim, cdim, rowptr_out, colidx_out);
    OP2HIP_LAUNCHED();
  }
  return OP2HIP_OK;
}

int op2hip_colour_greedy(int32_t nelem, int32_t nmaps, const int32_t *const *maps,
                         const int32_t *arity, const int32_t *target_id,
                         const int32_t *target_size, int32_t ntargets,
                         int32_t *colour, int32_t *ncolours) {
  OP2HIP_REQUIRE(nelem >= 0 && nmaps >= 0 && ntargets >= 0 && colour && ncolours,
                 "colour_greedy: bad arguments");
  for (int m = 0; m < nmaps; ++m)
    OP2HIP_REQUIRE(target_id[m] >= 0 && target_id[m] < ntargets,
                   "colour_greedy: map %d has target %d", m, target_id[m]);
  std::vector<std::vector<uint32_t>> masks(ntargets);
  for (int t = 0; t < ntargets; ++t) masks[t].assign(std::max(target_size[t], 1), 0u);
  std::fill(colour, colour + nelem, -1);
  int32_t left = nelem, base = 0, highest = 0;
  while (left > 0) {
    for (auto &m : masks) std::fill(m.begin(), m.end(), 0u);
    for (int32_t e = 0; e < nelem; ++e) {
      if (colour[e] >= 0) continue;
      uint32_t used = 0;
      for (int m = 0; m < nmaps; ++m) {
        const int32_t *row = maps[m] + (int64_t)e * arity[m];
        for (int i = 0; i < arity[m]; ++i)
          if (row[i] >= 0) {
            if (row[i] >= target_size[target_id[m]]) {
              set_error("colour_greedy: map %d entry %d out of range", m, row[i]);
              return OP2HIP_ERR_ARG;
            }
            used |= masks[target_id[m]][row[i]];
          }
      }
      if (used == 0xFFFFFFFFu) continue;  // try again in the next pass
      const int c = __builtin_ctz(~used);
      colour[e] = base + c;
      highest = std::max(highest, base + c + 1);
      --left;
      for (int m = 0; m < nmaps; ++m) {
        const int32_t *row = maps[m] + (int64_t)e * arity[m];
        for (int i = 0; i < arity[m]; ++i)
          if (row[i] >= 0) masks[target_id[m]][row[i]] |= (1u << c);
      }
    }
    base += 32;
  }
  *ncolours = highest;
  return OP2HIP_OK;
}

int op2hip_plan_tiles(int32_t start, int32_t end, int32_t nmaps, const int32_t *const *maps,
                      const int32_t *arity, const int32_t *target_size, int32_t tile_size,
                      int32_t node_cap, int32_t *ntiles_out, int32_t *tile_ptr,
                      int32_t *tile_elems, int32_t *const *node_ptr, int32_t *const *nodes,
                      int32_t *const *nexcl, uint16_t *const *local, int32_t *max_nodes) {
  OP2HIP_REQUIRE(end >= start && start >= 0 && nmaps >= 1 && nmaps <= 2 && tile_size > 0 &&
                     ntiles_out && tile_ptr && tile_elems && node_ptr && nodes && nexcl && local &&
                     max_nodes,
                 "plan_tiles: bad arguments");
  OP2HIP_REQUIRE(node_cap <= 0 || node_cap >= arity[0],
                 "plan_tiles: a node cap of %d cannot hold one element (arity %d)", node_cap,
                 arity[0]);
  for (int m = 0; m < nmaps; ++m)
    OP2HIP_REQUIRE(maps[m] && arity[m] > 0 && (int64_t)tile_size * arity[m] <= 65535,
                   "plan_tiles: map %d: arity %d, tile size %d (local ids are 16-bit)", m, arity[m],
                   tile_size);
  const int32_t n = end - start;
  // elements around each node of map 0 (the adjacency the regions grow over)
  const int32_t a0 = arity[0], nt0 = std::max(target_size[0], 1);
  std::vector<int32_t> adj_ptr(nt0 + 1, 0), adj;
  for (int32_t k = 0; k < n; ++k)
    for (int i = 0; i < a0; ++i) {
      const int32_t v = maps[0][(int64_t)(start + k) * a0 + i];
      OP2HIP_REQUIRE(v >= 0 && v < target_size[0], "plan_tiles: map 0 entry %d out of range", v);
      ++adj_ptr[v + 1];
    }
  for (int32_t v = 0; v < nt0; ++v) adj_ptr[v + 1] += adj_ptr[v];
  adj.resize(adj_ptr[nt0]);
  {
    std::vector<int32_t> fillp(adj_ptr.begin(), adj_ptr.end() - 1);
    for (int32_t k = 0; k < n; ++k)
      for (int i = 0; i < a0; ++i) adj[fillp[maps[0][(int64_t)(start + k) * a0 + i]]++] = k;
  }
  // regions: breadth first from the lowest unassigned element; elements queued
  // but not taken when the tile is full are released for later tiles
  // (and, with node_cap > 0, at most node_cap distinct nodes of map 0)
  std::vector<uint8_t> taken(n, 0), queued(n, 0);
  std::vector<int32_t> queue, mark(nt0, -1);
  queue.reserve(n);
  int32_t seed = 0, pos = 0, ntiles = 0;
  tile_ptr[0] = 0;
  while (pos < n) {
    const int32_t t = ntiles++;
    queue.clear();
    size_t head = 0;
    const int32_t want = std::min(tile_size, n - pos);
    int32_t got = 0, tile_nodes = 0;
    while (got < want) {
      if (head == queue.size()) {
        if (got > 0 && node_cap > 0) break;  // region exhausted: start a new tile
        while (taken[seed] || queued[seed]) ++seed;
        queued[seed] = 1;
        queue.push_back(seed);
      }
      const int32_t k = queue[head++];
      if (node_cap > 0) {
        int32_t fresh = 0;
        for (int i = 0; i < a0; ++i) fresh += mark[maps[0][(int64_t)(start + k) * a0 + i]] != t;
        if (got > 0 && tile_nodes + fresh > node_cap) {
          queued[k] = 0;
          continue;
        }
        for (int i = 0; i < a0; ++i) {
          int32_t &mk = mark[maps[0][(int64_t)(start + k) * a0 + i]];
          tile_nodes += mk != t;
          mk = t;
        }
      }
      taken[k] = 1;
      tile_elems[pos++] = start + k;
      ++got;
      for (int i = 0; i < a0 && got < want; ++i) {
        const int32_t v = maps[0][(int64_t)(start + k) * a0 + i];
        for (int32_t q = adj_ptr[v]; q < adj_ptr[v + 1]; ++q) {
          const int32_t k2 = adj[q];
          if (!taken[k2] && !queued[k2]) {
            queued[k2] = 1;
            queue.push_back(k2);
          }
        }
      }
    }
    for (size_t q = head; q < queue.size(); ++q) queued[queue[q]] = 0;
    tile_ptr[t + 1] = pos;
  }
  *ntiles_out = ntiles;
  // per map: the distinct nodes of each tile, those of no other tile first
  for (int m = 0; m < nmaps; ++m) {
    const int32_t am = arity[m], ntm = std::max(target_size[m], 1);
    std::vector<int32_t> ntile(ntm, 0), stamp(ntm, -1), slot(ntm, 0);
    for (int32_t t = 0; t < ntiles; ++t)
      for (int32_t p = tile_ptr[t]; p < tile_ptr[t + 1]; ++p)
        for (int i = 0; i < am; ++i) {
          const int32_t v = maps[m][(int64_t)tile_elems[p] * am + i];
          OP2HIP_REQUIRE(v >= 0 && v < target_size[m], "plan_tiles: map %d entry %d out of range",
                         m, v);
          if (stamp[v] != t) {
            stamp[v] = t;
            ++ntile[v];
          }
        }
    std::fill(stamp.begin(), stamp.end(), -1);
    std::vector<int32_t> own, shared;
    int32_t total = 0, mx = 0;
    node_ptr[m][0] = 0;
    for (int32_t t = 0; t < ntiles; ++t) {
      own.clear();
      shared.clear();
      for (int32_t p = tile_ptr[t]; p < tile_ptr[t + 1]; ++p)
        for (int i = 0; i < am; ++i) {
          const int32_t v = maps[m][(int64_t)tile_elems[p] * am + i];
          if (stamp[v] != t) {
            stamp[v] = t;
            (ntile[v] == 1 ? own : shared).push_back(v);
          }
        }
      std::sort(own.begin(), own.end());
      std::sort(shared.begin(), shared.end());
      int32_t c = 0;
      for (int32_t v : own) { nodes[m][total + c] = v; slot[v] = c++; }
      for (int32_t v : shared) { nodes[m][total + c] = v; slot[v] = c++; }
      nexcl[m][t] = (int32_t)own.size();
      for (int32_t p = tile_ptr[t]; p < tile_ptr[t + 1]; ++p)
        for (int i = 0; i < am; ++i)
          local[m][(int64_t)p * am + i] =
              static_cast<uint16_t>(slot[maps[m][(int64_t)tile_elems[p] * am + i]]);
      total += c;
      mx = std::max(mx, c);
      node_ptr[m][t + 1] = total;
    }
    max_nodes[m] = mx;
  }
  return OP2HIP_OK;
}

int op2hip_plan_tile_reduce(int32_t ntiles, const int32_t *node_ptr, const int32_t *nodes,
                            const int32_t *nexcl, int32_t nnodes, int32_t *shared_off,
                            int32_t *nshared, int32_t *shared_nodes, int32_t *shared_ptr,
                            int32_t *shared_slots) {
  OP2HIP_REQUIRE(ntiles >= 0 && nnodes >= 0 && node_ptr && nodes && nexcl && shared_off &&
                     nshared && shared_nodes && shared_ptr && shared_slots,
                 "plan_tile_reduce: bad arguments");
  // partial slots: the shared nodes of each tile, tiles in order
  shared_off[0] = 0;
  for (int32_t b = 0; b < ntiles; ++b) {
    const int32_t cnt = node_ptr[b + 1] - node_ptr[b];
    OP2HIP_REQUIRE(cnt >= 0 && nexcl[b] >= 0 && nexcl[b] <= cnt,
                   "plan_tile_reduce: tile %d has %d nodes, %d exclusive", b, cnt, nexcl[b]);
    shared_off[b + 1] = shared_off[b] + (cnt - nexcl[b]);
  }
  const int32_t nslots = shared_off[ntiles];
  // counting sort of the slots by node id (stable: tile order within a node)
  std::vector<int32_t> count((size_t)nnodes + 1, 0);
  for (int32_t b = 0; b < ntiles; ++b)
    for (int32_t k = node_ptr[b] + nexcl[b]; k < node_ptr[b + 1]; ++k) {
      const int32_t v = nodes[k];
      OP2HIP_REQUIRE(v >= 0 && v < nnodes, "plan_tile_reduce: node %d out of range", v);
      ++count[(size_t)v + 1];
    }
  int32_t ns = 0;
  std::vector<int32_t> first((size_t)nnodes, -1);
  for (int32_t v = 0; v < nnodes; ++v)
    if (count[(size_t)v + 1] > 0) {
      first[v] = ns;
      shared_nodes[ns] = v;
      ++ns;
    }
  shared_ptr[0] = 0;
  for (int32_t s = 0; s < ns; ++s) shared_ptr[s + 1] = shared_ptr[s] + count[(size_t)shared_nodes[s] + 1];
  std::vector<int32_t> fill(shared_ptr, shared_ptr + ns);
  for (int32_t b = 0; b < ntiles; ++b)
    for (int32_t k = node_ptr[b] + nexcl[b]; k < node_ptr[b + 1]; ++k) {
      const int32_t s = first[nodes[k]];
      shared_slots[fill[s]++] = shared_off[b] + (k - node_ptr[b] - nexcl[b]);
    }
  OP2HIP_REQUIRE(shared_ptr[ns] == nslots, "plan_tile_reduce: internal slot count mismatch");
  *nshared = ns;
  return OP2HIP_OK;
}

int op2hip_plan_row_batches(int32_t nrows, const int32_t *inc_ptr, const int32_t *rowptr,
                            int32_t max_inc, int32_t max_nnz, int32_t *batch_rows,
                            int32_t *nbatches, int32_t *max_batch_inc,
                            int32_t *max_batch_nnz, int32_t *max_batch_rows) {
  OP2HIP_REQUIRE(nrows >= 0 && inc_ptr && rowptr && batch_rows && nbatches &&
                     max_inc > 0 && max_nnz > 0,
                 "plan_row_batches: bad arguments");
  int32_t nb = 0, mi = 0, mn = 0, mr = 0;
  int32_t r = 0;
  batch_rows[0] = 0;
  while (r < nrows) {
    const int32_t r0 = r;
    int32_t inc = 0, nnz = 0;
    while (r < nrows) {
      const int32_t di = inc_ptr[r + 1] - inc_ptr[r];
      const int32_t dn = rowptr[r + 1] - rowptr[r];
      if (r > r0 && (inc + di > max_inc || nnz + dn > max_nnz)) break;
      inc += di;
      nnz += dn;
      ++r;
    }
    batch_rows[++nb] = r;
    mi = std::max(mi, inc);
    mn = std::max(mn, nnz);
    mr = std::max(mr, r - r0);
  }
  *nbatches = nb;
  if (max_batch_inc) *max_batch_inc = mi;
  if (max_batch_nnz) *max_batch_nnz = mn;
  if (max_batch_rows) *max_batch_rows = mr;
  return OP2HIP_OK;
}

}  // extern "C"

#include "rowgather.hpp"

namespace op2hip {

template <int kCar>
int plan_rowlist(int32_t nrows, const int32_t *rowptr, const int32_t *colidx,
                 const int32_t *inc_ptr, const int32_t *inc_ent, const int32_t *cmap,
                 int32_t rarity, int32_t max_inc, int32_t max_nnz, int32_t *row_order,
                 int32_t *nbatches, BatchDesc *desc, int32_t *ent, SlotEntry<kCar> *table,
                 int64_t *missing, int32_t *mi_out, int32_t *mn_out, int32_t *mr_out) {
  // rows by their first (lowest) incident element: incidences are sorted
  // by element within a row, so that is the row's first incidence
  std::vector<int32_t> idx(nrows);
  std::vector<int32_t> key(nrows);
  for (int32_t r = 0; r < nrows; ++r) {
    idx[r] = r;
    key[r] = inc_ptr[r + 1] > inc_ptr[r] ? inc_ent[inc_ptr[r]] / rarity : INT32_MAX;
  }
  std::stable_sort(idx.begin(), idx.end(), [&](int32_t x, int32_t y) { return key[x] < key[y]; });
  int32_t nb = 0, mi = 0, mn = 0, mr = 0;
  int64_t pos = 0, miss = 0;
  int32_t k = 0;
  while (k < nrows) {
    const int32_t b0 = k;
    int32_t inc = 0, nnz = 0;
    while (k < nrows) {
      const int32_t r = idx[k];
      const int32_t di = inc_ptr[r + 1] - inc_ptr[r], dn = rowptr[r + 1] - rowptr[r];
      if (k > b0 && (inc + di > max_inc || nnz + dn > max_nnz)) break;
      inc += di;
      nnz += dn;
      ++k;
    }
    if (nnz > 65535 || k - b0 > 65535) {
      set_error("row list: a batch of %d blocks / %d rows exceeds 16-bit offsets", nnz, k - b0);
      return OP2HIP_ERR_ARG;
    }
    BatchDesc d;
    d.r0 = b0;
    d.nr = k - b0;
    d.z0 = 0;
    d.nz = nnz;
    d.i0 = (int32_t)pos;
    d.ni = inc;
    d.pad0 = d.pad1 = 0;
    desc[nb++] = d;
    int32_t zoff = 0;
    for (int32_t q = b0; q < k; ++q) {
      const int32_t r = idx[q];
      row_order[2 * q] = r;
      row_order[2 * q + 1] = zoff;
      const int32_t zlo = rowptr[r], zhi = rowptr[r + 1];
      for (int32_t t = inc_ptr[r]; t < inc_ptr[r + 1]; ++t) {
        const int32_t e = inc_ent[t] / rarity;
        SlotEntry<kCar> s;
        s.row_off = static_cast<uint16_t>(zoff);
        s.lr = static_cast<uint16_t>(q - b0);
        for (int j = 0; j < kCar; ++j) {
          const int32_t c = cmap[(int64_t)e * kCar + j];
          int32_t p = -1;
          if (c >= 0) {
            const int32_t *hit = std::lower_bound(colidx + zlo, colidx + zhi, c);
            if (hit != colidx + zhi && *hit == c) p = int32_t(hit - colidx);
            else ++miss;
          }
          s.slot[j] = (p < 0 || p - zlo > 254) ? uint8_t(255) : static_cast<uint8_t>(p - zlo);
        }
        ent[pos] = inc_ent[t];
        table[pos++] = s;
      }
      zoff += zhi - zlo;
    }
    mi = std::max(mi, inc);
    mn = std::max(mn, nnz);
    mr = std::max(mr, k - b0);
  }
  *nbatches = nb;
  *missing = miss;
  *mi_out = mi;
  *mn_out = mn;
  *mr_out = mr;
  return OP2HIP_OK;
}

template <int kCar>
int plan_cells(int32_t nbatches, const BatchDesc *D, const SlotEntry<kCar> *table, int32_t rarity,
               const int32_t *inc_ent, int32_t *cell_ptr, int32_t *cells, uint8_t *gcount,
               uint16_t *order, int32_t *contrib_ptr, uint16_t *contrib) {
  std::vector<int32_t> es, uniq, cnt, pos, first;
  std::vector<int32_t> idx;
  int64_t cp = 0, gp = 0;
  cell_ptr[0] = 0;
  contrib_ptr[0] = 0;
  for (int32_t b = 0; b < nbatches; ++b) {
    const BatchDesc &d = D[b];
    es.resize(d.ni);
    for (int32_t t = 0; t < d.ni; ++t) es[t] = inc_ent[d.i0 + t] / rarity;
    uniq.assign(es.begin(), es.end());
    std::sort(uniq.begin(), uniq.end());
    uniq.erase(std::unique(uniq.begin(), uniq.end()), uniq.end());
    if (uniq.size() > 256) {
      set_error("cell gather: batch %d has %zu elements (at most 256)", b, uniq.size());
      return OP2HIP_ERR_ARG;
    }
    for (size_t k = 0; k < uniq.size(); ++k) cells[cp + (int64_t)k] = uniq[k];
    cnt.assign(d.nz, 0);
    for (int32_t t = 0; t < d.ni; ++t)
      for (int j = 0; j < kCar; ++j)
        if (table[d.i0 + t].slot[j] != 255) ++cnt[table[d.i0 + t].row_off + table[d.i0 + t].slot[j]];
    idx.resize(d.nz);
    for (int32_t z = 0; z < d.nz; ++z) {
      if (cnt[z] > 255) {
        set_error("cell gather: a block takes %d element blocks (at most 255)", cnt[z]);
        return OP2HIP_ERR_ARG;
      }
      gcount[(int64_t)d.z0 + z] = static_cast<uint8_t>(cnt[z]);
      idx[z] = z;
    }
    std::stable_sort(idx.begin(), idx.end(), [&](int32_t x, int32_t y) { return cnt[x] > cnt[y]; });
    first.assign(d.nz, 0);
    int32_t acc = 0;
    for (int32_t w = 0; w < d.nz; ++w) {
      order[(int64_t)d.z0 + w] = static_cast<uint16_t>(idx[w]);
      first[idx[w]] = acc;
      acc += cnt[idx[w]];
    }
    pos.assign(first.begin(), first.end());
    for (int32_t t = 0; t < d.ni; ++t) {
      const int32_t ent = inc_ent[d.i0 + t];
      const int32_t e = ent / rarity, i = ent - e * rarity;
      const int32_t u = int32_t(std::lower_bound(uniq.begin(), uniq.end(), e) - uniq.begin());
      for (int j = 0; j < kCar; ++j) {
        const uint8_t s = table[d.i0 + t].slot[j];
        if (s == 255) continue;
        contrib[gp + pos[table[d.i0 + t].row_off + s]++] =
            static_cast<uint16_t>((u << 8) | (i << 4) | j);
      }
    }
    cp += (int64_t)uniq.size();
    gp += acc;
    if (cp > INT32_MAX || gp > INT32_MAX) {
      set_error("cell gather: plan exceeds 2^31 entries");
      return OP2HIP_ERR_OVERFLOW;
    }
    cell_ptr[b + 1] = (int32_t)cp;
    contrib_ptr[b + 1] = (int32_t)gp;
  }
  return OP2HIP_OK;
}

}  // namespace op2hip

extern "C" {

int op2hip_slot_table_bytes(int32_t carity, size_t *entry_bytes) {
  OP2HIP_REQUIRE(entry_bytes, "slot_table_bytes: NULL");
  switch (carity) {
    case 3: *entry_bytes = sizeof(SlotEntry<3>); return OP2HIP_OK;
    case 4: *entry_bytes = sizeof(SlotEntry<4>); return OP2HIP_OK;
    case 10: *entry_bytes = sizeof(SlotEntry<10>); return OP2HIP_OK;
    default:
      set_error("slot tables exist for column arities 3, 4 and 10 (got %d)", carity);
      return OP2HIP_ERR_ARG;
  }
}

int op2hip_build_slot_table(int32_t nbatches, const int32_t *batch_rows, const int32_t *rowptr,
                            const int32_t *colidx, const int32_t *inc_ptr, const int32_t *inc_ent,
                            const int32_t *cmap, int32_t rarity, int32_t carity, void *table,
                            void *batch_desc, int32_t *bad, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nbatches >= 0 && batch_rows && rowptr && colidx && inc_ptr && inc_ent && cmap &&
                     table && batch_desc && rarity > 0 && bad,
                 "build_slot_table: bad arguments");
  int rc = fill(bad, 2, 0, s);
  if (rc) return rc;
  if (nbatches > 0) {
    auto *d = static_cast<BatchDesc *>(batch_desc);
    switch (carity) {
      case 3:
        build_slot_table<3><<<nbatches, 64, 0, s>>>(nbatches, batch_rows, rowptr, colidx, inc_ptr,
                                                     inc_ent, cmap, rarity,
                                                     static_cast<SlotEntry<3> *>(table), d, bad);
        break;
      case 4:
        build_slot_table<4><<<nbatches, 64, 0, s>>>(nbatches, batch_rows, rowptr, colidx, inc_ptr,
                                                     inc_ent, cmap, rarity,
                                                     static_cast<SlotEntry<4> *>(table), d, bad);
        break;
      case 10:
        build_slot_table<10><<<nbatches, 64, 0, s>>>(nbatches, batch_rows, rowptr, colidx, inc_ptr,
                                                      inc_ent, cmap, rarity,
                                                      static_cast<SlotEntry<10> *>(table), d, bad);
        break;
      default:
        set_error("slot tables exist for column arities 3, 4 and 10 (got %d)", carity);
        return OP2HIP_ERR_ARG;
    }
    OP2HIP_LAUNCHED();
  }
  return OP2HIP_OK;
}

int op2hip_plan_row_list(int32_t nrows, const int32_t *rowptr, const int32_t *colidx,
                         const int32_t *inc_ptr, const int32_t *inc_ent, const int32_t *cmap,
                         int32_t rarity, int32_t carity, int32_t max_inc, int32_t max_nnz,
                         int32_t *row_order, int32_t *nbatches, void *desc, int32_t *ent,
                         void *table, int64_t *missing, int32_t *max_inc_out,
                         int32_t *max_nnz_out, int32_t *max_rows_out) {
  OP2HIP_REQUIRE(nrows >= 0 && rowptr && colidx && inc_ptr && inc_ent && cmap && rarity > 0 &&
                     max_inc > 0 && max_nnz > 0 && row_order && nbatches && desc && ent && table &&
                     missing && max_inc_out && max_nnz_out && max_rows_out,
                 "plan_row_list: bad arguments");
  auto *D = static_cast<BatchDesc *>(desc);
  switch (carity) {
    case 3:
      return plan_rowlist<3>(nrows, rowptr, colidx, inc_ptr, inc_ent, cmap, rarity, max_inc,
                             max_nnz, row_order, nbatches, D, ent,
                             static_cast<SlotEntry<3> *>(table), missing, max_inc_out,
                             max_nnz_out, max_rows_out);
    case 4:
      return plan_rowlist<4>(nrows, rowptr, colidx, inc_ptr, inc_ent, cmap, rarity, max_inc,
                             max_nnz, row_order, nbatches, D, ent,
                             static_cast<SlotEntry<4> *>(table), missing, max_inc_out,
                             max_nnz_out, max_rows_out);
    case 10:
      return plan_rowlist<10>(nrows, rowptr, colidx, inc_ptr, inc_ent, cmap, rarity, max_inc,
                              max_nnz, row_order, nbatches, D, ent,
                              static_cast<SlotEntry<10> *>(table), missing, max_inc_out,
                              max_nnz_out, max_rows_out);
    default:
      set_error("row lists exist for column arities 3, 4 and 10 (got %d)", carity);
      return OP2HIP_ERR_ARG;
  }
}

int op2hip_plan_cell_gather(int32_t nbatches, const void *batch_desc, const void *table,
                            int32_t rarity, int32_t carity, const int32_t *inc_ent,
                            int32_t *cell_ptr, int32_t *cells, uint8_t *gcount, uint16_t *order,
                            int32_t *contrib_ptr, uint16_t *contrib) {
  OP2HIP_REQUIRE(nbatches >= 0 && batch_desc && table && inc_ent && cell_ptr && cells && gcount &&
                     order && contrib_ptr && contrib && rarity > 0 && rarity <= 16,
                 "plan_cell_gather: bad arguments");
  const auto *D = static_cast<const BatchDesc *>(batch_desc);
  switch (carity) {
    case 3:
      return plan_cells<3>(nbatches, D, static_cast<const SlotEntry<3> *>(table), rarity, inc_ent,
                           cell_ptr, cells, gcount, order, contrib_ptr, contrib);
    case 4:
      return plan_cells<4>(nbatches, D, static_cast<const SlotEntry<4> *>(table), rarity, inc_ent,
                           cell_ptr, cells, gcount, order, contrib_ptr, contrib);
    case 10:
      return plan_cells<10>(nbatches, D, static_cast<const SlotEntry<10> *>(table), rarity,
                            inc_ent, cell_ptr, cells, gcount, order, contrib_ptr, contrib);
    default:
      set_error("cell gather plans exist for column arities 3, 4 and 10 (got %d)", carity);
      return OP2HIP_ERR_ARG;
  }
}

int op2hip_task_plan_count(int32_t nbatches, const void *batch_desc, const uint8_t *gcount,
                           const int32_t *inc_ent, int32_t rarity, int32_t *counts,
                           void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nbatches >= 0 && batch_desc && gcount && inc_ent && rarity > 0 && counts,
                 "task_plan_count: bad arguments");
  const int rc = fill(counts + 3 * (int64_t)nbatches, 1, 0, s);
  if (rc || nbatches == 0) return rc;
  task_plan_kernel<false><<<nbatches, 256, 0, s>>>(
      nbatches, static_cast<const BatchDesc *>(batch_desc), gcount, nullptr, inc_ent, rarity, 1,
      nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, counts);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_task_plan_fill(int32_t nbatches, const void *batch_desc, const uint8_t *gcount,
                          const uint16_t *glist, const int32_t *inc_ent, int32_t rarity,
                          int32_t carity, const int32_t *first_cell, const int32_t *first_word,
                          const int32_t *first_multi, int32_t *cells, uint32_t *tasks,
                          uint16_t *multis, void *desc, void *stream) {
  OP2HIP_REQUIRE(nbatches >= 0 && batch_desc && gcount && glist && inc_ent && rarity > 0 &&
                     carity > 0 && rarity * carity <= 128 && first_cell && first_word &&
                     first_multi && cells && tasks && multis && desc,
                 "task_plan_fill: bad arguments");
  if (nbatches == 0) return OP2HIP_OK;
  task_plan_kernel<true><<<nbatches, 256, 0, stream_of(stream)>>>(
      nbatches, static_cast<const BatchDesc *>(batch_desc), gcount, glist, inc_ent, rarity, carity,
      first_cell, first_word, first_multi, cells, tasks, multis,
      static_cast<TaskDesc *>(desc), nullptr);
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_gather_table_count(int32_t nbatches, int32_t batch_max_nnz, const void *batch_desc,
                              const void *table, int32_t carity, uint8_t *gcount,
                              int32_t *batch_total, int32_t *over, void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nbatches >= 0 && batch_desc && table && gcount && batch_total && over,
                 "gather_table_count: bad arguments");
  OP2HIP_REQUIRE(batch_max_nnz <= kGatherMaxBlocks,
                 "gather tables take batches of at most %d blocks (got %d)", kGatherMaxBlocks,
                 batch_max_nnz);
  int rc = fill(over, 1, 0, s);
  if (rc || nbatches == 0) return rc;
  const auto *d = static_cast<const BatchDesc *>(batch_desc);
  switch (carity) {
    case 3:
      gather_count_kernel<3><<<nbatches, 256, 0, s>>>(
          nbatches, d, static_cast<const SlotEntry<3> *>(table), gcount, batch_total, over);
      break;
    case 4:
      gather_count_kernel<4><<<nbatches, 256, 0, s>>>(
          nbatches, d, static_cast<const SlotEntry<4> *>(table), gcount, batch_total, over);
      break;
    case 10:
      gather_count_kernel<10><<<nbatches, 256, 0, s>>>(
          nbatches, d, static_cast<const SlotEntry<10> *>(table), gcount, batch_total, over);
      break;
    default:
      set_error("gather tables exist for column arities 3, 4 and 10 (got %d)", carity);
      return OP2HIP_ERR_ARG;
  }
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

int op2hip_gather_table_fill(int32_t nbatches, int32_t batch_max_nnz, void *batch_desc,
                             const void *table, int32_t carity, const int32_t *batch_off,
                             const int32_t *batch_total, const uint8_t *gcount, uint16_t *glist,
                             void *stream) {
  hipStream_t s = stream_of(stream);
  OP2HIP_REQUIRE(nbatches >= 0 && batch_desc && table && batch_off && batch_total && gcount &&
                     glist,
                 "gather_table_fill: bad arguments");
  OP2HIP_REQUIRE(batch_max_nnz <= kGatherMaxBlocks,
                 "gather tables take batches of at most %d blocks (got %d)", kGatherMaxBlocks,
                 batch_max_nnz);
  if (nbatches == 0) return OP2HIP_OK;
  auto *d = static_cast<BatchDesc *>(batch_desc);
  switch (carity) {
    case 3:
      gather_fill_kernel<3><<<nbatches, 256, 0, s>>>(nbatches, d,
                                                      static_cast<const SlotEntry<3> *>(table),
                                                      batch_off, batch_total, gcount, glist);
      break;
    case 4:
      gather_fill_kernel<4><<<nbatches, 256, 0, s>>>(nbatches, d,
                                                      static_cast<const SlotEntry<4> *>(table),
                                                      batch_off, batch_total, gcount, glist);
      break;
    case 10:
      gather_fill_kernel<10><<<nbatches, 256, 0, s>>>(nbatches, d,
                                                       static_cast<const SlotEntry<10> *>(table),
                                                       batch_off, batch_total, gcount, glist);
      break;
    default:
      set_error("gather tables exist for column arities 3, 4 and 10 (got %d)", carity);
      return OP2HIP_ERR_ARG;
  }
  OP2HIP_LAUNCHED();
  return OP2HIP_OK;
}

}  // extern "C"
