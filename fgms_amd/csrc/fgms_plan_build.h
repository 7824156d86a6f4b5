// What the two ways to a plan share: from a caller's pair lists (fgms_plan.hip) and together with
// the map itself from voxel coordinates (fgms_kmap.hip).  Both end in the same row masks; from
// there on the row order, the tables and the dispatch orders are built by the launches declared here.
#pragma once

#include "fgms_device.h"
#include "fgms_internal.h"

namespace fgms {

// Blocks of one pool allocation, laid out by running the same `take` calls twice: without a base
// to add the sizes up, then with it.  (One block per build: a pool block costs two runtime calls
// on its way out and two on its way back.)
struct Arena {
  char *base = nullptr;
  size_t used = 0;
  template <typename T>
  void take(T *&p, size_t count) {
    p = base ? reinterpret_cast<T *>(base + used) : nullptr;
    used += (count * sizeof(T) + 255) & ~(size_t)255;
  }
};

// ---- fills of a build, all in one launch
struct FillRange {
  int32_t *p;
  size_t n;
  int32_t v;
};
struct FillBatch {
  FillRange range[6];
  int count;
  void add(void *p, size_t bytes, int32_t v) {
    if (bytes) range[count++] = FillRange{(int32_t *)p, bytes / 4, v};
  }
};
int launch_fills(const FillBatch &batch, hipStream_t s);

// ---- row order (see fgms_plan.hip)
struct SortSide {
  const unsigned long long *rmask;   // per row: the offsets it has a pair in
  unsigned long long *key;           // what the row is sorted by (sort_key); written with the histogram
  int32_t *perm_tmp;                 // order after the counting sort
  int32_t *perm;                     // final order: position -> row
  int32_t *inv;                      // row -> position
  int32_t *hist;                     // [chunks][kBins] rows per (chunk, bin)
  int32_t *hist_before;              // [chunks][kBins] rows of the bin in earlier chunks
  int32_t *bin_start;                // [kBins] rows per bin
  unsigned long long *block_mask;    // OR of the masks of every 64 positions
  int32_t *nbr;                      // the side's table (the middle offset's line, see Plan::centre_line)
  int n, chunks;                     // chunks == 0: one window, no counting sort
};
struct SortArgs {
  SortSide side[2];                  // output side, input side (n == 0: none)
  int k_vol;
  const int32_t *kpos;
  int *flags;
  bool by_mask;                      // false: natural order
};
constexpr int kBinBits = 13;
constexpr int kBins = 1 << kBinBits;
constexpr int kChunk = 2048;         // rows per workgroup of the histogram / scatter kernels
constexpr int kWindow = 1024;        // positions per workgroup of the window sort
constexpr int kSortThreads = 1024;
constexpr int kWindowThreads = kWindow / 2;

// An odd number of offsets without pairs in the middle one (-1: otherwise).
__device__ __forceinline__ int empty_centre(const int32_t *__restrict__ kpos, int k_vol) {
  const int mid = k_vol / 2;
  return k_vol % 2 == 1 && kpos[mid] == kpos[mid + 1] ? mid : -1;
}

// Bin of a key.
__device__ __forceinline__ int top_bits(unsigned long long key, int k_vol) {
  const int shift = k_vol > kBinBits ? k_vol - kBinBits : 0;
  return (int)((key >> shift) & (kBins - 1));
}

// The order of the offsets in a sort key, most significant first: by the number of their pairs,
// rarest first.  `order`: 64 bytes of LDS; the caller's barrier publishes it.  (A lane per offset, compared through
// shuffles: one trip to memory instead of one per offset.)
__device__ __forceinline__ void sort_offset_order(const int32_t *__restrict__ kpos, int k_vol, unsigned char *order) {
  const int k = threadIdx.x;
  if (k >= 64) return;
  const int mine = k < k_vol ? kpos[k + 1] - kpos[k] : 0;
  int rank = 0;
  for (int o = 0; o < k_vol; ++o) {
    const int theirs = __shfl(mine, o);
    rank += theirs < mine || (theirs == mine && o < k) ? 1 : 0;
  }
  if (k < k_vol) order[rank] = (unsigned char)k;
}

// A row's place among all sets of offsets: the set as a number whose high bits are the rare offsets,
// counted in Gray code, so that sets next to each other differ in few offsets.  Rows that have a rare
// offset are few: kept together they load few blocks with it.  (Counted with bins and
// windows of the sort's sizes, 64-row blocks x offsets over pairs / 64 on 120 k LiDAR voxels: by the mask
// as a number 1.39, rarest first 1.30, in Gray code too 1.28; 256-row tiles x offsets over pairs / 256
// 1.62, 1.47, 1.45; on 200 k indoor voxels 1.13, 1.12, 1.11 and 1.32, 1.28, 1.25.)
template <int N>
__device__ __forceinline__ void sort_keys(unsigned long long (&mask)[N], int k_vol, const unsigned char *order) {
  unsigned long long key[N] = {};
  for (int b = 0; b < k_vol; ++b) {
    const int bit = order[b];
#pragma unroll
    for (int r = 0; r < N; ++r) key[r] = key[r] << 1 | (mask[r] >> bit & 1);
  }
#pragma unroll
  for (int r = 0; r < N; ++r) {
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) key[r] ^= key[r] >> s;
    mask[r] = key[r];
  }
}
__device__ __forceinline__ unsigned long long sort_key(unsigned long long mask, int k_vol, const unsigned char *order) {
  unsigned long long key[1] = {mask};
  sort_keys<1>(key, k_vol, order);
  return key[0];
}

// Keys and rows per bin of one chunk; `hist`: kBins ints of LDS.  A thread's rows are loaded and turned into keys side by
// side, not one after the other: latencies bound this, not bytes.  (Launch of the lists and the histogram, together with
// the offsets' order from shuffles and the list blocks' loads in flight together: 27 offsets over 100 k LiDAR voxels 14.5 -> 13.0
// us, over the 30 k of the next level 13.3 -> 10.7, the 8 between them 10.2 -> 8.1.)
template <int THREADS>
__device__ __forceinline__ void sort_hist_body(const SortSide &sd, const SortArgs &a, int chunk, int *hist) {
  constexpr int kRows = kChunk / THREADS;
  __shared__ unsigned char order[64];
  const int first = chunk * kChunk + threadIdx.x;
  unsigned long long key[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) key[r] = first + r * THREADS < sd.n ? sd.rmask[first + r * THREADS] : 0ull;
  sort_offset_order(a.kpos, a.k_vol, order);
  for (int i = threadIdx.x; i < kBins; i += THREADS) hist[i] = 0;
  __syncthreads();
  sort_keys<kRows>(key, a.k_vol, order);
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    if (first + r * THREADS >= sd.n) break;
    sd.key[first + r * THREADS] = key[r];
    atomicAdd(&hist[top_bits(key[r], a.k_vol)], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kBins; i += THREADS) sd.hist[(size_t)chunk * kBins + i] = hist[i];
}

// Lays out a side's temporaries.
void sort_side_layout(SortSide &sd, int64_t n, Arena &tmp);
// Histogram (unless the caller's own launch took it), scan, scatter, window sort.
int launch_sort(const SortArgs &a, bool hist_done, hipStream_t s);

// Weight-gradient row bands: 8, 16, 32 or 64 (the XCDs take them in groups of 1, 2, 4 or 8;
// other counts measured worse), the fewest that leave an (offset, band) cell at most ~1 900
// pairs -- a workgroup's fixed costs (first loads, the four waves' partial tiles summed through
// LDS, 16 KB of atomic updates) are those of ~600 pairs, and with bigger cells the chip waits
// for the last ones -- then more while the cells are fewer than 1.5 per CU and keep ~400 pairs.
// 64 -> 64 fp16 backward launch with 64 bands throughout / with this rule: 50 k voxels 35.5 /
// 29.8 us, 80 k 55.6 / 45.2, 100 k 59.1 / 46.2, 120 k 61.5 / 55.6, 140 k 67.7 / 65.3 (32 bands
// each), 170 k and 200 k voxels 64 bands either way.
__host__ __device__ inline int band_count_of(int64_t n_pairs, int k_vol, int cus) {
  constexpr int kMaxBands = 64;
  int bands = 8;
  while (bands < kMaxBands && n_pairs / ((int64_t)k_vol * bands) > 1900) bands *= 2;
  while (bands < kMaxBands && (int64_t)bands * k_vol * 2 < 3 * (int64_t)cus && n_pairs / ((int64_t)k_vol * bands * 2) >= 384)
    bands *= 2;
  return bands;
}

// ---- the last launch of a build: tables by position, row bands, tile order, findings
struct TileSide {
  const int32_t *perm;
  const unsigned long long *block_masks;
  int32_t *order;                    // nullptr: none
  int n_rows, n_tiles, cap;
};
struct TablesArgs {
  const int32_t *kpos, *imap, *omap;
  int k_vol, n_pairs, n_in, n_out;
  // from the pair lists: position -> neighbour through offset k (tables pre-filled with -1; nullptr: not this one)
  const int32_t *inv_out, *inv_in;
  int32_t *nbr_out, *nbr_in;
  // from a table of the output rows, [n_out][row_ld] (nbr_in: where inv_in is given)
  const int32_t *rows;
  const int32_t *perm_out;
  int row_ld;
  // bands
  int32_t *band_start, *band_cells;
  int bands, band_rows;              // (bands == 0: as many as the pairs in kpos ask for, on `cus` compute units)
  bool bands_known;                  // band_start is filled in already
  TileSide tile[2];
  int cus;
  int *flags, *host;                 // findings and where they go on the host (nullptr: a copy follows)
  bool mirror, take_print;           // one side's counts stand for both; fingerprint of the lists
  // workgroups of each part, in this order
  int tile_blocks, band_blocks, print_blocks, row_blocks, pair_blocks;
};
int launch_tables(TablesArgs a, hipStream_t s);

// A plan from pair lists (fgms_plan_create; want_bands: with the weight gradient's row bands).
int plan_create(fgms_plan_t **plan, const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int64_t n_in,
                int64_t n_out, int k_vol, int64_t n_pairs, void *stream, bool want_bands);
// Plan objects without their tables.
Plan *plan_alloc(int k_vol, int64_t n_in, int64_t n_out, int64_t n_pairs, hipStream_t s);
void plan_bands(Plan *p);                                // band_count / band_rows from the sizes
int tile_table(int64_t n, int *cap);                     // tiles of a side that gets a table, else 0
void plan_fill_tables_args(const Plan *p, TablesArgs *t);
int plan_publish(Plan *p, bool written, hipStream_t s);  // findings on their way to the host, `ready` recorded

}  // namespace fgms
