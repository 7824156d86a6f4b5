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

// Lays out a side's temporaries.
void sort_side_layout(SortSide &sd, int64_t n, Arena &tmp);
bool plan_sorts_rows();                                  // false: rows stay in their natural order
int launch_sort_scatter(const SortArgs &a, hipStream_t s);
// Histogram, scan, scatter, window sort.
int launch_sort(const SortArgs &a, hipStream_t s);

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
