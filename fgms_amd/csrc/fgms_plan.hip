// Kernel-map plan: neighbour tables built on the device from the pair lists.
// nbr_out[k][o] = the input row that reaches output row o through offset k
// (-1 if none); nbr_in[k][i] = the output row that input row i reaches through
// offset k.  Offset-major, so a wave reads the entries of its 64 consecutive
// rows for one offset as one 256-byte line.  The reference keeps only the pair lists and scatters with atomics
// (backend/spconv.cuh:457-563); the tables let a workgroup own a block of
// output rows and sum all offsets in registers.
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>
#include <vector>

#include "fgms_device.h"
#include "fgms_internal.h"
#include "fgms_plan_build.h"
#include "fgms_plan_sort.h"

namespace fgms {
namespace {

__global__ __launch_bounds__(256) void fills_kernel(FillBatch batch) {
  typedef int int4v_ __attribute__((ext_vector_type(4)));
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
  for (int r = 0; r < batch.count; ++r) {
    const FillRange &f = batch.range[r];       // (16-byte aligned: pool blocks and what an Arena cuts from them)
    const int32_t v = f.v;
    for (size_t q = i; q < f.n / 4; q += stride) reinterpret_cast<int4v_ *>(f.p)[q] = int4v_{v, v, v, v};
    if (i < f.n % 4) f.p[f.n / 4 * 4 + i] = v;
  }
}

// flags[0]: an index is out of range; flags[1]: two pairs of one offset share
// an output row; flags[2]: two pairs of one offset share an input row;
// flags[3]: inside some offset the pairs are not ordered by output row;
// flags[4], flags[5]: (64-position block, offset) combinations in use, output / input side;
// flags[6..8]: unused; flags[9]: see kFlagInput; flags[10], flags[11]: offset bits
// set over all row masks of the output / input side; flags[12]: pairs in the map.  Two pairs of
// one offset that share a row set one bit between them, so a side whose bits do not add up to
// the pair count has such a pair (what flags[1] / flags[2] used to say).
//
// Step 1 of a plan: per row the set of offsets it has a pair in (bit k of rmask), both
// sides at once, straight from the pair lists.  An offset bit that is already set when a
// pair wants to set it means two pairs of that offset share the row.
__global__ void pair_masks_kernel(const int32_t *__restrict__ kpos, const int32_t *__restrict__ imap,
                                  const int32_t *__restrict__ omap, int k_vol, int n_pairs, int n_in,
                                  int n_out, unsigned long long *__restrict__ rmask_out,
                                  unsigned long long *__restrict__ rmask_in, int *__restrict__ flags,
                                  int32_t *__restrict__ band_start, int bands, int band_rows) {
  const int total = kpos[k_vol];
  if (blockIdx.x < kPrintParts) {
    // the launch's first workgroups take the fingerprint of the lists (fgms_plan_check re-takes
    // it); first, so that their chain of loads runs next to the others' work, not behind it
    plan_print_block(kpos, imap, omap, k_vol, n_pairs, flags, blockIdx.x);
    return;
  }
  const int j = kpos[0] + (blockIdx.x - kPrintParts) * blockDim.x + threadIdx.x;      // (kpos[0] > 0: a plan over a slice of the offsets)
  if (j >= total || j >= n_pairs) return;
  int lo = 0, hi = k_vol;          // offset of pair j: the last k with kpos[k] <= j
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (kpos[mid] <= j) lo = mid; else hi = mid;
  }
  const int k = lo;
  const int i = imap[j], o = omap[j];
  if (j == kpos[0]) flags[12] = min(total, n_pairs) - kpos[0];
  if (i < 0 || i >= n_in || o < 0 || o >= n_out) {
    flags[0] = 1;
    return;
  }
  const int before = j > kpos[k] ? omap[j - 1] : -1;
  if (before > o) flags[3] = 1;
  if (i != j - kpos[k] && kpos[k + 1] - kpos[k] == n_in) flags[kFlagInput] = 1;
  // the bounds of the weight gradient's row bands that fall between this pair and the one before it
  // (pre-set to 0; meaningful where the pairs are ordered by output row, in bounds always)
  if (band_start) {
    int32_t *row = band_start + k * (bands + 1);
    const int here = o / band_rows;
    for (int c = before < 0 ? 0 : before / band_rows + 1; c <= here; ++c) row[c] = j - kpos[k];
    if (j + 1 == min(min(kpos[k + 1], total), n_pairs))
      for (int c = here + 1; c <= bands; ++c) row[c] = j + 1 - kpos[k];
  }
  // the 32-bit half of the mask that holds bit k (little-endian words); the old value is not
  // asked for, so the atomics need no reply
  const unsigned bit = 1u << (k & 31);
  (void)__hip_atomic_fetch_or(reinterpret_cast<unsigned *>(rmask_out + o) + (k >> 5), bit, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
  (void)__hip_atomic_fetch_or(reinterpret_cast<unsigned *>(rmask_in + i) + (k >> 5), bit, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
}

// Step 2: the order in which a side's rows are visited.  Rows are sorted by the set of their offsets
// (sort_key), so that the 64 rows of a wave and the 256 of a workgroup use nearly the same offsets and
// whole (block, offset) steps can be skipped: on a surface-like cloud of 200 k voxels the number of
// such steps drops from 68.6 k to 36.3 k (33 k would be perfect).  Close keys share their high bits,
// which is what makes neighbours in the order similar; so the sort runs most
// significant bits first: a counting sort on the top kBinBits bits of the key over the whole
// side (histogram per chunk of rows, scan, stable scatter), then a full sort by (key, row) of
// every window of kWindow positions.  Inside a bin only rows of one window are ordered
// among themselves; that costs 1.5 % more (block, offset) steps than the exact sort on 200 k indoor
// voxels, 2 % on 120 k LiDAR voxels and 28 % on 50 k scattered ones (windows of 2048: 0.5 %, 0.7 % and
// 7 % fewer steps).  Both sides of a plan go through the same
// launches (blockIdx.y = side).
__global__ __launch_bounds__(kSortThreads) void sort_hist_kernel(SortArgs a) {
  const SortSide &sd = a.side[blockIdx.y];
  if ((int)blockIdx.x >= sd.chunks) return;
  __shared__ int hist[kBins];
  sort_hist_body(sd, a, blockIdx.x, hist, [] { return (const int *)nullptr; });
}

__global__ __launch_bounds__(256) void sort_scan_kernel(SortArgs a) { sort_scan_body(a.side[blockIdx.y], blockIdx.x); }

__global__ __launch_bounds__(kSortThreads) void sort_scatter_kernel(SortArgs a) {
  __shared__ int next[kBins];
  if ((int)blockIdx.x < a.side[blockIdx.y].chunks) sort_scatter_body(a.side[blockIdx.y], a, blockIdx.x, next);
}

__global__ __launch_bounds__(kWindowThreads) void sort_window_kernel(SortArgs a) {
  __shared__ unsigned long long buf[2 * kWindow];
  sort_window_body(a, blockIdx.y, blockIdx.x, buf);
}

// Pair view: the pair lists with every offset's run padded to a multiple of 64 rows
// (pv_in / pv_out pre-filled with -1, pv_mask with 0).  Pair j of offset k goes to row
// vpos[k] + j - kpos[k], vpos = the running sum of the padded run lengths.
__global__ void pair_view_kernel(const int32_t *__restrict__ kpos, const int32_t *__restrict__ imap,
                                 const int32_t *__restrict__ omap, int k_vol, int n_pairs,
                                 long long pv_rows, int32_t *__restrict__ pv_in,
                                 int32_t *__restrict__ pv_out,
                                 unsigned long long *__restrict__ pv_mask) {
  __shared__ int kp[65];
  __shared__ long long vp[65];
  if ((int)threadIdx.x <= k_vol) kp[threadIdx.x] = kpos[threadIdx.x];
  __syncthreads();
  if (threadIdx.x == 0) {
    long long v = 0;
    for (int k = 0; k < k_vol; ++k) {
      vp[k] = v;
      const int n = kp[k + 1] - kp[k];
      if (n > 0) v += (n + 63) / 64 * 64;
    }
    vp[k_vol] = v;
  }
  __syncthreads();
  const int j = kp[0] + blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= kp[k_vol] || j >= n_pairs) return;
  int lo = 0, hi = k_vol;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (kp[mid] <= j) lo = mid; else hi = mid;
  }
  const long long r = vp[lo] + (j - kp[lo]);
  if (j < kp[lo] || r < 0 || r >= pv_rows) return;     // (a kpos that does not ascend)
  pv_in[r] = imap[j];
  pv_out[r] = omap[j];
  if ((r & 63) == 0) pv_mask[r >> 6] = 1ull << lo;
}

// Dispatch order of the 256-position tiles of the output-stationary kernel.
// Workgroup b runs on XCD b % 8 and, inside an XCD, workgroup number q = b / 8
// lands on CU q % cus_per_xcd (the dispatcher goes round the CUs).
//  * A tile's weight is the number of offsets it uses and a little for its start and end.
//  * A tile's home XCD is the eighth of the cloud's weight its middle row lies in
//    (original row numbers follow the voxel order, i.e. space), so that
//    neighbouring rows meet in one L2 and the XCDs get equal work.
//  * Inside an XCD the tiles are ranked by weight, heaviest first: those must start first.  The
//    first kHeadRounds tiles of a CU are resident together, so the launch lasts as long as the
//    heaviest such sum: in every round the heaviest tile goes to the CU with the least so far.
//    Tiles behind those go to whichever CU has room.
//  * Every XCD takes at most cap tiles (tile_table); the lightest tiles of an
//    overfull XCD go to the XCDs that have room.
// Counted on 200 k indoor / 120 k LiDAR voxels, offsets of the busiest CU (the mean is 40 / 31): with
// eighths of the rows and a snake over the CUs 60 / 43, like this 48 / 37; 64 -> 64 over the former fp16
// forward 41.2 -> 40.1 us, in tf32 mode 110.7 -> 104.7, 128 -> 128 fp16 over the latter 82.0 -> 79.9.
// order[q * 8 + xcd] = tile | first offset << 24, -1 where no tile lands.  One workgroup; which of two
// equally heavy tiles comes first depends on timing, the results do not.
constexpr int kHeadRounds = 3, kHeadCus = 32, kHomeBuckets = 512;
__device__ __forceinline__ void tile_order_body(const TileSide &sd, int cus_per_xcd, int32_t *__restrict__ tiles) {
  const int32_t *__restrict__ perm = sd.perm;
  const unsigned long long *__restrict__ block_masks = sd.block_masks;
  int32_t *__restrict__ order = sd.order;
  const int n_rows = sd.n_rows, n_tiles = sd.n_tiles, cap = sd.cap;
  if (!order) return;
  constexpr int kPc = 65;                         // popcount classes 0..64
  __shared__ int rank_of[8][kPc];                 // tiles per (home, popcount), then the next rank of each
  __shared__ int total[8];
  __shared__ int before[kHomeBuckets];            // weight by middle row, then that in front of it
  __shared__ unsigned short head[8][kHeadRounds * kHeadCus];     // the first tiles by rank
  __shared__ int wave_sum[4];
  __shared__ int spill_count;
  const int tid = threadIdx.x, threads = blockDim.x;     // (256 threads)
  const int n_blocks = (n_rows + 63) / 64;
  const int head_ranks = cus_per_xcd <= kHeadCus ? min(kHeadRounds * cus_per_xcd, cap) : 0;
  constexpr unsigned short kNoTile = 0xffff;             // (tile_table: at most 15000 tiles)
  for (int i = tid; i < 8 * kPc; i += threads) (&rank_of[0][0])[i] = 0;
  for (int i = tid; i < kHomeBuckets; i += threads) before[i] = 0;
  for (int i = tid; i < 8 * kHeadRounds * kHeadCus; i += threads) (&head[0][0])[i] = kNoTile;
  if (tid == 0) spill_count = 0;
  for (int i = tid; i < cap * 8; i += threads) order[i] = -1;     // (slots no tile lands in)
  __syncthreads();
  // tiles[t] (n_tiles ints of LDS): number of offsets, first offset << 7, bucket or home << 13
  auto count_of = [](int info) { return info & 127; };
  auto weight_of = [](int info) { return (info & 127) + 2; };
  // entry of tile t in the table: t in the low 24 bits, the first offset the tile uses above
  // them (the kernel starts that offset's index load before it has seen the tile's masks)
  auto entry_of = [](int t, int info) { return t | (info >> 7 & 63) << 24; };
  for (int t = tid; t < n_tiles; t += threads) {
    const int mid = min(t * 256 + 128, n_rows - 1);
    const int bucket = (int)((long long)(perm ? perm[mid] : mid) * kHomeBuckets / n_rows);
    unsigned long long m = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) m |= block_masks[min(4 * t + q, n_blocks - 1)];
    const int info = __builtin_popcountll(m) | (m ? __builtin_ctzll(m) : 0) << 7 | bucket << 13;
    tiles[t] = info;
    atomicAdd(&before[bucket], weight_of(info));
  }
  __syncthreads();
  // weight in front of the middle of each bucket
  int all = 0;
  {
    constexpr int kPer = kHomeBuckets / 256;
    int w[kPer], sum = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) { w[i] = before[tid * kPer + i]; sum += w[i]; }
    int incl = sum;
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d);
      if (tid % 64 >= d) incl += up;
    }
    if (tid % 64 == 63) wave_sum[tid / 64] = incl;
    __syncthreads();
    int run = incl - sum;
    for (int q = 0; q < 4; ++q) {
      if (q < tid / 64) run += wave_sum[q];
      all += wave_sum[q];
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      before[tid * kPer + i] = run + w[i] / 2;
      run += w[i];
    }
  }
  __syncthreads();
  for (int t = tid; t < n_tiles; t += threads) {
    const int info = tiles[t];
    const int home = min(7, before[info >> 13] * 8 / max(all, 1));
    tiles[t] = (info & 0x1fff) | home << 13;
    atomicAdd(&rank_of[home][count_of(info)], 1);
  }
  __syncthreads();
  // start rank of each class, heaviest first: a wave per home, lane l takes class 64 - l
  for (int home = tid / 64; home < 8; home += threads / 64) {
    const int lane = tid % 64, pc = 64 - lane;
    const int n = rank_of[home][pc];
    int incl = n;
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    rank_of[home][pc] = incl - n;
    if (lane == 63) {
      const int n0 = rank_of[home][0];
      rank_of[home][0] = incl;
      total[home] = incl + n0;
    }
  }
  __syncthreads();
  auto place = [&](int home, int rank, int t, int info) {
    if (rank < head_ranks) head[home][rank] = (unsigned short)t;
    else order[rank * 8 + home] = entry_of(t, info);
  };
  constexpr int kSpilled = 1 << 16;
  for (int t = tid; t < n_tiles; t += threads) {
    const int info = tiles[t], home = info >> 13;
    const int rank = atomicAdd(&rank_of[home][count_of(info)], 1);
    if (rank < cap) place(home, rank, t, info);
    else tiles[t] = info | kSpilled;
  }
  __syncthreads();
  for (int t = tid; t < n_tiles; t += threads) {
    const int info = tiles[t];
    if (!(info & kSpilled)) continue;
    int left = atomicAdd(&spill_count, 1);
    for (int q = 0; q < 8; ++q) {
      const int filled = min(total[q], cap), room = cap - filled;
      if (left < room) {
        place(q, filled + left, t, info);
        break;
      }
      left -= room;
    }
  }
  __syncthreads();
  // the head: half a wave per home, a lane per CU
  {
    const int home = tid / 32, lane = tid % 32;
    int sum = 0;
    for (int first = 0; first < head_ranks; first += cus_per_xcd) {
      const int n = min(cus_per_xcd, head_ranks - first);
      int nth = 0;                                   // CUs of this round with less so far
      for (int o = 0; o < n; ++o) {
        const int theirs = __shfl(sum, o, 32);
        nth += theirs < sum || (theirs == sum && o < lane) ? 1 : 0;
      }
      if (lane < n) {
        const int t = head[home][first + nth];
        if (t != kNoTile) {
          order[(first + lane) * 8 + home] = entry_of(t, tiles[t]);
          sum += weight_of(tiles[t]);
        }
      }
    }
  }
}

// Row bands of the weight gradient and the dispatch order of its (offset, band) cells.
// band_start[k][c] = number of pairs of offset k whose output row is below c * band_rows (a lower
// bound over the offset's pairs, which are ordered by output row when the result is used);
// c = bands gives the offset's size.  Cell orders: one table per group size g in {1, 2, 4, 8}:
// cells[q * 8 + xcd] is the q-th cell of XCD xcd, cell = offset * 65536 + band.  XCD x owns the
// bands x, x + 8, ...; they are taken g at a time (g bands x all offsets are in flight together, so
// g is chosen at launch such that their rows fit the XCD's L2), and inside a group the cells
// are ranked by pair count, most first (the longest workgroups start first), ties
// by cell number.  Workgroup (x, shift) ranks XCD x's cells in groups of 1 << shift bands by
// comparing each with the others (a few hundred).  The bounds are there already (`bands_known`: the
// mask pass over the lists or the map builder left them), or -- plans over more than 64 offsets -- the
// workgroup finds them by bisection and the one with shift 0 writes them down.
__device__ __forceinline__ void bands_body(const TablesArgs &a, int x, int shift, int32_t *__restrict__ lds) {
  const int k_vol = a.k_vol, bands = a.bands ? a.bands : band_count_of(a.kpos[a.k_vol], a.k_vol, a.cus);
  const int per_xcd = (bands / 8) * k_vol;
  // [per_xcd], the last four's worth rounded up: the smaller, the earlier
  unsigned *key = reinterpret_cast<unsigned *>(lds);
  const int padded = (per_xcd + 3) & ~3;
  auto below = [&](int first, int n, long long target) {      // first pair with omap >= target
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (a.omap[first + mid] < target) lo = mid + 1; else hi = mid;
    }
    return lo;
  };
  for (int o = threadIdx.x; o < per_xcd; o += blockDim.x) {     // cell number inside the XCD: (band / 8) * k_vol + k
    const int k = o % k_vol, q = o / k_vol, band = q * 8 + x;
    const int first = min(max(a.kpos[k], 0), a.n_pairs);
    const int n = min(max(a.kpos[k + 1], first), a.n_pairs) - first;   // never reads past the map
    int b0, b1;
    if (a.bands_known) {
      b0 = a.band_start[k * (bands + 1) + band];
      b1 = a.band_start[k * (bands + 1) + band + 1];
    } else {
      b0 = below(first, n, (long long)band * a.band_rows);
      b1 = band + 1 == bands ? n : below(first, n, (long long)(band + 1) * a.band_rows);
    }
    key[o] = (unsigned)(q >> shift) << 27 | ((1u << 27) - 1 - min((unsigned)(b1 - b0), (1u << 27) - 1));
    if (shift == 0 && !a.bands_known) {
      a.band_start[k * (bands + 1) + band] = b0;
      if (band + 1 == bands) a.band_start[k * (bands + 1) + bands] = n;
    }
  }
  for (int o = per_xcd + threadIdx.x; o < padded; o += blockDim.x) key[o] = ~0u;
  __syncthreads();
  typedef unsigned uint4v_ __attribute__((ext_vector_type(4)));
  for (int c = threadIdx.x; c < per_xcd; c += blockDim.x) {
    const unsigned mine = key[c];
    int rank = 0;
    // (Bound by the reads' latency: four keys a read, four reads in flight.  Count and group of one cell at a time, 108 cells 14 us and
    // 216 cells 26, were what the launch waited for: over 100 k LiDAR and 200 k indoor voxels, 27 offsets, 17.2 -> 11.6 us
    // and 28.8 -> 17.2.)
#pragma unroll 4
    for (int o = 0; o < padded; o += 4) {
      const uint4v_ theirs = *reinterpret_cast<const uint4v_ *>(key + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) rank += theirs[e] < mine || (theirs[e] == mine && o + e < c) ? 1 : 0;
    }
    a.band_cells[(size_t)shift * bands * k_vol + rank * 8 + x] = (c % k_vol) * 65536 + (c / k_vol) * 8 + x;
  }
}

// The last launch of a build.  Step 3, the neighbour tables by POSITION: nbr_out[k][position of o] =
// i, nbr_in[k][position of i] = o -- scattered from the pair lists (tables pre-filled with -1), or,
// where the map builder left a table of the output rows, read from there in the output side's
// position order (whole lines both ways: no pre-fill, no scattered 4-byte stores on that side).  Next to it, as
// workgroups of the same launch: tile orders, row bands, the fingerprint of the lists, the findings'
// way to the host.  (Five launches of 3-12 us each and a second stream before.)
__global__ __launch_bounds__(256) void tables_kernel(TablesArgs a) {
  extern __shared__ __align__(16) int32_t lds[];      // (bands_body reads 16 bytes at a time; the static LDS in front of it ends anywhere)
  int b = blockIdx.x;
  if (b < a.tile_blocks) {
    if (b == 0 && threadIdx.x < kPlanFlags) {
      const int q = threadIdx.x;
      // (mirrored maps: one side's counts stand for both)
      const int v = a.flags[a.mirror && (q == 5 || q == 11) ? q - 1 : q];
      if (a.host && (q < kFlagPrint)) a.host[q] = v;
    }
    if (b < 2) tile_order_body(a.tile[b], a.cus >= 8 ? a.cus / 8 : 1, lds);
    return;
  }
  b -= a.tile_blocks;
  if (b < a.band_blocks) {
    bands_body(a, b % 8, b / 8, lds);
    return;
  }
  b -= a.band_blocks;
  if (b < a.print_blocks) {
    plan_print_block(a.kpos, a.imap, a.omap, a.k_vol, a.n_pairs, a.flags, b);
    return;
  }
  b -= a.print_blocks;
  if (b < a.row_blocks) {
    // 64 positions, transposed in LDS: rows come in as whole 16-byte pieces of neighbouring lanes
    // (a lane that reads its own row alone fetches every line as often as it has pieces)
    typedef int int4v_ __attribute__((ext_vector_type(4)));
    const int p0 = b * 64, lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int per_row = a.row_ld / 4, ld = a.row_ld + 1;
    for (int e = threadIdx.x; e < 64 * per_row; e += 256) {
      const int r = e / per_row, c = e % per_row, p = p0 + r;
      if (p < a.n_out) {
        const int4v_ v = *reinterpret_cast<const int4v_ *>(a.rows + (size_t)a.perm_out[p] * a.row_ld + c * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) lds[r * ld + c * 4 + q] = v[q];
      }
    }
    __syncthreads();
    const int centre = empty_centre(a.kpos, a.k_vol);
    if (p0 + lane < a.n_out) {
      const int o = a.inv_in || centre >= 0 ? a.perm_out[p0 + lane] : 0;
      for (int k = wave; k < a.k_vol; k += 4) {
        if (k == centre) {
          a.nbr_out[(size_t)k * a.n_out + p0 + lane] = o;
          continue;
        }
        const int i = lds[lane * ld + k];
        a.nbr_out[(size_t)k * a.n_out + p0 + lane] = i;
        if (a.inv_in && i >= 0) a.nbr_in[(size_t)k * a.n_in + a.inv_in[i]] = o;
      }
    }
    return;
  }
  b -= a.row_blocks;
  const int total = a.kpos[a.k_vol];
  const int j = a.kpos[0] + b * 256 + threadIdx.x;
  if (j >= total || j >= a.n_pairs) return;
  int lo = 0, hi = a.k_vol;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.kpos[mid] <= j) lo = mid; else hi = mid;
  }
  const int i = a.imap[j], o = a.omap[j];
  if (i < 0 || i >= a.n_in || o < 0 || o >= a.n_out) return;
  if (a.inv_out) a.nbr_out[(size_t)lo * a.n_out + a.inv_out[o]] = i;
  if (a.inv_in) a.nbr_in[(size_t)lo * a.n_in + a.inv_in[i]] = o;
}

// Pinned blocks for the builds' flag read-backs (hipHostMalloc costs as much as the whole
// build; freed blocks are kept).
std::mutex g_pinned_mutex;
std::vector<int *> g_pinned_free;

int *pinned_flags_get() {
  {
    std::lock_guard<std::mutex> lock(g_pinned_mutex);
    if (!g_pinned_free.empty()) {
      int *q = g_pinned_free.back();
      g_pinned_free.pop_back();
      return q;
    }
  }
  int *q = nullptr;
  note_allocation();
  if (hipHostMalloc((void **)&q, kPlanFlags * sizeof(int), hipHostMallocDefault) != hipSuccess) return nullptr;
  return q;
}

void pinned_flags_put(int *q) {
  std::lock_guard<std::mutex> lock(g_pinned_mutex);
  g_pinned_free.push_back(q);
}

// fgms_plan_check: the fingerprint taken again from the lists as they are now (a workgroup per
// part), compared with the build's; a difference raises the sticky flag, in device memory and in
// the plan's pinned block.
__global__ __launch_bounds__(256) void plan_check_kernel(const int32_t *__restrict__ kpos,
                                                          const int32_t *__restrict__ imap,
                                                          const int32_t *__restrict__ omap, int k_vol, int n_pairs,
                                                          int *__restrict__ flags, int *__restrict__ host) {
  plan_check_block(kpos, imap, omap, k_vol, n_pairs, flags, host, blockIdx.x);
}

}  // namespace
}  // namespace fgms

using namespace fgms;

namespace fgms {

int launch_fills(const FillBatch &batch, hipStream_t s) {
  size_t most = 0;
  for (int r = 0; r < batch.count; ++r)
    if (batch.range[r].n > most) most = batch.range[r].n;
  if (most == 0) return FGMS_OK;
  size_t blocks = (most / 4 + 255) / 256;          // one 16-byte store per thread, a few for big blocks
  if (blocks > 4096) blocks = 4096;
  fills_kernel<<<(unsigned)(blocks ? blocks : 1), 256, 0, s>>>(batch);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

void sort_side_layout(SortSide &sd, int64_t n, Arena &tmp) {
  sd.n = (int)n;
  sd.chunks = n > kWindow ? (int)((n + kChunk - 1) / kChunk) : 0;      // one window: no counting sort
  tmp.take(sd.inv, (size_t)n);
  if (sd.chunks) {
    tmp.take(sd.perm_tmp, (size_t)n);
    tmp.take(sd.hist, (size_t)kBins * sd.chunks);
    tmp.take(sd.hist_before, (size_t)kBins * sd.chunks);
    tmp.take(sd.bin_start, (size_t)kBins);
    tmp.take(sd.key, (size_t)n);
  }
}

// FGMS_PLAN_SORT=0 keeps the rows in their natural order (for comparison).
bool plan_sorts_rows() {
  static const bool sort_rows = !(getenv("FGMS_PLAN_SORT") && atoi(getenv("FGMS_PLAN_SORT")) == 0);
  return sort_rows;
}

static unsigned sides_of(const SortArgs &a) { return a.side[1].n > 0 ? 2 : 1; }
static int most_chunks(const SortArgs &a) { return a.side[0].chunks > a.side[1].chunks ? a.side[0].chunks : a.side[1].chunks; }

int launch_sort_scatter(const SortArgs &a, hipStream_t s) {
  sort_scatter_kernel<<<dim3((unsigned)most_chunks(a), sides_of(a)), kSortThreads, 0, s>>>(a);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

int launch_sort(const SortArgs &args, hipStream_t s) {
  SortArgs a = args;
  a.by_mask = plan_sorts_rows();
  if (!a.by_mask) a.side[0].chunks = a.side[1].chunks = 0;
  if (const int chunks = most_chunks(a)) {
    sort_hist_kernel<<<dim3((unsigned)chunks, sides_of(a)), kSortThreads, 0, s>>>(a);
    sort_scan_kernel<<<dim3(kBins / kScanBins, sides_of(a)), 256, 0, s>>>(a);
    const int rc = launch_sort_scatter(a, s);
    if (rc != FGMS_OK) return rc;
  }
  const int most = a.side[0].n > a.side[1].n ? a.side[0].n : a.side[1].n;
  if (most) sort_window_kernel<<<dim3((unsigned)((most + kWindow - 1) / kWindow), sides_of(a)), kWindowThreads, 0, s>>>(a);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

int launch_tables(TablesArgs a, hipStream_t s) {
  const int tiles = a.tile[0].n_tiles > a.tile[1].n_tiles ? a.tile[0].n_tiles : a.tile[1].n_tiles;
  size_t lds = (size_t)tiles * sizeof(int32_t);
  a.tile_blocks = 8;                               // (two at work; the parts behind start on a multiple of eight)
  a.band_blocks = 0;
  if (a.band_start) {
    const size_t need = ((size_t)((a.bands ? a.bands : 64) / 8) * a.k_vol + 3) * sizeof(int32_t);
    if (need > lds) lds = need;
    a.band_blocks = 32;
  }
  a.print_blocks = a.take_print ? kPrintParts : 0;
  a.row_blocks = a.rows ? (a.n_out + 63) / 64 : 0;
  if (a.rows && (size_t)64 * (a.row_ld + 1) * sizeof(int32_t) > lds) lds = (size_t)64 * (a.row_ld + 1) * sizeof(int32_t);
  a.pair_blocks = !a.rows && (a.inv_out || a.inv_in) ? (a.n_pairs + 255) / 256 : 0;
  a.cus = num_cus();
  if (lds > 48 * 1024) {
    const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(tables_kernel), lds);
    if (rc != FGMS_OK) return rc;
  }
  tables_kernel<<<(unsigned)(a.tile_blocks + a.band_blocks + a.print_blocks + a.row_blocks + a.pair_blocks), 256, lds, s>>>(a);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

Plan *plan_alloc(int k_vol, int64_t n_in, int64_t n_out, int64_t n_pairs, hipStream_t s) {
  Plan *p = new Plan();          // (value-initialised: every field starts out zero)
  p->k_vol = k_vol; p->n_in = n_in; p->n_out = n_out; p->n_pairs = n_pairs;
  p->last_stream = s;
  p->create_stream = s;
  if (hipGetDevice(&p->device) == hipSuccess && (p->host_flags = pinned_flags_get()) &&
      (p->ready = event_get(p->device))) {
    p->host_flags[kFlagStale] = 0;     // (a recycled block: the flag is read before the build has run)
    return p;
  }
  set_error("plan: pinned flag block / event creation failed");
  fgms_plan_destroy((fgms_plan_t *)p);
  return nullptr;
}

void plan_bands(Plan *p) {
  p->band_count = band_count_of(p->n_pairs, p->k_vol, num_cus());
  p->band_rows = (int)((p->n_out + p->band_count - 1) / p->band_count);
}

// Tile -> XCD homes pay off once every XCD has a few dozen tiles of its own.
// (cap: an eighth more than an eighth of them, for an XCD with many light tiles)
int tile_table(int64_t n, int *cap) {
  static const bool xcd_homes = !(getenv("FGMS_XCD_HOME") && atoi(getenv("FGMS_XCD_HOME")) == 0);
  const int64_t n_tiles = (n + 255) / 256;
  *cap = (int)((n_tiles * 9 / 8 + 7) / 8);
  return xcd_homes && n_tiles >= 256 && n_tiles * sizeof(int32_t) <= 60000 ? (int)n_tiles : 0;
}

void plan_fill_tables_args(const Plan *p, TablesArgs *t) {
  t->kpos = p->kpos; t->imap = p->in_map; t->omap = p->out_map;
  t->k_vol = p->k_vol; t->n_pairs = (int)p->n_pairs; t->n_in = (int)p->n_in; t->n_out = (int)p->n_out;
  t->band_start = p->band_start; t->band_cells = p->band_cells;
  t->bands = p->band_count;
  t->band_rows = p->band_rows > 0 ? p->band_rows : 1;
  for (int d = 0; d < 2; ++d) {
    int32_t *order = d ? p->tile_in : p->tile_out;
    if (!order || (d && order == p->tile_out)) continue;
    int cap;
    const int64_t n = d ? p->n_in : p->n_out;
    const int n_tiles = tile_table(n, &cap);
    t->tile[d] = TileSide{d ? p->perm_in : p->perm_out, d ? p->mask_in : p->mask_out, order, (int)n, n_tiles, cap};
  }
  t->flags = p->flags;
  if (hipHostGetDevicePointer((void **)&t->host, p->host_flags, 0) != hipSuccess) t->host = nullptr;
}

int plan_publish(Plan *p, bool written, hipStream_t s) {
  if ((!written && hipMemcpyAsync(p->host_flags, p->flags, kPlanFlags * sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess) ||
      hipEventRecord(p->ready, s) != hipSuccess) {
    set_error("plan: queuing the flag read-back failed");
    return FGMS_E_HIP;
  }
  return FGMS_OK;
}

// Builds a plan.  Everything is queued on `stream`; nothing waits for the GPU.  What
// the build finds out about the map (index out of range, rows shared inside an offset, pair
// order, block counts) travels to pinned host memory with the last kernel and is read by
// plan_resolve when the plan is first used.
int plan_create(fgms_plan_t **plan_out, const int32_t *kpos, const int32_t *in_map,
                const int32_t *out_map, int64_t n_in, int64_t n_out, int k_vol, int64_t n_pairs, void *stream,
                bool want_bands) {
  if (!plan_out) {
    set_error("plan output pointer is null");
    return FGMS_E_INVALID;
  }
  *plan_out = nullptr;
  if (!kpos || k_vol <= 0 || n_in < 0 || n_out < 0 || n_pairs < 0 ||
      (n_pairs > 0 && (!in_map || !out_map)) || n_in > INT32_MAX || n_out > INT32_MAX ||
      n_pairs > INT32_MAX - 65536) {
    set_error("fgms_plan_create: bad argument");
    return FGMS_E_INVALID;
  }
  hipStream_t s = (hipStream_t)stream;
  {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone) {
      set_error("fgms_plan_create: the stream is being captured (the build allocates; make the plan before)");
      return FGMS_E_INVALID;
    }
  }
  Plan *p = plan_alloc(k_vol, n_in, n_out, n_pairs, s);
  if (!p) return FGMS_E_NOMEM;
  p->kpos = kpos; p->in_map = in_map; p->out_map = out_map;
  plan_bands(p);
  const bool tables = k_vol <= 64;      // (64-bit offset masks; beyond that the plan is bands only)
  if (k_vol > 1500) want_bands = false;   // (the cell orders are ranked in LDS)
  p->has_tables = tables;
  p->has_bands = want_bands;
  const size_t so = tables ? (size_t)n_out * k_vol : 0, si = tables ? (size_t)n_in * k_vol : 0;
  const size_t bo = (size_t)(n_out + 63) / 64, bi = (size_t)(n_in + 63) / 64;
  SortArgs sa{};
  sa.k_vol = k_vol;
  unsigned long long *rmask = nullptr;          // [n_out] then [n_in]
  int cap_out = 0, cap_in = 0;
  const int tiles_out = tables ? tile_table(n_out, &cap_out) : 0, tiles_in = tables ? tile_table(n_in, &cap_in) : 0;
  void *scratch = nullptr;
  auto layout = [&](Arena &keep, Arena &tmp) {
    keep.take(p->flags, kPlanFlags);
    if (want_bands) {
      keep.take(p->band_start, (size_t)k_vol * (p->band_count + 1));
      keep.take(p->band_cells, (size_t)4 * k_vol * p->band_count);
    }
    if (!tables) return;
    keep.take(p->nbr_out, so + si);             // (nbr_in right behind: one fill)
    keep.take(p->mask_out, bo);
    keep.take(p->mask_in, bi);
    keep.take(p->perm_out, (size_t)n_out);
    keep.take(p->perm_in, (size_t)n_in);
    if (tiles_out) keep.take(p->tile_out, (size_t)cap_out * 8);
    if (tiles_in) keep.take(p->tile_in, (size_t)cap_in * 8);
    tmp.take(rmask, (size_t)(n_out + n_in));
    sort_side_layout(sa.side[0], n_out, tmp);
    sort_side_layout(sa.side[1], n_in, tmp);
  };
  int rc = FGMS_OK;
  auto fail = [&](int code) {
    if (scratch) pool_free(scratch, s, false);
    fgms_plan_destroy((fgms_plan_t *)p);
    return code;
  };
  {
    Arena keep, tmp;
    layout(keep, tmp);
    if ((rc = pool_alloc(&p->block, keep.used, s)) || (tmp.used && (rc = pool_alloc(&scratch, tmp.used, s)))) return fail(rc);
    Arena keep_at, tmp_at;
    keep_at.base = (char *)p->block;
    tmp_at.base = (char *)scratch;
    layout(keep_at, tmp_at);
  }
  if (tables) {
    p->nbr_in = p->nbr_out + so;
    p->tile_grid_out = p->tile_out ? cap_out * 8 : 0;
    p->tile_grid_in = p->tile_in ? cap_in * 8 : 0;
    sa.flags = p->flags;
    sa.kpos = kpos;
    sa.side[0].rmask = rmask; sa.side[0].perm = p->perm_out; sa.side[0].block_mask = p->mask_out; sa.side[0].nbr = p->nbr_out;
    sa.side[1].rmask = rmask + n_out; sa.side[1].perm = p->perm_in; sa.side[1].block_mask = p->mask_in; sa.side[1].nbr = p->nbr_in;
  }
  FillBatch fills{};
  fills.add(p->flags, kPlanFlags * sizeof(int), 0);
  if (tables) {
    fills.add(rmask, (size_t)(n_out + n_in) * sizeof(unsigned long long), 0);
    fills.add(p->nbr_out, (so + si) * sizeof(int32_t), -1);
    if (want_bands) fills.add(p->band_start, (size_t)k_vol * (p->band_count + 1) * sizeof(int32_t), 0);
  }
  if ((rc = launch_fills(fills, s))) return fail(rc);
  TablesArgs ta{};
  plan_fill_tables_args(p, &ta);
  if (tables) {
    if (n_pairs > 0)
      pair_masks_kernel<<<(unsigned)((n_pairs + 255) / 256) + kPrintParts, 256, 0, s>>>(
          kpos, in_map, out_map, k_vol, (int)n_pairs, (int)n_in, (int)n_out, rmask, rmask + n_out, p->flags,
          want_bands ? p->band_start : nullptr, p->band_count, p->band_rows > 0 ? p->band_rows : 1);
    if ((rc = launch_sort(sa, s))) return fail(rc);
    ta.inv_out = sa.side[0].inv; ta.inv_in = sa.side[1].inv;
    ta.nbr_out = p->nbr_out; ta.nbr_in = p->nbr_in;
    ta.bands_known = true;
  }
  if ((rc = launch_tables(ta, s)) || (rc = plan_publish(p, ta.host != nullptr, s))) return fail(rc);
  if (scratch) pool_free(scratch, s, false);
  scratch = nullptr;
  // More than 64 offsets: the tables and masks hold 64 offsets each, so the offsets are cut
  // into groups of 64, every group with tables of its own (the pairs of a group are one
  // contiguous run of the lists); the entry points walk the groups, the weight gradient uses
  // this plan's row bands over all offsets.
  if (!tables) {
    for (int k0 = 0; k0 < k_vol; k0 += 64) {
      fgms_plan_t *g = nullptr;
      rc = plan_create(&g, kpos + k0, in_map, out_map, n_in, n_out, k_vol - k0 < 64 ? k_vol - k0 : 64, n_pairs,
                       stream, false);
      if (rc != FGMS_OK) {
        fgms_plan_destroy((fgms_plan_t *)p);
        return rc;
      }
      p->groups.push_back((Plan *)g);
    }
  }
  *plan_out = (fgms_plan_t *)p;
  return FGMS_OK;
}

// What the build found out, once its last kernel has run.  Returns the plan when its flags are
// known (waiting for the build if it has not finished yet), nullptr when they cannot be had
// now (the stream is being captured into a graph: the caller then takes the kernels that need
// no plan) or when the map turned out to be invalid (*rc = FGMS_E_INVALID).
// The plan if its build results are already known to the host, else nullptr: never waits,
// never allocates, never launches (for the entry point that promises that).
const Plan *plan_if_resolved(fgms_plan_t *plan) {
  Plan *p = (Plan *)plan;
  if (!p) return nullptr;
  std::lock_guard<std::mutex> lock(p->mutex);
  return p->resolved && !p->invalid ? p : nullptr;
}

static Plan *check_owner(const Plan *p) { return const_cast<Plan *>(p->base ? p->base : p); }

bool plan_take_check(const Plan *p, SideJob *job) {
  Plan *b = check_owner(p);
  if (!b->check_pending || !b->has_tables || !b->flags || b->n_pairs == 0) return false;
  if (!b->resolved) return false;     // (the build may still be running: the fingerprint is not final)
  int *host_dev = nullptr;
  if (hipHostGetDevicePointer((void **)&host_dev, b->host_flags, 0) != hipSuccess) host_dev = nullptr;
  *job = SideJob{};
  job->kind = 3;
  job->blocks = kPrintParts;       // (a multiple of 8: the workgroups behind keep their XCDs)
  job->src = b->kpos;
  job->dst = const_cast<int32_t *>(b->in_map);
  job->omap = b->out_map;
  job->n = (size_t)b->n_pairs;
  job->k_vol = b->k_vol;
  job->flags = b->flags;
  job->host = host_dev;
  b->check_pending = false;
  b->checked = true;
  return true;
}

int plan_flush_check(const Plan *p, hipStream_t s) {
  Plan *b = check_owner(p);
  for (Plan *g : b->groups) {
    const int rc = plan_flush_check(g, s);
    if (rc != FGMS_OK) return rc;
  }
  if (!b->check_pending) return FGMS_OK;
  b->check_pending = false;
  if (!b->has_tables || !b->flags || b->n_pairs == 0) return FGMS_OK;
  int *host_dev = nullptr;
  if (hipHostGetDevicePointer((void **)&host_dev, b->host_flags, 0) != hipSuccess) host_dev = nullptr;
  // (queued behind the build if that ran on another stream: the fingerprint must be final)
  // (a resolved plan's build has finished; no event is queried then, which a stream under
  // capture would not allow)
  if (!b->resolved && s != b->create_stream) FGMS_HIP_TRY(hipStreamWaitEvent(s, b->ready, 0));
  plan_check_kernel<<<kPrintParts, 256, 0, s>>>(b->kpos, b->in_map, b->out_map, b->k_vol, (int)b->n_pairs, b->flags, host_dev);
  FGMS_HIP_TRY(hipGetLastError());
  b->checked = true;
  return FGMS_OK;
}

// Has an earlier fgms_plan_check found the lists changed?  (Reads the pinned block; no wait.)
static bool plan_is_stale(const Plan *p) {
  const Plan *b = p->base ? p->base : p;
  if (b->checked && b->host_flags && b->host_flags[kFlagStale]) return true;
  for (const Plan *g : b->groups)
    if (g->checked && g->host_flags && g->host_flags[kFlagStale]) return true;
  return false;
}

// The pair view of `p`, built by the first launch that is to walk it, from that call's own lists.
static bool build_pair_view(Plan *p, const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, hipStream_t s) {
  std::lock_guard<std::mutex> lock(p->mutex);
  if (p->pv_in) return true;
  if (!p->pv_rows || is_capturing(s)) return false;
  if (Plan *b = p->base) {                     // (a transposed view: the base's, the sides swapped)
    if (!build_pair_view(b, kpos, out_map, in_map, s)) return false;
    p->pv_stream = b->pv_stream; p->pv_ready = b->pv_ready;
    p->pv_out = b->pv_in; p->pv_mask = b->pv_mask; p->pv_in = b->pv_out;
    return true;
  }
  const int64_t rows = p->pv_rows;
  int32_t *in = nullptr, *out = nullptr;
  unsigned long long *mask = nullptr;
  FillBatch fills{};
  bool ok = pool_alloc((void **)&in, (size_t)rows * sizeof(int32_t), s) == FGMS_OK &&
            pool_alloc((void **)&out, (size_t)rows * sizeof(int32_t), s) == FGMS_OK &&
            pool_alloc((void **)&mask, (size_t)(rows / 64) * sizeof(unsigned long long), s) == FGMS_OK;
  if (ok) {
    fills.add(in, (size_t)rows * sizeof(int32_t), -1);
    fills.add(out, (size_t)rows * sizeof(int32_t), -1);
    fills.add(mask, (size_t)(rows / 64) * sizeof(unsigned long long), 0);
    ok = launch_fills(fills, s) == FGMS_OK;
  }
  if (!ok) {
    if (in) pool_free(in, s, false);
    if (out) pool_free(out, s, false);
    if (mask) pool_free(mask, s, false);
    p->pv_rows = 0;
    return false;
  }
  pair_view_kernel<<<(unsigned)((p->n_pairs + 255) / 256), 256, 0, s>>>(kpos, in_map, out_map, p->k_vol, (int)p->n_pairs, (long long)rows,
                                                                       in, out, mask);
  // launches on other streams wait for this event (launch_pair_view_gms, the destroy path)
  if (hipGetLastError() != hipSuccess || hipEventCreateWithFlags(&p->pv_ready, hipEventDisableTiming) != hipSuccess ||
      hipEventRecord(p->pv_ready, s) != hipSuccess) {
    // without the event nothing else can be ordered behind the build: finish it here
    (void)hipStreamSynchronize(s);
    if (p->pv_ready) (void)hipEventDestroy(p->pv_ready);
    p->pv_ready = nullptr;
  }
  p->pv_stream = s;
  p->pv_out = out; p->pv_mask = mask; p->pv_in = in;
  return true;
}

bool plan_pair_view(const Plan *p, const GmsArgs &a) {
  return build_pair_view(const_cast<Plan *>(p), a.kpos, a.transpose_w ? a.smap : a.gmap, a.transpose_w ? a.gmap : a.smap, a.stream);
}

const Plan *plan_resolve(fgms_plan_t *plan, hipStream_t stream, int *rc) {
  *rc = FGMS_OK;
  Plan *p = (Plan *)plan;
  if (!p) return nullptr;
  if (plan_is_stale(p)) {
    set_error("plan: the pair lists were rewritten after the plan was made (make a new plan)");
    *rc = FGMS_E_STALE;
    return nullptr;
  }
  if (p->base && !p->resolved) {
    // a transposed view: the base's tables with the sides swapped
    const Plan *b = plan_resolve((fgms_plan_t *)p->base, stream, rc);
    if (!b) return nullptr;
    std::lock_guard<std::mutex> lock(p->mutex);
    if (!p->resolved) {
      p->nbr_out = b->nbr_in; p->nbr_in = b->nbr_out;
      p->flip_out = b->flip_in; p->flip_in = b->flip_out;
      p->perm_out = b->perm_in; p->perm_in = b->perm_out;
      p->mask_out = b->mask_in; p->mask_in = b->mask_out;
      p->tile_out = b->tile_in; p->tile_in = b->tile_out;
      p->tile_grid_out = b->tile_grid_in; p->tile_grid_in = b->tile_grid_out;
      p->stages_out = b->stages_in; p->stages_in = b->stages_out;
      p->fwd_ok = b->dgrad_ok; p->dgrad_ok = b->fwd_ok;
      p->pv_rows = b->pv_rows;
      p->has_tables = b->has_tables;
      p->centre_line = b->centre_line;
      p->full_out = b->full_in; p->full_in = b->full_out;
      p->pairs_counted = b->pairs_counted;
      p->ordered = false;
      // (the weight gradient's row bands follow the base's output rows: not valid for the swapped lists)
      p->bands_ok = false; p->band_start = nullptr; p->band_cells = nullptr; p->band_count = 0;
      p->invalid = false;
      p->resolved = true;
    }
    return p;
  }
  if (!p->resolved) {
    std::lock_guard<std::mutex> lock(p->mutex);
    if (!p->resolved) {
      if (hipEventQuery(p->ready) != hipSuccess) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone)
          return nullptr;
        if (hipEventSynchronize(p->ready) != hipSuccess) {
          set_error("plan: waiting for the build failed");
          *rc = FGMS_E_HIP;
          return nullptr;
        }
      }
      const int *h = p->host_flags;
      p->invalid = h[0] != 0;
      p->fwd_ok = p->has_tables && !h[0] && !h[1] && h[10] == h[12];
      p->dgrad_ok = p->has_tables && !h[0] && !h[2] && h[11] == h[12];
      p->ordered = !h[0] && !h[3];
      p->bands_ok = p->has_bands && p->ordered;
      p->centre_line = p->has_tables && h[kFlagCentre];
      p->full_out = p->fwd_ok && p->ordered ? (h[kFlagFull] & 255) - 1 : -1;
      p->full_in = p->dgrad_ok && !h[kFlagInput] ? (h[kFlagFull] >> 8) - 1 : -1;
      p->stages_out = h[4];
      p->stages_in = h[5];
      p->pairs_counted = p->has_tables ? h[12] : p->n_pairs;
      // The pair view, for maps sparse enough that some layer would take it (fp32 layers prefer
      // it from about 1 + 45 / channels row slots per pair on, never below 1.4, where the products are many).  Its size is known now;
      // it is built when a layer does take it (plan_pair_view): fp16 layers want twice as sparse a map, and over 100 k LiDAR
      // voxels, 1.5 slots a pair, its two launches were 15 us that a network in fp16 never saw again.
      static const bool pair_view = !(getenv("FGMS_PAIR_VIEW") && atoi(getenv("FGMS_PAIR_VIEW")) == 0);
      const int most = p->stages_out > p->stages_in ? p->stages_out : p->stages_in;
      if (!p->invalid && pair_view && p->has_tables && p->pairs_counted > 0 &&
          (kernel_policy() == 5 || (double)most * 64.0 >= 1.35 * (double)p->pairs_counted))
        p->pv_rows = (p->pairs_counted + 64 * (int64_t)p->k_vol + 255) / 256 * 256;
      // (a plan over more than 64 offsets: its groups)
      for (Plan *g : p->groups) {
        int grc = FGMS_OK;
        const Plan *gr = plan_resolve((fgms_plan_t *)g, stream, &grc);
        if (!gr && grc == FGMS_E_INVALID) p->invalid = true;
        if (!gr && grc != FGMS_E_INVALID) return nullptr;        // (cannot be known now: try again later)
        if (gr) {
          p->fwd_ok = (g == p->groups.front() ? true : p->fwd_ok) && gr->fwd_ok;
          p->dgrad_ok = (g == p->groups.front() ? true : p->dgrad_ok) && gr->dgrad_ok;
          p->stages_out += gr->stages_out;
          p->stages_in += gr->stages_in;
          p->ordered = p->ordered && gr->ordered;
        }
      }
      if (!p->groups.empty()) p->bands_ok = p->has_bands && p->ordered && !p->invalid;
      p->resolved = true;
    }
  }
  if (p->invalid) {
    set_error("plan: a map index is outside [0, n_in) x [0, n_out)");
    *rc = FGMS_E_INVALID;
    return nullptr;
  }
  return p;
}
}  // namespace fgms

extern "C" {

int fgms_plan_create(fgms_plan_t **plan_out, const int32_t *kpos, const int32_t *in_map,
                     const int32_t *out_map, int64_t n_in, int64_t n_out, int k_vol,
                     int64_t n_pairs, void *stream) {
  return plan_create(plan_out, kpos, in_map, out_map, n_in, n_out, k_vol, n_pairs, stream, true);
}

int fgms_plan_transposed(fgms_plan_t **view_out, fgms_plan_t *base_plan) {
  Plan *b = (Plan *)base_plan;
  if (!view_out || !b || b->base || !b->groups.empty()) {
    set_error("fgms_plan_transposed: needs a plan made by fgms_plan_create over at most 64 offsets");
    return FGMS_E_INVALID;
  }
  Plan *v = new Plan();
  v->device = b->device;
  v->k_vol = b->k_vol; v->n_in = b->n_out; v->n_out = b->n_in; v->n_pairs = b->n_pairs;
  v->kpos = b->kpos; v->in_map = b->out_map; v->out_map = b->in_map;
  v->last_stream = b->last_stream;
  v->base = b;
  {
    std::lock_guard<std::mutex> lock(b->mutex);
    b->views += 1;
  }
  *view_out = (fgms_plan_t *)v;
  return FGMS_OK;
}

void fgms_plan_destroy(fgms_plan_t *plan) {
  Plan *p = (Plan *)plan;
  if (!p) return;
  if (p->base) {
    // a view owns nothing; the base goes with its last view if it was destroyed before
    Plan *b = p->base;
    bool free_base = false;
    {
      std::lock_guard<std::mutex> lock(b->mutex);
      if (p->last_stream != b->last_stream || p->many_streams) b->many_streams = true;
      b->views -= 1;
      free_base = b->views == 0 && b->destroyed;
    }
    delete p;
    if (free_base) fgms_plan_destroy((fgms_plan_t *)b);
    return;
  }
  {
    std::lock_guard<std::mutex> lock(p->mutex);
    p->destroyed = true;
    if (p->views > 0) return;       // (still shared: freed with the last view)
  }
  for (Plan *g : p->groups) {
    if (p->many_streams) g->many_streams = true;
    g->last_stream = p->last_stream;
    fgms_plan_destroy((fgms_plan_t *)g);
  }
  p->groups.clear();
  if (p->many_streams) (void)hipDeviceSynchronize();     // (blocks are handed back behind ONE stream's work)
  if (p->block) pool_free(p->block, p->last_stream, false);
  if (p->pv_ready) {
    // the view may have been built on another stream than the one the blocks are handed back behind
    if (p->pv_stream != p->last_stream) (void)hipStreamWaitEvent(p->last_stream, p->pv_ready, 0);
    (void)hipEventDestroy(p->pv_ready);
  }
  if (p->pv_in) pool_free(p->pv_in, p->last_stream, false);
  if (p->pv_out) pool_free(p->pv_out, p->last_stream, false);
  if (p->pv_mask) pool_free(p->pv_mask, p->last_stream, false);
  if (p->ready) {
    // the flag read-back must not land in freed host memory
    (void)hipEventSynchronize(p->ready);
    event_put(p->ready, p->device);
  }
  if (p->host_flags) pinned_flags_put(p->host_flags);
  delete p;
}

int fgms_plan_check(fgms_plan_t *plan, void *stream, int with_next_launch) {
  Plan *p = (Plan *)plan;
  if (!p) return FGMS_OK;
  Plan *b = p->base ? p->base : p;           // (a view shares its base's lists and flags)
  if (plan_is_stale(p)) {
    set_error("plan: the pair lists were rewritten after the plan was made (make a new plan)");
    return FGMS_E_STALE;
  }
  b->check_pending = true;
  for (Plan *g : b->groups) g->check_pending = true;
  if (with_next_launch) return FGMS_OK;
  return plan_flush_check(p, (hipStream_t)stream);
}

int fgms_plan_usable(const fgms_plan_t *plan, int for_dgrad) {
  int rc = FGMS_OK;
  const Plan *p = plan_resolve(const_cast<fgms_plan_t *>(plan), nullptr, &rc);
  if (!p) return 0;
  return for_dgrad ? (p->dgrad_ok ? 1 : 0) : (p->fwd_ok ? 1 : 0);
}

int fgms_plan_stats(const fgms_plan_t *plan, int64_t stats[4]) {
  if (!plan || !stats) {
    set_error("fgms_plan_stats: null argument");
    return FGMS_E_INVALID;
  }
  int rc = FGMS_OK;
  const Plan *p = plan_resolve(const_cast<fgms_plan_t *>(plan), nullptr, &rc);
  if (!p) return rc ? rc : FGMS_E_INVALID;
  stats[0] = p->groups.empty() ? p->pairs_counted : p->n_pairs;
  stats[1] = p->stages_out;
  stats[2] = p->stages_in;
  stats[3] = p->pv_rows;
  return FGMS_OK;
}

}  // extern "C"
