// Kernel-map builder on the device: from voxel coordinates to the pair lists the
// convolution kernels consume, and, if asked for, to the plan of the map as well.  The reference has
// no builder (its scripts load in_map / out_map / kernel_nnz / kernel_pos from files,
// cpu-check.py:89-94, spconv-test.py:64-73); this is the step right before the path.
//
// Pairs (i, o) with  in_coords[i] == out_coords[o] * stride + offsets[k],
// grouped by offset k, ascending o inside a group; when several input rows share
// a coordinate the smallest row index wins.  The result is a pure function of
// the inputs (no dependence on thread timing).
//
//   1. fill     everything that has to start from a value
//   2. insert   every input row enters its block of 2 x 2 x 4 voxels; the blocks are found through
//               an open-addressing hash table (buckets of four, load <= 0.5); equal coordinates keep the
//               smallest row
//   3. lookup   a table of the output rows, [n_out][offsets] -> input row or -1, the
//               set of offsets every row has a pair through, hits per (offset, 256 rows)
//   4. lists    prefix sums over those counts, hits compacted in (offset, row) order
//   5. plan     row order and tables (fgms_plan_sort.h, fgms_plan.hip), from the masks and the table of step 3: no atomics per
//               pair, no second pass over the lists.  A submanifold map (one coordinate list on
//               both sides, mirrored offsets) is its own mirror image, so one order and one table
//               serve both directions.  Steps 4 and 5 share launches (kmap_sizes_kernel).
// Bound by latencies: eight launches of one or two waves' worth of dependent accesses each.  At 100 k LiDAR voxels x 27 offsets they
// take 81 us of the stream; with a scan of its own and the lists in front of the plan's sort 98 us; lists alone and a plan from
// them afterwards 140 and 195 us, each behind a wait of the host for the one before.
#include <immintrin.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "fgms_device.h"
#include "fgms_internal.h"
#include "fgms_plan_build.h"
#include "fgms_plan_sort.h"

namespace fgms {
namespace {

typedef int int4v_ __attribute__((ext_vector_type(4)));

constexpr int kCoordLimit = 1 << 20;        // coordinates in [-2^20, 2^20)
constexpr int kListRows = 256;              // output rows per count
constexpr int kKernargOffsets = 128;        // offsets that travel as a kernel argument
// pinned read-back: [0] coordinates looked at, [1] bad one among them, [2] shared ones; [3] sizes there, [4] pairs, [16 ...] sizes
constexpr int kHostInts = 16 + 1024;
// A plan's offsets are also counted over all rows: in copies, a row of 64 sums each, so that the atomics of the lookup's workgroups
// spread over as many lines (all in one: a launch of 1 564 workgroups would wait for its 42 k atomics one behind the other).
constexpr int kTotalCopies = 64;

struct Offsets {
  int xyz[kKernargOffsets * 3];
};

// Voxels are found by blocks of 2 x 2 x 4: the hash table holds the blocks in use, and a block's 16 voxels lie in one 64-byte piece
// of `cells`, at its slot's number.  The 27 neighbours of a voxel lie in 8 blocks, and
// neighbouring rows share them: an eighth of the random accesses that a table of voxels costs, which
// is what such a table is bound by (100 k rows x 27 offsets: 2.7 M probes of a line each).  A slot holds its block's coordinates
// themselves (59 bits), so that a search is one access to it and one to the cells.
// A search waits for one bucket after another, and a wave for the longest chain of its lanes, most of which look for blocks that are not
// there.  Four slots to a bucket, read together, and two slots a row, whatever the number of rows: longest chain of a workgroup of the
// lookup, in the mean, 1.1 buckets over indoor and LiDAR surfaces, 2.0 over an indoor cloud thinned to a quarter, 2.7 to an
// eighth, 5.3 over 104 k voxels with a block each.  Single slots, two to four a row: 2.5, 4.6, 6.6 and 12; 1.25 to 2.5 a row: 3,
// 10, 18 and 141.  Whole builds with either of these / this, us: 200 k indoor voxels x 27 offsets 146 / 117 / 118, the eighth of them x 27
// 85 / 87 / 77 and x 125 144 / 231 / 105, 104 k with a block each x 27 123 / 277 / 104 and x 125 379 / 2 379 / 223.  (Three slots to
// two rows: 80 k with a block each x 125 314, of two a row 205, of two to four single ones 273.)
constexpr int kBlockX = 1, kBlockY = 1, kBlockZ = 2;      // bits of a coordinate inside its block
constexpr int kCells = 1 << (kBlockX + kBlockY + kBlockZ);
constexpr int kNoRow = INT32_MAX;
constexpr int kBucket = 4;
constexpr unsigned kNoSlot = ~0u;

// (Factors: the first three 32-bit primes of xxHash, Y. Collet; finaliser: prospector32, C. Wellons, "Prospecting for
// hash functions", 2018.)
__device__ __forceinline__ unsigned bucket_of(int bx, int by, int bz, unsigned buckets) {
  unsigned h = (unsigned)bx * 0x9E3779B1u ^ (unsigned)by * 0x85EBCA77u ^ (unsigned)bz * 0xC2B2AE3Du;
  h ^= h >> 15; h *= 0x2C1B3C6Du;
  h ^= h >> 12; h *= 0x297A2D39u;
  h ^= h >> 15;
  return __umulhi(h, buckets);
}
__device__ __forceinline__ int cell_of(int x, int y, int z) { return (x & 1) << 3 | (y & 1) << 2 | (z & 3); }
// A block as a slot holds it.  (Blocks of accepted coordinates only, block_exists; a free slot's ones are none of them.)
typedef unsigned long long BlockKey;
constexpr BlockKey kFreeSlot = ~0ull;
__device__ __forceinline__ bool block_exists(int bx, int by, int bz) {
  constexpr int x = kCoordLimit >> kBlockX, y = kCoordLimit >> kBlockY, z = kCoordLimit >> kBlockZ;
  return bx >= -x && bx < x && by >= -y && by < y && bz >= -z && bz < z;
}
__device__ __forceinline__ BlockKey block_key(int bx, int by, int bz) {
  constexpr int x = kCoordLimit >> kBlockX, y = kCoordLimit >> kBlockY, z = kCoordLimit >> kBlockZ;
  return (BlockKey)(unsigned)(bx + x) << 40 | (BlockKey)(unsigned)(by + y) << 20 | (unsigned)(bz + z);
}
// The slots of a bucket.  They fill from the front and keep what they hold, so that a free one ends every search.
typedef BlockKey keys2_ __attribute__((ext_vector_type(2)));
struct Bucket {
  keys2_ front, back;
  __device__ __forceinline__ BlockKey operator[](int e) const { return e < 2 ? front[e] : back[e - 2]; }
};
__device__ __forceinline__ Bucket bucket_at(const BlockKey *__restrict__ slots, unsigned bucket) {
  const keys2_ *const p = reinterpret_cast<const keys2_ *>(slots + (size_t)bucket * kBucket);
  return Bucket{p[0], p[1]};
}

// flags[0]: an input coordinate is outside the range; flags[1]: two input rows share their coordinates
__global__ __launch_bounds__(256) void kmap_insert_kernel(const int32_t *__restrict__ coords, int n, BlockKey *__restrict__ slots,
                                                          unsigned buckets, int32_t *__restrict__ cells, int *__restrict__ flags) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
  if (x < -kCoordLimit || x >= kCoordLimit || y < -kCoordLimit || y >= kCoordLimit || z < -kCoordLimit || z >= kCoordLimit) {
    flags[0] = 1;
    return;
  }
  const int bx = x >> kBlockX, by = y >> kBlockY, bz = z >> kBlockZ;
  unsigned bucket = bucket_of(bx, by, bz, buckets);
  const BlockKey key = block_key(bx, by, bz);
  int e = 0;
  while (true) {                       // ends: the table has more slots than rows
    const BlockKey prev = atomicCAS(&slots[(size_t)bucket * kBucket + e], kFreeSlot, key);
    if (prev == kFreeSlot || prev == key) break;
    // (what is read here may be old: a slot taken since then still looks free, and the exchange above tells)
    const Bucket b = bucket_at(slots, bucket);
    int next = kBucket;
#pragma unroll
    for (int q = kBucket - 1; q > 0; --q)
      if (q > e && (b[q] == kFreeSlot || b[q] == key)) next = q;
    e = next;
    if (e == kBucket) {
      e = 0;
      bucket = bucket + 1 == buckets ? 0 : bucket + 1;
    }
  }
  const size_t slot = (size_t)bucket * kBucket + e;
  if (atomicMin(&cells[slot * kCells + cell_of(x, y, z)], i) != kNoRow) flags[1] = 1;
}

struct LookupArgs {
  const int32_t *out_coords;
  int n_out, k_vol, stride, skip_offset, row_ld;
  const BlockKey *slots;
  const int32_t *cells;
  unsigned buckets;
  const int32_t *offsets;                      // device; nullptr: `offs`
  int32_t *rows;                               // [n_out][row_ld]
  int32_t *counts;                             // [k_vol][blocks of kListRows rows]
  int32_t *totals;                             // [kTotalCopies][64], nullptr: no plan
  int blocks;
  unsigned long long *rmask_out, *rmask_in;    // nullptr: no plan / a mirrored one
  const int *flags;
  int *host;                                   // pinned
};

// What the insertion found out, to the host.
__device__ __forceinline__ void publish_coordinates(const int *__restrict__ flags, int *__restrict__ host) {
  if (threadIdx.x != 0) return;
  host[1] = flags[0];
  host[2] = flags[1];
  __threadfence_system();
  __hip_atomic_store(&host[0], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The slots of N blocks (kNoSlot: not in use; want = false: not asked for), all searched together.
template <int N>
__device__ __forceinline__ void find_blocks(const LookupArgs &a, const int (&bx)[N], const int (&by)[N], const int (&bz)[N],
                                            const bool (&want)[N], unsigned (&at)[N]) {
  unsigned bucket[N];
  BlockKey key[N];
  bool open[N], any = false;
#pragma unroll
  for (int u = 0; u < N; ++u) {
    at[u] = kNoSlot;
    open[u] = want[u] && block_exists(bx[u], by[u], bz[u]);
    any = any || open[u];
    bucket[u] = bucket_of(bx[u], by[u], bz[u], a.buckets);
    key[u] = block_key(bx[u], by[u], bz[u]);
  }
  while (any) {                        // ends: every chain meets its block or a free slot
    Bucket b[N];
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (open[u]) b[u] = bucket_at(a.slots, bucket[u]);
    any = false;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (open[u]) {
#pragma unroll
        for (int e = 0; e < kBucket; ++e)
          if (b[u][e] == key[u]) at[u] = bucket[u] * kBucket + e;
      }
      open[u] = open[u] && at[u] == kNoSlot && b[u][kBucket - 1] != kFreeSlot;
      bucket[u] = bucket[u] + 1 == a.buckets ? 0 : bucket[u] + 1;
      any = any || open[u];
    }
  }
}

// The last workgroup sends the insertion's findings to the host.  The others take 64 output rows
// each.  NEAR (every offset within one voxel): its four waves find two of
// each row's eight blocks each, then every wave reads every fourth offset's cell from them.  Else
// (wider kernels) a lane finds the blocks of up to seven offsets at a time for itself.
// Bound by latency -- slot, cell: two dependent loads, with two to
// seven of each in flight per lane.  16.5 us at 100 k rows x 27 offsets; one probe chain per thread in a
// table of voxels took 14.5 us for half of the offsets, a table of voxels probed like this 116 us.
constexpr int kLookupRows = 64, kLookupChunk = 28;
template <bool NEAR>
__global__ __launch_bounds__(256) void kmap_lookup_kernel(LookupArgs a, Offsets offs) {
  constexpr int kMine = kLookupChunk / 4;
  __shared__ int32_t found[kLookupRows][kLookupChunk + 1];
  __shared__ unsigned long long wave_mask[4][kLookupRows];
  __shared__ unsigned near_slot[8][kLookupRows];
  if (blockIdx.x == gridDim.x - 1) {
    publish_coordinates(a.flags, a.host);
    return;
  }
  __shared__ int count_of[kLookupChunk];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int o = blockIdx.x * kLookupRows + lane;
  const bool live = o < a.n_out;
  const int oc = live ? o : a.n_out - 1;
  const long long lx = (long long)a.out_coords[3 * oc] * a.stride, ly = (long long)a.out_coords[3 * oc + 1] * a.stride,
                  lz = (long long)a.out_coords[3 * oc + 2] * a.stride;
  constexpr long long kFar = 1 << 30;          // (offsets are below it as well: sums stay in 32 bits)
  const bool sane = live && lx > -kFar && lx < kFar && ly > -kFar && ly < kFar && lz > -kFar && lz < kFar;
  const int x0 = sane ? (int)lx : 0, y0 = sane ? (int)ly : 0, z0 = sane ? (int)lz : 0;
  const int block = blockIdx.x * kLookupRows / kListRows;
  if constexpr (NEAR) {
    // block j of a row: the row's own (bits 0) or the nearer neighbour along x (bit 2), y (bit 1), z (bit 0)
    int bx[2], by[2], bz[2];
    unsigned at[2];
    bool want[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int j = wave * 2 + u;
      const int zi = z0 & 3, dz = zi == 0 ? -1 : zi == 3 ? 1 : 0;
      bx[u] = (x0 >> kBlockX) + (j & 4 ? ((x0 & 1) ? 1 : -1) : 0);
      by[u] = (y0 >> kBlockY) + (j & 2 ? ((y0 & 1) ? 1 : -1) : 0);
      bz[u] = (z0 >> kBlockZ) + (j & 1 ? dz : 0);
      want[u] = sane && !((j & 1) && dz == 0);
    }
    find_blocks<2>(a, bx, by, bz, want, at);
#pragma unroll
    for (int u = 0; u < 2; ++u) near_slot[wave * 2 + u][lane] = at[u];
    __syncthreads();
  }
  unsigned long long mine = 0;
  for (int k0 = 0; k0 < a.k_vol; k0 += kLookupChunk) {
    int hit[kMine], cell[kMine];
    unsigned at[kMine];
    if constexpr (NEAR) {
#pragma unroll
      for (int u = 0; u < kMine; ++u) {
        const int k = k0 + u * 4 + wave;
        at[u] = kNoSlot;
        cell[u] = 0;
        if (k < a.k_vol && k != a.skip_offset) {
          const int *d = a.offsets ? a.offsets + 3 * k : offs.xyz + 3 * k;
          const int x = x0 + d[0], y = y0 + d[1], z = z0 + d[2];
          const int j = (x >> kBlockX != x0 >> kBlockX) << 2 | (y >> kBlockY != y0 >> kBlockY) << 1 | (z >> kBlockZ != z0 >> kBlockZ);
          at[u] = near_slot[j][lane];
          cell[u] = cell_of(x, y, z);
        }
      }
    } else {
      int bx[kMine], by[kMine], bz[kMine];
      bool want[kMine];
#pragma unroll
      for (int u = 0; u < kMine; ++u) {
        const int k = k0 + u * 4 + wave;
        want[u] = false;
        bx[u] = by[u] = bz[u] = 0;
        cell[u] = 0;
        if (k < a.k_vol && k != a.skip_offset) {
          const int *d = a.offsets ? a.offsets + 3 * k : offs.xyz + 3 * k;
          const long long x = (long long)x0 + d[0], y = (long long)y0 + d[1], z = (long long)z0 + d[2];
          want[u] = sane && x == (int)x && y == (int)y && z == (int)z;
          bx[u] = (int)x >> kBlockX; by[u] = (int)y >> kBlockY; bz[u] = (int)z >> kBlockZ;
          cell[u] = cell_of((int)x, (int)y, (int)z);
        }
      }
      find_blocks<kMine>(a, bx, by, bz, want, at);
    }
#pragma unroll
    for (int u = 0; u < kMine; ++u) hit[u] = a.cells[(size_t)(at[u] == kNoSlot ? 0 : at[u]) * kCells + cell[u]];
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      const int k = k0 + u * 4 + wave;
      if (k >= a.k_vol) break;
      if (at[u] == kNoSlot || hit[u] == kNoRow) hit[u] = -1;
      found[lane][k - k0] = hit[u];
      const unsigned long long b = __ballot(hit[u] >= 0);
      if (lane == 0) count_of[k - k0] = __builtin_popcountll(b);
      if (a.rmask_out && hit[u] >= 0) {
        mine |= 1ull << k;
        if (a.rmask_in)
          (void)__hip_atomic_fetch_or(reinterpret_cast<unsigned *>(a.rmask_in + hit[u]) + (k >> 5), 1u << (k & 31),
                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
    // (the workgroup's counts in one instruction: a lane of every wave for itself took 3 us longer)
    if (threadIdx.x < kLookupChunk && k0 + (int)threadIdx.x < a.k_vol) {
      const int k = k0 + threadIdx.x;
      const int n = count_of[threadIdx.x];
      if (n) {
        atomicAdd(&a.counts[(size_t)k * a.blocks + block], n);
        if (a.totals) atomicAdd(&a.totals[blockIdx.x % kTotalCopies * 64 + k], n);
      }
    }
    // the chunk's part of every row, 16 bytes a thread
    const int width = min(kLookupChunk, a.row_ld - k0) / 4;
    for (int e = threadIdx.x; e < kLookupRows * width; e += 256) {
      const int r = e / width, c = e % width * 4, row = blockIdx.x * kLookupRows + r;
      if (row < a.n_out) {
        int4v_ v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = k0 + c + q < a.k_vol ? found[r][c + q] : -1;
        *reinterpret_cast<int4v_ *>(a.rows + (size_t)row * a.row_ld + k0 + c) = v;
      }
    }
    __syncthreads();
  }
  if (!a.rmask_out) return;
  wave_mask[wave][lane] = mine;
  __syncthreads();
  if (wave == 0 && live) a.rmask_out[o] = wave_mask[0][lane] | wave_mask[1][lane] | wave_mask[2][lane] | wave_mask[3][lane];
}

struct ScanArgs {
  const int32_t *counts;      // [k_vol][blocks]
  int32_t *bases;             // pairs before each of them, and the total behind
  int k_vol, blocks;
  int32_t *kernel_nnz, *kpos, *qkpos;      // (qkpos: nullptr: not wanted)
};

// Exclusive prefix sum by one workgroup, 4096 values a round: every thread takes four neighbouring
// values (the loads of a wave are contiguous; those of eight rounds are in flight together), the waves
// scan their threads' sums with lane shuffles, the 16 wave totals go through LDS, and the sum of the
// rounds so far is carried in a register.  The counts are few (offsets x 256-row blocks: 21 k for
// 200 k voxels), so one workgroup is enough; its first wave then writes the per-offset tables.
__global__ __launch_bounds__(1024) void kmap_scan_kernel(ScanArgs a) {
  __shared__ int wave_totals[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const size_t n = (size_t)a.k_vol * a.blocks;
  constexpr int kAhead = 8;
  int carry = 0, round = 0;
  for (size_t base0 = 0; base0 < n; base0 += 4096 * kAhead) {
    int v[kAhead][4];
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const size_t i = base0 + (size_t)q * 4096 + (size_t)tid * 4 + j;
        v[q][j] = i < n ? a.counts[i] : 0;
      }
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      const size_t i = base0 + (size_t)q * 4096 + (size_t)tid * 4;
      if (base0 + (size_t)q * 4096 >= n) break;
      const int mine = v[q][0] + v[q][1] + v[q][2] + v[q][3];
      int incl = mine;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d, 64);
        if (lane >= d) incl += up;
      }
      if (lane == 63) wave_totals[round][wave] = incl;
      __syncthreads();      // the other buffer is written next round, after every wave has passed this barrier
      int before = 0, total = 0;
#pragma unroll
      for (int w = 0; w < 16; ++w) {
        const int t = wave_totals[round][w];
        before += w < wave ? t : 0;
        total += t;
      }
      int run = carry + before + incl - mine;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (i + j < n) a.bases[i + j] = run;
        run += v[q][j];
      }
      carry += total;
      round ^= 1;
    }
  }
  if (tid == 0) a.bases[n] = carry;
  __threadfence_block();
  __syncthreads();
  if (wave != 0) return;
  int padded_before = 0;                       // (256-padded sizes of the offsets so far)
  for (int k0 = 0; k0 < a.k_vol; k0 += 64) {
    const int k = k0 + lane;
    int size = 0;
    if (k < a.k_vol) {
      const int first = a.bases[(size_t)k * a.blocks];
      size = a.bases[(size_t)(k + 1) * a.blocks] - first;
      a.kpos[k] = first;
      a.kernel_nnz[k] = size;
    }
    int padded = (size + 255) / 256 * 256;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(padded, d, 64);
      if (lane >= d) padded += up;
    }
    if (a.qkpos && k < a.k_vol) a.qkpos[k + 1] = padded_before + padded;
    padded_before += __shfl(padded, 63, 64);
  }
  if (lane == 0) {
    a.kpos[a.k_vol] = carry;
    if (a.qkpos) a.qkpos[0] = 0;
  }
}

struct ListArgs {
  const int32_t *rows;
  int n_out, k_vol, row_ld, blocks;
  const int32_t *bases;
  int32_t *in_map, *out_map;
  long long capacity;
  int32_t *band_start;        // of the plan, or nullptr
  int cus;
  const int32_t *kernel_nnz, *kpos;
  const int *flags;           // nullptr: the lookup's launch has sent them
  int *host;                  // pinned
};

// The sizes to the host; threads of the first wave.
__device__ __forceinline__ void publish_sizes(int k_vol, const int32_t *__restrict__ kernel_nnz, int pairs, int *__restrict__ host) {
  for (int k = threadIdx.x; k < min(k_vol, kHostInts - 16); k += 64) host[16 + k] = kernel_nnz[k];
  if (threadIdx.x == 0) host[4] = pairs;
  __threadfence_system();
  if (threadIdx.x == 0) __hip_atomic_store(&host[3], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// 256 output rows by THREADS threads, 28 offsets at a time through LDS (`tile`); a wave takes every (THREADS / 64)th offset
// and ranks its hits with ballots.
constexpr int kListWidth = 28, kListTile = kListRows * (kListWidth + 1);
template <int THREADS>
__device__ __forceinline__ void lists_body(const ListArgs &a, int list_block, int list_blocks, int32_t *__restrict__ tile) {
  constexpr int kWidth = kListWidth, kWaves = THREADS / 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
  const int row0 = list_block * kListRows;
  constexpr int kLoads = (kListRows * kWidth / 4 + THREADS - 1) / THREADS;      // 16-byte chunks of rows per thread
  constexpr int kTurns = (kWidth + kWaves - 1) / kWaves;                        // offsets per wave
  // bounds of the plan's row bands that fall into this block of rows (the last block has those behind
  // it, too): what lies below them inside the block is in the ballots anyway
  int bands = 0, band_rows = 1, c_first = 1, c_last = 0;
  if (a.band_start) {
    bands = band_count_of(a.kpos[a.k_vol], a.k_vol, a.cus);
    band_rows = (a.n_out + bands - 1) / bands;
    c_first = (row0 + band_rows - 1) / band_rows;
    c_last = list_block + 1 == list_blocks ? bands : min(bands, (row0 + kListRows - 1) / band_rows);
  }
  for (int k0 = 0; k0 < a.k_vol; k0 += kWidth) {
    const int width = min(kWidth, a.row_ld - k0) / 4, k_end = min(k0 + kWidth, a.k_vol);
    // (all of a part's loads in flight together)
    int4v_ v[kLoads];
    int block_first[kTurns], first[kTurns];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int e = threadIdx.x + THREADS * i, row = row0 + e / width;
      v[i] = int4v_{-1, -1, -1, -1};
      if (e < kListRows * width && row < a.n_out) v[i] = *reinterpret_cast<const int4v_ *>(a.rows + (size_t)row * a.row_ld + k0 + e % width * 4);
    }
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
      const size_t line = (size_t)min(k0 + wave + kWaves * i, a.k_vol - 1) * a.blocks;
      block_first[i] = a.bases[line + list_block];
      first[i] = a.bases[line];
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int e = threadIdx.x + THREADS * i;
      if (e >= kListRows * width) break;
#pragma unroll
      for (int q = 0; q < 4; ++q) tile[e / width * (kWidth + 1) + e % width * 4 + q] = v[i][q];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
      const int k = k0 + wave + kWaves * i;
      if (k >= k_end) break;
      const int before = block_first[i] - first[i];
      long long pos = block_first[i];
      unsigned long long hits[kListRows / 64];
#pragma unroll
      for (int q = 0; q < kListRows / 64; ++q) {
        const int r = q * 64 + lane, hit = tile[r * (kWidth + 1) + k - k0];
        const unsigned long long b = __ballot(hit >= 0);
        if (hit >= 0) {
          const long long at = pos + __builtin_popcountll(b & ((1ull << lane) - 1));
          if (at < a.capacity) {
            a.in_map[at] = hit;
            a.out_map[at] = row0 + r;
          }
        }
        pos += __builtin_popcountll(b);
        hits[q] = b;
      }
      for (int c = c_first + lane; c <= c_last; c += 64) {
        const long long end = (long long)c * band_rows - row0;      // rows of the block below the bound
        int below = before;
#pragma unroll
        for (int q = 0; q < kListRows / 64; ++q) {
          const long long r = end - q * 64;
          below += __builtin_popcountll(r >= 64 ? hits[q] : r > 0 ? hits[q] & ((1ull << r) - 1) : 0ull);
        }
        a.band_start[k * (bands + 1) + c] = below;
      }
    }
    __syncthreads();
  }
}

// Maps without a plan.  Workgroup 0 sends the sizes to the host, the others write the lists.
__global__ __launch_bounds__(256) void kmap_lists_kernel(ListArgs a, int list_blocks) {
  __shared__ int32_t tile[kListTile];
  if (blockIdx.x == 0) {
    if (threadIdx.x >= 64) return;
    publish_sizes(a.k_vol, a.kernel_nnz, a.kpos[a.k_vol], a.host);
    if (a.flags) publish_coordinates(a.flags, a.host);
    return;
  }
  lists_body<256>(a, blockIdx.x - 1, list_blocks, tile);
}

// Maps with a plan: its sort needs the row masks and the offsets' sizes only, so the lists keep out of its way.  Three launches,
// each of which runs what is ready side by side:
//   sizes   per-offset tables, and the sizes to the host (workgroup 0); the sort's histogram
//   bases   the sort's scan; pairs before every block of an offset (a workgroup per offset)
//   (the sort's scatter)
//   lists   the sort's windows, and next to them the lists
// (One workgroup scanning all counts, then lists and histogram, then scan, scatter and windows: 100 k LiDAR voxels x 27 offsets
// 8.3 + 12.7 + 5.4 + 9.7 + 11.6 us, so 7.0 + 4.5 + 8.9 + 13.4.  The lists next to the scatter instead, which needs 1 024 threads
// a workgroup: 200 k indoor voxels 25.2 us there and 11.4 for the windows, so 8.6 and 15.4.)
struct SizeArgs {
  const int32_t *totals;
  int32_t *kernel_nnz, *kpos, *qkpos;      // (qkpos: nullptr: not wanted)
  int *plan_flags;                         // flags[12] of the plan: its pair count; flags[9]
  int *host;                               // pinned
};
__global__ __launch_bounds__(kSortThreads) void kmap_sizes_kernel(SizeArgs a, SortArgs sort) {
  __shared__ int part[kSortThreads / 64][64];
  __shared__ int size_of[64];
  __shared__ int hist[kBins];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  auto sizes = [&]() -> const int * {
    constexpr int kWaves = kSortThreads / 64;
    int sum = 0;
#pragma unroll
    for (int c = 0; c < kTotalCopies / kWaves; ++c) sum += a.totals[(wave + kWaves * c) * 64 + lane];      // (0 from k_vol on)
    part[wave][lane] = sum;
    __syncthreads();
    if (wave == 0) {
      sum = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) sum += part[w][lane];
      size_of[lane] = sum;
    }
    __syncthreads();
    return size_of;
  };
  if (blockIdx.x > 0) {
    const int b = blockIdx.x - 1, side = b < sort.side[0].chunks ? 0 : 1;
    sort_hist_body(sort.side[side], sort, side ? b - sort.side[0].chunks : b, hist, sizes);
    return;
  }
  (void)sizes();
  if (wave != 0) return;
  const int mine = size_of[lane], k_vol = sort.k_vol;
  int upto = mine, padded = (mine + 255) / 256 * 256;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(upto, d, 64), padded_up = __shfl_up(padded, d, 64);
    if (lane >= d) {
      upto += up;
      padded += padded_up;
    }
  }
  if (lane < k_vol) {
    a.kernel_nnz[lane] = mine;
    a.kpos[lane] = upto - mine;
    if (a.qkpos) a.qkpos[lane + 1] = padded;
    a.host[16 + lane] = mine;
  }
  const int pairs = __shfl(upto, 63, 64);
  if (lane == 0) {
    a.kpos[k_vol] = pairs;
    if (a.qkpos) a.qkpos[0] = 0;
    a.plan_flags[12] = pairs;
    a.plan_flags[kFlagInput] = sort.side[1].n > 0;      // (a mirrored map's middle offset has every row for its own neighbour)
    a.host[4] = pairs;
  }
  __threadfence_system();
  if (lane == 0) __hip_atomic_store(&a.host[3], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct BaseArgs {
  const int32_t *counts, *kpos;
  int32_t *bases;
  int blocks, scans;          // workgroups of the sort's scan per side
};
__global__ __launch_bounds__(256) void kmap_bases_kernel(BaseArgs a, SortArgs sort) {
  const int sides = sort.side[1].n > 0 ? 2 : 1;
  int k = blockIdx.x - a.scans * sides;
  if (k < 0) {
    sort_scan_body(sort.side[blockIdx.x / a.scans], blockIdx.x % a.scans);
    return;
  }
  // exclusive prefix sum of an offset's line, four counts a thread and round
  __shared__ int wave_total[2][4];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int32_t *__restrict__ from = a.counts + (size_t)k * a.blocks;
  int32_t *__restrict__ to = a.bases + (size_t)k * a.blocks;
  int carry = a.kpos[k], round = 0;
  for (int base = 0; base < a.blocks; base += 1024, round ^= 1) {
    int v[4], mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = base + threadIdx.x * 4 + j;
      v[j] = i < a.blocks ? from[i] : 0;
      mine += v[j];
    }
    int incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64);
      if (lane >= d) incl += up;
    }
    if (lane == 63) wave_total[round][wave] = incl;
    __syncthreads();         // (the other buffer is written next round, after every wave has passed this barrier)
    int run = carry + incl - mine;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int t = wave_total[round][w];
      run += w < wave ? t : 0;
      carry += t;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = base + threadIdx.x * 4 + j;
      if (i < a.blocks) to[i] = run;
      run += v[j];
    }
  }
}

__global__ __launch_bounds__(kWindowThreads) void kmap_window_lists_kernel(ListArgs a, SortArgs sort, int windows, int list_blocks) {
  constexpr int kBuf = 2 * kWindow * (int)(sizeof(unsigned long long) / sizeof(int32_t));
  __shared__ __attribute__((aligned(16))) int32_t lds[kListTile > kBuf ? kListTile : kBuf];
  const int sides = sort.side[1].n > 0 ? 2 : 1, b = blockIdx.x;
  if (b < windows * sides) sort_window_body(sort, b / windows, b % windows, reinterpret_cast<unsigned long long *>(lds));
  else lists_body<kWindowThreads>(a, b - windows * sides, list_blocks, lds);
}

// Pinned read-back blocks, kept.
std::mutex g_host_mutex;
std::vector<int *> g_host_free;

int *host_block_get() {
  {
    std::lock_guard<std::mutex> lock(g_host_mutex);
    if (!g_host_free.empty()) {
      int *q = g_host_free.back();
      g_host_free.pop_back();
      return q;
    }
  }
  int *q = nullptr;
  note_allocation();
  if (hipHostMalloc((void **)&q, kHostInts * sizeof(int), hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) return nullptr;
  return q;
}

void host_block_put(int *q) {
  std::lock_guard<std::mutex> lock(g_host_mutex);
  g_host_free.push_back(q);
}

// Waits for a kernel's word, or, if that takes long, for everything queued so far.
int wait_for(volatile int *done, hipStream_t s) {
  for (int spins = 0; !*done; ++spins) {
    _mm_pause();
    if (spins > (1 << 20)) {
      FGMS_HIP_TRY(hipStreamSynchronize(s));
      if (*done) break;
      set_error("fgms_build_kernel_map: the build's kernels did not run");
      return FGMS_E_HIP;
    }
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  return FGMS_OK;
}

}  // namespace

// A build whose sizes have not been asked for yet.
struct MapBuild {
  int *host;
  hipStream_t stream;
  int k_vol;
  int64_t capacity, n_in, n_out;
  const int32_t *kernel_nnz, *kpos, *in_map, *out_map;
  Plan *plan;
  bool plan_from_lists;       // more offsets than one plan's tables hold
};

int map_build_begin(MapBuild **build, const int32_t *in_coords, int64_t n_in, const int32_t *out_coords, int64_t n_out,
                    const int32_t *offsets_host, int k_vol, int stride, int skip_offset,
                    int32_t *in_map, int32_t *out_map, int64_t capacity, int32_t *kernel_nnz,
                    int32_t *kpos, int32_t *qkpos, bool want_plan, bool allow_mirror, hipStream_t s) {
  *build = nullptr;
  {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone) {
      set_error("fgms_build_kernel_map: the stream is being captured (the build waits for its sizes)");
      return FGMS_E_INVALID;
    }
  }
  // the plan comes out of the same launches where its tables hold all offsets
  const bool with_plan = want_plan && k_vol <= 64 && n_in > 0 && n_out > 0;
  bool mirror = with_plan && allow_mirror && in_coords == out_coords && n_in == n_out && stride == 1 && k_vol % 2 == 1 &&
                (skip_offset < 0 || skip_offset == k_vol / 2);
  for (int k = 0; mirror && k < k_vol; ++k)
    for (int c = 0; c < 3; ++c)
      if (offsets_host[3 * (k_vol - 1 - k) + c] != -offsets_host[3 * k + c]) mirror = false;

  // (144 bytes of scratch a row, slots and cells, at every size)
  const unsigned buckets = (unsigned)((2 * (size_t)n_in + kBucket - 1) / kBucket + 1);
  const size_t slots = (size_t)buckets * kBucket;
  const int blocks = (int)((n_out + kListRows - 1) / kListRows);
  const int row_ld = (k_vol + 3) / 4 * 4;
  const size_t n_counts = (size_t)k_vol * blocks;

  int rc = FGMS_OK;
  Plan *p = with_plan ? plan_alloc(k_vol, n_in, n_out, 0, s) : nullptr;
  if (with_plan && !p) return FGMS_E_NOMEM;
  SortArgs sort{};
  sort.k_vol = k_vol;
  int cap_out = 0, cap_in = 0;
  const int tiles_out = with_plan ? tile_table(n_out, &cap_out) : 0, tiles_in = with_plan ? tile_table(n_in, &cap_in) : 0;
  const size_t so = (size_t)n_out * k_vol, si = mirror ? 0 : (size_t)n_in * k_vol;
  BlockKey *slot_table = nullptr;
  int32_t *cells = nullptr, *rows = nullptr, *counts = nullptr, *totals = nullptr, *bases = nullptr, *offs_dev = nullptr, *flags = nullptr;
  unsigned long long *rmask_out = nullptr, *rmask_in = nullptr;
  void *scratch = nullptr;
  auto layout = [&](Arena &keep, Arena &tmp) {
    tmp.take(slot_table, slots);
    tmp.take(cells, slots * kCells);
    tmp.take(rows, (size_t)n_out * row_ld);
    tmp.take(flags, 64);
    if (with_plan) tmp.take(totals, (size_t)kTotalCopies * 64);
    tmp.take(counts, n_counts);                     // (behind the flags: one fill)
    tmp.take(bases, n_counts + 1);
    if (k_vol > kKernargOffsets) tmp.take(offs_dev, (size_t)k_vol * 3);
    if (!with_plan) return;
    tmp.take(rmask_out, (size_t)n_out);
    if (!mirror) tmp.take(rmask_in, (size_t)n_in);
    sort_side_layout(sort.side[0], n_out, tmp);
    if (!mirror) sort_side_layout(sort.side[1], n_in, tmp);
    keep.take(p->flags, kPlanFlags);
    keep.take(p->band_start, (size_t)k_vol * (64 + 1));          // (the band count follows from the pair count)
    keep.take(p->band_cells, (size_t)4 * k_vol * 64);
    keep.take(p->nbr_out, so);
    if (!mirror) keep.take(p->nbr_in, si);
    keep.take(p->mask_out, (size_t)(n_out + 63) / 64);
    keep.take(p->perm_out, (size_t)n_out);
    if (!mirror) keep.take(p->mask_in, (size_t)(n_in + 63) / 64);
    if (!mirror) keep.take(p->perm_in, (size_t)n_in);
    if (tiles_out) keep.take(p->tile_out, (size_t)cap_out * 8);
    if (tiles_in && !mirror) keep.take(p->tile_in, (size_t)cap_in * 8);
  };
  int *host = host_block_get(), *host_dev = nullptr;
  auto fail = [&](int code) {
    (void)hipStreamSynchronize(s);
    if (scratch) pool_free(scratch, s, true);
    if (p) fgms_plan_destroy((fgms_plan_t *)p);
    if (host) host_block_put(host);
    return code;
  };
  if (!host || hipHostGetDevicePointer((void **)&host_dev, host, 0) != hipSuccess) {
    set_error("fgms_build_kernel_map: pinned allocation failed");
    return fail(FGMS_E_NOMEM);
  }
  host[0] = host[3] = 0;
  {
    Arena keep, tmp;
    layout(keep, tmp);
    if ((rc = pool_alloc(&scratch, tmp.used, s)) || (p && (rc = pool_alloc(&p->block, keep.used, s)))) return fail(rc);
    Arena keep_at, tmp_at;
    keep_at.base = p ? (char *)p->block : nullptr;
    tmp_at.base = (char *)scratch;
    layout(keep_at, tmp_at);
  }
  if (p) {
    p->kpos = kpos; p->in_map = in_map; p->out_map = out_map;
    p->has_tables = true;
    p->has_bands = true;
    if (mirror) {
      p->perm_in = p->perm_out;
      p->nbr_in = p->nbr_out;
      p->mask_in = p->mask_out;
      p->tile_in = p->tile_out;
      p->flip_in = k_vol - 1;
    }
    p->tile_grid_out = p->tile_out ? cap_out * 8 : 0;
    p->tile_grid_in = p->tile_in ? cap_in * 8 : 0;
    sort.flags = p->flags;
    sort.kpos = kpos;
    sort.side[0].rmask = rmask_out; sort.side[0].perm = p->perm_out; sort.side[0].block_mask = p->mask_out; sort.side[0].nbr = p->nbr_out;
    if (!mirror) {
      sort.side[1].rmask = rmask_in; sort.side[1].perm = p->perm_in; sort.side[1].block_mask = p->mask_in; sort.side[1].nbr = p->nbr_in;
    }
  }
  FillBatch fills{};
  fills.add(slot_table, slots * sizeof(BlockKey), -1);
  fills.add(cells, slots * kCells * sizeof(int32_t), kNoRow);
  fills.add(flags, (size_t)((char *)(counts + n_counts) - (char *)flags), 0);
  if (p) {
    fills.add(p->flags, kPlanFlags * sizeof(int), 0);
    if (!mirror) {
      fills.add(rmask_in, (size_t)n_in * sizeof(unsigned long long), 0);
      fills.add(p->nbr_in, si * sizeof(int32_t), -1);
    }
  }
  Offsets offs;
  if (offs_dev) {
    if (hipMemcpyAsync(offs_dev, offsets_host, (size_t)k_vol * 3 * sizeof(int32_t), hipMemcpyHostToDevice, s) != hipSuccess) {
      set_error("fgms_build_kernel_map: copying the offsets failed");
      return fail(FGMS_E_HIP);
    }
  } else {
    memcpy(offs.xyz, offsets_host, (size_t)k_vol * 3 * sizeof(int32_t));
  }
  if ((rc = launch_fills(fills, s))) return fail(rc);
  if (n_in > 0) {
    ProfileScope prof("kmap_insert_kernel", s);
    kmap_insert_kernel<<<(unsigned)((n_in + 255) / 256), 256, 0, s>>>(in_coords, (int)n_in, slot_table, buckets, cells, flags);
  }
  if (n_out > 0 && n_in > 0) {
    ProfileScope prof("kmap_lookup_kernel", s);
    LookupArgs la{out_coords, (int)n_out, k_vol, stride, skip_offset, row_ld, slot_table, cells, buckets, offs_dev,
                  rows, counts, totals, blocks, rmask_out, rmask_in, flags, host_dev};
    bool near = true;
    for (int q = 0; q < 3 * k_vol; ++q) near = near && offsets_host[q] >= -1 && offsets_host[q] <= 1;
    auto kern = near ? kmap_lookup_kernel<true> : kmap_lookup_kernel<false>;
    kern<<<(unsigned)((n_out + kLookupRows - 1) / kLookupRows) + 1, 256, 0, s>>>(la, offs);
  }
  ListArgs la{rows, (int)n_out, k_vol, row_ld, blocks, bases, in_map, out_map, (long long)capacity, p ? p->band_start : nullptr, num_cus(),
              kernel_nnz, kpos, n_out > 0 && n_in > 0 ? nullptr : flags, host_dev};
  const int list_blocks = n_in > 0 ? blocks : 0;
  if (p) {
    sort.by_mask = plan_sorts_rows();
    if (!sort.by_mask) sort.side[0].chunks = sort.side[1].chunks = 0;
    const int chunks = sort.side[0].chunks + sort.side[1].chunks, scans = chunks ? kBins / kScanBins : 0, sides = mirror ? 1 : 2;
    kmap_sizes_kernel<<<(unsigned)(1 + chunks), kSortThreads, 0, s>>>(SizeArgs{totals, kernel_nnz, kpos, qkpos, p->flags, host_dev}, sort);
    kmap_bases_kernel<<<(unsigned)(scans * sides + k_vol), 256, 0, s>>>(BaseArgs{counts, kpos, bases, blocks, scans}, sort);
    if (chunks && (rc = launch_sort_scatter(sort, s))) return fail(rc);
    ProfileScope prof("kmap_write_kernel", s);
    const int windows = (int)(((mirror || n_out > n_in ? n_out : n_in) + kWindow - 1) / kWindow);
    kmap_window_lists_kernel<<<(unsigned)(windows * sides + list_blocks), kWindowThreads, 0, s>>>(la, sort, windows, list_blocks);
  } else {
    kmap_scan_kernel<<<1, 1024, 0, s>>>(ScanArgs{counts, bases, k_vol, blocks, kernel_nnz, kpos, qkpos});
    ProfileScope prof("kmap_write_kernel", s);
    kmap_lists_kernel<<<(unsigned)(1 + list_blocks), 256, 0, s>>>(la, list_blocks);
  }
  if (hipGetLastError() != hipSuccess) {
    set_error("fgms_build_kernel_map: a kernel launch failed");
    return fail(FGMS_E_HIP);
  }
  if (p) {
    TablesArgs ta{};
    p->n_pairs = (int64_t)k_vol * n_out;         // (a bound; the count is known to the device only)
    plan_fill_tables_args(p, &ta);
    ta.rows = rows;
    ta.bands = 0;
    ta.bands_known = true;
    ta.row_ld = row_ld;
    ta.perm_out = p->perm_out;
    ta.nbr_out = p->nbr_out;
    if (!mirror) {
      ta.nbr_in = p->nbr_in;
      ta.inv_in = sort.side[1].inv;
    }
    ta.mirror = mirror;
    ta.take_print = true;
    if ((rc = launch_tables(ta, s)) || (rc = plan_publish(p, ta.host != nullptr, s))) return fail(rc);
  }
  // (the launches above are the longer way: the insertion's findings have arrived by now)
  if ((rc = wait_for(host, s))) return fail(rc);
  if (host[1]) {
    set_error("fgms_build_kernel_map: an input coordinate is outside [-2^20, 2^20)");
    return fail(FGMS_E_INVALID);
  }
  if (mirror && host[2]) {         // rows that share coordinates: the map is not its own mirror image
    (void)fail(FGMS_OK);
    return map_build_begin(build, in_coords, n_in, out_coords, n_out, offsets_host, k_vol, stride, skip_offset, in_map, out_map,
                           capacity, kernel_nnz, kpos, qkpos, want_plan, false, s);
  }
  pool_free(scratch, s, false);
  *build = new MapBuild{host, s, k_vol, capacity, n_in, n_out, kernel_nnz, kpos, in_map, out_map, p,
                        want_plan && !p && n_in > 0 && n_out > 0};
  return FGMS_OK;
}

// Waits for the build and takes it apart.
int map_build_end(MapBuild *b, int32_t *host_nnz, int64_t *n_pairs, fgms_plan_t **plan_out) {
  if (plan_out) *plan_out = nullptr;
  // (for the whole build: lists and tables can then be read on any stream)
  int rc = FGMS_OK;
  if ((b->plan ? hipEventSynchronize(b->plan->ready) : hipStreamSynchronize(b->stream)) != hipSuccess || !*(volatile int *)(b->host + 3)) {
    set_error("fgms_build_kernel_map: the build failed");
    rc = FGMS_E_HIP;
  }
  const int pairs = rc == FGMS_OK ? b->host[4] : 0;
  if (rc == FGMS_OK) {
    *n_pairs = pairs;
    if (host_nnz) {
      if (b->k_vol <= kHostInts - 16) {
        memcpy(host_nnz, b->host + 16, (size_t)b->k_vol * sizeof(int));
      } else if (hipMemcpyAsync(host_nnz, b->kernel_nnz, (size_t)b->k_vol * sizeof(int), hipMemcpyDeviceToHost, b->stream) != hipSuccess ||
                 hipStreamSynchronize(b->stream) != hipSuccess) {
        set_error("fgms_build_kernel_map: reading the sizes failed");
        rc = FGMS_E_HIP;
      }
    }
    if (pairs > b->capacity) {
      set_error("fgms_build_kernel_map: %d pairs do not fit the capacity of %lld", pairs, (long long)b->capacity);
      rc = FGMS_E_INVALID;
    }
  }
  if (rc == FGMS_OK && b->plan) {
    b->plan->n_pairs = pairs;
    plan_bands(b->plan);
    if (plan_out) {
      *plan_out = (fgms_plan_t *)b->plan;
      b->plan = nullptr;
    }
  } else if (rc == FGMS_OK && b->plan_from_lists && plan_out) {
    rc = plan_create(plan_out, b->kpos, b->in_map, b->out_map, b->n_in, b->n_out, b->k_vol, pairs, b->stream, true);
  }
  if (b->plan) fgms_plan_destroy((fgms_plan_t *)b->plan);
  host_block_put(b->host);
  delete b;
  return rc;
}

}  // namespace fgms
