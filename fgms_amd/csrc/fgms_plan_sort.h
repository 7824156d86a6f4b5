// Device code of a plan's row order: histogram, scan, scatter and window sort, for the launches of the two ways to a plan
// (fgms_plan.hip from pair lists, fgms_kmap.hip together with the map).
#pragma once

#include "fgms_plan_build.h"

namespace fgms {

// Bin of a key.
__device__ __forceinline__ int top_bits(unsigned long long key, int k_vol) {
  const int shift = k_vol > kBinBits ? k_vol - kBinBits : 0;
  return (int)((key >> shift) & (kBins - 1));
}

// A row's place among all sets of offsets: the set as a number whose high bits are the rare offsets,
// counted in Gray code, so that sets next to each other differ in few offsets.  Rows that have a rare
// offset are few: kept together they load few blocks with it.  (Counted with bins and
// windows of the sort's sizes, 64-row blocks x offsets over pairs / 64 on 120 k LiDAR voxels: by the mask
// as a number 1.39, rarest first 1.30, in Gray code too 1.28; 256-row tiles x offsets over pairs / 256
// 1.62, 1.47, 1.45; on 200 k indoor voxels 1.13, 1.12, 1.11 and 1.32, 1.28, 1.25.)
// The count in Gray code is linear: a set's key is the exclusive or of its offsets' keys, and that of an offset alone, bit p of the
// number, is all ones from p down.  key_of[k]: 64 entries of LDS; the caller's barrier publishes them.  (A lane per offset, compared
// through shuffles: one trip to memory instead of one per offset.)  `sizes`: the offsets' pairs, or nullptr: kpos has them.
__device__ __forceinline__ void sort_key_parts(const int32_t *__restrict__ kpos, int k_vol, unsigned long long *key_of, const int *sizes) {
  const int k = threadIdx.x;
  if (k >= 64) return;
  const int mine = k >= k_vol ? 0 : sizes ? sizes[k] : kpos[k + 1] - kpos[k];
  int rank = 0;
  for (int o = 0; o < k_vol; ++o) {
    const int theirs = __shfl(mine, o);
    rank += theirs < mine || (theirs == mine && o < k) ? 1 : 0;
  }
  key_of[k] = k < k_vol ? (2ull << (k_vol - 1 - rank)) - 1 : 0ull;
}
__device__ __forceinline__ unsigned long long sort_key(unsigned long long mask, int k_vol, const unsigned long long *key_of) {
  unsigned long long key = 0;
  for (int k = 0; k < k_vol; ++k) key ^= mask >> k & 1 ? key_of[k] : 0ull;
  return key;
}

// Keys and rows per bin of one chunk, by kSortThreads threads; `hist`: kBins ints of LDS.  A thread's rows are loaded and turned into
// keys side by side: latencies bound this, not bytes.  `sizes`: called while the rows are on their way, leaves the offsets' pairs in
// LDS or returns nullptr (kpos has them).  Keys come out of a table of the eight bits of a byte of the mask (offset by offset,
// 27 offsets, they were a third of the launch: 100 k rows 11.0 -> 7.0 us, together with sizes out of sums instead of counts).
template <typename F>
__device__ __forceinline__ void sort_hist_body(const SortSide &sd, const SortArgs &a, int chunk, int *hist, F &&sizes) {
  constexpr int kRows = kChunk / kSortThreads;
  __shared__ unsigned long long key_of[64];
  __shared__ unsigned long long of_byte[8][256];
  const int first = chunk * kChunk + threadIdx.x;
  unsigned long long mask[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) mask[r] = first + r * kSortThreads < sd.n ? sd.rmask[first + r * kSortThreads] : 0ull;
  sort_key_parts(a.kpos, a.k_vol, key_of, sizes());
  for (int i = threadIdx.x; i < kBins; i += kSortThreads) hist[i] = 0;
  __syncthreads();
  const int bytes = (a.k_vol + 7) / 8;
  for (int e = threadIdx.x; e < bytes * 256; e += kSortThreads) of_byte[e / 256][e % 256] = sort_key(e % 256, 8, key_of + e / 256 * 8);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    if (first + r * kSortThreads >= sd.n) break;
    unsigned long long key = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q < bytes) key ^= of_byte[q][mask[r] >> (8 * q) & 255];
    sd.key[first + r * kSortThreads] = key;
    atomicAdd(&hist[top_bits(key, a.k_vol)], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kBins; i += kSortThreads) sd.hist[(size_t)chunk * kBins + i] = hist[i];
}

// hist[chunk][bin] -> hist_before[chunk][bin] = rows of the bin in earlier chunks, and
// bin_total[bin].  Bins are independent: 64 of them per workgroup of 256 threads, a quarter of the
// chunks each (one workgroup alone reads the 800 KB of counts at 30 GB/s).
constexpr int kScanBins = 64;
__device__ __forceinline__ void sort_scan_body(const SortSide &sd, int block) {
  if (sd.chunks == 0) return;
  __shared__ int part_sum[4][kScanBins];
  const int part = threadIdx.x / kScanBins, b = threadIdx.x % kScanBins;
  const int bin = block * kScanBins + b;
  const int per = (sd.chunks + 3) / 4, c0 = min(part * per, sd.chunks), c1 = min(c0 + per, sd.chunks);
  const int32_t *__restrict__ h = sd.hist + bin;
  int32_t *__restrict__ hb = sd.hist_before + bin;
  int sum = 0;
#pragma unroll 8
  for (int c = c0; c < c1; ++c) sum += h[(size_t)c * kBins];
  part_sum[part][b] = sum;
  __syncthreads();
  int run = 0;
  for (int q = 0; q < part; ++q) run += part_sum[q][b];
#pragma unroll 8
  for (int c = c0; c < c1; ++c) {
    const int v = h[(size_t)c * kBins];
    hb[(size_t)c * kBins] = run;
    run += v;
  }
  if (part == 3) sd.bin_start[bin] = run;        // (the bin's total; the scatter kernel turns totals into starts)
}

// Value of the lane whose number differs from this lane's in bit J.
template <int J>
__device__ __forceinline__ unsigned lane_xor(unsigned v) {
  const int x = (int)v;
  if constexpr (J == 1) return (unsigned)__builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, true);           // quad_perm [1,0,3,2]
  else if constexpr (J == 2) return (unsigned)__builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, true);      // quad_perm [2,3,0,1]
  else if constexpr (J == 4)                                                                          // row_half_mirror, quad_perm [3,2,1,0]
    return (unsigned)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true);
  else if constexpr (J == 8) return (unsigned)__builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, true);     // row_ror:8
  else return (unsigned)__shfl_xor(x, J);
}
template <int J>
__device__ __forceinline__ unsigned long long lane_xor(unsigned long long v) {
  return (unsigned long long)lane_xor<J>((unsigned)v) | (unsigned long long)lane_xor<J>((unsigned)(v >> 32)) << 32;
}

// Bitonic sort of kWindow keys, ascending, by kWindowThreads threads: wave w holds elements w * 128 ...
// in two registers per lane (element w * 128 + r * 64 + lane in key[r]), so that 49 of the 55 phases
// are register exchanges inside a wave (most of them on the vector ALUs alone) and only the 6 with
// partners 128 or more apart go through LDS (`buf`: 2 x kWindow keys).  The vector ALUs are its
// limit, hence small windows on many CUs: 2048 keys by 1024 threads took 13 us, with every phase in LDS 25.
template <typename K, int K2, int J>
__device__ __forceinline__ void bitonic_phases(K (&key)[2], K *buf, int base, int lane, int &flip) {
  if constexpr (J >= 128) {
    K *to = buf + flip * kWindow;
    flip ^= 1;
    to[base + lane] = key[0];
    to[base + 64 + lane] = key[1];
    __syncthreads();
    const bool low = ((base & J) == 0) == ((base & K2) == 0);      // (J, K2 >= 128: bits of the wave's number)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const K o = to[(base ^ J) + r * 64 + lane];
      key[r] = (o < key[r]) == low ? o : key[r];
    }
  } else if constexpr (J == 64) {
    const bool asc = (base & K2) == 0;
    const K lo = key[0] < key[1] ? key[0] : key[1], hi = key[0] < key[1] ? key[1] : key[0];
    key[0] = asc ? lo : hi;
    key[1] = asc ? hi : lo;
  } else {
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int i = base + r * 64 + lane;
      const K o = lane_xor<J>(key[r]);
      const bool low = ((lane & J) == 0) == ((i & K2) == 0);
      key[r] = (o < key[r]) == low ? o : key[r];
    }
  }
  if constexpr (J > 1) bitonic_phases<K, K2, J / 2>(key, buf, base, lane, flip);
}
template <typename K, int K2 = 2>
__device__ __forceinline__ void bitonic_window(K (&key)[2], K *buf, int base, int lane, int &flip) {
  bitonic_phases<K, K2, K2 / 2>(key, buf, base, lane, flip);
  if constexpr (K2 < kWindow) bitonic_window<K, K2 * 2>(key, buf, base, lane, flip);
}

// Stable scatter of a chunk's rows into bin order.  Lanes of a wave that share a bin find each other
// with one ballot per bit of the bin; the waves then take their bins' counters in turn, the rows of a
// wave as one addition per bin.  (Sorting the chunk instead, in registers like the windows: 9 us.)  kSortThreads threads; `next`: kBins
// ints of LDS, where a bin's next row goes.
__device__ __forceinline__ void sort_scatter_body(const SortSide &sd, const SortArgs &a, int chunk, int *next) {
  __shared__ int part[kSortThreads / 64];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  constexpr int kBatches = kChunk / kSortThreads, kPer = kBins / kSortThreads;
  int bin[kBatches], rank[kBatches], peers[kBatches];
  bool first[kBatches];
  // (requested first, used last)
  int rows_of[kPer], before_of[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    rows_of[q] = sd.bin_start[threadIdx.x * kPer + q];
    before_of[q] = sd.hist_before[(size_t)chunk * kBins + threadIdx.x * kPer + q];
  }
#pragma unroll
  for (int r = 0; r < kBatches; ++r) {
    const int row = chunk * kChunk + (wave * kBatches + r) * 64 + lane;
    const bool live = row < sd.n;
    bin[r] = live ? top_bits(sd.key[row], a.k_vol) : -1;
    unsigned long long same = __ballot(live);
#pragma unroll
    for (int bit = 0; bit < kBinBits; ++bit) {
      const bool set = bin[r] >> bit & 1;
      const unsigned long long b = __ballot(set);
      same &= set ? b : ~b;
    }
    const unsigned long long below = same & ((1ull << lane) - 1);
    rank[r] = __builtin_popcountll(below);
    peers[r] = __builtin_popcountll(same);
    first[r] = live && below == 0;
  }
  // rows in smaller bins: exclusive scan of the bin totals (thread, wave, workgroup)
  {
    int local = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) local += rows_of[q];
    int incl = local;
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d);
      if (lane >= d) incl += up;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    int before = incl - local;
    for (int wv = 0; wv < wave; ++wv) before += part[wv];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int b = threadIdx.x * kPer + q;
      next[b] = before + before_of[q];
      before += rows_of[q];
    }
  }
  __syncthreads();
  int at[kBatches];
  for (int turn = 0; turn < kSortThreads / 64; ++turn) {
    if (wave == turn) {
#pragma unroll
      for (int r = 0; r < kBatches; ++r) {
        at[r] = bin[r] >= 0 ? next[bin[r]] : 0;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (first[r]) next[bin[r]] = at[r] + peers[r];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < kBatches; ++r)
    if (bin[r] >= 0) sd.perm_tmp[at[r] + rank[r]] = chunk * kChunk + (wave * kBatches + r) * 64 + lane;
}

// Full sort by (key, row) of a window of positions (of keys over more than 32 offsets: by the top
// 32 bits); writes the final order and its inverse, and what the window's blocks of 64 positions use:
// block_mask = the OR of their rows' masks, flags[4 + side] += (block, offset) combinations in use,
// flags[10 + side] += offset bits of all rows.  chunks == 0: the window starts from the identity
// order (sides of one window).  kWindowThreads threads; `buf`: 2 x kWindow keys of LDS.
__device__ __forceinline__ void sort_window_body(const SortArgs &a, int side, int window, unsigned long long *buf) {
  const SortSide &sd = a.side[side];
  const int p0 = window * kWindow;
  if (p0 >= sd.n) return;
  __shared__ int sums[kWindowThreads / 64][2];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, base = wave * 128;
  const int shift = a.k_vol > 32 ? a.k_vol - 32 : 0;
  unsigned long long key[2];
  __shared__ unsigned long long key_of[64];
  if (a.by_mask && sd.chunks == 0) {           // (no histogram has left keys)
    sort_key_parts(a.kpos, a.k_vol, key_of, nullptr);
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int p = p0 + base + r * 64 + lane;
    key[r] = ~0ull;
    if (p < sd.n) {
      const int row = sd.chunks ? sd.perm_tmp[p] : p;
      const unsigned long long full = !a.by_mask ? 0ull : sd.chunks ? sd.key[row] : sort_key(sd.rmask[row], a.k_vol, key_of);
      key[r] = (full >> shift) << 32 | (unsigned)row;
    }
  }
  int flip = 0;
  bitonic_window(key, buf, base, lane, flip);
  int bits = 0, row_bits = 0;
  const int centre = empty_centre(a.kpos, a.k_vol);
  if (window == 0 && side == 0 && wave == 0) {
    // (as many pairs as rows; that they are of different rows, and in order, is for the reader of the flags to ask)
    const int size = lane < a.k_vol ? a.kpos[lane + 1] - a.kpos[lane] : -1;
    const unsigned long long out = __ballot(size == a.side[0].n), in = __ballot(size == (a.side[1].n > 0 ? a.side[1].n : a.side[0].n));
    if (lane == 0) {
      a.flags[kFlagCentre] = centre >= 0;
      a.flags[kFlagFull] = (out ? __builtin_ctzll(out) + 1 : 0) | (in ? __builtin_ctzll(in) + 1 : 0) << 8;
    }
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int p = p0 + base + r * 64 + lane;
    unsigned long long m = 0;
    if (p < sd.n) {
      const int row = (int)(unsigned)key[r];
      sd.perm[p] = row;
      if (centre >= 0) sd.nbr[(size_t)centre * sd.n + p] = row;
      sd.inv[row] = p;
      m = sd.rmask[row];
    }
    int rb = __popcll(m);
    for (int d = 32; d > 0; d >>= 1) {
      m |= __shfl_xor(m, d);
      rb += __shfl_xor(rb, d);
    }
    if (p0 + base + r * 64 < sd.n) {
      const int block = (p0 + base) / 64 + r;
      if (lane == 0) sd.block_mask[block] = m;
      bits += __popcll(m);
      row_bits += rb;
    }
  }
  if (lane == 0) {
    sums[wave][0] = bits;
    sums[wave][1] = row_bits;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    int sum = 0;
    for (int i = 0; i < kWindowThreads / 64; ++i) sum += sums[i][threadIdx.x];
    if (sum) atomicAdd(&a.flags[(threadIdx.x ? 10 : 4) + side], sum);
  }
}

}  // namespace fgms
