// Layers with a narrow input side (1 .. 8 or, in fp16, 16 channels; up to 64 output channels), e.g. the
// 4 -> 32 first layer of a voxel network: forward and weight gradient on the matrix cores, through the
// plan's neighbour table.
//
// One (offset, channel) pair is one index of the contraction: a row's 27 neighbours of 4 channels are a
// row of 108 values, the weights [27][4][32] are a 108 x 32 matrix as they lie in memory.
//
//   forward          out[row][co] = sum over (k, ci) of in[nbr[k][row]][ci] * W[k][ci][co]
//   weight gradient  dW[(k, ci)][co] = sum over rows of in[nbr[k][row]][ci] * gout[row][co]
//
// The forward pass (fp16; on fp32 the matrix cores are no faster than the vector ALUs) needs no LDS for its rows: a lane of
// v_mfma_f32_32x32x16_f16 wants 8 consecutive contraction values of one row, i.e. two gathered rows of 4 channels or one of
// 8, which is what its gathers bring.  The weight gradient reads every output-gradient row once per row and not once per pair,
// and its gathers of 8-byte rows stay in the L2.
//
// Rows of 3, 5 or 7 halfs lie at odd 2-byte addresses: the aligned words around one are fetched and
// shifted, so that no padded copy is made of them.
//
// Bound by latency: a wave's few dependent loads (mask, index, row) and the launches.  4 -> 32 fp16 over 200 k voxels:
// forward 14 us (one lane per row and products on the vector ALUs: 20), weight gradient 18 + 4 (pair by pair: 33 + 4).
// 3 -> 32 over 125 offsets and 78 k voxels, both: 93 us with padded copies and the vector ALUs' kernels, 54 here.
#include "fgms_device.h"
#include "fgms_internal.h"
#include "fgms_mma.h"
#include "fgms_tile_ops.h"
#include "fgms_wgrad_bodies.h"

namespace fgms {
namespace {

typedef int int3v __attribute__((ext_vector_type(3)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));

constexpr int kNarrowCols = 64;                 // output channels at most
constexpr size_t kNarrowLds = 64 << 10;         // bytes the weights of a forward launch may take in LDS

// How a row of C channels is fetched.  SLOTS: contraction indices it takes (C and zeros behind).
// PARTS: lanes that share a row (16 halfs: two, 8 each).
template <typename T, int C>
struct NarrowRow {
  static constexpr bool kHalf = sizeof(T) == 2;
  static constexpr int SLOTS = C <= 4 ? 4 : C <= 8 ? 8 : 16;
  static constexpr int PARTS = SLOTS == 16 ? 2 : 1;
  static constexpr int W = kHalf ? (C == 16 ? 4 : (C + 1) / 2) : C;        // words fetched
  static constexpr int WS = SLOTS * (int)sizeof(T) / (4 * PARTS);          // words a lane holds of a row
  static_assert(kHalf ? C <= 8 || C == 16 : C == 4 || C == 8, "shape");

  __device__ static __forceinline__ unsigned offset(int row, int part) {
    if constexpr (C == 16) return (unsigned)row * 32u + (unsigned)part * 16u;
    else if constexpr (kHalf && C % 2 == 1) return ((unsigned)row * (2u * C)) & ~3u;
    else return (unsigned)row * (unsigned)(C * sizeof(T));
  }
  template <int N>
  __device__ static __forceinline__ void words(int *v, __amdgpu_buffer_rsrc_t rsrc, unsigned off) {
    if constexpr (N == 1) {
      v[0] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0);
    } else if constexpr (N == 2) {
      const int2v q = __builtin_bit_cast(int2v, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0));
      v[0] = q[0]; v[1] = q[1];
    } else if constexpr (N == 3) {
      const int3v q = __builtin_bit_cast(int3v, __builtin_amdgcn_raw_buffer_load_b96(rsrc, off, 0, 0));
      v[0] = q[0]; v[1] = q[1]; v[2] = q[2];
    } else {
      const int4v q = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
      v[0] = q[0]; v[1] = q[1]; v[2] = q[2]; v[3] = q[3];
    }
  }
  // (kAbsentRow: arrives as zeros)
  __device__ static __forceinline__ void load(int (&v)[WS], __amdgpu_buffer_rsrc_t rsrc, unsigned off) {
#pragma unroll
    for (int i = 0; i < WS; ++i) v[i] = 0;
    if constexpr (W <= 4) {
      words<W>(v, rsrc, off);
    } else {
      words<4>(v, rsrc, off);
      words<4>(v + 4, rsrc, off + 16);
    }
  }
  // The words around a row as its channels and zeros; `odd`: the row's number is.
  __device__ static __forceinline__ void settle(int (&v)[WS], unsigned odd) {
    if constexpr (kHalf && C % 2 == 1) {
      const unsigned shift = (odd & 1) * 16u;
#pragma unroll
      for (int i = 0; i < W; ++i) v[i] = (int)__builtin_amdgcn_alignbit(i + 1 < W ? (unsigned)v[i + 1] : 0u, (unsigned)v[i], shift);
      v[W - 1] &= 0xffff;
    }
  }
};

// Bytes of a tensor as a buffer's range, up to the end of its last word (odd counts of halfs; the word's
// other half is fetched and dropped).
size_t buffer_range(size_t bytes) { return (bytes + 3) & ~(size_t)3; }

struct NarrowFwd {
  const void *src, *w;
  void *dst;
  const int32_t *nbr;
  const unsigned long long *block_masks;
  const int32_t *perm;
  int n_dst, k_vol, c_out, overwrite, flip;
  unsigned src_bytes;
  SideJob side;
};

__device__ __forceinline__ unsigned long long uniform64(unsigned long long v) {
  return ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
         (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(v & 0xffffffffu));
}

template <typename T> __device__ __forceinline__ bool finite(T v) { return __builtin_fabsf(to_float(v)) < __builtin_inff(); }

// A wave owns 32 rows of the plan's order.  It walks the offsets that their 64-row block uses, 16 at a
// time (8 for 16 channels or wide fp32 rows): indices, gathers and matrix steps of a round are
// independent of each other, so a round is two memory latencies whatever its number of offsets.  The
// operands are swapped (weights as rows, gathered rows as columns), so that a lane ends up with four
// neighbouring channels of one row, four times, and stores them as they are.
// A weight that is not finite would reach rows without a pair through its offset (a zero row times
// infinity): a workgroup that meets one takes its products one by one.
template <int C, int NT>
__global__ __launch_bounds__(512, 4) void gms_narrow_kernel(NarrowFwd a) {
  using T = __half;
  using Row = NarrowRow<T, C>;
  constexpr int SLOTS = Row::SLOTS, WS = Row::WS, COLS = NT * 32;
  constexpr int LOADS = 8;                                                // rows a lane fetches a round
  constexpr int ROUND = SLOTS == 16 ? LOADS : 2 * LOADS;                  // offsets of a round
  int block_x = blockIdx.x;
  if (a.side.blocks) {
    if (block_x < a.side.blocks) {
      run_side_job(a.side, block_x);
      return;
    }
    block_x -= a.side.blocks;
  }
  extern __shared__ __align__(16) char narrow_lds[];
  T *w_lds = reinterpret_cast<T *>(narrow_lds);                           // [k][part][column][slots of a part]
  const T *w = reinterpret_cast<const T *>(a.w);
  const int lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
  const int tile = block_x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int p = tile * 32 + col, pc = min(p, a.n_dst - 1);
  unsigned long long todo = 0;
  if ((size_t)tile * 32 < (size_t)a.n_dst) todo = uniform64(a.block_masks[tile >> 1]);
  const bool touched = todo != 0;
  const __amdgpu_buffer_rsrc_t rsrc = rows_resource(a.src, a.src_bytes);

  int kk[LOADS], row[LOADS];
  int x[LOADS][WS];
  auto request = [&]() {      // indices and rows of the next ROUND offsets
    const int first = todo ? __builtin_ctzll(todo) : 0;
    int k[ROUND];
#pragma unroll
    for (int i = 0; i < ROUND; ++i) {
      k[i] = todo ? __builtin_ctzll(todo) : -1;
      todo &= todo - 1;
    }
    bool live[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int mine;
      if constexpr (SLOTS == 16) mine = k[i];
      else if constexpr (SLOTS == 4) mine = h ? k[4 * (i / 2) + 2 + i % 2] : k[4 * (i / 2) + i % 2];
      else mine = h ? k[2 * i + 1] : k[2 * i];
      live[i] = mine >= 0 && p < a.n_dst;
      kk[i] = mine >= 0 ? mine : first;
      row[i] = a.nbr[(size_t)kk[i] * a.n_dst + pc];
    }
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (!live[i]) row[i] = -1;
      Row::load(x[i], rsrc, row[i] < 0 ? kAbsentRow : Row::offset(row[i], h));
    }
  };
  request();

  // the weights, while the first rows are on their way
  bool odd = false;
  for (int e = threadIdx.x; e < a.k_vol * COLS; e += blockDim.x) {
    const int k = e / COLS, cd = e % COLS;
    const T *from = w + (size_t)(a.flip ? a.flip - k : k) * C * a.c_out + cd;
    T v[SLOTS];
#pragma unroll
    for (int c = 0; c < SLOTS; ++c) {
      v[c] = T(0.f);
      if (c < C && cd < a.c_out) v[c] = from[(size_t)c * a.c_out];
      odd = odd || !finite(v[c]);
    }
#pragma unroll
    for (int part = 0; part < Row::PARTS; ++part)
#pragma unroll
      for (int c = 0; c < SLOTS / Row::PARTS; ++c)
        w_lds[((size_t)(k * Row::PARTS + part) * COLS + cd) * (SLOTS / Row::PARTS) + c] = v[part * 8 + c];
  }
  const bool one_by_one = __syncthreads_or(odd);

  float16v acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nt][r] = 0.f;
  if (touched && one_by_one) {
    unsigned long long all = uniform64(a.block_masks[tile >> 1]);
    for (; all; all &= all - 1) {
      const int k = __builtin_ctzll(all);
      const int from = p < a.n_dst ? a.nbr[(size_t)k * a.n_dst + pc] : -1;
      if (from < 0) continue;
      for (int c = 0; c < C; ++c) {
        const float v = to_float(reinterpret_cast<const T *>(a.src)[(size_t)from * C + c]);
        const T *wk = w + ((size_t)(a.flip ? a.flip - k : k) * C + c) * a.c_out;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int cd = nt * 32 + (r / 4) * 8 + h * 4 + r % 4;
            if (cd < a.c_out) acc[nt][r] += v * to_float(wk[cd]);
          }
      }
    }
  } else if (touched) {
    while (true) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) Row::settle(x[i], (unsigned)row[i]);
      if constexpr (SLOTS == 4) {
#pragma unroll
        for (int s = 0; s < LOADS / 2; ++s) {
          const int4v b = {x[2 * s][0], x[2 * s][1], x[2 * s + 1][0], x[2 * s + 1][1]};
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            const int2v w0 = *reinterpret_cast<const int2v *>(w_lds + ((size_t)kk[2 * s] * COLS + nt * 32 + col) * 4);
            const int2v w1 = *reinterpret_cast<const int2v *>(w_lds + ((size_t)kk[2 * s + 1] * COLS + nt * 32 + col) * 4);
            mma<T>(acc[nt], int4v{w0[0], w0[1], w1[0], w1[1]}, b);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
          const int4v b = {x[i][0], x[i][1], x[i][2], x[i][3]};
          const int at = SLOTS == 16 ? kk[i] * 2 + h : kk[i];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            mma<T>(acc[nt], *reinterpret_cast<const int4v *>(w_lds + ((size_t)at * COLS + nt * 32 + col) * 8), b);
        }
      }
      if (!todo) break;
      request();
    }
  }
  // (a block no pair touches leaves its rows alone; overwrite: is zeroed)
  if (p >= a.n_dst || !(touched || a.overwrite)) return;
  T *out = reinterpret_cast<T *>(a.dst) + (size_t)(a.perm ? a.perm[p] : p) * a.c_out;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int cd = nt * 32 + g * 8 + h * 4;
      if (cd >= a.c_out) continue;
      half4v v = 0;
      if (!a.overwrite) v = *reinterpret_cast<const half4v *>(out + cd);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = (_Float16)((float)v[j] + acc[nt][g * 4 + j]);
      *reinterpret_cast<half4v *>(out + cd) = v;
    }
}

// ---------------------------------------------------------------------------
// Tables of up to 64 offsets: larger kernels have several sets, each with a row order of its own.
struct NarrowTables {
  const int32_t *nbr;
  const unsigned long long *block_masks;
  const int32_t *perm;
};
constexpr int kGroupOffsets = 64, kNarrowGroups = 6;      // (up to 384 offsets: 7 x 7 x 7)

struct NarrowWgrad {
  const void *in, *gout;
  float *partial;                               // [blockIdx.y][workgroup][128 slots][32]
  NarrowTables group[kNarrowGroups];
  int n_out, k_vol, c_out, col_blocks;
  unsigned in_bytes, gout_bytes;
  SideJob side;
};

constexpr int kTileBlocks = 4;                  // 32-slot blocks of (offset, channel) a wave accumulates
template <typename T> constexpr int narrow_wgrad_threads() { return sizeof(T) == 2 ? 1024 : 512; }

// A wave takes 32 rows at a time and holds dW for 128 (offset, channel) slots x 32 output channels in
// its accumulators; blockIdx.y walks the slots (of all
// groups of offsets) and the output channels.  The rows' gathered values and
// output gradients pass through the wave's own piece of LDS, which fp16 fragments leave transposed.  The
// waves of a workgroup meet in LDS; the workgroups leave a tile of sums each, which narrow_sums_kernel adds up
// (atomics instead: every workgroup has something for every element, and 256 adds to one address
// follow each other: 96 us for the launch).
// A row's output gradient is multiplied by zero where it has no pair: tiles in which one is not finite
// are left out and taken product by product afterwards, so that it stays out of those offsets.
template <typename T, int C>
__global__ __launch_bounds__(narrow_wgrad_threads<T>()) void wgrad_narrow_kernel(NarrowWgrad a) {
  using Row = NarrowRow<T, C>;
  constexpr bool kHalf = sizeof(T) == 2;
  constexpr int SLOTS = Row::SLOTS, WS = Row::WS;
  constexpr int THREADS = narrow_wgrad_threads<T>(), WAVES = THREADS / 64;
  constexpr int PIECES = 32 / SLOTS * Row::PARTS;          // lanes side by side on a row's block of 32 slots
  constexpr int ITS = PIECES * 32 / 64;                    // gathers a lane makes for a block
  constexpr int OFFSETS = 32 / SLOTS;                      // offsets of a block
  constexpr int GCHUNKS = 32 * (int)sizeof(T) / 16;        // 16-byte chunks of 32 output channels
  constexpr int GITS = GCHUNKS * 32 / 64;
  constexpr int LINE = 32 * (int)sizeof(T) / 4;            // words of 32 slots or channels
  int block_x = blockIdx.x;
  if (a.side.blocks) {
    if (block_x < a.side.blocks) {
      if (blockIdx.y == 0) run_side_job(a.side, block_x);
      return;
    }
    block_x -= a.side.blocks;
  }
  extern __shared__ __align__(16) char narrow_lds[];
  float *meet = reinterpret_cast<float *>(narrow_lds);                             // [waves][32 slots][32]
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  int *stage = reinterpret_cast<int *>(narrow_lds) + (size_t)wave * 32 * LINE;
  const int h = lane >> 5, col = lane & 31;
  const int k0 = (int)(blockIdx.y / a.col_blocks) * (kTileBlocks * OFFSETS), co0 = (int)(blockIdx.y % a.col_blocks) * 32;
  const int k_here = min(a.k_vol - k0, kTileBlocks * OFFSETS), group0 = k0 / kGroupOffsets * kGroupOffsets;
  const NarrowTables t = a.group[k0 / kGroupOffsets];
  const unsigned chunk_bits = k_here >= 32 ? ~0u : (1u << k_here) - 1;
  const __amdgpu_buffer_rsrc_t in_rsrc = rows_resource(a.in, a.in_bytes), gout_rsrc = rows_resource(a.gout, a.gout_bytes);

  float16v acc[kTileBlocks];
#pragma unroll
  for (int b = 0; b < kTileBlocks; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
  bool apart = false;
  const int tiles = (a.n_out + 31) / 32;
  const int walkers = (int)(gridDim.x - a.side.blocks) * WAVES;
  // (neighbouring tiles go to different workgroups, so that a small cloud fills the chip)
  for (int tile = block_x + wave * (walkers / WAVES); tile < tiles; tile += walkers) {
    const unsigned bits = (unsigned)(uniform64(t.block_masks[tile >> 1]) >> (k0 - group0)) & chunk_bits;
    if (!bits) continue;
    const int first = __builtin_ctz(bits), p0 = tile * 32;
    int grow[GITS];
#pragma unroll
    for (int it = 0; it < GITS; ++it) {
      const int p = min(p0 + it * (64 / GCHUNKS) + lane / GCHUNKS, a.n_out - 1);
      grow[it] = t.perm ? t.perm[p] : p;
    }
    int row[kTileBlocks][ITS];
#pragma unroll
    for (int b = 0; b < kTileBlocks; ++b)
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        const int q = b * OFFSETS + lane % PIECES / Row::PARTS, p = p0 + it * (64 / PIECES) + lane / PIECES;
        const int k = k0 + (bits >> q & 1 ? q : first);
        row[b][it] = t.nbr[(size_t)(k - group0) * a.n_out + min(p, a.n_out - 1)];
      }
    int4v g[GITS];
#pragma unroll
    for (int it = 0; it < GITS; ++it) {
      const int p = p0 + it * (64 / GCHUNKS) + lane / GCHUNKS, c = co0 + lane % GCHUNKS * (16 / (int)sizeof(T));
      const bool live = p < a.n_out && c < a.c_out;
      g[it] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(
                  gout_rsrc, live ? (unsigned)(((size_t)grow[it] * a.c_out + c) * sizeof(T)) : kAbsentRow, 0, 0));
    }
    int x[kTileBlocks][ITS][WS];
    unsigned odd_rows = 0;        // a bit per gather: the row's number is odd
#pragma unroll
    for (int b = 0; b < kTileBlocks; ++b)
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        const int q = b * OFFSETS + lane % PIECES / Row::PARTS, p = p0 + it * (64 / PIECES) + lane / PIECES;
        if (!(bits >> q & 1) || p >= a.n_out) row[b][it] = -1;
        odd_rows |= (unsigned)(row[b][it] & 1) << (b * ITS + it);
        Row::load(x[b][it], in_rsrc, row[b][it] < 0 ? kAbsentRow : Row::offset(row[b][it], lane % Row::PARTS));
      }
    bool odd = false;
#pragma unroll
    for (int it = 0; it < GITS; ++it)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (kHalf) odd = odd || (g[it][e] & 0x7c00) == 0x7c00 || (g[it][e] & 0x7c000000) == 0x7c000000;
        else odd = odd || (g[it][e] & 0x7f800000) == 0x7f800000;
      }
    if (__ballot(odd)) {
      apart = true;
      continue;
    }
    // output gradients: 32 rows x 32 channels through LDS into the fragments that all blocks share
    wave_lds_fence();
#pragma unroll
    for (int it = 0; it < GITS; ++it) *reinterpret_cast<int4v *>(stage + (it * 64 + lane) * 4) = g[it];
    wave_lds_fence();
    half8 gf[2];
    float gs[16];
    if constexpr (kHalf) {
#pragma unroll
      for (int s = 0; s < 2; ++s) gf[s] = tr_frag_dense<32>(reinterpret_cast<const __half *>(stage), s * 16, 0, lane);
    } else {
#pragma unroll
      for (int s = 0; s < 16; ++s) gs[s] = __builtin_bit_cast(float, stage[(2 * s + h) * LINE + col]);
    }
#pragma unroll
    for (int b = 0; b < kTileBlocks; ++b) {
      if (!(bits >> (b * OFFSETS) & ((1u << OFFSETS) - 1))) continue;
      wave_lds_fence();
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        Row::settle(x[b][it], odd_rows >> (b * ITS + it));
        int *to = stage + (it * 64 + lane) * WS;
        if constexpr (WS == 2) {
          *reinterpret_cast<int2v *>(to) = int2v{x[b][it][0], x[b][it][1]};
        } else {
#pragma unroll
          for (int q = 0; q < WS / 4; ++q)
            *reinterpret_cast<int4v *>(to + 4 * q) = int4v{x[b][it][4 * q], x[b][it][4 * q + 1], x[b][it][4 * q + 2], x[b][it][4 * q + 3]};
        }
      }
      wave_lds_fence();
      if constexpr (kHalf) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(tr_frag_dense<32>(reinterpret_cast<const __half *>(stage), s * 16, 0, lane),
                                                          gf[s], acc[b], 0, 0, 0);
      } else {
#pragma unroll
        for (int s = 0; s < 16; ++s)
          acc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, stage[(2 * s + h) * LINE + col]), gs[s], acc[b], 0, 0, 0);
      }
    }
  }
  // the waves' tiles, a block at a time: all write theirs, every thread adds up its elements of it
  float *mine = a.partial + ((size_t)blockIdx.y * (gridDim.x - a.side.blocks) + block_x) * (kTileBlocks * 32 * 32);
#pragma unroll
  for (int b = 0; b < kTileBlocks; ++b) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) meet[(wave * 32 + (r / 4) * 8 + h * 4 + r % 4) * 32 + col] = acc[b][r];
    __syncthreads();
#pragma unroll
    for (int e = threadIdx.x; e < 32 * 32; e += THREADS) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) v += meet[w * 32 * 32 + e];
      mine[b * 32 * 32 + e] = v;
    }
  }
  if (!__syncthreads_or(apart)) return;
  __threadfence();          // (a fence of every workgroup of the launch would double its time)
  __syncthreads();
  for (int tile = block_x + wave * (walkers / WAVES); tile < tiles; tile += walkers) {
    const unsigned bits = (unsigned)(uniform64(t.block_masks[tile >> 1]) >> (k0 - group0)) & chunk_bits;
    bool odd = false;
    for (int r = 0; r < 32; ++r) {
      const int p = tile * 32 + r;
      if (p < a.n_out && co0 + col < a.c_out)
        odd = odd || !finite(reinterpret_cast<const T *>(a.gout)[(size_t)(t.perm ? t.perm[p] : p) * a.c_out + co0 + col]);
    }
    if (!bits || !__ballot(odd) || h || co0 + col >= a.c_out) continue;
    for (int p = tile * 32; p < min(tile * 32 + 32, a.n_out); ++p) {
      const float g = to_float(reinterpret_cast<const T *>(a.gout)[(size_t)(t.perm ? t.perm[p] : p) * a.c_out + co0 + col]);
      for (unsigned m = bits; m; m &= m - 1) {
        const int q = __builtin_ctz(m), s = t.nbr[(size_t)(k0 - group0 + q) * a.n_out + p];
        for (int c = 0; s >= 0 && c < C; ++c)
          atomic_add(mine + (q * SLOTS + c) * 32 + col, to_float(reinterpret_cast<const T *>(a.in)[(size_t)s * C + c]) * g);
      }
    }
  }
}

// gw (+)= the workgroups' sums, rounded once.  A workgroup takes 32 output channels of one (offset, channel):
// eight runs of threads share the partial sums.
template <typename T>
__global__ __launch_bounds__(256) void narrow_sums_kernel(const float *__restrict__ partial, T *__restrict__ gw, int walkers,
                                                          int slots, int c_in, int c_out, int col_blocks, int flip, int overwrite,
                                                          SideJob side) {
  __shared__ float part[8][32];
  int block_x = blockIdx.x;
  if (side.blocks) {
    if (block_x < side.blocks) {
      run_side_job(side, block_x);
      return;
    }
    block_x -= side.blocks;
  }
  const int cb = block_x % col_blocks, kc = block_x / col_blocks, k = kc / c_in, c = kc % c_in;
  const int col = threadIdx.x % 32, run = threadIdx.x / 32, offsets = kTileBlocks * 32 / slots;
  const float *from = partial + ((size_t)(k / offsets * col_blocks + cb) * walkers) * (kTileBlocks * 32 * 32) +
                      (k % offsets * slots + c) * 32 + col;
  float sum = 0.f;
#pragma unroll 8
  for (int x = run; x < walkers; x += 8) sum += from[(size_t)x * (kTileBlocks * 32 * 32)];
  part[run][col] = sum;
  __syncthreads();
  const int co = cb * 32 + col;
  if (run != 0 || co >= c_out) return;
#pragma unroll
  for (int q = 1; q < 8; ++q) sum += part[q][col];
  T *to = gw + ((size_t)(flip ? flip - k : k) * c_in + c) * c_out + co;
  if (!overwrite) sum += to_float(*to);
  if constexpr (sizeof(T) == 2) *to = __float2half(sum);
  else *to = sum;
}

template <int C, int NT>
int launch_fwd(const GmsArgs &a, const Plan *p, size_t lds) {
  NarrowFwd n{a.src, a.w, a.dst, p->nbr_out, p->mask_out, p->perm_out, (int)a.n_dst, a.k_vol, a.c_out, a.overwrite ? 1 : 0,
              p->flip_out, (unsigned)buffer_range((size_t)a.n_src * C * sizeof(__half)), a.side};
  // (every workgroup reads all weights: bigger ones where these are many)
  const int threads = lds > (16 << 10) ? 512 : 256;
  const size_t tiles = ((size_t)a.n_dst + 31) / 32, per = threads / 64;
  auto kern = gms_narrow_kernel<C, NT>;
  { const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds); if (rc != FGMS_OK) return rc; }
  {
    ProfileScope prof("gms_narrow_kernel", a.stream);
    kern<<<(unsigned)((tiles + per - 1) / per) + (unsigned)a.side.blocks, threads, lds, a.stream>>>(n);
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

constexpr int kSlotPartials = 8;                // workspace of the workgroups' sums

// Workgroups of a weight gradient, one a CU or eight for each of blockIdx.y's range, whichever is more (each leaves a tile of
// sums), and that range.
struct NarrowGrid {
  size_t walkers;
  int ny, col_blocks;
  size_t bytes() const { return walkers * ny * (kTileBlocks * 32 * 32) * sizeof(float); }
};
NarrowGrid wgrad_grid(const WgradArgs &a) {
  NarrowGrid g;
  const int waves = (a.dtype == FGMS_F16 ? narrow_wgrad_threads<__half>() : narrow_wgrad_threads<float>()) / 64;
  const int offsets = kTileBlocks * 32 / (a.c_in <= 4 ? 4 : a.c_in <= 8 ? 8 : 16);
  g.col_blocks = (a.c_out + 31) / 32;
  g.ny = (a.k_vol + offsets - 1) / offsets * g.col_blocks;
  const size_t tiles = ((size_t)a.n_out + 31) / 32, most = (size_t)num_cus() / g.ny > 8 ? (size_t)num_cus() / g.ny : 8;
  g.walkers = (tiles + waves - 1) / waves < most ? (tiles + waves - 1) / waves : most;
  return g;
}

template <typename T, int C>
int launch_wgrad(const WgradArgs &a, const Plan *p) {
  constexpr int SLOTS = NarrowRow<T, C>::SLOTS, THREADS = narrow_wgrad_threads<T>();
  const NarrowGrid g = wgrad_grid(a);
  void *partial = nullptr;
  int rc = workspace_get(a.stream, kSlotPartials, g.bytes(), &partial);
  if (rc != FGMS_OK) return rc;
  NarrowWgrad n{};
  n.in = a.in; n.gout = a.gout; n.partial = (float *)partial;
  n.n_out = (int)a.n_out; n.k_vol = a.k_vol; n.c_out = a.c_out; n.col_blocks = g.col_blocks;
  n.in_bytes = (unsigned)buffer_range((size_t)a.n_in * C * sizeof(T));
  n.gout_bytes = (unsigned)((size_t)a.n_out * a.c_out * sizeof(T));
  n.side = a.side;
  // (pending fingerprint checks of the plan's groups ride along, one with either launch)
  SideJob second{};
  const std::vector<Plan *> alone{const_cast<Plan *>(p)}, &groups = p->groups.empty() ? alone : p->groups;
  for (size_t i = 0; i < groups.size(); ++i) {
    const Plan *q = groups[i];
    n.group[i] = NarrowTables{q->nbr_out, q->mask_out, q->perm_out};
    SideJob *free_job = !n.side.kind ? &n.side : !second.kind ? &second : nullptr;
    if (free_job) (void)plan_take_check(q, free_job);
  }
  const size_t lds = (size_t)THREADS / 64 * 32 * 32 * sizeof(float);
  auto kern = wgrad_narrow_kernel<T, C>;
  if ((rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds))) return rc;
  {
    ProfileScope prof("wgrad_narrow_kernel", a.stream);
    kern<<<dim3((unsigned)g.walkers + (unsigned)n.side.blocks, (unsigned)g.ny), THREADS, lds, a.stream>>>(n);
  }
  narrow_sums_kernel<T><<<(unsigned)(a.k_vol * C * g.col_blocks) + (unsigned)second.blocks, 256, 0, a.stream>>>(
      n.partial, (T *)a.gw, (int)g.walkers, SLOTS, C, a.c_out, g.col_blocks, p->flip_out, a.overwrite ? 1 : 0, second);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

size_t weights_lds(const GmsArgs &a) {
  return (size_t)a.k_vol * (a.c_in <= 4 ? 4 : a.c_in <= 8 ? 8 : 16) * ((a.c_out + 31) / 32 * 32) * sizeof(__half);
}

}  // namespace

bool narrow_gms_supported(const GmsArgs &a, const Plan *p) {
  if (!p || a.dtype != FGMS_F16 || a.transpose_w || a.dense_k >= 0 || a.k_vol > 64 || a.k_vol != p->k_vol || !p->has_tables || !p->nbr_out)
    return false;
  if (!p->fwd_ok || a.n_dst != p->n_out || a.n_src != p->n_in || a.n_dst == 0 || a.n_src == 0) return false;
  // (rows are fetched by words at 32-bit offsets and stored four channels at a time)
  return ((a.c_in >= 1 && a.c_in <= 8) || a.c_in == 16) && a.c_out <= kNarrowCols && a.c_out % 4 == 0 && weights_lds(a) <= kNarrowLds &&
         reinterpret_cast<uintptr_t>(a.src) % 4 == 0 && reinterpret_cast<uintptr_t>(a.dst) % 8 == 0 &&
         buffer_range((size_t)a.n_src * a.c_in * sizeof(__half)) <= kMaxBufferBytes;
}

int launch_narrow_gms(const GmsArgs &a, const Plan *p) {
  const size_t lds = weights_lds(a);
#define FGMS_NF(I) if (a.c_in == I) return a.c_out <= 32 ? launch_fwd<I, 1>(a, p, lds) : launch_fwd<I, 2>(a, p, lds);
  FGMS_NF(1) FGMS_NF(2) FGMS_NF(3) FGMS_NF(4) FGMS_NF(5) FGMS_NF(6) FGMS_NF(7) FGMS_NF(8) FGMS_NF(16)
#undef FGMS_NF
  set_error("launch_narrow_gms: unsupported shape");
  return FGMS_E_INVALID;
}

bool narrow_wgrad_supported(const WgradArgs &a, const Plan *p) {
  if (!p || a.k_vol != p->k_vol || a.crop_in || a.no_alloc) return false;
  auto tables = [&](const Plan *q) {
    return q->has_tables && q->nbr_out && q->fwd_ok && a.n_out == q->n_out && a.n_in == q->n_in && a.n_out > 0 && a.n_in > 0;
  };
  if (p->groups.empty()) {
    if (a.k_vol > kGroupOffsets || !tables(p)) return false;
  } else {
    if (p->groups.size() > (size_t)kNarrowGroups) return false;
    for (const Plan *q : p->groups)
      if (!tables(q) || q->flip_out || (q != p->groups.back() && q->k_vol != kGroupOffsets)) return false;
  }
  const size_t esz = a.dtype == FGMS_F16 ? 2 : 4;
  const bool channels = a.dtype == FGMS_F16 ? (a.c_in >= 1 && a.c_in <= 8) || a.c_in == 16
                                            : (a.c_in == 4 || a.c_in == 8) && (a.c_out == 32 || a.c_out == 64);
  // Where the vector ALUs' kernel takes the shape as it is, small launches are its: this one's two launches take 13 us
  // whatever the size (4 channels; 10.5 with 8 and 16, which always win in fp16).  27 offsets, vector ALUs / here:
  // 4 -> 32 fp16 20 k rows 12.9 / 14.5 us, 50 k 17.2 / 15.1, 200 k 38 / 22; 4 -> 64 5 k 11.6 / 13.1, 20 k 15.9 / 14.8;
  // 8 -> 32 fp32 10 k 13.7 / 14.1, 50 k 25.5 / 18.6; 16 -> 64 fp16 2 k 22.9 / 10.9, 50 k 65 / 19.
  const bool either = (a.c_out == 16 || a.c_out == 32 || a.c_out == 64) && (a.c_in == 4 || a.dtype != FGMS_F16);
  if (either && (double)a.n_out * a.c_out * a.k_vol < 27.0 * (1 << 20)) return false;
  return channels && a.c_out <= kNarrowCols && a.c_out * esz % 16 == 0 &&
         reinterpret_cast<uintptr_t>(a.in) % 4 == 0 && reinterpret_cast<uintptr_t>(a.gout) % 16 == 0 &&
         buffer_range((size_t)a.n_in * a.c_in * esz) <= kMaxBufferBytes &&
         // (a workspace cannot grow under stream capture)
         (!is_capturing(a.stream) || workspace_bytes(a.stream, kSlotPartials) >= wgrad_grid(a).bytes()) &&
         (size_t)a.n_out * a.c_out * esz <= kMaxBufferBytes;
}

int launch_narrow_wgrad(const WgradArgs &a, const Plan *p) {
#define FGMS_NW(T, I) if (a.c_in == I) return launch_wgrad<T, I>(a, p);
  if (a.dtype == FGMS_F16) {
    FGMS_NW(__half, 1) FGMS_NW(__half, 2) FGMS_NW(__half, 3) FGMS_NW(__half, 4) FGMS_NW(__half, 5)
    FGMS_NW(__half, 6) FGMS_NW(__half, 7) FGMS_NW(__half, 8) FGMS_NW(__half, 16)
  } else {
    FGMS_NW(float, 4) FGMS_NW(float, 8)
  }
#undef FGMS_NW
  set_error("launch_narrow_wgrad: unsupported shape");
  return FGMS_E_INVALID;
}

}  // namespace fgms
