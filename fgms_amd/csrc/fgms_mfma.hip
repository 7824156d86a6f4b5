// MFMA gather-GEMM-scatter kernels for gfx950 (forward and input gradient).
//
// Two dataflows share one fragment scheme:
//
//  * pair-stationary ("pairs"): a workgroup walks a run of 256-pair tiles of the
//    flat pair list, keeps op(W[k]) in LDS while the offset k does not change,
//    gathers the source rows through LDS and scatters the products with
//    atomics.  Works for any map.  This is the dataflow of the reference's fused
//    kernels (backend/spconv.cuh:1328-1477, backend/fwd_kernels.cuh:17-144,
//    backend/bwd_kernels.cuh:13-142, 281-408) re-tiled for 64-wide waves.
//  * output-stationary ("rows"): a workgroup owns 256 destination rows, walks the
//    offsets k through the plan's neighbour table, sums everything in MFMA
//    accumulators and writes each destination row once: no atomics, run-to-run
//    identical results.  Needs a plan whose map is functional.
//
// Fragment scheme.  A source row is cut into slabs of 2*S 16-byte chunks
// (S = 4, 2 or 1; a chunk is 8 halfs or 4 floats).  Lanes 0-31 of a wave carry
// the first S chunks of the slab, lanes 32-63 the last S, so one MFMA
// (v_mfma_f32_32x32x16_f16, or four v_mfma_f32_32x32x2_f32) contracts chunk s of
// both halves.  The order of the contraction index is free as long as both
// operands agree, and it lets every lane read one contiguous 16-byte piece.
// Weights are re-laid on the device into exactly that per-lane order before the
// main kernel runs (pack_weights_kernel), transposed for the input gradient.
//
// Gathered rows reach LDS with 16-byte loads, 2*S lanes per row (full 128-byte
// lines for S = 4), in an XOR-swizzled layout so that the b128 reads of the MFMA
// operand do not collide on banks.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "fgms_device.h"
#include "fgms_internal.h"
#include "fgms_mma.h"
#include "fgms_tile_ops.h"
#include "fgms_wgrad_bodies.h"

namespace fgms {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kWaveRows = 64;                 // two 32-row MFMA tiles per wave
constexpr int kTileRows = kWaves * kWaveRows; // 256 rows per workgroup tile

// ---------------------------------------------------------------------------
// Weight re-layout (see pack_weight_elements) in a launch of its own.
template <typename T>
__global__ void pack_weights_kernel(const T *__restrict__ w, T *__restrict__ packed, int k_vol,
                                    int c_in, int c_out, int S, bool transpose) {
  pack_weight_elements<T>(w, packed, k_vol, c_in, c_out, S, transpose,
                          (size_t)blockIdx.x * blockDim.x + threadIdx.x,
                          (size_t)gridDim.x * blockDim.x);
}

__global__ void side_job_kernel(SideJob job) { run_side_job(job, blockIdx.x); }

// Copies the packed weights of offset k, destination tiles [nt0, nt0 + NT), to LDS.
template <int NT>
__device__ __forceinline__ void load_weights(int4v *__restrict__ w_lds,
                                             const int4v *__restrict__ packed_k, int qs, int nts,
                                             int nt0) {
  const int n = qs * NT * 64;
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const int q = i / (NT * 64), rem = i % (NT * 64);
    w_lds[i] = packed_k[((size_t)q * nts + nt0) * 64 + rem];
  }
}

// The same for split weights (pack_weights_parts_kernel): per (slab, k-step) NT * 128 chunks.
template <int NT>
__device__ __forceinline__ void load_weights_split(int4v *__restrict__ w_lds,
                                                 const int4v *__restrict__ packed_k, int slabs, int nts,
                                                 int nt0) {
  const int n = slabs * 2 * NT * 128;
  for (int i = threadIdx.x; i < n; i += kThreads) {
    const int q = i / (NT * 128), rem = i % (NT * 128);
    w_lds[i] = packed_k[((size_t)q * nts + nt0) * 128 + rem];
  }
}

// acc[mt][nt] += A(slab) x W(slab).
template <typename T, int NT, int S, int MT>
__device__ __forceinline__ void mma_slab(float16v (&acc)[MT][NT], const int4v *__restrict__ a_lds,
                                         const int4v *__restrict__ w_lds, int slab, int lane) {
  const int h = lane / 32, r = lane % 32;
  if constexpr (sizeof(T) == 2 && NT <= 2) {
    // (pipelined like mma_slab_raw below: the next k-step's fragments are requested first)
    int4v a[2][MT], b[2][NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[0][nt] = w_lds[((slab * S) * NT + nt) * 64 + lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a[0][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S)];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      if (s + 1 < S) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) b[(s + 1) & 1][nt] = w_lds[((slab * S + s + 1) * NT + nt) * 64 + lane];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[(s + 1) & 1][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S + s + 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a[s & 1][mt], b[s & 1][nt]);
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
#pragma unroll
  for (int s = 0; s < S; ++s) {
    int4v b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) b[nt] = w_lds[((slab * S + s) * NT + nt) * 64 + lane];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int4v a = a_lds[a_slot<S>(mt * 32 + r, h * S + s)];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a, b[nt]);
    }
  }
}

// The MFMA phase of a stage, software-pipelined by hand: the fragments of k-step s + 1 are
// requested from LDS before the MFMAs of k-step s are issued (two sets of fragment registers),
// so that a wave's matrix instructions follow each other instead of each pair waiting out an
// LDS round trip.  The scheduling barriers keep the compiler from sinking the reads back to
// their uses (left alone it emits read, wait, two MFMAs, read, wait, ... in source order).
// acc[mt][nt] += A(slab) x W(slab), weights as raw_weight_frag reads them.
template <typename T, int NT, int S, int MT>
__device__ __forceinline__ void mma_slab_raw(float16v (&acc)[MT][NT], const int4v *__restrict__ a_lds,
                                             const int4v *__restrict__ w_lds, int lane) {
  const int h = lane / 32, r = lane % 32;
  int4v a[2][MT], b[2][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) b[0][nt] = raw_weight_frag<NT, S>(w_lds, 0, nt, lane);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) a[0][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S)];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (s + 1 < S) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[(s + 1) & 1][nt] = raw_weight_frag<NT, S>(w_lds, s + 1, nt, lane);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[(s + 1) & 1][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S + s + 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a[s & 1][mt], b[s & 1][nt]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The same for fp32 (forward): the stage's 2*S*4 rows of W[k] as they lie, NT*32 columns each; a lane's four values of a
// k-step are four reads down a column.
template <int NT, int S, int MT>
__device__ __forceinline__ void mma_slab_raw32(float16v (&acc)[MT][NT], const int4v *__restrict__ a_lds,
                                               const int4v *__restrict__ w_lds, int lane) {
  const int h = lane / 32, r = lane % 32;
  const float *w = reinterpret_cast<const float *>(w_lds) + h * S * 4 * (NT * 32) + r;
#pragma unroll
  for (int s = 0; s < S; ++s) {
    int4v b[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float4v f;
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = w[(s * 4 + j) * (NT * 32) + nt * 32];
      b[nt] = __builtin_bit_cast(int4v, f);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int4v a = a_lds[a_slot<S>(mt * 32 + r, h * S + s)];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma<float>(acc[mt][nt], a, b[nt]);
    }
  }
}

// --- input-gradient weights straight from the caller's tensor --------------------------
// The input gradient contracts over the COLUMNS of W[k] (dIn[ci] = sum over co of
// dOut[co] * W[k][ci][co]), and those are contiguous in memory: the 8 halfs (4 floats) an
// MFMA lane wants are one 16-byte piece of row ci.  A stage's weight tile (NT*32 rows ci x
// 2*S chunks of the co slab) goes to LDS as it lies in memory, swizzled like a wave's
// staging tile of gathered rows, and a fragment is one 16-byte read.  No re-layout at all.
template <typename T, int NT, int S, int MT>
__device__ __forceinline__ void mma_slab_rawt(float16v (&acc)[MT][NT], const int4v *__restrict__ a_lds,
                                              const int4v *__restrict__ w_lds, int lane) {
  const int h = lane / 32, r = lane % 32;
  if constexpr (sizeof(T) == 4) {
    // (fp32: a k-step is sixteen MFMAs of 64 cycles, long enough to cover the next reads)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      int4v b[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[nt] = w_lds[a_slot<S>(nt * 32 + r, h * S + s)];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int4v a = a_lds[a_slot<S>(mt * 32 + r, h * S + s)];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a, b[nt]);
      }
    }
    return;
  }
  int4v a[2][MT], b[2][NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) b[0][nt] = w_lds[a_slot<S>(nt * 32 + r, h * S)];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) a[0][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S)];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    if (s + 1 < S) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[(s + 1) & 1][nt] = w_lds[a_slot<S>(nt * 32 + r, h * S + s + 1)];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) a[(s + 1) & 1][mt] = a_lds[a_slot<S>(mt * 32 + r, h * S + s + 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a[s & 1][mt], b[s & 1][nt]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// --- fp32 tensors, products in split bf16 ("tf32" mode) ------------------------------------
// gfx950 has no tf32 matrix instruction, and its fp32 one runs at a sixteenth of the 16-bit
// rate.  Where the caller allows tf32 precision for the products (10 mantissa bits), every
// fp32 value is split into two bf16 numbers, x = hi + lo + O(2^-17 x), and a product becomes
// three bf16 MFMAs into the fp32 accumulator: hi*hi + hi*lo + lo*hi.  The dropped lo*lo term
// is below 2^-16 of the product, so this is more exact than tf32, at 3/16 of the fp32 matrix
// time.  Rows are split when they go from registers to LDS, the weights by their re-layout
// kernel.
//
// The same for fp32 tensors in full precision, with three parts and eight products (RAW = 5 and 6): x = h + m + l holds
// all 24 bits, and a product is rounded once, as by fp32 arithmetic (mma_parts).  Eight 16-bit matrix steps take half of the
// fp32 ones' time; a tile of rows takes half as much LDS again, which leaves two workgroups to a CU.  fp32 MFMAs / this:
// 64 -> 64 forward over 40 k voxels 88 / 76 us, 200 k 227 / 165; backward 116 / 91, 398 / 319; 128 -> 128 over 40 k 249 / 161
// and 349 / 271; 32 -> 32 over 20 k 25.4 / 23.2 and 25.6 / 24.0.
// What the parts cannot hold goes to fp32 MFMAs (RAW = 7 and 8): sums that an infinite value reaches come out as NaN or infinite
// whatever else is in them, and a value too small for them (below 2^-102 at most) is noted when it is split, so that a
// workgroup that has met either does its work again before it writes its tile, in that tile at the price of both.
//
// Slot (16 bytes = 8 bf16) of a split tile of P parts: row-major, a row holds its 32 values of the slab
// as 4 chunks of each part; the XOR spreads the rows one b128 read pass (16 lanes) touches over all banks: rows of
// 128 bytes go by pairs, of 192 bytes by fours.
template <int P>
__device__ __forceinline__ int part_slot(int row, int part, int j) {
  return row * (4 * P) + part * 4 + (j ^ ((row >> (P == 3 ? 2 : 1)) & 3));
}

// One fp32 chunk (4 values; chunk c of its row's slab) split and written to a split tile: 8 bytes of each part.
template <int P>
__device__ __forceinline__ void split_and_store(int4v *__restrict__ tile, const float4v &x, int row, int c, bool &lost) {
  int2v part[P];
  split_parts<P>(x, part, lost);
#pragma unroll
  for (int q = 0; q < P; ++q) reinterpret_cast<int2v *>(tile)[part_slot<P>(row, q, c / 2) * 2 + (c & 1)] = part[q];
}

// registers -> LDS for the split tile of gathered rows (absent rows as zeros).
template <int P, int N>
__device__ __forceinline__ void gather_commit_parts(int4v *__restrict__ a_lds, int4v (&v)[N],
                                                    const int (&g)[N], int lane) {
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const int slot = it * 64 + lane;
    const float4v x = g[it] < 0 ? float4v{0.f, 0.f, 0.f, 0.f} : __builtin_bit_cast(float4v, v[it]);
    bool lost = false;      // (two parts: not used)
    split_and_store<P>(a_lds, x, slot / 8, slot % 8, lost);
  }
}

// acc[mt][nt] += A(slab) x W(slab), both split.  Weights in LDS as [k-step][nt][part][lane], or (AS_ROWS: the input
// gradient) as a split tile of the NT*32 rows of W[k], the slab's 32 columns.
template <int P, bool AS_ROWS, int NT, int MT>
__device__ __forceinline__ void mma_slab_parts(float16v (&acc)[MT][NT], float16v (&low)[P == 3 ? MT : 1][P == 3 ? NT : 1],
                                               const int4v *__restrict__ a_lds, const int4v *__restrict__ w_lds, int lane) {
  const int h = lane / 32, r = lane % 32;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    bf16x8 b[NT][P];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < P; ++q)
        b[nt][q] = __builtin_bit_cast(bf16x8, w_lds[AS_ROWS ? part_slot<P>(nt * 32 + r, q, s * 2 + h)
                                                            : ((s * NT + nt) * P + q) * 64 + lane]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      bf16x8 a[P];
#pragma unroll
      for (int q = 0; q < P; ++q) a[q] = __builtin_bit_cast(bf16x8, a_lds[part_slot<P>(mt * 32 + r, q, s * 2 + h)]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma_parts<P>(acc[mt][nt], low[P == 3 ? mt : 0][P == 3 ? nt : 0], a, b[nt]);
    }
  }
}

// Split weights in the order mma_slab_parts reads them: chunk
//   ((((k * slabs + slab) * 2 + s) * nts + nt) * P + part) * 64 + lane
// holds the 8 values op(W[k])[slab*32 + s*16 + (lane/32)*8 + 0..7][nt*32 + lane%32] of that part.
// One thread per P chunks.
// (Channels that fill no whole tile: zeros behind them.)
// A chunk with a weight that three parts do not hold is marked with a NaN, which takes every tile that meets it to fp32 MFMAs
// and the weights as they are.
template <int P>
__global__ void pack_weights_parts_kernel(const float *__restrict__ w, int4v *__restrict__ packed,
                                          int k_vol, int c_in, int c_out, bool transpose) {
  // (transpose: the input gradient's view, W[k]^T -- source channels are the columns of W[k])
  const int c_src = transpose ? c_out : c_in, c_dst = transpose ? c_in : c_out, slabs = (c_src + 31) / 32, nts = (c_dst + 31) / 32;
  const size_t total = (size_t)k_vol * slabs * 2 * nts * 64;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
       t += (size_t)gridDim.x * blockDim.x) {
    const int lane = (int)(t % 64);
    size_t q = t / 64;
    const int nt = (int)(q % nts); q /= nts;
    const int s = (int)(q % 2); q /= 2;
    const int slab = (int)(q % slabs);
    const int k = (int)(q / slabs);
    const int cs0 = slab * 32 + s * 16 + (lane / 32) * 8, cd = nt * 32 + lane % 32;
    float4v x[2];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      x[e / 4][e % 4] = cs0 + e >= c_src || cd >= c_dst ? 0.f
                        : transpose ? w[((size_t)k * c_in + cd) * c_out + cs0 + e] : w[((size_t)k * c_in + cs0 + e) * c_out + cd];
    int2v lo[P], hi[P];
    bool lost = false;
    split_parts<P>(x[0], lo, lost);
    split_parts<P>(x[1], hi, lost);
    if (P == 3 && lost) lo[0][0] = 0x7fc07fc0;
    const size_t base = (t / 64) * (64 * P) + lane;
#pragma unroll
    for (int part = 0; part < P; ++part) packed[base + part * 64] = int4v{lo[part][0], lo[part][1], hi[part][0], hi[part][1]};
  }
}

// ---------------------------------------------------------------------------
// Row gathers in two steps, so that the loads of one slab run under the MFMAs of the
// previous one: issue (global -> registers, absent rows read row 0) and commit
// (registers -> the wave's LDS tile, absent rows as zeros; waits for the loads).
// (N chunks per lane: 2 * S for a wave tile of 64 rows, S for one of 32)
template <typename T, int S, int N>
__device__ __forceinline__ void gather_issue(int4v (&v)[N], int (&g)[N],
                                             const int *__restrict__ idx,
                                             const T *__restrict__ src, int c_src, int slab,
                                             int lane) {
  constexpr int E = Elem<T>::per_chunk;
  constexpr int C = 2 * S;
#pragma unroll
  for (int it = 0; it < N; ++it) g[it] = idx[(it * 64 + lane) / C];
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const int c = (it * 64 + lane) % C;
    v[it] = *reinterpret_cast<const int4v *>(src + (size_t)max(g[it], 0) * c_src +
                                             (size_t)(slab * C + c) * E);
  }
}

template <int S, int N>
__device__ __forceinline__ void gather_commit(int4v *__restrict__ a_lds, int4v (&v)[N],
                                              const int (&g)[N], int lane) {
  constexpr int C = 2 * S;
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const int slot = it * 64 + lane;
    a_lds[a_slot<S>(slot / C, slot % C)] = g[it] < 0 ? int4v{0, 0, 0, 0} : v[it];
  }
}

// The same two steps for the output-stationary kernel, through buffer loads (see kAbsentRow):
// `offs` holds a byte offset per row of the wave's tile, kAbsentRow for a row that has no
// neighbour through this offset, which then arrives as zeros by itself: no select on the way
// to LDS, no row index kept per load, 32-bit address arithmetic.
// (RAGGED: the slab's chunks from row_bytes on do not exist either; TAILS: of a row's last chunk the first half does, see take_tail)
template <int S, bool RAGGED = false, bool TAILS = false, int N>
__device__ __forceinline__ void gather_issue_buf(int4v (&v)[N], const unsigned *__restrict__ offs,
                                                 __amdgpu_buffer_rsrc_t rsrc, int slab, int lane, unsigned row_bytes = 0) {
  constexpr int C = 2 * S;
  unsigned off[N];
#pragma unroll
  for (int it = 0; it < N; ++it) off[it] = offs[(it * 64 + lane) / C] + (unsigned)((64 % C == 0 ? lane % C : (it * 64 + lane) % C) * 16);
  if constexpr (TAILS) {
    // (the slab in the lane's offset: a row's half chunk may start in front of it)
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const unsigned at = (unsigned)((slab * C + (it * 64 + lane) % C) * 16);
      off[it] = at >= row_bytes ? kAbsentRow : off[it] + (unsigned)(slab * (C * 16)) - (at + 16 > row_bytes ? kTailBytes : 0u);
    }
  } else if constexpr (RAGGED) {
#pragma unroll
    for (int it = 0; it < N; ++it)
      if ((unsigned)((slab * C + (it * 64 + lane) % C) * 16) >= row_bytes) off[it] = kAbsentRow;
  }
#pragma unroll
  for (int it = 0; it < N; ++it)
    v[it] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[it], TAILS ? 0 : slab * (C * 16), 0));
}

// The rows of a slab that ends in half a chunk.
template <int S, int N>
__device__ __forceinline__ void take_row_tails(int4v (&v)[N], int slab, int lane, unsigned row_bytes) {
  constexpr int C = 2 * S;
#pragma unroll
  for (int it = 0; it < N; ++it) v[it] = take_tail(v[it], (unsigned)((slab * C + (it * 64 + lane) % C) * 16) + 16 > row_bytes);
}

template <int S, int N>
__device__ __forceinline__ void gather_commit_buf(int4v *__restrict__ a_lds, const int4v (&v)[N], int lane) {
  constexpr int C = 2 * S;
  if constexpr (C == 8) {
    // a_slot(it * 8 + lane / 8, lane % 8) spelled out: the swizzle term (row >> 1) & 7 is
    // lane / 16 for even `it` and lane / 16 + 4 for odd ones, so two per-lane bases and
    // immediate offsets address all N writes
    const int base = (lane / 8) * 8, c = lane % 8, x = lane / 16;
    const int even = base + (c ^ x), odd = base + (c ^ (x + 4));
#pragma unroll
    for (int it = 0; it < N; ++it) a_lds[((it & 1) ? odd : even) + it * 64] = v[it];
  } else {
#pragma unroll
    for (int it = 0; it < N; ++it) {
      const int slot = it * 64 + lane;
      a_lds[a_slot<S>(slot / C, slot % C)] = v[it];
    }
  }
}

template <int P, int N>
__device__ __forceinline__ void gather_commit_parts_buf(int4v *__restrict__ a_lds, const int4v (&v)[N], int lane, bool &lost) {
#pragma unroll
  for (int it = 0; it < N; ++it) {
    const int slot = it * 64 + lane;
    split_and_store<P>(a_lds, __builtin_bit_cast(float4v, v[it]), slot / 8, slot % 8, lost);
  }
}

// ---------------------------------------------------------------------------
// Pair-stationary kernel.
// SPLIT: fp32 tensors whose caller allows tf32 precision, products in split bf16 (see
// mma_slab_parts); `packed` from pack_weights_parts_kernel.
// WALK: see kWalkAll.
template <typename T, int NT, int S, bool SPLIT, int WALK>
__global__ __launch_bounds__(kThreads) void gms_pairs_kernel(
    const T *__restrict__ src, const T *__restrict__ packed, T *__restrict__ dst,
    const int32_t *__restrict__ kpos, const int32_t *__restrict__ gmap,
    const int32_t *__restrict__ smap, int k_vol, int c_src, int c_dst, int tiles_per_wg,
    int offset, int dense_rows, SideJob side) {
  // the leading workgroups of the grid run the side job, if there is one
  int block_x = blockIdx.x;
  if (side.blocks) {
    if (block_x < side.blocks) {
      if (blockIdx.y == 0) run_side_job(side, block_x);
      return;
    }
    block_x -= side.blocks;
  }
  constexpr int E = Elem<T>::per_chunk;
  extern __shared__ int4v lds[];
  const int slabs = c_src / (2 * S * E);
  const int qs = slabs * S;
  const int nts = c_dst / 32;
  int4v *w_lds = lds;                                   // qs * NT * 64 chunks
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  int4v *a_lds = lds + qs * NT * 64 + wave * (kWaveRows * 2 * S);
  int *idx_all = reinterpret_cast<int *>(lds + qs * NT * 64 + kWaves * (kWaveRows * 2 * S));
  int *gidx = idx_all + wave * 2 * kWaveRows;
  int *sidx = gidx + kWaveRows;
  const int nt0 = blockIdx.y * NT;
  const size_t packed_per_k = (size_t)c_src * c_dst / E;  // chunks

  Strays strays;
  if constexpr (WALK == kWalkRest) {
    const int blocks = gridDim.x - side.blocks;
    strays = look_for_strays(kpos, smap, offset, block_x);
    tiles_per_wg = rest_tiles(kpos, k_vol, offset, kTileRows, tiles_per_wg, blocks);
  }
  int cur_k = -1;
  const int t_begin = block_x * tiles_per_wg;
  for (int t = t_begin; t < t_begin + tiles_per_wg; ++t) {
    int k, first, count;
    if constexpr (WALK == kWalkOwn) {
      k = offset >> 1;
      first = t * kTileRows;
      if (first >= dense_rows) break;
      count = min(kTileRows, dense_rows - first);
    } else if (!locate_tile(kpos, k_vol, kTileRows, t, k, first, count, WALK == kWalkRest ? offset : -1)) {
      break;
    }
    if (k != cur_k) {  // uniform over the workgroup
      __syncthreads();
      if constexpr (SPLIT)
        load_weights_split<NT>(w_lds, reinterpret_cast<const int4v *>(packed) + packed_per_k * k, slabs, nts, nt0);
      else
        load_weights<NT>(w_lds, reinterpret_cast<const int4v *>(packed) + packed_per_k * k, qs, nts, nt0);
      __syncthreads();
      cur_k = k;
    }
    const int wfirst = wave * kWaveRows;
    const int nrows = min(kWaveRows, count - wfirst);
    if (nrows <= 0) continue;
    const bool live = lane < nrows;
    const int j = first + wfirst + lane;
    if constexpr (WALK == kWalkOwn) {
      const int source = live ? own_source(kpos, gmap, smap, k, j) : -1;
      gidx[lane] = source;
      sidx[lane] = live ? own_row(source, j) : -1;
    } else {
      gidx[lane] = !live ? -1 : (gmap ? gmap[j] : j);
      sidx[lane] = !live ? -1 : (smap ? smap[j] : j);
    }
    wave_lds_fence();

    float16v acc[2][NT];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.f;

    float16v low[1][1];      // (two parts: not used)
    int4v v[2 * S];
    int gsel[2 * S];
    gather_issue<T, S>(v, gsel, gidx, src, c_src, 0, lane);
    for (int slab = 0; slab < slabs; ++slab) {
      if constexpr (SPLIT) gather_commit_parts<2>(a_lds, v, gsel, lane);
      else gather_commit<S>(a_lds, v, gsel, lane);
      wave_lds_fence();
      if (slab + 1 < slabs) gather_issue<T, S>(v, gsel, gidx, src, c_src, slab + 1, lane);   // under the MFMAs
      if constexpr (SPLIT) mma_slab_parts<2, false>(acc, low, a_lds, w_lds + slab * (2 * NT * 128), lane);
      else mma_slab<T, NT, S>(acc, a_lds, w_lds, slab, lane);
      wave_lds_fence();
    }
    if constexpr (WALK != kWalkOwn) write_tile<T, NT, kTileAtomic>(acc, dst, sidx, c_dst, nt0 * 32, lane);
    else if (offset & 1) write_tile<T, NT, kTileStore>(acc, dst, sidx, c_dst, nt0 * 32, lane);
    else write_tile<T, NT, kTileAdd>(acc, dst, sidx, c_dst, nt0 * 32, lane);
    if constexpr (WALK == kWalkOwn && sizeof(T) == 2)
      if (gmap) clear_rows<NT>(dst, sidx, c_dst, nt0 * 32, lane);
    wave_lds_fence();
  }
  if constexpr (WALK == kWalkRest)
    add_strays<S>(strays, src, reinterpret_cast<const int4v *>(packed) + packed_per_k * offset, dst, gmap, smap, dense_rows, c_src, c_dst,
                  nt0 * 32, NT * 32, gridDim.x - side.blocks);
}

// ---------------------------------------------------------------------------
// Output-stationary kernel.  nbr is the plan's table laid out [k_vol][n_dst]:
// nbr[k][d] = source row that reaches destination row d through offset k, or -1.
//
// The work of a workgroup is a list of stages (offset k, slab of the source
// row).  Stages are software-pipelined: while the MFMAs of stage t run, the
// weights and the gathered rows of stage t + 1 are already in flight in
// registers (the row index of the offset after that is in flight too); they are
// written to LDS after the MFMAs and one barrier closes the stage.  Weights are
// double-buffered in LDS, each wave's row tile is single-buffered (only its own
// wave reads it).
// RAW = 1: `packed` is the caller's weight tensor itself, forward (fp16: see raw_weight_frag);
// RAW = 2: the same for the input gradient (see mma_slab_rawt); RAW = 3: fp32 tensors with
// products in split bf16 (see mma_slab_parts), `packed` from pack_weights_parts_kernel; RAW = 4:
// the input gradient in split bf16, weights read as they lie and split on their way to LDS;
// RAW = 5 and 6: as 3 and 4 with three parts to a value, for fp32 tensors in full precision;
// RAW = 7 and 8: what a workgroup of those does where a sum is not finite, the same tile on fp32 MFMAs with the
// weights as they lie, forward (mma_slab_raw32) and input gradient; RAW = 0: the re-laid copy pack_weight_elements makes.
// (block_x, block_y, block_z) of a grid (tiles, column tiles, grid_z parts of a tile).
// MT: 32-row MFMA tiles per wave.  2 (a workgroup tile of 256 rows) is the layout every plan
// table is made for; 1 (tiles of 128 rows, half the work per wave and stage) serves launches
// too small to fill the chip, where a tile's chain of stages is all there is to the duration.
// KG > 1 (MT = 1): the workgroup is KG groups of four waves, every group walks its share of the
// tile's offsets with LDS of its own, and the groups' sums meet in LDS behind the last stage: the chain
// is a KG-th as long, without the atomics (and the zeroed result rows) that workgroups sharing a tile need.
constexpr int split_parts_of(int raw) { return raw == 3 || raw == 4 ? 2 : raw == 5 || raw == 6 ? 3 : 0; }
// 16-byte chunks of LDS per group: two stages of weights, row tiles, indices.  (Three bf16 parts take half as much
// again as the fp32 value.)
template <typename T, int NT, int S, int MT>
constexpr int rows_group_chunks(int raw) {
  return (2 * S * NT * 64 + kWaves * MT * 32 * 2 * S) * (split_parts_of(raw) == 3 ? 3 : 2) / 2 + kWaves * 3 * MT * 32 / 4;
}
template <int NT, int MT>
constexpr int rows_sum_chunks() { return kWaves * MT * NT * 4 * 64; }      // ... of a group's sums

// centre (forward only; 0: none): the bit of an offset through which every row is its own neighbour, and which the caller
// keeps out of its lists; the offset's line of the table says so, the masks do not (see Plan::centre_line).

// RAGGED (fp16, RAW 1 and 2; fp32, RAW 3 to 6): channel counts that fill no whole tile.  Chunks of rows and weights from
// c_src on, and of weights from c_dst on, are loaded from outside their buffers and arrive as zeros (re-laid weights hold
// zeros there); columns from c_dst on are not written.  TAILS (with it): 4 output channels more
// than a multiple of 8, so that rows of that side end in half a chunk (see take_tail); a variant of its own, because the moves into
// place and the addresses cost the masked tiles a tenth (48 -> 96 over 90 k LiDAR voxels, drop-in call 99.9 -> 112.3 us).
template <typename T, int NT, int S, int RAW, int MT = 2, int KG = 1, bool RAGGED = false, bool TAILS = false>
__device__ __forceinline__ void gms_rows_body(
    const T *__restrict__ src, const T *__restrict__ packed, T *__restrict__ dst,
    const int32_t *__restrict__ nbr, const unsigned long long *__restrict__ block_masks,
    const int32_t *__restrict__ perm, const int32_t *__restrict__ tile_order, int n_dst, int k_vol,
    int c_src, int c_dst, int part_stages, int block_x, int block_y, int block_z, int grid_z,
    unsigned src_bytes, int pair_view, int overwrite, int flip, unsigned long long centre, const T *__restrict__ w_raw) {
  constexpr int E = Elem<T>::per_chunk;
  constexpr int C = 2 * S;
  constexpr bool kAsRows = RAW == 2 || RAW == 4 || RAW == 6 || RAW == 8;      // weights as they lie, input gradient
  constexpr bool kAsLies = RAW == 1 || RAW == 7;                              // ... forward
  constexpr int WP = NT * 32 / E;                                             // 16-byte pieces of a weight row of the tile
  // 16-bit matrix instructions (fp16 tensors, fp32 tensors in split bf16): rows and weights come
  // through buffer loads and the MFMA phase is pipelined by hand; plain fp32, whose MFMA phase is
  // eight times as long, keeps pointer loads and interleaves them with its MFMAs instead
  constexpr int P = split_parts_of(RAW);
  constexpr bool kBuf = sizeof(T) == 2 || P > 0 || RAW >= 7;
  const __amdgpu_buffer_rsrc_t rsrc = rows_resource(src, src_bytes);
  const unsigned row_bytes = (unsigned)c_src * (unsigned)sizeof(T);
  // byte offset of source row g in the buffer (kAbsentRow: no neighbour, the loads return zeros)
  auto row_offset = [&](int g) { return !kBuf ? (unsigned)g : g < 0 ? kAbsentRow : (unsigned)g * row_bytes; };
  // pair view: `nbr` is one list of source rows for all offsets (a 64-row block belongs to
  // the one offset its mask names), `perm` the destination rows; results are added atomically
  const size_t nbr_stride = pair_view ? 0 : (size_t)n_dst;
  constexpr int kGrow = P == 3 ? 3 : 2;                   // (three parts: halves again)
  constexpr int WCH = S * NT * 64 * kGrow / 2;            // 16-byte chunks of one stage's weights in LDS
  constexpr int WLD = RAW == 6 ? S * NT * 64 : WCH;       // ... as they are read
  constexpr int NW = (WLD + kThreads - 1) / kThreads;     // ... per thread
  constexpr int CL = C * kGrow / 2;                       // chunks of a row of the wave's tile in LDS
  extern __shared__ int4v lds_all[];
  __shared__ unsigned long long wg_mask;
  const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / kThreads);
  const int tid = KG == 1 ? threadIdx.x : threadIdx.x % kThreads;
  int4v *const lds = KG == 1 ? lds_all : lds_all + group * rows_group_chunks<T, NT, S, MT>(RAW);
  // fp32 only: its MFMA phase is long enough (4 k clocks a stage) to absorb the loads'
  // issue waits; for fp16 the interleaved stage measured 2 us slower per launch
  constexpr bool kInterleave = !kBuf;
  static_assert(!RAGGED || (sizeof(T) == 2 ? RAW == 1 || RAW == 2 : P > 0 || RAW >= 7), "ragged: fp16 weights as they lie, fp32 in parts");
  static_assert(RAW < 7 || (sizeof(T) == 4 && S == 4), "the tiles of RAW 5 and 6");
  const int slabs = RAGGED ? (c_src + C * E - 1) / (C * E) : c_src / (C * E);
  const int nts = RAGGED ? (c_dst + 31) / 32 : c_dst / 32;
  int4v *w_lds = lds;                                     // [2][WCH]
  const int wave = tid / 64, lane = tid % 64;
  constexpr int WR = MT * 32;                             // rows per wave
  constexpr int TR = kWaves * WR;                         // rows per workgroup tile
  int4v *a_lds = lds + 2 * WCH + wave * (WR * CL);
  int *idx_all = reinterpret_cast<int *>(lds + 2 * WCH + kWaves * (WR * CL));
  // per wave: the rows to gather -- byte offsets, two sets (this offset's and the next one's), or
  // plain indices (!kBuf, one set) -- and the destination rows
  unsigned *goff = reinterpret_cast<unsigned *>(idx_all + wave * 3 * WR);
  const int *gidx = idx_all + wave * 3 * WR;
  int *didx = idx_all + wave * 3 * WR + 2 * WR;
  const int nt0 = block_y * NT;
  const int4v *packed4 = reinterpret_cast<const int4v *>(packed);
  // chunks of an offset's weights
  const size_t packed_per_k = RAW == 3 || RAW == 5 ? (size_t)slabs * nts * 128 * P : (size_t)c_src * c_dst / E;

  // the plan's table gives the tile and the first offset it uses
  int tile = block_x, k_first = -1;
  if (tile_order) {
    const int entry = tile_order[block_x];
    if (entry < 0) return;
    tile = entry & 0xFFFFFF;
    if (grid_z == 1 && !centre) k_first = entry >> 24;
  }
  const int row0 = tile * TR + wave * WR;
  const int my_row = row0 + lane;
  const bool owns_row = MT == 2 || lane < WR;             // (lanes past a 32-row wave tile own no row)
  const bool in_range = owns_row && my_row < n_dst;
  // that offset's neighbour index, fetched while the masks are still on their way: at the
  // start of a launch every workgroup walks this chain of dependent loads at the same time
  // and nothing else covers it (0.4 us of a 46 us launch)
  int g_first = -1;
  if (k_first >= 0 && in_range) g_first = nbr[(size_t)k_first * nbr_stride + my_row];
  if (owns_row) didx[lane] = in_range ? (perm ? perm[my_row] : my_row) : -1;   // my_row is a position in the plan's row order

  // which offsets touch this wave's rows / this workgroup's rows (from the plan)
  unsigned long long wave_mask = row0 < n_dst ? block_masks[row0 / 64] | centre : 0ull;
  // (one value for the whole wave: in scalar registers where vector registers are short)
  if constexpr (kBuf)
    wave_mask = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(wave_mask & 0xffffffffu)) |
              ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(wave_mask >> 32)) << 32);
  if (threadIdx.x == 0) wg_mask = 0;
  __syncthreads();
  if (lane == 0 && wave_mask) atomicOr(&wg_mask, wave_mask);
  __syncthreads();
  unsigned long long todo = wg_mask;
  if (!todo) {
    if (overwrite && group == 0) zero_rows<T, NT, WR, RAGGED>(dst, didx, c_dst, nt0 * 32, lane);
    return;
  }
  // The launch lasts as long as its longest tile, and the tiles with the longest
  // offset lists are few: they get the instruction issue priority, so that they run
  // at their own pace while the many short tiles share what is left.
  {
    const int n_off = __builtin_popcountll(todo);
    if (n_off * 4 > k_vol * 3) __builtin_amdgcn_s_setprio(3);
    else if (n_off * 2 > k_vol) __builtin_amdgcn_s_setprio(1);
  }
  // grid_z > 1: a tile is shared by up to grid_z workgroups, each takes a run
  // of the tile's offsets and adds its partial result with atomics.
  bool shared_tile = pair_view != 0;
  if (grid_z > 1) {
    const int n_off = __builtin_popcountll(todo);
    const int want = (n_off * slabs + part_stages - 1) / part_stages;
    const int parts = min(grid_z, max(want, 1));
    if (block_z >= parts) return;
    if (parts > 1) {
      shared_tile = true;
      const int per = (n_off + parts - 1) / parts;
      for (int i = 0; i < block_z * per; ++i) todo &= todo - 1;      // offsets of earlier parts
      unsigned long long mine = 0, rest = todo;
      for (int i = 0; i < per && rest; ++i) {
        mine |= rest & (0 - rest);
        rest &= rest - 1;
      }
      todo = mine;
      if (!todo) return;
    }
  }

  if constexpr (KG > 1) {
    // this group's run of the tile's offsets; a group with fewer than the others also walks some of
    // theirs, for which its rows count as absent, so that all groups meet at the same barriers
    const int per = (__builtin_popcountll(todo) + KG - 1) / KG;
    unsigned long long rest = todo, mine = 0;
    for (int i = 0; i < group * per; ++i) rest &= rest - 1;
    int count = 0;
    for (; count < per && rest; ++count) {
      mine |= rest & (0 - rest);
      rest &= rest - 1;
    }
    unsigned long long others = todo & ~mine;
    todo = mine;
    for (; count < per; ++count) {
      todo |= others & (0 - others);
      others &= others - 1;
    }
    wave_mask &= mine;
    k_first = -1;
  }

  float16v acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.f;

  float16v low[P == 3 ? MT : 1][P == 3 ? NT : 1];         // three parts: the small products (mma_parts)
  if constexpr (P == 3) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) low[mt][nt] = acc[mt][nt];
  }

  bool lost = false;                                      // ... met a value they do not hold (split_parts)

  // Weights of stage (k, slab), 16-byte chunk e = threadIdx.x + kThreads * i of the stage's tile,
  // through a buffer resource over the weight tensor: the part of a chunk's address that depends
  // on the thread is a per-lane constant (wvoff), the part that depends on the stage is scalar.
  //   RAW = 1, 7: row e / WP of the slab's C*E rows of W[k], 16-byte piece e % WP of the
  //            NT*32 columns from nt0*32 on
  //   RAW = 2, 4, 6, 8: row e / C of the NT*32 rows of W[k] from nt0*32 on (c_dst rows of c_src
  //            elements here), 16-byte piece e % C of the slab
  //   RAW = 3, 5: k-step e / (NT*64*P) of the stage, then [nt][part][lane]
  //   RAW = 0: chunks [(slab*S + s) * nts + nt0 + nt] * 64 + lane of the re-laid copy
  const __amdgpu_buffer_rsrc_t wrsrc =
      rows_resource(packed, RAW == 3 || RAW == 5 ? (unsigned)k_vol * (unsigned)packed_per_k * 16u
                                                   : (unsigned)k_vol * (unsigned)c_src * (unsigned)c_dst * (unsigned)sizeof(T));
  unsigned wvoff[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int e = tid + kThreads * i;
    if constexpr (kAsLies) wvoff[i] = (unsigned)(((e / WP) * c_dst + (e % WP) * E) * (int)sizeof(T));
    else if constexpr (kAsRows) wvoff[i] = (unsigned)(((e / C) * c_src + (e % C) * E) * (int)sizeof(T));
    else if constexpr (P > 0) wvoff[i] = (unsigned)(((e / (NT * 64 * P)) * nts * 64 * P + e % (NT * 64 * P)) * 16);
    else wvoff[i] = (unsigned)(((e / (NT * 64)) * nts * 64 + e % (NT * 64)) * 16);
  }
  // is chunk e of the stage's weights a row's last one, of which only half exists?
  auto weight_tail = [&](int e, int slab) {
    return kAsLies ? nt0 * 32 + e % WP * E + E > c_dst : slab * (C * E) + e % C * E + E > c_src;
  };
  // (flip: the tables number the offsets from the other end, see Plan)
  auto weights_issue = [&](int4v (&wreg)[NW], int k_, int slab) {
    const int k = flip ? flip - k_ : k_;
    if constexpr (!kBuf) {
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        const int e = tid + kThreads * i;
        if (NW * kThreads == WLD || e < WLD) {
          if constexpr (RAW == 2) {
            const int row = e / C, c = e % C;
            wreg[i] = *reinterpret_cast<const int4v *>(
                packed + ((size_t)k * c_dst + nt0 * 32 + row) * c_src + (size_t)(slab * C + c) * E);
          } else {
            const int q = e / (NT * 64), rem = e % (NT * 64);
            wreg[i] = packed4[packed_per_k * k + ((size_t)(slab * S + q) * nts + nt0) * 64 + rem];
          }
        }
      }
      return;
    }
    unsigned soff;                                       // (wave-uniform: goes to the scalar offset)
    if constexpr (kAsLies) soff = (unsigned)(((k * c_src + slab * (C * E)) * c_dst + nt0 * 32) * (int)sizeof(T));
    else if constexpr (kAsRows) soff = (unsigned)(((k * c_dst + nt0 * 32) * c_src + slab * (C * E)) * (int)sizeof(T));
    else if constexpr (P > 0) soff = (unsigned)(((int)packed_per_k * k + ((slab * 2) * nts + nt0) * 64 * P) * 16);
    else soff = (unsigned)(((int)packed_per_k * k + ((slab * S) * nts + nt0) * 64) * 16);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int e = tid + kThreads * i;
      if (NW * kThreads == WLD || e < WLD) {
        unsigned off = wvoff[i];
        if constexpr (TAILS) {
          const int from = slab * (C * E) + (kAsLies ? e / WP : e % C * E);
          const int to = nt0 * 32 + (kAsLies ? e % WP * E : e / C);
          off = from >= c_src || to >= c_dst ? kAbsentRow : off + soff - (weight_tail(e, slab) ? kTailBytes : 0u);
        } else if constexpr (RAGGED && RAW != 3 && RAW != 5) {
          const int from = slab * (C * E) + (kAsLies ? e / WP : e % C * E);
          const int to = nt0 * 32 + (kAsLies ? e % WP * E : e / C);
          if (from >= c_src || to >= c_dst) off = kAbsentRow;
        }
        wreg[i] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, off, TAILS ? 0 : soff, 0));
      }
    }
  };
  auto weights_commit = [&](int4v (&wreg)[NW], int buf, int slab) {
    if constexpr (TAILS) {
#pragma unroll
      for (int i = 0; i < NW; ++i) wreg[i] = take_tail(wreg[i], weight_tail(tid + kThreads * i, slab));
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int e = tid + kThreads * i;
      if (NW * kThreads == WLD || e < WLD) {
        if constexpr (RAW == 1) {
          const int row = e / (NT * 4), c = e % (NT * 4);
          w_lds[buf * WCH + row * (NT * 4) + (c ^ raw_swizzle<NT>(row))] = wreg[i];
        } else if constexpr (RAW == 2 || RAW == 8) {
          w_lds[buf * WCH + a_slot<S>(e / C, e % C)] = wreg[i];
        } else if constexpr (RAW == 4 || RAW == 6) {
          split_and_store<P>(w_lds + buf * WCH, __builtin_bit_cast(float4v, wreg[i]), e / C, e % C, lost);
        } else {
          w_lds[buf * WCH + e] = wreg[i];
        }
      }
    }
  };

  int k = __builtin_ctzll(todo);
  todo &= todo - 1;
  int slab = 0;
  int k_nxt = todo ? __builtin_ctzll(todo) : -1;
  if (todo) todo &= todo - 1;
  bool active = (wave_mask >> k) & 1;
  int4v wreg[NW];
  constexpr int NV = MT * S;                              // row chunks per lane and stage
  int4v v[NV];
  int gsel[kBuf ? 1 : NV];
  auto rows_issue = [&](int slab_, int slot_ = 0) {
    if constexpr (kBuf) gather_issue_buf<S, RAGGED, TAILS && kAsRows>(v, goff + slot_ * WR, rsrc, slab_, lane, row_bytes);
    else gather_issue<T, S>(v, gsel, gidx, src, c_src, slab_, lane);
  };
  auto rows_commit = [&](int slab_) {
    if constexpr (TAILS && kAsRows) take_row_tails<S>(v, slab_, lane, row_bytes);
    if constexpr (P > 0) gather_commit_parts_buf<P>(a_lds, v, lane, lost);
    else if constexpr (kBuf) gather_commit_buf<S>(a_lds, v, lane);
    else gather_commit<S>(a_lds, v, gsel, lane);
  };

  // prologue: stage 0 goes straight to LDS
  if (owns_row)
    goff[lane] = row_offset(k_first >= 0 ? g_first : (in_range && (KG == 1 || active) ? nbr[(size_t)k * nbr_stride + my_row] : -1));
  int g_nxt = (k_nxt >= 0 && in_range) ? nbr[(size_t)k_nxt * nbr_stride + my_row] : -1;
  wave_lds_fence();
  weights_issue(wreg, k, 0);
  if (active) rows_issue(0);
  weights_commit(wreg, 0, 0);
  if (active) rows_commit(0);
  __syncthreads();

  int buf = 0;
  if constexpr (kBuf) {
    // Every stage is the same straight run of instructions for every wave: a wave whose rows do
    // not use the next offset still issues its row loads (all its offsets are kAbsentRow, so
    // they fetch nothing and return zeros) and writes the zeros to its tile, and only skips the
    // MFMAs.  With no branch around the loads and their consumers the compiler knows exactly
    // which loads are in flight at every point and waits for none it does not need; in
    // particular the index load below stays in flight across the stage.
    const int safe_row = min(my_row, n_dst - 1);
    auto mma_stage = [&]() {
      if constexpr (RAW == 1) mma_slab_raw<T, NT, S>(acc, a_lds, w_lds + buf * WCH, lane);
      else if constexpr (RAW == 7) mma_slab_raw32<NT, S>(acc, a_lds, w_lds + buf * WCH, lane);
      else if constexpr (RAW == 2 || RAW == 8) mma_slab_rawt<T, NT, S>(acc, a_lds, w_lds + buf * WCH, lane);
      else if constexpr (P > 0) mma_slab_parts<P, RAW == 4 || RAW == 6>(acc, low, a_lds, w_lds + buf * WCH, lane);
      else mma_slab<T, NT, S>(acc, a_lds, w_lds + buf * WCH, 0, lane);
    };
    // Offsets are numbered in the order the tile walks them; offset j gathers through the index
    // set j & 1.  While stage (offset j, last slab) runs, set (j + 1) & 1 serves the loads of
    // offset j + 1 and set j & 1, which nothing reads any more, receives the offsets of offset
    // j + 2, whose indices were requested a whole stage earlier; the indices of offset j + 3 are
    // requested then.  So no stage starts by waiting for an index or for its way through LDS.
    int k1 = k_nxt;                                          // the next offset (-1: none)
    int k2 = todo ? __builtin_ctzll(todo) : -1;              // the one after
    if (todo) todo &= todo - 1;
    if (k1 >= 0) {                                           // (requested in the prologue, long landed)
      const bool a1 = (wave_mask >> k1) & 1;
      if (owns_row) goff[WR + lane] = row_offset(in_range && a1 ? g_nxt : -1);
      wave_lds_fence();
    }
    // (nothing of the prologue is in flight any more; said explicitly, because the compiler
    // cannot tell from the prologue's branches and would wait for loads that never were issued)
    __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
    if (k2 >= 0) g_nxt = nbr[(size_t)k2 * nbr_stride + safe_row];
    int slot = 0;
    // One pass of the loop per stage that has a successor: request the successor's weights and
    // rows, multiply this stage, move the successor to LDS; the last stage's products follow
    // the loop.  (One exit test, at the top: issue and commit always run together.)
    int nk = k, nslab = 1;
    if (nslab == slabs) { nk = k1; nslab = 0; }
    while (nk >= 0) {
      const bool adv = nk != k;
      const int nslot = adv ? slot ^ 1 : slot;
      weights_issue(wreg, nk, nslab);
      rows_issue(nslab, nslot);
      int k3 = -1;
      if (adv) {
        // (a wave that does not use an offset: all absent, also over the pair view, whose list
        // names a row whatever the offset)
        const bool a2 = k2 >= 0 && ((wave_mask >> k2) & 1);
        if (owns_row) goff[slot * WR + lane] = row_offset(in_range && a2 ? g_nxt : -1);
        wave_lds_fence();
        k3 = todo ? __builtin_ctzll(todo) : -1;
        if (todo) todo &= todo - 1;
        if (k3 >= 0) g_nxt = nbr[(size_t)k3 * nbr_stride + safe_row];
      }
      if (active) mma_stage();
      wave_lds_fence();
      rows_commit(nslab);
      weights_commit(wreg, buf ^ 1, nslab);
      __syncthreads();
      buf ^= 1;
      active = (wave_mask >> nk) & 1;
      k = nk;
      slot = nslot;
      if (adv) { k1 = k2; k2 = k3; }
      nslab += 1;
      if (nslab == slabs) { nk = k1; nslab = 0; }
    }
    if (active) mma_stage();
  } else {
    while (true) {
      int nk = k, nslab = slab + 1;
      if (nslab == slabs) { nk = k_nxt; nslab = 0; }
      const bool has_next = nk >= 0;
      const bool next_active = has_next && ((wave_mask >> nk) & 1);
      if (has_next) {
        if (nk != k) {          // the row loads that used the old indices were issued a stage ago
          if (owns_row) goff[lane] = row_offset(g_nxt);
          wave_lds_fence();
        }
      }
      if (kInterleave && has_next && active && next_active) {
        // The common stage: this stage's MFMAs with the next stage's loads between them,
        // one row load after each (k-step, row tile) group.  A load instruction waits at
        // issue while the CU's memory queue is full; issued in a block before the MFMAs
        // those waits come on top of the MFMA time, issued between them they pass while
        // the matrix pipe works off what it has.  (MFMAs and loads stay on their side of
        // each scheduling barrier, LDS reads and address arithmetic may cross.)
        const int4v *wl = w_lds + buf * WCH;
        const int h = lane / 32, r = lane % 32;
        weights_issue(wreg, nk, nslab);
  #pragma unroll
        for (int s = 0; s < S; ++s) {
          int4v b[NT];
  #pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            if constexpr (RAW == 1) b[nt] = raw_weight_frag<NT, S>(wl, s, nt, lane);
            else if constexpr (RAW == 2) b[nt] = wl[a_slot<S>(nt * 32 + r, h * S + s)];
            else b[nt] = wl[(s * NT + nt) * 64 + lane];
          }
  #pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const int4v a = a_lds[a_slot<S>(mt * 32 + r, h * S + s)];
  #pragma unroll
            for (int nt = 0; nt < NT; ++nt) mma<T>(acc[mt][nt], a, b[nt]);
            const int it = s * MT + mt;                      // one of the MT * S row loads
            gsel[it] = gidx[(it * 64 + lane) / C];
            v[it] = *reinterpret_cast<const int4v *>(src + (size_t)max(gsel[it], 0) * c_src +
                                                     (size_t)(nslab * C + (it * 64 + lane) % C) * E);
            __builtin_amdgcn_sched_barrier(0x386);
          }
        }
      } else {
        if (has_next) {
          weights_issue(wreg, nk, nslab);
          if (next_active) rows_issue(nslab);
        }
        if (active) {
          if constexpr (RAW == 1) mma_slab_raw<T, NT, S>(acc, a_lds, w_lds + buf * WCH, lane);
          else if constexpr (RAW == 2) mma_slab_rawt<T, NT, S>(acc, a_lds, w_lds + buf * WCH, lane);
          else mma_slab<T, NT, S>(acc, a_lds, w_lds + buf * WCH, 0, lane);
        }
      }
      if (!has_next) break;
      wave_lds_fence();
      if (next_active) rows_commit(nslab);
      weights_commit(wreg, buf ^ 1, nslab);
      if (nk != k) {
        k_nxt = todo ? __builtin_ctzll(todo) : -1;
        if (todo) todo &= todo - 1;
        g_nxt = (k_nxt >= 0 && in_range) ? nbr[(size_t)k_nxt * nbr_stride + my_row] : -1;
      }
      __syncthreads();
      buf ^= 1;
      k = nk;
      slab = nslab;
      active = next_active;
    }
  }
  if constexpr (P == 3) {
    float beyond = 0.f;                                      // (NaN where a sum is not finite: an infinity, a weight that is marked)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[mt][nt][r] += low[mt][nt][r];
          beyond = __builtin_fmaf(acc[mt][nt][r], 0.f, beyond);
        }
    if (__syncthreads_or(beyond != 0.f || lost)) {          // (also: every wave is through with LDS)
      gms_rows_body<T, NT, S, RAW + 2, MT, KG, RAGGED>(src, RAW == 5 ? w_raw : packed, dst, nbr, block_masks, perm, tile_order, n_dst, k_vol,
                                                       c_src, c_dst, part_stages, block_x, block_y, block_z, grid_z, src_bytes,
                                                       pair_view, overwrite, flip, centre, nullptr);
      return;
    }
  }
  if constexpr (KG > 1) {
    // the groups' sums meet in the LDS behind the first group's
    float4v *const sums = reinterpret_cast<float4v *>(lds_all + rows_group_chunks<T, NT, S, MT>(RAW));
    constexpr int per_group = rows_sum_chunks<NT, MT>();
    __syncthreads();                   // every group is through with its row tiles and weights
    if (group > 0) {
#pragma unroll
      for (int q = 0; q < MT * NT * 4; ++q) {
        float4v v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[q / 4 / NT][q / 4 % NT][q % 4 * 4 + e];
        sums[(group - 1) * per_group + (wave * (MT * NT * 4) + q) * 64 + lane] = v;
      }
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 0; g < KG - 1; ++g)
#pragma unroll
      for (int q = 0; q < MT * NT * 4; ++q) {
        const float4v v = sums[g * per_group + (wave * (MT * NT * 4) + q) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[q / 4 / NT][q / 4 % NT][q % 4 * 4 + e] += v[e];
      }
  }
  if (wave_mask || overwrite || KG > 1) {
    wave_lds_fence();
    if (shared_tile)
      add_rows_lds<T, NT, S, true, false, RAGGED>(acc, dst, didx, reinterpret_cast<float *>(a_lds), c_dst, nt0 * 32, lane);
    else if (overwrite)
      add_rows_lds<T, NT, S, false, true, RAGGED>(acc, dst, didx, reinterpret_cast<float *>(a_lds), c_dst, nt0 * 32, lane);
    else
      add_rows_lds<T, NT, S, false, false, RAGGED>(acc, dst, didx, reinterpret_cast<float *>(a_lds), c_dst, nt0 * 32, lane);
  }
}

template <typename T, int NT, int S, int RAW, int MT = 2, int KG = 1, bool RAGGED = false, bool TAILS = false>
__global__ __launch_bounds__(kThreads * KG, RAW >= 5 ? (MT == 2 || KG == 2 ? 2 : KG == 4 ? 4 : 3)
                                                      : MT == 1 ? (NT == 3 ? 3 : 4) : (NT >= 3 ? 2 : 3)) void gms_rows_kernel(
    const T *__restrict__ src, const T *__restrict__ packed, T *__restrict__ dst,
    const int32_t *__restrict__ nbr, const unsigned long long *__restrict__ block_masks,
    const int32_t *__restrict__ perm, const int32_t *__restrict__ tile_order, int n_dst, int k_vol,
    int c_src, int c_dst, int part_stages, SideJob side, int pair_view, unsigned src_bytes, int overwrite,
    int flip_centre, const T *__restrict__ w_raw) {
  // (flip, and the centre offset + 1 behind its 8 bits: as an argument of eight bytes its own, the centre's bit made every
  // launch 0.07 us longer, 10.20 instead of 10.13 us for 32 -> 32 fp16 over 2 k voxels)
  // the leading workgroups of the grid run the side job, if there is one
  int block_x = blockIdx.x;
  if (side.blocks) {
    if (block_x < side.blocks) {
      if (blockIdx.y == 0 && blockIdx.z == 0) run_side_job(side, block_x);
      return;
    }
    block_x -= side.blocks;
  }
  gms_rows_body<T, NT, S, RAW, MT, KG, RAGGED, TAILS>(src, packed, dst, nbr, block_masks, perm, tile_order, n_dst, k_vol, c_src,
                                   c_dst, part_stages, block_x, blockIdx.y, blockIdx.z, gridDim.z, src_bytes, pair_view,
                                   overwrite, flip_centre & 255, flip_centre >> 8 ? 1ull << ((flip_centre >> 8) - 1) : 0ull, w_raw);
}

// ---------------------------------------------------------------------------
struct Shape {
  int c_src, c_dst, S, NT, E;
  int NTR, SR;            // 32-column tiles per wave and k-steps per slab in the output-stationary kernel
  size_t lds_bytes;       // pair-stationary kernel
  bool ok;
};

Shape shape_of(const GmsArgs &a) {
  Shape s{};
  s.c_src = a.transpose_w ? a.c_out : a.c_in;
  s.c_dst = a.transpose_w ? a.c_in : a.c_out;
  s.E = a.dtype == FGMS_F16 ? 8 : 4;
  const size_t esz = a.dtype == FGMS_F16 ? 2 : 4;
  s.ok = false;
  if (s.c_dst % 32 != 0 || s.c_src % (2 * s.E) != 0) return s;
  s.S = (s.c_src % (8 * s.E) == 0) ? 4 : (s.c_src % (4 * s.E) == 0) ? 2 : 1;
  s.NT = (s.c_dst % 64 == 0) ? 2 : 1;
  // rows are read with 16-byte loads and fp16 results written as 4-byte pairs
  if (reinterpret_cast<uintptr_t>(a.src) % 16 || reinterpret_cast<uintptr_t>(a.dst) % 4) return s;
  const size_t tiles = (size_t)kWaves * kWaveRows * 2 * s.S * 16  // staging tiles
                       + (size_t)kWaves * 3 * kWaveRows * sizeof(int);
  s.lds_bytes = (size_t)s.c_src * s.NT * 32 * esz + tiles;      // + weights of one offset
  // wide fp16 layers: 128 columns per wave, so that a row is gathered once per 128
  // (not 64) output channels.  Costs 128 accumulator registers (2 waves per SIMD)
  // and halves the number of workgroups, so only when enough of them remain to
  // fill the chip; fp32 has 8x the MFMA time per gathered byte and gains nothing.
  const int64_t wide_wgs = (a.n_dst + kTileRows - 1) / kTileRows * (s.c_dst / 128);
  const bool wide = kernel_policy() == 3 || (a.dtype == FGMS_F16 && wide_wgs * 2 >= 3 * (int64_t)num_cus());
  // 96 columns: a row is gathered once for all of them, not once per 32; 48 channels (fp16; 24 fp32):
  // one slab, not three of 16.  96 -> 96 fp16 over 80 k voxels forward 57.5 -> 45.8 us, 48 -> 96 48.5 -> 26.5,
  // 24 -> 32 fp32 over 40 k 39.6 -> 27.1.  fp32 products keep 32 columns: they take 16 times the matrix
  // time, so that more waves are worth more than fewer gathers (96 -> 96 over 40 k: 127.5 us against 184.8
  // with 96); in tf32 mode the forward pass takes 96 once there are tiles enough (over 150 k 243.9 ->
  // 166.2 us, over 40 k the same).
  const bool tf32_fills_96 = a.reduced && !a.transpose_w && s.S == 4 && split_bf16_enabled() &&
                             (a.n_dst + kTileRows - 1) / kTileRows * (s.c_dst / 96) * 2 >= 3 * (int64_t)num_cus();
  const bool cols96 = s.c_dst % 96 == 0 && worth_96_columns(a.n_pairs, a.n_src, a.n_dst) && (a.dtype == FGMS_F16 || tf32_fills_96);
  s.NTR = (s.c_dst % 128 == 0 && wide) ? 4 : s.c_dst % 64 == 0 ? 2 : cols96 ? 3 : 1;
  s.SR = s.S < 4 && s.c_src % (6 * s.E) == 0 ? 3 : s.S;
  s.ok = s.lds_bytes <= 128 * 1024;
  return s;
}

// --- channel counts that fill no whole tile (RAGGED) --------------------------------------
// 32-column tiles per wave (and blocks of a weight-gradient tile) for c columns, 0: not served.
int ragged_tiles(int c, bool three) {
  const int t = (c + 31) / 32;
  if (t <= 2) return t;
  if (t % 3 == 0 && three) return 3;
  if (t % 2 == 0) return 2;
  return three ? 3 : 0;
}
// k-steps of a slab: a stage costs about two k-steps however few it has.  (160 channels: three slabs of 64, the
// last one half empty, not five of 32.)
int ragged_steps(int c) {
  int best = 4, least = 1 << 30;
  for (int S = 4; S >= 2; --S) {
    const int cost = (c + 16 * S - 1) / (16 * S) * (S + 2);
    if (cost < least) { least = cost; best = S; }
  }
  return best;
}
// The shapes that take it: multiples of 8 channels (16-byte chunks) that no whole tile fits -- a source of a pass
// that is no multiple of 16, anything else that is none of 32 -- or an odd number of 32s from five
// on (160), which whole tiles take 32 columns at a time.  Kernels on the vector ALUs keep the narrow ones.
// fp16 output layers of 20 and 28 channels too (half_chunk; counts of 4 more than a multiple of 8 above a tile are rare, and every tile of
// theirs would be one more instantiation): no copies of the gradient's rows and of the weights, no crop of either result; four launches
// instead of seven, 96 -> 20 over 60 k voxels 77.5 -> 69.2 us.
// fp32 (in bf16 parts): what is no multiple of 32 on either side.  Without (fp32 MFMAs, padded copies) / with masks:
// 48 -> 48 over 30 k voxels forward 83 / 50 us, both gradients 123 / 65; 48 -> 64 over 120 k 121 / 108 and 303 / 189, in
// tf32 mode 121 / 65 and 180 / 131.
bool ragged_channels(int c_in, int c_out, bool forward, bool f16) {
  if (c_in % 8 || c_out % (f16 && c_out <= 32 ? 4 : 8) || c_in < 16 || c_out < 16 || c_in * c_out <= 256) return false;
  if (!f16) return c_in % 32 != 0 || c_out % 32 != 0;
  auto odd = [](int c, int whole) { return c % whole != 0 || (c % 32 == 0 && c / 32 % 2 == 1 && c / 32 >= 5 && c / 32 % 3 != 0); };
  return odd(c_in, forward ? 16 : 32) || odd(c_out, 32);
}
bool half_chunk(const GmsArgs &a) { return a.c_out % 8 != 0; }      // (of the masked shapes)
Shape ragged_shape(const GmsArgs &a) {
  Shape s{};
  s.c_src = a.transpose_w ? a.c_out : a.c_in;
  s.c_dst = a.transpose_w ? a.c_in : a.c_out;
  const bool f16 = a.dtype == FGMS_F16;
  s.E = f16 ? 8 : 4;
  if ((!f16 && !split_bf16_enabled()) || !ragged_channels(a.c_in, a.c_out, !a.transpose_w, f16)) return s;
  if (reinterpret_cast<uintptr_t>(a.src) % 16 || reinterpret_cast<uintptr_t>(a.dst) % 16 ||
      reinterpret_cast<uintptr_t>(a.w) % 16 || !raw_weights_enabled())
    return s;
  s.NTR = f16 ? ragged_tiles(s.c_dst, worth_96_columns(a.n_pairs, a.n_src, a.n_dst)) : (s.c_dst + 31) / 32 % 2 ? 1 : 2;
  s.SR = f16 ? ragged_steps(s.c_src) : 4;
  s.ok = s.NTR > 0;
  return s;
}

template <typename T>
int pack_weights(const GmsArgs &a, int S, const T **packed) {
  void *ws = nullptr;
  const size_t n = (size_t)a.k_vol * a.c_in * a.c_out;
  bool fill = true;
  int rc = relaid_weights_buffer(a, (unsigned)S << 8 | (a.transpose_w ? 2u : 0u), n * sizeof(T), &ws, &fill);
  if (rc != FGMS_OK) return rc;
  *packed = (const T *)ws;
  if (!fill) return FGMS_OK;
  unsigned blocks = (unsigned)((n + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  pack_weights_kernel<T><<<blocks, 256, 0, a.stream>>>((const T *)a.w, (T *)ws, a.k_vol, a.c_in,
                                                       a.c_out, S, a.transpose_w);
  FGMS_HIP_TRY(hipGetLastError());
  relaid_weights_filled(a, ws);
  return FGMS_OK;
}

// The same for fp32 weights in bf16 parts (pack_weights_parts_kernel).
template <int P>
int pack_weights_parts(const GmsArgs &a, bool transpose, const void **packed) {
  void *ws = nullptr;
  const size_t n = (size_t)a.k_vol * ((a.c_in + 31) / 32 * 32) * ((a.c_out + 31) / 32 * 32);
  bool fill = true;
  int rc = relaid_weights_buffer(a, 1u | (transpose ? 2u : 0u) | (P == 3 ? 4u : 0u), n * 2 * P, &ws, &fill);
  if (rc != FGMS_OK) return rc;
  *packed = ws;
  if (!fill) return FGMS_OK;
  size_t blocks = (n / 8 + 255) / 256;
  pack_weights_parts_kernel<P><<<(unsigned)(blocks > 4096 ? 4096 : blocks), 256, 0, a.stream>>>(
      (const float *)a.w, (int4v *)ws, a.k_vol, a.c_in, a.c_out, transpose);
  FGMS_HIP_TRY(hipGetLastError());
  relaid_weights_filled(a, ws);
  return FGMS_OK;
}


template <typename T, int NT, int S>
int launch_pairs(const GmsArgs &a, const Shape &s) {
  const T *packed = nullptr;
  // fp32 tensors whose caller allows tf32 precision: products in split bf16
  constexpr bool kCanSplit = sizeof(T) == 4 && S == 4;
  const bool split = kCanSplit && a.reduced && split_bf16_enabled();
  if (split) {
    const void *ws = nullptr;
    int rc = pack_weights_parts<2>(a, a.transpose_w, &ws);
    if (rc != FGMS_OK) return rc;
    packed = (const T *)ws;
  } else {
    int rc = pack_weights<T>(a, S, &packed);
    if (rc != FGMS_OK) return rc;
  }
  // (a first launch for the offset that meets every row once, if there is one, then one for the other pairs)
  SideJob side = a.side;
  for (int part = a.first_offset ? 0 : 1; part < 2; ++part) {
    const bool dense = part == 0 || a.dense_k >= 0;
    const int64_t rows = part == 0 ? a.n_dst : dense ? a.n_dense : std::max<int64_t>(a.n_pairs - (a.first_offset ? a.n_dst : 0), 0);
    constexpr int kRest = sizeof(T) == 2 ? kWalkRest : kWalkAll;      // (first offsets: fp16)
    auto kern = dense            ? (split ? gms_pairs_kernel<T, NT, S, kCanSplit, kWalkOwn> : gms_pairs_kernel<T, NT, S, false, kWalkOwn>)
                : a.first_offset ? gms_pairs_kernel<T, NT, S, false, kRest>
                : split          ? gms_pairs_kernel<T, NT, S, kCanSplit, kWalkAll>
                                 : gms_pairs_kernel<T, NT, S, false, kWalkAll>;
    { const int rc_lds = allow_dynamic_lds(reinterpret_cast<const void *>(kern), (size_t)s.lds_bytes); if (rc_lds != FGMS_OK) return rc_lds; }
    const int64_t tiles = (rows + kTileRows - 1) / kTileRows + (dense ? 0 : a.k_vol);
    // a few workgroups per CU, each walking a contiguous run of tiles
    const int64_t want_wgs = (int64_t)num_cus() * 8;
    const int tiles_per_wg = (int)((tiles + want_wgs - 1) / want_wgs);
    const unsigned gx = (unsigned)((tiles + tiles_per_wg - 1) / tiles_per_wg);
    ProfileScope prof(split ? (a.transpose_w ? "gms_pairs_kernel(dgrad, bf16x3)" : "gms_pairs_kernel(fwd, bf16x3)")
                            : (a.transpose_w ? "gms_pairs_kernel(dgrad)" : "gms_pairs_kernel(fwd)"),
                      a.stream);
    kern<<<dim3(gx + (unsigned)side.blocks, (unsigned)(s.c_dst / (32 * NT))), kThreads, s.lds_bytes, a.stream>>>(
        (const T *)a.src, packed, (T *)a.dst, a.kpos, a.gmap, a.smap, a.k_vol, s.c_src, s.c_dst,
        tiles_per_wg, walk_offset(a, part == 0), (int)(dense ? rows : a.n_dst), side);
    side = SideJob{};
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

// Grid of an output-stationary launch over n_dst destination rows: tiles of 256 rows from the
// plan's tile table where there is one (65 k rows and more, `table_grid` entries), else plain tiles of 256 or --
// where those still fit the chip's workgroup slots in one round -- of 128 rows (32 per wave:
// twice the waves, half the work per wave and stage; such a launch lasts as long as one
// tile's chain of stages).  A small forward launch on 128-row tiles shortens the chain with groups of waves
// inside a workgroup (can_group, below).  Where there are no groups -- an input gradient, a forward launch on the
// plan's table or with 128-column wave tiles -- a launch that fills less than half of the slots shares every
// tile between two workgroups, each taking half of the tile's stages and adding its part with
// atomics: twice the workgroups, half the critical path.  (Two parts only: the sum of two
// partial results does not depend on their order.  On launches that fill the chip the atomics
// cost more than the split gains.)  The standalone and the one-grid backward launch share this
// choice, so that their input gradients agree bit for bit; an input gradient takes the small
// tiles only where they (times two, for the shared tiles) fill at most half of the slots, since
// in the backward launch its workgroups share the chip with the weight gradient's and more of
// them delay those.  Measured (MI355X, 64 -> 64 fp16 over 10 k / 20 k / 50 k / 60 k voxels of the
// indoor cloud, without / with the small tiles): backward launch 22.5 -> 17.0, 26.1 -> 20.9, 35.6 -> 36.0,
// 43.2 -> 47.8 us (128 -> 128 over 28 k voxels: 53.2 -> 63.0 us), hence the rule.
struct RowsGrid {
  bool half_tiles;
  bool drop_table;      // the launch does better on plain 128-row tiles than on the plan's tile table
  int groups;           // groups of four waves per workgroup (KG), 128-row tiles only
  unsigned gx, gz;
  int part_stages;
};
RowsGrid rows_grid(int64_t n_dst, unsigned gy, int stages, bool can_half, bool has_table, int table_grid,
                   bool pair_view, int wgs_per_cu, bool input_gradient, bool can_group) {
  RowsGrid g{};
  const int64_t small_tiles = (int64_t)((n_dst + 127) / 128) * gy;
  const int64_t tiles = (n_dst + kTileRows - 1) / kTileRows;      // (the table has more entries than tiles)
  // A forward launch too big to share its 256-row tiles between two workgroups (below) and
  // not yet a full round of them is neither short-chained nor busy: 128-row tiles in plain order
  // then beat the table's XCD-aware 256-row tiles (64 -> 64 fp16 over 100 k / 130 k voxels:
  // 40.9 -> 34.4, 41.2 -> 36.9 us; 70 k / 80 k voxels with shared 256-row tiles: 28.1 / 29.1 us).
  g.drop_table = can_half && half_tiles_enabled() && has_table && !pair_view && !input_gradient &&
                 small_tiles <= (int64_t)num_cus() * 4 &&
                 (tiles * gy * 2 > (int64_t)num_cus() * wgs_per_cu || stages < 8);
  if (g.drop_table) has_table = false;
  g.half_tiles = can_half && half_tiles_enabled() && !has_table && !pair_view &&
                 (input_gradient ? small_tiles * 4 <= (int64_t)num_cus() * 3 : small_tiles <= (int64_t)num_cus() * 4);
  const int tile_rows = g.half_tiles ? kTileRows / 2 : kTileRows;
  g.gx = has_table ? (unsigned)table_grid : (unsigned)((n_dst + tile_rows - 1) / tile_rows);
  // (an input gradient shares its launch with the weight gradient: its 256-row tiles are shared
  // only up to 2.25 workgroups per CU; 64 -> 64 fp16 backward launch over 70 k / 80 k / 90 k voxels
  // shared 50.7 / 58.6 / 60.4 us, not shared 54.7 / 55.8 / 56.4 us)
  const int64_t slots = g.half_tiles ? (int64_t)num_cus() * 4
                        : input_gradient ? (int64_t)num_cus() * 9 / 4 : (int64_t)num_cus() * wgs_per_cu;
  g.gz = 1;
  g.part_stages = 1;
  g.groups = 1;
  // Forward: no sharing between workgroups but groups of waves inside them, four where every CU has at
  // most one workgroup, two up to two of them (64 -> 64 fp16 over 20 k / 32 k / 45 k / 64 k voxels of
  // the indoor cloud, a whole call: 17.8 -> 15.8, 19.1 -> 17.2, 21.0 -> 19.8, 25.4 -> 22.3 us).  Four
  // waves already keep a CU's matrix cores busy, so groups hide latency but do not make the products
  // of one CU faster: launch_rows therefore takes 32-column tiles while these leave CUs idle.
  if (g.half_tiles && can_group && stages >= 4 && (int64_t)g.gx * gy <= (int64_t)num_cus() * 2) {
    g.groups = (int64_t)g.gx * gy <= num_cus() ? 4 : 2;
    return g;
  }
  if (!pair_view && (has_table ? tiles : (int64_t)g.gx) * gy * 2 <= slots && stages >= 8) {
    g.part_stages = (stages + 1) / 2;
    g.gz = 2;
  }
  return g;
}

template <typename T, int NT, int S, bool RAGGED = false, bool TAILS = false>
int launch_rows(const GmsArgs &a, const Shape &s, const int32_t *nbr,
                const unsigned long long *masks, const int32_t *perm, const int32_t *tile_order,
                int tile_grid, int flip, bool pair_view = false) {
  const int slabs = (s.c_src + 2 * S * s.E - 1) / (2 * S * s.E);
  const unsigned gy = (unsigned)((s.c_dst + 32 * NT - 1) / (32 * NT));
  constexpr bool kCanHalf = NT != 4;
  const RowsGrid rg = rows_grid(a.n_dst, gy, a.k_vol * slabs, kCanHalf, tile_order != nullptr, tile_grid, pair_view,
                                NT >= 3 || (sizeof(T) == 4 && S == 4 && !a.reduced && split_bf16_enabled()) ? 2 : 3, a.transpose_w,
                                kCanHalf && !a.transpose_w);
  // Few tiles: column tiles of 32 put them on twice the CUs, as long as each still has one to itself.
  // A tile's rows are then gathered twice, by CUs that had nothing to do.  Against two workgroups
  // per 64-column tile and atomics / 64-column tiles with four groups: 64 -> 64 fp16 over 1 k voxels
  // 14.3 / 15.3 -> 12.4 us, 5 k 14.4 / 15.0 -> 12.2, 12 k 15.3 / 15.4 -> 13.1; fp32 over 2 k
  // 47.2 / 66.4 -> 40.9; tf32 mode over 5 k 35.2 / 31.6 -> 27.4; 128 -> 128 fp16 over 2 k 21.8 / 24.1 -> 19.5.
  if constexpr (NT == 2 || NT == 3) {
    if (rg.groups == 4 && (int64_t)rg.gx * gy * NT <= num_cus())
      return launch_rows<T, 1, S, RAGGED, TAILS>(a, s, nbr, masks, perm, tile_order, tile_grid, flip, pair_view);
    // ... and where 96-column tiles would be partly empty and 32-column ones fit the chip in one round
    // (128 -> 160 fp16 over 20 k voxels 48.6 -> 37.5 us)
    if (RAGGED && NT == 3 && (s.c_dst + 31) / 32 % 3 != 0 &&
        (a.n_dst + 127) / 128 * ((s.c_dst + 31) / 32) <= (int64_t)num_cus() * 4) {
      if (s.c_dst % 32 == 0 && s.c_src % (2 * S * s.E) == 0)      // (nothing left to mask)
        return launch_rows<T, 1, S>(a, s, nbr, masks, perm, tile_order, tile_grid, flip, pair_view);
      return launch_rows<T, 1, S, RAGGED, TAILS>(a, s, nbr, masks, perm, tile_order, tile_grid, flip, pair_view);
    }
  }
  // With 64-column wave tiles the input gradient and the fp16 forward pass read the weight
  // tensor as it is (16-byte aligned rows of the tile) when the caller brings no re-laid
  // copy; the rest gets one, made here.  Measured: 64 -> 64 over 200k voxels, input gradient
  // 48.3 us raw against 47.3 us + a 4.4 us re-layout launch (the backward call re-lays
  // inside its other launch for free and keeps doing so); with 128-column wave tiles raw
  // weights lose either way (128 -> 128 over 120k voxels: forward 99.7 us against
  // 93.6 + 4.4 us, input gradient 92.9 against 87.7 + 4.4 us).  The fp32 forward pass has no
  // transposing LDS read to use.
  int raw = 0;
  if (NT != 4 && !a.prepacked && reinterpret_cast<uintptr_t>(a.w) % 16 == 0 && raw_weights_enabled())
    raw = a.transpose_w ? 2 : (sizeof(T) == 2 ? 1 : 0);
  // pinned weights: their re-laid copy is made once, and its plain fragment reads beat the
  // transposing ones of the raw tile (64 -> 64 fp16 forward over 200k voxels 41.9 -> 41.3 us)
  if (!RAGGED && raw == 1 && weights_pinned(a.w)) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (!(a.stream && hipStreamIsCapturing(a.stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone)) raw = 0;
  }
  // fp32 tensors: products of bf16 parts, two to a value in "tf32" mode, else three (three or eight 16-bit MFMAs instead
  // of sixteen fp32 ones per product tile); needs whole 32-channel slabs
  constexpr bool kCanSplit = sizeof(T) == 4 && S == 4 && NT != 4;
  // (The pair view's atomics hide fp32 products where there are workgroups enough, and better at three of them to a CU than at two;
  // at 32 columns a tile always.  fp32 MFMAs / three parts: 32 -> 32 over 5 k scattered voxels 16 / 18 us, 96 -> 96 over 60 k LiDAR ones
  // 144 / 162, 128 -> 128 over 20 k scattered ones 67 / 71, 256 -> 256 over 50 k 245 / 266, over 5 k 84 / 63, 64 -> 64 over 20 k 34 / 32.)
  const bool three_parts = NT != 3 && !(pair_view && (NT == 1 || (int64_t)rg.gx * gy > (int64_t)num_cus() * 2));
  // (Three parts take 6 bytes a weight, at 32-bit offsets: a stream under capture whose workspace holds only the 4 of the other
  // layouts stays on fp32 MFMAs.  Masked channel counts come here with room for them.)
  const size_t bytes = (size_t)a.k_vol * a.c_in * a.c_out * 6;
  auto room = [&]() { return bytes <= 0xfffffff0u && (!is_capturing(a.stream) || workspace_bytes(a.stream, 0) >= bytes); };
  const bool split = kCanSplit && !a.transpose_w && !a.prepacked && split_bf16_enabled() &&
                     (a.reduced || RAGGED || (three_parts && room()));
  if (kCanSplit && raw == 2 && split_bf16_enabled()) raw = a.reduced ? 4 : three_parts ? 6 : 2;   // (the input gradient splits as it reads)
  const T *packed = raw ? (const T *)a.w : (const T *)a.prepacked;
  if (split) {
    const void *ws = nullptr;
    int rc = a.reduced ? pack_weights_parts<2>(a, false, &ws) : pack_weights_parts<3>(a, false, &ws);
    if (rc != FGMS_OK) return rc;
    packed = (const T *)ws;
    raw = a.reduced ? 3 : 5;
  } else if (!packed) {
    int rc = pack_weights<T>(a, S, &packed);
    if (rc != FGMS_OK) return rc;
  }
  const bool half_tiles = rg.half_tiles;
  if (rg.drop_table) tile_order = nullptr;
  constexpr int kHalfMT = kCanHalf ? 1 : 2;
  const size_t kGroup = rows_group_chunks<T, NT, S, kHalfMT>(raw) * 16, kSums = rows_sum_chunks<NT, kHalfMT>() * 16;
  constexpr int kMaxGroups = NT == 3 ? 2 : 4;          // (four groups' sums of 96 columns do not fit LDS)
  // (three parts and 64 columns: 50 KB a group, half of the groups)
  const int kg = !half_tiles ? 1 : raw == 5 && NT == 2 ? (rg.groups + 1) / 2 : rg.groups < kMaxGroups ? rg.groups : kMaxGroups;
  size_t lds_rows = half_tiles ? kGroup * kg : rows_group_chunks<T, NT, S, 2>(raw) * 16;
  if (kg > 1 && lds_rows < kGroup + kSums * (kg - 1)) lds_rows = kGroup + kSums * (kg - 1);
  const unsigned gx = rg.gx;
  if (gx == 0) return a.side.kind ? launch_side_job(a.side, a.stream) : FGMS_OK;
  constexpr bool kCanRaw = NT != 4;
  constexpr int kRaw6 = kCanSplit && NT != 3 ? 6 : 0, kRaw5 = kCanSplit && NT != 3 ? 5 : 0;
  constexpr int kRaw4 = kCanSplit ? 4 : 0, kRaw3 = kCanSplit ? 3 : 0, kRaw2 = kCanRaw ? 2 : 0, kRaw1 = kCanRaw && sizeof(T) == 2 ? 1 : 0;
  constexpr int kRagRaw = !RAGGED ? 0 : sizeof(T) == 2 ? kRaw1 : kRaw3, kRagRaw5 = !RAGGED ? 0 : sizeof(T) == 2 ? kRaw1 : kRaw5;
  // (raw is one of those the type and the tile allow)
#define FGMS_BY_RAW(MTv, KGv)                                                                                       \
  (RAGGED && raw == 5 ? gms_rows_kernel<T, NT, S, kRagRaw5, MTv, KGv == 4 && NT == 2 && sizeof(T) == 4 ? 2 : KGv, RAGGED, TAILS> \
   : RAGGED   ? gms_rows_kernel<T, NT, S, kRagRaw, MTv, KGv, RAGGED, TAILS>                                         \
   : raw == 6 ? gms_rows_kernel<T, NT, S, kRaw6, MTv, 1>                                                            \
   : raw == 5 ? gms_rows_kernel<T, NT, S, kRaw5, MTv, KGv == 4 && NT == 2 ? 2 : KGv>                                \
   : raw == 4 ? gms_rows_kernel<T, NT, S, kRaw4, MTv, KGv>                                                          \
   : raw == 3 ? gms_rows_kernel<T, NT, S, kRaw3, MTv, KGv>                                                          \
   : raw == 2 ? gms_rows_kernel<T, NT, S, kRaw2, MTv, KGv>                                                          \
   : raw == 1 ? gms_rows_kernel<T, NT, S, kRaw1, MTv, KGv>                                                          \
              : gms_rows_kernel<T, NT, S, 0, MTv, KGv>)
  auto kern = FGMS_BY_RAW(2, 1);
  if constexpr (kCanHalf) {
    if (half_tiles) kern = kg == 4 ? FGMS_BY_RAW(1, kMaxGroups) : kg == 2 ? FGMS_BY_RAW(1, 2) : FGMS_BY_RAW(1, 1);
  }
#undef FGMS_BY_RAW
  { const int rc_lds = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds_rows); if (rc_lds != FGMS_OK) return rc_lds; }
  // (a tile shared by two workgroups is added up with atomics: its rows start from zero)
  const bool overwrite = a.overwrite && rg.gz == 1 && !pair_view;
  if (a.overwrite && !overwrite) {
    const int rc = launch_fill_zero(a.dst, (size_t)a.n_dst * s.c_dst * sizeof(T), a.stream);
    if (rc != FGMS_OK) return rc;
  }
  const int part_stages = rg.gz > 1 ? rg.part_stages : 0;
  const unsigned gz = rg.gz;
  {
    ProfileScope prof(pair_view  ? (a.transpose_w ? "gms_rows_kernel(dgrad, pair view)" : "gms_rows_kernel(fwd, pair view)")
                      : RAGGED   ? (raw == 3 ? "gms_rows_kernel(fwd, masked, bf16x3)" : "gms_rows_kernel(fwd, masked)")
                      : raw == 4 ? "gms_rows_kernel(dgrad, bf16x3)"
                      : raw == 3 ? "gms_rows_kernel(fwd, bf16x3)"
                      : a.transpose_w ? "gms_rows_kernel(dgrad)" : "gms_rows_kernel(fwd)",
                      a.stream);
    kern<<<dim3(gx + (unsigned)a.side.blocks, gy, gz), kThreads * kg, lds_rows, a.stream>>>(
        (const T *)a.src, packed, (T *)a.dst, nbr, masks, perm, tile_order, (int)a.n_dst, a.k_vol,
        s.c_src, s.c_dst, part_stages > 0 ? part_stages : 1, a.side, pair_view ? 1 : 0,
        (unsigned)((size_t)a.n_src * s.c_src * sizeof(T)), overwrite ? 1 : 0, flip | a.centre << 8, (const T *)a.w);
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

// ---------------------------------------------------------------------------
// Backward in one launch: the output-stationary input gradient (gms_rows_body, weights read
// as they lie) and the per-wave weight gradient (wgrad_wave_body) share a grid.  The two
// do not depend on each other, and workgroups of both kinds resident on the chip at the
// same time finish sooner than the two launches one after the other.
// Measured on 64 -> 64 fp16 over 200k voxels: the two kernels on two streams running
// freely 77 us per (input gradient, weight gradient) pair against 98 us back to back;
// ordering two streams with events costs more than that gain, one grid costs nothing
// (83 us + a 2 us launch that rounds the fp16 weight gradient).  The input gradient's
// workgroups come first in the grid (its longest tiles are the longest jobs of the launch;
// dealing the two kinds alternately or the weight gradient first measured 1-2 us slower).
// Their count is a multiple of 8, so that a workgroup's index mod 8, its XCD, is what the
// plan's XCD-aware orders of either kind assume.
// (2 waves per SIMD where the weight gradient's tile is 128 x 128: its 64 accumulators per lane and
// the rows in flight spill at 3.  128 -> 128 over 40k voxels, forward and backward: tf32 mode 477 -> 327 us.)
template <typename T, int NT, int S, int BI, int BJ, int RAWD, int MT = 2, bool RAGGED = false, bool TAILS = false>
__global__ __launch_bounds__(kThreads, NT >= 3 || RAWD == 6 || BI * BJ == 16 || ((BI == 3 || BJ == 3) && BI * BJ >= 6) ? 2 : 3)
void bwd_fused_kernel(
    const T *__restrict__ gout, const T *__restrict__ w, T *__restrict__ gin,
    const int32_t *__restrict__ nbr, const unsigned long long *__restrict__ block_masks,
    const int32_t *__restrict__ perm, const int32_t *__restrict__ tile_order, int n_in, int k_vol,
    int c_in, int c_out, int part_stages, const T *__restrict__ in, float *__restrict__ gw32,
    const int32_t *__restrict__ kpos, const int32_t *__restrict__ imap,
    const int32_t *__restrict__ omap, SliceMap smap, int row_x, int row_y, int row_z, int wgrad_x,
    unsigned gout_bytes, unsigned in_bytes, int wgrad_blocks, SideJob check, int overwrite, int flip) {
  // grid: row_x * row_y * row_z workgroups of the input gradient (tiles, column tiles,
  // parts of a tile), then wgrad_x * (tiles of dW[k]) of the weight gradient, then those of a
  // side job (the plan's fingerprint check), if there is one
  const int rows_total = row_x * row_y * row_z;
  if ((int)blockIdx.x >= rows_total + wgrad_blocks) {
    run_side_job(check, (int)blockIdx.x - rows_total - wgrad_blocks);
    return;
  }
  if ((int)blockIdx.x < rows_total) {
    const int bx = blockIdx.x % row_x, rest = blockIdx.x / row_x;
    gms_rows_body<T, NT, S, RAWD, MT, 1, RAGGED, TAILS>(gout, w, gin, nbr, block_masks, perm, tile_order, n_in, k_vol, c_out, c_in,
                                      part_stages, bx, rest % row_y, rest / row_y, row_z, gout_bytes, 0, overwrite, flip, 0, nullptr);
  } else {
    const int j = blockIdx.x - rows_total;
    if constexpr (BI <= 3 && BJ <= 3)
      wgrad_wave_body<T, BI, BJ, RAWD == 6 && BI * BJ == 1 ? 0 : split_parts_of(RAWD), RAGGED, TAILS>(      // (see wave_geometry)
          in, gout, gw32, kpos, imap, omap, k_vol, c_in, c_out, smap, j % wgrad_x, j / wgrad_x, in_bytes, gout_bytes);
    else
      wgrad_wg_body<T, BI, BJ, RAWD == 4>(in, gout, gw32, kpos, imap, omap, k_vol, c_in, c_out, smap,
                                          j % wgrad_x, j / wgrad_x);
  }
}

// FGMS_FUSED_BWD=0 keeps the backward call on its two launches (for comparison).
bool fused_bwd_enabled() {
  static const bool on = !(getenv("FGMS_FUSED_BWD") && atoi(getenv("FGMS_FUSED_BWD")) == 0);
  return on;
}

template <typename T, int NT, int S, int BI, int BJ, bool RAGGED = false, bool TAILS = false>
int launch_fused(const GmsArgs &d, const Shape &s, const Plan *p, const WgradArgs &w, const WgradGeometry &g,
                 float *acc32) {
  // the input gradient's grid, as launch_rows lays it out (tiles padded to a multiple of 8)
  const int slabs = (s.c_src + 2 * S * s.E - 1) / (2 * S * s.E);
  const unsigned row_y = (unsigned)((s.c_dst + 32 * NT - 1) / (32 * NT));
  constexpr bool kCanHalf = NT != 4;
  // RAWD: how the input gradient reads the weights (2: as they lie; 4, 6: also split into bf16
  // parts, for fp32 tensors)
  constexpr bool kCanSplit = sizeof(T) == 4 && S == 4 && NT != 4, kCan3 = kCanSplit && BI <= 2 && BJ <= 2;
  const int raw = !kCanSplit || !split_bf16_enabled() ? 2 : d.reduced ? 4 : kCan3 ? 6 : 2;
  const RowsGrid rg = rows_grid(d.n_dst, row_y, d.k_vol * slabs, kCanHalf, p->tile_in != nullptr, p->tile_grid_in,
                                false, NT >= 3 || raw == 6 ? 2 : 3, true, false);
  const unsigned row_x = (rg.gx + 7) / 8 * 8;
  const int part_stages = rg.part_stages;
  const unsigned row_z = rg.gz;
  // what the launch adds to with atomics starts from zero: shared tiles of the input gradient, a
  // weight gradient summed in the caller's fp32 tensor
  const bool zero_gin = d.overwrite && rg.gz > 1, zero_gw = w.overwrite && (void *)acc32 == w.gw;
  if (zero_gin || zero_gw) {
    const int rc = launch_fill_zero_two(d.dst, zero_gin ? (size_t)d.n_dst * s.c_dst * sizeof(T) : 0, w.gw,
                                        zero_gw ? (size_t)w.k_vol * w.c_in * w.c_out * sizeof(float) : 0, d.stream);
    if (rc != FGMS_OK) return rc;
  }
  constexpr int kRaw2 = RAGGED && sizeof(T) == 4 ? 4 : 2;        // (masked fp32 shapes come in parts only)
  constexpr int kHalfMT = kCanHalf ? 1 : 2;
  constexpr int kRaw4 = kCanSplit ? 4 : 2, kRaw6 = kCan3 ? 6 : 2;
  auto kern = rg.half_tiles ? (raw == 6 ? bwd_fused_kernel<T, NT, S, BI, BJ, kRaw6, kHalfMT, RAGGED, TAILS>
                               : raw == 4 ? bwd_fused_kernel<T, NT, S, BI, BJ, kRaw4, kHalfMT, RAGGED, TAILS>
                                          : bwd_fused_kernel<T, NT, S, BI, BJ, kRaw2, kHalfMT, RAGGED, TAILS>)
              : raw == 6    ? bwd_fused_kernel<T, NT, S, BI, BJ, kRaw6, 2, RAGGED, TAILS>
              : raw == 4    ? bwd_fused_kernel<T, NT, S, BI, BJ, kRaw4, 2, RAGGED, TAILS>
                            : bwd_fused_kernel<T, NT, S, BI, BJ, kRaw2, 2, RAGGED, TAILS>;
  size_t lds = g.lds;
  const size_t lds_rows = rg.half_tiles ? rows_group_chunks<T, NT, S, kHalfMT>(raw) * 16 : rows_group_chunks<T, NT, S, 2>(raw) * 16;
  if (lds < lds_rows) lds = lds_rows;
  // Tiles of 64 x 128 leave room for a third workgroup on a CU, which slows the other two down: it pays where workgroups wait for a slot, not
  // where nearly all of them start at once and the last to end is what the launch takes.  So two where the input gradient's tiles are
  // shared (it fills the chip about once) and there are cells for a round and a half of it, and up to seven workgroups to two CUs over dense maps.
  // Backward call, with three / two (indoor voxels, 27 offsets): 64 -> 128 over 30 k (672 workgroups) 38.8 / 36.4 us, 50 k (832) 55.5 / 51.7, 60 k (912)
  // 64.8 / 58.7, 70 k (1 056) 78.0 / 68.3, LiDAR 50 k 59.8 / 55.6 but 70 k 82.8 / 88.8; not shared 85 k (1 200) 70.6 / 73.4, 100 k 80.9 / 83.8, 120 k
  // 99.8 / 96.8, LiDAR 112.0 / 114.7.  128 -> 64 30 k (912, shared) 42.1 / 38.3, 50 k (832) 52.0 / 48.4, 60 k (902) 59.1 / 62.7, 70 k 71.7 / 75.1, 150 k
  // 107.5 / 107.6.  Transposed lists of a stride-2 map, 27 offsets, 64 -> 128 over 297 k pairs (704, 432 of them cells) 43.3 / 39.8, over 212 k (584, 216) 35.1 /
  // 41.0.  Over 140 launches of either kind the rule is 0.7 % over the better of the two, always three 1.5 %, always two 2.5 %.
  if constexpr (sizeof(T) == 2 && BI * BJ == 8) {
    const int64_t cus = num_cus(), wgs = (int64_t)row_x * row_y * row_z + g.tiles;
    const bool shared = row_z > 1 && 2 * g.tiles > 3 * cus;
    const bool dense = g.smap.band_start && w.n_pairs >= 5 * std::max(w.n_in, w.n_out);
    if (g.ty == 1 && (shared || (dense && 2 * wgs < 7 * cus)) && lds < kTwoToACu) lds = kTwoToACu;
  }
  { const int rc_lds = allow_dynamic_lds(reinterpret_cast<const void *>(kern), (size_t)lds); if (rc_lds != FGMS_OK) return rc_lds; }
  {
    ProfileScope prof(RAGGED     ? (raw == 4 ? "bwd_fused_kernel(masked, bf16x3)" : "bwd_fused_kernel(masked)")
                      : raw == 4 ? "bwd_fused_kernel(bf16x3)"
                      : g.smap.by_xcd ? "bwd_fused_kernel(by XCD)" : "bwd_fused_kernel",
                      d.stream);
    SideJob check{};
    (void)plan_take_check(p, &check);
    kern<<<row_x * row_y * row_z + (unsigned)(g.tiles * g.ty) + (unsigned)check.blocks, kThreads, lds, d.stream>>>(
        (const T *)d.src, (const T *)d.w, (T *)d.dst, p->nbr_in, p->mask_in, p->perm_in, p->tile_in,
        (int)d.n_dst, d.k_vol, d.c_in, d.c_out, part_stages, (const T *)w.in, acc32, w.kpos, w.imap, w.omap,
        g.smap, (int)row_x, (int)row_y, (int)row_z, (int)g.tiles,
        (unsigned)((size_t)d.n_src * s.c_src * sizeof(T)), (unsigned)((size_t)w.n_in * w.c_in * sizeof(T)),
        (int)(g.tiles * g.ty), check, d.overwrite && rg.gz == 1 ? 1 : 0, p->flip_in);
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

template <typename T, typename F>
int dispatch_shape(const Shape &s, F &&f);

template <int NT, typename F>
int dispatch_rows_slab(const Shape &s, F &&f) {
  if (s.SR == 4) return f(std::integral_constant<int, NT>{}, std::integral_constant<int, 4>{});
  if (s.SR == 3) return f(std::integral_constant<int, NT>{}, std::integral_constant<int, 3>{});
  if (s.SR == 2) return f(std::integral_constant<int, NT>{}, std::integral_constant<int, 2>{});
  return f(std::integral_constant<int, NT>{}, std::integral_constant<int, 1>{});
}

template <typename T, typename F>
int dispatch_rows_shape(const Shape &s, F &&f) {
  if (s.NTR == 4) return dispatch_rows_slab<4>(s, f);
  if (s.NTR == 3) return dispatch_rows_slab<3>(s, f);
  if (s.NTR == 2) return dispatch_rows_slab<2>(s, f);
  return dispatch_rows_slab<1>(s, f);
}

template <typename T, typename F>
int dispatch_shape(const Shape &s, F &&f) {
  if (s.NT == 2) {
    if (s.S == 4) return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 4>{});
    if (s.S == 2) return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
    return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  }
  if (s.S == 4) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{});
  if (s.S == 2) return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
  return f(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
}

}  // namespace

int num_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess)
      cus = p.multiProcessorCount;
    if (cus <= 0) cus = 256;
  }
  return cus;
}

int pack_weights_any(const GmsArgs &a, int S, const void **packed) {
  if (a.dtype == FGMS_F16) {
    const __half *p = nullptr;
    int rc = pack_weights<__half>(a, S, &p);
    *packed = p;
    return rc;
  }
  const float *p = nullptr;
  int rc = pack_weights<float>(a, S, &p);
  *packed = p;
  return rc;
}

// Input gradient `d` (output-stationary, through plan `p`) and weight gradient `w` of one
// layer in one launch where bwd_fused_kernel covers the shape; *done = false (and nothing
// launched) where it does not.
int launch_fused_bwd(const GmsArgs &d, const Plan *p, const WgradArgs &w, bool *done) {
  *done = false;
  if (!fused_bwd_enabled() || !d.transpose_w || d.prepacked || d.side.kind || w.side.kind ||
      d.k_vol != w.k_vol || d.c_in != w.c_in || d.c_out != w.c_out || d.dtype != w.dtype || d.stream != w.stream)
    return FGMS_OK;
  const Shape s = shape_of(d);
  if (!s.ok || reinterpret_cast<uintptr_t>(d.w) % 16 != 0 || !raw_weights_enabled()) return FGMS_OK;
  WgradGeometry g;
  if (!mfma_wgrad_supported(w) || wgrad_geometry(w, &g, true) != FGMS_OK) return FGMS_OK;
  float *acc32 = nullptr;
  int rc = wgrad_accumulator(w, &acc32);
  if (rc != FGMS_OK) return rc;
  bool found = false;
  // (wave tile columns NT of the input gradient, MFMA steps per slab S) follow from c_in and
  // c_out, and so do the block counts (BI, BJ) of the weight gradient's tile.  Input channels: NT 1, BI 1 for
  // odd numbers of 32s; 2, 2 for 64 and odd multiples; 2 or (launches that fill the chip) 4, BI 4 for multiples of 128; 3, 3
  // for odd multiples of 96 over dense maps.  Output channels: S 2, BJ 1 for 32 and other odd numbers of 32s; 4, 2
  // for 64 and odd multiples; 4, 4 for multiples of 128; 3, 3 for odd multiples of 96 over dense maps, 3, 1 over thin ones.
#define FGMS_FB(TT, NTv, Sv, BIv, BJv)                                             \
  if (!found && s.NTR == NTv && s.SR == Sv && g.bi == BIv && g.bj == BJv) {          \
    found = true;                                                                    \
    rc = launch_fused<TT, NTv, Sv, BIv, BJv>(d, s, p, w, g, acc32);                 \
  }
  if (d.dtype == FGMS_F16) {
    FGMS_FB(__half, 1, 2, 1, 1) FGMS_FB(__half, 1, 4, 1, 2) FGMS_FB(__half, 1, 4, 1, 4)
    FGMS_FB(__half, 2, 2, 2, 1) FGMS_FB(__half, 2, 4, 2, 2) FGMS_FB(__half, 2, 4, 2, 4)
    FGMS_FB(__half, 2, 2, 4, 1) FGMS_FB(__half, 2, 4, 4, 2) FGMS_FB(__half, 2, 4, 4, 4)
    FGMS_FB(__half, 4, 2, 4, 1) FGMS_FB(__half, 4, 4, 4, 2) FGMS_FB(__half, 4, 4, 4, 4)
    FGMS_FB(__half, 3, 2, 3, 1) FGMS_FB(__half, 3, 4, 3, 2) FGMS_FB(__half, 3, 3, 3, 3)
    FGMS_FB(__half, 1, 3, 1, 3) FGMS_FB(__half, 2, 3, 2, 3) FGMS_FB(__half, 4, 3, 2, 3)
    FGMS_FB(__half, 1, 3, 1, 1) FGMS_FB(__half, 2, 3, 2, 1) FGMS_FB(__half, 2, 3, 4, 1) FGMS_FB(__half, 4, 3, 4, 1)
  } else {
    FGMS_FB(float, 1, 4, 1, 1) FGMS_FB(float, 1, 4, 1, 2) FGMS_FB(float, 1, 4, 1, 4)
    FGMS_FB(float, 2, 4, 2, 1) FGMS_FB(float, 2, 4, 2, 2) FGMS_FB(float, 2, 4, 2, 4)
    FGMS_FB(float, 2, 4, 4, 1) FGMS_FB(float, 2, 4, 4, 2) FGMS_FB(float, 2, 4, 4, 4)
  }
#undef FGMS_FB
  if (!found) return FGMS_OK;     // (no such kernel: the caller's two launches)
  if (rc != FGMS_OK) return rc;
  *done = true;
  return wgrad_finish(w, acc32);
}

// The output-stationary kernel gathers through a buffer resource: 32-bit byte offsets, and
// offsets at or above 2^31 stand for "no row" (gather_issue_buf).
static bool rows_fit_buffer(const GmsArgs &a) {
  const size_t c_src = a.transpose_w ? a.c_out : a.c_in;
  return (size_t)a.n_src * c_src * (a.dtype == FGMS_F16 ? 2 : 4) <= kMaxBufferBytes;
}

// The same for channel counts that fill no whole tile.
int launch_ragged_bwd(const GmsArgs &d, const Plan *p, const WgradArgs &w, bool *done) {
  *done = false;
  if (!fused_bwd_enabled() || !p || !p->groups.empty() || d.k_vol > 64 || d.k_vol != p->k_vol || !p->dgrad_ok ||
      d.n_dst != p->n_in || d.n_src != p->n_out || !rows_fit_buffer(d))
    return FGMS_OK;
  const Shape s = ragged_shape(d);
  WgradGeometry g;
  const bool f16 = d.dtype == FGMS_F16;
  auto tiles = [&](int c) { return f16 ? ragged_tiles(c, worth_96_columns(w.n_pairs, w.n_in, w.n_out)) : (c + 31) / 32 % 2 ? 1 : 2; };
  if (!s.ok || !ragged_wgrad_geometry(w, tiles(w.c_in), tiles(w.c_out), &g)) return FGMS_OK;
  bool found = false;
  int rc = FGMS_OK;
  float *acc32 = nullptr;
  // (column tiles NT of the input gradient, k-steps S of its slab, blocks BJ of the weight gradient's tile; BI = NT.
  // NT: 1 up to 32 input channels, 2 up to 64 and for an even number of 32s, 3 for 72 .. 96, 136 .. 160 and the like.
  // S, BJ by output channels: 2, 1 up to 32; 3, 2 for 40 and 48; 4, 2 for 56, 64 and an even number of 32s; 3, 3 for
  // 72 .. 96; 4, 3 for 136 .. 160 and other odd numbers of 32s.)
#define FGMS_FRF(NTv, BJv)                                                                                        \
  if (!found && !f16 && s.NTR == NTv && g.bi == NTv && g.bj == BJv) {                                             \
    found = true;                                                                                                 \
    if ((rc = wgrad_accumulator(w, &acc32)) == FGMS_OK)                                                           \
      rc = launch_fused<float, NTv, 4, NTv, BJv, true>(d, s, p, w, g, acc32);                                     \
  }
  FGMS_FRF(1, 1) FGMS_FRF(1, 2) FGMS_FRF(2, 1) FGMS_FRF(2, 2)
#undef FGMS_FRF
#define FGMS_FR(NTv, Sv, BJv)                                                                                     \
  if (!found && f16 && !half_chunk(d) && s.NTR == NTv && s.SR == Sv && g.bi == NTv && g.bj == BJv) {                                \
    found = true;                                                                                                 \
    if ((rc = wgrad_accumulator(w, &acc32)) == FGMS_OK)                                                           \
      rc = launch_fused<__half, NTv, Sv, NTv, BJv, true>(d, s, p, w, g, acc32);                                   \
  }
#define FGMS_FT(NTv)                                                                                              \
  if (!found && f16 && half_chunk(d) && s.NTR == NTv && s.SR == 2 && g.bi == NTv && g.bj == 1) {                  \
    found = true;                                                                                                 \
    if ((rc = wgrad_accumulator(w, &acc32)) == FGMS_OK)                                                           \
      rc = launch_fused<__half, NTv, 2, NTv, 1, true, true>(d, s, p, w, g, acc32);                                \
  }
  FGMS_FT(1) FGMS_FT(2) FGMS_FT(3)
#undef FGMS_FT
  FGMS_FR(1, 2, 1) FGMS_FR(1, 3, 2) FGMS_FR(1, 4, 2) FGMS_FR(1, 3, 3) FGMS_FR(1, 4, 3)
  FGMS_FR(2, 2, 1) FGMS_FR(2, 3, 2) FGMS_FR(2, 4, 2) FGMS_FR(2, 3, 3) FGMS_FR(2, 4, 3)
  FGMS_FR(3, 2, 1) FGMS_FR(3, 3, 2) FGMS_FR(3, 4, 2) FGMS_FR(3, 3, 3) FGMS_FR(3, 4, 3)
#undef FGMS_FR
  if (!found) return FGMS_OK;
  if (rc != FGMS_OK) return rc;
  *done = true;
  return wgrad_finish(w, acc32);
}

int planned_pack_job(const GmsArgs &a, SideJob *job, const void **packed) {
  const Shape s = shape_of(a);
  if (!s.ok) {
    set_error("planned_pack_job: unsupported shape");
    return FGMS_E_INVALID;
  }
  const size_t esz = a.dtype == FGMS_F16 ? 2 : 4;
  const size_t n = (size_t)a.k_vol * a.c_in * a.c_out;
  void *ws = nullptr;
  int rc = workspace_get(a.stream, 0, n * esz, &ws);
  if (rc != FGMS_OK) return rc;
  *job = SideJob{};
  job->kind = 1;
  job->src = a.w;
  job->dst = ws;
  job->n = n;
  job->k_vol = a.k_vol; job->c_in = a.c_in; job->c_out = a.c_out;
  job->S = s.SR; job->transpose = a.transpose_w; job->dtype = a.dtype;
  // about 8 elements per thread of 256-thread workgroups
  size_t blocks = ((n + 2047) / 2048 + 7) / 8 * 8;
  job->blocks = (int)(blocks > 1024 ? 1024 : blocks);
  *packed = ws;
  return FGMS_OK;
}

int launch_side_job(const SideJob &job, hipStream_t stream) {
  if (job.kind == 0 || job.blocks <= 0) return FGMS_OK;
  side_job_kernel<<<(unsigned)job.blocks, 256, 0, stream>>>(job);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

// FGMS_RAW_WEIGHTS=0 keeps the forward pass on re-laid weights (for comparison).
bool raw_weights_enabled() {
  static const bool on = !(getenv("FGMS_RAW_WEIGHTS") && atoi(getenv("FGMS_RAW_WEIGHTS")) == 0);
  return on;
}

// FGMS_HALF_TILES=0 keeps small launches on 256-row tiles (for comparison).
bool half_tiles_enabled() {
  static const bool on = !(getenv("FGMS_HALF_TILES") && atoi(getenv("FGMS_HALF_TILES")) == 0);
  return on;
}

// FGMS_SPLIT_BF16=0 keeps fp32 tensors on fp32 MFMAs, in full precision and in "tf32" mode (for comparison).
bool split_bf16_enabled() {
  static const bool on = !(getenv("FGMS_SPLIT_BF16") && atoi(getenv("FGMS_SPLIT_BF16")) == 0);
  return on;
}

bool mfma_gms_supported(const GmsArgs &a) { return shape_of(a).ok; }

int launch_mfma_gms(const GmsArgs &a) {
  const Shape s = shape_of(a);
  if (!s.ok) {
    set_error("launch_mfma_gms: unsupported shape");
    return FGMS_E_INVALID;
  }
  if (a.dtype == FGMS_F16)
    return dispatch_shape<__half>(s, [&](auto nt, auto sv) {
      return launch_pairs<__half, decltype(nt)::value, decltype(sv)::value>(a, s);
    });
  return dispatch_shape<float>(s, [&](auto nt, auto sv) {
    return launch_pairs<float, decltype(nt)::value, decltype(sv)::value>(a, s);
  });
}

bool planned_gms_supported(const GmsArgs &a, const Plan *p) {
  if (!p || a.dense_k >= 0 || a.k_vol > 64 || a.k_vol != p->k_vol) return false;
  if (a.transpose_w) {
    if (!p->dgrad_ok || a.n_dst != p->n_in || a.n_src != p->n_out) return false;
  } else {
    if (!p->fwd_ok || a.n_dst != p->n_out || a.n_src != p->n_in) return false;
  }
  // result rows are updated with 8- and 16-byte accesses
  if (reinterpret_cast<uintptr_t>(a.dst) % 16) return false;
  if (!rows_fit_buffer(a)) return false;
  return shape_of(a).ok;
}

int launch_planned_gms(const GmsArgs &a, const Plan *p) {
  const Shape s = shape_of(a);
  if (!s.ok || !planned_gms_supported(a, p)) {
    set_error("launch_planned_gms: unsupported shape or plan");
    return FGMS_E_INVALID;
  }
  const int32_t *nbr = a.transpose_w ? p->nbr_in : p->nbr_out;
  const unsigned long long *masks = a.transpose_w ? p->mask_in : p->mask_out;
  const int32_t *perm = a.transpose_w ? p->perm_in : p->perm_out;
  const int32_t *tile_order = a.transpose_w ? p->tile_in : p->tile_out;
  const int tile_grid = a.transpose_w ? p->tile_grid_in : p->tile_grid_out;
  const int flip = a.transpose_w ? p->flip_in : p->flip_out;
  // (a pending fingerprint check of the plan rides along as the launch's side job)
  GmsArgs with_check = a;
  if (!with_check.side.kind) (void)plan_take_check(p, &with_check.side);
  const GmsArgs &a_ = with_check;
  if (a.dtype == FGMS_F16)
    return dispatch_rows_shape<__half>(s, [&](auto nt, auto sv) {
      return launch_rows<__half, decltype(nt)::value, decltype(sv)::value>(a_, s, nbr, masks, perm, tile_order, tile_grid,
                                                                              flip);
    });
  return dispatch_rows_shape<float>(s, [&](auto nt, auto sv) {
    return launch_rows<float, decltype(nt)::value, decltype(sv)::value>(a_, s, nbr, masks, perm, tile_order, tile_grid,
                                                                              flip);
  });
}

bool ragged_gms_supported(const GmsArgs &a, const Plan *p) {
  if (!p || !p->groups.empty() || a.dense_k >= 0 || a.transpose_w || a.k_vol > 64 || a.k_vol != p->k_vol) return false;
  return p->fwd_ok && a.n_dst == p->n_out && a.n_src == p->n_in && rows_fit_buffer(a) && ragged_shape(a).ok;
}

int launch_ragged_gms(const GmsArgs &a, const Plan *p) {
  const Shape s = ragged_shape(a);
  if (!ragged_gms_supported(a, p)) {
    set_error("launch_ragged_gms: unsupported shape or plan");
    return FGMS_E_INVALID;
  }
  GmsArgs a_ = a;
  if (!a_.side.kind) (void)plan_take_check(p, &a_.side);
  if (a.dtype != FGMS_F16) {
    if (s.NTR == 2)
      return launch_rows<float, 2, 4, true>(a_, s, p->nbr_out, p->mask_out, p->perm_out, p->tile_out, p->tile_grid_out, p->flip_out);
    return launch_rows<float, 1, 4, true>(a_, s, p->nbr_out, p->mask_out, p->perm_out, p->tile_out, p->tile_grid_out, p->flip_out);
  }
  if (half_chunk(a)) {                        // (one column tile)
    auto go = [&](auto sv) {
      return launch_rows<__half, 1, decltype(sv)::value, true, true>(a_, s, p->nbr_out, p->mask_out, p->perm_out, p->tile_out, p->tile_grid_out,
                                                                     p->flip_out);
    };
    return s.SR == 2 ? go(std::integral_constant<int, 2>{}) : s.SR == 3 ? go(std::integral_constant<int, 3>{}) : go(std::integral_constant<int, 4>{});
  }
#define FGMS_RG(NTv, Sv)                   \
  if (s.NTR == NTv && s.SR == Sv)          \
    return launch_rows<__half, NTv, Sv, true>(a_, s, p->nbr_out, p->mask_out, p->perm_out, p->tile_out, p->tile_grid_out, p->flip_out);
  FGMS_RG(1, 2) FGMS_RG(1, 3) FGMS_RG(1, 4) FGMS_RG(2, 2) FGMS_RG(2, 3) FGMS_RG(2, 4) FGMS_RG(3, 2) FGMS_RG(3, 3) FGMS_RG(3, 4)
#undef FGMS_RG
  set_error("launch_ragged_gms: no such tile");
  return FGMS_E_INVALID;
}

bool pair_view_gms_supported(const GmsArgs &a, const Plan *p) {
  if (!p || !p->pv_rows || a.dense_k >= 0 || a.k_vol != p->k_vol) return false;
  if (!p->pv_in && is_capturing(a.stream)) return false;
  if (a.transpose_w ? (a.n_dst != p->n_in || a.n_src != p->n_out) : (a.n_dst != p->n_out || a.n_src != p->n_in))
    return false;
  if (reinterpret_cast<uintptr_t>(a.dst) % 16 || !rows_fit_buffer(a)) return false;
  return shape_of(a).ok;
}

int launch_pair_view_gms(const GmsArgs &a, const Plan *p) {
  if (!pair_view_gms_supported(a, p) || !p->pv_in) {      // (plan_pair_view comes first)
    set_error("launch_pair_view_gms: unsupported shape or plan");
    return FGMS_E_INVALID;
  }
  // (the view was built on the stream of the first call that walked it)
  if (p->pv_ready && a.stream != p->pv_stream) FGMS_HIP_TRY(hipStreamWaitEvent(a.stream, p->pv_ready, 0));
  // the virtual rows stand in for the destination rows: tiles, the in-range test and the
  // choice of the wave tile's width go by their number
  GmsArgs v = a;
  v.n_dst = p->pv_rows;
  v.overwrite = false;
  if (a.overwrite) {
    const int rc = launch_fill_zero(a.dst, (size_t)a.n_dst * (a.transpose_w ? a.c_in : a.c_out) * (a.dtype == FGMS_F16 ? 2 : 4), a.stream);
    if (rc != FGMS_OK) return rc;
  }
  const Shape s = shape_of(v);
  const int32_t *nbr = a.transpose_w ? p->pv_out : p->pv_in;
  const int32_t *dest = a.transpose_w ? p->pv_in : p->pv_out;
  if (a.dtype == FGMS_F16)
    return dispatch_rows_shape<__half>(s, [&](auto nt, auto sv) {
      return launch_rows<__half, decltype(nt)::value, decltype(sv)::value>(v, s, nbr, p->pv_mask, dest, nullptr, 0, 0, true);
    });
  return dispatch_rows_shape<float>(s, [&](auto nt, auto sv) {
    return launch_rows<float, decltype(nt)::value, decltype(sv)::value>(v, s, nbr, p->pv_mask, dest, nullptr, 0, 0, true);
  });
}

// weight gradient: see fgms_wgrad.hip
}  // namespace fgms
