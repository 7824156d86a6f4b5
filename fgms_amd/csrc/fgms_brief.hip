// Small fp16 forward launches: every offset of a tile at once.
//
// Where a launch has fewer tiles than the chip has CUs, the output-stationary kernel's time is its start and one tile's chain
// of stages: each waits for its rows, and four groups of waves walk 27 offsets in seven of them.  Here a workgroup of sixteen waves takes 32 rows
// and 32 columns, a wave two of up to 32 offsets, and everything it needs is requested at once: the indices and the weights of all
// offsets (27 x 32 x 32 halfs are 54 KB of LDS), then the rows, straight into the registers the matrix
// instructions take them from.  So a launch is two dependent loads long whatever the number of offsets, and the waves' sums meet in
// LDS once.  The price is every weight once for 32 rows.  Bound by its latencies and the launch: 32 -> 32 over 2 k voxels 6.3 us
// a call among others, 10.3 before.
#include "fgms_device.h"
#include "fgms_internal.h"
#include "fgms_mma.h"
#include "fgms_tile_ops.h"

namespace fgms {
namespace {

constexpr int kBriefWaves = 16, kBriefRounds = 2, kBriefOffsets = kBriefWaves * kBriefRounds, kBriefRows = 32;

struct BriefArgs {
  const __half *src, *w;
  __half *dst;
  const int32_t *nbr, *perm;
  const unsigned long long *block_masks;
  unsigned long long centre;      // the bit of an offset through which every row is its own neighbour (see Plan::centre_line)
  int n_dst, k_vol, c_src, c_dst, overwrite, flip;
  unsigned src_bytes, w_bytes;
  SideJob side;
};

// S: 16 source channels each; those from c_src on and columns from c_dst on (multiples of 8) do not exist and arrive as zeros.
template <int S>
__global__ __launch_bounds__(kBriefWaves * 64, 4) void gms_brief_kernel(BriefArgs a) {
  constexpr int kChunks = 16 * S * 4;                                     // 16-byte chunks of an offset's 32 columns
  constexpr int NW = kBriefOffsets * kChunks / (kBriefWaves * 64);
  int block_x = blockIdx.x;
  if (a.side.blocks) {
    if (block_x < a.side.blocks) {
      if (blockIdx.y == 0) run_side_job(a.side, block_x);
      return;
    }
    block_x -= a.side.blocks;
  }
  extern __shared__ int4v lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nt0 = blockIdx.y * 32;
  const int pos = block_x * kBriefRows + (lane & 31), safe_pos = min(pos, a.n_dst - 1);
  const unsigned long long mask = a.block_masks[block_x * kBriefRows / 64] | a.centre;
  if (!mask && !a.overwrite) return;

  int g[kBriefRounds];
#pragma unroll
  for (int t = 0; t < kBriefRounds; ++t) g[t] = a.nbr[(size_t)min(wave + t * kBriefWaves, a.k_vol - 1) * a.n_dst + safe_pos];
  // the accumulator register `wave` of the tile: what this wave adds up and writes
  const int out_pos = block_x * kBriefRows + (wave / 4) * 8 + h * 4 + wave % 4;
  const int safe_out = min(out_pos, a.n_dst - 1);
  const int out_row = a.perm ? a.perm[safe_out] : safe_out;

  const __amdgpu_buffer_rsrc_t wrsrc = rows_resource(a.w, a.w_bytes), rsrc = rows_resource(a.src, a.src_bytes);
  int4v wreg[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int e = tid + i * kBriefWaves * 64, k = e / kChunks, c = e % kChunks / 4, to = nt0 + e % 4 * 8;
    const unsigned off = k < a.k_vol && c < a.c_src && to < a.c_dst ? (unsigned)((k * a.c_src + c) * a.c_dst + to) * 2u : kAbsentRow;
    wreg[i] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, off, 0, 0));
  }
  int4v v[kBriefRounds][S];
  unsigned rows[kBriefRounds];                                            // which of the 32 have a pair
#pragma unroll
  for (int t = 0; t < kBriefRounds; ++t) {
    const int k = wave + t * kBriefWaves;
    const bool live = pos < a.n_dst && g[t] >= 0 && k < a.k_vol && ((mask >> k) & 1);
    rows[t] = (unsigned)__builtin_amdgcn_ballot_w64(live);
    const unsigned off = live ? (unsigned)g[t] * (unsigned)(a.c_src * 2) : kAbsentRow;
#pragma unroll
    for (int s = 0; s < S; ++s)
      v[t][s] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(
                                              rsrc, (h * S + s) * 8 < a.c_src ? off + (unsigned)((h * S + s) * 16) : kAbsentRow, 0, 0));
  }
  const int out_col = nt0 + (lane & 30);
  __half2 *const out = reinterpret_cast<__half2 *>(a.dst + (size_t)out_row * a.c_dst + min(out_col, a.c_dst - 2));
  __half2 old = {};
  if (!a.overwrite) old = *out;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int e = tid + i * kBriefWaves * 64;
    if (e < a.k_vol * kChunks) lds[e] = wreg[i];
  }
  __syncthreads();

  const float16v zero = {};
  float16v acc = zero;
  auto products = [&](float16v &to, int t) {
    const int k = wave + t * kBriefWaves;
    const int4v *const w = lds + (size_t)(a.flip ? a.flip - k : k) * kChunks;
#pragma unroll
    for (int s = 0; s < S; ++s) mma<__half>(to, v[t][s], raw_weight_frag<1, S>(w, s, 0, lane));
  };
#pragma unroll
  for (int t = 0; t < kBriefRounds; ++t)
    if (rows[t]) products(acc, t);
  // a weight that is not finite reaches the rows with a pair through its offset and no others (a zero row times infinity)
  float beyond = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) beyond = __builtin_fmaf(acc[r], 0.f, beyond);
  if (__builtin_amdgcn_ballot_w64(beyond != 0.f)) {
    acc = zero;
#pragma unroll
    for (int t = 0; t < kBriefRounds; ++t) {
      float16v own = zero;
      if (rows[t]) products(own, t);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (rows[t] >> ((r / 4) * 8 + h * 4 + r % 4) & 1) acc[r] += own[r];
    }
  }
  __syncthreads();                          // every wave has read its weights
  float *const sums = reinterpret_cast<float *>(lds);
#pragma unroll
  for (int r = 0; r < 16; ++r) sums[(wave * 16 + r) * 64 + lane] = acc[r];
  __syncthreads();
  float sum = 0.f;
#pragma unroll
  for (int q = 0; q < kBriefWaves; ++q) sum += sums[(q * 16 + wave) * 64 + lane];
  const float next = swap_with_neighbour(sum);
  if (out_pos < a.n_dst && out_col < a.c_dst && !(lane & 1)) {
    const float2 o = __half22float2(old);
    *out = __floats2half2_rn(o.x + sum, o.y + next);
  }
}

// Layers of up to 32 channels in, 32 columns a workgroup: all weights of the layer stay in LDS, and a wave walks the offsets of its own 32 rows.
// Four offsets make a batch; the next batch's rows and the indices of the one behind it are in flight, and after the weights have come in
// there is no barrier: a stage of the output-stationary kernel, which brings 2 KB of weights and waits for four waves, does 32 channels' work of
// 128 clocks.  Bound by the L1's gathers where the launch is long: whole rows by neighbouring lanes, and through LDS to the lanes that want them
// (gathered as the matrix instructions take them, 16 bytes of another row a lane, 32 -> 32 over 100 k indoor voxels 14.8 us and 200 k 24.3,
// this way 12.3 and 22.2).
constexpr int kHeldWaves = 8, kHeldBatch = 4;

struct HeldBatch {
  int k[kHeldBatch];              // (-1: none)
};
__device__ __forceinline__ HeldBatch next_offsets(unsigned long long &todo) {
  HeldBatch b;
#pragma unroll
  for (int j = 0; j < kHeldBatch; ++j) {
    b.k[j] = todo ? __builtin_ctzll(todo) : -1;
    todo &= todo - 1;
  }
  return b;
}

template <int S>
__global__ __launch_bounds__(kHeldWaves * 64, 4) void gms_held_kernel(BriefArgs a, const int32_t *__restrict__ tile_order) {
  constexpr int C = 2 * S, kChunks = 16 * S * 4, kThreads_ = kHeldWaves * 64;
  constexpr int NW = kBriefOffsets * kChunks / kThreads_;
  int block_x = blockIdx.x;
  if (a.side.blocks) {
    if (block_x < a.side.blocks) {
      if (blockIdx.y == 0) run_side_job(a.side, block_x);
      return;
    }
    block_x -= a.side.blocks;
  }
  int tile = block_x;
  if (tile_order) {
    tile = tile_order[block_x];
    if (tile < 0) return;
    tile &= 0xFFFFFF;
  }
  if (tile * (kHeldWaves * 32) >= a.n_dst) return;
  extern __shared__ int4v lds[];
  __shared__ int out_rows[kHeldWaves][32];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, nt0 = blockIdx.y * 32;
  const int pos0 = tile * (kHeldWaves * 32) + wave * 32, pos = pos0 + (lane & 31), safe_pos = min(pos, a.n_dst - 1);
  const bool in_range = pos < a.n_dst;
  unsigned long long mask = a.block_masks[min(pos0, a.n_dst - 1) / 64] | a.centre;
  if (pos0 >= a.n_dst) mask = 0;
  unsigned long long todo = (unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(mask & 0xffffffffu)) |
                            ((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(mask >> 32)) << 32);

  const unsigned long long all = todo;
  int4v *const rows_lds = lds + a.k_vol * kChunks + wave * (32 * C);      // one offset's
  const __amdgpu_buffer_rsrc_t wrsrc = rows_resource(a.w, a.w_bytes), rsrc = rows_resource(a.src, a.src_bytes);
  // load `it` of an offset: rows it * (64 / C) + lane / C, piece lane % C of each
  auto row_of = [&](int it) { return it * (64 / C) + lane / C; };
  auto indices = [&](int (&g)[kHeldBatch][S], const HeldBatch &b) {
#pragma unroll
    for (int j = 0; j < kHeldBatch; ++j)
#pragma unroll
      for (int it = 0; it < S; ++it) g[j][it] = a.nbr[(size_t)max(b.k[j], 0) * a.n_dst + min(pos0 + row_of(it), a.n_dst - 1)];
  };
  auto gather = [&](int4v (&v)[kHeldBatch][S], const int (&g)[kHeldBatch][S], const HeldBatch &b) {
#pragma unroll
    for (int j = 0; j < kHeldBatch; ++j)
#pragma unroll
      for (int it = 0; it < S; ++it) {
        const bool live = pos0 + row_of(it) < a.n_dst && b.k[j] >= 0 && g[j][it] >= 0 && lane % C * 8 < a.c_src;
        const unsigned off = live ? (unsigned)g[j][it] * (unsigned)(a.c_src * 2) + (unsigned)(lane % C * 16) : kAbsentRow;
        v[j][it] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
      }
  };
  float16v acc[1][1] = {};
  auto product = [&](float16v &to, const int4v (&v)[S], int k) {
    const int4v *const w = lds + (size_t)(a.flip ? a.flip - k : k) * kChunks;
#pragma unroll
    for (int it = 0; it < S; ++it) rows_lds[a_slot<S>(row_of(it), lane % C)] = v[it];
    wave_lds_fence();
#pragma unroll
    for (int s = 0; s < S; ++s) mma<__half>(to, rows_lds[a_slot<S>(lane & 31, h * S + s)], raw_weight_frag<1, S>(w, s, 0, lane));
    wave_lds_fence();
  };
  auto products = [&](const int4v (&v)[kHeldBatch][S], const HeldBatch &b) {
#pragma unroll
    for (int j = 0; j < kHeldBatch; ++j)
      if (b.k[j] >= 0) product(acc[0][0], v[j], b.k[j]);
  };

  HeldBatch b0 = next_offsets(todo), b1 = next_offsets(todo);
  int g0[kHeldBatch][S], g1[kHeldBatch][S];
  indices(g0, b0);
  indices(g1, b1);
  const int out_row = a.perm ? a.perm[safe_pos] : safe_pos;
  int4v wreg[NW];
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int e = tid + i * kThreads_, k = e / kChunks, c = e % kChunks / 4, to = nt0 + e % 4 * 8;
    const unsigned off = k < a.k_vol && c < a.c_src && to < a.c_dst ? (unsigned)((k * a.c_src + c) * a.c_dst + to) * 2u : kAbsentRow;
    wreg[i] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, off, 0, 0));
  }
  int4v v0[kHeldBatch][S], v1[kHeldBatch][S];
  gather(v0, g0, b0);
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int e = tid + i * kThreads_;
    if (e < a.k_vol * kChunks) lds[e] = wreg[i];
  }
  if (lane < 32) out_rows[wave][lane] = in_range ? out_row : -1;
  __syncthreads();

  // (two batches a turn, so that each has registers of its own)
  while (b0.k[0] >= 0) {
    gather(v1, g1, b1);
    HeldBatch next = next_offsets(todo);
    indices(g0, next);
    products(v0, b0);
    b0 = next;
    if (b1.k[0] < 0) break;
    gather(v0, g0, b0);
    next = next_offsets(todo);
    indices(g1, next);
    products(v1, b1);
    b1 = next;
  }
  // a weight that is not finite reaches the rows with a pair through its offset and no others: one offset at a time
  float beyond = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) beyond = __builtin_fmaf(acc[0][0][r], 0.f, beyond);
  if (__builtin_amdgcn_ballot_w64(beyond != 0.f)) {
    acc[0][0] = float16v{};
    for (unsigned long long rest = all; rest; rest &= rest - 1) {
      HeldBatch one;
#pragma unroll
      for (int j = 0; j < kHeldBatch; ++j) one.k[j] = j ? -1 : __builtin_ctzll(rest);
      indices(g0, one);
      gather(v0, g0, one);
      float16v own = {};
      product(own, v0[0], one.k[0]);
      const unsigned rows = (unsigned)__builtin_amdgcn_ballot_w64(in_range && a.nbr[(size_t)one.k[0] * a.n_dst + safe_pos] >= 0);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (rows >> ((r / 4) * 8 + h * 4 + r % 4) & 1) acc[0][0][r] += own[r];
    }
  }
  // (Added to what is there: all old values requested before the first sum.  One by one, each behind the store before it, 32 -> 32 over 35 k
  // indoor voxels 13.6 us and 16 -> 64 over 60 k 15.8, 12.2 and 13.6 with the kernels that had these layers before; this way 12.4 and 12.2.)
  if (a.overwrite) write_tile<__half, 1, kTileStore, true>(acc, a.dst, out_rows[wave], a.c_dst, nt0, lane);
  else if (mask) add_rows<__half, 1, true>(acc, a.dst, out_rows[wave], a.c_dst, nt0, lane);
}

int brief_steps(const GmsArgs &a) { return (a.c_in + 15) / 16; }
size_t brief_lds(const GmsArgs &a) {
  const size_t weights = (size_t)a.k_vol * brief_steps(a) * 1024, sums = (size_t)kBriefWaves * 16 * 64 * sizeof(float);
  return weights > sums ? weights : sums;
}

}  // namespace

// What either kernel asks of a layer of up to `most` channels in.
static bool brief_layer(const GmsArgs &a, const Plan *p, int most) {
  if (a.dtype != FGMS_F16 || a.transpose_w || a.prepacked || a.dense_k >= 0 || a.n_pairs == 0 || a.n_dst == 0 || kernel_policy() != 0 || !raw_weights_enabled()) return false;
  if (!p || !p->groups.empty() || !p->has_tables || !p->fwd_ok || a.k_vol != p->k_vol || a.n_dst != p->n_out || a.n_src != p->n_in) return false;
  if (a.c_in % 8 || a.c_in < 16 || a.c_in > most || a.c_out % 8 || a.c_out < 16 || a.k_vol > kBriefOffsets) return false;
  if (reinterpret_cast<uintptr_t>(a.w) % 16 || reinterpret_cast<uintptr_t>(a.src) % 16 || reinterpret_cast<uintptr_t>(a.dst) % 4) return false;
  return (size_t)a.n_src * a.c_in * sizeof(__half) <= kMaxBufferBytes && (size_t)a.k_vol * a.c_in * a.c_out * sizeof(__half) <= kMaxBufferBytes;
}

static BriefArgs brief_args(const GmsArgs &a, const Plan *p) {
  BriefArgs b{};
  b.src = (const __half *)a.src;
  b.w = (const __half *)a.w;
  b.dst = (__half *)a.dst;
  b.nbr = p->nbr_out;
  b.perm = p->perm_out;
  b.block_masks = p->mask_out;
  b.centre = a.centre ? 1ull << (a.centre - 1) : 0;
  b.n_dst = (int)a.n_dst;
  b.k_vol = a.k_vol;
  b.c_src = a.c_in;
  b.c_dst = a.c_out;
  b.overwrite = a.overwrite ? 1 : 0;
  b.flip = p->flip_out;
  b.src_bytes = (unsigned)((size_t)a.n_src * a.c_in * sizeof(__half));
  b.w_bytes = (unsigned)((size_t)a.k_vol * a.c_in * a.c_out * sizeof(__half));
  b.side = a.side;
  if (!b.side.kind) (void)plan_take_check(p, &b.side);
  return b;
}

// Up to 32 channels two workgroups share a CU (64 KB of LDS each), and two rounds of them are faster than one of the kernels that bring
// the weights once for 128 or 256 rows; above, one and a half rounds of one (110 KB).  The others / this, us, indoor and scattered voxels:
// 32 -> 32 over 2 k 10.3 / 6.3 and 9.9 / 6.5, 16 k 10.5 / 6.5 and 9.8 / 6.5, 32 k (1 000 tiles) 10.4 / 8.8 and 10.5 / 8.6; 32 -> 64 over 16 k (1 000)
// 11.7 / 9.6 and 11.1 / 9.3, 24 k (1 500) 12.0 / 12.9 and 12.1 / 12.3; 24 -> 24 over 8 k 10.7 / 6.7 and 16.7 / 6.5; 16 -> 32 over 32 k 9.6 / 7.1;
// 64 -> 64 over 2 k 12.4 / 6.7 and 10.0 / 6.6, 4 k (250) 12.5 / 8.2 and 10.0 / 7.6, 6 k (376) 12.5 / 10.3, 8 k (500) 12.5 / 12.1 and 9.9 / 11.1;
// 48 -> 48 over 4 k 11.9 / 7.1 and 17.6 / 7.0; 64 -> 128 over 2 k (252) 12.5 / 8.2 and 10.5 / 7.6.
bool brief_gms_pays(const GmsArgs &a, const Plan *p) {
  if (!brief_layer(a, p, 64) || a.k_vol <= kBriefWaves || !half_tiles_enabled()) return false;
  const int64_t tiles = (a.n_dst + kBriefRows - 1) / kBriefRows * ((a.c_out + 31) / 32);
  return 2 * tiles <= (int64_t)num_cus() * (brief_lds(a) <= 80 << 10 ? 8 : 3);
}

int launch_brief_gms(const GmsArgs &a, const Plan *p) {
  const BriefArgs b = brief_args(a, p);
  const int S = brief_steps(a);
  auto kern = S == 1 ? gms_brief_kernel<1> : S == 2 ? gms_brief_kernel<2> : S == 3 ? gms_brief_kernel<3> : gms_brief_kernel<4>;
  const size_t lds = brief_lds(a);
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
  if (rc != FGMS_OK) return rc;
  {
    ProfileScope prof("gms_brief_kernel", a.stream);
    kern<<<dim3((unsigned)((a.n_dst + kBriefRows - 1) / kBriefRows) + (unsigned)b.side.blocks, (unsigned)((a.c_out + 31) / 32)), kBriefWaves * 64, lds, a.stream>>>(b);
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

// (The output-stationary, pair-view, first-layer or vector-ALU kernel that took the layer / this, us, indoor or scattered and LiDAR voxels in scan
// order: 32 -> 32 over 35 k 10.7 / 10.3 and 11.2 / 10.4, 60 k 12.1 / 10.5 and 14.2 / 11.3, 100 k 17.3 / 12.3 and 20.0 / 15.9, 130 k 19.2 / 14.0
// and 22.2 / 19.6, 200 k, where some workgroups wait for a second round, 22.6 / 22.2 and 28.3 / 28.9; 16 -> 32 over 60 k 10.1 / 7.6 and 10.6 / 8.0,
// 200 k 27.7 / 15.6 and 32.4 / 21.0; 32 -> 16 over 60 k 21.7 / 10.4 and 25.4 / 11.0, 200 k 50.1 / 21.4 and 57.1 / 27.8; 16 -> 16 over 100 k 11.4 / 8.1 and
// 14.9 / 11.7.  More than 32 columns gather their rows twice: 16 -> 48 over 60 k 13.5 / 11.0, 200 k 37.9 / 26.5; 16 -> 64 over 30 k 10.7 / 8.3, 100 k
// 17.1 / 14.7 and 20.3 / 19.4, 200 k 22.2 / 27.3, added to a result over 100 k 20.2 / 16.7 and 21.1 / 20.1, 120 k 21.5 / 20.8 and 22.4 / 24.9;
// 32 -> 64 over 30 k 12.2 / 11.7, 60 k 14.5 / 17.1.)
bool held_gms_pays(const GmsArgs &a, const Plan *p) {
  if (!brief_layer(a, p, 32) || a.c_out > 64 || a.k_vol <= 8) return false;
  const int64_t workgroups = (a.n_dst + kHeldWaves * 32 - 1) / (kHeldWaves * 32) * ((a.c_out + 31) / 32);
  if (a.c_in <= 16) return a.c_out <= 48 || 2 * workgroups <= (a.overwrite ? 8 : 7) * (int64_t)num_cus();
  return a.c_out <= 16 || (a.c_out <= 32 && workgroups <= 2 * (int64_t)num_cus());
}

int launch_held_gms(const GmsArgs &a, const Plan *p) {
  const BriefArgs b = brief_args(a, p);
  auto kern = brief_steps(a) == 1 ? gms_held_kernel<1> : gms_held_kernel<2>;
  const size_t lds = (size_t)(a.k_vol + kHeldWaves) * brief_steps(a) * 1024;
  const int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds);
  if (rc != FGMS_OK) return rc;
  // (without the plan's table a multiple of eight: the two workgroups of a tile of 64 columns write halves of the same lines, and belong on the
  // same XCD)
  const unsigned tiles = p->tile_out ? (unsigned)p->tile_grid_out : (unsigned)((a.n_dst + kHeldWaves * 32 - 1) / (kHeldWaves * 32) + 7) / 8 * 8;
  {
    ProfileScope prof("gms_held_kernel", a.stream);
    kern<<<dim3(tiles + (unsigned)b.side.blocks, (unsigned)((a.c_out + 31) / 32)), kHeldWaves * 64, lds, a.stream>>>(b, p->tile_out);
  }
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

}  // namespace fgms
