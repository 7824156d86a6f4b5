// Channel counts that no tuned kernel takes (3 or 5 input features, 20 classes) are widened to the next ones that
// a tuned kernel takes: zero-padded copies of the rows and of the weights, results cropped on their way back.
// The padding channels are zero in both operands of every product, so the results are those of the original shape.
//
// Not all of them: counts that are multiples of 8 (24, 48, 56) run without copies on dense maps, where the MFMA
// kernels mask the rest of a tile themselves (48 -> 48 fp16 over 80 k voxels, forward and backward, 100.7 us over copies,
// 64.6 without), fp16 output layers of 20 and 28 channels too (96 -> 20 over 60 k 77.5, 69.2 without), first layers of 1 to 8 channels have kernels of their own, and small fp32 calls stay on the vector ALUs, which take any count (padding_pays).
//
// Bound by memory: a copy reads n * c and writes n * c_padded elements once, 16 bytes per thread,
// where the shape-agnostic kernels spend a scalar atomic per result element: 96 -> 20 fp16 over
// 60 k voxels, forward and backward, 2378 us there and 78 us over copies.
#include "fgms_device.h"
#include "fgms_internal.h"

namespace fgms {
namespace {

// dst[o][rp][cp] (rp < r_to, cp < c_to) = src[o][rp][cp] inside [r][c], else 0; src == nullptr: all
// zeros.  c_to is a multiple of the V elements of a thread's store.
template <typename U, int V>
__device__ __forceinline__ void pad_chunk(const PadJob &job, size_t i) {
  typedef U vec __attribute__((ext_vector_type(V)));
  const int per_row = job.c_to / V;
  const size_t row = i / per_row;
  const int c0 = (int)(i % per_row) * V;
  vec v = 0;
  if (job.src) {
    size_t from_row = row;
    bool inside = true;
    if (job.r != job.r_to) {
      const size_t o = row / job.r_to;
      const int rr = (int)(row % job.r_to);
      inside = rr < job.r;
      from_row = o * job.r + rr;
    }
    const U *from = (const U *)job.src + from_row * job.c + c0;
    if (inside) {
      if (job.whole) {             // rows of whole chunks: a chunk is all data or all padding
        if (c0 < job.c) v = *reinterpret_cast<const vec *>(from);
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e)
          if (c0 + e < job.c) v[e] = from[e];
      }
    }
  }
  reinterpret_cast<vec *>(job.dst)[i] = v;
}

// All copies of a call in one launch (a launch in a chain of small ones costs 4 us whatever it does).
template <typename U>
__global__ __launch_bounds__(256) void pad_kernel(PadBatch batch) {
  int q = 0;
  while (q + 1 < batch.count && (int)blockIdx.x >= batch.job[q + 1].first_block) ++q;
  const PadJob &job = batch.job[q];
  const size_t stride = (size_t)job.blocks * 256;
  for (size_t i = (size_t)(blockIdx.x - job.first_block) * 256 + threadIdx.x; i < job.chunks; i += stride) {
    if (job.wide) pad_chunk<U, 16 / (int)sizeof(U)>(job, i);
    else pad_chunk<U, 4>(job, i);      // four halfs: the narrowest padded row
  }
}

// dst[row][0 .. c) += (overwrite: =) src[row][0 .. c), rows of c_from elements in src.
template <typename T>
__global__ __launch_bounds__(256) void crop_kernel(const T *__restrict__ src, T *__restrict__ dst, size_t n, int c, int c_from,
                                                   bool overwrite) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const float v = (float)src[i / c * c_from + i % c];
    dst[i] = (T)(overwrite ? v : (float)dst[i] + v);
  }
}

// The weight gradient's fp32 sums [k][r_from][c_from] -> dst[k][r][c] += (overwrite: =), rounded once; the sums
// are all zero afterwards, padding included (a product with an infinite operand leaves NaN there).
template <typename T>
__global__ __launch_bounds__(256) void crop_sums_kernel(float *__restrict__ sums, T *__restrict__ dst, size_t n, int r,
                                                        int r_from, int c, int c_from, bool overwrite) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const int cc = (int)(i % c_from);
    const size_t row = i / c_from;
    const int rr = (int)(row % r_from);
    if (cc < c && rr < r) {
      T *d = dst + (row / r_from * r + rr) * c + cc;
      *d = (T)(overwrite ? sums[i] : (float)*d + sums[i]);
    }
    sums[i] = 0.f;
  }
}

unsigned grid_for(size_t n) {
  const size_t blocks = (n + 255) / 256;
  return (unsigned)(blocks > 16384 ? 16384 : blocks);
}

}  // namespace

void PadBatch::add(const void *src, void *dst, size_t outer, int r, int r_to, int c, int c_to, int esz) {
  PadJob &j = job[count];
  j.src = src;
  j.dst = dst;
  j.r = r; j.r_to = r_to; j.c = c; j.c_to = c_to;
  const int v = 16 / esz;
  j.wide = c_to % v == 0;
  j.whole = j.wide && c % v == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0;
  j.chunks = outer * r_to * c_to / (j.wide ? v : 4);
  if (j.chunks == 0) return;
  j.first_block = total_blocks;
  j.blocks = (int)grid_for(j.chunks);
  total_blocks += j.blocks;
  ++count;
}

int launch_pad(const PadBatch &batch, int dtype, hipStream_t s) {
  if (batch.count == 0) return FGMS_OK;
  if (dtype == FGMS_F16) pad_kernel<unsigned short><<<(unsigned)batch.total_blocks, 256, 0, s>>>(batch);
  else pad_kernel<unsigned><<<(unsigned)batch.total_blocks, 256, 0, s>>>(batch);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

int launch_crop(const void *src, void *dst, size_t rows, int c, int c_from, bool overwrite, int dtype, hipStream_t s) {
  const size_t n = rows * c;
  if (n == 0) return FGMS_OK;
  if (dtype == FGMS_F16)
    crop_kernel<_Float16><<<grid_for(n), 256, 0, s>>>((const _Float16 *)src, (_Float16 *)dst, n, c, c_from, overwrite);
  else
    crop_kernel<float><<<grid_for(n), 256, 0, s>>>((const float *)src, (float *)dst, n, c, c_from, overwrite);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

int launch_crop_sums(float *sums, void *dst, size_t k_vol, int r, int r_from, int c, int c_from, bool overwrite, int dtype,
                     hipStream_t s) {
  const size_t n = k_vol * r_from * c_from;
  if (dtype == FGMS_F16)
    crop_sums_kernel<_Float16><<<grid_for(n), 256, 0, s>>>(sums, (_Float16 *)dst, n, r, r_from, c, c_from, overwrite);
  else
    crop_sums_kernel<float><<<grid_for(n), 256, 0, s>>>(sums, (float *)dst, n, r, r_from, c, c_from, overwrite);
  FGMS_HIP_TRY(hipGetLastError());
  return FGMS_OK;
}

}  // namespace fgms
