// Zeros in the part of an output that no group owns: the rows (2D x 3D) or columns (3D x 2D) past the largest offset.  A
// gradient has to hold zeros there, and clearing the whole matrix first wrote it twice: 32768 x 2048 bf16 18.5 us, nearly
// always for nothing, since the offsets usually end at the extent.  Here the workgroups read the offsets and leave (4.8 us).
#include "gmm_device.h"
#include "gmm_launch.h"

namespace {

constexpr int NT = 256;

// Groups follow each other, so what they own starts at 0 and ends at the largest offset, also for offsets that go back.
__device__ __forceinline__ int owned_end(const GmmParams& p, int extent, int* shared) {
  int end = 0;
  for (int g = threadIdx.x; g < p.G; g += NT) end = gmm_max(end, p.offs[g]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) end = gmm_max(end, __shfl_xor(end, o));
  if ((threadIdx.x & 63) == 0) shared[threadIdx.x >> 6] = end;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) end = gmm_max(end, shared[w]);
  return gmm_min(end, extent);
}

// Zeros in `lines` runs of `len` elements each, `pitch` elements apart: 16 bytes per thread, aligned wherever a run starts, the
// chunks that a run's ends cut element by element.  A run of up to 256 chunks takes as many threads as the next power of two, a
// longer one whole workgroups, piece by piece.  Columns were cleared element by element, with a division each: a training step
// of 4 groups, 512 x 131072 to 256, whose groups own half of the 131072, 263 us, with this 228 (all of the gradient cleared first
// 233).
template <typename T>
__device__ __forceinline__ void zero_runs(T* first, int64_t lines, int64_t pitch, int64_t len) {
  const int64_t chunks = len * int(sizeof(T)) / 16 + 2;      // at most: both ends cut
  const int shift = chunks > NT / 2 ? 8 : 32 - __clz(int(chunks) - 1);
  const int64_t pieces = chunks > NT ? (chunks + NT - 1) / NT : 1;
  const int at_once = NT >> shift, tid = threadIdx.x;
  const int64_t items = (lines + at_once - 1) / at_once * pieces;
  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    const int64_t set = pieces == 1 ? item : item / pieces, piece = item - set * pieces;
    const int64_t line = set * at_once + (tid >> shift);
    if (line >= lines) continue;
    const uintptr_t lo = reinterpret_cast<uintptr_t>(first + line * pitch), hi = lo + len * sizeof(T);
    const uintptr_t chunk = (lo & ~uintptr_t(15)) + (piece * NT + (tid & ((1 << shift) - 1))) * 16;
    if (chunk >= hi) continue;
    if (chunk >= lo && chunk + 16 <= hi) {
      *reinterpret_cast<uint4*>(chunk) = make_uint4(0, 0, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < 16 / int(sizeof(T)); ++i) {
        T* const e = reinterpret_cast<T*>(chunk) + i;
        if (reinterpret_cast<uintptr_t>(e) >= lo && reinterpret_cast<uintptr_t>(e) < hi) *e = T(0);
      }
    }
  }
}

// T: an unsigned type of the element's size.
template <typename T>
__global__ void __launch_bounds__(NT) zero_unowned_kernel(const GmmParams p) {
  __shared__ int shared[NT / 64];
  const bool rows = p.jag == GMM_JAG_M;
  const int extent = rows ? p.M : p.N, end = owned_end(p, extent, shared);
  if (end == extent) return;
  // the jagged dimension's rest x all of the other one
  const int64_t rest = extent - end, other = rows ? p.N : p.M;
  const int64_t s_rest = rows ? p.c_sm : p.c_sn, s_other = rows ? p.c_sn : p.c_sm;
  T* const out = static_cast<T*>(p.c) + end * s_rest;
  if (s_other == 1 && s_rest == other) {
    zero_runs(out, 1, 0, rest * other);
  } else if (s_other == 1) {
    zero_runs(out, rest, s_rest, other);
  } else if (s_rest == 1) {
    zero_runs(out, other, s_other, rest);
  } else {
    const int64_t total = rest * other, stride = int64_t(gridDim.x) * NT;
    for (int64_t i = int64_t(blockIdx.x) * NT + threadIdx.x; i < total; i += stride) {
      const int64_t r = i / other;
      out[r * s_rest + (i - r * other) * s_other] = T(0);
    }
  }
}

}  // namespace

int gmm_launch_zero_unowned(const GmmParams& p, int out_dtype, hipStream_t stream) {
  const int64_t elements = int64_t(p.M) * p.N;
  const int64_t want = (elements / 8 + NT - 1) / NT;
  const dim3 grid(unsigned(want < 1 ? 1 : want > 512 ? 512 : want)), block(NT);
  if (out_dtype == GMM_DT_F32) hipLaunchKernelGGL(zero_unowned_kernel<uint32_t>, grid, block, 0, stream, p);
  else hipLaunchKernelGGL(zero_unowned_kernel<uint16_t>, grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}
