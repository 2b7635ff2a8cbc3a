// Zeros in the part of an output that no group owns: the rows (2D x 3D) or columns (3D x 2D) past the largest offset.  A
// gradient has to hold zeros there, and clearing the whole matrix first wrote it twice: 32768 x 2048 bf16 18.5 us, nearly
// always for nothing, since the offsets usually end at the extent.  Here the workgroups read the offsets and leave (4.7 us).
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

// lines x width elements from `out`, `ld` and `step` elements apart; T: the element's size.
template <typename T>
__global__ void __launch_bounds__(NT) zero_unowned_kernel(const GmmParams p) {
  __shared__ int shared[NT / 64];
  const bool rows = p.jag == GMM_JAG_M;
  const int end = owned_end(p, rows ? p.M : p.N, shared);
  if (end == (rows ? p.M : p.N)) return;
  T* const out = static_cast<T*>(p.c);
  const int64_t first = int64_t(blockIdx.x) * NT + threadIdx.x, stride = int64_t(gridDim.x) * NT;
  if (rows && p.c_sn == 1 && p.c_sm == p.N) {
    // whole rows of a contiguous matrix: 16 bytes at a time between the ends
    constexpr int64_t PER = 16 / sizeof(T);
    const int64_t lo = int64_t(end) * p.N, hi = int64_t(p.M) * p.N;
    const int64_t skew = (reinterpret_cast<uintptr_t>(out + lo) & 15) / sizeof(T);
    const int64_t body = gmm_min(int(hi - lo < PER ? hi - lo : PER), int(skew ? PER - skew : 0)) + lo;
    const int64_t chunks = (hi - body) / PER;
    for (int64_t i = first; i < chunks; i += stride) *reinterpret_cast<uint4*>(out + body + i * PER) = make_uint4(0, 0, 0, 0);
    if (first < body - lo) out[lo + first] = T(0);
    if (first < hi - body - chunks * PER) out[body + chunks * PER + first] = T(0);
    return;
  }
  const int64_t width = rows ? p.N : p.N - end, total = (rows ? p.M - end : p.M) * width;
  for (int64_t i = first; i < total; i += stride) {
    const int64_t r = i / width, c = i - r * width;
    out[(rows ? end + r : r) * p.c_sm + (rows ? c : end + c) * p.c_sn] = T(0);
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
