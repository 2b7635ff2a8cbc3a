// Register-staged MFMA grouped GEMM for operands of any alignment: bf16, fp16 and fp32, each operand contiguous
// along K or along M / N, any leading dimension, any base address, with or without a row gather.
//
// What it replaces and why.  Operands that the assembly tile cannot take (an extent or a leading dimension that is
// not a multiple of 8 elements, fp32) went element by element: one 2- or 4-byte load, one bounds check and one 64-bit
// address per element, fp32 products whatever the type.  gfx950 loads 16 bytes from any address that is a multiple of
// the element size (measured: 29 us against 27 us aligned), so nothing has to go element by element but an operand's
// last chunk.  Before and after, us: bf16 8191 x 2047 x 2047 in 8 groups 2291 -> 153 (450 TFLOP/s), 6151 x 1031 x 519
// in 24 groups 472 -> 36, its weight gradient 437 -> 45; fp32 8192 x 1024 x 4096 920 -> 592 (116 TFLOP/s of 157),
// 1024 x 1024 x 8192 columns in 8 groups 330 -> 166.
//
//   * A K tile is 128 bytes of K per row (64 bf16 / fp16, 32 fp32): every thread carries its 16-byte chunks of the
//     next K tile in registers while the MFMAs of the present one run out of LDS (two buffers, one barrier per K
//     tile); two or four workgroups share a CU, so one computes while another stores, fetches or starts up.  fp32
//     fetches two K tiles ahead (5 % on large problems); for 16-bit operands a second one in flight gained nothing:
//     small problems are bound by start-up, which more code makes longer, large ones by the LDS.
//   * Operand contiguous along K: LDS [row][128 bytes], 16-byte chunk index XOR (row >> 1) & 7, a fragment (16 rows,
//     8 or 4 consecutive k per lane) is one ds_read_b128.  Operand contiguous along M / N: LDS [k][rows] as it comes
//     from memory; 16-bit fragments are two transposing ds_read_b64_tr_b16 (k rows 4 .. 7 and 8 .. 11 of 16 swap
//     places so that the 32 lanes served together hit all 64 banks once), fp32 fragments are four ds_read_b32.
//   * v_mfma_f32_16x16x32_{bf16,f16} / v_mfma_f32_16x16x4_f32, fp32 accumulators, one rounding.  Operands swapped, so
//     that a lane owns 4 consecutive columns; a wave stages 16 rows at a time in LDS and stores 16 bytes per lane in
//     whole rows.
//   * Loads never leave the operand: rows and columns past the extent are clamped (their products are not stored); K
//     tiles that are cut by the end of the group's range, or whose chunks touch the operand's last bytes, are fetched
//     with a check per chunk, without branches, in a loop of their own.
//   * What bounds it: 16-bit, 4 x 4 blocks per wave: LDS reads and writes take 1.5 times the cycles of the MFMAs; fp32:
//     the MFMA pipe (64 to 75 % busy), the rest is the last, partly filled round.
#include <cmath>

#include "gmm_device.h"
#include "gmm_launch.h"

namespace {

constexpr int NT = 256;            // threads: 2 x 2 waves
constexpr int ROW_BYTES = 128;     // bytes of K per row and K tile

// Workgroups per CU: what the LDS images (64 to 72 KB, 33 to 35 KB) and the registers allow.
constexpr int tile_wgs(int edge) { return edge == 128 ? 2 : 4; }

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4_ptr;

// 16 bytes from an address that is a multiple of the element size only (one global_load_dwordx4).
template <typename T>
__device__ __forceinline__ uint4 load16(const T* p) {
  uint4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// Elements [0, n) of the chunk at p, zeros behind them, without a branch and without reading at or past `end`: a chunk
// that would cross it is fetched from `last` (the operand's last 16 bytes) and shifted down.  p may lie anywhere if
// n <= 0.
template <typename T>
__device__ __forceinline__ uint4 load_part(const T* p, const T* last, int n) {
  constexpr int EPC = 16 / int(sizeof(T));
  const bool cross = p > last || n <= 0;
  uint4 v = load16(cross ? last : p);
  const int shift = cross ? int(p - last) : 0;           // elements; only looked at when n > 0
  if (__ballot(n > 0 && shift > 0)) {
    // rare (the operand's very last chunk): a loop over single elements.  Steps of 4, 2 and 1 elements are faster where it runs
    // (3 products of 726 x 14 x 1 1 us of 10), but make the code longer and every other launch 0.2 us slower.
#pragma unroll 1
    for (int s = EPC - 1; s > 0; --s) {
      const bool go = s <= shift;
      uint4 w;
      if constexpr (sizeof(T) == 2)
        w = make_uint4(__builtin_amdgcn_alignbit(v.y, v.x, 16), __builtin_amdgcn_alignbit(v.z, v.y, 16),
                       __builtin_amdgcn_alignbit(v.w, v.z, 16), v.w >> 16);
      else
        w = make_uint4(v.y, v.z, v.w, 0u);
      v.x = go ? w.x : v.x; v.y = go ? w.y : v.y; v.z = go ? w.z : v.z; v.w = go ? w.w : v.w;
    }
  }
  uint32_t* w = &v.x;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 2)
      w[i] = n > 2 * i + 1 ? w[i] : n > 2 * i ? (w[i] & 0xffffu) : 0u;
    else
      w[i] = n > i ? w[i] : 0u;
  }
  return v;
}

// LDS image of one operand's K tile of ROWS rows (or columns).
template <typename T, bool TR, int ROWS>
struct Image {
  static constexpr int ESZ = int(sizeof(T));
  static constexpr int BK = ROW_BYTES / ESZ;
  static constexpr int PITCH = TR ? ROWS * ESZ + (ESZ == 2 ? 32 : 16) : ROW_BYTES;   // bytes between LDS rows
  static constexpr int BYTES = TR ? BK * PITCH : ROWS * ROW_BYTES;
  // transposed 16-bit image: k rows 4..7 and 8..11 of every 16 trade places
  static __device__ __forceinline__ int slot(int k) { return ESZ == 2 ? (k & ~12) | ((k & 4) << 1) | ((k & 8) >> 1) : k; }
};

// Global -> registers -> LDS of one operand: NCH 16-byte chunks per thread and K tile.
template <typename T, bool TR, int ROWS>
struct Stage {
  using Im = Image<T, TR, ROWS>;
  static constexpr int EPC = 16 / Im::ESZ;             // elements of a chunk
  static constexpr int CPR = TR ? ROWS / EPC : 8;      // chunks per LDS row
  static constexpr int NCH = ROWS * 8 / NT;
  const T* ptr[NCH];                                   // the thread's chunks of K tile 0
  const T* last;                                       // the operand's last 16 bytes
  int64_t step;                                        // elements from one K tile to the next
  int zero_rows;                                       // bit i: chunk i belongs to a gathered row that does not exist
  int any_zero;                                        // some lane of the wave has one
  int n_fast;                                          // K tiles that need no check

  // base: element (row 0, k 0) of the group's operand; the tile's rows start at row0; `ext` rows exist.
  __device__ __forceinline__ void init(const T* base, int64_t ld, int row0, int ext, int k_lo, int k_hi, int k_ext,
                                       const int32_t* gather, int gather_end, int src_rows) {
    const int tid = threadIdx.x;
    zero_rows = 0;
    const int whole = (k_hi - k_lo) / Im::BK;          // K tiles that lie inside the range
    if constexpr (!TR) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int q = i * NT + tid, row = q >> 3, c = q & 7;
        int src = gmm_min(row0 + row, ext - 1);
        if (gather) {
          src = row0 + row < gather_end ? gather[row0 + row] : -1;
          if (src < 0 || src >= src_rows) { zero_rows |= 1 << i; src = 0; }
        }
        ptr[i] = base + int64_t(src) * ld + k_lo + c * EPC;
      }
      any_zero = gather ? __ballot(zero_rows != 0) != 0 : 0;
      last = base + int64_t((gather ? src_rows : ext) - 1) * ld + k_ext - EPC;
      step = Im::BK;
      n_fast = whole;
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int q = i * NT + tid, k = q / CPR, c = q % CPR;
        const int col = row0 + c * EPC;
        ptr[i] = base + int64_t(k_lo + k) * ld + (col < ext ? col : row0);
      }
      last = base + int64_t(k_ext - 1) * ld + ext - EPC;
      step = int64_t(Im::BK) * ld;
      // the last chunk of a row may reach past the extent, into the next k row: fine as long as there is one
      const int over = row0 + gmm_min(ROWS, (ext - row0 + EPC - 1) / EPC * EPC) - ext;
      const int slack = over > 0 ? int((over + ld - 1) / ld) : 0;
      const int safe = gmm_min(k_hi, k_ext - slack) - k_lo;
      n_fast = safe > 0 ? safe / Im::BK : 0;
    }
  }

  __device__ __forceinline__ void load_fast(uint4 (&r)[NCH], int t) const {
#pragma unroll
    for (int i = 0; i < NCH; ++i) r[i] = load16(ptr[i] + int64_t(t) * step);
  }

  // the same for a K tile that needs checks; k_left = k elements of the range from K tile t on
  __device__ __forceinline__ void load_checked(uint4 (&r)[NCH], int t, int k_left) const {
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int q = i * NT + tid;
      const int n = TR ? (q / CPR < k_left ? EPC : 0) : k_left - (q & 7) * EPC;
      r[i] = load_part<T>(ptr[i] + int64_t(t) * step, last, n);
    }
  }

  __device__ __forceinline__ void store(uint4 (&r)[NCH], char* image) const {
    const int tid = threadIdx.x;
    if (!TR && __builtin_amdgcn_readfirstlane(any_zero)) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) r[i] = (zero_rows & (1 << i)) ? make_uint4(0, 0, 0, 0) : r[i];
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int q = i * NT + tid;
      int at;
      if constexpr (!TR) {
        const int row = q >> 3, c = q & 7;
        at = row * ROW_BYTES + ((c ^ ((row >> 1) & 7)) << 4);
      } else {
        at = Im::slot(q / CPR) * Im::PITCH + (q % CPR) * 16;
      }
      *reinterpret_cast<uint4*>(image + at) = r[i];
    }
  }
};

// Fragment of 16 rows starting at `row0` and k half `half` of a K tile: lane l holds row l % 16, the k elements of
// 16-byte chunk 4 * half + l / 16.
template <typename T, bool TR, int ROWS>
__device__ __forceinline__ uint4 read_fragment(const char* image, int row0, int half, int lane) {
  using Im = Image<T, TR, ROWS>;
  const int q = lane >> 4, ii = lane & 15;
  if constexpr (!TR) {
    const int row = row0 + ii;
    return *reinterpret_cast<const uint4*>(image + row * ROW_BYTES + (((4 * half + q) ^ ((row >> 1) & 7)) << 4));
  } else if constexpr (Im::ESZ == 2) {
    // k = 32 half + 8 q + 0..3 and + 4..7; each group of 16 lanes reads 4 k rows x 16 columns, transposed
    const int s0 = 32 * half + 16 * (q >> 1) + 4 * (q & 1) + (ii >> 2);
    const char* p = image + s0 * Im::PITCH + (row0 + 4 * (ii & 3)) * 2;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 8 * Im::PITCH));
    uint4 v;
    __builtin_memcpy(&v.x, &lo, 8);
    __builtin_memcpy(&v.z, &hi, 8);
    return v;
  } else {
    const char* p = image + (16 * half + 4 * q) * Im::PITCH + (row0 + ii) * 4;
    uint4 v;
    v.x = *reinterpret_cast<const uint32_t*>(p);
    v.y = *reinterpret_cast<const uint32_t*>(p + Im::PITCH);
    v.z = *reinterpret_cast<const uint32_t*>(p + 2 * Im::PITCH);
    v.w = *reinterpret_cast<const uint32_t*>(p + 3 * Im::PITCH);
    return v;
  }
}

// acc += first operand's fragments x second operand's; operands swapped, so that a lane owns 4 consecutive columns.
template <typename T, int TM, int TN>
__device__ __forceinline__ void multiply(const uint4 (&a)[TM], const uint4 (&b)[TN], f32x4 (&acc)[TM][TN]) {
  if constexpr (sizeof(T) == 4) {
    // element e of every lane's chunk is one k of four: no two MFMAs in a row add to the same accumulator
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const uint32_t x = e == 0 ? a[i].x : e == 1 ? a[i].y : e == 2 ? a[i].z : a[i].w;
          const uint32_t y = e == 0 ? b[j].x : e == 1 ? b[j].y : e == 2 ? b[j].z : b[j].w;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(y), __uint_as_float(x), acc[i][j], 0, 0, 0);
        }
  } else {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if constexpr (__is_same(T, gmm_f16)) {
          f16x8 x, y;
          __builtin_memcpy(&x, &a[i], 16);
          __builtin_memcpy(&y, &b[j], 16);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(y, x, acc[i][j], 0, 0, 0);
        } else {
          bf16x8 x, y;
          __builtin_memcpy(&x, &a[i], 16);
          __builtin_memcpy(&y, &b[j], 16);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(y, x, acc[i][j], 0, 0, 0);
        }
      }
  }
}

// ---- jagged contractions cut along K ---------------------------------------------------------------- //
// A weight gradient of small matrices has few tiles and a contraction as long as the group: 64 groups of 32 x 64 with 2048
// elements each are 64 tiles, two groups of 88 x 48 over 64920 elements two.  A group longer than p.k_chunk is cut into
// parts (gmm_group_parts); a tile of a part is an entry of the tile list like any other, number `id`, and leaves its
// accumulators in slot `id` of the workspace as they lie in the registers.  Up to GMM_K_CLUSTER neighbouring parts form a
// cluster: the part that finds all others of its cluster there adds the slots in the order of the parts, and so, one level
// up, does the cluster that comes last.  The sum does not depend on timing, and nobody waits.  Counters (word `id` of the
// workspace's header: of the cluster's first part for the cluster, of the tile's second part for the tile) are left
// at zero.  A part's tiles are neighbours in the list, so that what they share of A and B is read together.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <int TM, int TN, int EDGE>
struct Partial {
  static constexpr int SLOT = EDGE * EDGE * 4;
  __amdgpu_buffer_rsrc_t slots;
  int rows, cols;    // 16 x 16 blocks of the wave that hold something

  __device__ __forceinline__ Partial(const GmmParams& p, const GmmTile& tile, int wm, int wn) {
    slots = __builtin_amdgcn_make_buffer_rsrc(static_cast<char*>(p.ws) + GMM_WS_HEADER, 0, 0x7fffffff, 0x00020000);
    rows = gmm_min(gmm_max(gmm_cdiv(tile.m_hi - tile.m0 - wm, 16), 0), TM);
    cols = gmm_min(gmm_max(gmm_cdiv(tile.n_hi - tile.n0 - wn, 16), 0), TN);
  }
  static __device__ __forceinline__ int at(int slot, int i, int j) {
    return slot * SLOT + ((i * TN + j) * NT + int(threadIdx.x)) * 16;
  }
  // Stored through to memory at device scope and read past this XCD's L2 (sc1).
  __device__ __forceinline__ void store(const f32x4 (&acc)[TM][TN], int slot) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        u32x4 v;
        __builtin_memcpy(&v, &acc[i][j], 16);
        if (i < rows && j < cols) __builtin_amdgcn_raw_buffer_store_b128(v, slots, at(slot, i, j), 0, 16 /* sc1 */);
      }
  }
  // acc = sum of n slots `stride` apart.
  __device__ __forceinline__ void add(f32x4 (&acc)[TM][TN], int slot, int stride, int n) const {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int x = 0; x < n; ++x) {
      u32x4 v[TM][TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          v[i][j] = u32x4{0u, 0u, 0u, 0u};
          if (i < rows && j < cols) v[i][j] = __builtin_amdgcn_raw_buffer_load_b128(slots, at(slot + x * stride, i, j), 0, 16 /* sc1 */);
        }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          f32x4 f;
          __builtin_memcpy(&f, &v[i][j], 16);
          acc[i][j] += f;
        }
    }
  }
};

// Count this workgroup in on counter `word`; true in all threads of the one that completes `n`.  Everything that the
// workgroup stored before is visible to the device by then.
__device__ __forceinline__ bool arrive(const GmmParams& p, int word, int n, int* flag) {
  unsigned* const counter = static_cast<unsigned*>(p.ws) + word;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == unsigned(n - 1);
    if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last ? 1 : 0;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

// Part `part` of `parts` of a tile whose first part is entry `id0` of the list and whose parts are `per` entries apart.
// True if acc now holds the whole tile.
template <int TM, int TN, int EDGE>
__device__ __forceinline__ bool join_parts(const GmmParams& p, const GmmTile& tile, f32x4 (&acc)[TM][TN], int wm, int wn,
                                           int id0, int per, int part, int parts, int* flag) {
  const Partial<TM, TN, EDGE> partial(p, tile, wm, wn);
  const int first = part / GMM_K_CLUSTER * GMM_K_CLUSTER, in_cluster = gmm_min(GMM_K_CLUSTER, parts - first);
  const int clusters = gmm_cdiv(parts, GMM_K_CLUSTER);
  partial.store(acc, id0 + part * per);
  if (!arrive(p, id0 + first * per, in_cluster, flag)) return false;
  partial.add(acc, id0 + first * per, per, in_cluster);
  if (clusters == 1) return true;
  partial.store(acc, id0 + first * per);
  if (!arrive(p, id0 + per, clusters, flag)) return false;
  partial.add(acc, id0, GMM_K_CLUSTER * per, clusters);
  return true;
}

// Parts of each of the `tail` tiles of a last, partly filled round behind `whole` tiles on `wgs` workgroups: as many as there are
// places for, and behind whole rounds only if that makes four of each.  Places: the workgroups.  Of 128 x 128 tiles half of them, one
// to a compute unit, where that is enough for four parts of each: a second part on a unit slows the first, and each is stored and
// read again.  us uncut / one part to a unit / two: a last round of 64 tiles of 2047 x 1667 (31 groups, 2247 columns) 82.1 / 64.6 /
// 82.1, 48 of 2255 100 / 76 / 85; 1024 x 1024 x 2304 on 64 tiles 26.8 on the assembly tile / 25.7 / 38.2.  Where they alone make the
// launch, parts past k_alone elements are better on two, full tiles later (1024 x 1024 x 5000, 64 tiles with A contiguous along M 34 /
// 47) than those with few rows or columns (8 products of 64 x 1024 x 2560 22.0 / 24.1, x 4000 28.3 / 28.1, x 6144 35.6 / 32.7).  Behind whole rounds of 64 x 64 tiles, four of which share a CU's matrix cores, always half (a tile
// that is alone on its CU already runs three times as fast as in a full round).
__host__ __device__ inline int tail_parts(int tail, int whole, int wgs, int edge, const GmmParams& p) {
  if (tail == 0) return 1;
  const bool one_each = edge == 64 ? whole > 0 : 8 * tail <= wgs && (whole || int64_t(p.K) * tail <= int64_t(p.k_alone) * (wgs / 2));
  const int places = one_each ? wgs / 2 : wgs, room = places < p.k_parts ? places : p.k_parts;
  const int parts = room / tail < p.k_split ? room / tail : p.k_split;
  return parts < (whole ? 4 : 2) ? 1 : parts;
}

// SPLIT = 1: a jagged contraction whose groups may be cut along K.  SPLIT = 2: any other product, the tiles of the last round
// cut along K.
template <typename T, typename OutT, bool A_TR, bool B_TR, int EDGE, int SPLIT>
__global__ void __launch_bounds__(NT, tile_wgs(EDGE)) gmm_staged_kernel(const GmmParams p) {
  constexpr int BM = EDGE, BN = EDGE;
  constexpr int AHEAD = sizeof(T) == 4 ? 2 : 1;   // K tiles fetched ahead (see the top of the file)
  using ImA = Image<T, A_TR, BM>;
  using ImB = Image<T, B_TR, BN>;
  constexpr int BK = ImA::BK;
  constexpr int WTM = BM / 2, WTN = BN / 2, TM = WTM / 16, TN = WTN / 16;
  // epilogue: a wave stages 16 rows of its columns, padded by 16 bytes against bank conflicts
  constexpr int OSZ = int(sizeof(OutT)), OEC = 16 / OSZ;
  constexpr int EPITCH = WTN * OSZ + 16, ECPR = WTN * OSZ / 16;
  constexpr int PIPE = 2 * (ImA::BYTES + ImB::BYTES), EPI = 4 * 16 * EPITCH;
  __shared__ __attribute__((aligned(16))) char lds[PIPE > EPI ? PIPE : EPI];
  __shared__ int32_t cum[GMM_MAX_GROUPS + 1];
  __shared__ int flag;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave & 1) * WTM, wn = (wave >> 1) * WTN;
  const int64_t lda = A_TR ? p.a_sk : p.a_sm, ldb = B_TR ? p.b_sk : p.b_sn;
  const bool in_registers = p.jag != GMM_JAG_NONE && p.G <= 64;
  GmmWaveGroups groups{0, 0, 0, 0};
  int chunk = SPLIT == 1 ? p.k_chunk : 0;
  auto build = [&]() {
    return __builtin_amdgcn_readfirstlane(in_registers ? groups.build(p, BM, BN, chunk) : gmm_build_tile_table<NT>(p, BM, BN, cum, chunk));
  };
  int total = build();
  const int tail = SPLIT == 2 ? total % int(gridDim.x) : 0, whole = total - tail;
  const int split = SPLIT == 2 ? tail_parts(tail, whole, gridDim.x, EDGE, p) : 1;
  if (SPLIT == 2) total = whole + tail * split;
  if (SPLIT == 1 && chunk && total > p.k_parts) {   // offsets that overlap: more parts than K elements have room for
    chunk = 0;
    __syncthreads();
    total = build();
  }

  for (int t = blockIdx.x; t < total; t += gridDim.x) {
    int id = gmm_xcd_remap(t, total, gridDim.x);
    int g, local, lo, hi;
    int part = 0, parts = 1, per = 1, number = id;
    if (SPLIT == 2 && id >= whole) {
      per = tail;
      parts = split;
      id -= whole;
      part = id / tail;
      number = whole + id - part * tail;
    }
    if (in_registers) groups.find(number, g, local, lo, hi);
    else gmm_find_tile(p, cum, number, BM, BN, g, local, lo, hi);
    if (SPLIT == 1) {
      parts = gmm_group_parts(hi - lo, chunk);
      per = gmm_cdiv(p.M, BM) * gmm_cdiv(p.N, BN);
      part = local / per;
      local -= part * per;
    }
    GmmTile tile = gmm_tile_of_group(p, g, local, lo, hi, BM, BN);
    if (SPLIT && parts > 1) {
      const int k_lo = tile.k_lo, k_hi = tile.k_hi;
      int first, last;
      gmm_part_ktiles(gmm_cdiv(k_hi - k_lo, BK), parts, part, first, last);
      tile.k_lo = k_lo + first * BK;
      tile.k_hi = gmm_min(k_lo + last * BK, k_hi);
    }
    const T* a = static_cast<const T*>(p.a) + int64_t(tile.g) * p.a_sg;
    const T* b = static_cast<const T*>(p.b) + int64_t(tile.g) * p.b_sg;
    OutT* c = static_cast<OutT*>(p.c) + int64_t(tile.g) * p.c_sg;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int klen = tile.k_hi - tile.k_lo;
    if (klen > 0) {
      Stage<T, A_TR, BM> sa;
      Stage<T, B_TR, BN> sb;
      sa.init(a, lda, tile.m0, p.M, tile.k_lo, tile.k_hi, p.K, SPLIT == 1 ? nullptr : p.gather, tile.m_hi, p.a_rows);
      sb.init(b, ldb, tile.n0, p.N, tile.k_lo, tile.k_hi, p.K, nullptr, 0, 0);
      const int n_fast = gmm_min(sa.n_fast, sb.n_fast), nk = (klen + BK - 1) / BK;
      // K tile t + 1 .. t + AHEAD are on their way in registers while K tile t is multiplied
      uint4 ra[AHEAD][sa.NCH], rb[AHEAD][sb.NCH];
      auto load = [&](int t, int set) {
        sa.load_checked(ra[set], t, klen - t * BK);
        sb.load_checked(rb[set], t, klen - t * BK);
      };
      auto store = [&](int t, int set) {
        sa.store(ra[set], lds + (t & 1) * ImA::BYTES);
        sb.store(rb[set], lds + 2 * ImA::BYTES + (t & 1) * ImB::BYTES);
      };
#pragma unroll
      for (int d = 0; d < AHEAD; ++d)
        if (d < nk) load(d, d);
      store(0, 0);
      __syncthreads();
      auto compute = [&](int t) {
        const char* la = lds + (t & 1) * ImA::BYTES;
        const char* lb = lds + 2 * ImA::BYTES + (t & 1) * ImB::BYTES;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          uint4 fa[TM], fb[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) fa[i] = read_fragment<T, A_TR, BM>(la, wm + 16 * i, half, lane);
#pragma unroll
          for (int j = 0; j < TN; ++j) fb[j] = read_fragment<T, B_TR, BN>(lb, wn + 16 * j, half, lane);
          multiply<T, TM, TN>(fa, fb, acc);
        }
      };
      // interior: the K tiles fetched here need no check.  A loop of its own: with the checked fetch in the same loop
      // the compiler waits for every load in flight where the two meet.
      int k0 = 0;
      for (; k0 + 2 * AHEAD <= n_fast; k0 += AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
          sa.load_fast(ra[d], k0 + d + AHEAD);
          sb.load_fast(rb[d], k0 + d + AHEAD);
          compute(k0 + d);
          store(k0 + d + 1, (d + 1) % AHEAD);
          __syncthreads();
        }
      }
      for (; k0 < nk; k0 += AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
          const int kt = k0 + d;
          if (kt >= nk) break;
          if (kt + AHEAD < nk) load(kt + AHEAD, d);
          compute(kt);
          if (kt + 1 < nk) store(kt + 1, (d + 1) % AHEAD);
          __syncthreads();
        }
      }
    }

    if (SPLIT && parts > 1 && !join_parts<TM, TN, EDGE>(p, tile, acc, wm, wn, id - part * per, per, part, parts, &flag)) continue;

    // Block (i, j), register r: row 16 i + lane % 16, column 16 j + 4 (lane / 16) + r of the wave's part.
    char* const stage = lds + wave * (16 * EPITCH);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const float f[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
        gmm_store4<OutT>(stage + (lane & 15) * EPITCH + (16 * j + 4 * (lane >> 4)) * OSZ, f);
      }
      asm volatile("" ::: "memory");   // the wave's LDS accesses complete in order; the compiler must keep it
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int x = lane; x < 16 * ECPR; x += 64) {
        const int row = tile.m0 + wm + 16 * i + x / ECPR, col = tile.n0 + wn + (x % ECPR) * OEC;
        if (row < tile.m_lo || row >= tile.m_hi || col >= tile.n_hi || col + OEC <= tile.n_lo) continue;
        const char* src = stage + (x / ECPR) * EPITCH + (x % ECPR) * 16;
        OutT* dst = c + int64_t(row) * p.c_sm + int64_t(col) * p.c_sn;
        // The row's ragged end, or an output that is not contiguous along its columns, goes out element by element: out of
        // registers, or with a loop over the elements there are, as each pair of types is faster (a loop over all elements that
        // waits for the LDS for each of them takes 3 us of a launch).  us, that loop / this: bf16 2087 x 1034 in 80 groups of 3
        // elements 130 / 123, 3 products of 1000 x 1001 x 515 28 / 26, fp32 60 of 300 x 65 x 131 16.1 / 14.9.
        constexpr bool MIXED = sizeof(T) == 2 && OSZ == 4;
        uint4 v;
        if constexpr (sizeof(T) == 2) v = *reinterpret_cast<const uint4*>(src);   // fp32 has no registers to spare here
        const void* const chunk = sizeof(T) == 2 ? static_cast<const void*>(&v) : __builtin_assume_aligned(src, 16);
        if (p.c_sn == 1 && col >= tile.n_lo && col + OEC <= tile.n_hi) {
          __builtin_memcpy(dst, chunk, 16);
        } else if constexpr (MIXED) {
          const int first = gmm_max(tile.n_lo - col, 0), end = gmm_min(tile.n_hi - col, OEC);
#pragma unroll 1
          for (int e = first; e < end; ++e) __builtin_memcpy(dst + e * p.c_sn, src + e * OSZ, OSZ);
        } else {
          OutT out[OEC];
          __builtin_memcpy(out, chunk, 16);
#pragma unroll
          for (int e = 0; e < OEC; ++e)
            if (col + e >= tile.n_lo && col + e < tile.n_hi) dst[e * p.c_sn] = out[e];
        }
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();   // the next tile's images overwrite the staging area
  }
}

template <typename T, typename OutT, int EDGE, int SPLIT>
int launch_layout(const GmmParams& p, bool a_tr, bool b_tr, hipStream_t stream) {
  const dim3 grid(p.num_wg), block(NT);
  if (a_tr && b_tr)
    hipLaunchKernelGGL((gmm_staged_kernel<T, OutT, true, true, EDGE, SPLIT>), grid, block, 0, stream, p);
  else if (a_tr)
    hipLaunchKernelGGL((gmm_staged_kernel<T, OutT, true, false, EDGE, SPLIT>), grid, block, 0, stream, p);
  else if (b_tr)
    hipLaunchKernelGGL((gmm_staged_kernel<T, OutT, false, true, EDGE, SPLIT>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((gmm_staged_kernel<T, OutT, false, false, EDGE, SPLIT>), grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Tiles of a launch with square tiles of `edge`, the group boundaries taken to cut half a tile each on average.
int64_t expected_tiles(const GmmParams& p, int edge) {
  const int64_t tm = (p.M + edge - 1) / edge, tn = (p.N + edge - 1) / edge;
  if (p.jag == GMM_JAG_M) return (p.M / edge + (p.G + 1) / 2) * tn;
  if (p.jag == GMM_JAG_N) return tm * (p.N / edge + (p.G + 1) / 2);
  return p.G * tm * tn;
}

// The same if every group boundary cuts a whole tile more.
int64_t most_tiles(const GmmParams& p, int edge) {
  const int64_t tm = (p.M + edge - 1) / edge, tn = (p.N + edge - 1) / edge;
  if (p.jag == GMM_JAG_M) return (p.M / edge + (p.G < p.M ? p.G : p.M)) * tn;
  if (p.jag == GMM_JAG_N) return tm * (p.N / edge + (p.G < p.N ? p.G : p.N));
  return p.G * tm * tn;
}

// Cut the groups of a jagged contraction along K?  A group longer than a chunk is cut into even parts of up to a chunk (more
// than half of one), up to GMM_K_PARTS_MAX of them.  A chunk is an even share of one round of the grid, so that the chip is
// full whatever the groups' lengths, but not shorter than GMM_K_CHUNK_MIN: a part costs its start, a store and a read of its
// partial tile.  Sets k_chunk and k_parts; returns the most entries of the list, 0 if nothing is cut.
constexpr int GMM_K_CHUNK_MIN = 256;
template <int EDGE>
int64_t cut_contraction(GmmParams& p, int64_t most_wgs) {
  p.k_chunk = p.k_parts = 0;
  if (p.jag != GMM_JAG_K || p.ws_parts <= 0) return 0;
  const int64_t per = int64_t((p.M + EDGE - 1) / EDGE) * ((p.N + EDGE - 1) / EDGE);
  const int64_t share = (p.K * per + most_wgs - 1) / most_wgs;
  const int64_t chunk = share < GMM_K_CHUNK_MIN ? GMM_K_CHUNK_MIN : (share + 63) / 64 * 64;
  // entries of the list: every group's tiles once, and once more for every whole chunk; they need a counter and a slot
  const int64_t entries = p.G * per + p.K / chunk * per;
  int64_t room = int64_t(p.ws_parts) * GMM_WS_SLOT / (EDGE * EDGE * 4);
  if (room > GMM_WS_TICKET) room = GMM_WS_TICKET;
  if (entries > room || p.K < 2 * chunk) return 0;
  p.k_chunk = int32_t(chunk);
  p.k_parts = int32_t(room);
  return entries;
}

// Rows of a group on average: the tiles of one are full, the other's mostly hold rows that do not exist.
bool full_rows(const GmmParams& p) { return p.jag == GMM_JAG_M ? int64_t(p.M) >= 96 * int64_t(p.G) : p.M >= 96; }

// Cut the tiles of any other product along K?  A launch of few tiles with a long contraction leaves most of the chip idle and
// takes as long as one tile: each is cut into as many parts as there are workgroups for (the device knows the number of tiles),
// of at least GMM_K_SPLIT_MIN elements, joined like those of a jagged contraction.  Joining costs 8 to 12 us.  us, whole / cut:
// 16 rows, 8 groups of 4001 x 2047 112 / 47; 3 x 4 tiles of 331 x 517 x 4099, four products 86 / 40; fp32 500 x 500 x 8000, two
// 173 / 92.  Random launches of up to 256 tiles 2.7 (16-bit) and 2.8 (fp32) times as fast, 0.99 at worst.  The line leaves out what
// lost: K up to 1024 (two products of 512 x 1024 x 1024 17 / 22), more than 64 full tiles up to 1536 (two of 1000 x 1001 x 1101 27 /
// 33) or, with a first operand contiguous along M, up to 2048, more than 80 fp32 tiles up to 3072 (0.9 to 1.4).
constexpr int GMM_K_SPLIT_MIN = 256;
template <int EDGE>
bool split_tiles(GmmParams& p, int64_t most_wgs) {
  p.k_split = 0;
  if (p.jag == GMM_JAG_K || p.ws_parts <= 0) return false;
  const int64_t tiles = most_tiles(p, EDGE);
  int64_t room = int64_t(p.ws_parts) * GMM_WS_SLOT / (EDGE * EDGE * 4);
  if (room > GMM_WS_TICKET) room = GMM_WS_TICKET;
  if (tiles > 256 || 2 * tiles > most_wgs || 2 * tiles > room) return false;
  int least = 1024;
  if (EDGE == 64 && tiles > 80) least = 3072;
  if (EDGE == 128 && (tiles > 128 || (tiles > 64 && p.jag == GMM_JAG_NONE && full_rows(p)))) least = 1536;
  if (EDGE == 128 && tiles > 64 && p.a_sk != 1 && full_rows(p)) least = 2048;
  if (p.K <= least) return false;
  p.k_split = int32_t(p.K / GMM_K_SPLIT_MIN < GMM_K_PARTS_MAX ? p.K / GMM_K_SPLIT_MIN : GMM_K_PARTS_MAX);
  p.k_parts = int32_t(room);
  p.k_alone = full_rows(p) && (p.jag == GMM_JAG_N ? int64_t(p.N) >= 96 * int64_t(p.G) : p.N >= 96) ? 1280 : 640;
  return true;
}

// Does a number of tiles that the launch may well have leave a last round that is cut?  p.k_split and p.k_parts are set.
bool may_be_cut(const GmmParams& p, int edge, int wgs) {
  const int tm = (p.M + edge - 1) / edge, tn = (p.N + edge - 1) / edge;
  int lo = p.G * tm, hi = lo, step = tn;      // step times so many tiles
  if (p.jag != GMM_JAG_NONE) {
    const bool rows = p.jag == GMM_JAG_M;
    const int extent = rows ? p.M : p.N, groups = p.G < extent ? p.G : extent;
    const float full = float(extent) / edge, away = 2.0f * sqrtf(groups / 12.0f);
    step = rows ? tn : tm;
    lo = int(ceilf(full + groups / 3.0f - away));
    hi = int(floorf(full + groups / 2.0f + away));
    if (lo < (rows ? tm : tn)) lo = rows ? tm : tn;
    if (hi < groups) hi = groups;
  }
  for (int n = lo; n <= hi; ++n) {
    const int tiles = n * step, tail = tiles % wgs;
    if (tail_parts(tail, tiles - tail, wgs, edge, p) > 1) return true;
  }
  return false;
}

// Cut the tiles of the last round along K where it holds only a few?  Only the device knows how many there are, and the kernel
// that can cut them is 0.6 % slower where it does not (up to 4.5 %), a captured launch also clears a workspace for it (2 us).  So
// launches of one to four rounds with at least 24 K tiles that may well be cut: equal products make a known number of tiles;
// groups end anywhere in a tile, each makes half a tile more on average, all together with a deviation of the square root of
// G / 12, up to a third of the groups may be empty, and groups that are short make a tile each.  Any number in between, two
// deviations added, has to be one that is cut.  us, whole / cut: fp32 1024 x 1024 x 8192 columns in 8 uneven groups (2.1 rounds) 166 /
// 159; bf16 8191 x 2047 x 2047 in 8 groups 142 / 135, 5 products of 7 x 13204 x 2148 (520 tiles, 512 workgroups) 97 / 69; 3827 rows
// in 31 groups, 6 of them empty, of 3189 x 1841 198 / 151.  170 random 16-bit launches whose last
// round is cut 1.24 times as fast (0.99 to 1.6); with K below 2048 and most of the time spent on memory it can lose (28 products of
// 2048 x 1835 to 7305 columns in all, 80 to 128 tiles in the last round 0.79 to 1.0).  fp32, 24 launches 1.06 (1.01 to 1.18).
template <int EDGE>
bool split_tail(GmmParams& p, int64_t most_wgs, int esz) {
  p.k_split = 0;
  if (p.jag == GMM_JAG_K || p.ws_parts <= 0 || int64_t(p.K) * esz < 24 * ROW_BYTES) return false;
  const int64_t tiles = expected_tiles(p, EDGE);
  int64_t room = int64_t(p.ws_parts) * GMM_WS_SLOT / (EDGE * EDGE * 4);
  if (room > GMM_WS_TICKET) room = GMM_WS_TICKET;
  if (tiles <= most_wgs || tiles > 4 * most_wgs) return false;
  p.k_split = p.K / (GMM_K_SPLIT_MIN / 2) < GMM_K_CLUSTER ? p.K / (GMM_K_SPLIT_MIN / 2) : GMM_K_CLUSTER;
  p.k_parts = int32_t(room);
  if (may_be_cut(p, EDGE, int(most_wgs))) return true;
  p.k_split = 0;
  return false;
}

template <typename T, typename OutT, int EDGE>
int launch_layout(GmmParams p, bool a_tr, bool b_tr, int num_cus, hipStream_t stream) {
  const int64_t most = int64_t(tile_wgs(EDGE)) * num_cus;
  int64_t bound = cut_contraction<EDGE>(p, most);
  if (bound == 0) bound = gmm_tile_bound(p.jag, p.G, p.M, p.N, EDGE, EDGE);
  const bool split = split_tiles<EDGE>(p, most) || split_tail<EDGE>(p, most, sizeof(T));
  if (split) bound = gmm_tile_bound(p.jag, p.G, p.M, p.N, EDGE, EDGE) * p.k_split;
  const int64_t want = (bound + 7) / 8 * 8;
  p.num_wg = int(want < most ? (want < 8 ? 8 : want) : most);
  if (split) return launch_layout<T, OutT, EDGE, 2>(p, a_tr, b_tr, stream);
  return p.k_chunk ? launch_layout<T, OutT, EDGE, 1>(p, a_tr, b_tr, stream) : launch_layout<T, OutT, EDGE, 0>(p, a_tr, b_tr, stream);
}

// fp32: 64 x 64 tiles (four workgroups per CU) or 128 x 128 (two)?  A launch takes whole rounds of its grid, and a
// round of large tiles takes 1.84 times a round of small ones (2048 x 2048 x 2048, four products: 2 rounds of 258 us
// against 4 of 140 us), so the cheaper count wins.  Measured, us, small / large: 1024 rows, K 1024, 8192 columns in
// 8 groups 166 / 216; 4096 x 2048 x 2048 in 8 groups 316 / 394; 1024 x 1024 x 1024 in 8 groups 45 / 77; 8192 x 1024
// x 4096 in 8 groups 599 / 592; four products of 2048^3 562 / 517.
// 16-bit operands always take 128 x 128: twice the MFMA rate makes the small tile's LDS reads the bound (8191 x 2047
// x 2047 in 8 groups: 218 us against 153; 24 groups of 6151 x 1031 x 519: 32 against 36).
bool small_tiles(const GmmParams& p, int in_dtype, int num_cus) {
  if (in_dtype != GMM_DT_F32) return false;
  const int64_t small_round = int64_t(tile_wgs(64)) * num_cus, large_round = int64_t(tile_wgs(128)) * num_cus;
  const int64_t small = (expected_tiles(p, 64) + small_round - 1) / small_round;
  const int64_t large = (expected_tiles(p, 128) + large_round - 1) / large_round;
  return 100 * small < 184 * large;
}

}  // namespace

// Aligned 16-bit products that this kernel runs faster than the assembly tile, which takes up to 256 x 256 elements
// of output and needs 3.3 us before its first tile (1 us here): little work, spread over more and smaller tiles by four
// times as many workgroups.  T tiles of 128 x 128 with nk K tiles each; us, assembly tile / here:
//   A contiguous along K: six groups of 32 x 64 x 48 9.5 / 5.5; 131072 x 32 x 64 in 64 groups 28 / 13.7; 8192 x 256 x
//   384 in 64 groups 13.5 / 9.9.  Over 260 random shapes, operands from memory, the ratio is 1.46 at nk = 1, 1.33 at 2, 1.17
//   at 4, 1.12 at 6 and 1.05 with every third shape slower at 8, where the assembly tile has three K tiles in flight.  Past
//   T nk = 3072 its larger tile moves less between L2 and LDS (16384 x 256 x 4096 in 8 groups 55 / 72), and groups shorter
//   than its 64-row tile fill half a tile here (750 tiles of 264 x 424 x 1264 in 73 groups 26 / 29).
//   A contiguous along M: the assembly tile always has 256 rows.  1256 x 824 x 456 in 11 groups 32 / 21; 1392 x 1312 x
//   352 in 40 groups 47 / 37; 2160 tiles of 1880 x 144 x 1120 35 / 37.  It wins once there are rounds to fill.
//   Few tiles, K past 1024: cut along K (split_tiles).  The assembly tile cuts its own tiles from K = 4096 on, into longer
//   parts.  us, assembly tile / here: one row each of 8 groups of 2048 x 1536 30 / 20; 8 products of 64 x 1024 x 4000 53 / 29;
//   512 rows, 8 groups of 4000 x 1024 55 / 30; A contiguous along M, 1024 x 1024 x 8192 81 / 52.  Full tiles want more K or fewer of
//   them: 1024 x 1024 x 2056 26 / 27, x 2816 31 / 27; 512 x 1024 x 1288 19 / 21, x 1800 23 / 22; 1472 x 1264 x 2304 29 / 33, x 3456 40 /
//   38 (groups make fewer tiles than the most).  150 random launches of up to 256 tiles 1.55 times as fast (0.95 to 3.6, those that
//   stay on the assembly tile among them).
//   Jagged contraction: cut along K (above) it fills the chip whatever the groups' lengths.  A contiguous along M, up to 384
//   tiles: 64 groups of 32 x 64 with 2048 elements each 46 / 13; 24 groups of 328 x 360, 95496 elements 201 / 98; two groups
//   of 328 x 712, 40424 elements 652 / 62; past 384 the larger tile catches up (496 tiles of 184 x 464 in 62 even groups
//   70 / 78), but for very short groups (1230 tiles of 104 x 1248 in 123 groups, 16464 elements 69 / 52).  A contiguous along
//   K stays with the assembly tile, never cut: its 16-byte loads start at any element here (80 tiles of 200 x 968 in 5
//   groups, 2960 elements 19 / 26), and the bits of such a product do not depend on there being a workspace.
//   The line does not ask whether the launch can be cut: uncut, for want of a workspace, 570 random calls with A contiguous
//   along M are 1.31 times as fast here on average (12 groups of 176 x 368, 4936 elements 19.4 / 11.8), and slower by 8 % at
//   most (7 groups of 352 x 1976, 50880 elements 636 / 686).
bool gmm_staged_preferred(const GmmParams& p, int num_cus) {
  if (p.act || !gmm_staged_eligible(p)) return false;
  const int64_t tiles = most_tiles(p, 128), nk = (p.K + 63) / 64, cus = num_cus;
  if (p.jag == GMM_JAG_K) {
    return p.a_sk != 1 && (2 * tiles <= 3 * cus || (p.K <= 64 * int64_t(p.G) && tiles <= 4 * cus));
  }
  if (gmm_staged_cut_preferred(p, num_cus)) return true;
  if (p.a_sk != 1 && tiles <= tile_wgs(128) * cus && nk <= 32) return true;
  const bool rows_fill = p.jag == GMM_JAG_M ? p.M >= 64 * int64_t(p.G) : p.M >= 64;
  return nk <= 6 && tiles * nk <= 12 * cus && (nk == 1 || rows_fill || tiles <= cus);
}

bool gmm_staged_cut_preferred(const GmmParams& p, int num_cus) {
  GmmParams cut = p;
  if (!gmm_staged_eligible(p) || !split_tiles<128>(cut, tile_wgs(128) * int64_t(num_cus))) return false;
  const int64_t tiles = most_tiles(p, 128), parts = tile_wgs(128) * int64_t(num_cus) / tiles;
  if (p.a_sk != 1) return p.K >= 2560 && (parts >= 4 || p.K <= 6144);
  const bool equal = p.jag == GMM_JAG_NONE && p.N >= 96;    // full tiles; of groups most_tiles() is more than there are
  if (parts >= 16) return !(equal && p.M > 128) || p.K >= (parts >= 20 ? 1280 : 1664);
  if (full_rows(p)) return p.K > (equal && p.M > 192 && parts < 8 ? 3072 : 2048) && (parts >= 8 || (parts >= 4 && p.K <= 4096));
  return parts >= 5 && p.K <= 6144;
}

// Products without alignment, 16-bit, that are over before a tile of 128 x 128 has started: K up to 16 and no more such tiles
// than compute units.  The element-wise kernel's 64 x 64 tiles are then so many times as fast as the staged kernel (3000 random
// calls; first operand contiguous along K, 129 to 256 tiles / along M, up to 128): K 1 and 2 1.18 / 1.11, 3 and 4 1.27 / 1.13, 5
// to 8 1.17 / 1.14, 9 to 12 1.13 / 1.21, 13 to 16 0.93 / 1.15; K 17 to 20 1.0 / 0.93; 257 to 512 tiles 1.07 / 0.99 (64 products of
// 466 x 7 x 3 5.9 us against 11.3; at worst 53 of 5 x 7 x 186 8.0 against 6.3).  In fp32 the staged kernel is faster at any K.
bool gmm_element_preferred(const GmmParams& p, int in_dtype, int num_cus) {
  return in_dtype != GMM_DT_F32 && p.K <= 16 && most_tiles(p, 128) <= num_cus;
}

bool gmm_staged_eligible(const GmmParams& p) {
  // each operand contiguous along one of its dimensions; gathered rows only along K; element offsets are 64-bit, so
  // no extent is too large
  const bool a_kc = p.a_sk == 1, b_kc = p.b_sk == 1;
  if (!a_kc && (p.a_sm != 1 || p.gather)) return false;
  if (!b_kc && p.b_sn != 1) return false;
  const int64_t lda = a_kc ? p.a_sm : p.a_sk, ldb = b_kc ? p.b_sn : p.b_sk;
  // a chunk of 16 bytes has to fit into every operand
  const int64_t rows = p.gather ? p.a_rows : p.M;
  const int64_t a_len = a_kc ? (rows - 1) * lda + p.K : (p.K - 1) * lda + p.M;
  const int64_t b_len = b_kc ? (p.N - 1) * ldb + p.K : (p.K - 1) * ldb + p.N;
  return lda >= 1 && ldb >= 1 && p.K >= 1 && rows >= 1 && a_len >= 8 && b_len >= 8;
}

template <int EDGE>
static bool uses_workspace(GmmParams& p, int64_t most_wgs, int esz) {
  return cut_contraction<EDGE>(p, most_wgs) > 0 || split_tiles<EDGE>(p, most_wgs) || split_tail<EDGE>(p, most_wgs, esz);
}

bool gmm_staged_uses_workspace(const GmmParams& p, int in_dtype, int num_cus) {
  GmmParams cut = p;
  if (small_tiles(p, in_dtype, num_cus))
    return uses_workspace<64>(cut, int64_t(tile_wgs(64)) * num_cus, 4);
  return uses_workspace<128>(cut, int64_t(tile_wgs(128)) * num_cus, in_dtype == GMM_DT_F32 ? 4 : 2);
}

int gmm_launch_staged(GmmParams p, int in_dtype, int out_dtype, int num_cus, hipStream_t stream) {
  p.align = 1;
  const bool a_tr = p.a_sk != 1, b_tr = p.b_sk != 1;
  if (in_dtype == GMM_DT_F32 && out_dtype == GMM_DT_F32)
    return small_tiles(p, in_dtype, num_cus) ? launch_layout<float, float, 64>(p, a_tr, b_tr, num_cus, stream)
                                             : launch_layout<float, float, 128>(p, a_tr, b_tr, num_cus, stream);
#define GMM_STAGED_CASE(IN_CODE, OUT_CODE, IN_T, OUT_T) \
  if (in_dtype == IN_CODE && out_dtype == OUT_CODE) return launch_layout<IN_T, OUT_T, 128>(p, a_tr, b_tr, num_cus, stream);
  GMM_STAGED_CASE(GMM_DT_BF16, GMM_DT_BF16, gmm_bf16, gmm_bf16)
  GMM_STAGED_CASE(GMM_DT_BF16, GMM_DT_F32, gmm_bf16, float)
  GMM_STAGED_CASE(GMM_DT_F16, GMM_DT_F16, gmm_f16, gmm_f16)
  GMM_STAGED_CASE(GMM_DT_F16, GMM_DT_F32, gmm_f16, float)
#undef GMM_STAGED_CASE
  return -1;
}
