// Device-side helpers shared by the gfx950 kernels: the per-workgroup tile
// table (prefix sum of per-group tile counts kept in LDS) and dtype conversion.
#pragma once
#include <hip/hip_runtime.h>
#include "gmm_sched.h"

// Exclusive prefix sum of per-group tile counts into cum[0..G] (LDS), returns
// the total.  All NT threads of the workgroup must call it; it ends with a
// barrier.  For 3D x 3D there is no table: every group has the same grid.
// chunk > 0: a group counts once for each of its parts along K (gmm_group_parts).
template <int NT>
__device__ __forceinline__ int gmm_build_tile_table(const GmmParams& p, int bm, int bn, int32_t* cum, int chunk = 0) {
  const int tid = threadIdx.x;
  if (p.jag == GMM_JAG_NONE) return p.G * gmm_cdiv(p.M, bm) * gmm_cdiv(p.N, bn);

  const int extent = p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K);
  for (int g = tid; g < GMM_MAX_GROUPS; g += NT) {
    int cnt = 0;
    if (g < p.G) {
      int lo, hi, tm, tn;
      gmm_group_range(p.offs, g, extent, lo, hi);
      gmm_group_grid(p.jag, lo, hi, p.M, p.N, bm, bn, p.align, tm, tn);
      cnt = tm * tn * gmm_group_parts(hi - lo, chunk);
    }
    cum[g + 1] = cnt;
  }
  if (tid == 0) cum[0] = 0;
  __syncthreads();
  if (tid < 64) {
    // lane l owns entries 1 + 16 l .. 16 + 16 l
    constexpr int PER = GMM_MAX_GROUPS / 64;
    int v[PER];
    int run = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) { run += cum[1 + tid * PER + i]; v[i] = run; }
    int incl = run;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64);
      if (tid >= d) incl += up;
    }
    const int before = incl - run;
#pragma unroll
    for (int i = 0; i < PER; ++i) cum[1 + tid * PER + i] = v[i] + before;
  }
  __syncthreads();
  return cum[p.G];
}

// Linear tile id -> group, index inside the group and the group's range, using the table above; uniform.
__device__ __forceinline__ void gmm_find_tile(const GmmParams& p, const int32_t* cum, int t, int bm, int bn, int& g,
                                              int& local, int& lo, int& hi) {
  lo = hi = 0;
  if (p.jag == GMM_JAG_NONE) {
    const int per = gmm_cdiv(p.M, bm) * gmm_cdiv(p.N, bn);
    g = t / per;
    local = t - g * per;
  } else {
    g = gmm_find_group(cum, p.G, t);
    local = t - cum[g];
    gmm_group_range(p.offs, g, p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K), lo, hi);
  }
  g = __builtin_amdgcn_readfirstlane(g);
  local = __builtin_amdgcn_readfirstlane(local);
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
}

// Tile `local` of group g.
__device__ __forceinline__ GmmTile gmm_tile_of_group(const GmmParams& p, int g, int local, int lo, int hi, int bm, int bn) {
  int tm, tn, mt, nt;
  gmm_group_grid(p.jag, lo, hi, p.M, p.N, bm, bn, p.align, tm, tn);
  gmm_decode_in_group(local, tm, tn, mt, nt);
  return gmm_make_tile(p, g, lo, hi, mt, nt, bm, bn);
}

// Linear tile id -> tile, using the table above.
__device__ __forceinline__ GmmTile gmm_locate_tile(const GmmParams& p, const int32_t* cum, int t, int bm, int bn) {
  int g, local, lo, hi;
  gmm_find_tile(p, cum, t, bm, bn, g, local, lo, hi);
  return gmm_tile_of_group(p, g, local, lo, hi, bm, bn);
}

// ---- the same table for up to 64 groups in registers ------------------------------------------------ //
// Lane g of every wave holds group g; a tile's group is the number of groups that end at or before it.  No LDS, no
// barrier, no search: 1 us from the kernel's start to the first tile where the table in LDS takes 3.3 us (it is a
// chain of loads, barriers and dependent LDS reads, and every workgroup of a small launch waits for it).
__device__ __forceinline__ int gmm_wave_inclusive_scan(int v) {
  // prefix sums inside each row of 16 lanes, then lane 15 of a row into the next row, lane 31 into rows 2 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

struct GmmWaveGroups {
  int lo, hi, count, incl;   // of the lane's group: its range, its tiles, tiles up to and including it

  // Returns the total number of tiles.
  __device__ __forceinline__ int build(const GmmParams& p, int bm, int bn, int chunk = 0) {
    const int lane = threadIdx.x & 63;
    const int extent = p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K);
    lo = hi = count = 0;
    if (lane < p.G) {
      int tm, tn;
      gmm_group_range(p.offs, lane, extent, lo, hi);
      gmm_group_grid(p.jag, lo, hi, p.M, p.N, bm, bn, p.align, tm, tn);
      count = tm * tn * gmm_group_parts(hi - lo, chunk);
    }
    incl = gmm_wave_inclusive_scan(count);
    return __builtin_amdgcn_readlane(incl, 63);
  }

  // Group of tile t, the tile's index inside it, the group's range: uniform over the wave.
  __device__ __forceinline__ void find(int t, int& g, int& local, int& glo, int& ghi) const {
    g = __popcll(__ballot(incl <= t));
    local = t - __builtin_amdgcn_readlane(incl, g) + __builtin_amdgcn_readlane(count, g);
    glo = __builtin_amdgcn_readlane(lo, g);
    ghi = __builtin_amdgcn_readlane(hi, g);
  }
};

// ---- two-height tile list (gmm_sched.h): tables cum[0] (tall) and cum[1] (short), each G + 1 entries ---- //
template <int NT>
__device__ __forceinline__ void gmm_scan_table(int32_t* cum) {
  const int tid = threadIdx.x;
  if (tid < 64) {
    constexpr int PER = GMM_MAX_GROUPS / 64;
    int v[PER];
    int run = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) { run += cum[1 + tid * PER + i]; v[i] = run; }
    int incl = run;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64);
      if (tid >= d) incl += up;
    }
    const int before = incl - run;
#pragma unroll
    for (int i = 0; i < PER; ++i) cum[1 + tid * PER + i] = v[i] + before;
  }
}

// Returns the total number of tiles; total_tall gets the number of tall ones (they come first in the launch
// order: the workgroups of all XCDs then work on tiles of one height in every round and stay in step, which
// keeps the operand panels they share in the Infinity Cache).
template <int NT>
__device__ __forceinline__ int gmm_build_tile_table2(const GmmParams& p, int bn, int32_t* cum_tall, int32_t* cum_short,
                                                     int& total_tall) {
  const int tid = threadIdx.x;
  if (p.jag == GMM_JAG_NONE) {
    const int tn = gmm_cdiv(p.N, bn);
    int n_tall, n_short, rem_rows;
    gmm_split_rows(p.M, p.tall, p.shrt, n_tall, n_short, rem_rows);
    total_tall = p.G * n_tall * tn;
    return total_tall + p.G * n_short * tn;
  }
  const int extent = p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K);
  for (int g = tid; g < GMM_MAX_GROUPS; g += NT) {
    int ct = 0, cs = 0;
    if (g < p.G) {
      int lo, hi, n_tall, n_short, rem_rows;
      gmm_group_range(p.offs, g, extent, lo, hi);
      gmm_split_rows(gmm_group_rows(p.jag, lo, hi, p.M, p.align), p.tall, p.shrt, n_tall, n_short, rem_rows);
      const int tn = gmm_group_tile_cols(p.jag, lo, hi, p.N, p.align, bn);
      ct = n_tall * tn;
      cs = n_short * tn;
    }
    cum_tall[g + 1] = p.group_major ? ct + cs : ct;
    cum_short[g + 1] = p.group_major ? 0 : cs;
  }
  if (tid == 0) { cum_tall[0] = 0; cum_short[0] = 0; }
  __syncthreads();
  gmm_scan_table<NT>(cum_tall);
  gmm_scan_table<NT>(cum_short);
  __syncthreads();
  total_tall = cum_tall[p.G];
  return total_tall + cum_short[p.G];   // group-major order: everything is in the first table
}

// Tile id -> tile, per lane (ids differ between lanes).
__device__ __forceinline__ GmmTile gmm_locate_tile2(const GmmParams& p, const int32_t* cum_tall, const int32_t* cum_short,
                                                    int total_tall, int t, int bn) {
  int cls = t < total_tall ? 0 : 1;
  const int tc = cls ? t - total_tall : t;
  int g, local, lo = 0, hi = 0;
  if (p.group_major && p.jag != GMM_JAG_NONE) {
    // one table: a group's tall tiles, then its remainder tiles
    g = gmm_find_group(cum_tall, p.G, t);
    local = t - cum_tall[g];
    gmm_group_range(p.offs, g, p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K), lo, hi);
    int n_tall, n_short, rem_rows;
    gmm_split_rows(gmm_group_rows(p.jag, lo, hi, p.M, p.align), p.tall, p.shrt, n_tall, n_short, rem_rows);
    const int tall_tiles = n_tall * gmm_group_tile_cols(p.jag, lo, hi, p.N, p.align, bn);
    cls = local < tall_tiles ? 0 : 1;
    if (cls) local -= tall_tiles;
  } else if (p.jag == GMM_JAG_NONE) {
    int n_tall, n_short, rem_rows;
    gmm_split_rows(p.M, p.tall, p.shrt, n_tall, n_short, rem_rows);
    const int per = (cls ? n_short : n_tall) * gmm_cdiv(p.N, bn);
    g = tc / per;
    local = tc - g * per;
  } else {
    const int32_t* cum = cls ? cum_short : cum_tall;
    g = gmm_find_group(cum, p.G, tc);
    local = tc - cum[g];
    gmm_group_range(p.offs, g, p.jag == GMM_JAG_M ? p.M : (p.jag == GMM_JAG_N ? p.N : p.K), lo, hi);
  }
  return gmm_make_tile2(p, g, lo, hi, cls, local, bn);
}

// ---- tile queue of a jagged contraction -------------------------------------------------------------- //
// Every group has the same grid of tiles, but its contraction is as long as the group, so dealing tiles round by round
// leaves whole chips waiting for the workgroups that drew the long groups.  Here the groups are sorted by length, longest
// first, and a workgroup draws its next tile when it is free.  128 groups, 20 of them empty, the others skewed (log-normal,
// sigma 2.4), 32768 elements, 2048 x 768 each, bf16: dealt in group order 230 us, drawn 161; fp32 result 306 and 212.
// The sorted list is cut into spans of one tile per workgroup and every span into one block per XCD, so that the tiles
// an XCD runs together are neighbours; each XCD has a counter of its own, in the head of the workspace, and a workgroup
// whose XCD has nothing left draws from the others.  The first tile needs no draw, the following ticket is drawn
// before a tile runs and looked at after it.
// A drawn tile is located alone, on the critical path: 1.4 us each, where tiles that are dealt are located several at a
// time.  Dealt round by round, the sorted list leaves workgroups apart by no more than the longest tile's time less the
// shortest's, 1.5 us per K tile of 64.  So tiles are drawn when the longest group exceeds the mean by two K tiles a round
// (at one a round, groups of 64 to 128 elements on average lost 4 to 8 %), and dealt otherwise or without a workspace.  Without
// one, where the spread may be any, every other round is dealt backwards: the skewed groups above take 196 us (212 with every
// round forwards, 226 in group order), 33 groups of 1208 x 352, 21600 elements 39 (51).  With a workspace, where the spread
// is small, it gains as often as it loses (223 and 238 us for 201 groups of 1072 x 1360, 6432 elements).
// Dealing what is not worth drawing, us, every list drawn / dealt, the matrices above: 1280 elements 108 / 91, 32768 of 256
// each 153 / 147.
// One thread of the workgroup uses the queue; it ends when all eight counters have run out.
struct GmmKQueue {
  int per, total, chunk;   // tiles per group, of the launch, of an XCD's block in a span
  int turn;                // counters that have run out, counted from the workgroup's own
  bool drawn;              // tiles are drawn, not dealt; the same in all threads
  bool back;               // dealt: every other round backwards
  int next;                // drawn: tile to run, -1: none left
  int ticket;              // drawn ticket (index in the counter's part of the list)

  // order[i] = group of rank i, bound[g] .. bound[g + 1] = range of group g.  All threads; ends with a barrier.
  // keys: room for G + 3 words, aligned to 16 bytes.  A group's rank is the number of greater keys (gmm_k_queue_key, no two
  // are equal), counted four to a broadcast read, for two groups of a thread at a time.  Every workgroup does it, so it is part
  // of every launch: 512 groups of 512 x 512, 16384 elements 71 us (67 in group order; 105 with lengths compared one by one).
  // Up to about 450 groups a bitonic sort takes longer (128 groups 5 us more, 512 groups 1 us less than one group at a time).
  template <int NT>
  __device__ __forceinline__ void build(const GmmParams& p, int bn, int32_t* order, int32_t* bound, uint32_t* keys) {
    const int tid = threadIdx.x;
    for (int g = tid; g < p.G; g += NT) {
      int lo, hi;
      gmm_group_range(p.offs, g, p.K, lo, hi);
      if (g == 0) bound[0] = 0;
      bound[g + 1] = gmm_min(gmm_max(p.offs[g], 0), p.K);
      keys[g] = gmm_k_queue_key(g, hi - lo, p.K);
    }
    if (tid < 3) keys[p.G + tid] = 0;
    int n_tall, n_short, rem_rows;
    gmm_split_rows(p.M, p.tall, p.shrt, n_tall, n_short, rem_rows);
    per = (n_tall + n_short) * gmm_cdiv(p.N, bn);
    total = p.G * per;
    chunk = int(gridDim.x) >> 3;
    turn = 0;
    ticket = int(blockIdx.x) >> 3;
    next = tile_of(int(blockIdx.x) & 7, ticket);
    back = p.ws == nullptr;
    drawn = false;
    if (!gmm_k_queue_sorts(per, p.G, int(gridDim.x))) {
      for (int g = tid; g < p.G; g += NT) order[g] = g;
      __syncthreads();
      return;
    }
    __syncthreads();
    for (int g = tid; g < p.G; g += 2 * NT) {
      const bool two = g + NT < p.G;
      const uint32_t u = keys[g], v = two ? keys[g + NT] : ~0u;
      int before_u = 0, before_v = 0;
#pragma unroll 8
      for (int h = 0; h < p.G; h += 4) {
        const uint4 k = *reinterpret_cast<const uint4*>(keys + h);
        before_u += (k.x > u) + (k.y > u) + (k.z > u) + (k.w > u);
        before_v += (k.x > v) + (k.y > v) + (k.z > v) + (k.w > v);
      }
      order[before_u] = g;
      if (two) order[before_v] = g + NT;
    }
    __syncthreads();
    const int longest = gmm_max(bound[order[0] + 1] - bound[order[0]], 0);
    drawn = p.ws && longest - p.K / p.G >= 128 * gmm_cdiv(total, int(gridDim.x));
  }

  // Tiles that the workgroup is dealt, and the i-th of them.  Backwards, the workgroups with the longest tiles of one round
  // get the shortest of the next.
  __device__ __forceinline__ int dealt() const {
    const int rounds = total / int(gridDim.x);
    return rounds + (tile_number(rounds) < total ? 1 : 0);
  }
  __device__ __forceinline__ int tile_number(int i) const {
    const int place = (int(blockIdx.x) & 7) * chunk + (int(blockIdx.x) >> 3);
    return i * int(gridDim.x) + (back && (i & 1) ? int(gridDim.x) - 1 - place : place);
  }

  // Tile number `i` of an XCD's part of the list, or -1 past its end.
  __device__ __forceinline__ int tile_of(int xcd, int i) const {
    const int span = i / chunk;
    const int t = (span * 8 + xcd) * chunk + (i - span * chunk);
    return t < total ? t : -1;
  }

  __device__ __forceinline__ void draw(const GmmParams& p) {
    if (turn < 8)
      ticket = chunk + int(__hip_atomic_fetch_add(static_cast<unsigned*>(p.ws) + ((blockIdx.x + turn) & 7) * GMM_WS_QUEUE_PITCH, 1u,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }

  // The drawn ticket becomes the next tile; a counter that has run out is left for the next one.
  __device__ __forceinline__ void advance(const GmmParams& p) {
    next = tile_of(int(blockIdx.x + turn) & 7, ticket);
    while (next < 0 && ++turn < 8) {
      draw(p);
      next = tile_of(int(blockIdx.x + turn) & 7, ticket);
    }
  }

  __device__ __forceinline__ GmmTile locate(const GmmParams& p, int t, const int32_t* order, const int32_t* bound, int bn) const {
    const int rank = t / per, g = order[rank];
    int n_tall, n_short, rem_rows, local = t - rank * per;
    gmm_split_rows(p.M, p.tall, p.shrt, n_tall, n_short, rem_rows);
    const int tall_tiles = n_tall * gmm_cdiv(p.N, bn);
    const int cls = local < tall_tiles ? 0 : 1;
    const int lo = bound[g];
    return gmm_make_tile2(p, g, lo, gmm_max(bound[g + 1], lo), cls, cls ? local - tall_tiles : local, bn);
  }

  // The last workgroup to leave puts the counters back to zero for the next launch: all others have drawn their last
  // tickets.
  __device__ __forceinline__ void leave(const GmmParams& p) const {
    unsigned* const header = static_cast<unsigned*>(p.ws);
    if (__hip_atomic_fetch_add(&header[GMM_WS_EXITED], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != gridDim.x - 1) return;
    for (int x = 0; x < 8; ++x)
      __hip_atomic_store(&header[x * GMM_WS_QUEUE_PITCH], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&header[GMM_WS_EXITED], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

// Source row of product row m under a row gather; -1 if the index is outside the source matrix.
__device__ __forceinline__ int gmm_gather_row(const GmmParams& p, int m) {
  const int s = p.gather[m];
  return (s >= 0 && s < p.a_rows) ? s : -1;
}

// ---- element types -------------------------------------------------------- //
struct gmm_bf16 { uint16_t bits; };
struct gmm_f16 { _Float16 v; };

__device__ __forceinline__ float gmm_to_float(gmm_bf16 x) { return __uint_as_float(uint32_t(x.bits) << 16); }
__device__ __forceinline__ float gmm_to_float(gmm_f16 x) { return float(x.v); }
__device__ __forceinline__ float gmm_to_float(float x) { return x; }

// fp32 -> bf16 bits, round to nearest even, NaN stays NaN.
__device__ __forceinline__ uint16_t gmm_bf16_bits(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x0040u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}

// Four at a time: v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32 where there is one.
template <typename OutT>
__device__ __forceinline__ void gmm_store4(void* dst, const float* f) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef __bf16 b4 __attribute__((ext_vector_type(4)));
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  const f4 v = {f[0], f[1], f[2], f[3]};
  if constexpr (__is_same(OutT, float)) {
    __builtin_memcpy(dst, &v, 16);
  } else if constexpr (__is_same(OutT, gmm_f16)) {
    const h4 h = __builtin_convertvector(v, h4);
    __builtin_memcpy(dst, &h, 8);
  } else {
    const b4 b = __builtin_convertvector(v, b4);
    __builtin_memcpy(dst, &b, 8);
  }
}

template <typename T> __device__ __forceinline__ T gmm_from_float(float f);
template <> __device__ __forceinline__ gmm_bf16 gmm_from_float<gmm_bf16>(float f) { return gmm_bf16{gmm_bf16_bits(f)}; }
template <> __device__ __forceinline__ gmm_f16 gmm_from_float<gmm_f16>(float f) { return gmm_f16{_Float16(f)}; }
template <> __device__ __forceinline__ float gmm_from_float<float>(float f) { return f; }
