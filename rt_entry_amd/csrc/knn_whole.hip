// kNN lists of data whose values are whole numbers of magnitude <= 256 (image
// descriptors are bytes).  They are bf16 values, so one bf16 MFMA product of 16
// times the FP32 rate gives what the FP32 kernel (knn.hip) computes.  The
// accumulator starts at -|x|^2 / 2 and ends at q.x - |x|^2 / 2.  With norms below
// 2^23 and no negative value (below 2^22 with negative ones) every partial sum
// is a multiple of 1/2 of at most 2^23 in magnitude, and so are the sums with
// |q|^2 / 2 and half distances: exact in FP32 in any order.
//
// Points are visited by cells.  np / 320 rows are pivots, half of them evenly
// spaced, the others among the quarter of the points that lie farthest from those
// (a cluster without a pivot leaves rows that every block holding one must compare
// with everything); every point goes to the cell of its nearest one, by one
// product, and the cells' points are sorted by a few bits of that distance and laid
// out as tiles of 64 (a cell's last one padded).  A tile knows its cell and the range [a, b] of its points'
// distances from the pivot.  Rows are taken in the same order, so that a
// workgroup's rows are near each other: it visits its own cells first, which gives
// nearly all neighbours and tight thresholds, and then every tile that could hold
// a nearer point than some row's k-th best: by the triangle inequality none of its
// points is nearer than max(D - b, a - D) for a row at distance D from the pivot.
//
// 160k x 128, k = 64: 2.3 ms in 160 clusters, of which 1.9 go to picking points in
// about 30 tiles a block; 18 ms for uniform values, where every tile is visited
// (products and operand reads 5, picking the rest); 73 ms with the FP32 kernel.
#include <hip/hip_runtime.h>
#include <float.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "key_sort.h"
#include "knn.h"

namespace rte {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr int kWnCols = 64;    // points per tile
constexpr int kWnQueue = 416;  // queued points per wave: a block's 256 and some
constexpr int kWnWaves = 4;    // of a workgroup
constexpr int kWnRows = 32 * kWnWaves;
constexpr int kWnPerCu = 2;    // workgroups
constexpr int kWnKeys = 128;   // of a row: 64 list, 64 buffer
constexpr int kWnPivots = 1024;
constexpr int kWnBuckets = 32;  // of a cell, by distance from its pivot
constexpr int kWnFarBins = 2048;
constexpr int64_t kWnStep = 1 << 19;  // rows per launch
constexpr int kWnList = 2048;  // tiles looked at together

template <int KS>  // d / 32
struct WnTile {
  static constexpr int CPR = 4 * KS;              // 16-byte units per point
  static constexpr int SWM = (CPR & -CPR) - 1;    // 3, 7, 3, 15
  static constexpr int UNITS = kWnCols * CPR;     // per tile
  static constexpr int SLOT = UNITS + 32;         // and 64 floats -|x|^2 / 2, 64 ids
};

// a tile's points, the range of their distances from its cell's pivot
struct WnMeta {
  float a, b;
  int cell, pad;
};

// The cells' layout and the scratch of a call, all in one allocation.
struct WnLayout {
  int64_t np, slots;  // slots: of the sorted points, pads included, at most
  int d, pivots, ppad;
  int pivots1;  // those evenly spaced
  int launches;
  uint16_t* Xs;   // slots x d: the points by cell
  float* hs;      // slots: -|x|^2 / 2 (-inf: no point)
  int32_t* sid;   // slots: row of X (-1: no point)
  float* sd;      // slots: squared distance from the pivot
  WnMeta* meta;   // slots / 64
  int32_t* cell;  // np
  float* d2;      // np
  int32_t* hist;  // pivots x kWnBuckets: points; then, of the rows asked for, rhist
  int32_t* rhist;
  int32_t* pos;  // next free slot
  int32_t* rpos;
  int32_t* cstart;  // pivots + 1: first slot of a cell
  uint16_t* Pb;     // ppad x d
  float* ph;        // ppad
  int32_t* far;     // kWnFarBins counts of points by distance, and a counter
  int32_t* next;    // of a launch: next block of rows
  int32_t* rows;    // rows asked for, by cell
  uint64_t* keys;   // of every row in flight: kWnKeys
};

static size_t wn_layout(int64_t np, int d, int64_t nrows, int cus, char* w, WnLayout& l) {
  l.np = np;
  l.d = d;
  l.pivots = (int)std::min<int64_t>(std::max<int64_t>(np / 320, 1), kWnPivots);
  l.pivots1 = (l.pivots + 1) / 2;
  l.ppad = (l.pivots + kWnCols - 1) / kWnCols * kWnCols;
  l.slots = (np + kWnCols - 1) / kWnCols * kWnCols + (int64_t)kWnCols * l.pivots;
  const int64_t nk = (int64_t)l.pivots * kWnBuckets;
  const int64_t blocks = std::min<int64_t>((nrows + kWnRows - 1) / kWnRows, kWnPerCu * cus);
  l.launches = (int)((nrows + kWnStep - 1) / kWnStep);
  size_t at = 0;
  auto take = [&](auto*& p, size_t n) {
    p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(w + at);
    at = (at + n * sizeof(*p) + 255) & ~(size_t)255;
  };
  take(l.Xs, (size_t)l.slots * d);
  take(l.hs, l.slots);
  take(l.sid, l.slots);
  take(l.sd, l.slots);
  take(l.meta, l.slots / kWnCols);
  take(l.cell, np);
  take(l.d2, np);
  take(l.hist, nk);
  take(l.rhist, nk);
  take(l.pos, nk);
  take(l.rpos, nk);
  take(l.cstart, l.pivots + 1);
  take(l.Pb, (size_t)l.ppad * d);
  take(l.ph, l.ppad);
  take(l.far, kWnFarBins + 1);
  take(l.next, l.launches);
  take(l.rows, nrows);
  take(l.keys, (size_t)blocks * kWnRows * kWnKeys);
  return at;
}

// ---- the cells ------------------------------------------------------------
__device__ __forceinline__ int wn_far_bin(float d2) {  // three bits of mantissa
  return (int)(__float_as_uint(d2) >> 20) & (kWnFarBins - 1);
}

// no point in any slot, no count; the first pivots' rows, and no second ones yet
__global__ __launch_bounds__(256) void wn_init_kernel(WnLayout l, const uint16_t* __restrict__ Xb,
                                                      const float* __restrict__ half) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t e = i; e < l.slots; e += step) {
    l.sid[e] = -1;
    l.hs[e] = -INFINITY;
  }
  for (int64_t e = i; e < (int64_t)l.pivots * kWnBuckets; e += step) l.hist[e] = l.rhist[e] = 0;
  for (int64_t e = i; e < kWnFarBins + 1; e += step) l.far[e] = 0;
  for (int64_t e = i; e < l.launches; e += step) l.next[e] = 0;
  const int units = l.d / 8;
  for (int64_t e = i; e < (int64_t)l.ppad * units; e += step) {
    const int p = (int)(e / units), u = (int)(e - (int64_t)p * units);
    const int64_t id = (int64_t)min(p, l.pivots1 - 1) * l.np / l.pivots1;
    reinterpret_cast<uint4*>(l.Pb)[e] = reinterpret_cast<const uint4*>(Xb)[id * units + u];
    if (u == 0) l.ph[p] = p < l.pivots1 ? half[id] : -INFINITY;
  }
}

__device__ __forceinline__ int wn_key(int cell, float d2) {  // two bits of mantissa
  return cell * kWnBuckets + (int)((__float_as_uint(d2) >> 21) & (kWnBuckets - 1));
}

// nearest pivot of every point (the first of equally near ones); 32 rows a wave.
// FAR: of the first pivots, and counts of the distances.
template <int KS, bool FAR>
__global__ __launch_bounds__(256) void wn_assign_kernel(WnLayout l, const uint16_t* __restrict__ Xb,
                                                        const float* __restrict__ half,
                                                        int64_t row0, int64_t nrows) {
  constexpr int D = 32 * KS;
  __shared__ int bins[FAR ? kWnFarBins : 1];
  if (FAR) {
    for (int i = threadIdx.x; i < kWnFarBins; i += 256) bins[i] = 0;
    __syncthreads();
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 128 + 32 * wave;  // past np: nothing is written
  uint4 A[2][KS];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) {
    const int64_t row = min(m0 + 16 * rb + r, l.np - 1);
#pragma unroll
    for (int s = 0; s < KS; ++s)
      A[rb][s] = *reinterpret_cast<const uint4*>(Xb + row * D + 32 * s + 8 * g);
  }
  float best[2][4];
  int at[2][4];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      best[rb][v] = -INFINITY;
      at[rb][v] = 0;
    }
  const int pend = FAR ? l.pivots1 : l.pivots;
  for (int p0 = 0; p0 < pend; p0 += kWnCols) {
    floatx4 acc[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float hx = l.ph[p0 + 16 * j + r];
      acc[0][j] = acc[1][j] = floatx4{hx, hx, hx, hx};
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint4 b = *reinterpret_cast<const uint4*>(l.Pb + (int64_t)(p0 + 16 * j + r) * D +
                                                        32 * s + 8 * g);
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
          acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, A[rb][s]), __builtin_bit_cast(bf16x8, b), acc[rb][j], 0, 0,
              0);
      }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (acc[rb][j][v] > best[rb][v]) {
            best[rb][v] = acc[rb][j][v];
            at[rb][v] = p0 + 16 * j + r;
          }
  }
#pragma unroll
  for (int rb = 0; rb < 2; ++rb)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const float ob = __shfl_xor(best[rb][v], o, 64);
        const int oa = __shfl_xor(at[rb][v], o, 64);
        if (ob > best[rb][v] || (ob == best[rb][v] && oa < at[rb][v])) {
          best[rb][v] = ob;
          at[rb][v] = oa;
        }
      }
      const int64_t row = m0 + 16 * rb + 4 * g + v;
      if (r == 0 && row < l.np) {
        const float d2 = __builtin_fmaf(-2.f, best[rb][v] + half[row], 0.f);
        l.d2[row] = d2;
        if (FAR) {
          atomicAdd(&bins[wn_far_bin(d2)], 1);
          continue;
        }
        l.cell[row] = at[rb][v];
        const int key = wn_key(at[rb][v], d2);
        atomicAdd(&l.hist[key], 1);
        if (row >= row0 && row < row0 + nrows) atomicAdd(&l.rhist[key], 1);
      }
    }
  if (FAR) {
    __syncthreads();
    for (int i = threadIdx.x; i < kWnFarBins; i += 256)
      if (bins[i]) atomicAdd(&l.far[i], bins[i]);
  }
}

// the other pivots: evenly spaced among the points of the farthest bins that hold
// a quarter of the points, in the order in which the waves come
__global__ __launch_bounds__(256) void wn_pick_kernel(WnLayout l, const uint16_t* __restrict__ Xb,
                                                      const float* __restrict__ half) {
  __shared__ int part[256];
  const int t = threadIdx.x, lane = t & 63;
  constexpr int kPer = kWnFarBins / 256;
  // bins from the far end: thread t has bins [hi - kPer + 1, hi]
  const int hi = kWnFarBins - 1 - kPer * t;
  int n = 0;
  for (int i = 0; i < kPer; ++i) n += l.far[hi - i];
  part[t] = n;
  __syncthreads();
  for (int o = 1; o < 256; o <<= 1) {
    const int y = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += y;
    __syncthreads();
  }
  __shared__ int first, total;
  const int64_t want = (l.np + 3) / 4;
  const int before = part[t] - n;
  if (before < want && part[t] >= want) {  // one thread: the last one's sum is np
    int sum = before, bin = hi + 1;
    while (sum < want) sum += l.far[--bin];
    first = bin;
    total = sum;
  }
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * 256 + t;
  const bool is = i < l.np && wn_far_bin(l.d2[i]) >= first;
  const uint64_t m = __builtin_amdgcn_ballot_w64(is);
  if (!m) return;
  int base = 0;
  if (lane == 0) base = atomicAdd(&l.far[kWnFarBins], __popcll(m));
  const int64_t rank = __builtin_amdgcn_readfirstlane(base) +
                       (int)__builtin_amdgcn_mbcnt_hi(
                           (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  // of `total` ranks, those where rank * seconds / total steps up
  const int64_t seconds = l.pivots - l.pivots1;
  const int64_t q = rank * seconds / total;
  if (!is || (rank > 0 && (rank - 1) * seconds / total == q) || q >= seconds) return;
  const int p = l.pivots1 + (int)q, units = l.d / 8;
  for (int u = 0; u < units; ++u)
    reinterpret_cast<uint4*>(l.Pb)[(int64_t)p * units + u] =
        reinterpret_cast<const uint4*>(Xb)[i * units + u];
  l.ph[p] = half[i];
}

// first slot of every key, cells padded to whole tiles; first place of a key's
// rows.  One workgroup, thread p has cell p.
__global__ __launch_bounds__(kWnPivots) void wn_scan_kernel(WnLayout l) {
  __shared__ int sp[kWnPivots], sr[kWnPivots];
  const int p = threadIdx.x;
  int n = 0, nr = 0;
  if (p < l.pivots)
    for (int b = 0; b < kWnBuckets; ++b) {
      n += l.hist[p * kWnBuckets + b];
      nr += l.rhist[p * kWnBuckets + b];
    }
  const int padded = (n + kWnCols - 1) / kWnCols * kWnCols;
  sp[p] = padded;
  sr[p] = nr;
  __syncthreads();
  for (int o = 1; o < kWnPivots; o <<= 1) {
    const int y = p >= o ? sp[p - o] : 0, yr = p >= o ? sr[p - o] : 0;
    __syncthreads();
    sp[p] += y;
    sr[p] += yr;
    __syncthreads();
  }
  if (p >= l.pivots) return;
  int at = sp[p] - padded, rat = sr[p] - nr;
  l.cstart[p] = at;
  if (p == l.pivots - 1) l.cstart[l.pivots] = sp[p];
  for (int b = 0; b < kWnBuckets; ++b) {
    const int key = p * kWnBuckets + b;
    l.pos[key] = at;
    l.rpos[key] = rat;
    at += l.hist[key];
    rat += l.rhist[key];
  }
}

// every point to its slot (in any order inside a key: lists do not depend on it)
__global__ __launch_bounds__(256) void wn_scatter_kernel(WnLayout l, const uint16_t* __restrict__ Xb,
                                                         const float* __restrict__ half,
                                                         int64_t row0, int64_t nrows) {
  __shared__ int slot[256];
  const int64_t i0 = (int64_t)blockIdx.x * 256, i = i0 + threadIdx.x;
  if (i < l.np) {
    const float d2 = l.d2[i];
    const int key = wn_key(l.cell[i], d2);
    const int at = atomicAdd(&l.pos[key], 1);
    slot[threadIdx.x] = at;
    l.sid[at] = (int32_t)i;
    l.hs[at] = half[i];
    l.sd[at] = d2;
    if (i >= row0 && i < row0 + nrows) l.rows[atomicAdd(&l.rpos[key], 1)] = (int32_t)i;
  }
  __syncthreads();
  const int units = l.d / 8;
  const int64_t n = min<int64_t>(256, l.np - i0) * units;
  for (int64_t e = threadIdx.x; e < n; e += 256) {
    const int q = (int)(e / units), u = (int)(e - (int64_t)q * units);
    reinterpret_cast<uint4*>(l.Xs)[(int64_t)slot[q] * units + u] =
        reinterpret_cast<const uint4*>(Xb)[(i0 + q) * units + u];
  }
}

// range of a tile's distances; zeros in its pads.  One wave a tile.
__global__ __launch_bounds__(256) void wn_meta_kernel(WnLayout l) {
  const int lane = threadIdx.x & 63;
  const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile * kWnCols >= l.cstart[l.pivots]) return;  // whole waves, no barrier
  const int64_t at = tile * kWnCols + lane;
  const int id = l.sid[at];
  const float d = id >= 0 ? sqrtf(l.sd[at]) : 0.f;
  float a = id >= 0 ? d : INFINITY, b = d;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a = fminf(a, __shfl_xor(a, o, 64));
    b = fmaxf(b, __shfl_xor(b, o, 64));
  }
  if (lane == 0) l.meta[tile] = WnMeta{a, b, l.cell[id], 0};  // a tile starts with a point
  if (id < 0)
    for (int u = 0; u < l.d / 8; ++u)
      reinterpret_cast<uint4*>(l.Xs)[at * (l.d / 8) + u] = make_uint4(0, 0, 0, 0);
}

// ---- the lists --------------------------------------------------------------
// 64 lanes x 16 (or 4) bytes from global memory to LDS at `dst` + 16 (4) * lane.
// As asm, so that the compiler does not wait for it before every LDS read that
// might alias; the kernel waits once, before the tile's barrier.
__device__ __forceinline__ void wn_copy16(const void* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
               : "memory", "m0");
}
__device__ __forceinline__ void wn_copy4(const void* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src)
               : "memory", "m0");
}

// the tile of points from n0 to LDS at `dst`, by the workgroup
template <int KS>
__device__ __forceinline__ void wn_copy_tile(const uint16_t* X, const float* half,
                                             const int32_t* ids, int64_t n0, uint32_t dst, int wave,
                                             int lane) {
  using W = WnTile<KS>;
#pragma unroll
  for (int i = 0; i < (W::UNITS / 64 + kWnWaves - 1) / kWnWaves; ++i) {
    const int u0 = 64 * (kWnWaves * i + wave);
    if (u0 < W::UNITS) {
      const int u = u0 + lane, c = u / W::CPR, q = (u % W::CPR) ^ (c & W::SWM);
      wn_copy16(X + (n0 + c) * (32 * KS) + 8 * q, dst + 16u * (uint32_t)u0);
    }
  }
  if (wave == 0) wn_copy4(half + n0 + lane, dst + 16u * W::UNITS);
  if (wave == 1 && ids) wn_copy4(ids + n0 + lane, dst + 16u * W::UNITS + 256u);
}

struct WnArgs {
  WnLayout l;
  const uint16_t* Xb;  // np x d
  const float* half;   // np
  int64_t row0;        // of the outputs
  int64_t first, nq;   // of l.rows
  int launch;
  int k;
  int32_t* ids_out;
  float* dists_out;
};

// A workgroup of four waves owns 32 rows a wave (their operands in registers, so
// that a 16-byte operand read of a tile feeds two MFMAs: with 16 rows the LDS
// reads take twice the MFMAs' time).  Tiles come straight into an LDS ring of two
// tiles (16-byte units XOR-swizzled per point), one barrier a tile; two
// workgroups a compute unit, since a wave's points to pick differ from tile to tile
// and a workgroup waits for its slowest wave (one of eight waves, three tiles to a
// barrier: 4.0 ms at 160k x 128, two: 2.6).  A point nearer than its row's
// threshold (the k-th best of the row's list) goes to the wave's queue -- writes
// only, no round trip through LDS -- and 64 at a time to the rows' buffers.  A
// buffer is sorted across the wave and merged with its row's sorted list when it
// is full, in all rows at tiles 0, 1, 2, 4, ... times 1.8 (a point enters the k
// best of n seen with probability k / n, so that a buffer of 64 lasts while n
// grows by a factor), and after each list of tiles.  Lists and buffers lie in global
// memory, 1 KiB a row, touched by the row's wave only; the workgroups are as many as
// the card holds at once and take block after block of rows, so they stay in L2.
// Points come in any order of ids, so one at the k-th best distance
// passes if its id is lower.
template <int KS>
__global__ __launch_bounds__(64 * kWnWaves, 2) void knn_whole_kernel(WnArgs a) {
  using W = WnTile<KS>;
  constexpr int D = 32 * KS;
  constexpr int ROWS = kWnRows;
  constexpr uint64_t kNone = ~0ull;
  __shared__ __attribute__((aligned(16))) uint4 ring[2 * W::SLOT];
  __shared__ uint2 qe[kWnWaves][kWnQueue];  // a wave's queue: product, row << 27 | id
  __shared__ int cnt[ROWS];
  __shared__ float thr[ROWS];  // -(k-th best distance) / 2 + |q|^2 / 2
  __shared__ float kth[ROWS];  // k-th best distance
  __shared__ int kid[ROWS];    // its id
  __shared__ float hrow[ROWS];
  __shared__ int rid[ROWS];
  __shared__ float dmin[kWnPivots], dmax[kWnPivots];  // of the block's rows from a pivot
  __shared__ int list[kWnList];                       // tiles to visit
  __shared__ int listed;  // their number; before that, the block
  __shared__ float wk[kWnWaves];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int lrow0 = 32 * wave;  // the wave's rows in the workgroup
  const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_void_t*)ring;
  constexpr uint32_t kHalf = 16u * W::SLOT;
  const int ntile = a.l.cstart[a.l.pivots] / kWnCols;
  uint64_t* const keys = a.l.keys + ((int64_t)blockIdx.x * ROWS + lrow0) * kWnKeys + lane;
  while (true) {
    __syncthreads();  // every wave is done with the block before
    if (t == 0) listed = atomicAdd(&a.l.next[a.launch], 1);
    __syncthreads();
    const int64_t j0 = (int64_t)listed * ROWS;
    if (j0 >= a.nq) break;
    const int last = (int)min<int64_t>(ROWS, a.nq - j0) - 1;  // the block's last row
    for (int i = t; i < ROWS; i += 64 * kWnWaves) {
      const int id = a.l.rows[a.first + j0 + min(i, last)];
      rid[i] = id;
      hrow[i] = a.half[id];
      cnt[i] = 0;
      // nothing passes in a row past the end; pads (-inf) pass in none
      thr[i] = i <= last ? -FLT_MAX : INFINITY;
      kth[i] = i <= last ? INFINITY : 0.f;
      kid[i] = INT_MAX;
    }
    for (int i = t; i < a.l.pivots; i += 64 * kWnWaves) {
      reinterpret_cast<uint32_t*>(dmin)[i] = 0x7f800000u;
      reinterpret_cast<uint32_t*>(dmax)[i] = 0u;
    }
    __syncthreads();
    uint4 A[2][KS];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t row = rid[lrow0 + 16 * rb + r];
#pragma unroll
      for (int s = 0; s < KS; ++s)
        A[rb][s] = *reinterpret_cast<const uint4*>(a.Xb + row * D + 32 * s + 8 * g);
    }
#pragma unroll 4
    for (int i = 0; i < 32; ++i) keys[i * kWnKeys] = kNone;
    // the rows' distances from the pivots
    for (int p0 = 0; p0 < a.l.ppad; p0 += kWnCols) {
      __syncthreads();
      wn_copy_tile<KS>(a.l.Pb, a.l.ph, nullptr, p0, ring0, wave, lane);
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
      const float* ht = reinterpret_cast<const float*>(ring + W::UNITS);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float hx = ht[16 * j + r];
        floatx4 acc[2];
        acc[0] = acc[1] = floatx4{hx, hx, hx, hx};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const uint4 x = ring[(16 * j + r) * W::CPR + ((4 * s + g) ^ (r & W::SWM))];
#pragma unroll
          for (int rb = 0; rb < 2; ++rb)
            acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[rb][s]),
                                                              __builtin_bit_cast(bf16x8, x),
                                                              acc[rb], 0, 0, 0);
        }
        float lo = -INFINITY, hi = INFINITY;  // halves of negated distances
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float x = acc[rb][v] + hrow[lrow0 + 16 * rb + 4 * g + v];
            lo = fmaxf(lo, x);
            hi = fminf(hi, x);
          }
        lo = fmaxf(lo, __shfl_xor(lo, 16, 64));
        hi = fminf(hi, __shfl_xor(hi, 16, 64));
        lo = fmaxf(lo, __shfl_xor(lo, 32, 64));
        hi = fminf(hi, __shfl_xor(hi, 32, 64));
        const int p = p0 + 16 * j + r;
        if (g == 0 && p < a.l.pivots) {  // order of bits = order of values, none negative
          atomicMin(reinterpret_cast<uint32_t*>(dmin) + p,
                    __float_as_uint(__builtin_fmaf(-2.f, lo, 0.f)));
          atomicMax(reinterpret_cast<uint32_t*>(dmax) + p,
                    __float_as_uint(__builtin_fmaf(-2.f, hi, 0.f)));
        }
      }
    }
    __syncthreads();
    for (int i = t; i < a.l.pivots; i += 64 * kWnWaves) {
      dmin[i] = sqrtf(dmin[i]);
      dmax[i] = sqrtf(dmax[i]);
    }
    float th[2][4];
    auto load_thr = [&]() {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) th[rb][v] = thr[lrow0 + 16 * rb + 4 * g + v];
    };
    load_thr();
    // list and buffer (c entries) of row i of the wave, and their merge
    auto take = [&](int i, int c, uint64_t& fresh, uint64_t& old) {
      fresh = lane < c ? keys[i * kWnKeys + 64] : kNone;
      old = keys[i * kWnKeys];
    };
    auto merge = [&](int i, uint64_t fresh, uint64_t old) {
      fresh = sort_keys_desc(fresh, lane);
      const uint64_t key = merge_keys_asc(fresh < old ? fresh : old, lane);
      keys[i * kWnKeys] = key;
      const uint32_t kd = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(key >> 32), a.k - 1);
      const int ki = __builtin_amdgcn_readlane((int)(uint32_t)key, a.k - 1);
      if (lane == 0) {
        cnt[lrow0 + i] = 0;
        if (kd != 0xffffffffu) {
          kth[lrow0 + i] = __uint_as_float(kd);
          kid[lrow0 + i] = ki;
          thr[lrow0 + i] = -0.5f * __uint_as_float(kd) - hrow[lrow0 + i];
        }
      }
    };
    // the lanes of mask m queue point id of row i with their product x
    int queued = 0;
    auto push = [&](uint64_t m, float x, int i, int id) {
      if (__builtin_expect(m == 0, 1)) return;
      const int at = queued + (int)__builtin_amdgcn_mbcnt_hi(
                                  (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      if (__builtin_amdgcn_inverse_ballot_w64(m))
        qe[wave][at] = make_uint2(__float_as_uint(x), (uint32_t)i << 27 | (uint32_t)id);
      queued += __popcll(m);
    };
    // the queued points (but a row itself) into their rows' buffers, 64 at a time
    auto drain = [&]() {
      wave_sync();
      while (queued > 0) {
        const int n = min(queued, 64);
        queued -= n;
        bool left = lane < n;
        uint64_t key = kNone;
        int i = -1;
        if (left) {
          const uint2 e = qe[wave][queued + lane];
          i = (int)(e.y >> 27);
          const uint32_t id = e.y & 0x7ffffffu;
          // + 0: a distance of zero is +0, as a key too
          const float dist = __builtin_fmaf(-2.f, __uint_as_float(e.x) + hrow[lrow0 + i], 0.f);
          key = (uint64_t)__float_as_uint(dist) << 32 | id;
          left = (int)id != rid[lrow0 + i];
        }
        while (true) {
          if (left) {
            const int at = atomicAdd(&cnt[lrow0 + i], 1);
            if (at < 64) {
              (keys - lane)[i * kWnKeys + 64 + at] = key;
              left = false;
            }
          }
          wave_sync();
          uint64_t full = __builtin_amdgcn_ballot_w64(left);
          if (!full) break;
          __builtin_amdgcn_s_waitcnt(0x0f70);  // the buffers' entries are written
          while (full) {
            const int f = __builtin_amdgcn_readlane(i, __builtin_ctzll(full));
            uint64_t fresh, old;
            take(f, 64, fresh, old);
            merge(f, fresh, old);
            full &= ~__builtin_amdgcn_ballot_w64(i == f);
          }
          wave_sync();
          load_thr();
        }
      }
    };
    // every row's buffer into its list, the next row's keys in flight
    auto flush_all = [&]() {
      drain();
      __builtin_amdgcn_s_waitcnt(0x0f70);
      wave_sync();
      const int c = lane < 32 ? min(cnt[lrow0 + lane], 64) : 0;
      uint64_t todo = __builtin_amdgcn_ballot_w64(c > 0);
      int i = 0;
      uint64_t fresh = 0, old = 0;
      if (todo) {
        i = __builtin_ctzll(todo);
        take(i, __builtin_amdgcn_readlane(c, i), fresh, old);
      }
      while (todo) {
        todo &= todo - 1;
        const int i1 = todo ? __builtin_ctzll(todo) : i;
        uint64_t fresh1, old1;
        take(i1, __builtin_amdgcn_readlane(c, i1), fresh1, old1);
        merge(i, fresh, old);
        i = i1;
        fresh = fresh1;
        old = old1;
      }
      wave_sync();
      load_thr();
    };
    // one tile: products, then the points that pass.  All its operands are asked
    // for before the first product: left to itself the compiler reads them between
    // the products and waits for each (160k x 128 uniform 17.5 -> 19.1 ms).
    auto tile = [&](const uint4* Bt) {
      const float* ht = reinterpret_cast<const float*>(Bt + W::UNITS);
      uint4 b[KS][4];
      float hx[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) hx[j] = ht[16 * j + r];
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          b[s][j] = Bt[(16 * j + r) * W::CPR + ((4 * s + g) ^ (r & W::SWM))];
      __builtin_amdgcn_sched_barrier(0);
      floatx4 acc[2][4];
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb)
            acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, A[rb][s]), __builtin_bit_cast(bf16x8, b[s][j]),
                s ? acc[rb][j] : floatx4{hx[j], hx[j], hx[j], hx[j]}, 0, 0, 0);
      int idx[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        idx[j] = reinterpret_cast<const int*>(Bt + W::UNITS + 16)[16 * j + r];
      asm volatile("" ::: "memory");  // the reads stay here
      // points that pass, block (rb, v) by block; a block that the queue may
      // have no room for (the first tiles) is left for the loop below.  What
      // is done with them lies out of line: a tile's branches fall through
      // unless a point passes
      uint32_t left = 0;
      // of lanes whose products are at least a row's threshold, those whose
      // point precedes the k-th best in (distance, id)
      auto nearer = [&](uint64_t m, float x, float tb, int i, int id) {
        const uint64_t equal = __builtin_amdgcn_ballot_w64(x == tb) & m;
        if (__builtin_expect(equal == 0, 1)) return m;
        return m & ~(equal & __builtin_amdgcn_ballot_w64(id >= kid[lrow0 + i]));
      };
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          uint64_t m[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            m[j] = __builtin_amdgcn_ballot_w64(acc[rb][j][v] >= th[rb][v]);
          if (__builtin_expect(((m[0] | m[1]) | (m[2] | m[3])) != 0, 0)) {
            if (queued > kWnQueue - 256) {
              left |= 1u << (4 * rb + v);
            } else {
              int i = 4 * g;
              asm volatile("" : "+v"(i));  // formed here, not kept in registers for every block
              i += 16 * rb + v;
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (m[j])
                  push(nearer(m[j], acc[rb][j][v], th[rb][v], i, idx[j]), acc[rb][j][v], i, idx[j]);
            }
          }
        }
      if (__builtin_expect(queued >= 64, 0)) drain();
      // a rolled loop, draining as it goes; the block's values are picked by a
      // scalar branch
      while (__builtin_expect(left != 0, 0)) {
        const int q = __builtin_ctz(left);
        left &= left - 1;
        float x[4], tb = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (e == q) {
            tb = th[e >> 2][e & 3];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = acc[e >> 2][j][e & 3];
          }
        const int i = 16 * (q >> 2) + 4 * g + (q & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint64_t m = __builtin_amdgcn_ballot_w64(x[j] >= tb);
          push(nearer(m, x[j], tb, i, idx[j]), x[j], i, idx[j]);
        }
        drain();
      }
    };
    // Phase 0: the tiles of the block's own cells.  1: those with a row inside
    // their range, where most rows that are far from their own cells' points find
    // theirs.  2: those within the k-th best distances of some wave's rows, so
    // that a few rows without near points so far do not have the block look at
    // everything.  3: what is left within every row's.  kWnList tiles at a time.
    const int own0 = a.l.cstart[a.l.cell[rid[0]]] / kWnCols;
    const int own1 = a.l.cstart[a.l.cell[rid[last]] + 1] / kWnCols;
    int seen = 0, next = 0;
    float above = 0.f, bound = 0.f;  // tiles of a phase: above < distance <= bound
    for (int phase = 0; phase < 4; ++phase) {
      const int hi = phase ? ntile : own1;
      if (phase == 3) above = bound;
      for (int c0 = phase ? 0 : own0; c0 < hi; c0 += kWnList) {
        if (phase >= 2) {  // the largest k-th best distance of the wave's rows
          float d = kth[lrow0 + (lane & 31)];
#pragma unroll
          for (int o = 16; o > 0; o >>= 1) d = fmaxf(d, __shfl_xor(d, o, 64));
          if (lane == 0) wk[wave] = d;
        }
        if (t == 0) listed = 0;
        __syncthreads();  // wk; every wave is done with the list and the ring
        if (phase == 3 || (phase == 2 && c0 == 0)) {
          float d = wk[0];
#pragma unroll
          for (int w = 1; w < kWnWaves; ++w) d = phase == 2 ? fminf(d, wk[w]) : fmaxf(d, wk[w]);
          // distances as rounded: a margin of a ten-thousandth and 0.01
          bound = sqrtf(d) * 1.0002f + 0.01f;
          if (phase == 3 && bound <= above) break;
        }
        for (int c = t; c < kWnList; c += 64 * kWnWaves) {
          const int tl = c0 + c;
          bool keep = tl < hi;
          if (phase && keep) {
            const WnMeta m = a.l.meta[tl];
            const float near = fmaxf(dmin[m.cell] - m.b, m.a - dmax[m.cell]);
            keep = (tl < own0 || tl >= own1) &&
                   (phase == 1 ? near <= 0.f : near > above && !(near > bound));
          }
          const uint64_t km = __builtin_amdgcn_ballot_w64(keep);
          int base = 0;
          if (lane == 0 && km) base = atomicAdd(&listed, __popcll(km));
          base = __builtin_amdgcn_readfirstlane(base);
          if (keep)
            list[base + (int)__builtin_amdgcn_mbcnt_hi(
                            (uint32_t)(km >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)km, 0u))] = tl;
        }
        __syncthreads();
        const int n = __builtin_amdgcn_readfirstlane(listed);
        if (n == 0) continue;
        auto copy_tile = [&](int i, uint32_t dst) {
          wn_copy_tile<KS>(a.l.Xs, a.l.hs, a.l.sid,
                           (int64_t)__builtin_amdgcn_readfirstlane(list[i]) * kWnCols, dst, wave,
                           lane);
        };
        copy_tile(0, ring0);
        uint32_t here = 0;  // the ring's half that holds the tile
        for (int i = 0; i < n; ++i) {
          // the tile's copies have landed (each wave waits for its own) and
          // every wave is done with the other half
          __builtin_amdgcn_s_waitcnt(0x0f70);
          __syncthreads();
          if (i + 1 < n) copy_tile(i + 1, ring0 + (kHalf - here));
          tile(ring + here / 16);
          if (seen >= next) {
            flush_all();
            next = seen + 1 + 8 * seen / 10;
          }
          ++seen;
          here = kHalf - here;
        }
        flush_all();
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll 4
    for (int i = 0; i < 32; ++i) {
      const uint64_t key = keys[i * kWnKeys];
      if (lrow0 + i <= last && lane < a.k) {
        const int64_t o = ((int64_t)rid[lrow0 + i] - a.row0) * a.k + lane;
        a.ids_out[o] = (int32_t)(uint32_t)key;
        if (a.dists_out) a.dists_out[o] = __uint_as_float((uint32_t)(key >> 32));
      }
    }
  }
}

size_t knn_whole_bytes(int64_t np, int d, int64_t nrows, int cus) {
  WnLayout l;
  return wn_layout(np, d, nrows, cus, nullptr, l);
}

template <int KS>
static void launch_wn(WnArgs a, int64_t nrows, int cus, int32_t* ids, float* dists,
                      hipStream_t st) {
  const WnLayout& l = a.l;
  hipLaunchKernelGGL(wn_init_kernel, dim3(1024), dim3(256), 0, st, l, a.Xb, a.half);
  const dim3 by128((unsigned)((l.np + 127) / 128)), by256((unsigned)((l.np + 255) / 256));
  hipLaunchKernelGGL((wn_assign_kernel<KS, true>), by128, dim3(256), 0, st, l, a.Xb, a.half, a.row0,
                     nrows);
  if (l.pivots > l.pivots1)
    hipLaunchKernelGGL(wn_pick_kernel, by256, dim3(256), 0, st, l, a.Xb, a.half);
  hipLaunchKernelGGL((wn_assign_kernel<KS, false>), by128, dim3(256), 0, st, l, a.Xb, a.half, a.row0,
                     nrows);
  hipLaunchKernelGGL(wn_scan_kernel, dim3(1), dim3(kWnPivots), 0, st, l);
  hipLaunchKernelGGL(wn_scatter_kernel, by256, dim3(256), 0, st, l, a.Xb, a.half, a.row0, nrows);
  hipLaunchKernelGGL(wn_meta_kernel, dim3((unsigned)((l.slots / kWnCols + 3) / 4)), dim3(256), 0, st,
                     l);
  a.ids_out = ids;
  a.dists_out = dists;
  for (int i = 0; i < l.launches; ++i) {
    a.launch = i;
    a.first = i * kWnStep;
    a.nq = std::min(kWnStep, nrows - a.first);
    hipLaunchKernelGGL(
        knn_whole_kernel<KS>,
        dim3((unsigned)std::min<int64_t>((a.nq + kWnRows - 1) / kWnRows, kWnPerCu * cus)),
        dim3(64 * kWnWaves), 0, st, a);
  }
}

hipError_t launch_knn_whole(const uint16_t* Xb, const float* half, int64_t np, int d, int64_t row0,
                            int64_t nrows, int k, int cus, void* work, int32_t* ids, float* dists,
                            hipStream_t st) {
  if (nrows <= 0) return hipSuccess;
  WnArgs a{};
  wn_layout(np, d, nrows, cus, static_cast<char*>(work), a.l);
  a.Xb = Xb;
  a.half = half;
  a.row0 = row0;
  a.k = k;
  switch (d / 32) {
    case 1: launch_wn<1>(a, nrows, cus, ids, dists, st); break;
    case 2: launch_wn<2>(a, nrows, cus, ids, dists, st); break;
    case 3: launch_wn<3>(a, nrows, cus, ids, dists, st); break;
    case 4: launch_wn<4>(a, nrows, cus, ids, dists, st); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace rte
