// Exact kNN of a base against itself on FP32 MFMA, for building the search
// graph.  The reference has no graph builder (graph.cu:117-121 leaves a TODO;
// its .nsw files come from an external tool, flags.cpp:14).
//
// Distances are |q|^2 + |x|^2 - 2 q.x with q.x from v_mfma_f32_16x16x4_f32
// tiles.  For integer-valued data with |x|^2 < 2^24 (the 1M x 128 workload:
// values 0..255, d = 128) every term is an exact FP32 integer, so the lists
// equal the FP64 ones, ties broken by id.
//
// Tiling: a workgroup of 8 waves owns 128 query rows (16 per wave, their
// operands in registers as float4 per 16 k) and walks all base points in
// tiles of 64, double-buffered through LDS transposed ([point][k]).  Every
// tile gives a wave 16 x 64 distances; a distance enters its row's list only
// if it beats the row's current k-th best (kept in registers), so after the
// first tiles almost nothing is inserted.  Lists live in LDS, one per row,
// sorted by (dist, id); an insertion is done by the whole wave (lane i =
// list position i): the position is a ballot count and the tail shifts one
// lane up.  Points arrive in increasing id order, so a tie never displaces
// an earlier id.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "knn.h"
#include "search_impl.h"

namespace rte {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kKnnRows = 128;  // rows per workgroup
constexpr int kKnnCols = 64;   // base points per tile

// |x|^2 per row (FP32, dims in order) and, for the whole-number kernel, the
// bf16 copy of the rows (npad x d, zero past np), -|x|^2 / 2 (-inf past np) and
// what rules that kernel out: flag bits are set when a value is no whole number
// of magnitude <= 256 or a row's norm too large for exact sums
// (knn_whole_numbers).  One workgroup takes 64 rows, staged through LDS so that
// the base is read in whole lines once; bound by that traffic.
__global__ __launch_bounds__(256) void row_norms_kernel(const float* __restrict__ X, int64_t np,
                                                        int d, int64_t stride, int64_t npad,
                                                        float* __restrict__ norms,
                                                        uint16_t* __restrict__ Xb,
                                                        float* __restrict__ half,
                                                        uint32_t* __restrict__ flag) {
  __shared__ float rows[64][128 + 1];
  const int t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * 64;
  uint32_t bad = 0;
  for (int e = t; e < 64 * (d / 2); e += 256) {
    const int r = e / (d / 2), c = 2 * (e - r * (d / 2));
    float2 v = make_float2(0.f, 0.f);
    if (r0 + r < np) v = *reinterpret_cast<const float2*>(X + (r0 + r) * stride + c);
    rows[r][c] = v.x;
    rows[r][c + 1] = v.y;
    const bool whole = v.x == rintf(v.x) && fabsf(v.x) <= 256.f && v.y == rintf(v.y) &&
                       fabsf(v.y) <= 256.f;
    bad |= whole ? 0u : kKnnNotWhole;
    bad |= v.x < 0.f || v.y < 0.f ? kKnnNegative : 0u;
    // whole numbers up to 256 are bf16 values: the upper halves are exact
    if (Xb && r0 + r < npad)
      reinterpret_cast<uint32_t*>(Xb)[((r0 + r) * d + c) >> 1] =
          (__float_as_uint(v.x) >> 16) | (__float_as_uint(v.y) & 0xffff0000u);
  }
  __syncthreads();
  if (t < 64 && r0 + t < npad) {
    float s = 0.f;
    for (int j = 0; j < d; ++j) s = __builtin_fmaf(rows[t][j], rows[t][j], s);
    if (r0 + t < np) {
      norms[r0 + t] = s;
      bad |= s < 8388608.f ? 0u : kKnnLarge;        // 2^23
      bad |= s < 4194304.f ? 0u : kKnnLargeSigned;  // 2^22
    }
    if (half) half[r0 + t] = r0 + t < np ? -0.5f * s : -INFINITY;
  }
  for (int o = 32; o > 0; o >>= 1) bad |= __shfl_xor(bad, o, 64);
  if (flag && (t & 63) == 0 && bad) atomicOr(flag, bad);
}

template <int S>  // S = d / 16 (float4 operands per lane)
__global__ __launch_bounds__(512) void knn_kernel(const float* __restrict__ X, int64_t np, int d,
                                                  int64_t stride, const float* __restrict__ norms,
                                                  int64_t row0, int64_t nq, int k,
                                                  int32_t* __restrict__ ids_out,
                                                  float* __restrict__ dists_out) {
  constexpr int LDB = 16 * S + 4;  // floats per point in LDS (padding breaks bank conflicts)
  __shared__ __attribute__((aligned(16))) float Bt[2][kKnnCols * LDB];
  __shared__ float Ld[kKnnRows * kKnnK];
  __shared__ int Li[kKnnRows * kKnnK];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int64_t mrow0 = row0 + (int64_t)blockIdx.x * kKnnRows + 16 * wave;  // wave's first row
  // lists empty
  for (int i = t; i < kKnnRows * kKnnK; i += 512) {
    Ld[i] = INFINITY;
    Li[i] = 0x7fffffff;
  }
  // A operands: row mrow0 + r, dims 16 s + 4 g .. + 3
  float4 A[S];
  {
    const int64_t row = mrow0 + r;
    const bool ok = row < row0 + nq;
#pragma unroll
    for (int s = 0; s < S; ++s)
      A[s] = ok ? *reinterpret_cast<const float4*>(X + row * stride + 16 * s + 4 * g)
                : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // lane (r, g) holds distances of rows 4 g + v (v < 4): their norms and thresholds
  float qn[4], thr[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int64_t row = mrow0 + 4 * g + v;
    qn[v] = row < row0 + nq ? norms[row] : 0.f;
    thr[v] = INFINITY;
  }
  // tile loader: 64 points x d floats = 16 S float4 per point; thread t moves
  // float4 chunks t + 512 i
  constexpr int CH = kKnnCols * 4 * S;  // float4 chunks per tile
  constexpr int PER = (CH + 511) / 512;
  float4 pre[PER];
  auto chunk_src = [&](int64_t n0, int c, bool& ok) -> const float4* {
    const int p = c / (4 * S), q4 = c % (4 * S);
    ok = n0 + p < np;
    return reinterpret_cast<const float4*>(X + (n0 + p) * stride + 4 * q4);
  };
  const int64_t ntile = (np + kKnnCols - 1) / kKnnCols;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = t + 512 * i;
    bool ok = false;
    const float4* src = c < CH ? chunk_src(0, c, ok) : nullptr;
    pre[i] = (c < CH && ok) ? *src : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int c = t + 512 * i;
    if (c < CH) {
      const int p = c / (4 * S), q4 = c % (4 * S);
      *reinterpret_cast<float4*>(&Bt[0][p * LDB + 4 * q4]) = pre[i];
    }
  }
  __syncthreads();
  for (int64_t tile = 0; tile < ntile; ++tile) {
    const int64_t n0 = tile * kKnnCols;
    const int buf = (int)(tile & 1);
    const int64_t nn = tile + 1 < ntile ? n0 + kKnnCols : 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = t + 512 * i;
      bool ok = false;
      const float4* src = c < CH ? chunk_src(nn, c, ok) : nullptr;
      pre[i] = (c < CH && ok) ? *src : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    floatx4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const float a4[4] = {A[s].x, A[s].y, A[s].z, A[s].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 b4 = *reinterpret_cast<const float4*>(&Bt[buf][(16 * j + r) * LDB + 16 * s + 4 * g]);
        const float b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[c], b[c], acc[j], 0, 0, 0);
      }
    }
    // distances: lane holds rows 4 g + v, points n0 + 16 j + r
    float xn[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t col = n0 + 16 * j + r;
      xn[j] = col < np ? norms[col] : 0.f;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t row = mrow0 + 4 * g + v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t col = n0 + 16 * j + r;
        const float dist = __builtin_fmaf(-2.f, acc[j][v], qn[v] + xn[j]);
        const bool pass = col < np && col != row && dist < thr[v];
        uint64_t m = __ballot(pass);
        while (m) {  // wave-uniform: one insertion per candidate, lowest lane first
          const int src = __ffsll((unsigned long long)m) - 1;
          m &= m - 1;
          const float cd = __shfl(dist, src, 64);
          const int ci = (int)(n0 + 16 * j + (src & 15));
          const int lrow = 16 * wave + 4 * (src >> 4) + v;  // row in the workgroup
          float* ld = Ld + lrow * kKnnK;
          int* li = Li + lrow * kKnnK;
          const float ed = ld[lane];
          const int ei = li[lane];
          const bool less = ed < cd || (ed == cd && ei < ci);
          const int pos = __popcll(__ballot(less));
          const float pd = __shfl_up(ed, 1, 64);
          const int pi = __shfl_up(ei, 1, 64);
          if (pos < kKnnK && lane >= pos) {
            ld[lane] = lane == pos ? cd : pd;
            li[lane] = lane == pos ? ci : pi;
          }
          // the row's k-th best, to the 16 lanes holding the row
          const float kth = __shfl(lane == pos ? cd : (lane > pos ? pd : ed), k - 1, 64);
          if ((lane >> 4) == (src >> 4)) thr[v] = kth;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = t + 512 * i;
      if (c < CH) {
        const int p = c / (4 * S), q4 = c % (4 * S);
        *reinterpret_cast<float4*>(&Bt[buf ^ 1][p * LDB + 4 * q4]) = pre[i];
      }
    }
    __syncthreads();
  }
  // lists out: row lrow = wave's 16 rows, lanes = positions
  for (int lr = 0; lr < 16; ++lr) {
    const int lrow = 16 * wave + lr;
    const int64_t row = mrow0 + lr;
    if (row < row0 + nq && lane < k) {
      ids_out[(row - row0) * k + lane] = Li[lrow * kKnnK + lane];
      if (dists_out) dists_out[(row - row0) * k + lane] = Ld[lrow * kKnnK + lane];
    }
  }
}

// ---- whole-number data ----------------------------------------------------
// kNN lists of data whose values are whole numbers of magnitude <= 256 (image
// descriptors are bytes): they are bf16 values, so one bf16 MFMA product of 16
// times the FP32 rate gives the same numbers.  The accumulator starts at
// -(|q|^2 + |x|^2) / 2 and ends at -dist / 2.  With norms below 2^23 and no
// negative value (below 2^22 with negative ones) every partial sum is a
// multiple of 1/2 below 2^23 in magnitude: exact in FP32 in any order, and
// equal to what the FP32 kernel computes.
//
// A workgroup of 8 waves owns 256 rows, 32 per wave (their operands in
// registers), so that a 16-byte operand read of the tile feeds two MFMAs: with
// 16 rows the LDS reads take twice the MFMAs' time.  Tiles of 64 points come
// straight into an LDS ring of two groups of four (16-byte units XOR-swizzled
// per point), one barrier a group: a wave's points to pick differ from tile to
// tile, and with a barrier every tile each tile took as long as its slowest wave
// and the waves of a SIMD were all at the matrix unit or all away from it.  A
// point nearer than its row's threshold (the k-th best of the row's list) goes
// to the wave's queue -- writes only, no round trip through LDS -- and 64 at a
// time to the rows' buffers.  A buffer is sorted across the wave and merged
// with its row's sorted list when it is full, and in all rows at tiles 0, 1, 3,
// 6, ... times 1.7: a point enters the k best of n seen with probability k / n,
// so that a buffer of 64 lasts while n grows by a factor.  Lists and buffers lie
// in global memory, 1 KiB a row, touched by the row's wave only; the workgroups
// are as many as the card holds at once and take block after block of rows, so
// they stay in L2.
//
// 160k x 128, k = 64: 13.8 ms, 16.5 with two tiles in LDS and a barrier a tile.
// 5 ms of it are products and operand reads, the rest points that pass.
constexpr int kWnQueue = 416;  // queued points per wave: a block's 256 and some
constexpr int kWnGroup = 4;    // tiles between barriers
constexpr int kWnKeys = 128;   // of a row: 64 list, 64 buffer

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void global_void_t;

// compare-exchange of 64-bit keys at lane distance SUB: ascending, or
// descending where DESC(lane) holds
template <int SUB>
__device__ __forceinline__ uint64_t cas_key(uint64_t k, int lane, bool want_larger) {
  const uint32_t lo = (uint32_t)xor_lane<SUB>((int)(uint32_t)k, lane);
  const uint32_t hi = (uint32_t)xor_lane<SUB>((int)(uint32_t)(k >> 32), lane);
  const uint64_t p = ((uint64_t)hi << 32) | lo;
  return (p > k) == want_larger ? p : k;
}
template <int STEP, int SUB>
__device__ __forceinline__ uint64_t sort_keys_step(uint64_t k, int lane) {
  // pairs of a step are descending where (lane & 2 * STEP) == 0
  k = cas_key<SUB>(k, lane, ((lane & SUB) == 0) == ((lane & (2 * STEP)) == 0));
  if constexpr (SUB > 1) return sort_keys_step<STEP, SUB / 2>(k, lane);
  return k;
}
template <int STEP = 1>
__device__ __forceinline__ uint64_t sort_keys_desc(uint64_t k, int lane) {
  k = sort_keys_step<STEP, STEP>(k, lane);
  if constexpr (STEP < 32) return sort_keys_desc<STEP * 2>(k, lane);
  return k;
}
template <int SUB = 32>
__device__ __forceinline__ uint64_t merge_keys_asc(uint64_t k, int lane) {
  k = cas_key<SUB>(k, lane, (lane & SUB) != 0);
  if constexpr (SUB > 1) return merge_keys_asc<SUB / 2>(k, lane);
  return k;
}

template <int KS>  // d / 32
struct WnTile {
  static constexpr int CPR = 4 * KS;            // 16-byte units per point
  static constexpr int SWM = (CPR & -CPR) - 1;  // 3, 7, 3, 15
  static constexpr int UNITS = kKnnCols * CPR;  // per tile
  static constexpr int SLOT = UNITS + 16;       // and 64 floats: -|x|^2 / 2
};

// 64 lanes x 16 (or 4) bytes from global memory to LDS at `dst` + 16 (4) * lane.
// As asm, so that the compiler does not wait for it before every LDS read that
// might alias; the kernel waits once, before the group's barrier.
__device__ __forceinline__ void wn_copy16(const void* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
               : "memory", "m0");
}
__device__ __forceinline__ void wn_copy4(const void* src, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src)
               : "memory", "m0");
}

// the kWnGroup tiles from `tile` (past the last: the last again, never read)
template <int KS, int NW>
__device__ __forceinline__ void wn_copy_group(const uint16_t* Xb, const float* half, int64_t tile,
                                              int64_t ntile, uint32_t dst, int wave, int lane) {
  using W = WnTile<KS>;
#pragma unroll 1
  for (int j = 0; j < kWnGroup; ++j) {
    const int64_t n0 = min(tile + j, ntile - 1) * kKnnCols;
    const uint32_t at = dst + 16u * (uint32_t)(j * W::SLOT);
#pragma unroll
    for (int i = 0; i < (W::UNITS / 64 + NW - 1) / NW; ++i) {
      const int u0 = 64 * (NW * i + wave);
      if (u0 < W::UNITS) {
        const int u = u0 + lane, c = u / W::CPR, q = (u % W::CPR) ^ (c & W::SWM);
        wn_copy16(Xb + (n0 + c) * (32 * KS) + 8 * q, at + 16u * (uint32_t)u0);
      }
    }
    if (wave == j % NW) wn_copy4(half + n0 + lane, at + 16u * W::UNITS);
  }
}

struct WnArgs {
  const uint16_t* Xb;  // npad x d
  const float* half;   // npad
  int64_t np, npad;    // npad: a multiple of 64
  int64_t row0, nq;
  int k;
  uint64_t* keys;  // gridDim x 32 NW rows x kWnKeys (distance bits << 32 | id), lists ascending
  int32_t* ids_out;
  float* dists_out;
};

template <int KS, int NW>
__global__ __launch_bounds__(64 * NW, 1) void knn_whole_kernel(WnArgs a) {
  using W = WnTile<KS>;
  constexpr int D = 32 * KS;
  constexpr int ROWS = 32 * NW;
  constexpr uint64_t kNone = ~0ull;
  __shared__ __attribute__((aligned(16))) uint4 ring[2 * kWnGroup * W::SLOT];
  __shared__ uint2 qe[NW][kWnQueue];  // a wave's queue: product, row << 27 | id
  __shared__ int cnt[ROWS];
  __shared__ float thr[ROWS];  // -(k-th best distance) / 2 + |q|^2 / 2
  __shared__ float hrow[ROWS];
  const int t = threadIdx.x;
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int lrow0 = 32 * wave;  // the wave's rows in the workgroup
  const uint32_t ring0 = (uint32_t)(uintptr_t)(lds_void_t*)ring;
  constexpr uint32_t kHalf = 16u * kWnGroup * W::SLOT;
  const int64_t rend = a.row0 + a.nq;
  const int64_t ntile = a.npad / kKnnCols;
  uint64_t* const keys = a.keys + ((int64_t)blockIdx.x * ROWS + lrow0) * kWnKeys + lane;
  for (int64_t blk = blockIdx.x; blk * ROWS < a.nq; blk += gridDim.x) {
    const int64_t mrow0 = a.row0 + blk * ROWS + lrow0;
    __syncthreads();  // every wave is done with the ring
    wn_copy_group<KS, NW>(a.Xb, a.half, 0, ntile, ring0, wave, lane);
    uint4 A[2][KS];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const int64_t row = min(mrow0 + 16 * rb + r, a.np - 1);
#pragma unroll
      for (int s = 0; s < KS; ++s)
        A[rb][s] = *reinterpret_cast<const uint4*>(a.Xb + row * D + 32 * s + 8 * g);
    }
    if (lane < 32) {  // nothing passes in a row past the end
      cnt[lrow0 + lane] = 0;
      thr[lrow0 + lane] = mrow0 + lane < rend ? -INFINITY : INFINITY;
      hrow[lrow0 + lane] = a.half[min(mrow0 + lane, a.np - 1)];
    }
#pragma unroll 4
    for (int i = 0; i < 32; ++i) keys[i * kWnKeys] = kNone;
    wave_sync();
    float th[2][4];
    auto load_thr = [&]() {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) th[rb][v] = thr[lrow0 + 16 * rb + 4 * g + v];
    };
    load_thr();
    // rows' list and buffer (c entries) of row i of the wave, and their merge
    auto take = [&](int i, int c, uint64_t& fresh, uint64_t& old) {
      fresh = lane < c ? keys[i * kWnKeys + 64] : kNone;
      old = keys[i * kWnKeys];
    };
    auto merge = [&](int i, uint64_t fresh, uint64_t old) {
      fresh = sort_keys_desc(fresh, lane);
      const uint64_t key = merge_keys_asc(fresh < old ? fresh : old, lane);
      keys[i * kWnKeys] = key;
      const uint32_t kth = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(key >> 32), a.k - 1);
      if (lane == 0) {
        cnt[lrow0 + i] = 0;
        thr[lrow0 + i] = kth == 0xffffffffu
                             ? -INFINITY
                             : -0.5f * __uint_as_float(kth) - hrow[lrow0 + i];
      }
    };
    // the lanes of mask m queue point col of row i with their product x
    int queued = 0;
    auto push = [&](uint64_t m, float x, int i, int col) {
      if (__builtin_expect(m == 0, 1)) return;
      const int at = queued + (int)__builtin_amdgcn_mbcnt_hi(
                                  (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
      if (__builtin_amdgcn_inverse_ballot_w64(m))
        qe[wave][at] = make_uint2(__float_as_uint(x), (uint32_t)i << 27 | (uint32_t)col);
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
          const float dist =
              __builtin_fmaf(-2.f, __uint_as_float(e.x) + hrow[lrow0 + i], 0.f);
          key = (uint64_t)__float_as_uint(dist) << 32 | id;
          left = (int64_t)id != mrow0 + i;
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
    // a tile's operands in registers: a step's are read again, for the next
    // tile, as soon as its products are under way, so that LDS and the matrix
    // unit work at the same time and the picking waits for neither
    uint4 b[KS][4];
    float hx[4];
    auto fetch_half = [&](const uint4* Bt, float (&h)[4]) {
      const float* ht = reinterpret_cast<const float*>(Bt + W::UNITS);
#pragma unroll
      for (int j = 0; j < 4; ++j) h[j] = ht[16 * j + r];
    };
    auto fetch_step = [&](const uint4* Bt, int s) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[s][j] = Bt[(16 * j + r) * W::CPR + ((4 * s + g) ^ (r & W::SWM))];
    };
    // one tile: products, then the points that pass
    auto tile = [&](int64_t n0, const uint4* following) {
      floatx4 acc[2][4];
      float hn[4] = {0.f, 0.f, 0.f, 0.f};
      fetch_half(following, hn);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int rb = 0; rb < 2; ++rb)
            acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, A[rb][s]), __builtin_bit_cast(bf16x8, b[s][j]),
                s ? acc[rb][j] : floatx4{hx[j], hx[j], hx[j], hx[j]}, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_step(following, s);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" ::: "memory");  // the reads stay here
#pragma unroll
      for (int j = 0; j < 4; ++j) hx[j] = hn[j];
      // points that pass, block (rb, v) by block; a block that the queue may
      // have no room for (the first tiles) is left for the loop below.  What
      // is done with them lies out of line: a tile's branches fall through
      // unless a point passes (a taken branch costs a wave as much as ten
      // instructions, and there were eight a tile)
      uint32_t left = 0;
      const int col0 = (int)n0 + r;
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          uint64_t m[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) m[j] = __builtin_amdgcn_ballot_w64(acc[rb][j][v] > th[rb][v]);
          if (__builtin_expect(((m[0] | m[1]) | (m[2] | m[3])) != 0, 0)) {
            if (queued > kWnQueue - 256) {
              left |= 1u << (4 * rb + v);
            } else {
              const int i = 16 * rb + 4 * g + v;
#pragma unroll
              for (int j = 0; j < 4; ++j) push(m[j], acc[rb][j][v], i, col0 + 16 * j);
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
        for (int j = 0; j < 4; ++j)
          push(__builtin_amdgcn_ballot_w64(x[j] > tb), x[j], i, col0 + 16 * j);
        drain();
      }
    };
    int64_t next = 0;
    uint32_t here = 0;  // the ring's half that holds the group
    for (int64_t t0 = 0; t0 < ntile; t0 += kWnGroup) {
      // the group's copies have landed (each wave waits for its own) and every
      // wave is done with the other half
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __syncthreads();
      if (t0 + kWnGroup < ntile)
        wn_copy_group<KS, NW>(a.Xb, a.half, t0 + kWnGroup, ntile, ring0 + (kHalf - here), wave, lane);
      const int n = (int)min<int64_t>(kWnGroup, ntile - t0);
      const uint4* Bt = ring + here / 16;
      fetch_half(Bt, hx);
#pragma unroll
      for (int s = 0; s < KS; ++s) fetch_step(Bt, s);
#pragma unroll 1
      for (int j = 0; j < n; ++j) {
        const int64_t tl = t0 + j;
        Bt += W::SLOT;
        tile(tl * kKnnCols, j + 1 < n ? Bt : Bt - W::SLOT);  // past the group's last: not used
        if (tl >= next) {
          flush_all();
          next = tl + 1 + 7 * tl / 10;
        }
      }
      here = kHalf - here;
    }
    flush_all();
    __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll 4
    for (int i = 0; i < 32; ++i) {
      const int64_t row = mrow0 + i;
      const uint64_t key = keys[i * kWnKeys];
      if (row < rend && lane < a.k) {
        a.ids_out[(row - a.row0) * a.k + lane] = (int32_t)(uint32_t)key;
        if (a.dists_out)
          a.dists_out[(row - a.row0) * a.k + lane] = __uint_as_float((uint32_t)(key >> 32));
      }
    }
  }
}

// ---- search graph from kNN lists -----------------------------------------
// Candidate edges of u: forward u -> knn[u][j] (rank j, type 0) and reverse
// u -> v for every v with knn[v][j] == u, j < rev_rank (rank j, type 1); a
// pair (u, v) keeps its smallest (rank, type); row u keeps the `degree`
// candidates of smallest (rank, type, v), padded with np.

__global__ void rev_count_kernel(const int32_t* __restrict__ knn, int64_t np, int kf, int kr,
                                 int32_t* __restrict__ cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np * kr) return;
  const int64_t v = i / kr;
  const int j = (int)(i - v * kr);
  const int32_t u = knn[v * kf + j];
  if (u >= 0 && u < np && u != v) atomicAdd(&cnt[u], 1);
}

// exclusive scan in blocks of 1024 (block totals to `sums`), then the block
// totals by one workgroup, then the carry-in
__global__ __launch_bounds__(1024) void scan_blocks_kernel(const int32_t* __restrict__ in, int64_t n,
                                                          int64_t* __restrict__ out,
                                                          int64_t* __restrict__ sums) {
  __shared__ int64_t sh[1024];
  const int t = threadIdx.x;
  const int64_t i = (int64_t)blockIdx.x * 1024 + t;
  const int64_t x = i < n ? in[i] : 0;
  sh[t] = x;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {
    const int64_t y = t >= o ? sh[t - o] : 0;
    __syncthreads();
    sh[t] += y;
    __syncthreads();
  }
  if (i < n) out[i] = sh[t] - x;
  if (t == 1023) sums[blockIdx.x] = sh[t];
}

__global__ __launch_bounds__(1024) void scan_sums_kernel(int64_t* __restrict__ sums, int64_t nb,
                                                        int64_t* __restrict__ total) {
  __shared__ int64_t sh[1024];
  const int t = threadIdx.x;
  int64_t carry = 0;
  for (int64_t b0 = 0; b0 < nb; b0 += 1024) {
    const int64_t b = b0 + t;
    const int64_t x = b < nb ? sums[b] : 0;
    sh[t] = x;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
      const int64_t y = t >= o ? sh[t - o] : 0;
      __syncthreads();
      sh[t] += y;
      __syncthreads();
    }
    if (b < nb) sums[b] = carry + sh[t] - x;
    const int64_t blk = sh[1023];
    __syncthreads();
    carry += blk;
  }
  if (t == 0) total[0] = carry;
}

__global__ void scan_add_kernel(int64_t* __restrict__ out, int64_t n,
                                const int64_t* __restrict__ sums, const int64_t* __restrict__ total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] += sums[i / 1024];
  if (i == n) out[n] = total[0];
}

__global__ void rev_fill_kernel(const int32_t* __restrict__ knn, int64_t np, int kf, int kr,
                                const int64_t* __restrict__ off, int32_t* __restrict__ cur,
                                int64_t* __restrict__ rev) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np * kr) return;
  const int64_t v = i / kr;
  const int j = (int)(i - v * kr);
  const int32_t u = knn[v * kf + j];
  if (u >= 0 && u < np && u != v) {
    const int slot = atomicAdd(&cur[u], 1);
    rev[off[u] + slot] = ((int64_t)j << 32) | (int64_t)v;  // key (rank, id)
  }
}

// (rank, type, id) order of two candidates
__device__ __forceinline__ bool cand_less(int r1, int t1, int v1, int r2, int t2, int v2) {
  return r1 < r2 || (r1 == r2 && (t1 < t2 || (t1 == t2 && v1 < v2)));
}

// one wave per node u
__global__ __launch_bounds__(256) void graph_rows_kernel(const int32_t* __restrict__ knn,
                                                         int64_t np, int kf, int degree,
                                                         const int64_t* __restrict__ off,
                                                         const int64_t* __restrict__ rev,
                                                         int32_t* __restrict__ graph) {
  const int lane = threadIdx.x & 63;
  const int64_t u = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (u >= np) return;  // whole waves, no workgroup barrier
  const int32_t fv = lane < kf ? knn[u * kf + lane] : -1;
  const bool fvalid = lane < kf && fv >= 0 && fv < np && fv != u;
  uint64_t fdrop = 0;  // forward positions displaced by a smaller-rank reverse edge
  constexpr int64_t kNone = 0x7fffffffffffffffLL;
  int64_t tk = kNone;  // lane i < degree: i-th best reverse key (rank << 32 | id)
  const int64_t r0 = off[u], r1 = off[u + 1];
  for (int64_t c0 = r0; c0 < r1; c0 += 64) {
    const int64_t idx = c0 + lane;
    int64_t key = idx < r1 ? rev[idx] : kNone;
    const int rj = (int)(key >> 32);
    const int rv = (int)(key & 0xffffffff);
    bool keep = key != kNone;
    for (int p = 0; p < kf; ++p) {  // is rv also a forward neighbour, at rank p?
      const int fp = __shfl(fv, p, 64);
      const bool match = keep && rv == fp;
      if (__ballot(match && p > rj)) fdrop |= 1ull << p;
      if (match && p <= rj) keep = false;
    }
    uint64_t m = __ballot(keep);
    while (m) {  // insert the survivors into the sorted top-`degree` list
      const int src = __ffsll((unsigned long long)m) - 1;
      m &= m - 1;
      const int64_t ck = __shfl(key, src, 64);
      const bool less = lane < degree && tk < ck;
      const int pos = __popcll(__ballot(less));
      const int64_t prev = __shfl_up(tk, 1, 64);
      if (pos < degree && lane >= pos && lane < degree) tk = lane == pos ? ck : prev;
    }
  }
  // merge: forward survivors (rank = position, type 0) and the reverse list
  const bool fs = fvalid && !((fdrop >> lane) & 1ull);
  const uint64_t fmask = __ballot(fs);
  const int nf_before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(fmask >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)fmask, 0u));
  const bool ts = lane < degree && tk != kNone;
  const uint64_t tmask = __ballot(ts);
  const int tr = (int)(tk >> 32), tv = (int)(tk & 0xffffffff);
  // output position of each surviving element = its rank in its own list +
  // the number of elements of the other list that precede it
  int fpos = nf_before, tpos = lane;
  for (int q = 0; q < 64; ++q) {
    if ((tmask >> q) & 1ull) {  // reverse element q against this lane's forward element
      const int qr = __shfl(tr, q, 64), qv = __shfl(tv, q, 64);
      if (fs && cand_less(qr, 1, qv, lane, 0, fv)) ++fpos;
    }
    if ((fmask >> q) & 1ull) {  // forward element q against this lane's reverse element
      const int qv = __shfl(fv, q, 64);
      if (ts && cand_less(q, 0, qv, tr, 1, tv)) ++tpos;
    }
  }
  int32_t* row = graph + u * degree;
  const int total = __popcll(fmask) + __popcll(tmask);
  if (lane < degree && lane >= total) row[lane] = (int32_t)np;
  if (fs && fpos < degree) row[fpos] = fv;
  if (ts && tpos < degree) row[tpos] = tv;
}

hipError_t launch_graph_from_knn(const int32_t* knn, int64_t np, int kf, int degree, int rev_rank,
                                 int32_t* graph, void* work, hipStream_t st) {
  const int kr = rev_rank < kf ? rev_rank : kf;
  // work: cnt (np) | cur (np) | off (np + 1) | sums | total | rev
  char* w = static_cast<char*>(work);
  int32_t* cnt = reinterpret_cast<int32_t*>(w);
  int32_t* cur = cnt + np;
  int64_t* off = reinterpret_cast<int64_t*>(w + ((2 * np * 4 + 255) & ~255LL));
  const int64_t nb = (np + 1023) / 1024;
  int64_t* sums = off + np + 1;
  int64_t* total = sums + nb;
  int64_t* rev = total + 1;
  hipError_t e = hipMemsetAsync(cnt, 0, 2 * np * sizeof(int32_t), st);
  if (e != hipSuccess) return e;
  const int64_t ne = np * (int64_t)kr;
  if (kr > 0) {
    hipLaunchKernelGGL(rev_count_kernel, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, st, knn,
                       np, kf, kr, cnt);
  }
  hipLaunchKernelGGL(scan_blocks_kernel, dim3((unsigned)nb), dim3(1024), 0, st, cnt, np, off, sums);
  hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(1024), 0, st, sums, nb, total);
  hipLaunchKernelGGL(scan_add_kernel, dim3((unsigned)((np + 1 + 255) / 256)), dim3(256), 0, st, off,
                     np, sums, total);
  if (kr > 0) {
    hipLaunchKernelGGL(rev_fill_kernel, dim3((unsigned)((ne + 255) / 256)), dim3(256), 0, st, knn,
                       np, kf, kr, off, cur, rev);
  }
  hipLaunchKernelGGL(graph_rows_kernel, dim3((unsigned)((np + 3) / 4)), dim3(256), 0, st, knn, np,
                     kf, degree, off, rev, graph);
  return hipGetLastError();
}

size_t graph_from_knn_work_bytes(int64_t np, int kf, int rev_rank) {
  const int kr = rev_rank < kf ? rev_rank : kf;
  const int64_t nb = (np + 1023) / 1024;
  return (size_t)((2 * np * 4 + 255) & ~255LL) + (size_t)(np + 1 + nb + 1) * 8 +
         (size_t)np * kr * 8;
}

hipError_t launch_row_norms(const float* X, int64_t np, int d, int64_t stride, float* norms,
                            uint16_t* Xb, float* half, uint32_t* flag, hipStream_t st) {
  const int64_t npad = knn_padded(np);
  hipLaunchKernelGGL(row_norms_kernel, dim3((unsigned)(npad / 64)), dim3(256), 0, st, X, np, d,
                     stride, npad, norms, Xb, half, flag);
  return hipGetLastError();
}

hipError_t launch_knn_whole(const uint16_t* Xb, const float* half, int64_t np, int d, int64_t row0,
                            int64_t nq, int k, int slots, uint64_t* keys, int32_t* ids,
                            float* dists, hipStream_t st) {
  WnArgs a{Xb, half, np, knn_padded(np), row0, nq, k, keys, ids, dists};
  // whole rounds of 256-row blocks first; what is left over in blocks of 128
  // rows where they still run all at once (a round of them takes 0.6 of one of
  // 256-row blocks)
  const int64_t blocks = (nq + 255) / 256, rest = blocks % slots;
  const bool split = 2 * rest <= slots;
  const int64_t n8 = split ? std::min(nq, (blocks - rest) * 256) : nq;
#define KNNW(KS)                                                                                 \
  {                                                                                              \
    a.nq = n8;                                                                                   \
    if (a.nq > 0)                                                                                \
      hipLaunchKernelGGL((knn_whole_kernel<KS, 8>),                                              \
                         dim3((unsigned)std::min<int64_t>((a.nq + 255) / 256, slots)), dim3(512), \
                         0, st, a);                                                              \
    a.row0 = row0 + n8;                                                                          \
    a.nq = nq - n8;                                                                              \
    a.ids_out = ids + n8 * k;                                                                    \
    a.dists_out = dists ? dists + n8 * k : nullptr;                                              \
    if (a.nq > 0)                                                                                \
      hipLaunchKernelGGL((knn_whole_kernel<KS, 4>), dim3((unsigned)((a.nq + 127) / 128)),        \
                         dim3(256), 0, st, a);                                                   \
    break;                                                                                       \
  }
  switch (d / 32) {
    case 1: KNNW(1)
    case 2: KNNW(2)
    case 3: KNNW(3)
    case 4: KNNW(4)
    default: return hipErrorInvalidValue;
  }
#undef KNNW
  return hipGetLastError();
}

hipError_t launch_knn(const float* X, int64_t np, int d, int64_t stride, const float* norms,
                      int64_t row0, int64_t nq, int k, int32_t* ids, float* dists,
                      hipStream_t st) {
  if (nq <= 0) return hipSuccess;
  const dim3 grid((unsigned)((nq + kKnnRows - 1) / kKnnRows));
#define KNN(S)                                                                                    \
  hipLaunchKernelGGL(knn_kernel<S>, grid, dim3(512), 0, st, X, np, d, stride, norms, row0, nq, k, \
                     ids, dists)
  switch (d / 16) {
    case 2: KNN(2); break;
    case 4: KNN(4); break;
    case 6: KNN(6); break;
    case 8: KNN(8); break;
    default: return hipErrorInvalidValue;
  }
#undef KNN
  return hipGetLastError();
}

}  // namespace rte
