// kd-tree over the first three coordinates of the rows of a device array,
// built on the GPU.  Same output as the host build (kdtree.cpp in this
// library) and the reference's Kdtree + computeAabbPid (kdtree.cpp:4-195):
// the same leaf point sets, the same tight boxes (as values: where a
// coordinate is +0 in some points and -0 in others, the sign of a zero box
// bound may differ), the same left-first DFS leaf order and the same
// ascending, np-padded pid table.
//
// The rules (kdtree.cpp:30-62, 103-125, 171-185): a node with at most
// max_node points is a leaf; otherwise it splits its tight box's widest axis
// (ties to the lowest axis) at the bisection value of findxM, and values
// below the split go left.  Every output depends only on the set of points
// in a node, never on their order, which the parallel partitions below use.
//
// Points travel as 16-byte records (three coordinates, id) between two buffers,
// and the device plans its own work: large nodes (more than kKdSmall points) are
// split in rounds of five launches on grids of the largest possible size, which
// the host queues for the expected depth at once and checks afterwards.
//   count x 3  findxM's loop, four steps a launch: a workgroup per 2048-point
//              chunk counts its points at or below the 15 midpoints that four
//              steps can meet; who needs a node's state walks its counts
//   partition  slots from both ends of the node's segment, one atomic per side
//              and workgroup; the children's boxes on the way, as order-preserving
//              integer keys; a node whose search has not ended is carried over
//   plan       one workgroup makes the next round's nodes of the children, the map
//              from chunks to nodes and the list of small nodes
// 1M points, cap 256: ten rounds of 58 us, 0.9 ms in all; 3.4 with a launch per
// step, boxes and split-axis values gathered from the rows by id, and a read-back
// every four steps.
// Small nodes (at most kKdSmall points) are finished by one workgroup each:
// ids, coordinates and a local permutation in LDS, an explicit stack of
// segments, block-wide counts for the bisection.  Left children always come
// before right children in the index array, so the left-first DFS order of
// the leaves is the order of their segment starts: starts are marked and counted
// in order.  Each leaf's ids are sorted by a bitonic network in LDS to form its
// pid row.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "ctx.h"
#include "kd_chunk.h"

namespace rte {

namespace {

constexpr int kKdSmall = 2048;   // nodes up to this size: one workgroup in LDS
constexpr int kKdMaxIter = 64;   // findxM ends within about 11 steps
constexpr int kKdSteps = 4;      // of findxM in a launch
constexpr int kKdPasses = 3;     // launches in a round
constexpr int kKdMids = (1 << kKdSteps) - 1;

struct LevelNode {
  int l, r;               // segment [l, r)
  int blk0;               // first workgroup of this node in the round's grids
  int axis, done, steps;  // done: the search has ended, xm is the split
  float bl, br, xm, eps;
  unsigned nl, nr;                         // points left and right of the split
  unsigned cnt[kKdPasses][kKdMids + 1];    // points at or below midpoint i of a pass
  unsigned key[2][6];  // children's ordered keys: min x, y, z, max x, y, z
};

struct Seg {
  int l, r, buf, pad;  // a small node, in record buffer `buf`
};

struct Header {
  int m[2], blocks[2];  // nodes and workgroups, by parity of the round
  int ns;               // small nodes
  unsigned err, leaves;
};

struct KdWork {
  float4* rec[2];
  int* idx;    // np: ids in leaf order
  int* mark;   // np: leaf record + 1 at a leaf's start, 0 elsewhere
  int* marks;  // marks per chunk
  LevelNode* nodes[2];
  int* map[2];  // node of a workgroup
  Seg* segs;
  Header* h;
  int64_t np;
  int cap;  // of segs and leaves
};

struct LeafRec {
  int64_t start;
  int cnt, pad;
  float box[6];
};

__device__ __forceinline__ unsigned fkey(float f) {
  const unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float funkey(unsigned k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// findxM's midpoint (kdtree.cpp:103-125): the float sum, halved in double
__device__ __forceinline__ float kd_mid(float l, float r) {
  return (float)((double)(r + l) / 2.0);
}

__device__ __forceinline__ unsigned lanes_below(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// 6 keys: min of the first three, max of the last three, over the workgroup
__device__ __forceinline__ void block_minmax6(unsigned v[6], unsigned (*red)[4]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = min(v[k], (unsigned)__shfl_xor((int)v[k], o));
#pragma unroll
    for (int k = 3; k < 6; ++k) v[k] = max(v[k], (unsigned)__shfl_xor((int)v[k], o));
  }
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 6; ++k) red[k][wave] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k) v[k] = min(min(red[k][0], red[k][1]), min(red[k][2], red[k][3]));
#pragma unroll
  for (int k = 3; k < 6; ++k) v[k] = max(max(red[k][0], red[k][1]), max(red[k][2], red[k][3]));
  __syncthreads();
}

__device__ __forceinline__ unsigned block_sum(unsigned v, unsigned* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += (unsigned)__shfl_xor((int)v, o);
  if (lane == 0) red[wave] = v;
  __syncthreads();
  v = red[0] + red[1] + red[2] + red[3];
  __syncthreads();
  return v;
}

// widest axis (strictly wider wins, so ties go to the lowest axis) and the
// initial bisection state (kdtree.cpp:30-42, 103-110)
__device__ __forceinline__ void split_setup(const float lo[3], const float hi[3], int& axis,
                                            float& bl, float& br, float& xm, float& eps) {
  float maxw = 0.0f;
  axis = 0;
  for (int a = 0; a < 3; ++a)
    if (hi[a] - lo[a] > maxw) {
      maxw = hi[a] - lo[a];
      axis = a;
    }
  bl = lo[axis];
  br = hi[axis];
  xm = kd_mid(bl, br);
  eps = fmaxf((br - bl) / 1000.0f, 0.00001f);
}

// findxM's state after the steps that the counts of the first `passes` launches
// decide (kdtree.cpp:111-124)
struct KdState {
  float bl, br, xm;
  int done, steps;
};
__device__ __forceinline__ KdState kd_walk(const LevelNode& n, int passes) {
  KdState s{n.bl, n.br, n.xm, n.done, n.steps};
  const unsigned half = (unsigned)(n.r - n.l) / 2;
  for (int p = 0; p < passes; ++p) {
    int q = 1;  // midpoints as a heap: 2q where the upper half goes, 2q + 1 the lower
    for (int i = 0; i < kKdSteps && !s.done && s.steps < kKdMaxIter; ++i) {
      const float mid = kd_mid(s.bl, s.br);
      const unsigned c = n.cnt[p][q];
      ++s.steps;
      if (c <= half) {
        s.bl = mid;
        s.xm = mid;
        if (c == half) s.done = 1;
        q = 2 * q + 1;
      } else {
        s.br = mid;
        q = 2 * q;
      }
      if (!(s.br - s.bl > n.eps)) s.done = 1;
    }
  }
  return s;
}

// records of the points; the root's box goes to `root` as a left child's
__global__ __launch_bounds__(256) void kd_root_kernel(const float* __restrict__ pts, int64_t stride,
                                                      KdWork w, LevelNode* root) {
  __shared__ unsigned red[6][4];
  const int64_t s0 = (int64_t)blockIdx.x * kKdChunk, s1 = min(w.np, s0 + kKdChunk);
  unsigned v[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
#pragma unroll 4
  for (int64_t i = s0 + threadIdx.x; i < s1; i += 256) {
    const float* p = pts + i * stride;
    const float4 c = make_float4(p[0], p[1], p[2], __int_as_float((int)i));
    w.rec[0][i] = c;
    w.mark[i] = 0;
    const float x[3] = {c.x, c.y, c.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const unsigned k = fkey(x[a]);
      v[a] = min(v[a], k);
      v[3 + a] = max(v[3 + a], k);
    }
  }
  block_minmax6(v, red);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      atomicMin(&root->key[0][a], v[a]);
      atomicMax(&root->key[0][3 + a], v[3 + a]);
    }
  }
}

// the root as the left child of a node that is done, nothing to its right
__global__ void kd_start_kernel(KdWork w) {
  if (threadIdx.x) return;
  *w.h = Header{};
  w.h->m[1] = 1;
  LevelNode& n = w.nodes[1][0];
  n = LevelNode{};
  n.r = (int)w.np;
  n.done = 1;
  n.nl = (unsigned)w.np;
  for (int c = 0; c < 2; ++c)
    for (int k = 0; k < 3; ++k) n.key[c][k] = 0xffffffffu;
}

// Pass `pass` of a round: points of a chunk at or below each midpoint of the next
// four steps.  Bound by the launch and three dependent loads.
__global__ __launch_bounds__(256) void kd_count_kernel(KdWork w, int par, int pass) {
  if ((int)blockIdx.x >= w.h->blocks[par]) return;
  LevelNode& n = w.nodes[par][w.map[par][blockIdx.x]];
  __shared__ unsigned tot[kKdMids + 1];
  const int t = threadIdx.x;
  if (t <= kKdMids) tot[t] = 0;
  const KdState s = kd_walk(n, pass);
  if (s.done || s.steps >= kKdMaxIter) return;  // all threads
  float bl[kKdMids + 1], br[kKdMids + 1], mid[kKdMids + 1];
  bl[1] = s.bl;
  br[1] = s.br;
#pragma unroll
  for (int q = 1; q <= kKdMids; ++q) {
    mid[q] = kd_mid(bl[q], br[q]);
    if (2 * q + 1 <= kKdMids) {
      bl[2 * q] = bl[q];
      br[2 * q] = mid[q];
      bl[2 * q + 1] = mid[q];
      br[2 * q + 1] = br[q];
    }
  }
  const KdChunk ch = kd_chunk(n.l, n.r, (int)blockIdx.x - n.blk0);
  const float* x = reinterpret_cast<const float*>(w.rec[par]) + n.axis;
  constexpr int PER = kKdChunk / 256;
  float v[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k)  // past the end: above every midpoint, or NaN
    v[k] = 256 * k + t < ch.count ? x[4 * (int64_t)(ch.first + 256 * k + t)] : INFINITY;
  __syncthreads();
#pragma unroll
  for (int q = 1; q <= kKdMids; ++q) {
    unsigned c = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k)
      c += (unsigned)__popcll(__ballot(256 * k + t < ch.count && v[k] <= mid[q]));
    if ((t & 63) == 0 && c) atomicAdd(&tot[q], c);
  }
  __syncthreads();
  if (t >= 1 && t <= kKdMids && tot[t]) atomicAdd(&n.cnt[pass][t], tot[t]);
}

// Points of a chunk below the split go to the front of the node's segment in the
// other buffer, the rest to the back, with their boxes.  The workgroup counts both
// sides, takes its slots with one atomic per side and node, and the waves place
// their points from per-wave bases.  Where the search has not ended the points
// keep their places.
__global__ __launch_bounds__(256) void kd_partition_kernel(KdWork w, int par) {
  if ((int)blockIdx.x >= w.h->blocks[par]) return;
  constexpr int PER = kKdChunk / 256;
  __shared__ unsigned cnt_w[2][4];
  __shared__ unsigned base_w[2][4];
  __shared__ unsigned red[6][4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  LevelNode& n = w.nodes[par][w.map[par][blockIdx.x]];
  const int l = n.l, r = n.r;
  const KdChunk ch = kd_chunk(l, r, (int)blockIdx.x - n.blk0);
  const float4* in = w.rec[par] + ch.first;
  float4* out = w.rec[par ^ 1];
  const KdState s = kd_walk(n, kKdPasses);
  float4 p[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = 256 * k + t;
    p[k] = i < ch.count ? in[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (!s.done) {
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if (256 * k + t < ch.count) out[ch.first + 256 * k + t] = p[k];
    return;  // all threads
  }
  const int axis = n.axis;
  unsigned v[2][6];
  for (int c = 0; c < 2; ++c)
    for (int k = 0; k < 6; ++k) v[c][k] = k < 3 ? 0xffffffffu : 0u;
  unsigned lmask = 0, vmask = 0;  // bit k: element k is valid / goes left
  unsigned nl = 0, nr = 0;        // this wave's counts (uniform)
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool valid = 256 * k + t < ch.count;
    const float x[3] = {p[k].x, p[k].y, p[k].z};
    const float xa = axis == 0 ? x[0] : axis == 1 ? x[1] : x[2];
    const bool left = valid && xa < s.xm;
    vmask |= (unsigned)valid << k;
    lmask |= (unsigned)left << k;
    nl += (unsigned)__popcll(__ballot(left));
    nr += (unsigned)__popcll(__ballot(valid && !left));
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const unsigned key = fkey(x[a]);
      if (left) {
        v[0][a] = min(v[0][a], key);
        v[0][3 + a] = max(v[0][3 + a], key);
      } else if (valid) {
        v[1][a] = min(v[1][a], key);
        v[1][3 + a] = max(v[1][3 + a], key);
      }
    }
  }
  if (lane == 0) {
    cnt_w[0][wave] = nl;
    cnt_w[1][wave] = nr;
  }
  __syncthreads();
  if (t == 0) {
    const unsigned tl = cnt_w[0][0] + cnt_w[0][1] + cnt_w[0][2] + cnt_w[0][3];
    const unsigned tr = cnt_w[1][0] + cnt_w[1][1] + cnt_w[1][2] + cnt_w[1][3];
    unsigned bl = tl ? atomicAdd(&n.nl, tl) : 0u;
    unsigned br = tr ? atomicAdd(&n.nr, tr) : 0u;
    for (int i = 0; i < 4; ++i) {
      base_w[0][i] = bl;
      base_w[1][i] = br;
      bl += cnt_w[0][i];
      br += cnt_w[1][i];
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    block_minmax6(v[c], red);
    if (t < 6) {  // v is the same in all threads
      unsigned x = v[c][0];
#pragma unroll
      for (int k = 1; k < 6; ++k) x = t == k ? v[c][k] : x;
      if (t < 3) atomicMin(&n.key[c][t], x);
      else atomicMax(&n.key[c][t], x);
    }
  }
  unsigned ol = base_w[0][wave], orr = base_w[1][wave];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const bool valid = (vmask >> k) & 1u, left = (lmask >> k) & 1u;
    const unsigned long long ml = __ballot(left), mr = __ballot(valid && !left);
    if (left) out[l + ol + lanes_below(ml)] = p[k];
    if (valid && !left) out[r - 1 - (int)(orr + lanes_below(mr))] = p[k];
    ol += (unsigned)__popcll(ml);
    orr += (unsigned)__popcll(mr);
  }
}

// The next round's nodes: children of nodes that are done, and those that are not.
// One workgroup; nodes of the round `par` to the other parity.
__global__ __launch_bounds__(1024) void kd_plan_kernel(KdWork w, int par) {
  __shared__ int sn[1024], sb[1024];
  __shared__ int nseg;
  const int t = threadIdx.x, m = w.h->m[par];
  int base_n = 0, base_b = 0;
  if (t == 0) nseg = w.h->ns;
  for (int i0 = 0; i0 < m; i0 += 1024) {
    LevelNode c[2];
    int large = 0, blocks = 0;
    if (i0 + t < m) {
      const LevelNode& n = w.nodes[par][i0 + t];
      const KdState s = kd_walk(n, kKdPasses);
      if (!s.done) {
        if (s.steps >= kKdMaxIter) {
          atomicOr(&w.h->err, 2u);
        } else {
          c[0] = n;
          c[0].bl = s.bl;
          c[0].br = s.br;
          c[0].xm = s.xm;
          c[0].steps = s.steps;
          large = 1;
        }
      } else {
        const int mid = n.l + (int)n.nl;
        if ((mid == n.l || mid == n.r) && n.axis >= 0 && n.eps > 0.f) atomicOr(&w.h->err, 1u);
        else
          for (int k = 0; k < 2; ++k) {
            const int l = k ? mid : n.l, r = k ? n.r : mid;
            if (r - l > kKdSmall) {
              LevelNode& d = c[large++];
              d.l = l;
              d.r = r;
              float lo[3], hi[3];
              for (int a = 0; a < 3; ++a) {
                lo[a] = funkey(n.key[k][a]);
                hi[a] = funkey(n.key[k][3 + a]);
              }
              split_setup(lo, hi, d.axis, d.bl, d.br, d.xm, d.eps);
              d.done = !(d.br - d.bl > d.eps);
              d.steps = 0;
            } else if (r > l) {
              const int at = atomicAdd(&nseg, 1);
              if (at < w.cap) w.segs[at] = Seg{l, r, par ^ 1, 0};
            }
          }
      }
      for (int k = 0; k < large; ++k) blocks += kd_chunks(c[k].r - c[k].l);
    }
    __syncthreads();
    sn[t] = large;
    sb[t] = blocks;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
      const int x = t >= o ? sn[t - o] : 0, y = t >= o ? sb[t - o] : 0;
      __syncthreads();
      sn[t] += x;
      sb[t] += y;
      __syncthreads();
    }
    int at = base_n + sn[t] - large, b = base_b + sb[t] - blocks;
    for (int k = 0; k < large; ++k) {
      LevelNode& d = c[k];
      d.blk0 = b;
      d.nl = d.nr = 0;
      for (int p = 0; p < kKdPasses; ++p)
        for (int q = 0; q <= kKdMids; ++q) d.cnt[p][q] = 0;
      for (int e = 0; e < 2; ++e)
        for (int a = 0; a < 6; ++a) d.key[e][a] = a < 3 ? 0xffffffffu : 0u;
      w.nodes[par ^ 1][at] = d;
      for (int j = kd_chunks(d.r - d.l); j > 0; --j) w.map[par ^ 1][b++] = at;
      ++at;
    }
    base_n += sn[1023];
    base_b += sb[1023];
  }
  __syncthreads();
  if (t == 0) {
    w.h->m[par ^ 1] = base_n;
    w.h->blocks[par ^ 1] = base_b;
    w.h->ns = nseg;
    if (nseg > w.cap) atomicOr(&w.h->err, 4u);
  }
}

// marks of a chunk
__global__ __launch_bounds__(256) void kd_mark_kernel(KdWork w) {
  __shared__ unsigned red[4];
  const int64_t s0 = (int64_t)blockIdx.x * kKdChunk, s1 = min(w.np, s0 + kKdChunk);
  unsigned c = 0;
  for (int64_t i = s0 + threadIdx.x; i < s1; i += 256) c += w.mark[i] != 0;
  c = block_sum(c, red);
  if (threadIdx.x == 0) w.marks[blockIdx.x] = (int)c;
}

// leaves in the order of their starts
__global__ __launch_bounds__(256) void kd_order_kernel(KdWork w, const LeafRec* __restrict__ leaves,
                                                       int* __restrict__ start,
                                                       int* __restrict__ count,
                                                       float* __restrict__ boxes) {
  __shared__ unsigned red[4];
  __shared__ unsigned wsum[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  unsigned before = 0;
  for (int i = t; i < (int)blockIdx.x; i += 256) before += (unsigned)w.marks[i];
  before = block_sum(before, red);
  const int64_t s0 = (int64_t)blockIdx.x * kKdChunk, s1 = min(w.np, s0 + kKdChunk);
  for (int64_t i0 = s0; i0 < s1; i0 += 256) {  // 256 in a row at a time
    const int64_t i = i0 + t;
    const int k = i < s1 ? w.mark[i] : 0;
    const unsigned long long mk = __ballot(k != 0);
    if (lane == 0) wsum[wave] = (unsigned)__popcll(mk);
    __syncthreads();
    unsigned at = before + lanes_below(mk);
    for (int x = 0; x < 4; ++x) {
      if (x < wave) at += wsum[x];
      before += wsum[x];
    }
    if (k) {
      const LeafRec& rec = leaves[k - 1];
      start[at] = (int)i;
      count[at] = rec.cnt;
      for (int b = 0; b < 6; ++b) boxes[(int64_t)at * 6 + b] = rec.box[b];
    }
    __syncthreads();
  }
}

// err bits: 1 = split failed, 2 = findxM did not end, 4 = leaf capacity
__global__ __launch_bounds__(256) void kd_small_kernel(KdWork w, int max_node,
                                                       LeafRec* __restrict__ leaves,
                                                       int max_leaves) {
  __shared__ int ids[kKdSmall];
  __shared__ float cs[3][kKdSmall];
  __shared__ uint16_t perm[2][kKdSmall];
  __shared__ unsigned stack[kKdSmall];  // a << 16 | b, local offsets
  __shared__ unsigned red[6][4];
  __shared__ unsigned cnts[2];
  const int t = threadIdx.x;
  const Seg sg = w.segs[blockIdx.x];
  const int l = sg.l, n = sg.r - sg.l;
  int* const idx = w.idx;
  unsigned* const err = &w.h->err;
  for (int j = t; j < n; j += 256) {
    const float4 p = w.rec[sg.buf][l + j];
    ids[j] = __float_as_int(p.w);
    cs[0][j] = p.x;
    cs[1][j] = p.y;
    cs[2][j] = p.z;
    perm[0][j] = (uint16_t)j;
  }
  if (t == 0) stack[0] = (unsigned)n;
  int top = 1;
  __syncthreads();
  while (top > 0) {
    const unsigned e = stack[--top];
    const int a = (int)(e >> 16), b = (int)(e & 0xffffu);
    const int cnt = b - a;
    unsigned v[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
    for (int j = a + t; j < b; j += 256) {
      const int p = perm[0][j];
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        const unsigned k = fkey(cs[ax][p]);
        v[ax] = min(v[ax], k);
        v[3 + ax] = max(v[3 + ax], k);
      }
    }
    block_minmax6(v, red);
    float lo[3], hi[3];
    for (int ax = 0; ax < 3; ++ax) {
      lo[ax] = funkey(v[ax]);
      hi[ax] = funkey(v[3 + ax]);
    }
    if (cnt <= max_node) {  // leaf (kdtree.cpp:171-174)
      if (t == 0) {
        const unsigned s = atomicAdd(&w.h->leaves, 1u);
        if (s < (unsigned)max_leaves) {
          LeafRec& rec = leaves[s];
          w.mark[l + a] = (int)s + 1;
          rec.start = l + a;
          rec.cnt = cnt;
          rec.pad = 0;
          for (int ax = 0; ax < 3; ++ax) {
            rec.box[ax] = lo[ax];
            rec.box[3 + ax] = hi[ax];
          }
        } else {
          atomicOr(err, 4u);
        }
      }
      for (int j = a + t; j < b; j += 256) idx[l + j] = ids[perm[0][j]];
      __syncthreads();
      continue;
    }
    int axis;
    float bl, br, xm, eps;
    split_setup(lo, hi, axis, bl, br, xm, eps);
    const unsigned half = (unsigned)cnt / 2;
    int steps = 0;
    while (br - bl > eps) {  // findxM (kdtree.cpp:111-124), block-uniform
      if (++steps > kKdMaxIter) break;
      const float mid = kd_mid(bl, br);
      unsigned c = 0;
      for (int j = a + t; j < b; j += 256) c += cs[axis][perm[0][j]] <= mid;
      c = block_sum(c, &red[0][0]);
      if (c <= half) {
        bl = mid;
        xm = mid;
        if (c == half) break;
      } else {
        br = mid;
      }
    }
    if (steps > kKdMaxIter) {
      if (t == 0) atomicOr(err, 2u);
      return;
    }
    if (t < 2) cnts[t] = 0;
    __syncthreads();
    for (int base = a; base < b; base += 256) {
      const int j = base + t;
      const bool valid = j < b;
      const int p = valid ? perm[0][j] : 0;
      const bool left = valid && cs[axis][p] < xm;
      const bool right = valid && !left;
      const unsigned long long ml = __ballot(left), mr = __ballot(right);
      unsigned lb = 0, rb = 0;
      if ((t & 63) == 0) {
        if (ml) lb = atomicAdd(&cnts[0], (unsigned)__popcll(ml));
        if (mr) rb = atomicAdd(&cnts[1], (unsigned)__popcll(mr));
      }
      lb = (unsigned)__builtin_amdgcn_readfirstlane((int)lb);
      rb = (unsigned)__builtin_amdgcn_readfirstlane((int)rb);
      if (left) perm[1][a + lb + lanes_below(ml)] = (uint16_t)p;
      if (right) perm[1][b - 1 - (int)(rb + lanes_below(mr))] = (uint16_t)p;
    }
    __syncthreads();
    const int nl = (int)cnts[0];
    for (int j = a + t; j < b; j += 256) perm[0][j] = perm[1][j];
    if (nl == 0 || nl == cnt) {  // kdtree.cpp:182-185
      if (t == 0) atomicOr(err, 1u);
      return;
    }
    if (t == 0) {
      stack[top] = ((unsigned)(a + nl) << 16) | (unsigned)b;
      stack[top + 1] = ((unsigned)a << 16) | (unsigned)(a + nl);
    }
    top += 2;
    __syncthreads();
  }
}

// pid row of leaf i: its ids ascending, padded with np (kdtree.cpp:91-101)
__global__ __launch_bounds__(256) void kd_pids_kernel(const int* __restrict__ idx,
                                                      const int* __restrict__ start,
                                                      const int* __restrict__ count, int max_node,
                                                      int P, int64_t np,
                                                      int32_t* __restrict__ pids) {
  __shared__ int s[kKdSmall];
  const int leaf = blockIdx.x;
  const int64_t st = start[leaf];
  const int cnt = count[leaf];
  for (int j = threadIdx.x; j < P; j += 256) s[j] = j < cnt ? idx[st + j] : INT_MAX;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int jj = k >> 1; jj > 0; jj >>= 1) {
      for (int i = threadIdx.x; i < P; i += 256) {
        const int ixj = i ^ jj;
        if (ixj > i) {
          const int x = s[i], y = s[ixj];
          const bool up = (i & k) == 0;
          if ((x > y) == up) {
            s[i] = y;
            s[ixj] = x;
          }
        }
      }
      __syncthreads();
    }
  for (int j = threadIdx.x; j < max_node; j += 256)
    pids[(int64_t)leaf * max_node + j] = j < cnt ? s[j] : (int32_t)np;
}

}  // namespace

}  // namespace rte

extern "C" {

int rte_build_kdtree_gpu(rte_ctx* c, const float* pts, int64_t np, int64_t stride, int max_node,
                         int max_leaves, float* aabbs_out, int32_t* pids_out, int* n_leaf_out,
                         int where) {
  using namespace rte;
  if (!c) return RTE_EINVAL;
  if (!pts || !aabbs_out || !pids_out || !n_leaf_out || np <= 0 || max_node <= 0 ||
      max_leaves <= 0 || stride < 3)
    return rte_fail(c, RTE_EINVAL, "bad kd-tree arguments");
  *n_leaf_out = 0;
  if (np > INT_MAX) return rte_fail(c, RTE_EINVAL, "kd-tree: np %lld exceeds int32 ids", (long long)np);
  if (max_node > kKdSmall)
    return rte_fail(c, RTE_EUNSUP, "GPU kd-tree: max_node %d > %d (use rte_build_kdtree)",
                    max_node, kKdSmall);
  if (hipSetDevice(c->device) != hipSuccess) return rte_fail(c, RTE_EHIP, "hipSetDevice");
  hipStream_t st = c->stream;
  auto ck = [&](hipError_t e, const char* what) {
    return e == hipSuccess ? RTE_OK : rte_fail(c, RTE_EHIP, "%s: %s", what, hipGetErrorString(e));
  };
#define KCK(expr, what) \
  do {                                  \
    if (int r_ = ck((expr), what)) return r_; \
  } while (0)
  DevBuf pin, work, outb;  // freed on return (hipFree waits for the device)
  const float* dp = pts;
  int64_t ds = stride;
  if (where == RTE_HOST) {  // only the three coordinates travel
    std::vector<float> p3((size_t)np * 3);
    for (int64_t i = 0; i < np; ++i)
      for (int a = 0; a < 3; ++a) p3[(size_t)i * 3 + a] = pts[i * stride + a];
    KCK(pin.reserve(p3.size() * sizeof(float)), "hipMalloc");
    KCK(hipMemcpyAsync(pin.p, p3.data(), p3.size() * sizeof(float), hipMemcpyHostToDevice, st),
        "copy");
    KCK(hipStreamSynchronize(st), "sync");
    dp = pin.as<float>();
    ds = 3;
  }
  // leaves and small nodes: no more than points
  const int cap = (int)std::min<int64_t>(max_leaves, np);
  const int64_t chunks = (np + kKdChunk - 1) / kKdChunk;
  const int64_t max_nodes = np / (kKdSmall + 1) + 1, max_blocks = np / kKdChunk + max_nodes;
  KdWork w{};
  LeafRec* leaves = nullptr;
  int *dstart = nullptr, *dcount = nullptr;
  auto lay = [&](char* base) {
    size_t at = 0;
    auto take = [&](auto*& p, size_t n) {
      p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(base + at);
      at = (at + n * sizeof(*p) + 255) & ~(size_t)255;
    };
    for (int i = 0; i < 2; ++i) {
      take(w.rec[i], np);
      take(w.nodes[i], max_nodes);
      take(w.map[i], max_blocks);
    }
    take(w.idx, np);
    take(w.mark, np);
    take(w.marks, chunks);
    take(w.segs, cap);
    take(w.h, 1);
    take(leaves, cap);
    take(dstart, cap);
    take(dcount, cap);
    return at;
  };
  KCK(work.reserve(lay(nullptr)), "hipMalloc(kd-tree work)");
  lay(work.as<char>());
  w.np = np;
  w.cap = cap;
  hipLaunchKernelGGL(kd_start_kernel, dim3(1), dim3(64), 0, st, w);
  hipLaunchKernelGGL(kd_root_kernel, dim3((unsigned)chunks), dim3(256), 0, st, dp, ds, w,
                     w.nodes[1]);
  // the root's plan, then rounds: two more than halving takes, one of them empty
  // as a rule, and then two at a time while nodes are left
  hipLaunchKernelGGL(kd_plan_kernel, dim3(1), dim3(1024), 0, st, w, 1);
  int rounds = 0;
  for (int64_t n = np; n > kKdSmall; n = (n + 1) / 2) ++rounds;
  if (rounds) ++rounds;
  Header hh{};
  hh.ns = 1;  // a root that is a small node needs no rounds and no read-back
  for (int r = 0; rounds > 0; ++r) {
    const int par = r & 1;
    if (r >= rounds) {
      KCK(hipGetLastError(), "kd-tree kernels");
      KCK(hipMemcpyAsync(&hh, w.h, sizeof hh, hipMemcpyDeviceToHost, st), "copy");
      KCK(hipStreamSynchronize(st), "sync");
      if (hh.err & 1u) return rte_fail(c, RTE_EBUILD, "kd-tree split failed");
      if (hh.err & 2u) return rte_fail(c, RTE_EBUILD, "kd-tree split search did not end");
      if (hh.err & 4u) break;
      if (hh.m[par] == 0) break;
      rounds = r + 2;
    }
    for (int p = 0; p < kKdPasses; ++p)
      hipLaunchKernelGGL(kd_count_kernel, dim3((unsigned)max_blocks), dim3(256), 0, st, w, par, p);
    hipLaunchKernelGGL(kd_partition_kernel, dim3((unsigned)max_blocks), dim3(256), 0, st, w, par);
    hipLaunchKernelGGL(kd_plan_kernel, dim3(1), dim3(1024), 0, st, w, par);
  }
  if (!(hh.err & 4u)) {
    // boxes straight to the caller where it can hold all there may be
    KCK(outb.reserve(where == RTE_HOST ? (size_t)cap * 24 : 1), "hipMalloc");
    float* boxes = where == RTE_HOST ? outb.as<float>() : aabbs_out;
    hipLaunchKernelGGL(kd_small_kernel, dim3((unsigned)hh.ns), dim3(256), 0, st, w, max_node,
                       leaves, max_leaves);
    hipLaunchKernelGGL(kd_mark_kernel, dim3((unsigned)chunks), dim3(256), 0, st, w);
    hipLaunchKernelGGL(kd_order_kernel, dim3((unsigned)chunks), dim3(256), 0, st, w, leaves, dstart,
                       dcount, boxes);
    KCK(hipGetLastError(), "kd_small_kernel");
    KCK(hipMemcpyAsync(&hh, w.h, sizeof hh, hipMemcpyDeviceToHost, st), "copy");
    KCK(hipStreamSynchronize(st), "sync");
  }
  if (hh.err & 1u) return rte_fail(c, RTE_EBUILD, "kd-tree split failed");
  if (hh.err & 2u) return rte_fail(c, RTE_EBUILD, "kd-tree split search did not end");
  if ((hh.err & 4u) || hh.leaves > (unsigned)max_leaves)
    return rte_fail(c, RTE_EINVAL, "kd-tree: more than max_leaves=%d leaves", max_leaves);
  const int nl = (int)hh.leaves;
  int P = 1;
  while (P < max_node) P <<= 1;
  int32_t* dpids = pids_out;
  DevBuf pidb;
  if (where == RTE_HOST) {
    KCK(pidb.reserve((size_t)nl * max_node * sizeof(int32_t)), "hipMalloc");
    dpids = pidb.as<int32_t>();
  }
  hipLaunchKernelGGL(kd_pids_kernel, dim3(nl), dim3(256), 0, st, w.idx, dstart, dcount, max_node, P,
                     np, dpids);
  KCK(hipGetLastError(), "kd_pids_kernel");
  if (where == RTE_HOST) {
    KCK(hipMemcpyAsync(pids_out, dpids, (size_t)nl * max_node * sizeof(int32_t),
                       hipMemcpyDeviceToHost, st),
        "copy");
    KCK(hipMemcpyAsync(aabbs_out, outb.p, (size_t)nl * 24, hipMemcpyDeviceToHost, st), "copy");
  }
  KCK(hipStreamSynchronize(st), "sync");
#undef KCK
  *n_leaf_out = nl;
  return RTE_OK;
}

}  // extern "C"
