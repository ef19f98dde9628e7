// Chunks of a kd-tree node's points, one a workgroup.  Points are counted by int,
// and a node may hold up to INT_MAX of them: no sum here exceeds the node's end.
#pragma once

#ifdef __HIPCC__
#define RTE_KD_HD __host__ __device__ __forceinline__
#else
#define RTE_KD_HD inline
#endif

namespace rte {

constexpr int kKdChunk = 2048;  // points per workgroup in the rounds' kernels

struct KdChunk {
  int first, count;  // points [first, first + count)
};

// chunks of n points
RTE_KD_HD constexpr int kd_chunks(int n) { return n / kKdChunk + (n % kKdChunk != 0); }

// chunk i < kd_chunks(r - l) of the node [l, r)
RTE_KD_HD KdChunk kd_chunk(int l, int r, int i) {
  const int first = l + i * kKdChunk, left = r - first;
  return KdChunk{first, left < kKdChunk ? left : kKdChunk};
}

}  // namespace rte
