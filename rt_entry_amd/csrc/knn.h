// Exact k-nearest-neighbour lists and the search graph built from them (knn.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rte {

constexpr int kKnnK = 64;        // list length computed by the kernel (k <= 64)
constexpr int kKnnMaxD = 256;    // dims held in registers

// ids/dists: nq x k (k <= kKnnK), the k nearest rows of X (np x d, row stride
// `stride`) to each of rows [row0, row0 + nq) of X, excluding the row itself,
// ordered by (squared distance, id).  With `unless`, nothing for whole-number data.
struct KnnFlags;
hipError_t launch_knn(const float* X, int64_t np, int d, int64_t stride, const float* norms,
                      int64_t row0, int64_t nq, int k, int32_t* ids, float* dists,
                      const KnnFlags* unless, hipStream_t st);
// Search graph from kNN lists (np x kf, by (dist, id)): forward and reverse
// (ranks < rev_rank) candidates, duplicates keep their smallest (rank, type),
// each row keeps `degree` by (rank, type, id), padded with np.  `work` holds
// graph_from_knn_work_bytes() bytes.
hipError_t launch_graph_from_knn(const int32_t* knn, int64_t np, int kf, int degree, int rev_rank,
                                 int32_t* graph, void* work, hipStream_t st);
size_t graph_from_knn_work_bytes(int64_t np, int kf, int rev_rank);
// What rules the whole-number kernel out, a word a bit: the call's epoch where the
// bit is set, so that nothing is cleared between calls.
constexpr uint32_t kKnnNotWhole = 1, kKnnNegative = 2, kKnnLarge = 4, kKnnLargeSigned = 8;
constexpr uint32_t kKnnVaried = 16;  // not most distances are equal
constexpr int kKnnFlagWords = 5;
struct KnnFlags {
  uint32_t* dev;   // device memory
  uint32_t* host;  // the same in mapped host memory
  uint32_t epoch;
  bool varied;  // the whole-number kernel is for varied data only
};
// Where most distances are equal the FP32 kernel, which meets the points in the
// order of their ids, passes over nearly all of them; the whole-number kernel looks
// at the ids of each.  Below one row of workgroups (128 rows a CU) that is the
// slower way: k = 64, equal points, 0.55 against 1.25 ms at 8000 x 32 and 1.85 against
// 2.6 at 20000 x 128 (8.2 against 5.7 at 50000; 0.32 against 0.23 at 256).
inline bool knn_varied_only(int64_t np, int cus) { return np >= 768 && np <= (int64_t)128 * cus; }
__host__ __device__ inline uint32_t knn_flag_bits(const uint32_t* words, uint32_t epoch) {
  uint32_t bits = 0;
  for (int b = 0; b < kKnnFlagWords; ++b) bits |= words[b] == epoch ? 1u << b : 0u;
  return bits;
}
__host__ __device__ inline bool knn_whole_numbers(uint32_t flag, bool varied) {
  return !(flag & (kKnnNotWhole | kKnnLarge)) && (!varied || (flag & kKnnVaried)) &&
         (flag & (kKnnNegative | kKnnLargeSigned)) != (kKnnNegative | kKnnLargeSigned);
}
inline int64_t knn_padded(int64_t np) { return (np + 63) / 64 * 64; }
// Row norms of X and, unless null, what the whole-number kernel needs: the bf16
// rows (knn_padded(np) x d), half = -norm / 2 (-inf past np), and the flags.
hipError_t launch_row_norms(const float* X, int64_t np, int d, int64_t stride, float* norms,
                            uint16_t* Xb, float* half, const KnnFlags* flags, hipStream_t st);
// launch_knn for data of which knn_whole_numbers(flags, false) holds and np <= kKnnWholeMax;
// same lists, for rows [row0, row0 + nrows).  cus: the card's compute units;
// `work` has knn_whole_bytes() bytes.
constexpr int64_t kKnnWholeMax = 1 << 27;
size_t knn_whole_bytes(int64_t np, int d, int64_t nrows, int cus);
hipError_t launch_knn_whole(const uint16_t* Xb, const float* half, int64_t np, int d, int64_t row0,
                            int64_t nrows, int k, int cus, void* work, int32_t* ids, float* dists,
                            hipStream_t st);

}  // namespace rte
