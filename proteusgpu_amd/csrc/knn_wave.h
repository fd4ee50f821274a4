// The wave-per-query KNN kernel (knn_core.h) and its launch, one instance per
// row length and sub-grid use (knn.hip: rows up to 256, knn_long.hip: longer).
#pragma once

#include "knn_core.h"

namespace pg {
namespace {

// waves per SIMD the register budget is sized for: 6 for rows up to 128,
// 5 up to 256; the long restart rows (up to 1024) are rare
template <int M>
constexpr int knn_wave_occupancy() { return M <= 2 ? 6 : (M <= 4 ? 5 : 2); }

// SUB: the grid has crowded cells with sub-grids (a separate instance, so
// that the uniform case keeps its registers)
template <int DIM, int M, bool SUB>
__global__ void __launch_bounds__(64, knn_wave_occupancy<M>())
    k_knn_wave(const double* __restrict__ sorted, const uint32_t* __restrict__ perm, int N,
               const int32_t* __restrict__ starts, const int32_t* __restrict__ counts,
               const uint32_t* __restrict__ queries, int64_t q0, int64_t nq, int k, uint32_t* __restrict__ out,
               KnnTail tail, SubGrid sg) {
    __shared__ KnnSmem<M> smem;
    const int64_t qi = q0 + xcd_block(blockIdx.x, gridDim.x);
    if (qi >= nq) return;  // whole block
    const uint32_t q = queries ? queries[qi] : (uint32_t)qi;
    int kp = 0;
    uint32_t lo = 0;
    tail_of(tail, q, k, kp, lo);
    knn_wave_query<DIM, M, SUB>(sorted, perm, N, 0, starts, counts, q, k, out + (size_t)qi * k, smem, kp, lo, sg);
}

template <int DIM, int M>
void run_wave(const double* sorted, const uint32_t* perm, int N, const int32_t* starts,
              const int32_t* counts, const uint32_t* queries, int64_t nq, int k, uint32_t* out,
              KnnTail tail, SubGrid sg, hipStream_t s) {
    // a launch of 2^32 threads or more wraps without an error: one block of 64
    // per query goes up to 2^26 queries (67.1M 2D points, k = 16: 44 ms a
    // call, the heap 51)
    constexpr int64_t MOST = (int64_t)1 << 25;
    for (int64_t q0 = 0; q0 < nq; q0 += MOST) {
        const unsigned nb = (unsigned)(nq - q0 < MOST ? nq - q0 : MOST);
        if (sg.m != nullptr)
            k_knn_wave<DIM, M, true><<<nb, 64, 0, s>>>(sorted, perm, N, starts, counts, queries, q0, nq, k, out, tail, sg);
        else
            k_knn_wave<DIM, M, false><<<nb, 64, 0, s>>>(sorted, perm, N, starts, counts, queries, q0, nq, k, out, tail, sg);
    }
}

}  // namespace
}  // namespace pg
