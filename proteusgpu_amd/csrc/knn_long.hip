// KNN rows of 257 to 1024 (certificate restarts of seeds beside dense
// clusters); a unit of its own, since these two instances take longest to
// compile.
#include "kernels.h"
#include "knn_wave.h"

namespace pg {

void launch_knn_long(int dim, const double* sorted, const uint32_t* perm, int N, const int32_t* starts,
                     const int32_t* counts, const uint32_t* queries, int64_t nq, int k, uint32_t* out, KnnTail tail,
                     SubGrid sg, hipStream_t s) {
    auto go = [&](auto f2, auto f3) { dim == 2 ? f2() : f3(); };
    if (k <= 512)
        go([&] { run_wave<2, 8>(sorted, perm, N, starts, counts, queries, nq, k, out, tail, sg, s); },
           [&] { run_wave<3, 8>(sorted, perm, N, starts, counts, queries, nq, k, out, tail, sg, s); });
    else
        go([&] { run_wave<2, 16>(sorted, perm, N, starts, counts, queries, nq, k, out, tail, sg, s); },
           [&] { run_wave<3, 16>(sorted, perm, N, starts, counts, queries, nq, k, out, tail, sg, s); });
}

}  // namespace pg
