// Kernel entry points for the Voronoi clip and the restart bookkeeping.
#include <atomic>
#include <cstdio>
#include <cstdlib>

#include "voronoi_kernel.h"

namespace pg {
namespace {

// Fast kernel: in 3D 16 lanes x 4 slots = 64 vertex slots and 48 planes per
// seed, 4 seeds per wave; in 2D 8 lanes x 2 slots = 16 vertices and 24 planes, 8
// seeds per wave.  Large kernel: 16 lanes x 8 slots = 128 slots and 64 planes,
// for seeds whose cell outgrows these before max_t and max_p (rare).
template <int DIM, int G, int S>
__global__ void __launch_bounds__(64, (VoroCfg<DIM, G, S>::WAVES)) k_voronoi(ClipArgs a) {
    __shared__ VoroSmem<DIM, G, S> sm[VoroCfg<DIM, G, S>::SPW];
    // a first pass resumes nothing, and sets every seed's resume entry
    voronoi_group<DIM, G, S>(a.pts, a.n_total, a.seeds, a.nq, a.knn, a.k, a.max_p, a.max_t, nullptr, nullptr, a.fa.key, sm,
                             xcd_block(blockIdx.x, gridDim.x));
}

// Certificate restarts, which resume saved cells.
template <int DIM, int G, int S>
__global__ void __launch_bounds__(64, (VoroCfg<DIM, G, S>::WAVES)) k_voronoi_restart(ClipArgs a) {
    __shared__ VoroSmem<DIM, G, S> sm[VoroCfg<DIM, G, S>::SPW];
    voronoi_group<DIM, G, S>(a.pts, a.n_total, a.seeds, a.nq, a.knn, a.k, a.max_p, a.max_t, a.fa.resume, a.fa.cstate,
                             a.fa.key, sm, xcd_block(blockIdx.x, gridDim.x));
}

// Cells whose filtered predicate was degenerate, again with the exact
// predicate (128 vertex slots).
template <int DIM>
__global__ void __launch_bounds__(64, 1) k_voronoi_exact(ClipArgs a) {
    __shared__ VoroSmem<DIM, 16, 8> sm[VoroCfg<DIM, 16, 8>::SPW];
    voronoi_group<DIM, 16, 8, true>(a.pts, a.n_total, a.seeds, a.nq, a.knn, a.k, a.max_p, a.max_t, a.fa.resume,
                                    a.fa.cstate, a.fa.key, sm, blockIdx.x);
}

// Vertex-ball completion of seeds no row certifies (128 vertex slots).
template <int DIM>
__global__ void __launch_bounds__(64, 1) k_voronoi_ball(ClipArgs a, BallGrid bg) {
    using C = VoroCfg<DIM, 16, 8>;
    __shared__ VoroSmem<DIM, 16, 8> sm[C::SPW];
    __shared__ int32_t scr[C::SPW * (2 * 16 + 1)];
    bg.scr = scr;
    voronoi_group<DIM, 16, 8, false, true>(a.pts, a.n_total, a.seeds, a.nq, a.knn, a.k, a.max_p, a.max_t, a.fa.resume,
                                           a.fa.cstate, a.fa.key, sm, blockIdx.x, bg);
}

template <int DIM, int G, int S>
void run(const ClipArgs& a, bool restart, hipStream_t s) {
    using C = VoroCfg<DIM, G, S>;
    const unsigned nb = (unsigned)((a.nq + C::SPW - 1) / C::SPW);
    if (restart) k_voronoi_restart<DIM, G, S><<<dim3(nb), dim3(64), 0, s>>>(a);
    else k_voronoi<DIM, G, S><<<dim3(nb), dim3(64), 0, s>>>(a);
}

constexpr int TB = 256;
constexpr int PER = 8;  // seeds per thread of a collect

// A block's matches are counted first (per wave and round of 256 seeds), take
// one range of the list by one atomic, and are written in order; the tallies of
// the other statuses are the block's sums as well (a set of degenerate cells
// would queue an atomic per thread at one address; a mesh of 1M such cells
// 8.48 -> 8.44 ms).  One launch per collect; flags, a scan and a compaction were
// five.
__global__ void __launch_bounds__(TB) k_collect(int64_t nq_host, const int64_t* __restrict__ nq_dev,
                                                const uint32_t* __restrict__ seeds, const int32_t* __restrict__ status,
                                                int code, uint32_t* __restrict__ list, unsigned long long* tally,
                                                int counts) {
    __shared__ int32_t cnt[PER][TB / WAVE];
    __shared__ int32_t sum[2][TB / WAVE];
    __shared__ int64_t base_s;
    const int64_t nq = nq_dev ? *nq_dev : nq_host;
    const int64_t b0 = (int64_t)blockIdx.x * TB * PER;
    if (b0 >= nq) return;  // whole block
    const int w = threadIdx.x / WAVE, l = threadIdx.x & (WAVE - 1);
    uint32_t id[PER];
    bool hit[PER];
    int ov = 0, other = 0;
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const int64_t i = b0 + r * TB + threadIdx.x;
        id[r] = i < nq ? (seeds ? seeds[i] : (uint32_t)i) : 0u;
        const int st = i < nq ? status[id[r]] : SUCCESS;
        hit[r] = code < 0 ? st != SUCCESS : st == code && i < nq;
        const uint64_t m = (uint64_t)__ballot(hit[r]);
        if (l == 0) cnt[r][w] = __popcll(m);
        if (counts) {
            ov += __popcll(__ballot(st == SLOT_OVERFLOW));
            other += __popcll(__ballot(!hit[r] && st != SUCCESS && st != SLOT_OVERFLOW));
        }
    }
    if (l == 0) {  // the wave's
        sum[0][w] = ov;
        sum[1][w] = other;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        if (counts)
            for (int q = 0; q < 2; q++) {
                int t = 0;
                for (int v = 0; v < TB / WAVE; v++) t += sum[q][v];
                if (t) atomicAdd(tally + 1 + q, (unsigned long long)t);
            }
        int t = 0;
        for (int r = 0; r < PER; r++)
            for (int v = 0; v < TB / WAVE; v++) {
                const int c = cnt[r][v];
                cnt[r][v] = t;
                t += c;
            }
        base_s = t ? (int64_t)atomicAdd(tally, (unsigned long long)t) : 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; r++) {
        const uint64_t m = (uint64_t)__ballot(hit[r]);
        if (hit[r]) list[base_s + cnt[r][w] + __popcll(m & ((1ull << l) - 1ull))] = id[r];
    }
}

}  // namespace

// Fast-kernel shape in 3D: lanes per seed x vertex slots per lane.  16 x 4 (64
// slots, 4 seeds per wave), 16 x 3 (48 slots; less work per clip, a few
// more seeds overflow into the 128-slot kernel), 8 x 6 and 8 x 8 (8 seeds
// per wave: the group-wide work of a clip is shared by twice as many seeds,
// at twice the LDS per wave).  Chosen by the autotuner or PGPU_CLIP_CFG
// ("16x4", "16x3", "8x6", "8x8").  2D clips have one shape (CLIP2D_LANES).
static std::atomic<int> g_clip_lanes{16}, g_clip_slots{64};
static const bool g_clip_env = [] {
    const char* e = getenv("PGPU_CLIP_CFG");
    int l = 0, sl = 0;
    if (e && sscanf(e, "%dx%d", &l, &sl) == 2) set_clip_config(l, l * sl);
    const char* e2 = getenv("PGPU_CLIP_SLOTS");
    if (e2 && atoi(e2) == 48) set_clip_config(16, 48);
    return true;
}();
bool valid_clip_config(int lanes, int slots) {
    return (lanes == 16 || lanes == 8) && (slots == 48 || slots == 64);
}
void set_clip_config(int lanes, int slots) {
    if (!valid_clip_config(lanes, slots)) return;
    g_clip_lanes = lanes;
    g_clip_slots = slots;
}
int clip_lanes() { return g_clip_lanes; }
int clip_slots() { return g_clip_slots; }

// Certificate restarts resume the saved cell (default) or clip again from
// the first neighbour (PGPU_CLIP_RESUME=0); the results are the same.
static std::atomic<bool> g_clip_resume{[] {
    const char* e = getenv("PGPU_CLIP_RESUME");
    return !(e && atoi(e) == 0);
}()};
bool clip_resume() { return g_clip_resume; }
void set_clip_resume(bool on) { g_clip_resume = on; }

template <int DIM>
void launch_dim(const ClipArgs& a, int big, hipStream_t s, bool restart, int lanes, int slots, bool exact) {
    if (exact) {
        using C = VoroCfg<DIM, 16, 8>;
        k_voronoi_exact<DIM><<<dim3((unsigned)((a.nq + C::SPW - 1) / C::SPW)), dim3(64), 0, s>>>(a);
    } else if (big) run<DIM, 16, 8>(a, true, s);
    else if constexpr (DIM == 2) run<2, CLIP2D_LANES, CLIP2D_SLOTS / CLIP2D_LANES>(a, restart, s);
    else if (lanes == 8 && slots == 48) run<DIM, 8, 6>(a, restart, s);
    else if (lanes == 8) run<DIM, 8, 8>(a, restart, s);
    else if (slots == 48) run<DIM, 16, 3>(a, restart, s);
    else run<DIM, 16, 4>(a, restart, s);
}

void launch_voronoi(int dim, const double* sorted, int64_t n, const uint32_t* seeds, int64_t nq,
                    const uint32_t* knn, int k, int max_p, int max_t, int big, FaceArrays fa, int lanes, int slots,
                    hipStream_t s, bool restart, bool exact) {
    if (nq <= 0) return;
    (void)g_clip_env;
    const ClipArgs a{sorted, n, seeds, nq, nullptr, knn, nullptr, fa, k, max_p, max_t};
    if (dim == 2) launch_dim<2>(a, big, s, restart, lanes, slots, exact);
    else launch_dim<3>(a, big, s, restart, lanes, slots, exact);
}

void launch_voronoi_ball(int dim, const double* sorted, int64_t n, const uint32_t* seeds, int64_t nq,
                         const uint32_t* knn, int k, int max_p, int max_t, FaceArrays fa, int N,
                         const int32_t* starts, const int32_t* counts, const uint32_t* perm, int kmark,
                         hipStream_t s, SubGrid sg) {
    if (nq <= 0) return;
    BallGrid bg;
    bg.N = N;
    bg.starts = starts;
    bg.counts = counts;
    bg.perm = perm;
    bg.kmark = kmark;
    bg.sg = sg;
    const unsigned nb = (unsigned)((nq + 3) / 4);  // 4 seeds per wave
    const ClipArgs a{sorted, n, seeds, nq, nullptr, knn, nullptr, fa, k, max_p, max_t};
    if (dim == 2) k_voronoi_ball<2><<<dim3(nb), dim3(64), 0, s>>>(a, bg);
    else k_voronoi_ball<3><<<dim3(nb), dim3(64), 0, s>>>(a, bg);
}

void launch_collect(int64_t nq, const int64_t* nq_dev, const uint32_t* seeds, const int32_t* status, int code,
                    uint32_t* list, unsigned long long* tally, bool counts, hipStream_t s) {
    if (nq <= 0) return;
    k_collect<<<(unsigned)((nq + TB * PER - 1) / (TB * PER)), TB, 0, s>>>(nq, nq_dev, seeds, status, code, list, tally,
                                                                          counts ? 1 : 0);
}

}  // namespace pg
