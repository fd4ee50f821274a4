// Meshless Voronoi clipping on CDNA4: one 16-lane group per seed.
//
// Algorithm (cell.cpp:42-411, voronoi.cpp:115-156, after Ray et al. 2018):
// a seed's cell starts as the box [-1e-14, 1+1e-14]^d and is clipped by the
// bisector planes of its neighbours in KNN order; after every clip the cell
// is certified once the just-clipped neighbour is farther than twice the
// largest seed-vertex distance.  Vertices are plane triples (pairs in 2D).
//
// Layout on the GPU (differs from the reference, results do not):
//   * a wave64 holds SPW = 64/G seeds, G lanes each; a lane owns S vertex
//     slots, slot id gs = s*G + lane.  Per slot the lane keeps in registers
//     the vertex position, its squared seed distance and three float bounds
//     used by the filter below; which slots are live, removed or on the
//     cavity's rim are lane masks in scalar registers.
//   * planes (FP64), plane->neighbour ids, vertex plane triples and the
//     vertex adjacency (slot across each edge) live in LDS.
//   * row entries are taken in windows of 16; the ones whose plane cannot
//     reach the cell are passed over (see vertex_good), the matrix cores
//     making the 16 x vertices products of a window.
//   * a clip tests every live vertex in parallel.  The reference decides
//     with a 4x4 (3x3 in 2D) FP64 determinant per vertex; here
//     det ~= W * (e . p + e.w) is judged by its second factor, from the
//     cached vertex, against the test's rounding and eps bound over |W|
//     (SlotRegs, clip_step); a value below it goes to the reference
//     determinant and its eps test, evaluated exactly as written.  Decisions
//     and needs_exact_predicates flags are therefore identical to the
//     reference.
//   * the cavity boundary is found from the adjacency (an edge of a removed
//     vertex whose neighbour is kept), in parallel over removed vertices,
//     instead of the reference's serial walk; new vertices are the same
//     plane triples (cur, a, b) with the same orientation, so vertex
//     positions and the certificate are bit-identical to the reference.
//   * extraction walks each face's vertex cycle through the adjacency; face
//     order is plane order as in the reference (box planes, then KNN order).
//
// What bounds it: VALU issue (87 % of the SIMD cycles at three waves per SIMD,
// LDS 13.2 KB per wave).  At 1M uniform 3D seeds and k = 64 a wave of four
// seeds takes 24 clip steps of about 500 VALU instructions, a fifth of them
// the new vertices' Cramer rule, and 1.5k for the extraction: 16.0k in all,
// 8.7 ms (k = 32: 7.4 ms).  With one conflict bound in double per test, slot
// masks in vector registers, a loop per lane over its cavity edges, one
// vector prefix per use and the extraction by plane index it was 19.9k
// and 10.8 ms (9.3 ms).
#pragma once

#include "common.h"
#include "exact.h"
#include "kernels.h"
#include "simt.h"
#include "subgrid.h"

namespace pg {

struct Plane {
    double x, y, z, w;
};

// Fast kernels (at most 64 vertex slots) hold 48 planes per seed in 3D, which
// keeps a seed's LDS below 3.4 KB (three waves per SIMD), and 24 in 2D; a
// seed that needs more planes before max_p, or more vertex slots, is redone
// by the 128-slot kernel, which holds the full 64 planes.  2D cells have six
// vertices and a clip makes two: 8 lanes x 2 slots per seed, 8 seeds per
// wave.  At 16 x 4, 4 seeds per wave, as in 3D, three lanes of four had
// nothing to do: 1M uniform seeds at k = 16 2.66 -> 1.06 ms.
template <int DIM, int G, int S>
struct VoroCfg {
    static constexpr int NS = G * S;               // vertex slots per seed
    static constexpr int SPW = 64 / G;             // seeds per wave (= block)
    static constexpr int MAXP = NS > 64 ? 64 : (DIM == 3 ? 48 : 24);  // plane slots per seed
    static constexpr int NW = (NS + 63) / 64;      // 64-bit words of a slot mask
    static constexpr int PPL = MAXP / G;           // planes per lane at extraction
    // waves per SIMD the register budget is sized for: the 16-lane fast
    // kernels fit three in LDS (under 3.4 KB per seed), the 2D one four
    static constexpr int WAVES = NS > 64 ? 1 : (DIM == 2 ? 4 : (G == 16 ? 3 : 1));
    static_assert(NS <= 128, "slot ids are bytes below 255");
    static_assert(G <= 64 && 64 % G == 0, "groups tile the wave");
    static_assert(MAXP % G == 0, "planes tile the group");
};

// A plane in LDS (2D: without z).
template <int DIM>
struct alignas(DIM == 3 ? 16 : 8) PlaneMem {
    double v[DIM + 1];
    PG_DEV PlaneMem& operator=(const Plane& p) {
        v[0] = p.x;
        v[1] = p.y;
        if (DIM == 3) v[2] = p.z;
        v[DIM] = p.w;
        return *this;
    }
    PG_DEV operator Plane() const { return Plane{v[0], v[1], DIM == 3 ? v[2] : 0.0, v[DIM]}; }
};

template <int DIM, int NS, int MAXP, int G>
struct SeedSmem {
    union {
        PlaneMem<DIM> plane[MAXP];  // planes while clipping
        double vpos[3 * NS];    // vertex positions during extraction
    };
    float pn1[MAXP];        // |x|+|y|+|z|+|w| rounded up
    int32_t pvid[MAXP];     // neighbour (sorted id) of each plane, -1 = box
    // per vertex x: its planes a | b << 8 | c << 16; y: the neighbour slots
    // across its edges (lines in 2D), byte e across edge e
    uint2 va[NS];
    union {
        struct {
            uint32_t edge[NS];        // boundary edges of the current clip
            uint8_t newslot[NS];      // slot of the j-th new vertex
            uint8_t by_start[DIM == 3 ? MAXP : 1];  // 3D: boundary edge starting at a plane
            uint8_t by_end[DIM == 3 ? MAXP : 1];    // 3D: boundary edge ending at a plane
            uint32_t nbi[G];   // window of the neighbour row, one entry per lane
            double nbp[G][DIM];  // and the neighbours' positions
        };
        struct {  // extraction
            uint32_t first[MAXP];  // vertex of each plane with the lowest plane key
            uint8_t plist[MAXP];   // planes holding a vertex, in plane order
        };
    };
};

template <int DIM, int G, int S>
using VoroSmem = SeedSmem<DIM, VoroCfg<DIM, G, S>::NS, VoroCfg<DIM, G, S>::MAXP, G>;

// Round a non-negative double up to float (next float above on inexact).
PG_DEV float f2f_up(double d) {
    float f = (float)d;
    if ((double)f < d) f = __int_as_float(__float_as_int(f) + 1);
    return f;
}
PG_DEV int tri_p(uint32_t t, int e) { return (int)((t >> (8 * e)) & 0xffu); }
// write byte e of a vertex's adjacency
PG_DEV void set_adj(uint2& v, int e, int slot) { reinterpret_cast<uint8_t*>(&v.y)[e] = (uint8_t)slot; }

// Slot-independent identity of a vertex: its planes, sorted, packed in 24
// bits (16 in 2D).
template <int DIM>
PG_DEV uint32_t vertex_key(uint32_t t) {
    uint32_t a = t & 0xffu, b = (t >> 8) & 0xffu;
    if (DIM == 2) return a < b ? (a << 8) | b : (b << 8) | a;
    uint32_t c = (t >> 16) & 0xffu, x;
    if (a > b) { x = a; a = b; b = x; }
    if (b > c) { x = b; b = c; c = x; }
    if (a > b) { x = a; a = b; b = x; }
    return (a << 16) | (b << 8) | c;
}

// bit gs < 64 NW of a slot mask
template <int NW>
PG_DEV bool mask_has(const uint64_t (&m)[NW], int gs) {
    return (m[NW == 1 ? 0 : gs >> 6] >> (gs & 63)) & 1ull;
}
// Vertex of three planes (two lines in 2D) by the reference's Cramer rule
// (cell.cpp:388-411), homogeneous part (X, Y, Z, W).
template <int DIM>
PG_DEV void cramer(const Plane& a, const Plane& b, const Plane& c, double& X, double& Y, double& Z,
                   double& W) {
    if (DIM == 2) {
        X = -det2(a.w, a.y, b.w, b.y);
        Y = -det2(a.x, a.w, b.x, b.w);
        Z = 0.0;
        W = det2(a.x, a.y, b.x, b.y);
    } else {
        X = -det3(a.w, a.y, a.z, b.w, b.y, b.z, c.w, c.y, c.z);
        Y = -det3(a.x, a.w, a.z, b.x, b.w, b.z, c.x, c.w, c.z);
        Z = -det3(a.x, a.y, a.w, b.x, b.y, b.w, c.x, c.y, c.w);
        W = det3(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z);
    }
}

// The reference conflict predicate (cell.cpp:175-221), evaluated exactly.
template <int DIM>
PG_DEV bool conflict_exact(const Plane& p1, const Plane& p2, const Plane& p3, const Plane& e,
                           bool& flag, double xb = 0.0) {
    double det, eps;
    if (DIM == 2) {
        det = det3(p1.x, p2.x, e.x, p1.y, p2.y, e.y, p1.w, p2.w, e.w);
        double mx = fmax(fmax(fabs(p1.x), fabs(p2.x)), fabs(e.x));
        double my = fmax(fmax(fabs(p1.y), fabs(p2.y)), fabs(e.y));
        double mw = fmax(fmax(fabs(p1.w), fabs(p2.w)), fabs(e.w));
        double mm = fmax(fmax(mx, my), mw);
        eps = 1e-14 * mx * my * mw;
        eps *= mm;
    } else {
        det = det4(p1.x, p2.x, p3.x, e.x, p1.y, p2.y, p3.y, e.y, p1.z, p2.z, p3.z, e.z, p1.w, p2.w,
                   p3.w, e.w);
        double mx = fmax(fmax(fmax(fabs(p1.x), fabs(p2.x)), fabs(p3.x)), fabs(e.x));
        double my = fmax(fmax(fmax(fabs(p1.y), fabs(p2.y)), fabs(p3.y)), fabs(e.y));
        double mz = fmax(fmax(fmax(fabs(p1.z), fabs(p2.z)), fabs(p3.z)), fabs(e.z));
        eps = 1e-14 * mx * my * mz;
        double mm = fmax(fmax(mx, my), mz);
        eps *= (mm * mm);
    }
    if (fabs(det) < eps || fabs(det) < xb) flag = true;
    return det > 0.0;
}

// |x| + |y| + |z| + wm rounded up to float, wm = |w| (or, in exact mode, the
// magnitude that bounds the rounding error of w, see XTOL)
PG_DEV float plane_n1(const Plane& p, double wm) { return f2f_up(fabs(p.x) + fabs(p.y) + fabs(p.z) + wm); }

// Per-seed register state of one lane.  Per slot: the vertex position, its
// squared seed distance (float, +inf when not finite), and its share of the
// conflict test's bound over |W|, W the vertex's Cramer denominator (floats
// rounded up; see clip_step): qw = q / |W|, q bounding the product of the
// planes' 1-norms, ew = eps / |W|, eps the eps_bound of the largest of them,
// iw = 1 / |W|, made once with the vertex.  iw = +inf (every test of the vertex
// is decided exactly) unless W is negative, as it is for a proper vertex.
template <int S>
struct SlotRegs {
    double px[S], py[S], pz[S];
    float d2[S], qw[S], ew[S], iw[S];
    bool live[S];  // slot s holds a vertex (lane masks in scalar registers)
};

// An upper bound (float, at least the smallest normal float) of 1.0000001e-14
// m^5 (m^4 in 2D): the reference's conflict eps (cell.cpp:175-221) is 1e-14
// times a product of five, or four, component maxima, each at most the
// largest 1-norm m of the planes involved.  Rounding of the products is
// monotone, so the bound of max(a, b) is the max of the bounds.
template <int DIM>
PG_DEV float eps_bound(float m) {
    // The constant, 1.000001e-14 as a float (relative error below 6e-8), and
    // at most four products, each within 2^-24 of the exact one, stay above
    // 1.0000001e-14 m^5.  When that bound is a normal float every
    // intermediate is normal too (m^k >= m^5 / 1e-14 for m < 1); a result
    // below the smallest normal float, subnormal or flushed to zero, is
    // raised to it by the integer max on its bit pattern (non-negative).
    const float m2 = m * m;
    const float mp = DIM == 3 ? m2 * m2 * m : m2 * m2;
    return __uint_as_float(max(__float_as_uint(mp * 1.000001e-14f), 0x00800000u));
}

template <int DIM, int S>
PG_DEV void slot_write(SlotRegs<S>& r, int s, double px, double py, double pz, float d2, float qw, float ew,
                       float iw) {
#pragma unroll
    for (int i = 0; i < S; i++) {
        if (i == s) {
            r.px[i] = px;
            r.py[i] = py;
            r.pz[i] = pz;
            r.d2[i] = d2;
            r.qw[i] = qw;
            r.ew[i] = ew;
            r.iw[i] = iw;
            r.live[i] = true;
        }
    }
}

// Squared seed distance of a vertex (cell.cpp:369-384's arithmetic).
PG_DEV double vertex_d2(double px, double py, double pz, double sx, double sy, double sz) {
    const double dx = px - sx, dy = py - sy, dz = pz - sz;
    return dx * dx + dy * dy + dz * dz;
}

// A new vertex of planes a, b, c (reference arithmetic for the position,
// cell.cpp:388-411) into slot s; na, nb, nc: the planes' 1-norms.
template <int DIM, int S>
PG_DEV void make_vertex(SlotRegs<S>& r, int s, const Plane& a, const Plane& b, const Plane& c, float na, float nb,
                        float nc, double sx, double sy, double sz, float& qw, float& ew, float& iw) {
    double X, Y, Z, W;
    cramer<DIM>(a, b, c, X, Y, Z, W);
    const double px = X / W, py = Y / W, pz = DIM == 3 ? Z / W : 0.0;
    const float d = (float)vertex_d2(px, py, pz, sx, sy, sz);
    // the bounds' products and v_rcp_f32 are each within 2^-22; 1.00001 covers them
    const float aw = -(float)W;
    iw = aw > 1e-37f ? __builtin_amdgcn_rcpf(aw) * 1.00001f : __builtin_inff();
    qw = (DIM == 3 ? na * nb * nc : na * nb) * 1.000001f * iw;
    ew = eps_bound<DIM>(fmaxf(fmaxf(na, nb), nc)) * iw;
    slot_write<DIM, S>(r, s, px, py, pz, d <= 3e38f ? d : __builtin_inff(), qw, ew, iw);
}

// The initial box cell (cell.cpp:84-103): per vertex its planes, and the
// vertices across its edges (edge e of a 3D vertex joins planes e, e + 1 mod
// 3 and leads to the vertex holding them in the other order; line e of a 2D
// vertex to the other vertex on it).
template <int DIM>
struct InitCell {
    uint32_t tri[8], adj[8];
};
template <int DIM>
constexpr InitCell<DIM> init_cell() {
    InitCell<DIM> c{};
    const uint32_t T3[8] = {2 | 5 << 8 | 0 << 16, 5 | 3 << 8 | 0 << 16, 1 | 5 << 8 | 2 << 16, 5 | 1 << 8 | 3 << 16,
                            4 | 2 << 8 | 0 << 16, 4 | 0 << 8 | 3 << 16, 2 | 4 << 8 | 1 << 16, 4 | 3 << 8 | 1 << 16};
    const uint32_t T2[4] = {2 | 0 << 8, 1 | 2 << 8, 3 | 1 << 8, 0 | 3 << 8};
    const int n = DIM == 3 ? 8 : 4;
    for (int i = 0; i < n; i++) c.tri[i] = DIM == 3 ? T3[i] : T2[i];
    for (int i = 0; i < n; i++)
        for (int e = 0; e < DIM; e++)
            for (int j = 0; j < n; j++)
                for (int f = 0; f < DIM; f++) {
                    if (j == i) continue;
                    const uint32_t ae = (c.tri[i] >> (8 * e)) & 0xff, be = (c.tri[i] >> (8 * ((e + 1) % DIM))) & 0xff;
                    const uint32_t af = (c.tri[j] >> (8 * f)) & 0xff, bf = (c.tri[j] >> (8 * ((f + 1) % DIM))) & 0xff;
                    if (DIM == 3 ? (af == be && bf == ae) : (af == ae)) c.adj[i] |= (uint32_t)j << (8 * e);
                }
    return c;
}

// Saved clip state (CLIP_STATE_BYTES per seed): planes, their bounds and
// neighbour ids, then per vertex slot its planes (0xffffffff: empty slot)
// and adjacency (as in LDS), then the plane and live-vertex counts.
struct ClipState {
    Plane plane[64];
    float pn1[64];
    int32_t pvid[64];
    uint2 va[64];
    int32_t nb_v, nlive;
};
static_assert(sizeof(ClipState) <= CLIP_STATE_BYTES, "clip state layout");

// Exact decision of a degenerate conflict test (exact.h) from the vertex's
// plane triple tt, the new plane's point b (sorted id z) and the seed.
template <int DIM, class SM>
__device__ __noinline__ int exact_conflict(uint32_t tt, const SM& sm, const double* pts,
                                           uint32_t sid, const double* sp, uint32_t z, const double* bp,
                                           const uint32_t* key) {
    XRow rows[DIM + 1];
    for (int r = 0; r < DIM; r++) {
        const int pid = (int)tri_p(tt, r);
        XRow& x = rows[r];
        x.box = pid < 2 * DIM;
        x.p[0] = x.p[1] = x.p[2] = 0.0;
        x.key = 0;
        x.axis = pid >> 1;
        x.sg = (pid & 1) ? -1.0 : 1.0;
        x.c = (pid & 1) ? 1.0 + 1e-14 : -1e-14;  // the box bounds of the initial cell
        if (!x.box) {
            const uint32_t q = (uint32_t)sm.pvid[pid];
            for (int d = 0; d < DIM; d++) x.p[d] = pts[(size_t)DIM * q + d];
            x.key = key ? key[q] : q;
        }
    }
    XRow& e = rows[DIM];
    e.box = false;
    e.axis = 0;
    e.sg = 1.0;
    e.c = 0.0;
    e.p[0] = bp[0];
    e.p[1] = bp[1];
    e.p[2] = bp[2];
    e.key = key ? key[z] : z;
    return conflict_sos<DIM>(sp, key ? key[sid] : sid, rows);
}

// Vertex-ball completion (BALL kernels; no reference counterpart): a seed
// whose certificate no row of k_max neighbours reaches is finished by the
// empty-sphere test.  After the first kb neighbours of its row, while the
// ball of some vertex v (centre v, radius |v - s|) strictly holds a point
// that is not one of the cell's planes, the cell is clipped by the
// candidate nearest the seed ((distance, input index) order) among the
// vertices' candidates, each the point nearest its vertex (smallest input
// index on ties); when no ball holds one, every vertex is a vertex of the
// Voronoi diagram and the cell is certified (kcert = kmark).  A candidate
// stays valid while its vertex lives: a clip by p removes every vertex whose
// ball holds p.  A ball search visits grid rings out to BALL_RINGS; one that
// would need more leaves the seed uncertified.
constexpr int BALL_RINGS = 32;

struct BallGrid {
    int N = 0;                        // grid cells per axis of the sorted points
    const int32_t* starts = nullptr;  // first sorted id per grid cell
    const int32_t* counts = nullptr;  // points per grid cell
    const uint32_t* perm = nullptr;   // input index per sorted id (ties)
    int kmark = 0;                    // kcert of a cell the completion certifies
    int32_t* scr = nullptr;           // LDS, 2 G + 1 ints per seed group (the group search's tables)
    SubGrid sg;                       // sub-grids of the crowded cells (none: sg.m == nullptr)
};

// Lower bound of the squared distance from v to any point of grid cell ix:
// boundary cells are open outwards (points beyond the unit box are clamped
// into them); a slack of 1e-9 cell widths per axis and a factor 1 - 1e-12
// keep it below the rounded distance of every point of the cell, so a cell
// whose bound is at least the best distance so far holds no point that
// would be picked.
template <int DIM>
PG_DEV double ball_cell_lb2(int N, const double (&v)[3], const int (&ix)[3]) {
    const double h = 1.0 / N;
    double s = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const double lo = ix[d] == 0 ? -1e300 : ix[d] * h;
        const double hi = ix[d] == N - 1 ? 1e300 : (ix[d] + 1) * h;
        const double e = fmax(fmax(lo - v[d], v[d] - hi) - 1e-9 * h, 0.0);
        s += e * e;
    }
    return s * (1.0 - 1e-12);
}

// The point nearest v strictly inside the ball (v, r2) that is neither the
// seed nor a plane of the cell ((distance, input index) order); -1: none;
// -2: beyond BALL_RINGS.  Found by the whole group: the cells of a grid
// ring are taken G at a time, their points spread over the group's lanes
// (prefix sum of the cell counts, a binary search per lane), and the
// group's best is reduced at the end of every ring.  With the bounds of
// ball_cell_lb2 the answer is the argmin over all points, and the ring at
// which the walk stops depends only on the rings before it: the order the
// points are visited in does not matter.  A crowded cell (one with a
// sub-grid) is taken sub-cell by sub-cell, only the sub-cells the ball of
// the best so far reaches (sub_lower_d2 bounds them the same way).  v, r2,
// sid: the same on every lane of the group, every lane of which is active;
// shift / gmask: the group's lanes in a ballot; cst / cpf: the group's LDS
// tables (G and G + 1 entries).
template <int DIM, int G>
PG_DEV int32_t ball_search_group(const BallGrid& bg, const double* __restrict__ pts, const double (&v)[3], double r2,
                                 uint32_t sid, const int32_t* pvid, int nb_v, int gl, int shift, uint64_t gmask,
                                 int32_t* cst, int32_t* cpf) {
    const int N = bg.N;
    const double h = 1.0 / N;
    int cc[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < DIM; d++) cc[d] = max(0, min(N - 1, (int)floor(v[d] * N)));
    double best = r2;
    int32_t pick = -1;
    for (int ring = 0;; ring++) {
        if (ring > 1) {
            // a point of ring r lies more than r - 1 cell widths away
            const double lb = ((ring - 1) - 1e-9) * h;
            if (lb * lb * (1.0 - 1e-12) >= best) break;
        }
        if (ring > N) break;
        if (ring > BALL_RINGS) return -2;
        const int side = 2 * ring + 1;
        const int ncube = DIM == 3 ? side * side * side : side * side;
        double lbest = best;
        int32_t lpick = pick;
        // points 0 .. total-1 of the cells (or sub-cells) in cst / cpf
        // (first position, exclusive prefix), G at a time; positions are
        // sorted ids, or indices into indir
        auto scan = [&](int total, const uint32_t* __restrict__ indir) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int cb = 0; cb < total; cb += G) {
                const int j = cb + gl;
                if (j >= total) continue;
                // cell holding point j: largest a with cpf[a] <= j
                int lo = 0, hi = G - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (cpf[mid] <= j) lo = mid;
                    else hi = mid - 1;
                }
                int32_t q = cst[lo] + (j - cpf[lo]);
                if (indir != nullptr) q = (int32_t)indir[q];
                if ((uint32_t)q == sid) continue;
                double d2 = 0.0;
#pragma unroll
                for (int d = 0; d < DIM; d++) {
                    const double df = pts[(size_t)DIM * q + d] - v[d];
                    d2 += df * df;
                }
                // strictly inside; on ties the smaller input index
                if (d2 > lbest || (d2 == lbest && (lpick < 0 || bg.perm[q] > bg.perm[lpick]))) continue;
                bool plane = false;
                for (int pl = 0; pl < nb_v && !plane; pl++) plane = pvid[pl] == q;
                if (plane) continue;
                lbest = d2;
                lpick = q;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        for (int base = 0; base < ncube; base += G) {
            const int t = base + gl;
            int32_t st = 0, cnt = 0;
            bool crowded = false;  // a cell with a sub-grid: taken sub-cell by sub-cell below
            int ix[3] = {0, 0, 0};
            if (t < ncube) {
                const int di = t % side - ring, dj = (t / side) % side - ring;
                const int dk = DIM == 3 ? t / (side * side) - ring : 0;
                const int cheb = max(abs(di), max(abs(dj), abs(dk)));
                ix[0] = cc[0] + di;
                ix[1] = cc[1] + dj;
                ix[2] = cc[2] + dk;
                if (cheb == ring && ix[0] >= 0 && ix[1] >= 0 && ix[2] >= 0 && ix[0] < N && ix[1] < N &&
                    (DIM == 2 || ix[2] < N) && ball_cell_lb2<DIM>(N, v, ix) < best) {
                    const int64_t cell = ix[0] + (int64_t)ix[1] * N + (int64_t)ix[2] * N * N;
                    if (bg.sg.m != nullptr && bg.sg.m[cell] > 0) {
                        crowded = true;
                    } else {
                        st = bg.starts[cell];
                        cnt = bg.counts[cell];
                    }
                }
            }
            const int incl = group_incl_sum<G>(cnt, gl);
            const int total = group_last<G>(incl);
            if (total > 0) {
                cst[gl] = st;
                cpf[gl + 1] = incl;
                if (gl == 0) cpf[0] = 0;
                scan(total, nullptr);
            }
            // the crowded cells of this batch, one at a time: their
            // sub-cells that the ball of the ring-start best can reach
            uint64_t crowd = (wave_ballot(crowded) >> shift) & gmask;
            while (crowd != 0ull) {
                const int a = ffs64(crowd);
                crowd &= crowd - 1ull;
                const int cx[3] = {shfl(ix[0], a, G), shfl(ix[1], a, G), shfl(ix[2], a, G)};
                const int64_t cell = cx[0] + (int64_t)cx[1] * N + (int64_t)cx[2] * N * N;
                const int m = bg.sg.m[cell];
                const int64_t sbase = bg.sg.ptr[cell];
                const double P[3] = {v[0] * N, v[1] * N, DIM == 3 ? v[2] * N : 0.0};
                int lo[3], hi[3];
                sub_box<DIM>(P, cx, m, N, best, lo, hi);
                const int nx = hi[0] - lo[0] + 1, ny = hi[1] - lo[1] + 1, nz = hi[2] - lo[2] + 1;
                const int nbox = nx * ny * nz;
                for (int b0 = 0; b0 < nbox; b0 += G) {
                    const int u = b0 + gl;
                    int32_t sst = 0, scnt = 0;
                    if (u < nbox) {
                        const int sx[3] = {lo[0] + u % nx, lo[1] + (u / nx) % ny, lo[2] + u / (nx * ny)};
                        if (sub_lower_d2<DIM>(P, cx, sx, m, N) < best) {
                            const int64_t j = sbase + sx[0] + (int64_t)m * (sx[1] + (int64_t)m * sx[2]);
                            sst = bg.sg.start[j];
                            scnt = bg.sg.cnt[j];
                        }
                    }
                    const int sincl = group_incl_sum<G>(scnt, gl);
                    const int stotal = group_last<G>(sincl);
                    if (stotal == 0) continue;
                    cst[gl] = sst;
                    cpf[gl + 1] = sincl;
                    if (gl == 0) cpf[0] = 0;
                    scan(stotal, bg.sg.idx);
                }
            }
        }
        // the group's best after this ring
        best = lbest;
        pick = lpick;
#pragma unroll
        for (int d = 1; d < G; d <<= 1) {
            const double od = shfl_xor(best, d, G);
            const int32_t oq = shfl_xor(pick, d, G);
            if (oq >= 0 && (pick < 0 || od < best || (od == best && bg.perm[oq] < bg.perm[pick]))) {
                best = od;
                pick = oq;
            }
        }
    }
    return pick;
}

// ---- passing over row entries that cannot cut the cell
//
// In a uniform 3D set about 45 row entries are walked per seed and 16 of
// them cut the cell; a step that cuts nothing costs a conflict test of every
// vertex, and idles the wave's other seeds or waits for their cuts.  With
// the entries passed over, a wave of four seeds takes 24 steps at k = 64,
// 22 of which cut a cell of it, and 19.5 of which each seed uses.  Measured
// (1M uniform seeds, first pass): k = 64 12.7 -> 10.8 ms (26.2k -> 19.9k
// VALU per wave), k = 32 10.1 -> 9.3 ms, 2D k = 16 3.4 -> 3.1 ms.  An entry with offset d = b - s cuts nothing when
// d . (v - s) < |d|^2 / 2 for every vertex v, and then neither it nor any
// later test of it can cut the cell, which only shrinks: the vertices made
// later lie in the hull of the present ones.  The filter tests that in
// float with a margin of SKIP_MARGIN |d|^2 and a slack for its own rounding.
//
// What is passed over would have been tested exactly: the reference flags a
// cell when a conflict determinant W f (f = |d|^2/2 - d . (v - s)) is below
// its eps, which a tiny W can bring about whatever f is, and a vertex with a
// tiny W has an uncertain position.  A vertex is good when its W < 0 and
// |W| SKIP_F E^2 exceeds twice the bound the conflict test trusts its
// filtered value above (5.4e-15 n1(e) q + the eps bounds) for every offset
// length E of the window (E0 <= E <= E1; n1(e) <= a E, a = 1.75 + |s|_1 +
// E1/2, since |w| = |d . (s + b)| / 2).  Its position is then within
// SKIP_F E0 / 4 of exact, so with f >= SKIP_MARGIN E^2 at every vertex at the
// time of the filter, f >= SKIP_F E^2 at every good vertex made later, and
// every test passed over would have ended in "kept", unflagged.  While a
// vertex that is not good lives, nothing is passed over.
constexpr float SKIP_MARGIN = 1.0f / 32;
constexpr float SKIP_F = 1.0f / 64;
// clips after which the rest of a window is filtered again
constexpr int REFILTER = 4;
// 4 with the margin of the certificate's float compare
constexpr float CERT_HI = 4.0f * (1.0f + 4e-7f), CERT_LO = 4.0f * (1.0f - 4e-7f);

struct SkipBounds {
    float g1, g2, g3;  // SKIP_F > g1 qw + g2 ew + g3 iw
};
PG_DEV bool vertex_good(const SkipBounds& g, float qw, float ew, float iw) {
    return fmaf(g.g1, qw, fmaf(g.g2, ew, g.g3 * iw)) < SKIP_F;
}
// wf: squared distance of this lane's entry, ascending over the pend
// entries of the window (lanes 0 ..).
template <int D, int G>
PG_DEV SkipBounds window_bounds(float wf, uint32_t pend, double sx, double sy, double sz) {
    const float lo = shfl(wf, 0, G), hi = shfl(wf, pend ? 31 - __builtin_clz(pend) : 0, G);
    const float iE0 = __builtin_amdgcn_rsqf(lo) * 1.001f, E1 = __builtin_amdgcn_sqrtf(hi) * 1.001f;
    const float a = 1.75f + (float)(fabs(sx) + fabs(sy) + fabs(sz)) + 0.5f * E1;
    const float a2 = a * a;
    SkipBounds g;
    g.g1 = 1.2e-14f * a * iE0;
    g.g2 = 2.1f * (iE0 * iE0);
    g.g3 = D == 3 ? 2.1e-14f * a2 * a2 * a * E1 * E1 * E1 : 2.1e-14f * a2 * a2 * E1 * E1;
    return g;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
// Lane l's max over the lanes of equal l % 16 of m_(l / 16): the maxima of
// the four rows' values, row r keeping that of m_r (two row swaps).
PG_DEV int rows_max_scatter(int m0, int m1, int m2, int m3) {
    const auto a = __builtin_amdgcn_permlane32_swap((uint32_t)m0, (uint32_t)m2, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap((uint32_t)m1, (uint32_t)m3, false, false);
    const int x = max((int)a[0], (int)a[1]), y = max((int)b[0], (int)b[1]);
    const auto c = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
    return max((int)c[0], (int)c[1]);
}

// Arguments of the clip kernels: the first (explicit) kernel argument, so
// that it starts the kernel-argument segment.  The output arrays are read
// from the segment again when the outputs are written: as ordinary arguments
// they would be loaded once and stay live across the clip, whose scalar
// registers hold the lane masks of its slots and would spill.
struct ClipArgs {
    const double* pts;      // sorted points
    int64_t n_total;        // seeds of the problem (exhaustive rows)
    const uint32_t* seeds;  // sorted ids to clip (nullptr: all)
    int64_t nq;             // their number,
    const int64_t* nq_dev;  // or its device address (batches)
    const uint32_t* knn;    // rows of length k
    unsigned long long* ticket;
    FaceArrays fa;
    int k, max_p, max_t;
    const int32_t* from = nullptr;  // batches: resume entries the pass goes on from (first pass: none)
};

// The first argument of the running kernel, through a pointer the compiler
// must treat as new.
template <class A>
PG_DEV const __attribute__((address_space(4))) A* fresh_args() {
    const __attribute__((address_space(4))) A* p =
        (const __attribute__((address_space(4))) A*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}
// a FaceArrays out of the argument segment, field by field
PG_DEV FaceArrays face_arrays_of(const __attribute__((address_space(4))) FaceArrays& a) {
    FaceArrays f;
    f.stride = a.stride;
    f.nbr = a.nbr;
    f.area = a.area;
    f.nrm = a.nrm;
    f.cen = a.cen;
    f.count = a.count;
    f.vol = a.vol;
    f.ccen = a.ccen;
    f.status = a.status;
    f.kcert = a.kcert;
    f.cstate = a.cstate;
    f.resume = a.resume;
    f.lastnb = a.lastnb;
    f.key = a.key;
    f.nbr_cm = a.nbr_cm;
    return f;
}

// Exact mode (fa.key set, or EXACT): a conflict test is trusted in floating
// point only above XTOL times the product of its rows' 1-norms (w measured
// by the magnitude its rounding is relative to), a valid bound on how far the
// rounding of the planes and of the determinant can move it; below, EXACT
// kernels decide it with exact_conflict and the others flag the cell
// (needs_exact_predicates) for them.  The certificate of EXACT kernels keeps
// a relative margin (CERT_TIE): a neighbour tied with twice the largest
// vertex distance can still cut a zero-area face under the symbolic
// perturbation, so only neighbours clearly beyond it certify the cell; the
// other kernels flag a near tie.
// BALL: the row is clipped whole, then the vertex-ball completion above
// certifies the cell.
template <int DIM, int G, int S, bool EXACT = false, bool BALL = false>
__device__ __forceinline__ void voronoi_group(const double* __restrict__ pts, int64_t n_total, const uint32_t* __restrict__ seeds,
                              int64_t nq, const uint32_t* __restrict__ knn, int k, int max_p, int max_t,
                              const int32_t* resume, const uint8_t* cstate, const uint32_t* key,
                              VoroSmem<DIM, G, S>* smem, int64_t vblock, BallGrid bg = {}) {
    using C = VoroCfg<DIM, G, S>;
    constexpr int NS = C::NS, NW = C::NW, MAXP = C::MAXP;
    constexpr int D = DIM;
    constexpr bool SKIP = !EXACT && (G == 16 || G == 8);  // row entries may be passed over
    const int tid = (int)threadIdx.x;
    const int grp = tid / G, gl = tid % G;
    const int shift = grp * G;
    const uint64_t gmask = (G == 64) ? ~0ull : ((1ull << G) - 1ull);
    const int64_t qi = vblock * C::SPW + grp;
    const bool valid = qi < nq;
    VoroSmem<DIM, G, S>& sm = smem[grp];
    if (max_p > FACE_SLOTS) max_p = FACE_SLOTS;
    // exact mode (a build with the exact-predicate fallback): every test
    // whose sign the rounding of the planes could flip is decided exactly
    // (EXACT kernels) or flags the cell for them (the others)
    const bool xmode = EXACT || key != nullptr;

    const uint32_t sid = valid ? (seeds ? seeds[qi] : (uint32_t)qi) : 0u;
    const uint32_t* row = knn + (valid ? (size_t)qi * (size_t)k : 0);
    const double sx = pts[(size_t)D * sid], sy = pts[(size_t)D * sid + 1];
    const double sz = D == 3 ? pts[(size_t)D * sid + 2] : 0.0;

    // ---------------------------------------------------------------- init
    // A seed whose previous pass (same shape, shorter row) stopped
    // uncertified resumes from its saved cell at neighbour v0: clipping the
    // same planes in the same order is deterministic, so the cell equals a
    // pass over the longer row from scratch.
    const int32_t shape_tag = (G << 24) | (S << 16);
    int v0 = 0;
    if (valid && resume != nullptr && NS <= 64) {
        const int32_t r = resume[sid];
        if (r > 0 && (r & 0x7fff0000) == shape_tag && (r & 0xffff) < k) v0 = r & 0xffff;
    }
    const ClipState* cst = v0 ? reinterpret_cast<const ClipState*>(cstate + (size_t)sid * CLIP_STATE_BYTES)
                              : nullptr;
    int nb_v0 = 2 * D, nlive0 = D == 3 ? 8 : 4;
    if (v0) {
        nb_v0 = cst->nb_v;
        nlive0 = cst->nlive;
        for (int p = gl; p < nb_v0; p += G) {
            sm.plane[p] = cst->plane[p];
            sm.pn1[p] = cst->pn1[p];
            sm.pvid[p] = cst->pvid[p];
        }
#pragma unroll
        for (int i = 0; i < S; i++) {
            const int gs = i * G + gl;
            sm.va[gs] = cst->va[gs];
        }
    }
    // Box planes (cell.cpp:44-82): eps = 1e-14 margin.
    if (!v0 && gl < 2 * D) {
        const double eps = 1e-14, lo = -eps, hi = 1.0 + eps;
        Plane p;
        switch (gl) {
            case 0: p = {1.0, 0.0, 0.0, -lo}; break;
            case 1: p = {-1.0, 0.0, 0.0, hi}; break;
            case 2: p = {0.0, 1.0, 0.0, -lo}; break;
            case 3: p = {0.0, -1.0, 0.0, hi}; break;
            case 4: p = {0.0, 0.0, 1.0, -lo}; break;
            default: p = {0.0, 0.0, -1.0, hi}; break;
        }
        sm.plane[gl] = p;
        sm.pn1[gl] = plane_n1(p, fabs(p.w));
        sm.pvid[gl] = -1;
    }
    // Initial vertices (cell.cpp:84-103): planes, and the vertices across
    // their edges (edge e of a 3D vertex joins planes e and e + 1 mod 3).
    constexpr int NV0 = D == 3 ? 8 : 4;
    if (!v0 && gl < NV0) {
        constexpr InitCell<D> T = init_cell<D>();
        uint2 t = {0, 0};
#pragma unroll
        for (int i = 0; i < NV0; i++)
            if (gl == i) t = make_uint2(T.tri[i], T.adj[i]);
        sm.va[gl] = t;
    }
    block_sync();
    SlotRegs<S> R;
#pragma unroll
    for (int s = 0; s < S; s++) {
        R.live[s] = false;
        R.px[s] = R.py[s] = R.pz[s] = 0.0;
        R.d2[s] = R.qw[s] = R.ew[s] = R.iw[s] = 0.f;
    }
    // vertex of slot i from its planes (of a resumed cell: with the same
    // arithmetic and operand order as when it was made)
    auto slot_from_planes = [&](int i, uint32_t t) __attribute__((always_inline)) {
        const int ia = tri_p(t, 0), ib = tri_p(t, 1), ic = D == 3 ? tri_p(t, 2) : tri_p(t, 1);
        float qw, ew, iw;
        make_vertex<D, S>(R, i, sm.plane[ia], sm.plane[ib], sm.plane[ic], sm.pn1[ia], sm.pn1[ib], sm.pn1[ic], sx, sy,
                          sz, qw, ew, iw);
    };
    if (v0) {
#pragma unroll
        for (int i = 0; i < S; i++) {
            const uint32_t t = sm.va[i * G + gl].x;
            if (t != 0xffffffffu) slot_from_planes(i, t);
        }
    } else if (gl < NV0) {
        slot_from_planes(0, sm.va[gl].x);  // NV0 <= G: vertex j lives in slot 0 of lane j
    }

    int nb_v = nb_v0;
    int nlive = nlive0;
    int status = SUCCESS;
    int kc = 0;
    bool done = !valid;
    // Largest squared seed-vertex distance of the cell: r2 in float for the
    // certificate's clear decisions (a float compare against 4 r2 with a
    // relative margin of 4e-7, several roundings), exact_R2 for the others.
    auto exact_R2 = [&]() __attribute__((always_inline)) {
        double m = 0.0;
#pragma unroll
        for (int s = 0; s < S; s++)
            if (R.live[s]) m = smax(vertex_d2(R.px[s], R.py[s], R.pz[s], sx, sy, sz), m);
        return group_butterfly_d<G>(m, [](double a, double b) { return smax(a, b); });
    };
    auto group_r2 = [&]() __attribute__((always_inline)) {
        float m = 0.f;
#pragma unroll
        for (int s = 0; s < S; s++) m = fmaxf(m, R.live[s] ? R.d2[s] : 0.f);
        return group_max_f<G>(m);
    };
    float r2 = group_r2();

    // Row entries may be passed over without the conflict test only while
    // every live vertex is good (vertex_good): nb_skip, per group.
    SkipBounds win = {0.f, 0.f, 0.f};
    bool nb_skip = true;
    const int cap_v = max_p < MAXP ? max_p : MAXP;  // planes the cell may have

    // One clip of the cell by the bisector of neighbour z at (bx, by, bz)
    // (act: this group clips in this step; every lane of the wave calls it):
    // new plane, conflict test of every live vertex, cavity, consistency and
    // new vertices.  Returns whether any seed of the wave clipped.
    auto clip_step = [&](bool act, uint32_t z, double bx, double by, double bz) __attribute__((always_inline)) -> bool {
            // -- new half plane (cell.cpp:158-172)
            if (wave_ballot(act && nb_v >= cap_v) != 0ull) {
                // SLOT_OVERFLOW: more planes than this kernel holds
                if (act && nb_v >= cap_v) status = nb_v >= max_p ? VERTEX_OVERFLOW : SLOT_OVERFLOW;
            }
            const bool go = act && nb_v < cap_v;
            const int cur = nb_v;
            const double ax = sx + bx, ay = sy + by, az = sz + bz;
            Plane e = {sx - bx, sy - by, sz - bz, 0.0};
            const double dot = ax * e.x + ay * e.y + az * e.z;
            e.w = -dot / 2.0;
            double ewm = fabs(e.w);
            if (xmode) ewm = 0.5 * (fabs(ax * e.x) + fabs(ay * e.y) + fabs(az * e.z));
            // 1-norm of e for the bounds (see plane_n1)
            const double en1 = fabs(e.x) + fabs(e.y) + fabs(e.z) + ewm;
            const float cn1 = f2f_up(en1);
            if (go && gl == 0) {
                sm.plane[cur] = e;
                sm.pn1[cur] = cn1;
                sm.pvid[cur] = (int32_t)z;
            }
            nb_v += go ? 1 : 0;
            // -- conflict test of every live vertex.  The reference's
            //    determinant is W f up to rounding, f = e . p + e.w >= 0 on the
            //    seed's side and W < 0: the vertex goes when f < 0.  |W f|
            //    above 5.4e-15 n1(e) q plus the eps bound of the four planes
            //    decides as the reference does (48 u n1 q bounds the rounding of
            //    both; exact mode: XTOL n1 q, below which the rounding of the
            //    planes themselves may flip the sign, which the reference's eps
            //    does not bound); here divided by |W| and compared in float
            //    (1.00001: f's and the bound's float roundings).
            const float c1 = (5.4e-15f + (xmode ? (float)XTOL : 0.f)) * 1.00001f * cn1;
            const float e_eps = 1.00001f * eps_bound<D>(cn1);
            bool rem[S];
            uint32_t doubt = 0;  // slots to decide exactly
    #pragma unroll
            for (int s = 0; s < S; s++) {
                rem[s] = false;
                const bool lv = go && R.live[s];
                if (s > 0 && wave_ballot(lv) == 0ull) continue;  // levels no lane uses cost a branch
                const double f = D == 3 ? fma(e.x, R.px[s], fma(e.y, R.py[s], fma(e.z, R.pz[s], e.w)))
                                        : fma(e.x, R.px[s], fma(e.y, R.py[s], e.w));
                const float ff = (float)f;
                const float bnd = fmaf(c1, R.qw[s], fmaxf(R.ew[s], e_eps * R.iw[s]));
                rem[s] = lv && ff < -bnd;
                doubt |= lv && !(fabsf(ff) > bnd) ? 1u << s : 0u;
            }
            bool gflag = false;
            if (wave_ballot(doubt != 0u) != 0ull) {
                bool flag = false;
                while (doubt) {
                    const int s = __builtin_ctz(doubt);
                    doubt &= doubt - 1u;
                    const uint32_t tt = sm.va[s * G + gl].x;
                    const int i1 = tri_p(tt, 0), i2 = tri_p(tt, 1), i3 = D == 3 ? tri_p(tt, 2) : i2;
                    double xb = 0.0;
                    if (xmode) {
                        const float q = D == 3 ? sm.pn1[i1] * sm.pn1[i2] * sm.pn1[i3] : sm.pn1[i1] * sm.pn1[i2];
                        xb = XTOL * (en1 * (1.0 + 1e-15)) * (double)(q * 1.000001f);
                    }
                    bool c;
                    if (EXACT) {
                        bool fl = false;
                        c = conflict_exact<D>(sm.plane[i1], sm.plane[i2], sm.plane[i3], e, fl, xb);
                        if (fl) {
                            const double sp[3] = {sx, sy, sz}, bp[3] = {bx, by, bz};
                            const int r = exact_conflict<D>(tt, sm, pts, sid, sp, z, bp, key);
                            if (r == 0) flag = true;  // outside the exact predicate's range
                            else c = r > 0;
                        }
                    } else {
                        c = conflict_exact<D>(sm.plane[i1], sm.plane[i2], sm.plane[i3], e, flag, xb);
                    }
    #pragma unroll
                    for (int i = 0; i < S; i++)
                        if (i == s) rem[i] = c;
                }
                gflag = ((wave_ballot(flag) >> shift) & gmask) != 0ull;
            }
            // -- the group's removed slots
            uint64_t Rm[NW];
            int nb_r = 0;
    #pragma unroll
            for (int w = 0; w < NW; w++) Rm[w] = 0ull;
    #pragma unroll
            for (int s = 0; s < S; s++) {
                Rm[(s * G) >> 6] |= ((wave_ballot(rem[s]) >> shift) & gmask) << ((s * G) & 63);
                R.live[s] = R.live[s] && !rem[s];  // removed vertices leave the cell (also on failure)
            }
    #pragma unroll
            for (int w = 0; w < NW; w++) nb_r += popc64(Rm[w]);
            const bool doclip = go && !gflag && nb_r > 0;
            if (go && !doclip) {
                if (gflag) status = NEEDS_EXACT_PREDICATES;
                else nb_v--;  // the plane clipped nothing (cell.cpp:132-136)
            }
            // The cavity, consistency and new-vertex machinery runs only when a
            // seed of the wave clips (a wave-uniform branch; a block is one wave).
            const bool anyclip = wave_ballot(doclip) != 0ull;
            if (anyclip) {
                // -- cavity boundary: edges of removed vertices whose neighbour
                //    is kept
                bool be[S][D];
                uint2 va[S];
                int mycnt = 0;
    #pragma unroll
                for (int s = 0; s < S; s++) {
    #pragma unroll
                    for (int ee = 0; ee < D; ee++) be[s][ee] = false;
                    va[s] = make_uint2(0u, 0u);
                    const bool rm = doclip && rem[s];
                    if (wave_ballot(rm) == 0ull) continue;
                    if (rm) va[s] = sm.va[s * G + gl];
    #pragma unroll
                    for (int ee = 0; ee < D; ee++) {
                        be[s][ee] = rm && !mask_has<NW>(Rm, tri_p(va[s].y, ee));
                        mycnt += be[s][ee] ? 1 : 0;
                    }
                }
                // -- slots for the new vertices: each lane with a free slot
                //    offers its lowest one, and the boundary edges take the
                //    offers lowest level first, so one new vertex per lane
                //    unless lanes are full.  One prefix sum over the lanes for
                //    both: the boundary edges in the high bits, one count of
                //    offers per level (at most G = 16) in 5 bits each below
                constexpr int FB = 5, EB = S <= 4 ? FB * S : 0;
                int fl = S;
    #pragma unroll
                for (int s = S - 1; s >= 0; s--) fl = R.live[s] ? fl : s;
                uint32_t in = (uint32_t)mycnt << EB;
                if (S <= 4) in += fl < S ? 1u << (FB * fl) : 0u;
                in = (uint32_t)group_incl_sum<G>((int)in, gl);
                const uint32_t all = (uint32_t)group_last<G>((int)in);
                const int Bt = (int)(all >> EB);
                int j = (int)(in >> EB) - mycnt;
                int offers = 0, rank = 0;  // of the group; of my offer
                if (S <= 4) {
    #pragma unroll
                    for (int s = 0; s < S; s++) {
                        const int c = (int)((all >> (FB * s)) & 31u);
                        offers += c;
                        rank += s < fl ? c : 0;
                    }
                    rank += (int)((in >> (FB * (fl & 3))) & 31u) - 1;
                } else {
    #pragma unroll
                    for (int s = 0; s < S; s++) {
                        const uint64_t b = (wave_ballot(fl == s) >> shift) & gmask;
                        const int c = popc64(b);
                        offers += c;
                        rank += s < fl ? c : (s == fl ? popc64(b & ((1ull << gl) - 1ull)) : 0);
                    }
                }
                // boundary edges in (slot, edge) order, as counted: plane a |
                // plane b << 8 | kept neighbour << 16 (3D edge e joins planes e
                // and e + 1 of the vertex; 2D: the line, 0, the neighbour)
    #pragma unroll
                for (int s = 0; s < S; s++) {
                    if (s > 0 && wave_ballot(be[s][0] || be[s][1] || be[s][D - 1]) == 0ull) continue;
    #pragma unroll
                    for (int ee = 0; ee < D; ee++) {
                        if (be[s][ee]) {
                            const uint32_t sel = D == 3 ? (uint32_t)(ee | (ee + 1) % 3 << 8 | (4 + ee) << 16 | 0x0c << 24)
                                                        : (uint32_t)(ee | 0x0c << 8 | (4 + ee) << 16 | 0x0c << 24);
                            const uint32_t ed = __builtin_amdgcn_perm(va[s].y, va[s].x, sel);
                            if (S > 3 || j < NS) {  // more boundary edges than slots: overflow below
                                sm.edge[j < NS ? j : NS - 1] = ed;
                                if (D == 3) {
                                    sm.by_start[ed & 0xffu] = (uint8_t)j;
                                    sm.by_end[(ed >> 8) & 0xffu] = (uint8_t)j;
                                }
                            }
                            j++;
                        }
                    }
                }
                block_sync();
                // -- consistency and capacity.  3D: the boundary edges form one
                //    cycle, each edge starting at the plane the one before it
                //    ends at.  Around every plane the boundary edges that
                //    start and end at it alternate, so when no two edges
                //    start at one plane the successor map is a permutation.
                bool ok = doclip;
                bool bad = false;
                if (D == 3) {
                    const int base = shift + gl;  // lane of the wave
                    int nxt = base * 4, lab = gl;  // successor's lane (as a byte address), smallest edge seen
                    if (doclip) {
                        for (int jj = gl; jj < Bt && jj < NS; jj += G)
                            if (sm.by_start[sm.edge[jj] & 0xffu] != jj) bad = true;
                        if (Bt <= G && gl < Bt && !bad) {
                            const int nx = sm.by_start[(sm.edge[gl] >> 8) & 0xffu];
                            if (nx < Bt) nxt = (shift + nx) * 4;
                            else bad = true;
                        }
                        if (gl >= Bt) lab = 0;
                    }
                    // the smallest edge index on each orbit, by pointer jumping
                    // over the group's lanes (all groups of the wave take part;
                    // lanes without an edge point to themselves), must be 0
                    const int jmax = doclip && Bt <= G ? Bt : 0;
    #pragma unroll
                    for (int r = 1; r < 16 && r < G; r <<= 1) {
                        if (wave_ballot(jmax > r) == 0ull) break;
                        lab = min(lab, __builtin_amdgcn_ds_bpermute(nxt, lab));
                        nxt = __builtin_amdgcn_ds_bpermute(nxt, nxt);
                    }
                    if (doclip) {
                        if (Bt <= G) {
                            if (lab != 0) bad = true;
                        } else if (gl == 0 && !bad && Bt <= NS) {
                            int jj = 0, steps = 0;
                            do {
                                jj = sm.by_start[(sm.edge[jj] >> 8) & 0xffu];
                                steps++;
                            } while (jj != 0 && jj < Bt && steps <= Bt);
                            if (steps != Bt || jj != 0) bad = true;
                        }
                    }
                } else {
                    bad = doclip && Bt != 2;
                }
                const bool gbad = ((wave_ballot(bad) >> shift) & gmask) != 0ull;
                bad = false;  // from here: a new vertex no skip can pass (see vertex_good)
                if (doclip) {
                    const int nl_after = nlive - nb_r + Bt;
                    if (gbad) {
                        status = INCONSISTENT_BOUNDARY;
                        ok = false;
                    } else if (nl_after >= max_t) {
                        status = TRIANGLE_OVERFLOW;  // cell.cpp:347-350
                        ok = false;
                    } else if (nl_after > NS) {
                        status = SLOT_OVERFLOW;
                        ok = false;
                    }
                    nlive -= nb_r;
                }
                // the offers' slots, then, where lanes hold several new
                // vertices, more rounds of offers (an edge past the first
                // round waits in its slot's va entry)
                uint32_t more = 0;
                const bool mine = ok && fl < S && rank < Bt;
                if (mine) sm.newslot[rank] = (uint8_t)(fl * G + gl);
                if (wave_ballot(ok && offers < Bt) != 0ull) {
                    uint32_t fr = 0;
    #pragma unroll
                    for (int s = 0; s < S; s++) fr |= ok && !R.live[s] && s != fl ? 1u << s : 0u;
                    int base = offers;
                    while (wave_ballot(ok && base < Bt) != 0ull) {
                        const uint64_t b = (wave_ballot(fr != 0u) >> shift) & gmask;
                        const int r = base + popc64(b & ((1ull << gl) - 1ull));
                        if (fr && r < Bt) {
                            const int s = __builtin_ctz(fr);
                            sm.newslot[r] = (uint8_t)(s * G + gl);
                            sm.va[s * G + gl].x = (uint32_t)r;
                            more |= 1u << s;
                        }
                        fr &= fr - 1u;
                        base += popc64(b);
                    }
                }
                block_sync();
                // -- new vertices (cell.cpp:346-364 orientation, :388-411 position)
                auto new_vertex = [&](int s, int r) __attribute__((always_inline)) {
                    const int gs = s * G + gl;
                    const uint32_t ed = sm.edge[r];
                    const int K = (int)(ed >> 16);
                    float qw, ew, iw;
                    if (D == 3) {
                        const int a = ed & 0xff, b = (ed >> 8) & 0xff;
                        const uint32_t prev = sm.newslot[sm.by_end[a]], next = sm.newslot[sm.by_start[b]];
                        const uint32_t tk = sm.va[K].x;
                        make_vertex<D, S>(R, s, e, sm.plane[a], sm.plane[b], cn1, sm.pn1[a], sm.pn1[b], sx, sy, sz, qw, ew,
                                          iw);
                        sm.va[gs] = make_uint2((uint32_t)cur | (ed & 0xffffu) << 8, prev | (uint32_t)K << 8 | next << 16);
                        // the kept neighbour's edge (b, a) now leads here
                        const uint32_t rk = tk | tk << 24, ba = (uint32_t)(b | a << 8);
                        const int f = (rk & 0xffffu) == ba ? 0 : (((rk >> 8) & 0xffffu) == ba ? 1 : 2);
                        if (f < 2 || (rk >> 16) == ba) set_adj(sm.va[K], f, gs);
                    } else {
                        const int L = ed & 0xff;
                        const Plane pa = sm.plane[L];
                        const float nL = sm.pn1[L];
                        const uint32_t other = sm.newslot[1 - r], tk = sm.va[K].x;
                        const bool swap = det2(e.x, e.y, pa.x, pa.y) > 0;
                        const Plane& p1 = swap ? pa : e;
                        const Plane& p2 = swap ? e : pa;
                        make_vertex<D, S>(R, s, p1, p2, p2, swap ? nL : cn1, swap ? cn1 : nL, swap ? cn1 : nL, sx, sy, sz,
                                          qw, ew, iw);
                        sm.va[gs] = swap ? make_uint2((uint32_t)L | (uint32_t)cur << 8, (uint32_t)K | other << 8)
                                         : make_uint2((uint32_t)cur | (uint32_t)L << 8, other | (uint32_t)K << 8);
                        set_adj(sm.va[K], tri_p(tk, 0) == L ? 0 : 1, gs);
                    }
                    bad = bad || !vertex_good(win, qw, ew, iw);
                };
                if (mine) new_vertex(fl, rank);
                if (wave_ballot(more != 0u) != 0ull) {
                    while (more) {
                        const int s = __builtin_ctz(more);
                        more &= more - 1u;
                        new_vertex(s, (int)sm.va[s * G + gl].x);
                    }
                }
                if (ok) nlive += Bt;
                if (((wave_ballot(bad) >> shift) & gmask) != 0ull) nb_skip = false;
                block_sync();
            }
        return anyclip;
    };

    // --------------------------------------------------------- clip loop
    // The group walks its row in windows of G entries, one per lane.
    // Every window entry that may cut the cell is clipped in row order; the
    // others are passed over (window_filter).  Passing over an entry leaves
    // the cell as it is, so the certificate of a passed entry is judged with
    // the R2 of the last clip, all entries of the window at once.  Seeds of a
    // wave walk their own windows: every step of the wave clips a candidate
    // of each of its seeds.
    int wb = v0;                 // row entry of the window's lane 0
    uint32_t pend = 0, cand = 0; // window entries ahead; of those, the ones to clip
    float wf = 0.f, wx = 0.f, wy = 0.f, wz = 0.f;  // this lane's entry: squared distance and offset
    bool first = true;
    int since = 0;
    // entries of the window ahead whose bisector may cut the cell: the
    // others keep every live vertex on the seed's side by a margin
    auto window_filter = [&]() __attribute__((always_inline)) {
        float mx = 0.f;  // largest offset . vertex of this lane's entry (the seed as origin)
        bool vbad = false;
        if constexpr (SKIP) {
            // offsets (columns) times vertices (rows) of the wave's four
            // seeds, one 16 x 16 block per seed and slot level, on the
            // matrix cores: entry (i, j) of block b sits in register 4 b +
            // i % 4 of lane 16 (i / 4) + j
            // (maxima of at least 0 as signed integers: no NaN handling)
            int m4[4] = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < S; s++) {
                const bool lv = R.live[s];
                if (wave_ballot(lv) == 0ull) continue;
                vbad = vbad || (lv && !vertex_good(win, R.qw[s], R.ew[s], R.iw[s]));
                f32x16 c = {0.f};
                c = __builtin_amdgcn_mfma_f32_16x16x1f32(lv ? (float)(R.px[s] - sx) : 0.f, wx, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x1f32(lv ? (float)(R.py[s] - sy) : 0.f, wy, c, 0, 0, 0);
                if (D == 3) c = __builtin_amdgcn_mfma_f32_16x16x1f32(lv ? (float)(R.pz[s] - sz) : 0.f, wz, c, 0, 0, 0);
#pragma unroll
                for (int b = 0; b < 4; b++)
                    m4[b] = max(max(max(m4[b], __float_as_int(c[4 * b])), max(__float_as_int(c[4 * b + 1]), __float_as_int(c[4 * b + 2]))),
                                __float_as_int(c[4 * b + 3]));
            }
            if (G == 8 && ((tid >> 5) & 1) != ((tid >> 3) & 1)) m4[0] = m4[1] = m4[2] = m4[3] = 0;
            mx = __int_as_float(rows_max_scatter(m4[0], m4[1], m4[2], m4[3]));
        }
        const float h = wx * wx + wy * wy + wz * wz;
        const float slack = 2e-6f * (fabsf(wx) + fabsf(wy) + fabsf(wz)) * __builtin_amdgcn_sqrtf(r2 * 1.001f);
        const bool cut = !(mx < h * (0.5f - SKIP_MARGIN) - slack);
        const uint32_t cm = (uint32_t)((wave_ballot(cut) >> shift) & gmask);
        const bool gb = ((wave_ballot(vbad) >> shift) & gmask) != 0ull;
        nb_skip = !gb;
        cand = gb || nb_v >= cap_v ? pend : pend & cm;
        since = 0;
    };
    for (;;) {
        if (!BALL) {
            // passed entries the certificate holds at (a group's lanes act
            // on their own entries; entries ascend, so a doubtful one can
            // only precede the clear ones)
            bool cert = wf > r2 * CERT_HI;
            const bool ahead = !done && ((pend >> gl) & 1u);
            if (wave_ballot(ahead && !cert && !(wf < r2 * CERT_LO)) != 0ull) {
                const double R2 = exact_R2();
                if (ahead) {
                    const double dx = sm.nbp[gl][0] - sx, dy = sm.nbp[gl][1] - sy;
                    const double dz = D == 3 ? sm.nbp[gl][D - 1] - sz : 0.0;
                    cert = dx * dx + dy * dy + dz * dz > 4 * R2;
                }
            }
            const uint32_t cm = (uint32_t)((wave_ballot(cert) >> shift) & gmask) & pend;
            if (!done && cm != 0u && (cand == 0u || __builtin_ctz(cm) < __builtin_ctz(cand))) {
                kc = wb + __builtin_ctz(cm) + 1;
                done = true;
            }
        }
        const bool refill = wave_ballot(!done && cand == 0u) != 0ull;
        bool filter = since >= REFILTER;
        if (refill) {
            // a seed has passed its window: every seed's next one
            if (!done) {
                if (!first) wb += cand != 0u ? __builtin_ctz(cand) : G;
                if (wb >= k) done = true;
            }
            pend = done ? 0u : (uint32_t)((1ull << min(G, k - wb)) - 1ull);
            cand = pend;
            wf = wx = wy = wz = 0.f;
            if ((pend >> gl) & 1u) {
                const uint32_t zz = row[wb + gl];
                double bp[3] = {0, 0, 0};
                sm.nbi[gl] = zz;
#pragma unroll
                for (int d = 0; d < D; d++) sm.nbp[gl][d] = bp[d] = pts[(size_t)D * zz + d];
                const double dx = bp[0] - sx, dy = bp[1] - sy, dz = D == 3 ? bp[2] - sz : 0.0;
                wf = (float)(dx * dx + dy * dy + dz * dz);
                wx = (float)dx;
                wy = (float)dy;
                wz = (float)dz;
            }
            win = window_bounds<D, G>(wf, pend, sx, sy, sz);
            block_sync();
            filter = !first;
            first = false;
        }
        if (wave_ballot(!done) == 0ull) break;
        filter = filter && SKIP && !xmode;
        if (filter) window_filter();
        if (refill || filter) continue;
        const bool act = !done;
        // the step's neighbour
        uint32_t z = 0;
        double bx = 0, by = 0, bz = 0;
        int j = 0;
        if (act) {
            j = __builtin_ctz(cand);
            pend &= ~((2u << j) - 1u);
            cand &= pend;
            z = sm.nbi[j];
            bx = sm.nbp[j][0];
            by = sm.nbp[j][1];
            bz = D == 3 ? sm.nbp[j][D - 1] : 0.0;
        }
        const bool anyclip = clip_step(act, z, bx, by, bz);
        since++;
        // -- certificate (cell.cpp:369-384) with the just-clipped neighbour;
        //    the largest seed-vertex distance only changes with a clip
        if (anyclip) r2 = group_r2();
        const double dx = bx - sx, dy = by - sy, dz = bz - sz;
        const double dz2 = dx * dx + dy * dy + dz * dz;
        bool cert = !BALL && (float)dz2 > r2 * CERT_HI;
        if (!BALL && wave_ballot(act && (xmode || (!cert && !((float)dz2 < r2 * CERT_LO)))) != 0ull) {
            const double R2 = exact_R2();
            cert = dz2 > 4 * R2 * (EXACT ? CERT_TIE : 1.0);
            if (!EXACT && xmode && act && cert && status == SUCCESS && !(dz2 > 4 * R2 * CERT_TIE)) {
                status = NEEDS_EXACT_PREDICATES;  // a near tie: the exact kernel decides
                cert = false;
            }
        }
        if (act) {
            if (cert) {
                kc = wb + j + 1;
                done = true;
            }
            if (status != SUCCESS) done = true;
            if (!nb_skip || nb_v >= cap_v) cand = pend;
        }
    }

    // -- vertex-ball completion
    const int first_ball = nb_v;
    if (BALL) {
        bool bdone = !valid || status != SUCCESS;
        int32_t cand[S];
        uint32_t ctri[S];
        uint32_t known = 0;  // bit s: cand[s] belongs to the vertex now in slot s
#pragma unroll
        for (int s = 0; s < S; s++) {
            cand[s] = -1;
            ctri[s] = 0xffffffffu;
        }
        for (int iter = 0;; iter++) {
            if (wave_ballot(!bdone) == 0ull) break;
            // candidates of the live vertices not searched yet
            double bd = 0.0;
            int32_t bq = -1;
            bool far = false;
            // the group searches its vertices one at a time, slot by slot
            // (the wave walks until every group has searched its own)
            int32_t* const cst = bg.scr + grp * (2 * G + 1);
            int32_t* const cpf = cst + G;
#pragma unroll
            for (int s = 0; s < S; s++) {
                const uint32_t t = sm.va[s * G + gl].x;
                const bool need = !bdone && R.live[s] && (!((known >> s) & 1u) || ctri[s] != t);
                uint64_t m = (wave_ballot(need) >> shift) & gmask;
                while (wave_ballot(m != 0ull) != 0ull) {
                    if (m == 0ull) continue;
                    const int src = ffs64(m);
                    m &= m - 1ull;
                    const double vv[3] = {shfl(R.px[s], src, G), shfl(R.py[s], src, G), shfl(R.pz[s], src, G)};
                    const double r2v = vertex_d2(vv[0], vv[1], vv[2], sx, sy, sz);
                    const int32_t cq =
                        ball_search_group<D, G>(bg, pts, vv, r2v, sid, sm.pvid, nb_v, gl, shift, gmask, cst, cpf);
                    if (gl == src) cand[s] = cq;
                }
                if (need) {
                    ctri[s] = t;
                    known |= 1u << s;
                }
            }
            if (!bdone) {
#pragma unroll
                for (int s = 0; s < S; s++) {
                    if (!R.live[s]) continue;
                    if (cand[s] == -2) far = true;
                    if (cand[s] < 0) continue;
                    const int32_t q = cand[s];
                    const double dx = pts[(size_t)D * q] - sx, dy = pts[(size_t)D * q + 1] - sy;
                    const double dz = D == 3 ? pts[(size_t)D * q + 2] - sz : 0.0;
                    const double d2 = dx * dx + dy * dy + dz * dz;
                    if (bq < 0 || d2 < bd || (d2 == bd && bg.perm[q] < bg.perm[bq])) {
                        bd = d2;
                        bq = q;
                    }
                }
            }
            // the group's candidate nearest the seed
#pragma unroll
            for (int d = 1; d < G; d <<= 1) {
                const double od = shfl_xor(bd, d, G);
                const int32_t oq = shfl_xor(bq, d, G);
                if (oq >= 0 && (bq < 0 || od < bd || (od == bd && bg.perm[oq] < bg.perm[bq]))) {
                    bd = od;
                    bq = oq;
                }
            }
            far = ((wave_ballot(far) >> shift) & gmask) != 0ull;
            bool act = false;
            if (!bdone) {
                if (far) {
                    status = SECURITY_RADIUS_NOT_REACHED;  // a ball beyond BALL_RINGS: gives up
                    bdone = true;
                } else if (bq < 0) {
                    kc = bg.kmark;  // every vertex ball is empty
                    bdone = true;
                } else if (iter >= 4 * max_p) {
                    status = SECURITY_RADIUS_NOT_REACHED;
                    bdone = true;
                } else {
                    act = true;
                }
            }
            const uint32_t zb = act ? (uint32_t)bq : 0u;
            const double bx = act ? pts[(size_t)D * zb] : 0.0, by = act ? pts[(size_t)D * zb + 1] : 0.0;
            const double bz = (act && D == 3) ? pts[(size_t)D * zb + 2] : 0.0;
            clip_step(act, zb, bx, by, bz);
            if (act && status != SUCCESS) bdone = true;
        }
        if (valid && status != SUCCESS) kc = 0;
    }

    // final certificate with the k-th neighbour (voronoi.cpp:145-147); a row
    // holding every other seed certifies the cell by exhaustion
    // (a slot overflow keeps its code: the 128-slot kernel redoes the seed
    // at the same row length and applies this test itself)
    const int loop_status = status;
    const uint32_t zl = valid ? row[k - 1] : 0u;
    const double R2 = BALL ? 0.0 : exact_R2();
    if (valid && !BALL) {
        const double dx = pts[(size_t)D * zl] - sx, dy = pts[(size_t)D * zl + 1] - sy;
        const double dz = D == 3 ? pts[(size_t)D * zl + 2] - sz : 0.0;
        const double dl2 = dx * dx + dy * dy + dz * dz;
        if (!EXACT && xmode && status == SUCCESS && dl2 > 4 * R2 && !(dl2 > 4 * R2 * CERT_TIE))
            status = NEEDS_EXACT_PREDICATES;
        if (!(dl2 > 4 * R2 * (EXACT ? CERT_TIE : 1.0))) {
            if ((int64_t)k >= n_total - 1 && status == SUCCESS)
                kc = k;
            else if (status != SLOT_OVERFLOW)
                status = SECURITY_RADIUS_NOT_REACHED;
        }
        if (status != SUCCESS) kc = 0;
    }

    const FaceArrays fa = face_arrays_of(fresh_args<ClipArgs>()->fa);
    // save an uncertified cell that ran through its whole row, for a resume
    // at a longer row
    if (fa.resume != nullptr && NS <= 64) {
        const bool save = valid && loop_status == SUCCESS && status == SECURITY_RADIUS_NOT_REACHED;
        if (save) {
            ClipState* out = reinterpret_cast<ClipState*>(fa.cstate + (size_t)sid * CLIP_STATE_BYTES);
            for (int p = gl; p < nb_v; p += G) {
                out->plane[p] = sm.plane[p];
                out->pn1[p] = sm.pn1[p];
                out->pvid[p] = sm.pvid[p];
            }
#pragma unroll
            for (int i = 0; i < S; i++) {
                const int gs = i * G + gl;
                const uint2 v = sm.va[gs];
                out->va[gs] = make_uint2(R.live[i] ? v.x : 0xffffffffu, v.y);
            }
            if (gl == 0) {
                out->nb_v = nb_v;
                out->nlive = nlive;
            }
        }
        if (valid && gl == 0) {
            fa.resume[sid] = save ? (shape_tag | k) : 0;
            if (save) fa.lastnb[sid] = zl;
        }
    }

    // ---------------------------------------------------------- extraction
    const bool ext = valid && status == SUCCESS;
#pragma unroll
    for (int i = 0; i < C::PPL; i++) sm.first[gl + G * i] = 0xffffffffu;
    block_sync();
    // lowest vertex per plane
    if (ext) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            if (!R.live[s]) continue;
            const int gs = s * G + gl;
            const uint32_t t = sm.va[gs].x;
            // a face's cycle starts at its vertex with the smallest sorted
            // plane tuple: the same vertex whatever slot it occupies, so the
            // fan sums round identically for every kernel shape
            const uint32_t key = vertex_key<D>(t);
#pragma unroll
            for (int ee = 0; ee < D; ee++) atomicMin(&sm.first[tri_p(t, ee)], (key << 8) | (uint32_t)gs);
        }
    }
    block_sync();
    // the planes that hold a vertex, listed in plane order: face r is lane r %
    // G's in pass r / G (of 26 planes of a cell some 16 are faces; by plane
    // index the passes would take most lanes through planes without one)
    bool has[C::PPL];
    int nface = 0, fb_rank = 0;
#pragma unroll
    for (int i = 0; i < C::PPL; i++) {
        const int p = gl + G * i;
        has[i] = ext && p < nb_v && sm.first[p] != 0xffffffffu;
        const uint64_t b = (wave_ballot(has[i]) >> shift) & gmask;
        if (has[i]) sm.plist[nface + popc64(b & ((1ull << gl) - 1ull))] = (uint8_t)p;
        nface += popc64(b);
        if (BALL) fb_rank += popc64((wave_ballot(has[i] && p < first_ball) >> shift) & gmask);
    }
    block_sync();
    // normals and neighbour ids of my faces (cell.cpp:575-579, 646-669)
    double nx[C::PPL], ny[C::PPL], nz[C::PPL];
    int fp[C::PPL];  // plane of my face (-1: none)
#pragma unroll
    for (int i = 0; i < C::PPL; i++) {
        const int r = gl + G * i;
        nx[i] = ny[i] = nz[i] = 0.0;
        fp[i] = -1;
        if (r < nface) {
            fp[i] = sm.plist[r];
            const Plane pe = sm.plane[fp[i]];
            const double nl = sqrt(pe.x * pe.x + pe.y * pe.y + pe.z * pe.z);
            nx[i] = pe.x / nl;
            ny[i] = pe.y / nl;
            nz[i] = pe.z / nl;
        }
    }
    block_sync();
    // vertex positions to LDS (over the planes)
    if (ext) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            if (!R.live[s]) continue;
            const int gs = s * G + gl;
            sm.vpos[3 * gs] = R.px[s];
            sm.vpos[3 * gs + 1] = R.py[s];
            sm.vpos[3 * gs + 2] = R.pz[s];
        }
    }
    block_sync();
    // faces: walk each plane's vertex cycle through the adjacency; per plane
    // the volume and centroid moments of its fan
    double pvol[C::PPL], pcx[C::PPL], pcy[C::PPL], pcz[C::PPL];
    bool isface[C::PPL];
    double farea[C::PPL], fcx[C::PPL], fcy[C::PPL], fcz[C::PPL];
    const double* vpos = sm.vpos;
#pragma unroll
    for (int i = 0; i < C::PPL; i++) {
        isface[i] = false;
        farea[i] = fcx[i] = fcy[i] = fcz[i] = 0.0;
        pvol[i] = pcx[i] = pcy[i] = pcz[i] = 0.0;
        double vol = 0.0, cxs = 0.0, cys = 0.0, czs = 0.0;
        if (fp[i] < 0) continue;
        const int p = fp[i];
        const uint32_t v0 = sm.first[p] & 0xffu;
        const double x0 = vpos[3 * v0], y0 = vpos[3 * v0 + 1], z0 = vpos[3 * v0 + 2];
        if (D == 2) {
            const uint2 t0 = sm.va[v0];
            const int v1 = tri_p(t0.y, tri_p(t0.x, 0) == p ? 0 : 1);
            const double x1 = vpos[3 * v1], y1 = vpos[3 * v1 + 1];
            const double dx = x1 - x0, dy = y1 - y0;
            farea[i] = sqrt(dx * dx + dy * dy);
            fcx[i] = 0.5 * (x0 + x1);
            fcy[i] = 0.5 * (y0 + y1);
            const double ta = 0.5 * fabs((x0 - sx) * (y1 - sy) - (x1 - sx) * (y0 - sy));
            vol += ta;
            cxs += ta * (sx + x0 + x1) / 3.0;
            cys += ta * (sy + y0 + y1) / 3.0;
            isface[i] = true;
            pvol[i] = vol;
            pcx[i] = cxs;
            pcy[i] = cys;
        } else {
            int cnt = 0;
            uint32_t cv = v0;
            double ax = 0, ay = 0, az = 0;  // area-weighted centroid sums
            double area = 0.0;
            double px = 0, py = 0, pz = 0;
            bool have_prev = false;
            do {
                const double x = vpos[3 * cv], y = vpos[3 * cv + 1], zz = vpos[3 * cv + 2];
                if (have_prev && cnt >= 2) {
                    const double e1x = px - x0, e1y = py - y0, e1z = pz - z0;
                    const double e2x = x - x0, e2y = y - y0, e2z = zz - z0;
                    const double crx = e1y * e2z - e1z * e2y;
                    const double cry = e1z * e2x - e1x * e2z;
                    const double crz = e1x * e2y - e1y * e2x;
                    const double ta = 0.5 * sqrt(crx * crx + cry * cry + crz * crz);
                    area += ta;
                    ax += ta * (x0 + px + x) / 3.0;
                    ay += ta * (y0 + py + y) / 3.0;
                    az += ta * (z0 + pz + zz) / 3.0;
                    // tetra (seed, v0, prev, cur): seed inside => same sign on a face
                    const double a1 = x0 - sx, a2 = y0 - sy, a3 = z0 - sz;
                    const double b1 = px - sx, b2 = py - sy, b3 = pz - sz;
                    const double c1 = x - sx, c2 = y - sy, c3 = zz - sz;
                    const double tv =
                        fabs(a1 * (b2 * c3 - b3 * c2) + a2 * (b3 * c1 - b1 * c3) + a3 * (b1 * c2 - b2 * c1)) /
                        6.0;
                    vol += tv;
                    cxs += tv * (sx + x0 + px + x) / 4.0;
                    cys += tv * (sy + y0 + py + y) / 4.0;
                    czs += tv * (sz + z0 + pz + zz) / 4.0;
                }
                px = x;
                py = y;
                pz = zz;
                have_prev = true;
                cnt++;
                const uint2 t = sm.va[cv];
                const int ee = tri_p(t.x, 0) == p ? 0 : (tri_p(t.x, 1) == p ? 1 : 2);
                cv = (uint32_t)tri_p(t.y, ee);
            } while (cv != v0 && cnt <= NS);
            pvol[i] = vol;
            pcx[i] = cxs;
            pcy[i] = cys;
            pcz[i] = czs;
            if (cnt >= 3) {
                isface[i] = true;
                farea[i] = area;
                if (area > 0) {
                    fcx[i] = ax / area;
                    fcy[i] = ay / area;
                    fcz[i] = az / area;
                }
            }
        }
    }
    // face order = plane order among planes that form a face
    uint64_t fm = 0;  // by rank in the list
#pragma unroll
    for (int i = 0; i < C::PPL; i++) {
        uint64_t b = (wave_ballot(isface[i]) >> shift) & gmask;
        fm |= b << (G * i);
    }
    // cell volume and centroid moments: a pairwise sum over the plane index,
    // lowest bit first (lanes hold bits below log2 G, the planes of a lane
    // the bits above), i.e. the same tree for every kernel shape; the faces'
    // moments go back to their planes' lanes through LDS (over the positions)
    block_sync();
#pragma unroll
    for (int i = 0; i < C::PPL; i++)
        if (fp[i] >= 0) sm.plane[fp[i]] = Plane{pvol[i], pcx[i], pcz[i], pcy[i]};
    block_sync();
    const auto add = [](double theirs, double mine) { return mine + theirs; };
#pragma unroll
    for (int i = 0; i < C::PPL; i++) {
        Plane m = {0.0, 0.0, 0.0, 0.0};
        if (has[i]) m = sm.plane[gl + G * i];
        pvol[i] = group_butterfly_d<G>(m.x, add);
        pcx[i] = group_butterfly_d<G>(m.y, add);
        pcy[i] = group_butterfly_d<G>(m.w, add);
        pcz[i] = group_butterfly_d<G>(m.z, add);
    }
#pragma unroll
    for (int w = 1; w < C::PPL; w <<= 1)
#pragma unroll
        for (int i = 0; i + w < C::PPL; i += 2 * w) {  // absent planes add nothing
            pvol[i] += pvol[i + w];
            pcx[i] += pcx[i + w];
            pcy[i] += pcy[i + w];
            pcz[i] += pcz[i + w];
        }
    const double vol = pvol[0], cxs = pcx[0], cys = pcy[0], czs = pcz[0];
    if (valid) {
        const int64_t st = fa.stride;
#pragma unroll
        for (int i = 0; i < C::PPL; i++) {
            if (!isface[i]) continue;
            const int r = gl + G * i;
            const int32_t pv = sm.pvid[fp[i]];
            int fi = popc64(fm & ((1ull << r) - 1ull));
            if (BALL && r >= fb_rank) {
                // faces of the completion's planes in (distance, input
                // index) order, after the row's
                const uint32_t zp = (uint32_t)pv;
                const double kp = dist2<D>(pts + (size_t)D * zp, pts + (size_t)D * sid);
                fi = popc64(fb_rank >= 64 ? fm : (fm & ((1ull << fb_rank) - 1ull)));
                for (int q = fb_rank; q < nface; q++) {
                    if (q == r || !((fm >> q) & 1ull)) continue;
                    const uint32_t zq = (uint32_t)sm.pvid[sm.plist[q]];
                    const double kq = dist2<D>(pts + (size_t)D * zq, pts + (size_t)D * sid);
                    if (kq < kp || (kq == kp && bg.perm[zq] < bg.perm[zp])) fi++;
                }
            }
            const int64_t at = (int64_t)fi * st + sid;
            fa.nbr[at] = pv;
            if (fa.nbr_cm) fa.nbr_cm[(int64_t)sid * FACE_SLOTS + fi] = pv;
            fa.area[at] = farea[i];
            const int64_t plane_stride = st * FACE_SLOTS;
            fa.nrm[at] = nx[i];
            fa.nrm[plane_stride + at] = ny[i];
            fa.nrm[2 * plane_stride + at] = nz[i];
            fa.cen[at] = fcx[i];
            fa.cen[plane_stride + at] = fcy[i];
            fa.cen[2 * plane_stride + at] = D == 3 ? fcz[i] : 0.0;
        }
        if (gl == 0) {
            fa.count[sid] = ext ? (uint8_t)popc64(fm) : (uint8_t)0;
            fa.vol[sid] = ext ? vol : 0.0;
            const double iv = vol != 0.0 ? 1.0 / vol : 0.0;
            fa.ccen[sid] = ext ? cxs * iv : 0.0;
            fa.ccen[st + sid] = ext ? cys * iv : 0.0;
            fa.ccen[2 * st + sid] = ext ? czs * iv : 0.0;
            fa.status[sid] = status;
            fa.kcert[sid] = kc;
        }
    }
}

}  // namespace pg
