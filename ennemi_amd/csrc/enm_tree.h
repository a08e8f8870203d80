// Box trees: k-th-neighbour radii and ball counts of spaces of two or more
// columns, replacing cKDTree.query and cKDTree.query_ball_point of the
// reference (ennemi/_entropy_estimators.py:39,108,142,152-154,194,196,240,
// 243-245) where no strip of two columns fits in LDS.
//
// A wave takes one query at a time, or counts four.  Its 64 lanes test the boxes
// of 64 children of a node at once (groups, then cells, then leaves), and the
// points of a leaf are evaluated one per lane, so each (query, leaf) pair
// whose ball and box meet costs one coalesced load and one difference and
// maximum per column, and nothing is evaluated for the sake of other queries:
// the boxes are tight in every column, where a window shared by 64 queries is
// their union and is cut by two columns only.  Measured against such windows
// (one conditional MI of 2,000,000 points with two conditions, k = 5): kNN in
// four columns 51.6 -> 4.5 ms, the three counts 51.4 -> 8.0 ms; 100,000 points
// with three conditions, kNN in five columns 2.77 -> 0.24 ms, counts 3.97 ->
// 0.45 ms; joint entropy of four columns, 100,000 points, 1.48 -> 0.13 ms; 60
// conditional MIs of 1,800 points, kNN 0.110 -> 0.062 ms, counts 0.305 ->
// 0.05 ms.  The kNN is bound by its instructions (800 vector ones a query in
// four columns).  The counts were bound by their loads from L2, about 85 of 512
// bytes a query; four neighbouring queries at once share them (the 8.0 ms above
// are 15.3 one at a time, 10.5 two, and 9.9 eight, whose coordinates no longer fit
// the scalar registers).
//
// Everything is decided by the reference's own FP64 expressions.  For a box
// side lo <= a <= hi, fl(a - q) >= fl(lo - q) and fl(q - a) >= fl(q - hi)
// (rounding is monotone), so the largest of these over the columns bounds
// every point's distance from below exactly, and the largest of fl(hi - q),
// fl(q - lo) bounds it from above: a leaf is passed over, or counted whole,
// only where every one of its points would be.
#pragma once
#include "enm_device.h"
#include "enm_launch.h"

#include <algorithm>

namespace {

// v of the lane that the DPP control names, `old` where there is none.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double old, double v) {
    const long long o = __double_as_longlong(old), b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)o, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float old, float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// DPP controls: shifts within rows of 16 and broadcasts across them (a
// reduction into lane 63), one lane up across the wave, and the fixed
// exchanges inside a row.
enum { DPP_SHR1 = 0x111, DPP_SHR2 = 0x112, DPP_SHR4 = 0x114, DPP_SHR8 = 0x118, DPP_ROR8 = 0x128, DPP_WSHR1 = 0x138,
       DPP_MIRROR = 0x140, DPP_HALF_MIRROR = 0x141, DPP_BCAST15 = 0x142, DPP_BCAST31 = 0x143,
       DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_XOR3 = 0x1B };

// Smallest and largest value of the wave (never NaN).
__device__ __forceinline__ float wave_min_f32(float v) {
    v = fminf(v, dpp_f32<DPP_SHR1>(INFINITY, v));
    v = fminf(v, dpp_f32<DPP_SHR2>(INFINITY, v));
    v = fminf(v, dpp_f32<DPP_SHR4>(INFINITY, v));
    v = fminf(v, dpp_f32<DPP_SHR8>(INFINITY, v));
    v = fminf(v, dpp_f32<DPP_BCAST15>(INFINITY, v));
    v = fminf(v, dpp_f32<DPP_BCAST31>(INFINITY, v));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ double lane_f64(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <bool MAX>
__device__ __forceinline__ double wave_ext_f64(double v) {
    const double id = MAX ? -INFINITY : INFINITY;
    auto f = [](double a, double b) { return MAX ? vmax(a, b) : vmin(a, b); };
    v = f(v, dpp_f64<DPP_SHR1>(id, v));
    v = f(v, dpp_f64<DPP_SHR2>(id, v));
    v = f(v, dpp_f64<DPP_SHR4>(id, v));
    v = f(v, dpp_f64<DPP_SHR8>(id, v));
    v = f(v, dpp_f64<DPP_BCAST15>(id, v));
    v = f(v, dpp_f64<DPP_BCAST31>(id, v));
    return lane_f64(v, 63);
}

// The value of lane ^ X.
template <int X>
__device__ __forceinline__ double xor_f64(double v) {
    if constexpr (X == 1) return dpp_f64<DPP_XOR1>(v, v);
    else if constexpr (X == 2) return dpp_f64<DPP_XOR2>(v, v);
    else if constexpr (X == 3) return dpp_f64<DPP_XOR3>(v, v);
    else if constexpr (X == 4) return dpp_f64<DPP_XOR3>(v, dpp_f64<DPP_HALF_MIRROR>(v, v));
    else if constexpr (X == 7) return dpp_f64<DPP_HALF_MIRROR>(v, v);
    else if constexpr (X == 8) return dpp_f64<DPP_ROR8>(v, v);
    else if constexpr (X == 15) return dpp_f64<DPP_MIRROR>(v, v);
    else return __shfl_xor(v, X, ENM_WAVE);
}

// One stage of a bitonic network: lanes l and l ^ X, the lower one keeps the
// smaller value.  Lane masks of "keeps the larger": lanes with the highest
// bit of X set.
template <int X>
__device__ __forceinline__ double bitonic_stage(double v) {
    constexpr int TOP = X >= 32 ? 32 : X >= 16 ? 16 : X >= 8 ? 8 : X >= 4 ? 4 : X >= 2 ? 2 : 1;
    const double o = xor_f64<X>(v);
    const bool upper = ((int)(threadIdx.x & (ENM_WAVE - 1)) & TOP) != 0;
    return (o < v) != upper ? o : v;
}

// A bitonic sequence of 64 values (one per lane) into ascending order.
__device__ __forceinline__ double wave_clean64(double v) {
    v = bitonic_stage<32>(v);
    v = bitonic_stage<16>(v);
    v = bitonic_stage<8>(v);
    v = bitonic_stage<4>(v);
    v = bitonic_stage<2>(v);
    return bitonic_stage<1>(v);
}

// 64 values (one per lane, never NaN) into ascending order: Batcher's bitonic
// sort, each merge beginning with a mirrored stage so that every run ascends.
__device__ __forceinline__ double wave_sort64(double v) {
    v = bitonic_stage<1>(v);
    v = bitonic_stage<3>(v); v = bitonic_stage<1>(v);
    v = bitonic_stage<7>(v); v = bitonic_stage<2>(v); v = bitonic_stage<1>(v);
    v = bitonic_stage<15>(v); v = bitonic_stage<4>(v); v = bitonic_stage<2>(v); v = bitonic_stage<1>(v);
    v = bitonic_stage<31>(v); v = bitonic_stage<8>(v); v = bitonic_stage<4>(v); v = bitonic_stage<2>(v);
    v = bitonic_stage<1>(v);
    v = bitonic_stage<63>(v); v = bitonic_stage<16>(v); v = bitonic_stage<8>(v); v = bitonic_stage<4>(v);
    v = bitonic_stage<2>(v);
    return bitonic_stage<1>(v);
}

// The 64 * NR smallest distances seen, ascending across the lanes (rank
// 64 r + lane in L[r]); unset ranks are +inf.
template <int NR>
struct LaneList {
    double L[NR];

    // From the 64 distances of the first leaf.
    __device__ __forceinline__ void seed(double d) {
        L[0] = wave_sort64(d);
#pragma unroll
        for (int r = 1; r < NR; ++r) L[r] = INFINITY;
    }

    __device__ __forceinline__ double rank(int t) const {
        double v = lane_f64(L[0], t & 63);
#pragma unroll
        for (int r = 1; r < NR; ++r)
            if (t >= 64 * r) v = lane_f64(L[r], t & 63);
        return v;
    }

    // One value (the same in every lane): every rank takes
    // min(L[t], max(v, L[t-1])).
    __device__ __forceinline__ void insert(double v) {
        double below = -INFINITY;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double last = NR > 1 && r + 1 < NR ? lane_f64(L[r], 63) : 0.0;
            const double prev = dpp_f64<DPP_WSHR1>(below, L[r]);
            L[r] = vmin(L[r], vmax(prev, v));
            below = last;
        }
    }

    // 64 values, one per lane (+inf: none): sorted, and merged from the
    // highest ranks down (reversed and paired, the smaller of each pair are
    // the lowest 64 of the two runs, the larger ones the rest, both bitonic).
    __device__ __forceinline__ void merge(double d) {
        double s = wave_sort64(d);
#pragma unroll
        for (int r = NR - 1; r >= 0; --r) {
            const double rev = xor_f64<63>(s);
            const double lo = vmin(L[r], rev), hi = vmax(L[r], rev);
            s = wave_clean64(lo);   // the lowest 64 of L[r] and what came from above
            if (r < NR - 1) L[r + 1] = wave_clean64(hi);
            L[r] = s;
        }
    }
};

// Distance of this lane's point a to the query q, max over the columns of
// fl64(|a - q|) (NaN differences are passed over, as fmax does).
template <int D>
__device__ __forceinline__ double point_dist(const double (&a)[D], const double (&q)[D]) {
    double e;
    {
        const double d0 = a[0] - q[0], d1 = a[D > 1 ? 1 : 0] - q[D > 1 ? 1 : 0];
        asm("v_max_f64 %0, |%1|, |%2|" : "=v"(e) : "v"(d0), "v"(d1));
    }
#pragma unroll
    for (int d = 2; d < D; ++d) e = vmax_abs(e, a[d] - q[d]);
    return e;
}

// Offset in a leaf of dimension d's values: classes up to 6 are exact, wider
// ones repeat column 0 beyond the tree's columns (which leaves the max-norm
// unchanged).
template <int D>
__device__ __forceinline__ int col_of(int d, int ncol) {
    return D <= 6 || d < ncol ? d : 0;
}

// This lane's point of a leaf (NaN past the last point).
template <int D>
__device__ __forceinline__ void load_leaf(double (&a)[D], const double* __restrict__ leaf, int ncol) {
    const int lane = (int)(threadIdx.x & (ENM_WAVE - 1));
#pragma unroll
    for (int d = 0; d < D; ++d) a[d] = leaf[col_of<D>(d, ncol) * ENM_LEAF + lane];
}

// The queries' distances to this lane's box, from below (FAR: and from above).
template <int D, int Q, bool FAR>
__device__ __forceinline__ void box_gap(const double* __restrict__ b, int ncol, const double (&q)[Q][D], double (&gap)[Q],
                                        double (&far)[Q]) {
    const int lane = (int)(threadIdx.x & (ENM_WAVE - 1));
    double lo[D], hi[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        const int c = col_of<D>(d, ncol);
        lo[d] = b[(2 * c) * 64 + lane];
        hi[d] = b[(2 * c + 1) * 64 + lane];
    }
    // Equal infinities differ by NaN, which the maxima pass over here as they
    // do in point_dist (all NaN: not inside).
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        double g = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            g = vmax(g, vmax(lo[d] - q[k][d], q[k][d] - hi[d]));
            if (FAR) {
                const double s = vmax(hi[d] - q[k][d], q[k][d] - lo[d]);
                far[k] = d == 0 ? s : vmax(far[k], s);
            }
        }
        gap[k] = g;
    }
}

// One query's distance to this lane's box, from below.
template <int D>
__device__ __forceinline__ double box_gap(const double* __restrict__ b, int ncol, const double (&q)[D]) {
    double gap[1], far[1];
    box_gap<D, 1, false>(b, ncol, reinterpret_cast<const double(&)[1][D]>(q), gap, far);
    return gap[0];
}

__device__ __forceinline__ unsigned long long low_mask(int n) {
    return n >= 64 ? ~0ull : ((1ull << n) - 1ull);
}

// c[k] += points within r[k] of q[k], max_d fl64(|a_d - q_d|) <= r, of Q queries
// at once: a node whose box lies within the radius in every column adds its
// points unopened, one out of reach adds none; the others are opened, leaves by
// their points.  A node is opened for all the queries if one of them needs it:
// neighbours in a leaf mostly need the same ones, and the loads (48 KB a query
// by itself, from L2) are what bounds the counts.
template <int D, int Q>
__device__ __forceinline__ void count_cell(const TreeDev& T, const double* __restrict__ col64, int cell,
                                           const double (&q)[Q][D], const double (&r)[Q], int (&c)[Q], unsigned& opened) {
    const int ncol = T.ncol;
    const int cnt = min(T.cell, T.n - cell * T.cell);
    const int nleaf = (cnt + ENM_LEAF - 1) / ENM_LEAF;
    unsigned long long part = 1;
    if (T.n > ENM_LEAF) {
        double gap[Q], far[Q];
        box_gap<D, Q, true>(col64 + T.box + (int64_t)cell * 2 * ncol * 64, ncol, q, gap, far);
        const unsigned long long valid = low_mask(nleaf);
        unsigned long long inside[Q];
        part = 0;
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            inside[k] = __builtin_amdgcn_ballot_w64(far[k] <= r[k]) & valid;
            part |= __builtin_amdgcn_ballot_w64(gap[k] <= r[k]) & valid & ~inside[k];
        }
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const unsigned long long whole = inside[k] & ~part;
            c[k] += (int)__popcll(whole) * ENM_LEAF;
            if ((whole >> (nleaf - 1)) & 1) c[k] -= nleaf * ENM_LEAF - cnt;
        }
    }
    opened += (unsigned)__popcll(part) * Q;
    const double* leaves = col64 + T.col + (int64_t)cell * T.cell * ncol;
    // Two leaves at a time, so that their loads overlap (an odd last one is
    // loaded twice and counted once).
    while (part) {
        const int l0 = __builtin_ctzll(part);
        part &= part - 1;
        const int l1 = part ? __builtin_ctzll(part) : l0;
        const bool two = part != 0;
        part &= part - 1;
        double a[D], b[D];
        load_leaf<D>(a, leaves + l0 * ENM_LEAF * ncol, ncol);
        load_leaf<D>(b, leaves + l1 * ENM_LEAF * ncol, ncol);
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const int ca = (int)__popcll(__builtin_amdgcn_ballot_w64(point_dist<D>(a, q[k]) <= r[k]));
            const int cb = (int)__popcll(__builtin_amdgcn_ballot_w64(point_dist<D>(b, q[k]) <= r[k]));
            c[k] += ca + (two ? cb : 0);
        }
    }
}

template <int D, int Q>
__device__ __forceinline__ void count_queries(const TreeDev& T, const double* __restrict__ col64, const double (&q)[Q][D],
                                              const double (&r)[Q], int (&c)[Q], unsigned& opened) {
    const int ncell = T.ncell, ncol = T.ncol;
#pragma unroll
    for (int k = 0; k < Q; ++k) c[k] = 0;
    if (ncell == 1) {
        count_cell<D, Q>(T, col64, 0, q, r, c, opened);
        return;
    }
    const int ngroup = (ncell + 63) / 64;
    double gap[Q], far[Q];
    // Groups that the balls meet, 64 at a time; then their cells.
    for (int gb = 0; gb < ngroup; gb += 64) {
        unsigned long long gm = 1;
        if (ngroup > 1) {
            box_gap<D, Q, false>(col64 + T.gbox + (int64_t)(gb / 64) * 2 * ncol * 64, ncol, q, gap, far);
            gm = 0;
#pragma unroll
            for (int k = 0; k < Q; ++k) gm |= __builtin_amdgcn_ballot_w64(gap[k] <= r[k]);
            gm &= low_mask(ngroup - gb);
        }
        while (gm) {
            const int gr = gb + __builtin_ctzll(gm);
            gm &= gm - 1;
            box_gap<D, Q, true>(col64 + T.cbox + (int64_t)gr * 2 * ncol * 64, ncol, q, gap, far);
            const unsigned long long valid = low_mask(ncell - gr * 64);
            unsigned long long inside[Q], part = 0;
#pragma unroll
            for (int k = 0; k < Q; ++k) {
                inside[k] = __builtin_amdgcn_ballot_w64(far[k] <= r[k]) & valid;
                part |= __builtin_amdgcn_ballot_w64(gap[k] <= r[k]) & valid & ~inside[k];
            }
            const int last = ncell - 1 - gr * 64;   // the scope's last cell, if it is here
#pragma unroll
            for (int k = 0; k < Q; ++k) {
                const unsigned long long whole = inside[k] & ~part;
                c[k] += (int)__popcll(whole) * T.cell;
                if (last < 64 && ((whole >> last) & 1)) c[k] -= ncell * T.cell - T.n;
            }
            while (part) {
                const int k = gr * 64 + __builtin_ctzll(part);
                part &= part - 1;
                count_cell<D, Q>(T, col64, k, q, r, c, opened);
            }
        }
    }
}

// Waves per SIMD that the kernels of dimension class D are held to registers
// for, and waves per workgroup (each with an item of its own).
constexpr int tree_waves(int D) { return D <= 4 ? 8 : D <= 6 ? 6 : D <= 8 ? 4 : 2; }
constexpr int TREE_WG = 4;

struct TreeArgs {
    const Item* items;    // leaves
    const int* qoff;
    int share;            // waves of a leaf (a power of two)
    const TreeDev* trees;
    const int* perm;
    const double* psi_tab;
};

// This wave's queries: nq positions of tree `tile` from t0 on, for descriptor
// desc (nq = 0: none).  Every share of a leaf is a wave of the launch: the
// dispatcher balances them, and there are no tickets, whose counters would
// cost as much as the queries (conditional MI of 60 x 1,800 points: kNN 239 us
// with tickets for 8 queries, 62 us so).  Workgroup b serves queue
// b % ENM_NQ, whose leaves share one XCD's L2.
struct TreeWork {
    int desc, tile, t0, nq;
};
__device__ __forceinline__ TreeWork tree_work(const TreeArgs& A) {
    const int q = (int)(blockIdx.x % ENM_NQ);
    const int k = uni((int)(blockIdx.x / ENM_NQ * TREE_WG + threadIdx.x / ENM_WAVE));
    const int i = A.qoff[q] + k / A.share;
    TreeWork w{0, 0, 0, 0};
    if (i < A.qoff[q + 1]) {
        const Item& it = A.items[i];
        const int step = ENM_LEAF / A.share;
        w.desc = it.desc;
        w.tile = it.tile;
        w.t0 = it.t0 + k % A.share * step;
        w.nq = min(step, it.t1 - w.t0);
    }
    return w;
}
inline int tree_grid(int qmax, int share) { return (qmax * share + TREE_WG - 1) / TREE_WG * ENM_NQ; }

}  // namespace
