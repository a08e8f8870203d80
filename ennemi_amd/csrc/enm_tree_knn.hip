// k-th-neighbour radii on box trees: eps_i is the (k+1)-th smallest distance
// over the scope, the query itself included (+inf with fewer points).
//
// A wave takes the queries of one leaf one after the other.  The leaf's own 64
// points, held one per lane for all of its queries, are sorted across the
// lanes and give the first k+1 neighbours and radius T; then the leaves of the
// own cell and of the other cells whose boxes come nearer than T are visited,
// the nearest first, so T is close to its final value after a leaf or two.  A
// leaf's few distances below T go into the list one at a time (a shift by one
// lane, a minimum and a maximum for up to 64 neighbours); where there are
// many, as with long lists, they are sorted and merged.  Lists longer than
// 64 * ENM_TREE_LISTS are taken in passes: each finds the next ranks above the
// last pass's highest distance B, after counting the points within B.  4 x
// 50,000 points in two columns: k = 126 in 0.59 ms, 200 in 1.13, 600 in 8.5,
// where walks with a heap per lane took 3.1, 6.4 and 28; in four columns 1.6,
// 3.3 and 23 ms, where sweeps shared by 64 queries took 49, 77 and 267.
#include "enm_tree.h"

namespace {

// Distances below T at which sorting and merging all 64 beats inserting one by
// one: about 140, 210, 350 or 630 instructions (1, 2, 4 or 8 registers of
// ranks) against 11, 15, 23 or 39 each.
constexpr int MERGE_FROM = 14;

template <int D, int NR>
struct TreeQuery {
    const TreeDev& T;
    const double* col64;
    int ncol;
    double q[D];
    LaneList<NR> list;
    int K1;
    double t;            // the current radius
    double above;        // only distances above this are ranked (last registers only)
    unsigned visited;    // leaves

    static constexpr bool PASSES = NR == ENM_TREE_LISTS;

    __device__ __forceinline__ void visit_leaf(const double* leaf) {
        double a[D];
        load_leaf<D>(a, leaf, ncol);
        double e = point_dist<D>(a, q);
        if (PASSES) e = e > above ? e : INFINITY;
        unsigned long long m = __builtin_amdgcn_ballot_w64(e < t);
        ++visited;
        if (__popcll(m) >= MERGE_FROM) {
            list.merge(e < t ? e : INFINITY);
            t = list.rank(K1 - 1);
        } else {
            while (m) {
                list.insert(lane_f64(e, __builtin_ctzll(m)));
                t = list.rank(K1 - 1);
                m &= (m - 1) & __builtin_amdgcn_ballot_w64(e < t);
            }
        }
    }

    // The nearest of the lanes in m by their gaps.
    __device__ __forceinline__ int nearest(unsigned long long m, double gap) {
        const int lane = (int)(threadIdx.x & (ENM_WAVE - 1));
        const float g = (m >> lane) & 1 ? (float)gap : INFINITY;
        const unsigned long long s = __builtin_amdgcn_ballot_w64(g == wave_min_f32(g)) & m;
        return __builtin_ctzll(s ? s : m);
    }

    // The leaves of a cell but leaf `own` (-1: all).
    __device__ __forceinline__ void visit_cell(int cell, int own) {
        const int nleaf = (min(T.cell, T.n - cell * T.cell) + ENM_LEAF - 1) / ENM_LEAF;
        const double g = box_gap<D>(col64 + T.box + (int64_t)cell * 2 * ncol * 64, ncol, q);
        unsigned long long open = low_mask(nleaf);
        if (own >= 0) open &= ~(1ull << own);
        const double* leaves = col64 + T.col + (int64_t)cell * T.cell * ncol;
        for (;;) {
            const unsigned long long m = __builtin_amdgcn_ballot_w64(g < t) & open;
            if (!m) break;
            const int l = nearest(m, g);
            open &= ~(1ull << l);
            visit_leaf(leaves + l * ENM_LEAF * ncol);
        }
    }

    __device__ __forceinline__ void visit_others(int own_cell) {
        const int ncell = T.ncell, ngroup = (ncell + 63) / 64;
        for (int gb = 0; gb < ngroup; gb += 64) {
            double gg = 0.0;
            unsigned long long gopen = low_mask(ngroup - gb);
            if (ngroup > 1) gg = box_gap<D>(col64 + T.gbox + (int64_t)(gb / 64) * 2 * ncol * 64, ncol, q);
            for (;;) {
                const unsigned long long gm = ngroup > 1 ? __builtin_amdgcn_ballot_w64(gg < t) & gopen : gopen;
                if (!gm) break;
                const int gl = ngroup > 1 ? nearest(gm, gg) : 0;
                gopen &= ~(1ull << gl);
                const int gr = gb + gl;
                const double g = box_gap<D>(col64 + T.cbox + (int64_t)gr * 2 * ncol * 64, ncol, q);
                unsigned long long open = low_mask(ncell - gr * 64);
                if (own_cell / 64 == gr) open &= ~(1ull << (own_cell % 64));
                for (;;) {
                    const unsigned long long m = __builtin_amdgcn_ballot_w64(g < t) & open;
                    if (!m) break;
                    const int c = nearest(m, g);
                    open &= ~(1ull << c);
                    visit_cell(gr * 64 + c, -1);
                }
            }
        }
    }
};

template <int D, int NR>
__global__ __launch_bounds__(TREE_WG* ENM_WAVE, std::min(tree_waves(D), NR <= 2 ? 8 : NR <= 4 ? 6 : 4))
void tree_knn_kernel(TreeArgs A, const KnnDev* __restrict__ descs, const double* __restrict__ col64,
                     double* __restrict__ res64, unsigned long long* __restrict__ stats) {
    const TreeWork it = tree_work(A);
    if (it.nq <= 0) return;
    const int lane = (int)(threadIdx.x & (ENM_WAVE - 1));
    const KnnDev& kd = descs[it.desc];
    const TreeDev& T = A.trees[it.tile];
    const int t0 = it.t0, nq = it.nq;
    const int ncol = T.ncol;
    // The queries' leaf, one point per lane.
    const int leaf = t0 / ENM_LEAF, j0 = t0 % ENM_LEAF;
    const int cell = leaf * ENM_LEAF / T.cell;
    double own[D];
    load_leaf<D>(own, col64 + T.col + (int64_t)leaf * ncol * ENM_LEAF, ncol);
    constexpr bool PASSES = TreeQuery<D, NR>::PASSES;
    double mine = 0.0;
    unsigned visited = 0;
    for (int j = 0; j < nq; ++j) {
        TreeQuery<D, NR> w{T, col64, ncol};
#pragma unroll
        for (int d = 0; d < D; ++d) w.q[d] = lane_f64(own[d], j0 + j);
        const int k1 = kd.k + 1;
        const double e0 = vmin(point_dist<D>(own, w.q), INFINITY);   // (NaN: +inf)
        w.visited = visited;
        w.above = -INFINITY;
        int found = 0;   // points ranked by the passes before
        for (;;) {
            w.K1 = PASSES ? min(k1 - found, 64 * NR) : k1;
            w.list.seed(PASSES ? (e0 > w.above ? e0 : INFINITY) : e0);
            w.t = w.list.rank(w.K1 - 1);
            ++w.visited;
            if (T.n > ENM_LEAF) w.visit_cell(cell, leaf - cell * (T.cell / ENM_LEAF));
            if (T.ncell > 1) w.visit_others(cell);
            if (!PASSES || found + w.K1 == k1 || !(w.t < INFINITY)) break;
            const double radius[1] = {w.t};
            int within[1];
            count_queries<D, 1>(T, col64, reinterpret_cast<const double(&)[1][D]>(w.q), radius, within, w.visited);
            found = within[0];
            if (found >= k1) break;   // ties at the last rank
            w.above = w.t;
        }
        if (lane == j) mine = w.t;
        visited = w.visited;
    }
    if (lane < nq) res64[kd.eps_orig + A.perm[T.perm + t0 + lane]] = mine;
    if (lane == 0) add_stat(stats, ST_KNN_PAIRS, (unsigned long long)visited * ENM_LEAF);
}

template <int D>
hipError_t launch(const TreeArgs& a, int qmax, int lists, const KnnDev* descs, const double* col64, double* res64,
                  unsigned long long* stats, hipStream_t st) {
    const dim3 grid(tree_grid(qmax, a.share)), block(TREE_WG * ENM_WAVE);
#define ENM_TREE_KNN(NR) \
    case NR: hipLaunchKernelGGL((tree_knn_kernel<D, NR>), grid, block, 0, st, a, descs, col64, res64, stats); break;
    switch (lists) {
        ENM_TREE_KNN(1)
        ENM_TREE_KNN(2)
        ENM_TREE_KNN(4)
        ENM_TREE_KNN(ENM_TREE_LISTS)
        default: return hipErrorInvalidValue;
    }
#undef ENM_TREE_KNN
    return hipGetLastError();
}

}  // namespace

int enm_tree_list_class(int k1) { return k1 <= 64 ? 1 : k1 <= 128 ? 2 : k1 <= 256 ? 4 : ENM_TREE_LISTS; }

hipError_t enm_launch_tree_knn(const Item* items, const int* qoff, int n_items, int qmax, int share,
                               const KnnDev* descs,
                               const TreeDev* trees, const int* perm, const double* col64, double* res64,
                               unsigned long long* stats, int dclass, int lists, hipStream_t st) {
    if (n_items <= 0) return hipSuccess;
    const TreeArgs a{items, qoff, share, trees, perm, nullptr};
    switch (dclass) {
        case 2: return launch<2>(a, qmax, lists, descs, col64, res64, stats, st);
        case 3: return launch<3>(a, qmax, lists, descs, col64, res64, stats, st);
        case 4: return launch<4>(a, qmax, lists, descs, col64, res64, stats, st);
        case 5: return launch<5>(a, qmax, lists, descs, col64, res64, stats, st);
        case 6: return launch<6>(a, qmax, lists, descs, col64, res64, stats, st);
        case 8: return launch<8>(a, qmax, lists, descs, col64, res64, stats, st);
        case 12: return launch<12>(a, qmax, lists, descs, col64, res64, stats, st);
        case 16: return launch<16>(a, qmax, lists, descs, col64, res64, stats, st);
        default: return hipErrorInvalidValue;
    }
}
