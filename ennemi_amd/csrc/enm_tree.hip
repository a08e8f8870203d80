// Build of the box trees, the ball counts on them, and the dispatch of both
// tree queries (the kNN kernels are in enm_tree_knn.hip).
#include "enm_sort_lds.h"
#include "enm_tree.h"

namespace {

// ---------------------------------------------------------------------------
// Build.  One workgroup per cell: its points (a run of the slab order, or of
// the point order where the whole scope is one cell) are sorted in LDS by one
// column, the sorted run cut into equal runs, each sorted by the next column,
// and so on down to runs of a leaf.  Every halving goes to the column that is
// widest so far in the cell, by the middle half of 64 of its points (which
// outliers do not move), so that leaves come out about as long in every column
// whatever the columns' scales: radii are in the largest one's.  Then the columns
// are gathered from the arena in tree order and every leaf's box is taken.
// (The first column 10^6 times wider than the others, joint entropies of 500,000
// points in three, four and five columns: 18, 45 and 57 ms with the halvings dealt
// out evenly, 3.3, 4.9 and 6.3 so; equal widths 2.0, 3.4 and 5.4 ms both ways.  To
// measure the widths takes a cell 3 us of 80.)

constexpr int TB_THREADS = 512;

// The width of a column in a cell of cnt points (si: their numbers), by one wave:
// that of the middle half of 64 of them, and of a tiny one at least, so that
// columns without any take turns.
__device__ __forceinline__ double cell_width(const double* __restrict__ src, const int* si, int cnt) {
    const int lane = (int)threadIdx.x & (ENM_WAVE - 1);
    const double v = wave_sort64(vmin(src[si[lp(lane * cnt / ENM_WAVE)]], INFINITY));   // (NaN: +inf)
    const double w = lane_f64(v, 48) - lane_f64(v, 16);
    return w < 1e300 ? vmax(w, 1e-250) : w >= 1e300 ? 1e300 : 1e-250;   // (equal infinities: NaN)
}

// The steps of a cell, by one wave.  The column that the slab order has sorted
// comes first, the others in their order.
__device__ void cell_steps(const TreeDev& T, const double* widths, int* dim, int* run, int* nstep) {
    const int lane = (int)threadIdx.x & (ENM_WAVE - 1);
    double width = lane < T.ncol ? widths[lane] : -1.0;
    // A column that is not cut yet costs a sort (one cell of 4,096 points 18 us, which
    // few cells wait for), and is taken up only if it is wider by a factor than the
    // widest that is; the one sorted already costs none.  Build and kNN of 20,000 and
    // of 400,000 points in five columns, us: factor 4, 272 and 1800; 2.5, 272 and
    // 1700; 2, 277 and 1678; 1.5, 293 and 1681.
    const double least = T.ncell <= 64 ? 0.25 : 0.5;
    if (lane != T.sorted) width *= least;
    int bits = 0;
    for (int h = 0; h < T.halvings; ++h) {
        const unsigned long long widest = __builtin_amdgcn_ballot_w64(width == wave_ext_f64<true>(width));
        if (lane == __builtin_ctzll(widest)) {
            width *= bits == 0 && lane != T.sorted ? 0.5 / least : 0.5;
            ++bits;
        }
    }
    unsigned long long cut = __builtin_amdgcn_ballot_w64(bits > 0);
    int n = 0, log2run = 6 + T.halvings;
    auto step = [&](int c) {
        if (lane == 0) {
            dim[n] = c;
            run[n] = log2run;
        }
        ++n;
        log2run -= __builtin_amdgcn_readlane(bits, c);
        cut &= ~(1ull << c);
    };
    if (T.sorted >= 0 && (cut >> T.sorted) & 1) step(T.sorted);
    while (cut) step(__builtin_ctzll(cut));
    if (lane == 0) *nstep = n;
}

template <int TILE>
__global__ __launch_bounds__(TB_THREADS)
void tree_build_kernel(const CellItem* __restrict__ items, const TreeDev* __restrict__ trees,
                       const double* __restrict__ arena, double* __restrict__ col64, int* perm) {
    constexpr int NW = TB_THREADS / ENM_WAVE;
    constexpr int PER = TILE / TB_THREADS;
    constexpr int LPW = TILE / ENM_LEAF / NW;   // leaves per wave
    __shared__ double sk[ENM_LDS_PAD(TILE)];
    __shared__ int si[ENM_LDS_PAD(TILE)];
    __shared__ int s_dim[ENM_TREE_STEPS], s_run[ENM_TREE_STEPS], s_nstep;
    __shared__ double s_width[16];
    const CellItem it = items[blockIdx.x];
    const TreeDev& T = trees[it.tree];
    const int tid = (int)threadIdx.x, lane = tid & (ENM_WAVE - 1), wave = tid / ENM_WAVE;
    const int p0 = it.cell * T.cell;
    const int cnt = min(T.cell, T.n - p0);
    // Padding (+inf, INT_MAX) sorts last; NaN keys sort as +inf, ahead of it.
    {
        int id[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int t = k * TB_THREADS + tid;
            id[k] = t >= cnt ? 0x7fffffff : T.slab >= 0 ? perm[T.slab + T.p0 + p0 + t] : T.p0 + p0 + t;
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) si[lp(k * TB_THREADS + tid)] = id[k];
    }
    __syncthreads();
    // The columns to sort by and the lengths (powers of two) of the runs sorted.
    int nstep = 0;
    if (T.halvings > 0) {
        for (int c = wave; c < T.ncol; c += NW) {
            const double w = cell_width(arena + T.src[c], si, cnt);
            if (lane == 0) s_width[c] = w;
        }
        __syncthreads();
        if (wave == 0) cell_steps(T, s_width, s_dim, s_run, &s_nstep);
        __syncthreads();
        nstep = s_nstep;
    }
    for (int s = 0; s < nstep; ++s) {
        if (s == 0 && s_dim[0] == T.sorted) continue;   // the slab order has it
        const double* src = arena + T.src[s_dim[s]];
        double key[PER];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int id = si[lp(k * TB_THREADS + tid)];
            key[k] = id != 0x7fffffff ? src[id] : INFINITY;
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) sk[lp(k * TB_THREADS + tid)] = vmin(key[k], INFINITY);
        block_sort_lds<TILE, TB_THREADS>(sk, si, 1 << s_run[s]);
    }
    __syncthreads();
    // Wave w takes leaves w * LPW onwards.
    const int ncol = T.ncol;
    double* box = col64 + T.box + (int64_t)it.cell * 2 * ncol * 64;
    double* leaves = col64 + T.col + (int64_t)p0 * ncol;
    int id[LPW];
    bool in[LPW];
#pragma unroll
    for (int k = 0; k < LPW; ++k) {
        const int t = (wave * LPW + k) * ENM_LEAF + lane;
        in[k] = t < cnt;
        id[k] = in[k] ? si[lp(t)] : 0;
        if (in[k]) perm[T.perm + p0 + t] = id[k];
    }
    const bool boxes = T.n > ENM_LEAF;
    __syncthreads();   // sk holds boxes from here on
    for (int c = 0; c < ncol; ++c) {
        const double* src = arena + T.src[c];
        double v[LPW];
#pragma unroll
        for (int k = 0; k < LPW; ++k) v[k] = in[k] ? src[id[k]] : __builtin_nan("");
#pragma unroll
        for (int k = 0; k < LPW; ++k) {
            const int leaf = wave * LPW + k;
            if (leaf * ENM_LEAF >= cnt) continue;   // wave-uniform
            leaves[((int64_t)leaf * ncol + c) * ENM_LEAF + lane] = v[k];
            if (!boxes) continue;
            const double lo = wave_ext_f64<false>(in[k] ? v[k] : INFINITY);
            const double hi = wave_ext_f64<true>(in[k] ? v[k] : -INFINITY);
            if (lane == 0) {
                box[(2 * c) * 64 + leaf] = lo;
                box[(2 * c + 1) * 64 + leaf] = hi;
                // Kept for the cell's box where there are several cells (of
                // 64 leaves: 2 * ncol * 64 <= TILE values).
                if (T.ncell > 1) {
                    sk[(2 * c) * 64 + leaf] = lo;
                    sk[(2 * c + 1) * 64 + leaf] = hi;
                }
            }
        }
    }
    if (T.ncell == 1) return;
    __syncthreads();
    const int nleaf = (cnt + ENM_LEAF - 1) / ENM_LEAF;
    double* cbox = col64 + T.cbox + (int64_t)(it.cell / 64) * 2 * ncol * 64 + it.cell % 64;
    for (int r = wave; r < 2 * ncol; r += NW) {
        const bool ok = lane < nleaf;
        const double v = sk[r * 64 + (ok ? lane : 0)];
        const double e = (r & 1) ? wave_ext_f64<true>(ok ? v : -INFINITY) : wave_ext_f64<false>(ok ? v : INFINITY);
        if (lane == 0) cbox[r * 64] = e;
    }
}

// Boxes of the groups of 64 cells: one wave per group (trees of more than 64
// cells).
__global__ __launch_bounds__(ENM_WAVE)
void tree_group_kernel(const CellItem* __restrict__ items, const TreeDev* __restrict__ trees,
                       double* __restrict__ col64) {
    const CellItem it = items[blockIdx.x];   // cell: the group
    const TreeDev& T = trees[it.tree];
    const int lane = (int)threadIdx.x, ncol = T.ncol;
    const bool in = it.cell * 64 + lane < T.ncell;
    const double* cbox = col64 + T.cbox + (int64_t)it.cell * 2 * ncol * 64;
    double* gbox = col64 + T.gbox + (int64_t)(it.cell / 64) * 2 * ncol * 64 + it.cell % 64;
    for (int r = 0; r < 2 * ncol; ++r) {
        const double v = in ? cbox[r * 64 + lane] : 0.0;
        const double e = (r & 1) ? wave_ext_f64<true>(in ? v : -INFINITY) : wave_ext_f64<false>(in ? v : INFINITY);
        if (lane == 0) gbox[r * 64] = e;
    }
}

// ---------------------------------------------------------------------------
// Ball counts, n_i = #{ j : max_d fl64(|a_d[j] - a_d[i]|) <= fl64(eps_i - 1e-12) }.
// The counts of a wave's queries are collected one per lane.

template <int D>
__global__ __launch_bounds__(TREE_WG* ENM_WAVE, tree_waves(D))
void tree_count_kernel(TreeArgs A, const CountDev* __restrict__ descs, const double* __restrict__ col64,
                       const double* __restrict__ eps, double* __restrict__ res64, int* __restrict__ res32,
                       unsigned long long* __restrict__ stats) {
    const TreeWork it = tree_work(A);
    if (it.nq <= 0) return;
    constexpr int Q = enm_tree_queries(D);
    const int lane = (int)(threadIdx.x & (ENM_WAVE - 1));
    const CountDev& cd = descs[it.desc];
    const TreeDev& T = A.trees[it.tile];
    const int t0 = it.t0, nq = it.nq;
    const int ncol = T.ncol;
    // Lane j holds query j: its point, radius and coordinates.
    const int pos = t0 + min(lane, nq - 1);
    const int pt = A.perm[T.perm + pos];
    const double rl = eps[cd.eps + pt] - 1e-12;
    const double* leaf = col64 + T.col + (int64_t)(t0 / ENM_LEAF) * ncol * ENM_LEAF;
    double ql[D];
#pragma unroll
    for (int d = 0; d < D; ++d) ql[d] = leaf[col_of<D>(d, ncol) * ENM_LEAF + pos % ENM_LEAF];
    int mine = 0;
    unsigned opened = 0;
    for (int j = 0; j < nq; j += Q) {
        // (Past the last query: a radius that no point is within.)
        double q[Q][D], r[Q];
        int c[Q];
        bool any = false;
#pragma unroll
        for (int k = 0; k < Q; ++k) {
            const int t = min(j + k, nq - 1);
            r[k] = j + k < nq ? lane_f64(rl, t) : -1.0;
            any = any || !(r[k] < 0.0);
#pragma unroll
            for (int d = 0; d < D; ++d) q[k][d] = lane_f64(ql[d], t);
        }
        if (!any) continue;
        count_queries<D, Q>(T, col64, q, r, c, opened);
#pragma unroll
        for (int k = 0; k < Q; ++k)
            if (lane == j + k) mine = c[k];
    }
    if (lane < nq) {
        res32[cd.counts + pt] = mine;
        // A zero count is +inf (psi_tab[0]), as psi(0) poisons the mean.
        res64[cd.psi_pt + pt] = A.psi_tab[mine];
    }
    if (lane == 0) add_stat(stats, ST_CNT_PAIRS, (unsigned long long)opened * ENM_LEAF);
}

}  // namespace

hipError_t enm_launch_tree_build(const CellItem* items, int n_items, const CellItem* groups, int n_groups, int tile,
                                 const TreeDev* trees, const double* arena, double* col64, int* perm, int* n_launch,
                                 hipStream_t st) {
    if (n_items <= 0) return hipSuccess;
    if (tile <= 1024)
        hipLaunchKernelGGL((tree_build_kernel<1024>), dim3(n_items), dim3(TB_THREADS), 0, st, items, trees, arena,
                           col64, perm);
    else if (tile <= 2048)
        hipLaunchKernelGGL((tree_build_kernel<2048>), dim3(n_items), dim3(TB_THREADS), 0, st, items, trees, arena,
                           col64, perm);
    else
        hipLaunchKernelGGL((tree_build_kernel<4096>), dim3(n_items), dim3(TB_THREADS), 0, st, items, trees, arena,
                           col64, perm);
    hipError_t e = hipGetLastError();
    ++*n_launch;
    if (e != hipSuccess || n_groups <= 0) return e;
    hipLaunchKernelGGL(tree_group_kernel, dim3(n_groups), dim3(ENM_WAVE), 0, st, groups, trees, col64);
    ++*n_launch;
    return hipGetLastError();
}

hipError_t enm_launch_tree_count(const Item* items, const int* qoff, int n_items, int qmax, int share,
                                 const CountDev* descs,
                                 const TreeDev* trees, const int* perm, const double* psi_tab, const double* col64,
                                 double* res64, int* res32, unsigned long long* stats, int dclass, hipStream_t st) {
    if (n_items <= 0) return hipSuccess;
    const TreeArgs a{items, qoff, share, trees, perm, psi_tab};
#define ENM_TREE_COUNT(D) \
    case D: \
        hipLaunchKernelGGL((tree_count_kernel<D>), dim3(tree_grid(qmax, share)), dim3(TREE_WG * ENM_WAVE), 0, st, a, descs, \
                           col64, res64, res64, res32, stats); \
        break;
    switch (dclass) {
        ENM_TREE_COUNT(2)
        ENM_TREE_COUNT(3)
        ENM_TREE_COUNT(4)
        ENM_TREE_COUNT(5)
        ENM_TREE_COUNT(6)
        ENM_TREE_COUNT(8)
        ENM_TREE_COUNT(12)
        ENM_TREE_COUNT(16)
        default: return hipErrorInvalidValue;
    }
#undef ENM_TREE_COUNT
    return hipGetLastError();
}
