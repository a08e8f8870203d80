// Sorting of (key, index) pairs in registers and LDS by one workgroup, shared
// by the segmented sorts (enm_sort.hip) and the box-tree build (enm_tree.hip).
#pragma once
#include "enm_device.h"

namespace {

__device__ __forceinline__ bool kless(double ka, int ia, double kb, int ib) {
    return ka < kb || (ka == kb && ia < ib);
}

// Compare-exchange of two (key, index) pairs.
__device__ __forceinline__ void cex_pair(double& ka, int& ia, double& kb, int& ib) {
    const bool sw = kless(kb, ib, ka, ia);
    const double k0 = sw ? kb : ka, k1 = sw ? ka : kb;
    const int i0 = sw ? ib : ia, i1 = sw ? ia : ib;
    ka = k0; ia = i0; kb = k1; ib = i1;
}

// Sort PER (key, index) pairs held in registers (PER = 2, 4, 8 or 16;
// Batcher's odd-even merge sorting networks: 1, 5, 19 and 63 comparators).
template <int PER>
__device__ __forceinline__ void sort_regs(double (&k)[PER], int (&x)[PER]) {
#define ENM_CX(a, b) cex_pair(k[a], x[a], k[b], x[b])
    if constexpr (PER == 2) {
        ENM_CX(0, 1);
    } else if constexpr (PER == 4) {
        ENM_CX(0, 1); ENM_CX(2, 3); ENM_CX(0, 2); ENM_CX(1, 3); ENM_CX(1, 2);
    } else if constexpr (PER == 8) {
        ENM_CX(0, 1); ENM_CX(2, 3); ENM_CX(4, 5); ENM_CX(6, 7);
        ENM_CX(0, 2); ENM_CX(1, 3); ENM_CX(4, 6); ENM_CX(5, 7);
        ENM_CX(1, 2); ENM_CX(5, 6);
        ENM_CX(0, 4); ENM_CX(1, 5); ENM_CX(2, 6); ENM_CX(3, 7);
        ENM_CX(2, 4); ENM_CX(3, 5);
        ENM_CX(1, 2); ENM_CX(3, 4); ENM_CX(5, 6);
    } else {
        static_assert(PER == 16, "2, 4, 8 or 16 per thread");
        // Two sorted halves of 8 (the 19-comparator network on each) ...
        ENM_CX(0, 1); ENM_CX(2, 3); ENM_CX(0, 2); ENM_CX(1, 3); ENM_CX(1, 2);
        ENM_CX(4, 5); ENM_CX(6, 7); ENM_CX(4, 6); ENM_CX(5, 7); ENM_CX(5, 6);
        ENM_CX(0, 4); ENM_CX(2, 6); ENM_CX(2, 4); ENM_CX(1, 5); ENM_CX(3, 7); ENM_CX(3, 5);
        ENM_CX(1, 2); ENM_CX(3, 4); ENM_CX(5, 6);
        ENM_CX(8, 9); ENM_CX(10, 11); ENM_CX(8, 10); ENM_CX(9, 11); ENM_CX(9, 10);
        ENM_CX(12, 13); ENM_CX(14, 15); ENM_CX(12, 14); ENM_CX(13, 15); ENM_CX(13, 14);
        ENM_CX(8, 12); ENM_CX(10, 14); ENM_CX(10, 12); ENM_CX(9, 13); ENM_CX(11, 15); ENM_CX(11, 13);
        ENM_CX(9, 10); ENM_CX(11, 12); ENM_CX(13, 14);
        // ... and their odd-even merge (25 comparators).
        ENM_CX(0, 8); ENM_CX(4, 12); ENM_CX(4, 8); ENM_CX(2, 10); ENM_CX(6, 14); ENM_CX(6, 10);
        ENM_CX(2, 4); ENM_CX(6, 8); ENM_CX(10, 12); ENM_CX(1, 9); ENM_CX(5, 13); ENM_CX(5, 9);
        ENM_CX(3, 11); ENM_CX(7, 15); ENM_CX(7, 11); ENM_CX(3, 5); ENM_CX(7, 9); ENM_CX(11, 13);
        ENM_CX(1, 2); ENM_CX(3, 4); ENM_CX(5, 6); ENM_CX(7, 8); ENM_CX(9, 10); ENM_CX(11, 12);
        ENM_CX(13, 14);
    }
#undef ENM_CX
}

// LDS tiles of (key, index) pairs keep one unused slot after every 32
// elements (element i at lp(i)).  A thread's PER consecutive elements then
// start at a different bank from its neighbour's: without the slot, the 64
// lanes' 8-element runs (64 B apart) fall on the same few banks and every
// register-phase read and write serializes 16 ways.
#define ENM_LDS_PAD(n) ((n) + ((n) >> 5))
__device__ __forceinline__ int lp(int i) { return i + (i >> 5); }

// co_rank over an LDS tile: A at elements [a0, a0 + na), B at [b0, b0 + nb).
__device__ __forceinline__ int co_rank_lds(int d, const double* sk, const int* si, int a0, int na,
                                           int b0, int nb) {
    int lo = max(0, d - nb), hi = min(d, na);
    while (lo < hi) {
        const int i = (lo + hi) >> 1;
        const int pa = lp(a0 + i), pb = lp(b0 + d - i - 1);
        const double x = sk[pa], y = sk[pb];
        bool lt = x < y;
        if (x == y) lt = si[pa] < si[pb];
        if (lt) lo = i + 1; else hi = i;
    }
    return lo;
}

// The PER outputs of merge(A, B) of an LDS tile (A at [a0, a0 + na), B at
// [b0, b0 + nb), na, nb >= 1) from merge-path split (a, b): the two heads
// stay in registers and each step reloads only the side it consumed.
// Clamped reads stay inside the slices; the flags decide.
template <int PER>
__device__ __forceinline__ void seq_merge(const double* sk, const int* si, int a0, int na, int b0, int nb,
                                          int a, int b, int ne, double (&k)[PER], int (&x)[PER]) {
    double ha = sk[lp(a0 + min(a, na - 1))], hb = sk[lp(b0 + min(b, nb - 1))];
    int xa = si[lp(a0 + min(a, na - 1))], xb = si[lp(b0 + min(b, nb - 1))];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        if (e < ne) {
            const bool take_a = b >= nb || (a < na && kless(ha, xa, hb, xb));
            k[e] = take_a ? ha : hb;
            x[e] = take_a ? xa : xb;
            if (e + 1 < PER) {
                a += take_a ? 1 : 0;
                b += take_a ? 0 : 1;
                const int src = lp(take_a ? a0 + min(a, na - 1) : b0 + min(b, nb - 1));
                const double v = sk[src];
                const int vi = si[src];
                ha = take_a ? v : ha;
                xa = take_a ? vi : xa;
                hb = take_a ? hb : v;
                xb = take_a ? xb : vi;
            }
        }
    }
}

// Sort the TILE (key, index) pairs of an LDS tile (ENM_LDS_PAD(TILE) slots)
// with an NT-thread block: each thread sorts TILE/NT consecutive pairs in
// registers, then merge levels of doubling run width, each thread producing
// TILE/NT consecutive outputs of its pair of runs from a merge-path split
// (outputs kept in registers across a barrier, so the merge works in place).
// Padding keys (+inf, INT_MAX) sort last.  With `seg` (a power of two of at
// least TILE/NT), runs of seg pairs are sorted, each by itself.  Starts and
// ends with a barrier.
template <int TILE, int NT = ENM_SORT_THREADS>
__device__ __forceinline__ void block_sort_lds(double* sk, int* si, int seg = TILE) {
    constexpr int PER = TILE / NT;
    __syncthreads();
    const int e0 = threadIdx.x * PER;
    double k[PER];
    int x[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) { k[e] = sk[lp(e0 + e)]; x[e] = si[lp(e0 + e)]; }
    sort_regs<PER>(k, x);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < PER; ++e) { sk[lp(e0 + e)] = k[e]; si[lp(e0 + e)] = x[e]; }
    __syncthreads();
    for (int run = PER; run < seg; run <<= 1) {
        const int pb = (e0 / (2 * run)) * (2 * run);
        const int d = e0 - pb;
        const int a = co_rank_lds(d, sk, si, pb, run, pb + run, run);
        seq_merge<PER>(sk, si, pb, run, pb + run, run, a, d - a, PER, k, x);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < PER; ++e) { sk[lp(e0 + e)] = k[e]; si[lp(e0 + e)] = x[e]; }
        __syncthreads();
    }
}

}  // namespace
