// Dispatch of the kNN launches by joint dimension and list depth; the
// kernels themselves are in enm_knn.h, instantiated per dimension class
// by enm_knn_d*.hip.
#include "enm_knn.h"

namespace {

// One column: the k+1 nearest of position i are k+1 consecutive sorted keys
// that include it, and with L(a) = fl64(x_i - x_{i-a}) and R(b) =
// fl64(x_{i+b} - x_i), both non-decreasing, the radius is the least of
// max(L(a), R(k - a)) over the windows inside the scope.  L rises and R(k - a)
// falls with a, so a binary search finds the first a with L(a) >= R(k - a),
// and the answer is L there or R just before it.  The few keys a thread reads
// lie around its own position, so they come from the lines its neighbours
// read (three variables of 1,000,000 points in 16 classes, k = 3: 11.5 ms by
// scanning the sorted keys in steps of 64 for all lanes of a wave, 0.07 so).
__global__ __launch_bounds__(ENM_LINE_THREADS)
void knn_line_kernel(const Item* __restrict__ items, const KnnDev* __restrict__ descs,
                     const OrderDev* __restrict__ orders, const int* __restrict__ perm,
                     const double* __restrict__ col64, double* __restrict__ res64,
                     unsigned long long* __restrict__ stats) {
    const Item it = items[blockIdx.x];
    const KnnDev kd = descs[it.desc];
    const OrderDev& od = orders[kd.order];
    const double* x = col64 + od.c64;
    const int64_t at = od.perm;
    const int k = kd.k;
    unsigned read = 0;
    for (int i = it.t0 + (int)threadIdx.x; i < it.t1; i += ENM_LINE_THREADS) {
        double e = INFINITY;
        if (it.hi - it.lo > k) {
            const double xi = x[i];
            // Windows [i - a, i + k - a] inside [lo, hi).
            int a = max(0, k - (it.hi - 1 - i));
            const int a1 = min(k, i - it.lo);
            int n = a1 - a;   // L(a) >= R(k - a) first holds at a + n at most (or nowhere)
            const int a0 = a;
            while (n > 0) {
                const int h = n >> 1;
                const double l = xi - x[i - a - h], r = x[i + k - a - h] - xi;
                if (l >= r) n = h;
                else { a += h + 1; n -= h + 1; }
                read += 2;
            }
            const double l = xi - x[i - a], r = x[i + k - a] - xi;
            e = l >= r ? l : r;
            if (a > a0) e = vmin(e, x[i + k - a + 1] - xi);
            read += 3;
            // Equal infinities differ by NaN: no neighbour.
            if (!(e < INFINITY)) e = INFINITY;
        }
        if (kd.eps >= 0) res64[kd.eps + i] = e;
        if (kd.eps_orig >= 0) res64[kd.eps_orig + perm[at + i]] = e;
    }
    const unsigned long long total = wave_sum_u64(read);
    if ((threadIdx.x & (ENM_WAVE - 1)) == 0) add_stat(stats, ST_KNN_PAIRS, total);
}

}  // namespace

hipError_t enm_launch_knn_line(const Item* items, int n_items, const KnnDev* descs, const OrderDev* orders,
                               const int* perm, const double* col64, double* res64, unsigned long long* stats,
                               hipStream_t st) {
    if (n_items <= 0) return hipSuccess;
    hipLaunchKernelGGL(knn_line_kernel, dim3(n_items), dim3(ENM_LINE_THREADS), 0, st, items, descs, orders, perm,
                       col64, res64, stats);
    return hipGetLastError();
}

int enm_knn_dim_class(int d) {
    if (d <= 6) return d;
    if (d <= 8) return 8;
    if (d <= 12) return 12;
    if (d <= 16) return 16;
    return -1;
}

int enm_knn_list_class(int k1) {
    if (k1 <= 4) return 4;
    if (k1 <= 8) return 8;
    if (k1 <= 16) return 16;
    if (k1 <= 32) return 32;
    if (k1 <= ENM_LIST_LDS_MAX) return ENM_LIST_HEAP_LDS;
    return ENM_LIST_HEAP_GLOBAL;
}

hipError_t enm_launch_knn(const Item* items, const int* qoff, int n_items, unsigned* counter,
                          const KnnDev* descs, const OrderDev* orders,
                          const unsigned long long* maxabs, const int* perm,
                          const double* col64, const float* col32, double* res64,
                          unsigned long long* stats, int dclass, int pclass, bool f32, bool brute,
                          int walk, int grid, int k1max, double* heap, int ticket, int smax, char* far,
                          unsigned* far_count, int64_t far_bytes, hipStream_t st) {
    if (n_items <= 0) return hipSuccess;
    // Tickets of up to ENM_KCHUNK items (or the tuned items per ticket), but
    // at least four per wave of the grid, so small launches still fill it.
    const int chunk = std::max(1, std::min(ticket > 0 ? ticket : ENM_KCHUNK, n_items / (4 * std::max(1, grid))));
    KnnArgs a{items, qoff, counter, chunk, descs, orders, maxabs, perm, brute ? 1 : 0,
              heap, (int64_t)ENM_WAVE * k1max, smax, far, far_count, far_bytes};
    if (pclass == ENM_LIST_HEAP_GLOBAL && heap == nullptr) return hipErrorInvalidValue;
    switch (dclass) {
        case 1: return enm_knn_launch_d1(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 2: return enm_knn_launch_d2(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 3: return enm_knn_launch_d3(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 4: return enm_knn_launch_d4(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 5: return enm_knn_launch_d5(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 6: return enm_knn_launch_d6(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 8: return enm_knn_launch_d8(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 12: return enm_knn_launch_d12(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        case 16: return enm_knn_launch_d16(a, pclass, f32, walk, grid, col64, col32, res64, stats, st);
        default: return hipErrorInvalidValue;
    }
}

int enm_knn_heap_grid(int grid, int k1max) {
    const int64_t per_block = (int64_t)ENM_WAVE * k1max * (int64_t)sizeof(double);
    const int64_t most = std::max<int64_t>(1, ENM_HEAP_GLOBAL_BYTES / std::max<int64_t>(1, per_block));
    return (int)std::max<int64_t>(1, std::min<int64_t>(grid, most));
}
