// Rows grouped by class: every column of a task scattered so that the rows of
// a class are consecutive, classes in ascending order and rows in their own
// order within a class, as np.unique's order and a stable argsort give them in
// the reference (ennemi/_entropy_estimators.py:177-196 visits the classes in
// turn).  The labels are whole numbers in a small range.
//
// A counting sort: the rows of each class in every block of 2,048 rows
// (group_count_kernel), running sums over the blocks of a class and the
// classes of a task (group_scan_kernel), and the scatter, in which each wave
// owns 512 consecutive rows, 64 at a time, and ranks equal labels by ballots.
// Bound by the scattered stores (whole runs of a class inside a block).
#include "enm_device.h"
#include "enm_launch.h"

namespace {

constexpr int GR_THREADS = 256;
constexpr int GR_WAVES = GR_THREADS / ENM_WAVE;
constexpr int GR_ROUNDS = ENM_PREP_BLOCK / GR_THREADS;   // 64-row rounds of a wave

__device__ __forceinline__ int label_of(const GroupTaskDev& t, const double* __restrict__ src, int64_t i) {
    return (int)(src[t.label + i] - t.least);
}

// Row of a wave's round: waves own consecutive rows of the block.
__device__ __forceinline__ int64_t wave_row(int64_t r0, int round) {
    return r0 + (int64_t)(threadIdx.x / ENM_WAVE) * (GR_ROUNDS * ENM_WAVE) + round * ENM_WAVE +
           (threadIdx.x & (ENM_WAVE - 1));
}

__global__ __launch_bounds__(GR_THREADS)
void group_count_kernel(const GroupTaskDev* __restrict__ tasks, int64_t stride, const double* __restrict__ src,
                        int classes, int* __restrict__ counts) {
    extern __shared__ int s_cnt[];
    const int ti = (int)(blockIdx.x / stride);
    const GroupTaskDev& t = tasks[ti];
    const int64_t r0 = (blockIdx.x - ti * stride) * ENM_PREP_BLOCK;
    if (r0 >= t.n) return;
    for (int c = threadIdx.x; c < classes; c += GR_THREADS) s_cnt[c] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < GR_ROUNDS; ++j) {
        const int64_t i = r0 + j * GR_THREADS + threadIdx.x;
        if (i < t.n) atomicAdd(&s_cnt[label_of(t, src, i)], 1);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < classes; c += GR_THREADS) counts[(int64_t)blockIdx.x * classes + c] = s_cnt[c];
}

// One workgroup per task: counts become the first position of each block's
// rows of each class; sizes[c] the rows of class c.
__global__ __launch_bounds__(GR_THREADS)
void group_scan_kernel(const GroupTaskDev* __restrict__ tasks, int64_t stride, int classes, int* __restrict__ counts,
                       int64_t* __restrict__ sizes) {
    extern __shared__ int s_base[];   // rows of every class, then their first position
    const GroupTaskDev& t = tasks[blockIdx.x];
    const int nb = (int)((t.n + ENM_PREP_BLOCK - 1) / ENM_PREP_BLOCK);
    int* cnt = counts + (int64_t)blockIdx.x * stride * classes;
    constexpr int BATCH = 16;   // blocks read together
    for (int c = threadIdx.x; c < classes; c += GR_THREADS) {
        int run = 0;
        for (int b = 0; b < nb; b += BATCH) {
            int v[BATCH];
#pragma unroll
            for (int k = 0; k < BATCH; ++k) v[k] = b + k < nb ? cnt[(int64_t)(b + k) * classes + c] : 0;
#pragma unroll
            for (int k = 0; k < BATCH; ++k) {
                if (b + k < nb) cnt[(int64_t)(b + k) * classes + c] = run;
                run += v[k];
            }
        }
        s_base[c] = run;
        sizes[(int64_t)blockIdx.x * classes + c] = run;
    }
    __syncthreads();
    // First positions of the classes: one wave, 64 classes at a time.
    if (threadIdx.x < ENM_WAVE) {
        const int lane = threadIdx.x;
        int carry = 0;
        for (int c0 = 0; c0 < classes; c0 += ENM_WAVE) {
            const int v = c0 + lane < classes ? s_base[c0 + lane] : 0;
            int inc = v;
            for (int off = 1; off < ENM_WAVE; off <<= 1) {
                const int o = __shfl_up(inc, off, ENM_WAVE);
                if (lane >= off) inc += o;
            }
            if (c0 + lane < classes) s_base[c0 + lane] = carry + inc - v;
            carry += __shfl(inc, ENM_WAVE - 1, ENM_WAVE);
        }
    }
    __syncthreads();
    for (int64_t e = threadIdx.x; e < (int64_t)nb * classes; e += GR_THREADS) cnt[e] += s_base[e % classes];
}

__global__ __launch_bounds__(GR_THREADS)
void group_scatter_kernel(const GroupTaskDev* __restrict__ tasks, int64_t stride, const double* __restrict__ src,
                          int classes, const int* __restrict__ counts, double* __restrict__ dst) {
    extern __shared__ int s_next[];   // [wave][class]: where the wave's next row of the class goes
    const int ti = (int)(blockIdx.x / stride);
    const GroupTaskDev& t = tasks[ti];
    const int64_t r0 = (blockIdx.x - ti * stride) * ENM_PREP_BLOCK;
    if (r0 >= t.n) return;
    const int lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    for (int c = threadIdx.x; c < GR_WAVES * classes; c += GR_THREADS) s_next[c] = 0;
    __syncthreads();
    int label[GR_ROUNDS];
#pragma unroll
    for (int j = 0; j < GR_ROUNDS; ++j) {
        const int64_t i = wave_row(r0, j);
        label[j] = i < t.n ? label_of(t, src, i) : -1;
        if (label[j] >= 0) atomicAdd(&s_next[wv * classes + label[j]], 1);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < classes; c += GR_THREADS) {
        int at = counts[(int64_t)blockIdx.x * classes + c];
#pragma unroll
        for (int w = 0; w < GR_WAVES; ++w) {
            const int v = s_next[w * classes + c];
            s_next[w * classes + c] = at;
            at += v;
        }
    }
    __syncthreads();
    volatile int* next = s_next + wv * classes;
    int pos[GR_ROUNDS];
#pragma unroll
    for (int j = 0; j < GR_ROUNDS; ++j) {
        pos[j] = 0;
        unsigned long long open = __builtin_amdgcn_ballot_w64(label[j] >= 0);
        while (open) {
            const int c = __builtin_amdgcn_readlane(label[j], __builtin_ctzll(open));
            const unsigned long long m = __builtin_amdgcn_ballot_w64(label[j] == c);
            const int at = next[c];
            if (label[j] == c) pos[j] = at + (int)__popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) next[c] = at + (int)__popcll(m);
            __builtin_amdgcn_wave_barrier();
            open &= ~m;
        }
    }
    for (int c = 0; c < t.ncol; ++c) {
        const double* from = src + t.src[c];
        double* to = dst + t.dst[c];
        double v[GR_ROUNDS];
#pragma unroll
        for (int j = 0; j < GR_ROUNDS; ++j) v[j] = label[j] >= 0 ? from[wave_row(r0, j)] : 0.0;
#pragma unroll
        for (int j = 0; j < GR_ROUNDS; ++j)
            if (label[j] >= 0) to[pos[j]] = v[j];
    }
}

}  // namespace

hipError_t enm_launch_group(const GroupTaskDev* tasks, int n_tasks, int64_t stride, int classes, const double* src,
                            int* counts, int64_t* sizes, double* dst, hipStream_t st) {
    const dim3 grid((unsigned)(stride * n_tasks)), block(GR_THREADS);
    hipLaunchKernelGGL(group_count_kernel, grid, block, (size_t)classes * 4, st, tasks, stride, src, classes, counts);
    hipLaunchKernelGGL(group_scan_kernel, dim3(n_tasks), block, (size_t)classes * 4, st, tasks, stride, classes,
                       counts, sizes);
    hipLaunchKernelGGL(group_scatter_kernel, grid, block, (size_t)GR_WAVES * classes * 4, st, tasks, stride, src,
                       classes, counts, dst);
    return hipGetLastError();
}
