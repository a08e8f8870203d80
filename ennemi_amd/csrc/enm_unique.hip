// Distinct rows and their counts, on the device: np.unique(rows, axis=0,
// return_inverse=True, return_counts=True) for the discrete plug-in
// estimators of the reference (ennemi/_entropy_estimators.py:44-56 entropy,
// :257-289 MI, :291-320 conditional MI), which spend their time there.
//
// A row set is one or more float64 columns of n values.  Each distinct
// column is sorted once (the library's segmented merge sort, keys compared
// as doubles and ties by point index, so -0.0 and 0.0 are one value, as for
// np.unique, and every NaN is a value of its own after the others); a run head
// is a position whose key differs from the previous one, and a value's code is
// the number of run heads up to it, minus one: codes number the distinct values
// in increasing order.  A row set of
// several columns is keyed by the mixed-radix number of its columns' codes
// (column 0 most significant: the order of np.unique's lexicographic row
// sort), exact in float64 while the product of the columns' distinct counts
// is at most 2^53, and factorised the same way.  Counts are run lengths.
#include "enm_device.h"
#include "enm_launch.h"

#include <algorithm>

namespace {

constexpr int UQ_THREADS = 256;
constexpr int UQ_PER = 8;                       // elements per thread of a tile
constexpr int UQ_TILE = UQ_THREADS * UQ_PER;    // as the sort's chunks
static_assert(UQ_TILE == ENM_SORT_TILE, "tiles are numbered by the segments' first_tile");

__device__ __forceinline__ int uq_seg(const UqSeg* __restrict__ segs, int nsegs, int tile) {
    int lo = 0, hi = nsegs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (segs[mid].first_tile <= tile) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Run heads among a thread's UQ_PER consecutive positions.
__device__ __forceinline__ int uq_heads(const UqSeg& sg, const double* __restrict__ skeys, int64_t i0,
                                        bool (&h)[UQ_PER]) {
    int heads = 0;
#pragma unroll
    for (int j = 0; j < UQ_PER; ++j) {
        const int64_t i = i0 + j;
        h[j] = i < sg.n && (i == 0 || skeys[sg.sbase + i] != skeys[sg.sbase + i - 1]);
        heads += h[j];
    }
    return heads;
}

// The sort holds NaN as +inf, in point order among the infinities.  np.unique
// puts NaN last and keeps every one apart: the points of the last run are laid
// out again, infinities first, and the keys of the others become NaN, which
// differ from whatever stands before them.  Next to nothing where the greatest
// key is finite.
constexpr int UQ_SEG_THREADS = 1024;
__device__ __forceinline__ void nan_last(const UqSeg& sg, const double* __restrict__ values, double* skeys, int* sidx,
                                         int* tmp, int* s_wave) {
    constexpr int NW = UQ_SEG_THREADS / ENM_WAVE;
    skeys += sg.sbase;
    sidx += sg.sbase;
    tmp += sg.sbase;
    if (skeys[sg.n - 1] < INFINITY) return;
    int64_t lo = 0, hi = sg.n - 1;   // the first infinite key
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (skeys[mid] < INFINITY) lo = mid + 1; else hi = mid;
    }
    const int lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    // Real infinities, then, given their number, every point's place.
    int64_t infinities = 0;
    for (int place = 0; place < 2; ++place) {
        int64_t before = 0;   // infinities among the positions done
        for (int64_t base = lo; base < sg.n; base += UQ_SEG_THREADS) {
            const int64_t i = base + threadIdx.x;
            const int pt = i < sg.n ? sidx[i] : 0;
            const bool real = i < sg.n && values[sg.src + pt] == INFINITY;
            const unsigned long long m = __builtin_amdgcn_ballot_w64(real);
            __syncthreads();   // the counts of the step before are read
            if (lane == 0) s_wave[wv] = (int)__popcll(m);
            __syncthreads();
            int64_t mine = before + (int)__popcll(m & ((1ull << lane) - 1ull));
            for (int w = 0; w < NW; ++w) {
                mine += w < wv ? s_wave[w] : 0;
                before += s_wave[w];
            }
            if (place && i < sg.n) tmp[real ? lo + mine : lo + infinities + (i - lo - mine)] = pt;
        }
        infinities = before;
        if (infinities == sg.n - lo) return;   // no NaN
    }
    __syncthreads();
    for (int64_t i = lo + threadIdx.x; i < sg.n; i += UQ_SEG_THREADS) {
        sidx[i] = tmp[i];
        if (i >= lo + infinities) skeys[i] = __builtin_nan("");
    }
}

__global__ __launch_bounds__(UQ_SEG_THREADS)
void uq_nan_kernel(const UqSeg* __restrict__ segs, const double* __restrict__ values, double* skeys, int* sidx,
                   int* tmp) {
    __shared__ int s_wave[UQ_SEG_THREADS / ENM_WAVE];
    nan_last(segs[blockIdx.x], values, skeys, sidx, tmp, s_wave);
}

// Codes, run starts, counts and the number of distinct values of short segments,
// one workgroup each, 1,024 positions at a time.  Bound by launches, of which a
// call has four fewer and, in its second stage, three; longer ones are bound by
// the positions in sequence.  The rows of two columns, both ways: 300 positions
// 197 us and 225 in passes, 5,000 283 and 311, 16,384 both 370, 30,000 486 and 451.
constexpr int64_t UQ_SEG_MAX = 16384;
__global__ __launch_bounds__(UQ_SEG_THREADS)
void uq_seg_kernel(const UqSeg* __restrict__ segs, const double* __restrict__ values, double* skeys, int* sidx, int* tmp,
                   int* codes, int64_t* starts, int64_t* counts, int64_t* distinct) {
    constexpr int NW = UQ_SEG_THREADS / ENM_WAVE;
    __shared__ int s_wave[NW];
    const UqSeg sg = segs[blockIdx.x];
    if (values) {
        nan_last(sg, values, skeys, sidx, tmp, s_wave);
        __syncthreads();
    }
    skeys += sg.sbase;
    sidx += sg.sbase;
    starts += sg.start_off;
    const int n = (int)sg.n, lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    int heads = 0;   // before this step
    for (int base = 0; base < n; base += UQ_SEG_THREADS) {
        const int i = base + (int)threadIdx.x;
        const bool head = i < n && (i == 0 || skeys[i] != skeys[i - 1]);
        const unsigned long long m = __builtin_amdgcn_ballot_w64(head);
        __syncthreads();   // the counts of the step before are read
        if (lane == 0) s_wave[wv] = (int)__popcll(m);
        __syncthreads();
        int rank = heads + (int)__popcll(m & ((2ull << lane) - 1ull)) - 1;
        for (int w = 0; w < NW; ++w) {
            rank += w < wv ? s_wave[w] : 0;
            heads += s_wave[w];
        }
        if (i < n) {
            codes[sg.code_off + sidx[i]] = rank;
            if (head) starts[rank] = i;
        }
    }
    if (threadIdx.x == 0) {
        starts[heads] = n;
        distinct[sg.slot] = heads;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < heads; r += UQ_SEG_THREADS) counts[sg.count_off + r] = starts[r + 1] - starts[r];
}

// Longer segments: three passes over tiles of 2,048 sorted positions (one workgroup per segment
// walked its tiles in sequence: 1.9 ms for two columns of 1,000,000): the run
// heads of every tile, their running sums per segment, then codes (by point)
// and run starts.
__global__ __launch_bounds__(UQ_THREADS)
void uq_heads_kernel(const UqSeg* __restrict__ segs, int nsegs, const double* __restrict__ skeys,
                     int* __restrict__ tile_heads) {
    __shared__ int s_wave[UQ_THREADS / ENM_WAVE];
    const UqSeg& sg = segs[uq_seg(segs, nsegs, (int)blockIdx.x)];
    const int64_t t0 = ((int64_t)blockIdx.x - sg.first_tile) * UQ_TILE;
    bool h[UQ_PER];
    int c = uq_heads(sg, skeys, t0 + threadIdx.x * UQ_PER, h);
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, ENM_WAVE);
    if ((threadIdx.x & (ENM_WAVE - 1)) == 0) s_wave[threadIdx.x / ENM_WAVE] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
        for (int w = 0; w < UQ_THREADS / ENM_WAVE; ++w) total += s_wave[w];
        tile_heads[blockIdx.x] = total;
    }
}

__global__ __launch_bounds__(ENM_WAVE)
void uq_scan_kernel(const UqSeg* __restrict__ segs, int* __restrict__ tile_heads, int64_t* __restrict__ starts,
                    int64_t* __restrict__ distinct) {
    const UqSeg sg = segs[blockIdx.x];
    const int lane = threadIdx.x;
    const int nt = (int)((sg.n + UQ_TILE - 1) / UQ_TILE);
    int carry = 0;
    for (int base = 0; base < nt; base += ENM_WAVE) {
        const int v = base + lane < nt ? tile_heads[sg.first_tile + base + lane] : 0;
        int inc = v;
        for (int off = 1; off < ENM_WAVE; off <<= 1) {
            const int o = __shfl_up(inc, off, ENM_WAVE);
            if (lane >= off) inc += o;
        }
        if (base + lane < nt) tile_heads[sg.first_tile + base + lane] = carry + inc - v;
        carry += __shfl(inc, ENM_WAVE - 1, ENM_WAVE);
    }
    if (lane == 0) {
        starts[sg.start_off + carry] = sg.n;
        distinct[sg.slot] = carry;
    }
}

__global__ __launch_bounds__(UQ_THREADS)
void uq_codes_kernel(const UqSeg* __restrict__ segs, int nsegs, const double* __restrict__ skeys,
                     const int* __restrict__ sidx, const int* __restrict__ tile_heads, int* __restrict__ codes,
                     int64_t* __restrict__ starts) {
    __shared__ int s_wave[UQ_THREADS / ENM_WAVE];
    const UqSeg& sg = segs[uq_seg(segs, nsegs, (int)blockIdx.x)];
    const int64_t i0 = ((int64_t)blockIdx.x - sg.first_tile) * UQ_TILE + threadIdx.x * UQ_PER;
    const int lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    bool h[UQ_PER];
    const int heads = uq_heads(sg, skeys, i0, h);
    int inc = heads;
    for (int off = 1; off < ENM_WAVE; off <<= 1) {
        const int o = __shfl_up(inc, off, ENM_WAVE);
        if (lane >= off) inc += o;
    }
    if (lane == ENM_WAVE - 1) s_wave[wv] = inc;
    __syncthreads();
    int64_t rank = tile_heads[blockIdx.x] + inc - heads - 1;   // code of the position before this thread's first
    for (int w = 0; w < wv; ++w) rank += s_wave[w];
#pragma unroll
    for (int j = 0; j < UQ_PER; ++j) {
        const int64_t i = i0 + j;
        if (i < sg.n) {
            rank += h[j];
            codes[sg.code_off + sidx[sg.sbase + i]] = (int)rank;
            if (h[j]) starts[sg.start_off + rank] = i;
        }
    }
}

// Points per code: run lengths.
__global__ __launch_bounds__(UQ_THREADS)
void uq_counts_kernel(const UqSeg* __restrict__ segs, int nsegs, const int64_t* __restrict__ starts,
                      const int64_t* __restrict__ distinct, int64_t* __restrict__ counts) {
    const UqSeg& sg = segs[uq_seg(segs, nsegs, (int)blockIdx.x)];
    const int64_t m = distinct[sg.slot];
    const int64_t r0 = ((int64_t)blockIdx.x - sg.first_tile) * UQ_TILE;
    for (int64_t r = r0 + threadIdx.x; r < min(m, r0 + UQ_TILE); r += UQ_THREADS)
        counts[sg.count_off + r] = starts[sg.start_off + r + 1] - starts[sg.start_off + r];
}

// ---------------------------------------------------------------------------
// Rows of whole numbers in small ranges (class labels, levels): counted
// directly, without a sort.

// An order-preserving integer image of a double, for atomic extrema.
__device__ __forceinline__ unsigned long long uq_image(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return b >> 63 ? ~b : b | (1ull << 63);
}

// Per column: the images of its least and greatest value, and whether a value
// is not a whole number below 2^53.  ext[3 c] starts at all ones, the others
// at 0.
__global__ __launch_bounds__(UQ_THREADS)
void uq_range_kernel(EnmRowsDev rows, const double* __restrict__ values, unsigned long long* __restrict__ ext) {
    __shared__ unsigned long long s_ext[UQ_THREADS / ENM_WAVE][3];
    const double* v = values + rows.col[blockIdx.y];
    unsigned long long lo = ~0ull, hi = 0;
    bool odd = false;
    for (int64_t i = (int64_t)blockIdx.x * UQ_THREADS + threadIdx.x; i < rows.n; i += (int64_t)gridDim.x * UQ_THREADS) {
        const double x = v[i] + 0.0;   // (-0.0 is 0.0)
        odd = odd || !(fabs(x) < 9007199254740992.0 && x == floor(x));
        const unsigned long long m = uq_image(x);
        lo = m < lo ? m : lo;
        hi = m > hi ? m : hi;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long a = __shfl_xor(lo, off, ENM_WAVE), b = __shfl_xor(hi, off, ENM_WAVE);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
    const bool any = wave_any(odd);
    const int wv = threadIdx.x / ENM_WAVE;
    if ((threadIdx.x & (ENM_WAVE - 1)) == 0) {
        s_ext[wv][0] = lo;
        s_ext[wv][1] = hi;
        s_ext[wv][2] = any ? 1 : 0;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long o = s_ext[0][2];
        lo = s_ext[0][0];
        hi = s_ext[0][1];
        for (int w = 1; w < UQ_THREADS / ENM_WAVE; ++w) {
            lo = s_ext[w][0] < lo ? s_ext[w][0] : lo;
            hi = s_ext[w][1] > hi ? s_ext[w][1] : hi;
            o |= s_ext[w][2];
        }
        atomicMin(ext + 3 * blockIdx.y, lo);
        atomicMax(ext + 3 * blockIdx.y + 1, hi);
        if (o) atomicOr(ext + 3 * blockIdx.y + 2, 1ull);
    }
}

// Points per mixed-radix key of their values' offsets from the columns' least.
// Bound by the reads of the columns; the counters of a workgroup are in LDS
// where they fit (a few labels are many additions to few addresses).
template <bool LDS>
__global__ __launch_bounds__(UQ_THREADS)
void uq_hist_kernel(EnmRowsDev rows, const double* __restrict__ values, int keys, unsigned* __restrict__ counts) {
    extern __shared__ unsigned s_counts[];
    if (LDS) {
        for (int k = threadIdx.x; k < keys; k += UQ_THREADS) s_counts[k] = 0;
        __syncthreads();
    }
    for (int64_t i = (int64_t)blockIdx.x * UQ_THREADS + threadIdx.x; i < rows.n; i += (int64_t)gridDim.x * UQ_THREADS) {
        int key = 0;
        for (int c = 0; c < rows.ncol; ++c)
            key = key * rows.radix[c] + (int)(values[rows.col[c] + i] - rows.least[c]);
        atomicAdd((LDS ? s_counts : counts) + key, 1u);
    }
    if (LDS) {
        __syncthreads();
        for (int k = threadIdx.x; k < keys; k += UQ_THREADS) {
            const unsigned c = s_counts[k];
            if (c) atomicAdd(counts + k, c);
        }
    }
}

// Both of a short row set by one workgroup, straight to host memory: the columns'
// extrema, and the counts where the keys fit LDS (out->keys of them; 0: not
// counted).  A call on a thousand labels then waits once for one kernel (9 us),
// where clearing, two kernels and two read-backs took 69 us of it.
constexpr int UQ_SHORT_THREADS = 1024;
__global__ __launch_bounds__(UQ_SHORT_THREADS)
void uq_short_kernel(EnmRowsDev rows, const double* __restrict__ values, int cap, UqShort* __restrict__ out) {
    constexpr int NW = UQ_SHORT_THREADS / ENM_WAVE;
    __shared__ unsigned s_counts[UQ_LDS_KEYS];
    __shared__ double s_lo[NW], s_hi[NW], s_least[16];
    __shared__ int s_odd[NW], s_radix[16];
    __shared__ double s_keys;
    const int n = (int)rows.n, tid = (int)threadIdx.x, wv = tid / ENM_WAVE;
    if (tid == 0) s_keys = 1.0;
    for (int c = 0; c < rows.ncol; ++c) {
        const double* v = values + rows.col[c];
        double lo = INFINITY, hi = -INFINITY;
        bool odd = false;
        for (int i = tid; i < n; i += UQ_SHORT_THREADS) {
            const double x = v[i] + 0.0;   // (-0.0 is 0.0)
            odd = odd || !(fabs(x) < 9007199254740992.0 && x == floor(x));
            lo = fmin(lo, x);
            hi = fmax(hi, x);
        }
        for (int off = 32; off > 0; off >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, off, ENM_WAVE));
            hi = fmax(hi, __shfl_xor(hi, off, ENM_WAVE));
        }
        const bool any = wave_any(odd);
        __syncthreads();
        if ((tid & (ENM_WAVE - 1)) == 0) {
            s_lo[wv] = lo;
            s_hi[wv] = hi;
            s_odd[wv] = any ? 1 : 0;
        }
        __syncthreads();
        if (tid == 0) {
            for (int w = 1; w < NW; ++w) {
                lo = fmin(lo, s_lo[w]);
                hi = fmax(hi, s_hi[w]);
                s_odd[0] |= s_odd[w];
            }
            lo = fmin(lo, s_lo[0]);
            hi = fmax(hi, s_hi[0]);
            out->least[c] = lo;
            out->most[c] = hi;
            out->odd[c] = s_odd[0];
            const double range = s_odd[0] ? INFINITY : hi - lo + 1.0;
            s_keys *= range;
            s_least[c] = lo;
            s_radix[c] = range <= UQ_LDS_KEYS ? (int)range : 0;
        }
    }
    __syncthreads();
    const int keys = s_keys <= (double)min(cap, UQ_LDS_KEYS) ? (int)s_keys : 0;
    if (tid == 0) out->keys = keys;
    if (keys == 0) return;
    for (int k = tid; k < keys; k += UQ_SHORT_THREADS) s_counts[k] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += UQ_SHORT_THREADS) {
        int key = 0;
        for (int c = 0; c < rows.ncol; ++c) key = key * s_radix[c] + (int)(values[rows.col[c] + i] - s_least[c]);
        atomicAdd(s_counts + key, 1u);
    }
    __syncthreads();
    for (int k = tid; k < keys; k += UQ_SHORT_THREADS) out->counts[k] = s_counts[k];
}

// Mixed-radix keys of the rows of multi-column row sets (exact doubles).
__global__ void uq_key_kernel(const UqRowKey* __restrict__ rk, int n_rk, const int* __restrict__ ccodes,
                              double* __restrict__ keys) {
    const int s = blockIdx.y;
    if (s >= n_rk) return;
    const UqRowKey r = rk[s];
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < r.n; p += (int64_t)gridDim.x * blockDim.x) {
        int64_t key = 0;
        for (int c = 0; c < r.ncol; ++c) key = key * r.radix[c] + ccodes[r.code_off[c] + p];
        keys[r.key_off + p] = (double)key;
    }
}

}  // namespace

hipError_t enm_launch_uq_codes(const UqSeg* segs, int nsegs, int ntiles, int64_t maxlen, const double* values,
                               double* skeys, int* sidx, int* tmp, int* tile_heads, int* codes, int64_t* starts,
                               int64_t* counts, int64_t* distinct, hipStream_t st) {
    if (nsegs <= 0) return hipSuccess;
    if (maxlen <= UQ_SEG_MAX) {
        hipLaunchKernelGGL(uq_seg_kernel, dim3(nsegs), dim3(UQ_SEG_THREADS), 0, st, segs, values, skeys, sidx, tmp,
                           codes, starts, counts, distinct);
        return hipGetLastError();
    }
    if (values)
        hipLaunchKernelGGL(uq_nan_kernel, dim3(nsegs), dim3(UQ_SEG_THREADS), 0, st, segs, values, skeys, sidx, tmp);
    hipLaunchKernelGGL(uq_heads_kernel, dim3(ntiles), dim3(UQ_THREADS), 0, st, segs, nsegs, skeys, tile_heads);
    hipLaunchKernelGGL(uq_scan_kernel, dim3(nsegs), dim3(ENM_WAVE), 0, st, segs, tile_heads, starts, distinct);
    hipLaunchKernelGGL(uq_codes_kernel, dim3(ntiles), dim3(UQ_THREADS), 0, st, segs, nsegs, skeys, sidx, tile_heads,
                       codes, starts);
    hipLaunchKernelGGL(uq_counts_kernel, dim3(ntiles), dim3(UQ_THREADS), 0, st, segs, nsegs, starts, distinct, counts);
    return hipGetLastError();
}

hipError_t enm_launch_uq_short(const EnmRowsDev& rows, const double* values, int cap, UqShort* out, hipStream_t st) {
    hipLaunchKernelGGL(uq_short_kernel, dim3(1), dim3(UQ_SHORT_THREADS), 0, st, rows, values, cap, out);
    return hipGetLastError();
}

hipError_t enm_launch_uq_range(const EnmRowsDev& rows, const double* values, unsigned long long* ext, hipStream_t st) {
    const int blocks = (int)std::min<int64_t>((rows.n + UQ_TILE - 1) / UQ_TILE, 256);
    hipLaunchKernelGGL(uq_range_kernel, dim3(blocks, rows.ncol), dim3(UQ_THREADS), 0, st, rows, values, ext);
    return hipGetLastError();
}

hipError_t enm_launch_uq_hist(const EnmRowsDev& rows, const double* values, int keys, unsigned* counts,
                              hipStream_t st) {
    const int blocks = (int)std::min<int64_t>((rows.n + UQ_TILE - 1) / UQ_TILE, 512);
    if (keys <= UQ_LDS_KEYS)
        hipLaunchKernelGGL(uq_hist_kernel<true>, dim3(blocks), dim3(UQ_THREADS), (size_t)keys * 4, st, rows, values,
                           keys, counts);
    else
        hipLaunchKernelGGL(uq_hist_kernel<false>, dim3(blocks), dim3(UQ_THREADS), 0, st, rows, values, keys, counts);
    return hipGetLastError();
}

hipError_t enm_launch_uq_keys(const UqRowKey* rk, int n_rk, int64_t max_n, const int* ccodes, double* keys,
                              hipStream_t st) {
    if (n_rk <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((max_n + 255) / 256, 4096);
    hipLaunchKernelGGL(uq_key_kernel, dim3((unsigned)std::max<int64_t>(blocks, 1), (unsigned)n_rk), dim3(256), 0, st,
                       rk, n_rk, ccodes, keys);
    return hipGetLastError();
}
