// Device-side preparation of estimate_mi tasks: the lag windows, mask and
// NaN compaction, and the rescaling of ennemi's _lagged_mi
// (ennemi/_driver.py:795-806 windows, :834-854 _apply_masks, :871-902
// _rescale_data), producing the float64 instance columns of a batch directly
// in HBM from the raw series.
//
// Every value is bit-identical to NumPy's:
//   * compaction keeps the rows in order (a stable prefix scan per block);
//   * x.mean() and x.std() of a column (and of a one-column condition) sum
//     in NumPy's order: 8192-element chunks, each by its pairwise recursion
//     (halves cut at a multiple of 8, leaves of at most 128 elements summed
//     by 8 interleaved accumulators), the chunk sums added in order to -0.0;
//   * zs.mean(axis=0) and zs.std(axis=0) of a condition of two or more
//     columns accumulate each column row by row;
//   * std = sqrt(sum((v - mean)^2) / n); the scaled value is
//     ((v - mean) / std) + noise, each operation rounded once (the library
//     is built without FP contraction).
// The noise is the reference's: every task draws from a fresh
// default_rng(2_718281828) in the order x, y, z (z row-major), so its draws
// are prefixes of one stream, which the host generates once per call.  A
// variable with std < 1e-20 is left as it is and draws nothing (for the
// condition: if any of its columns is constant).
#include "enm_device.h"
#include "enm_launch.h"
#include "enm_tree.h"

namespace {

constexpr int PB_THREADS = 256;
constexpr int PB_ROWS = ENM_PREP_BLOCK;          // rows per block
constexpr int PB_ROUNDS = PB_ROWS / PB_THREADS;  // rows per thread
constexpr int PW_CHUNK = 8192;                   // NumPy's reduction buffer
constexpr int PW_LEAF = 128;                     // NumPy's pairwise block

// Window row r of task t in two steps, so that a thread issues the loads of
// all its rows before it uses any: row_load reads x, y and the mask byte;
// row_keep says whether the row is kept (the mask first, then, with
// drop_nan, no NaN in x, y or the condition) and whether a row that passes
// the mask holds a NaN.  Rows at or past the window's end are neither kept
// nor NaN (row 0 is read instead, so every load stays inside the series).
__device__ __forceinline__ void row_load(const PrepTaskDev& t, const double* __restrict__ raw,
                                         const unsigned char* __restrict__ mask, int64_t r0,
                                         double (&xv)[PB_ROUNDS], double (&yv)[PB_ROUNDS], int (&mk)[PB_ROUNDS]) {
#pragma unroll
    for (int j = 0; j < PB_ROUNDS; ++j) {
        const int64_t r = r0 + j * PB_THREADS + threadIdx.x;
        const int64_t rr = r < t.w ? r : 0;
        xv[j] = raw[t.x_col + t.x0 + rr];
        yv[j] = raw[t.y_col + t.y0 + rr];
    }
    if (mask != nullptr) {   // uniform: the bytes' loads go out together too
#pragma unroll
        for (int j = 0; j < PB_ROUNDS; ++j) {
            const int64_t r = r0 + j * PB_THREADS + threadIdx.x;
            mk[j] = mask[t.y0 + (r < t.w ? r : 0)];
        }
    } else {
#pragma unroll
        for (int j = 0; j < PB_ROUNDS; ++j) mk[j] = 1;
    }
}

__device__ __forceinline__ bool row_keep(const PrepTaskDev& t, const double* __restrict__ raw, int drop_nan,
                                         int64_t r, double xv, double yv, int mk, bool& has_nan) {
    const bool in = r < t.w;
    const int64_t rr = in ? r : 0;
    const bool pass = in && mk != 0;
    bool nan = isnan(xv) || isnan(yv);
    for (int c = 0; c < t.dz; ++c) nan = nan || isnan(raw[t.z_col[c] + t.z0[c] + rr]);
    has_nan = pass && nan;
    return pass && !(drop_nan && nan);
}

// Rows of m columns (row-major, as NumPy holds a table) to columns of n rows:
// 64 x 64 tiles through LDS, both sides in whole lines.
constexpr int PC_TILE = 64;
constexpr int PC_THREADS = 256;
__global__ __launch_bounds__(PC_THREADS)
void prep_columns_kernel(const double* __restrict__ rows, int64_t n, int m, double* __restrict__ cols) {
    __shared__ double tile[PC_TILE][PC_TILE + 1];
    const int64_t r0 = (int64_t)blockIdx.x * PC_TILE;
    const int c0 = (int)blockIdx.y * PC_TILE;
    // Narrow tables: consecutive threads read consecutive values of the rows.
    const int w = min(PC_TILE, m - c0), h = (int)min((int64_t)PC_TILE, n - r0);
    for (int t = (int)threadIdx.x; t < h * w; t += PC_THREADS) {
        const int r = t / w, c = t - r * w;
        tile[r][c] = rows[(r0 + r) * m + c0 + c];
    }
    __syncthreads();
    for (int t = (int)threadIdx.x; t < w * PC_TILE; t += PC_THREADS) {
        const int c = t / PC_TILE, r = t % PC_TILE;
        if (r < h) cols[(int64_t)(c0 + c) * n + r0 + r] = tile[r][c];
    }
}

// Blocks are laid out `stride` per task (the most any task needs; the
// rest of a shorter task's blocks find no rows), so a block's task is a
// division, not a search.

// Phase 1: kept rows per block, and a NaN among the masked rows per task.
// Every row's loads are issued before any of them is used.
__global__ __launch_bounds__(PB_THREADS)
void prep_count_kernel(const PrepTaskDev* __restrict__ tasks, int64_t stride, const double* __restrict__ raw,
                       const unsigned char* __restrict__ mask, int drop_nan, int* __restrict__ blk_count,
                       unsigned* __restrict__ nan_flag, int64_t* __restrict__ blk_off,
                       PrepCounted* __restrict__ out) {
    __shared__ int s_cnt[PB_THREADS / ENM_WAVE];
    __shared__ int s_nan;
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);   // a task's blocks on one XCD
    const int ti = (int)(b / stride);
    const PrepTaskDev& t = tasks[ti];   // read in place: a copy indexed by c would sit in scratch
    const int64_t r0 = (b - ti * stride) * PB_ROWS;
    if (threadIdx.x == 0) s_nan = 0;
    __syncthreads();
    int cnt = 0;
    bool any_nan = false;
    double xv[PB_ROUNDS], yv[PB_ROUNDS];
    int mk[PB_ROUNDS];
    row_load(t, raw, mask, r0, xv, yv, mk);
#pragma unroll
    for (int j = 0; j < PB_ROUNDS; ++j) {
        bool nan;
        cnt += row_keep(t, raw, drop_nan, r0 + j * PB_THREADS + threadIdx.x, xv[j], yv[j], mk[j], nan) ? 1 : 0;
        any_nan = any_nan || nan;
    }
    const int lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, ENM_WAVE);
    if (lane == 0) s_cnt[wv] = cnt;
    if (wave_any(any_nan) && lane == 0) s_nan = 1;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < PB_THREADS / ENM_WAVE; ++w) tot += s_cnt[w];
        const unsigned nan = s_nan && !drop_nan ? 1u : 0u;
        if (stride == 1) {   // the task's only block: nothing to scan
            blk_off[b] = 0;
            out[ti] = PrepCounted{tot, nan, 0};
        } else {
            blk_count[b] = tot;
            if (nan) atomicOr(nan_flag + ti, 1u);
        }
    }
}

// Per task: block offsets (exclusive scan of the block counts, in place in
// blk_off), and to host memory the kept rows n and whether a NaN is among them
// (two copies less per call).  One wave per task.
__global__ __launch_bounds__(ENM_WAVE)
void prep_scan_kernel(const PrepTaskDev* __restrict__ tasks, int64_t stride, int n_tasks,
                      const int* __restrict__ blk_count, int64_t* __restrict__ blk_off,
                      const unsigned* __restrict__ nan_flag, PrepCounted* __restrict__ out) {
    const int ti = blockIdx.x;
    if (ti >= n_tasks) return;
    const int64_t b0 = ti * stride, nb = tasks[ti].nblk;
    const int lane = threadIdx.x;
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += ENM_WAVE) {
        const int64_t v = base + lane < nb ? blk_count[b0 + base + lane] : 0;
        int64_t inc = v;
        for (int off = 1; off < ENM_WAVE; off <<= 1) {
            const int64_t o = __shfl_up(inc, off, ENM_WAVE);
            if (lane >= off) inc += o;
        }
        if (base + lane < nb) blk_off[b0 + base + lane] = carry + inc - v;
        carry += __shfl(inc, ENM_WAVE - 1, ENM_WAVE);
    }
    if (lane == 0) out[ti] = PrepCounted{carry, nan_flag[ti], 0};
}

// Phase 2a: the kept rows of every block, in row order, to the task's
// arena columns (x, y, then the condition columns, n values each); with a
// kept-row map, each 32 window rows' kept bits and the kept rows before
// them, for the sort hints.  Every
// row's state and x, y values are read first; one barrier then gives each
// wave the kept rows of the waves before it, round by round.
__device__ __forceinline__ void compact_rows(const PrepTaskDev& t, int64_t r0, int64_t pos, const double* __restrict__ raw,
                                             const unsigned char* __restrict__ mask, int drop_nan,
                                             double* __restrict__ arena, KeptWord* __restrict__ kept) {
    constexpr int NW = PB_THREADS / ENM_WAVE;
    __shared__ int s_wcnt[PB_ROUNDS][NW];
    const int lane = threadIdx.x & (ENM_WAVE - 1), wv = threadIdx.x / ENM_WAVE;
    bool keep[PB_ROUNDS];
    double xv[PB_ROUNDS], yv[PB_ROUNDS];
    int below[PB_ROUNDS];
    int mk[PB_ROUNDS];
    row_load(t, raw, mask, r0, xv, yv, mk);
#pragma unroll
    for (int j = 0; j < PB_ROUNDS; ++j) {
        bool nan;
        keep[j] = row_keep(t, raw, drop_nan, r0 + j * PB_THREADS + threadIdx.x, xv[j], yv[j], mk[j], nan);
    }
    unsigned long long wm[PB_ROUNDS];
#pragma unroll
    for (int j = 0; j < PB_ROUNDS; ++j) {
        const unsigned long long m = __builtin_amdgcn_ballot_w64(keep[j]);
        wm[j] = m;
        below[j] = __popcll(m & ((1ull << lane) - 1ull));
        if (lane == 0) s_wcnt[j][wv] = __popcll(m);
    }
    __syncthreads();
    double* out = arena + t.arena_off;
#pragma unroll
    for (int j = 0; j < PB_ROUNDS; ++j) {
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            before += w < wv ? s_wcnt[j][w] : 0;
            total += s_wcnt[j][w];
        }
        const int64_t r = r0 + j * PB_THREADS + threadIdx.x;
        const int64_t p = pos + before + below[j];
        if (keep[j]) {
            out[p] = xv[j];
            out[t.n + p] = yv[j];
            for (int c = 0; c < t.dz; ++c) out[(2 + c) * t.n + p] = raw[t.z_col[c] + t.z0[c] + r];
        }
        if (kept != nullptr && lane < 2) {
            // The wave's 64 rows are two words of the map.
            const int64_t row = r0 + j * PB_THREADS + wv * ENM_WAVE + 32 * lane;
            if (row < t.w) {
                const uint32_t lo = (uint32_t)wm[j];
                const uint32_t bits = lane ? (uint32_t)(wm[j] >> 32) : lo;
                const int64_t pre = pos + before + (lane ? __popc(lo) : 0);
                kept[t.pmap + row / 32] = KeptWord{bits, (int32_t)pre};
            }
        }
        pos += total;
    }
}

__global__ __launch_bounds__(PB_THREADS)
void prep_compact_kernel(const PrepTaskDev* __restrict__ tasks, int64_t stride,
                         const double* __restrict__ raw, const unsigned char* __restrict__ mask, int drop_nan,
                         const int64_t* __restrict__ blk_off, double* __restrict__ arena,
                         KeptWord* __restrict__ kept) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);   // a task's blocks on one XCD
    const int ti = (int)(b / stride);
    // (The task is read in place: a copy indexed by c would sit in scratch.)
    compact_rows(tasks[ti], (b - ti * stride) * PB_ROWS, blk_off[b], raw, mask, drop_nan, arena, kept);
}

// One term of a sum: the value, or its squared deviation from `mean`.
struct Term {
    const double* v;
    double mean;
    bool dev;
    __device__ __forceinline__ double operator()(int64_t i) const {
        if (!dev) return v[i];
        const double d = v[i] - mean;
        return d * d;
    }
};

// NumPy's pairwise recursion over n <= PW_CHUNK values as a heap-ordered
// binary tree (node 1 the root, nodes 2i and 2i+1 the halves of node i): a
// node of more than PW_LEAF values splits at half its length rounded down
// to a multiple of 8; smaller nodes are leaves.  Right halves are at most
// half their parent plus 8 values, so every leaf of an 8191-value chunk is
// within depth 7: heap slots 1 .. PW_HEAP - 1.
constexpr int PW_HEAP = 256;
constexpr int PW_DEPTH = 7;

// The sum of a full PW_CHUNK-value chunk in NumPy's order, by one wave: the
// recursion's 64 leaves of 128 values form a balanced tree.  Lane l takes
// accumulator l % 8 of leaf 8 * pass + l / 8 (sixteen values, added in
// order), so one load instruction reads eight 64-byte runs.  Butterfly
// shuffles then combine the accumulators as the leaf does,
// ((r0 + r1) + (r2 + r3)) + ((r4 + r5) + (r6 + r7)), and the pass's eight
// leaves pairwise; IEEE addition commutes, so both lanes of a pair hold the
// same bits.  The eight passes' subtree sums end the tree.
__device__ __forceinline__ double pw_full_chunk(const Term& f) {
    const int lane = threadIdx.x & (ENM_WAVE - 1);
    const int j = lane & 7, g = lane >> 3;
    double part[8];
#pragma unroll
    for (int pass = 0; pass < 8; ++pass) {
        const int64_t base = (int64_t)(pass * 8 + g) * PW_LEAF + j;
        double v[PW_LEAF / 8];
#pragma unroll
        for (int i = 0; i < PW_LEAF / 8; ++i) v[i] = f(base + 8 * i);
        double acc = v[0];
#pragma unroll
        for (int i = 1; i < PW_LEAF / 8; ++i) acc += v[i];
        acc += __shfl_xor(acc, 1, ENM_WAVE);
        acc += __shfl_xor(acc, 2, ENM_WAVE);
        acc += __shfl_xor(acc, 4, ENM_WAVE);
        acc += __shfl_xor(acc, 8, ENM_WAVE);
        acc += __shfl_xor(acc, 16, ENM_WAVE);
        acc += __shfl_xor(acc, 32, ENM_WAVE);
        part[pass] = acc;
    }
    return ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
}

// LDS of one wave's sum.
struct PwTree {
    int lo[PW_HEAP], len[PW_HEAP];
    double val[PW_HEAP];
    short leaf[PW_HEAP];
    int nl;
};

// Orders a wave's own LDS accesses.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

// The pairwise sum of m <= PW_CHUNK values (pass 0) or squared deviations (pass
// 1) by one wave, in every lane.  A full chunk takes pw_full_chunk; otherwise the
// wave builds the recursion's tree in LDS level by level (slot lengths; -1 for no
// node), sums its leaves, eight lanes to a leaf, and adds every node's two halves
// bottom-up, left + right, as NumPy does.
template <bool FULL>   // whether m may be PW_CHUNK
__device__ double pw_chunk(const Term& f, int m, PwTree& L) {
    if (FULL && m == PW_CHUNK) return pw_full_chunk(f);
    const int lane = (int)threadIdx.x & (ENM_WAVE - 1);
    // The tree, top-down: slot 1 is the whole chunk; a slot's halves exist
    // when it has more than PW_LEAF values.
    for (int i = lane; i < PW_HEAP; i += ENM_WAVE) L.len[i] = -1;
    if (lane == 0) {
        L.lo[1] = 0;
        L.len[1] = m;
        L.nl = 0;
    }
    wave_sync();
    for (int d = 0; d < PW_DEPTH; ++d) {
        for (int i = (1 << d) + lane; i < (2 << d); i += ENM_WAVE) {
            const int len = L.len[i];
            if (len > PW_LEAF) {
                int n2 = len / 2;
                n2 -= n2 % 8;
                L.lo[2 * i] = L.lo[i];
                L.len[2 * i] = n2;
                L.lo[2 * i + 1] = L.lo[i] + n2;
                L.len[2 * i + 1] = len - n2;
            }
        }
        wave_sync();
    }
    // The leaves, listed in any order (each is summed on its own).
    for (int i = 1 + lane; i < PW_HEAP; i += ENM_WAVE) {
        const int len = L.len[i];
        if (len >= 0 && len <= PW_LEAF) L.leaf[atomicAdd(&L.nl, 1)] = (short)i;
    }
    wave_sync();
    // A leaf is NumPy's pairwise_sum leaf: fewer than 8 values summed from
    // 0.0; up to 128 by 8 interleaved accumulators combined as
    // ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)), the remainder added after.
    // Eight lanes per leaf, eight leaves per round: lane j of a group takes
    // accumulator j (its up to sixteen values loaded at once, added in
    // order), butterfly shuffles within the group combine the accumulators,
    // and the group's first lane adds the remainder.
    const int j = lane & 7;
    const int nl = L.nl;
    for (int l0 = 0; l0 < nl; l0 += ENM_WAVE / 8) {
        const int l = l0 + (lane >> 3);
        const int slot = l < nl ? L.leaf[l] : 0;
        const int lo = l < nl ? L.lo[slot] : 0, len = l < nl ? L.len[slot] : 0;
        const int full = len >= 8 ? len - len % 8 : 0;
        double v[PW_LEAF / 8];
#pragma unroll
        for (int i = 0; i < PW_LEAF / 8; ++i) v[i] = 8 * i < full ? f(lo + 8 * i + j) : 0.0;
        double acc = v[0];
#pragma unroll
        for (int i = 1; i < PW_LEAF / 8; ++i)
            if (8 * i < full) acc += v[i];
        acc += __shfl_xor(acc, 1, ENM_WAVE);
        acc += __shfl_xor(acc, 2, ENM_WAVE);
        acc += __shfl_xor(acc, 4, ENM_WAVE);
        if (j == 0 && l < nl) {
            double res;
            if (len < 8) {
                res = 0.0;
                for (int t = 0; t < len; ++t) res += f(lo + t);
            } else {
                res = acc;
                for (int t = full; t < len; ++t) res += f(lo + t);
            }
            L.val[slot] = res;
        }
    }
    wave_sync();
    // Bottom-up: every split node is its left half plus its right half.
    for (int d = PW_DEPTH - 1; d >= 0; --d) {
        for (int i = (1 << d) + lane; i < (2 << d); i += ENM_WAVE)
            if (L.len[i] > PW_LEAF) L.val[i] = L.val[2 * i] + L.val[2 * i + 1];
        wave_sync();
    }
    return L.val[1];
}

// Phase 2b: one wave per chunk of every array, four waves per block (no barriers:
// each wave sums its own chunk).
__global__ __launch_bounds__(4 * ENM_WAVE)
void prep_chunk_kernel(const PrepSumDev* __restrict__ sums, const int* __restrict__ chunk_sum_of,
                       const int* __restrict__ chunk_index, const int* __restrict__ list, int n_list,
                       const double* __restrict__ arena, const double* __restrict__ stats, int pass,
                       double* __restrict__ chunk_val) {
    __shared__ PwTree s_tree[4];
    const int wave = (int)(threadIdx.x / ENM_WAVE), idx = (int)blockIdx.x * 4 + wave;
    if (idx >= n_list) return;
    const int c = list[idx];
    const PrepSumDev& sd = sums[chunk_sum_of[c]];
    const int64_t first = (int64_t)chunk_index[c] * PW_CHUNK;
    const int m = (int)min((int64_t)PW_CHUNK, sd.n - first);
    const Term f{arena + sd.src + first, pass ? stats[sd.stat] : 0.0, pass != 0};
    const double sum = pw_chunk<true>(f, m, s_tree[wave]);
    if ((threadIdx.x & (ENM_WAVE - 1)) == 0) chunk_val[c] = sum;
}

// ---- Row-by-row sums -------------------------------------------------------
// The columns of a multi-column condition are summed one row after the other,
// each addition rounded: s' = RN(s + x).  As one chain of additions that takes
// 4.4 ns per row however wide the chip is (5.5 before a row was read by the
// addition itself; two passes over two million rows: 22 ms).  The same sum, bit
// for bit, in parallel:
//
// While |s| stays inside one binade, (2^e, 2^(e+1)), s is an integer S in units
// of u = 2^(e-52), and an addition adds x rounded to whole units: S' = S +
// rint(x / u), where S matters only if x / u lies exactly between two integers
// (a tie): then S' is the even one of the two around S + x / u.  So a run of
// rows adds an amount that depends on S by its parity alone; it is known before
// S is.  A TILE of 64 rows keeps, for the binade e that its predicted start
// lies in: the amount `add` for an even S, the change `odd` of it for an odd S
// (-1, 0 or 1), whether there was a tie (then S' is of the same parity for
// both), and the least and greatest sum inside it, so that whoever knows S can
// tell that no sum inside the tile leaves the binade.
//
// prep_seq_block_kernel: sums of blocks of 4096 rows, in any order, for the
// prediction.  prep_seq_tile_kernel: the tiles.  prep_finish_kernel: one wave
// per array takes 64 tiles at a time: every lane finds the S its tile starts
// with, and checks its tile; the tiles before the first that fails are done.
// That one's rows are added one by one (the start, where |s| is small; sums
// that cross a binade; mispredictions; anything not finite), and so on.  Tiles
// that the prediction expects to fail have their rows loaded ahead.
//
// Mean and deviation of two columns of 2,000,000 rows: 22.0 -> 2.5 ms, of
// 100,000: 1.10 -> 0.57.  What is left is the tiles that fail, at 0.4 us each:
// next to none in the sum of squares, and in a mean near 0, where the sum is a
// walk about 0, 4 to 14 % of two million rows and 10 to 45 % of 100,000.

constexpr int SEQ_THREADS = 256;
constexpr int SEQ_BLOCK = ENM_PREP_SEQ_BLOCK;             // rows per block
constexpr int SEQ_TILE = 64;                              // rows per tile
constexpr int SEQ_PER = SEQ_BLOCK / SEQ_THREADS;          // rows per thread
constexpr int SEQ_AHEAD = 32;                             // tiles of a block whose rows are loaded ahead
constexpr double SEQ_LO = 0x1p52, SEQ_HI = 0x1p53;        // |S|

constexpr int SEQ_EXP = 0x7ff, SEQ_BAD = 1 << 11, SEQ_TIE = 1 << 12, SEQ_ODD = 1 << 13, SEQ_SUSPECT = 1 << 14,
              SEQ_ZERO = 1 << 15;

__device__ __forceinline__ int exp_bits(double v) { return (int)((__double_as_longlong(v) >> 52) & 0x7ff); }

__device__ __forceinline__ double seq_term(double v, double mean, int pass) {
    if (!pass) return v;
    const double d = v - mean;
    return d * d;
}

// The parity of a whole number below 2^53.
__device__ __forceinline__ int parity(double v) { return (int)((long long)v & 1); }

// S, S + lo and S + hi inside the binade (`gap` units from its ends at least).
__device__ __forceinline__ bool inside(double S, double lo, double hi, double gap) {
    return S > 0.0 ? S + lo - gap > SEQ_LO && S + hi + gap < SEQ_HI : S + hi + gap < -SEQ_LO && S + lo - gap > -SEQ_HI;
}

// The sum of the lanes up to and with this one.
__device__ __forceinline__ double seq_scan(double v) {
    const int lane = threadIdx.x & (ENM_WAVE - 1);
    v += dpp_f64<DPP_SHR1>(0.0, v);
    v += dpp_f64<DPP_SHR2>(0.0, v);
    v += dpp_f64<DPP_SHR4>(0.0, v);
    v += dpp_f64<DPP_SHR8>(0.0, v);
    const double row = dpp_f64<DPP_BCAST15>(0.0, v);
    if (lane & 16) v += row;
    const double half = lane_f64(v, 31);
    return lane >= 32 ? v + half : v;
}

__device__ __forceinline__ double block_sum(double v, double* s_part) {
    v = lane_f64(seq_scan(v), ENM_WAVE - 1);
    __syncthreads();
    if ((threadIdx.x & (ENM_WAVE - 1)) == 0) s_part[threadIdx.x / ENM_WAVE] = v;
    __syncthreads();
    v = 0.0;
    for (int w = 0; w < SEQ_THREADS / ENM_WAVE; ++w) v += s_part[w];
    return v;
}

__global__ __launch_bounds__(SEQ_THREADS)
void prep_seq_block_kernel(const PrepSumDev* __restrict__ sums, const int* __restrict__ sum_of,
                           const double* __restrict__ arena, const double* __restrict__ stats, int pass,
                           double* __restrict__ block_val) {
    __shared__ double s_part[SEQ_THREADS / ENM_WAVE];
    const PrepSumDev& sd = sums[sum_of[blockIdx.x]];
    const int64_t first = (int64_t)((int)blockIdx.x - sd.chunk0) * SEQ_BLOCK;
    const double mean = pass ? stats[sd.stat] : 0.0;
    double v[SEQ_PER], sum = 0.0;
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j) {
        const int64_t i = first + j * SEQ_THREADS + threadIdx.x;
        v[j] = arena[sd.src + (i < sd.n ? i : sd.n - 1)];
    }
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j)
        sum += first + j * SEQ_THREADS + threadIdx.x < sd.n ? seq_term(v[j], mean, pass) : 0.0;
    sum = block_sum(sum, s_part);
    if (threadIdx.x == 0) block_val[blockIdx.x] = sum;
}

// What a run of rows does to S (see above).
struct SeqRun {
    double add, odd, lo, hi;
    bool tie;
};

// One run, then another.
__device__ __forceinline__ SeqRun seq_then(const SeqRun& f, const SeqRun& g) {
    const int p0 = parity(f.add), p1 = parity(1.0 + f.add + f.odd);
    SeqRun r;
    r.add = f.add + g.add + (p0 ? g.odd : 0.0);
    r.odd = (f.add + f.odd) + g.add + (p1 ? g.odd : 0.0) - r.add;
    r.lo = fmin(f.lo, f.add + g.lo);
    r.hi = fmax(f.hi, f.add + g.hi);
    r.tie = f.tie || g.tie;
    return r;
}

// Four threads per tile, 16 rows each.  Bound by its loads (8 bytes per row).
__global__ __launch_bounds__(SEQ_THREADS)
void prep_seq_tile_kernel(const PrepSumDev* __restrict__ sums, const int* __restrict__ sum_of,
                          const double* __restrict__ arena, const double* __restrict__ stats, int pass,
                          const double* __restrict__ block_val, PrepSeqTile* __restrict__ tiles) {
    __shared__ double s_part[SEQ_THREADS / ENM_WAVE];
    __shared__ double s_rows[SEQ_BLOCK + SEQ_THREADS];   // 16 rows, then one unused: no bank conflicts
    const PrepSumDev& sd = sums[sum_of[blockIdx.x]];
    const int block = (int)blockIdx.x - sd.chunk0;
    const int64_t first = (int64_t)block * SEQ_BLOCK;
    const double mean = pass ? stats[sd.stat] : 0.0;
    const int tid = threadIdx.x, lane = tid & (ENM_WAVE - 1);
    double v[SEQ_PER];
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j) {
        const int64_t i = first + j * SEQ_THREADS + tid;
        v[j] = arena[sd.src + (i < sd.n ? i : sd.n - 1)];
    }
    double before = 0.0;
    for (int b = tid; b < block; b += SEQ_THREADS) before += block_val[sd.chunk0 + b];
    before = block_sum(before, s_part);
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j) {
        const int i = j * SEQ_THREADS + tid;
        s_rows[i + i / SEQ_PER] = first + i < sd.n ? seq_term(v[j], mean, pass) : -0.0;
    }
    __syncthreads();
    const double* rows = s_rows + tid * (SEQ_PER + 1);
    double own = 0.0;
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j) own += rows[j];
    // The sum before this thread's rows.
    const double upto = seq_scan(own);
    __syncthreads();
    if (lane == ENM_WAVE - 1) s_part[tid / ENM_WAVE] = upto;
    __syncthreads();
    double start = before + (upto - own);
    for (int w = 0; w < tid / ENM_WAVE; ++w) start += s_part[w];
    start = __shfl(start, lane & ~3, ENM_WAVE);

    const int e = exp_bits(start);
    bool bad = e == 0 || e == 0x7ff, zero = true;
    SeqRun run{0.0, 0.0, 0.0, 0.0, false};
#pragma unroll
    for (int j = 0; j < SEQ_PER; ++j) {
        const double t = ldexp(rows[j], 1075 - e);
        const double r = rint(t);
        bad = bad || !(fabs(t) < SEQ_HI);
        zero = zero && rows[j] == 0.0;
        if (fabs(t - r) == 0.5) {
            const double q = floor(t);
            const double even = q + (parity(run.add + q) ? 1.0 : 0.0);
            const double odd = q + (parity(1.0 + run.add + run.odd + q) ? 1.0 : 0.0);
            run.add += even;
            run.odd += odd - even;
            run.tie = true;
        } else {
            run.add += r;
        }
        run.lo = fmin(run.lo, run.add);
        run.hi = fmax(run.hi, run.add);
        bad = bad || !(fabs(run.add) < SEQ_HI);   // also keeps the parities' arguments exact
        if (bad) run.add = run.odd = 0.0;
    }
    for (int d = 1; d <= 2; d <<= 1) {
        SeqRun o;
        o.add = __shfl_down(run.add, d, ENM_WAVE);
        o.odd = __shfl_down(run.odd, d, ENM_WAVE);
        o.lo = __shfl_down(run.lo, d, ENM_WAVE);
        o.hi = __shfl_down(run.hi, d, ENM_WAVE);
        o.tie = __shfl_down((int)run.tie, d, ENM_WAVE) != 0;
        bad = __shfl_down((int)bad, d, ENM_WAVE) != 0 || bad;
        zero = __shfl_down((int)zero, d, ENM_WAVE) != 0 && zero;
        run = seq_then(run, o);
    }
    bad = bad || !(run.lo > -SEQ_HI && run.hi < SEQ_HI);
    if (tid % 4 == 0) {
        PrepSeqTile T;
        T.add = bad ? 0.0 : run.add;
        T.lo = run.lo;
        T.hi = run.hi;
        T.odd = bad ? 0 : (int)run.odd;
        // The prediction is good to far less than 2^20 units.
        const bool suspect = bad || !inside(ldexp(start, 1075 - e), run.lo, run.hi, 0x1p20);
        T.bits = e | (bad ? SEQ_BAD : 0) | (run.tie ? SEQ_TIE : 0) | (parity(T.add) ? SEQ_ODD : 0) |
                 (suspect && !zero ? SEQ_SUSPECT : 0) | (zero ? SEQ_ZERO : 0);
        tiles[(int64_t)blockIdx.x * (SEQ_BLOCK / SEQ_TILE) + tid / 4] = T;
    }
}

// s plus the rows of one tile, one per lane, in order.  fma(row, 1, s) is s + row;
// as an fma it can read the row of another lane itself (one of its own 16), so
// nothing but the additions is on the chain (through a scalar register: 10.5 ns
// a row).
#define SEQ_ROW(k) "v_fmac_f64_dpp %0, %1, %2 row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n"
__device__ __forceinline__ double seq_add_rows(double s, double row) {
    const double one = 1.0;
#pragma unroll
    for (int r = 0; r < SEQ_TILE; r += 16) {
        // A register may be read by another lane two instructions after it is written.
        asm("s_nop 1\n" SEQ_ROW(0) SEQ_ROW(1) SEQ_ROW(2) SEQ_ROW(3) SEQ_ROW(4) SEQ_ROW(5) SEQ_ROW(6) SEQ_ROW(7)
            SEQ_ROW(8) SEQ_ROW(9) SEQ_ROW(10) SEQ_ROW(11) SEQ_ROW(12) SEQ_ROW(13) SEQ_ROW(14) SEQ_ROW(15)
            : "+v"(s) : "v"(row), "v"(one));
        s = lane_f64(s, r);
    }
    return s;
}
#undef SEQ_ROW

// Rows of tiles of one block that are expected to be added one by one.
struct SeqAhead {
    double v[SEQ_AHEAD];
    unsigned long long which;
};

__device__ __forceinline__ void seq_load_ahead(SeqAhead& a, const PrepSeqTile& T, const double* v, int64_t block,
                                               int64_t n) {
    a.which = __ballot((T.bits & SEQ_SUSPECT) != 0);
    unsigned long long m = a.which;
#pragma unroll
    for (int j = 0; j < SEQ_AHEAD; ++j) {
        if (!m) break;
        const int64_t i = block * SEQ_BLOCK + (int64_t)__builtin_ctzll(m) * SEQ_TILE + (threadIdx.x & (ENM_WAVE - 1));
        a.v[j] = v[i < n ? i : n - 1];
        m &= m - 1;
    }
}

// The row-by-row sum of one array from its tiles; one wave.
__device__ double seq_sum(const PrepSumDev& sd, const double* v, double mean, int pass,
                          const PrepSeqTile* __restrict__ tiles, double (*s_ahead)[ENM_WAVE]) {
    const int lane = threadIdx.x & (ENM_WAVE - 1);
    const int64_t n = sd.n;
    const int n_blocks = sd.n_chunks;
    const unsigned long long below = (1ull << lane) - 1;
    tiles += (int64_t)sd.chunk0 * ENM_WAVE + lane;
    PrepSeqTile T = tiles[0], next = tiles[n_blocks > 1 ? ENM_WAVE : 0];
    SeqAhead ahead;
    seq_load_ahead(ahead, T, v, 0, n);
    double s = -0.0;
    for (int b = 0; b < n_blocks; ++b) {
        const unsigned long long which = ahead.which;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < SEQ_AHEAD; ++j) s_ahead[j][lane] = ahead.v[j];
        __syncthreads();
        if (b + 1 < n_blocks) seq_load_ahead(ahead, next, v, b + 1, n);
        const PrepSeqTile later = tiles[(int64_t)(b + 2 < n_blocks ? b + 2 : b) * ENM_WAVE];

        const int n_tiles = (int)min((int64_t)ENM_WAVE, (n - (int64_t)b * SEQ_BLOCK + SEQ_TILE - 1) / SEQ_TILE);
        const unsigned long long ties = __ballot((T.bits & SEQ_TIE) != 0), odds = __ballot((T.bits & SEQ_ODD) != 0);
        for (int at = 0; at < n_tiles;) {
            const int e = exp_bits(s);
            const unsigned long long from = ~0ull << at;
            if ((which >> at) & 1) {
                // Expected to fail: nothing to be gained from a look at the others.
            } else if (e != 0 && e != 0x7ff) {
                const double S = ldexp(s, 1075 - e);
                const bool same = lane >= at && (T.bits & (SEQ_EXP | SEQ_BAD)) == e;
                // The parity of S where this lane's tile starts: that after
                // the last tile with a tie, turned by the odd ones since.
                const unsigned long long mine = from & below, t = ties & mine;
                unsigned long long turns = odds & mine;
                int odd = parity(S);
                if (t) {
                    const int j = 63 - __builtin_clzll(t);
                    turns &= ~0ull << j;
                    odd = 0;
                }
                odd ^= __builtin_popcountll(turns) & 1;
                const double add = same ? T.add + (odd ? (double)T.odd : 0.0) : 0.0;
                const double upto = seq_scan(add);
                // Three units: `odd` inside the tile, and what rounding to one does.
                const bool ok = same && inside(S + (upto - add), T.lo, T.hi, 3.0);
                const unsigned long long fails = ~__ballot(ok) & from;
                const int stop = min(n_tiles, fails ? __builtin_ctzll(fails) : ENM_WAVE);
                if (stop > at) {
                    s = ldexp(S + lane_f64(upto, stop - 1), e - 1075);
                    at = stop;
                    if (at == n_tiles) break;
                }
            } else if (__double_as_longlong(s) == 0) {
                // 0 stays 0 over rows of 0.
                const unsigned long long fails = ~__ballot((T.bits & SEQ_ZERO) != 0) & from;
                at = min(n_tiles, fails ? __builtin_ctzll(fails) : ENM_WAVE);
                if (at == n_tiles) break;
            }
            const int64_t i = (int64_t)b * SEQ_BLOCK + (int64_t)at * SEQ_TILE + lane;
            const int slot = __builtin_popcountll(which & ((1ull << at) - 1));   // (`at` has moved since `from`)
            const double x = ((which >> at) & 1) && slot < SEQ_AHEAD ? s_ahead[slot][lane] : v[i < n ? i : n - 1];
            s = seq_add_rows(s, i < n ? seq_term(x, mean, pass) : -0.0);
            ++at;
        }
        T = next;
        next = later;
    }
    return s;
}

// The row-by-row sum of one array as one chain; one wave.  64 rows at a time,
// the next 256 on their way.
__device__ double seq_chain(const double* v, int64_t n, double mean, int pass) {
    constexpr int AHEAD = 4;
    const int lane = threadIdx.x & (ENM_WAVE - 1);
    double acc = -0.0, rows[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) {
        const int64_t i = j * ENM_WAVE + lane;
        rows[j] = i < n ? v[i] : 0.0;
    }
    for (int64_t base = 0; base < n; base += AHEAD * ENM_WAVE) {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const int64_t i = base + j * ENM_WAVE + lane, k = i + AHEAD * ENM_WAVE;
            const double term = i < n ? seq_term(rows[j], mean, pass) : -0.0;
            rows[j] = k < n ? v[k] : 0.0;
            if (base + j * ENM_WAVE < n) acc = seq_add_rows(acc, term);
        }
    }
    return acc;
}

// Phase 2c: per array, the chunk sums added in order to -0.0 (pairwise
// arrays), or the whole column accumulated row by row (columns of a
// multi-column condition; from its tiles if it has any); then mean = sum / n
// (pass 0) or std = sqrt(sum / n) (pass 1).  One wave per array.  A row-by-row
// sum starts at -0.0, which leaves the first row's term unchanged
// (x + -0.0 == x for every x), as a sum that starts from the first row does.
__global__ __launch_bounds__(ENM_WAVE)
void prep_finish_kernel(const PrepSumDev* __restrict__ sums, int n_sums, const double* __restrict__ arena,
                        const double* __restrict__ chunk_val, const PrepSeqTile* __restrict__ tiles, int pass,
                        double* __restrict__ stats) {
    __shared__ double s_ahead[SEQ_AHEAD][ENM_WAVE];
    const int s = blockIdx.x;
    if (s >= n_sums) return;
    const PrepSumDev& sd = sums[s];
    const int lane = threadIdx.x;
    double acc = -0.0;
    if (sd.sequential) {
        const double* v = arena + sd.src;
        const double mean = pass ? stats[sd.stat] : 0.0;
        if (sd.n_chunks > 0) {
            acc = seq_sum(sd, v, mean, pass, tiles, s_ahead);
        } else {
            acc = seq_chain(v, sd.n, mean, pass);
        }
    } else {
        for (int c = 0; c < sd.n_chunks; ++c) acc += chunk_val[sd.chunk0 + c];
    }
    if (lane != 0) return;
    const double q = acc / (double)sd.n;
    if (pass == 0) stats[sd.stat] = q;
    else stats[sd.stat + 1] = sqrt(q);
}

// Which variables of a task are rescaled, where their noise starts, and its
// flag bits (bit 0 x, bit 1 y, bit 2 z constant), which are returned.
// Variables of raw_vars (bit 0 x, bit 1 y) are class labels: never rescaled, no
// noise drawn, not called constant.
__device__ __forceinline__ unsigned place_noise(PrepTaskDev& t, const double* stats, unsigned raw_vars) {
    unsigned fl = 0;
    if (!(raw_vars & 1u) && fabs(stats[t.stat + 1]) < 1e-20) fl |= 1u;
    if (!(raw_vars & 2u) && fabs(stats[t.stat + 3]) < 1e-20) fl |= 2u;
    for (int c = 0; c < t.dz; ++c)
        if (fabs(stats[t.stat + 4 + 2 * c + 1]) < 1e-20) fl |= 4u;
    const unsigned constant = fl;
    fl |= raw_vars;
    int64_t drawn = 0;
    t.noise_x = drawn;
    if (!(fl & 1u)) drawn += t.n;
    t.noise_y = drawn;
    if (!(fl & 2u)) drawn += t.n;
    t.noise_z = drawn;
    t.flags = fl;
    return constant;
}

// (v - mean) / std + noise for row i of every rescaled variable, in place.
__device__ __forceinline__ void scale_row(const PrepTaskDev& t, int64_t i, const double* stats,
                                          const double* __restrict__ noise, double* arena) {
    double* col = arena + t.arena_off;
    if (!(t.flags & 1u)) {
        const double v = (col[i] - stats[t.stat]) / stats[t.stat + 1];
        col[i] = v + noise[t.noise_x + i];
    }
    if (!(t.flags & 2u)) {
        const double v = (col[t.n + i] - stats[t.stat + 2]) / stats[t.stat + 3];
        col[t.n + i] = v + noise[t.noise_y + i];
    }
    if (!(t.flags & 4u)) {
        for (int c = 0; c < t.dz; ++c) {
            const double mean = stats[t.stat + 4 + 2 * c], sd = stats[t.stat + 5 + 2 * c];
            const double v = (col[(2 + c) * t.n + i] - mean) / sd;
            col[(2 + c) * t.n + i] = v + noise[t.noise_z + i * t.dz + c];
        }
    }
}

// Phase 2d.  One thread per task.
__global__ void prep_noise_kernel(PrepTaskDev* __restrict__ tasks, int n_tasks, const double* __restrict__ stats,
                                  unsigned raw_vars, unsigned* __restrict__ const_flag) {
    const int ti = blockIdx.x * blockDim.x + threadIdx.x;
    if (ti >= n_tasks) return;
    const_flag[ti] = place_noise(tasks[ti], stats, raw_vars);
}

// Phase 2e.
__global__ __launch_bounds__(PB_THREADS)
void prep_scale_kernel(const PrepTaskDev* __restrict__ tasks, int64_t stride, const double* __restrict__ stats,
                       const double* __restrict__ noise, double* __restrict__ arena) {
    const int64_t b = xcd_block(blockIdx.x, gridDim.x);   // a task's blocks on one XCD
    const int ti = (int)(b / stride);
    const PrepTaskDev& t = tasks[ti];   // read in place: a copy indexed by c would sit in scratch
    const int64_t i = (b - ti * stride) * PB_THREADS + threadIdx.x;
    if (i < t.n) scale_row(t, i, stats, noise, arena);
}

// Phase 2 of short tasks (at most PREP_SHORT kept rows each), one workgroup per
// task: every array's mean and deviation by a wave of its own, then the
// rescaling.  Bound by latency and launches: for a few short tasks the phases
// take some 5 us each, mostly to be launched.  (36 tasks of 2,500 rows 37 us, in
// phases 32 and five launches more; of 8,000 rows 117 and 40.)  With `whole` (windows of one block
// of rows) it does the compaction too.
__global__ __launch_bounds__(PB_THREADS)
void prep_short_kernel(PrepTaskDev* tasks, const double* __restrict__ raw, const unsigned char* __restrict__ mask,
                       int drop_nan, int whole, double* stats, const double* __restrict__ noise, unsigned raw_vars,
                       unsigned* __restrict__ const_flag, double* arena, KeptWord* __restrict__ kept) {
    constexpr int NW = PB_THREADS / ENM_WAVE;
    __shared__ PwTree s_tree[NW];
    PrepTaskDev& t = tasks[blockIdx.x];
    const int lane = threadIdx.x & (ENM_WAVE - 1), wave = threadIdx.x / ENM_WAVE;
    if (whole) {
        compact_rows(t, 0, 0, raw, mask, drop_nan, arena, kept);
        __syncthreads();
    }
    for (int a = wave; a < 2 + t.dz; a += NW) {
        if (a < 2 && ((raw_vars >> a) & 1u)) continue;
        const double* v = arena + t.arena_off + a * t.n;
        double mean = 0.0;
        for (int pass = 0; pass < 2; ++pass) {
            const double sum = a >= 2 && t.dz >= 2 ? seq_chain(v, t.n, mean, pass)
                                                   : -0.0 + pw_chunk<false>(Term{v, mean, pass != 0}, (int)t.n, s_tree[wave]);
            const double q = sum / (double)t.n;
            if (pass == 0) mean = q;
            if (lane == 0) stats[t.stat + 2 * a + pass] = pass ? sqrt(q) : q;
            wave_sync();
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) const_flag[blockIdx.x] = place_noise(t, stats, raw_vars);
    __syncthreads();
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < t.n; i += PB_THREADS) scale_row(t, i, stats, noise, arena);
}

}  // namespace

hipError_t enm_launch_prep_columns(const double* rows, int64_t n, int m, double* cols, hipStream_t st) {
    const dim3 grid((unsigned)((n + PC_TILE - 1) / PC_TILE), (unsigned)((m + PC_TILE - 1) / PC_TILE));
    hipLaunchKernelGGL(prep_columns_kernel, grid, dim3(PC_THREADS), 0, st, rows, n, m, cols);
    return hipGetLastError();
}

hipError_t enm_launch_prep_count(const PrepTaskDev* tasks, int64_t stride, int n_tasks,
                                 const double* raw, const unsigned char* mask, int drop_nan, int* blk_count,
                                 int64_t* blk_off, unsigned* nan_flag, PrepCounted* out, hipStream_t st) {
    const int64_t n_blocks = stride * n_tasks;
    if (n_tasks <= 0) return hipSuccess;
    if (n_blocks > 0)
        hipLaunchKernelGGL(prep_count_kernel, dim3((unsigned)n_blocks), dim3(PB_THREADS), 0, st, tasks, stride,
                           raw, mask, drop_nan, blk_count, nan_flag, blk_off, out);
    if (stride != 1)
        hipLaunchKernelGGL(prep_scan_kernel, dim3((unsigned)n_tasks), dim3(ENM_WAVE), 0, st, tasks, stride, n_tasks,
                       blk_count, blk_off, nan_flag, out);
    return hipGetLastError();
}

hipError_t enm_launch_prep_write(PrepTaskDev* tasks, int64_t stride, int n_tasks,
                                 const double* raw, const unsigned char* mask, int drop_nan, int rescale,
                                 const int64_t* blk_off, const PrepSumDev* sums, int n_sums,
                                 const int* chunk_sum_of, const int* chunk_index, const int* chunk_list,
                                 int n_chunks, double* chunk_val, const int* seq_sum_of, int n_seq,
                                 double* seq_val, PrepSeqTile* seq_tiles, double* stats, int64_t sstride,
                                 const double* noise, unsigned raw_vars, unsigned* const_flag, double* arena,
                                 KeptWord* kept, hipStream_t st) {
    if (n_tasks <= 0) return hipSuccess;
    const int64_t n_blocks = stride * n_tasks, n_sblocks = sstride * n_tasks;
    static_assert(ENM_PREP_SHORT < PW_CHUNK, "a short task's sums are of less than a chunk");
    const bool short_tasks = rescale && sstride * PB_THREADS <= ENM_PREP_SHORT;
    const bool whole = short_tasks && stride == 1;
    if (n_blocks > 0 && !whole)
        hipLaunchKernelGGL(prep_compact_kernel, dim3((unsigned)n_blocks), dim3(PB_THREADS), 0, st, tasks, stride,
                           raw, mask, drop_nan, blk_off, arena, kept);
    if (short_tasks)
        hipLaunchKernelGGL(prep_short_kernel, dim3((unsigned)n_tasks), dim3(PB_THREADS), 0, st, tasks, raw, mask,
                           drop_nan, whole ? 1 : 0, stats, noise, raw_vars, const_flag, arena, kept);
    if (!rescale || short_tasks) return hipGetLastError();
    for (int pass = 0; pass < 2; ++pass) {
        if (n_chunks > 0) {
            hipLaunchKernelGGL(prep_chunk_kernel, dim3((unsigned)((n_chunks + 3) / 4)), dim3(4 * ENM_WAVE), 0, st,
                               sums, chunk_sum_of, chunk_index, chunk_list, n_chunks, arena, stats, pass,
                               chunk_val);
        }
        if (n_seq > 0) {
            hipLaunchKernelGGL(prep_seq_block_kernel, dim3((unsigned)n_seq), dim3(SEQ_THREADS), 0, st, sums,
                               seq_sum_of, arena, stats, pass, seq_val);
            hipLaunchKernelGGL(prep_seq_tile_kernel, dim3((unsigned)n_seq), dim3(SEQ_THREADS), 0, st, sums,
                               seq_sum_of, arena, stats, pass, seq_val, seq_tiles);
        }
        hipLaunchKernelGGL(prep_finish_kernel, dim3((unsigned)n_sums), dim3(ENM_WAVE), 0, st, sums, n_sums, arena,
                           chunk_val, seq_tiles, pass, stats);
    }
    hipLaunchKernelGGL(prep_noise_kernel, dim3((unsigned)((n_tasks + 63) / 64)), dim3(64), 0, st, tasks, n_tasks,
                       stats, raw_vars, const_flag);
    if (n_sblocks > 0)
        hipLaunchKernelGGL(prep_scale_kernel, dim3((unsigned)n_sblocks), dim3(PB_THREADS), 0, st, tasks, sstride,
                           stats, noise, arena);
    return hipGetLastError();
}
