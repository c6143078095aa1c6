// Norm-cost (l1 / linf / l2) pricing scan on VALU for gfx950.
//
// Semantics (pricing.cu:65-161 VALU scan, cost.cu:10-85 direct_norm tiles, matrix_selection.cuh:20-26):
//   c_ij = fp32 distance; features are combined sequentially inside 32-feature chunks and the chunk results
//          are then combined in order (l1: sum |x-y|, linf: max |x-y|, l2: sqrtf(sum fmaf(z, z, .))),
//   sigma_ij = (g_j - (double)c_ij) + f_i   (fp64).
// Every value is reproduced bit for bit, so the per-row lists hold exact fp64 scores: an fp32 estimate of
// sigma with a rigorous slack only decides whether a pair needs its fp64 score.
//
// One thread owns one or two X rows (features in registers up to d = 128); a Y row is the same for the whole wave, so
// its features are scalar loads and enter the vector instructions as scalar operands. Per pair the loop computes the
// cost and one test against the lowest of the row's, the column's and the certificate's thresholds; what passes (a few
// pairs in a thousand) is handled out of line, with the row lists in LDS (long ones in memory, see norm_plan). The certificate adds the squares of violated
// scores in fp64 and those of all costs in fp32, flushed to fp64 per tile or more often (cost_span).
//
// Column lists, k <= 2 with rows and columns requested: they ride on the row sweep, so every pair is evaluated
// once. Every column keeps its running top-2 values in global memory (the largest and second largest score
// inserted so far, two atomic maxima: inserting v raises the first to max(v, first) and the second to
// min(v, previous first)); the running k-th value is a lower bound of the column's true k-th value. The tile's columns
// have their fp32 entry thresholds in LDS beside their duals, and the workgroup's own top-k values of each; a pair that
// beats its column's threshold enters the own values (LDS atomics), raises the threshold, and is appended to a
// candidate buffer when at or above the own k-th value. After the tile each thread inserts one column's own values into
// the running ones: the global atomics of 256 columns overlap, where a wave that inserted each pair as it met it waited
// for one chain of atomics after another. Workgroups start their Y sweep at staggered tiles, so most workgroups reach a
// column after its running values are set. The buffer's candidates at or above their column's final k-th value are then
// grouped by column (counting sort) and each column keeps its k best. Should the buffer overflow, the column lists come
// from the role-swapped sweep instead (the same launches, gated on the overflow count).
// Otherwise, column lists come from a second sweep with the roles swapped (the score keeps the original
// association).
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"

namespace hm {
namespace {

constexpr int NB_ROWS = 256;   // X rows per workgroup of the fp64 sweep (one per thread)
constexpr int NT = 256;        // Y rows per tile of the sweeps' segments
constexpr int LDS_FLOATS = 15872;  // fp64 sweep: 62 KiB of dynamic LDS, leaving room for the static reduction buffer

// one appended column candidate of the fused sweep
struct ColCand {
    int j;     // column
    int i;     // row
    double v;  // exact fp64 score
};

// column state of the fused sweep (all per call, in the workspace)
struct ColArgs {
    unsigned long long* gthr;   // per column: double_key of the largest (gthr[j]) and second largest (gthr[n + j])
                                // values inserted so far
    ColCand* buf;               // appended candidates (capacity cap)
    unsigned long long* count;  // reserved slots; above cap means the buffer overflowed
    int* ccount;                // per column: candidates stored in the buffer (n + 1, last 0)
    int* coff;                  // exclusive scan of ccount (n + 1)
    int* order;                 // buffer slots grouped by column
    const unsigned long long* xmaxima;  // [max ||x||_1, max |f|] of the row side (the column slack)
    const unsigned int* seeds;          // the columns' entry floors (norm_seed), or none
    int64_t cap;
    int64_t n;
};

// the running k-th value of column j (k <= 2): a lower bound of the column's k-th best score
__device__ inline double running_kth(const ColArgs& ca, int64_t j, int k) {
    return key_double(__hip_atomic_load(ca.gthr + (k == 1 ? j : ca.n + j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// insert a score (its key) into column j's running top-2 values
__device__ inline void running_insert(const ColArgs& ca, int64_t j, unsigned long long kv) {
    const unsigned long long o1 = atomicMax(ca.gthr + j, kv);
    const unsigned long long lo = kv < o1 ? kv : o1;
    if (lo != double_key(-INFINITY)) atomicMax(ca.gthr + ca.n + j, lo);
}

// the fused sweep's candidate capacity: each column receives its first workgroup's k entries and, after that,
// the entries that beat its threshold when their workgroup reaches it
inline int64_t fused_cap(int64_t n, int k) { return 16 * n * k + 65536; }

// buffer slots a wave reserves at a time: one atomic on the shared count per CHUNK appends, or per append of more. (A
// wave's unused slots are marked empty when its run ends; 64 at a time, thousands of waves of a tall problem filled the
// buffer with them.)
constexpr int CHUNK = 16;

// a wave's current run of reserved buffer slots (uniform over the wave)
struct SlotRun {
    int64_t base = -1;  // first slot; -1: none yet
    int size = 0, used = 0;
};

template <int KIND>
__device__ inline float feature_op(float part, float z) {
    if (KIND == HM_COST_L1) return part + fabsf(z);
    if (KIND == HM_COST_LINF) return fmaxf(part, fabsf(z));
    return fmaf(z, z, part);
}

// Y features are uniform over the wave: read through constant-address pointers they are scalar loads (rows need only
// 4-byte alignment) and enter the VALU as scalar operands, so a column costs neither LDS bandwidth nor vector loads.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x8u __attribute__((ext_vector_type(8), aligned(4)));
typedef const float __attribute__((address_space(4))) * ScalarRow;
typedef const f32x4u __attribute__((address_space(4))) * ScalarRow4;
typedef const f32x8u __attribute__((address_space(4))) * ScalarRow8;

__device__ __forceinline__ ScalarRow scalar_row(const float* p) { return (ScalarRow)(uintptr_t)p; }

// register widths: rows of d features take the smallest of these that holds them; a sweep at width DR knows that its
// rows have more than below(DR) features
constexpr int below(int dr) {
    return dr == 4 ? 0 : dr == 8 ? 4 : dr == 16 ? 8 : dr == 24 ? 16 : dr == 32 ? 24 : dr == 48 ? 32 : dr == 64 ? 48
           : dr == 96 ? 64 : 96;
}
constexpr int PAD = 32;  // readable floats after every row of a scalar-loaded side (SweepSide): at most DR - d are used

// W features of a Y row from `base` on, read whole (the row is followed by PAD readable floats)
template <int W>
__device__ __forceinline__ void scalar_features(float (&y)[W], ScalarRow row, int base) {
    if constexpr (W == 8) {
        const f32x8u v = *(ScalarRow8)(row + base);
#pragma unroll
        for (int t = 0; t < W; ++t) y[t] = v[t];
    } else {
        const f32x4u v = *(ScalarRow4)(row + base);
#pragma unroll
        for (int t = 0; t < W; ++t) y[t] = v[t];
    }
}

// Accumulated differences (l2: the squared distance) of J Y rows and R register rows of at most DR features: 32-feature
// chunks accumulated sequentially, chunk results combined in order. A chunk's scalar loads go out together, then its
// products run: one wait per up to 32 features of J rows. TAIL: d is not a whole number of feature groups; features at
// or past d read as 0 (x is padded with 0 there, and a zero difference leaves every partial result as it is, bit for
// bit); groups past d are skipped.
template <int KIND, int DR, int R, int J, bool TAIL>
__device__ __forceinline__ void accumulate_reg(const float (&x)[R][DR], const ScalarRow (&y)[J], int d,
                                               float (&acc)[J][R]) {
    constexpr int W = DR < 8 ? DR : 8;
#pragma unroll
    for (int base = 0; base < DR; base += 32) {
        constexpr int NG = (DR < 32 ? DR : 32) / W;  // groups of a whole chunk
        float yv[NG][J][W], part[J][R];
#pragma unroll
        for (int g = 0; g < NG; ++g)
            if (base + g * W < DR)
#pragma unroll
                for (int u = 0; u < J; ++u) scalar_features<W>(yv[g][u], y[u], base + g * W);
#pragma unroll
        for (int u = 0; u < J; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r) part[u][r] = 0.0f;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int f = base + g * W;  // (a constant once unrolled)
            if (f < DR && (f <= below(DR) || f < d)) {
#pragma unroll
                for (int t = 0; t < W; ++t)
#pragma unroll
                    for (int u = 0; u < J; ++u) {
                        float yt = yv[g][u][t];
                        if (TAIL && f + W > below(DR)) yt = __int_as_float(__float_as_int(yt) & (f + t < d ? -1 : 0));
#pragma unroll
                        for (int r = 0; r < R; ++r) part[u][r] = feature_op<KIND>(part[u][r], x[r][f + t < DR ? f + t : 0] - yt);
                    }
            }
        }
#pragma unroll
        for (int u = 0; u < J; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)  // (0 + part has part's bits: part is never -0)
                acc[u][r] = base == 0 ? part[u][r]
                                      : (KIND == HM_COST_LINF) ? fmaxf(acc[u][r], part[u][r]) : acc[u][r] + part[u][r];
    }
}

// the same for any d, one X row streamed from memory 32 features at a time against J Y rows
template <int KIND, int J>
__device__ __forceinline__ void accumulate_mem(const float* __restrict__ x, const ScalarRow (&y)[J], int d,
                                               float (&acc)[J][1]) {
#pragma unroll
    for (int u = 0; u < J; ++u) acc[u][0] = 0.0f;
    for (int base = 0; base < d; base += 32) {
        float xv[32], part[J];
        if (base + 32 <= d) {
#pragma unroll
            for (int t = 0; t < 32; t += 4) {
                const f32x4u v = *reinterpret_cast<const f32x4u*>(x + base + t);
                xv[t] = v.x;
                xv[t + 1] = v.y;
                xv[t + 2] = v.z;
                xv[t + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int t = 0; t < 32; ++t) xv[t] = base + t < d ? x[base + t] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < J; ++u) part[u] = 0.0f;
#pragma unroll
        for (int g = 0; g < 32; g += 8) {
            if (base + g < d) {
#pragma unroll
                for (int u = 0; u < J; ++u) {
                    float yv[8];
                    if (base + g + 8 <= d) {
                        scalar_features<8>(yv, y[u], base + g);
                    } else {  // nothing past the row is read
#pragma unroll
                        for (int t = 0; t < 8; ++t) {
                            const float v = y[u][base + g + t < d ? base + g + t : d - 1];
                            yv[t] = base + g + t < d ? v : 0.0f;
                        }
                    }
#pragma unroll
                    for (int t = 0; t < 8; ++t) part[u] = feature_op<KIND>(part[u], xv[g + t] - yv[t]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < J; ++u)
            acc[u][0] = (KIND == HM_COST_LINF) ? fmaxf(acc[u][0], part[u]) : acc[u][0] + part[u];
    }
}

// the cost of an accumulated difference; l2: the correctly rounded square root (fp64, rounded once)
template <int KIND>
__device__ __forceinline__ float cost_of(float acc) {
    return (KIND == HM_COST_L2) ? (float)sqrt((double)acc) : acc;
}

// maxima[0] = max ||y||_1, maxima[1] = max |g| (ordered keys): reduced per wave, one atomic each
__global__ __launch_bounds__(256) void norm_prep(const float* __restrict__ Y, int64_t n, int d,
                                                 const double* __restrict__ g,
                                                 unsigned long long* __restrict__ maxima) {
    double s = 0.0, gm = 0.0;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
        double a = 0.0;
        for (int k = 0; k < d; ++k) a += fabs((double)Y[j * d + k]);
        s = fmax(s, a);
        gm = fmax(gm, fabs(g[j]));
    }
    for (int o = 32; o >= 1; o >>= 1) {
        s = fmax(s, __shfl_xor(s, o, 64));
        gm = fmax(gm, __shfl_xor(gm, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMax(&maxima[0], double_key(s));
        atomicMax(&maxima[1], double_key(gm));
    }
}

inline unsigned prep_blocks(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return (unsigned)(b < 512 ? b : 512);
}

// the fp32 entry threshold of a column whose running k-th value is kth: any pair whose fp32 score is at or below
// it has an exact score below kth (one ulp down keeps it strictly below kth - slack). A slack that is not finite (a dual
// that is infinite, or whose slack is beyond fp32) leaves none: inf - inf would be a threshold that nothing passes.
__device__ inline float column_threshold(double kth, float cslack) {
    return (kth == -INFINITY || !(cslack < INFINITY)) ? -INFINITY : nextafterf((float)(kth - (double)cslack), -INFINITY);
}

// marks the unused slots of the wave's run empty (every lane of the wave calls it)
__device__ inline void slot_run_close(const ColArgs& ca, const SlotRun& run) {
    if (run.base < 0 || run.base + run.size > ca.cap) return;
    for (int e = run.used + (int)(threadIdx.x & 63); e < run.size; e += 64) ca.buf[run.base + e].j = -1;
}

// lanes with `app` append (j, row, v) to the buffer through the wave's run of slots (every lane calls it)
__device__ inline void column_append(const ColArgs& ca, SlotRun& run, bool app, int64_t j, int row, double v) {
    const unsigned long long am = __ballot(app);
    if (!am) return;
    const int na = __popcll(am);
    if (run.used + na > run.size) {
        slot_run_close(ca, run);
        run.size = na > CHUNK ? na : CHUNK;
        unsigned long long b = 0;
        if ((threadIdx.x & 63) == 0) b = atomicAdd(ca.count, (unsigned long long)run.size);
        run.base = (int64_t)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32)) << 32) |
                             (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b));
        run.used = 0;
    }
    if (app && run.base + run.size <= ca.cap) {  // a run past the capacity: the buffer overflowed
        const int rank = __popcll(am & ((1ull << (threadIdx.x & 63)) - 1ull));
        ColCand cc;
        cc.j = (int)j;
        cc.i = row;
        cc.v = v;
        ca.buf[run.base + run.used + rank] = cc;
    }
    run.used += na;
}

// A sweep's tile of Y rows in LDS: the column's dual in fp32 and, in a fused sweep, its fp32 entry threshold.
struct TileCol {
    float g;
    float thr;
};

// Lanes with `pass` (score sig of row `row`) beat the threshold of column j: they enter the workgroup's own top-2 values
// own1 / own2 of the column (keys in LDS; k = 1 leaves own2), those at or above the own k-th value are appended, and the
// column's threshold rises with it. Every lane of the wave calls it.
__device__ __forceinline__ void column_enter(const ColArgs& ca, SlotRun& run, bool pass, int64_t j, double sig, int row,
                                             int k, unsigned long long* own1, unsigned long long* own2, float* thr,
                                             float cslack) {
    const unsigned long long kv = double_key(sig);
    if (pass) {
        const unsigned long long o = atomicMax(own1, kv);
        if (k > 1) atomicMax(own2, kv < o ? kv : o);
    }
    const unsigned long long kth =
        __hip_atomic_load(k > 1 ? own2 : own1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const double own = key_double(kth);  // (compared as values: -0 and 0 tie)
    column_append(ca, run, pass && sig >= own, j, row, sig);
    // (any value up to the column's final k-th one is a valid bound, whichever wave writes last)
    const float t = column_threshold(own, cslack);
    if ((threadIdx.x & 63) == 0 && t > *thr) *thr = t;
}

// dynamic LDS of a sweep workgroup of T threads, R rows each, lists of k entries there; fused sweeps add the columns' own
// values
inline size_t sweep_lds(int T, int R, int k, bool fused) {
    return (size_t)R * T * (sizeof(double) + 3 * sizeof(float) + (size_t)k * (sizeof(double) + sizeof(int))) +
           (size_t)(NT + 8) * sizeof(TileCol) + (fused ? 2 * NT * sizeof(unsigned long long) : 0);
}

// The Y side of a sweep. At up to 128 features they are read in groups up to the register width, past the end of a row:
// rows from `tail_row` on (the last one or two tiles, where that could be past the end of Y) are read from `tail`, a
// copy of them with PAD floats of padding. (Longer rows: no copy, tail_row = n.)
struct SweepSide {
    const float* Y;
    const float* tail;
    int64_t tail_row;
};

constexpr int REG_FEATURES = 128;  // longest rows kept in registers
inline int64_t tail_start(int64_t n, int d) {
    if (d > REG_FEATURES) return n;
    const int64_t last = (n - 1) / NT * NT;
    return last >= NT ? last - NT : 0;
}
inline size_t tail_floats(int64_t n, int d) { return d > REG_FEATURES ? 1 : (size_t)(n - tail_start(n, d)) * d + PAD; }

__global__ __launch_bounds__(256) void norm_tail(const float* __restrict__ Y, int64_t first, int64_t count,
                                                 float* __restrict__ out) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < count + PAD; e += (int64_t)gridDim.x * blockDim.x)
        out[e] = e < count ? Y[first + e] : 0.0f;
}

// Y rows per step of a sweep: two while their features fit the scalar registers, eight per read of a streamed row
constexpr int step_columns(int dr) { return dr == 0 ? 8 : dr <= 32 ? 2 : 1; }

// waves per SIMD the register allocation aims at (rows of dr features, r of them per thread): the out-of-line part then
// spills rather than take waves from the pair loop
constexpr int sweep_waves(int dr, int r) {
    return dr == 0 ? 3 : dr * r <= 32 ? 5 : dr * r <= 64 ? 4 : 3;
}

// squared costs added up in fp32 before they go to the fp64 sum (0: each goes there): a chain of L rounds by up to L / 2
// units of 2^-24. A tile where a pair is cheap; 32 for wider rows, where the flush is lost in the pairs' work (as is one
// fp64 operation a pair for streamed rows).
constexpr int cost_span(int dr) { return dr == 0 ? 0 : dr <= 48 ? NT : 32; }

// Entry floors of the row lists, before the sweep: the k-th best score of a row is at least the smallest of k maxima over
// disjoint samples of its columns. Sample q of `samples` (grid y) takes every samples-th of `count` columns spread over
// the side and raises seeds[(q % k) * m + row] (an ordered key) to its largest fp32 score. Without floors every segment
// of every row list starts by taking in nearly all it sees, one out-of-line insertion after another.
template <int KIND, int DR, bool TAIL>
__global__ __launch_bounds__(256) void norm_seed(const float* __restrict__ X, SweepSide side, int64_t m, int64_t n,
                                                 int d, const double* __restrict__ rb, const double* __restrict__ cb,
                                                 int k, int count, int samples, unsigned int* __restrict__ seeds) {
    constexpr int J = step_columns(DR);
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool ok = row < m;
    float x[1][DR > 0 ? DR : 1];
    if constexpr (DR > 0) {
#pragma unroll
        for (int t = 0; t < DR; ++t) x[0][t] = (ok && t < d) ? X[row * d + t] : 0.0f;
    }
    float top = -INFINITY;
    for (int t = blockIdx.y; t < count; t += samples * J) {
        ScalarRow y[J];
        float g[J], acc[J][1];
#pragma unroll
        for (int u = 0; u < J; ++u) {
            const int tu = t + u * samples < count ? t + u * samples : t;  // (past the sample: the first again)
            const int64_t j = (int64_t)tu * n / count;
            y[u] = scalar_row(j >= side.tail_row ? side.tail + (j - side.tail_row) * d : side.Y + j * d);
            g[u] = (float)cb[j];
        }
        if constexpr (DR > 0) accumulate_reg<KIND, DR, 1, J, TAIL>(x, y, d, acc);
        else accumulate_mem<KIND, J>(X + (ok ? row : 0) * d, y, d, acc);
#pragma unroll
        for (int u = 0; u < J; ++u)
            top = fmaxf(top, g[u] - (KIND == HM_COST_L2 ? __builtin_amdgcn_sqrtf(acc[u][0]) : acc[u][0]));
    }
    if (ok) atomicMax(&seeds[(int64_t)(blockIdx.y % k) * m + row], float_key(top + (float)rb[row]));
}

// The threshold a row's seeds give: fp32 scores at or below it belong to pairs whose exact score is below the row's k-th
// best. A seed is within slack of an exact score (l2: within 1.5 of them, its square root being off by one unit in the
// last place, and by up to 2^-63 where the instruction takes a denormal square for 0), and a pair's fp32 score within slack
// of its exact one. None for a slack that is not finite (column_threshold).
template <int KIND>
__device__ __forceinline__ float seed_threshold(const unsigned int* __restrict__ seeds, int64_t m, int64_t row, int k,
                                                float slack) {
    unsigned int lo = 0xffffffffu;
    for (int q = 0; q < k; ++q) {
        const unsigned int s = seeds[(int64_t)q * m + row];
        lo = s < lo ? s : lo;
    }
    const float v = key_float(lo);
    const double off = 2.5 * (double)slack + (KIND == HM_COST_L2 ? 1.0842021724855044e-19 : 0.0);
    return v > -INFINITY && slack < INFINITY ? nextafterf((float)((double)v - off), -INFINITY) : -INFINITY;
}

// Bound: fp32 VALU (two operations per feature and pair; l1 at d = 8: 16 of about 23 instructions per pair). So the
// loop holds nothing else it can avoid: Y features are scalar operands, the row's, the column's and the certificate's
// tests are one compare against their lowest threshold (a wave vote sends the rest out of line), lists and fp64 duals
// live in LDS, which leaves the registers to the features (R rows of DR) and the waves in flight.
// l2 compares squared: a pair can matter when c <= B = g + f - T, decided as acc <= B|B| without a square root per
// pair; the rounding of B (3 u (|g| + |f|) + u |T|) and of the square is within the slack that T carries. Its
// certificate takes sum c^2 from acc and max c as the root of the largest acc.
// DR: register features (d <= DR, padded with zeros; 0: rows streamed from memory). TAIL: d is not a multiple of 8 (of
// 4 at DR = 4). R rows per thread share each Y row.
// FUSED (k <= 2, rows and columns): column lists as described at the top of this file; tiles start staggered.
// ST: certificate sums. gate: the role-swapped column sweep of a fused call runs only when the fused buffer
// overflowed (*gate > cap).
// Measured, whole calls with k = 2, rows, columns and certificate, before (features in LDS, one row per thread held to 64
// registers, per-pair certificate branches) and now: 262144 x 262144, l1, d = 8: 80.1 -> 38.9 ms (21.5 instructions per
// pair at 39.3e12 lane operations a second are 37.6 ms); 30000 x 40961, l2, d = 50: 75-85 -> 5.9 ms (3.8 ms).
// Violated scores beyond the slack are counted and summed for the whole step without branches, since a scan far from the
// optimum has one in most votes. 131072 x 131072, l1, d = 8, a third of the pairs violated: 14.2 ms (10.2 with few); pair by
// pair in the part for rare ones 36.4, and 23.2 with the certificate branching per pair.
template <int KIND, int DR, int R, bool TAIL, bool FUSED, bool ST, bool GL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sweep_waves(DR, R)))) void norm_sweep(const float* __restrict__ X, SweepSide side, int64_t m,
                                                  int64_t n, int d, const double* __restrict__ rb,
                                                  const double* __restrict__ cb,
                                                  const unsigned long long* __restrict__ ymaxima, int k,
                                                  int64_t seg_len, double* __restrict__ part_v, int* __restrict__ part_i,
                                                  double* __restrict__ blockstats, int TRANSPOSED,
                                                  const unsigned int* __restrict__ seeds, ColArgs ca,
                                                  const unsigned long long* __restrict__ gate, int64_t gate_cap) {
    static_assert(DR > 0 || R == 1, "streamed rows: one per thread");
    constexpr int J = step_columns(DR);
    if (gate != nullptr && *gate <= (unsigned long long)gate_cap) return;  // uniform: the fused lists are complete
    extern __shared__ double smem[];
    __shared__ double sRed[4][5];
    const int T = blockDim.x;
    const int tid = threadIdx.x;
    const int kl = GL ? 0 : k;  // list entries in LDS
    const int ls = GL ? 1 : T;  // between the entries of a list
    double* const sF = smem + tid;                                  // [R][T] row duals
    double* sV = smem + (size_t)R * T + tid;                        // [R][k][T] list scores
    int* sI = reinterpret_cast<int*>(smem + (size_t)R * T * (1 + kl)) + tid;  // [R][k][T] list indices
    float* const sThr = reinterpret_cast<float*>(sI - tid + (size_t)R * T * kl) + tid;  // [R][T] list entry thresholds
    float* const sSlack = sThr + R * T;                             // [R][T] certificate slacks
    int* const sWorst = reinterpret_cast<int*>(sSlack + R * T);     // [R][T] place of the list's worst entry
    TileCol* const sG = reinterpret_cast<TileCol*>(sWorst - tid + R * T);  // [NT + 8]
    unsigned long long* const sOwn = reinterpret_cast<unsigned long long*>(sG + NT + 8);  // [2][NT], fused
    const int64_t row0 = (int64_t)blockIdx.x * (T * R) + tid;       // rows row0 + r T
    const int64_t seg = blockIdx.y;
    if constexpr (GL) {  // [R][T][k], in place
        sV = part_v + (seg * m + row0) * k;
        sI = part_i + (seg * m + row0) * k;
    }
    const int64_t y_begin = seg * seg_len;
    const int64_t y_end = y_begin + seg_len < n ? y_begin + seg_len : n;
    const double ymax1 = key_double(ymaxima[0]);
    const double gmax = key_double(ymaxima[1]);

    float x[R][DR > 0 ? DR : 1];
    float fi32[R];  // -inf for rows past m: their scores never pass a test
    float low[R];   // a pair whose fp32 score is at or below it matters neither to the row's list nor to the certificate
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = row0 + (int64_t)r * T;
        const bool ok = row < m;
        double x1 = 0.0;
        if constexpr (DR > 0) {
#pragma unroll
            for (int t = 0; t < DR; ++t) {
                x[r][t] = (ok && t < d) ? X[row * d + t] : 0.0f;
                x1 += fabs((double)x[r][t]);
            }
        } else if (ok) {
            for (int t = 0; t < d; ++t) x1 += fabs((double)X[row * d + t]);
        }
        const double fi = ok ? rb[row] : 0.0;
        // slack >= |sigma32 - sigma64|: every fp32 operand is within u of its fp64 value and the two fp32 sums
        // round by at most u each; magnitudes are bounded by |g| + c + |f| with c <= ||x||_1 + max||y||_1.
        const float slack = (float)((x1 + ymax1 + gmax + fabs(fi)) * 4.0 * 5.9604644775390625e-08 * (1.0 + 1e-6) + 1e-37);
        const float thr = ok && seeds ? seed_threshold<KIND>(seeds, m, row, k, slack) : -INFINITY;
        fi32[r] = ok ? (float)fi : -INFINITY;
        low[r] = ST ? fminf(thr, -slack) : thr;
        sF[r * T] = fi;
        sThr[r * T] = thr;
        sSlack[r * T] = slack;
        sWorst[r * T] = 0;
        for (int s = 0; s < k && (!GL || ok); ++s) {
            sV[(size_t)r * k * T + s * ls] = -INFINITY;
            sI[(size_t)r * k * T + s * ls] = -1;
        }
    }
    // the same bound over every pair of a column (row side at its maxima)
    const float cslack = FUSED ? (float)((key_double(ca.xmaxima[0]) + ymax1 + gmax + key_double(ca.xmaxima[1])) * 4.0 *
                                         5.9604644775390625e-08 * (1.0 + 1e-6) + 1e-37)
                               : 0.0f;
    double num64 = 0.0, den64[R];
    unsigned int count = 0u;           // violated pairs of this lane's rows in one segment within the slack
    unsigned long long wcount = 0ull;  // and those of the wave beyond the slack
    float cm[R];              // largest acc
#pragma unroll
    for (int r = 0; r < R; ++r) {
        den64[r] = 0.0;
        cm[r] = 0.0f;
    }
    SlotRun run;  // fused: this wave's buffer slots
    // fused: the tiles in rotated order, starting along a Weyl sequence (stride about 0.618 of the tiles), so that the
    // workgroups resident at any time start spread over all tiles and each column is reached by one workgroup after
    // another; a column that many workgroups reach before its running values are set costs each of them slow paths
    int64_t shift = 0, span = 0;
    if constexpr (FUSED) {
        const int64_t ntiles = (y_end - y_begin + NT - 1) / NT;
        shift = (((int64_t)blockIdx.x * (((ntiles * 633) >> 10) | 1)) % ntiles) * NT;
        span = ntiles * NT;
    }
    const unsigned long long none = double_key(-INFINITY);
    // fused (T = NT): thread e moves the own values of the tile's column e into the running ones
    auto flush = [&](int64_t tile) {
        const unsigned long long o1 = sOwn[tid], o2 = sOwn[NT + tid];
        if (o1 != none) running_insert(ca, tile + tid, o1);
        if (o2 != none) running_insert(ca, tile + tid, o2);
    };
    int64_t t0 = -1;
    for (int64_t th = y_begin; th < y_end; th += NT) {
        __syncthreads();
        if (FUSED && t0 >= 0) flush(t0);
        t0 = th;
        if constexpr (FUSED) {
            t0 += shift;
            if (t0 >= y_begin + span) t0 -= span;
            sOwn[tid] = sOwn[NT + tid] = none;
        }
        const int cnt = (int)((y_end - t0) < NT ? (y_end - t0) : NT);
        for (int e = tid; e < cnt; e += T) {
            TileCol c;
            c.g = (float)cb[t0 + e];
            // (any value of a column's monotone running k-th value is a valid lower bound)
            c.thr = INFINITY;
            if constexpr (FUSED) {
                c.thr = column_threshold(running_kth(ca, t0 + e, k), cslack);
                if (ca.seeds) c.thr = fmaxf(c.thr, seed_threshold<KIND>(ca.seeds, ca.n, t0 + e, k, cslack));
            }
            sG[e] = c;
        }
        if (tid < J - 1) sG[cnt + tid] = TileCol{-INFINITY, INFINITY};  // columns past the tile never pass a test
        __syncthreads();
        const float* const yt = t0 >= side.tail_row ? side.tail + (t0 - side.tail_row) * d : side.Y + t0 * d;
        constexpr int SPAN = ST && cost_span(DR) > 0 ? cost_span(DR) : NT;
        for (int j0 = 0; j0 < (SPAN < NT ? cnt : 1); j0 += SPAN) {
            const int j1 = SPAN < NT && cnt > j0 + SPAN ? j0 + SPAN : cnt;
            std::conditional_t<cost_span(DR) == 0, double, float> tden[R];
#pragma unroll
            for (int r = 0; r < R; ++r) tden[r] = 0;
            for (int jj = j0; jj < j1; jj += J) {
                // columns jj .. jj + J - 1 of the tile (past its end: the last one again)
                ScalarRow y[J];
#pragma unroll
                for (int u = 0; u < J; ++u) y[u] = scalar_row(yt + (unsigned)((jj + u < cnt ? jj + u : cnt - 1) * d));
                TileCol col[J];
#pragma unroll
                for (int u = 0; u < J; ++u) col[u] = sG[jj + u];
                float acc[J][R];
                if constexpr (DR > 0) accumulate_reg<KIND, DR, R, J, TAIL>(x, y, d, acc);
                else accumulate_mem<KIND, J>(X + (row0 < m ? row0 : 0) * d, y, d, acc);  // lanes past m read row 0
                unsigned long long hits = 0ull;
#pragma unroll
                for (int u = 0; u < J; ++u) {
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        if constexpr (KIND == HM_COST_L2) {
                            const float t = FUSED ? fminf(low[r], col[u].thr) : low[r];
                            const float b = (col[u].g + fi32[r]) - t;
                            hits |= __ballot(acc[u][r] <= b * fabsf(b));
                        } else {
                            const float sc = (col[u].g - acc[u][r]) + fi32[r];
                            hits |= __ballot(sc > low[r]);
                            if (FUSED) hits |= __ballot(sc > col[u].thr);
                        }
                        if (ST) cm[r] = fmaxf(cm[r], acc[u][r]);  // (a column past the tile repeats its last one)
                    }
                    if (ST) {
                        if (u == 0 || jj + u < cnt) {
                            asm volatile("");  // a scalar branch, not a select per accumulator
#pragma unroll
                            for (int r = 0; r < R; ++r) {
                                if constexpr (cost_span(DR) == 0) {
                                    const double c = acc[u][r];
                                    tden[r] = KIND == HM_COST_L2 ? tden[r] + c : fma(c, c, tden[r]);
                                } else {
                                    tden[r] = KIND == HM_COST_L2 ? tden[r] + acc[u][r] : fmaf(acc[u][r], acc[u][r], tden[r]);
                                }
                            }
                        }
                    }
                }
                if (!hits) continue;
                // some lane has a pair that may matter. Violated scores beyond the slack, of which a state far from the optimum
                // has many, are counted and squared here; only list and column entries and scores within the slack go on
                unsigned int todo = (1u << (J * R)) - 1u;  // pair e = u R + r
                if constexpr (ST) {
                    unsigned long long rare[J][R], any = 0ull;
                    float tnum = 0.0f;
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float slack = sSlack[r * T], thr = sThr[r * T];
#pragma unroll
                        for (int u = 0; u < J; ++u) {
                            const float s32 = (col[u].g - cost_of<KIND>(acc[u][r])) + fi32[r];
                            const bool over = s32 > slack;
                            const float sp = over ? s32 : 0.0f;
                            tnum = fmaf(sp, sp, tnum);
                            wcount += (unsigned long long)__popcll(__ballot(over));
                            rare[u][r] = __ballot(s32 > thr) | __ballot(fabsf(s32) <= slack);
                            if (FUSED) rare[u][r] |= __ballot(s32 > col[u].thr);
                            any |= rare[u][r];
                        }
                    }
                    num64 += (double)tnum;
                    if (!any) continue;
                    todo = 0u;
#pragma unroll
                    for (int e = 0; e < J * R; ++e) todo |= rare[e / R][e % R] ? 1u << e : 0u;
                }
                // rare: each of those pairs in turn
#pragma unroll 1
                for (; todo != 0u; todo &= todo - 1u) {
                    const int e = __builtin_ctz(todo);
                    float a = acc[0][0], f32 = fi32[0];
#pragma unroll
                    for (int u = 0; u < J; ++u)
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            if (e == u * R + r) {
                                a = acc[u][r];
                                f32 = fi32[r];
                            }
                    const int u = e / R, r = e % R;
                    const float gj32 = sG[jj + u].g;
                    const int64_t j = t0 + jj + u;
                    const float c = cost_of<KIND>(a);
                    const float s32 = (gj32 - c) + f32;
                    if constexpr (FUSED) {
                        const bool over = s32 > sG[jj + u].thr;
                        if (__any(over)) {
                            const double sig = (cb[j] - (double)c) + sF[r * T];
                            column_enter(ca, run, over && sig == sig, j, sig, (int)(row0 + (int64_t)r * T), k, sOwn + jj + u,
                                         sOwn + NT + jj + u, &sG[jj + u].thr, cslack);
                        }
                    }
                    const bool enters = s32 > sThr[r * T];
                    const float slack = sSlack[r * T];
                    const bool near = ST && s32 > -slack && !(s32 > slack);
                    if (enters || near) {
                        const double cd = (double)c, fi = sF[r * T], gj = cb[j];
                        const double sig = TRANSPOSED ? (fi - cd) + gj : (gj - cd) + fi;
                        double* const v = sV + (size_t)r * k * T;
                        int* const id = sI + (size_t)r * k * T;
                        const int w = sWorst[r * T];
                        if (enters && sig == sig && better(sig, (int)j, v[w * ls], id[w * ls])) {
                            // the list is unordered: the new entry replaces the worst, and the worst of the rest is found by
                            // independent reads (a sorted insertion is a chain of dependent ones)
                            v[w * ls] = sig;
                            id[w * ls] = (int)j;
                            double kth = v[0];
                            int kid = id[0], at = 0;
#pragma unroll 4
                            for (int s = 1; s < k; ++s) {
                                const double vs = v[s * ls];
                                const int is = id[s * ls];
                                if (better(kth, kid, vs, is)) {
                                    kth = vs;
                                    kid = is;
                                    at = s;
                                }
                            }
                            sWorst[r * T] = at;
                            float thr = sThr[r * T];
                            thr = fmaxf(thr, column_threshold(kth, slack));
                            sThr[r * T] = thr;
                            const float lo = ST ? fminf(thr, -slack) : thr;
#pragma unroll
                            for (int q = 0; q < R; ++q)
                                if (q == r) low[q] = lo;
                        }
                        // beyond the slack the fp32 score decided; within it the exact fp64 score does (the maximum
                        // comes from the exact row lists afterwards)
                        if (near && sig > 0.0) {
                            num64 = fma(sig, sig, num64);
                            ++count;
                        }
                    }
                }
            }
            if (ST) {
#pragma unroll
                for (int r = 0; r < R; ++r) den64[r] += (double)tden[r];
            }
        }
    }
    if constexpr (FUSED) {
        __syncthreads();
        flush(t0);
        slot_run_close(ca, run);
    }
    double den = 0.0;
    float cmax = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = row0 + (int64_t)r * T;
        if (row < m) {
            double* ov = part_v + (seg * m + row) * k;
            int* oi = part_i + (seg * m + row) * k;
            double* const v = sV + (size_t)r * k * T;
            int* const id = sI + (size_t)r * k * T;
            for (int s = 0; GL && s + 1 < k; ++s) {  // in order, best first
                double bv = v[s];
                int bi = id[s], at = s;
#pragma unroll 4
                for (int q = s + 1; q < k; ++q) {
                    const double vq = v[q];
                    const int iq = id[q];
                    if (better(vq, iq, bv, bi)) {
                        bv = vq;
                        bi = iq;
                        at = q;
                    }
                }
                v[at] = v[s];
                id[at] = id[s];
                v[s] = bv;
                id[s] = bi;
            }
            for (int s = 0; !GL && s < k; ++s) {
                double bv = v[0];
                int bi = id[0], at = 0;
#pragma unroll 4
                for (int q = 1; q < k; ++q) {
                    const double vq = v[q * T];
                    const int iq = id[q * T];
                    if (better(vq, iq, bv, bi)) {
                        bv = vq;
                        bi = iq;
                        at = q;
                    }
                }
                ov[s] = bv;
                oi[s] = bi;
                v[at * T] = -INFINITY;
                id[at * T] = -1;
            }
            den += den64[r];
            cmax = fmaxf(cmax, cost_of<KIND>(cm[r]));
        }
    }
    if (ST) {
        const int lane = tid & 63, wave = tid >> 6;
        // (slot 3: exact row maximum later)
        double v[5] = {num64, den, (double)count + (lane == 0 ? (double)wcount : 0.0), 0.0, (double)cmax};
#pragma unroll
        for (int e = 0; e < 5; ++e)
            for (int o = 32; o >= 1; o >>= 1) {
                const double t = __shfl_xor(v[e], o, 64);
                v[e] = e >= 3 ? fmax(v[e], t) : v[e] + t;
            }
        if (lane == 0)
            for (int e = 0; e < 5; ++e) sRed[wave][e] = v[e];
        __syncthreads();
        if (tid == 0) {
            double* dst = blockstats + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 5;
            for (int e = 0; e < 5; ++e) {
                double o = sRed[0][e];
                for (int w = 1; w < T / 64; ++w) o = e >= 3 ? fmax(o, sRed[w][e]) : o + sRed[w][e];
                dst[e] = o;
            }
        }
    }
}

// fp64 costs (HM_FP64, the reference's direct_norm_fp64: cost.cu:10-104 with CHAINS = 1 and a double accumulator):
// each feature difference is taken in fp64 from the fp32 inputs and the features combine one after another in
// feature order; l2 accumulates fma(z, z, acc) (nvcc contracts the multiply-add) and takes one fp64 sqrt.
template <int KIND>
__device__ inline double feature_op64(double part, double z) {
    if (KIND == HM_COST_L1) return part + fabs(z);
    if (KIND == HM_COST_LINF) return fmax(part, fabs(z));
    return fma(z, z, part);
}

// One thread per X row (its features in registers as fp64 when DR > 0, else read from memory), Y tiles in LDS as
// fp32 with their duals as fp64. Scores sigma = (g_j - c) + f_i, the row lists and the certificate are fp64; there
// is no fp32 filter. The lists are exact whatever the order of the pairs, the certificate sums fp64-grade.
template <int KIND, int K, int DR>
__global__ __launch_bounds__(256) void norm_sweep64(const float* __restrict__ X, const float* __restrict__ Y, int64_t m,
                                                    int64_t n, int d, const double* __restrict__ rb,
                                                    const double* __restrict__ cb, int k, int64_t seg_len,
                                                    double* __restrict__ part_v, int* __restrict__ part_i,
                                                    double* __restrict__ blockstats, int STATS, int TRANSPOSED,
                                                    int ntile) {
    extern __shared__ float4 smem4[];
    double* scb = reinterpret_cast<double*>(smem4);   // ntile column duals
    float* sy = reinterpret_cast<float*>(scb + ntile);  // ntile * d features
    __shared__ double sRed[4][5];
    const int tid = threadIdx.x;
    const int64_t row = (int64_t)blockIdx.x * NB_ROWS + tid;
    const bool row_ok = row < m;
    const int64_t y_begin = (int64_t)blockIdx.y * seg_len;
    const int64_t y_end = y_begin + seg_len < n ? y_begin + seg_len : n;

    double x[DR > 0 ? DR : 1];
    if (DR > 0) {
#pragma unroll
        for (int t = 0; t < (DR > 0 ? DR : 1); ++t) x[t] = (row_ok && t < d) ? (double)X[row * d + t] : 0.0;
    }
    const float* xr = X + (row_ok ? row : 0) * d;
    const double fi = row_ok ? rb[row] : 0.0;
    double v[K];
    int id[K];
#pragma unroll
    for (int s = 0; s < K; ++s) { v[s] = -INFINITY; id[s] = -1; }
    double num = 0.0, den = 0.0, cnt = 0.0, cmax = 0.0;
    for (int64_t t0 = y_begin; t0 < y_end; t0 += ntile) {
        const int tn = (int)((y_end - t0) < ntile ? (y_end - t0) : ntile);
        __syncthreads();
        for (int e = tid; e < tn * d; e += 256) sy[e] = Y[t0 * d + e];
        for (int e = tid; e < tn; e += 256) scb[e] = cb[t0 + e];
        __syncthreads();
        if (!row_ok) continue;
        for (int jj = 0; jj < tn; ++jj) {
            const float* yj = sy + (size_t)jj * d;
            double c = 0.0;
            if (DR > 0) {
#pragma unroll
                for (int t = 0; t < (DR > 0 ? DR : 1); ++t)
                    if (t < d) c = feature_op64<KIND>(c, x[t] - (double)yj[t]);
            } else {
                for (int t = 0; t < d; ++t) c = feature_op64<KIND>(c, (double)xr[t] - (double)yj[t]);
            }
            if (KIND == HM_COST_L2) c = sqrt(c);
            const double sig = TRANSPOSED ? (fi - c) + scb[jj] : (scb[jj] - c) + fi;
            const int j = (int)(t0 + jj);
            if (sig == sig && better(sig, j, v[k - 1], id[k - 1])) put_sorted<K>(v, id, k, sig, j);
            if (STATS) {
                den = fma(c, c, den);
                cmax = fmax(cmax, c);
                if (sig > 0.0) {
                    num = fma(sig, sig, num);
                    cnt += 1.0;
                }
            }
        }
    }
    if (row_ok) {
        double* ov = part_v + ((int64_t)blockIdx.y * m + row) * k;
        int* oi = part_i + ((int64_t)blockIdx.y * m + row) * k;
        for (int s = 0; s < k; ++s) { ov[s] = v[s]; oi[s] = id[s]; }
    }
    if (STATS) {
        const int lane = tid & 63, wave = tid >> 6;
        double r[5] = {num, den, cnt, 0.0, cmax};  // slot 3: exact row maximum later
#pragma unroll
        for (int e = 0; e < 5; ++e)
            for (int o = 32; o >= 1; o >>= 1) {
                const double t = __shfl_xor(r[e], o, 64);
                r[e] = e >= 3 ? fmax(r[e], t) : r[e] + t;
            }
        if (lane == 0)
            for (int e = 0; e < 5; ++e) sRed[wave][e] = r[e];
        __syncthreads();
        if (tid == 0) {
            double* dst = blockstats + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 5;
            for (int e = 0; e < 5; ++e) {
                double o = sRed[0][e];
                for (int w = 1; w < 4; ++w) o = e >= 3 ? fmax(o, sRed[w][e]) : o + sRed[w][e];
                dst[e] = o;
            }
        }
    }
}

// Merge S sorted exact segment lists per row (tie rule): G lanes per row (a power of two of at least S), each at the
// head of one list, take the best head k times. Gated like norm_sweep. rowmax (or null) receives the largest first entry
// of all rows (an ordered key, one atomic per wave).
__global__ __launch_bounds__(256) void norm_merge(const double* __restrict__ part_v, const int* __restrict__ part_i,
                                                  int64_t m, int S, int G, int k, double* __restrict__ out_v,
                                                  int* __restrict__ out_i, const unsigned long long* gate,
                                                  int64_t gate_cap, unsigned long long* __restrict__ rowmax) {
    if (gate != nullptr && *gate <= (unsigned long long)gate_cap) return;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t row = t / G;
    const int l = (int)(t % G);
    const bool live = row < m && l < S;
    const double* pv = part_v + (live ? ((int64_t)l * m + row) * k : 0);
    const int* pi = part_i + (live ? ((int64_t)l * m + row) * k : 0);
    double hv = live ? pv[0] : -INFINITY, top = 0.0;
    int hi = live ? pi[0] : -1, at = 0;
    for (int s = 0; s < k; ++s) {
        double bv = hv;
        int bi = hi, bl = l;
        for (int o = G / 2; o >= 1; o >>= 1) {
            const double ov = __shfl_xor(bv, o, 64);
            const int oi = __shfl_xor(bi, o, 64), ol = __shfl_xor(bl, o, 64);
            if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; bl = ol; }
        }
        if (s == 0) top = fmax(bv, 0.0);
        if (row < m && l == 0) {
            out_v[row * k + s] = bv;
            out_i[row * k + s] = bi;
        }
        if (live && bl == l && bi >= 0) {  // this head was taken
            ++at;
            hv = at < k ? pv[at] : -INFINITY;
            hi = at < k ? pi[at] : -1;
        }
    }
    if (rowmax) {
        for (int o = 32; o >= 1; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
        if ((threadIdx.x & 63) == 0) atomicMax(rowmax, double_key(top));
    }
}

// fused column state: thresholds at double_key(-inf), counts at zero
__global__ void cols_clear(unsigned long long* __restrict__ gthr, int* __restrict__ ccount, int64_t n,
                           unsigned long long* __restrict__ count) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) gthr[j] = gthr[n + j] = double_key(-INFINITY);
    if (j <= n) ccount[j] = 0;
    if (j == 0) *count = 0ull;
}

// Candidates per column (empty slots skipped) among those that can be in its list: after the sweep a column's running
// k-th value is its exact k-th best score, so only candidates at or above it count, k per column and ties with the
// k-th, of the 16 to 20 a column collects (one atomic each).
__global__ void cols_count(const ColCand* __restrict__ buf, const unsigned long long* __restrict__ count, int64_t cap,
                           const unsigned long long* __restrict__ kth, int* __restrict__ ccount) {
    const unsigned long long c = *count;
    if (c > (unsigned long long)cap) return;
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < (int64_t)c; s += (int64_t)gridDim.x * blockDim.x) {
        const ColCand cc = buf[s];
        if (cc.j >= 0 && cc.v >= key_double(kth[cc.j])) atomicAdd(ccount + cc.j, 1);
    }
}

// buffer slots grouped by column: slot s of column j goes to coff[j] + (its rank among the column's arrivals);
// ccount counts back down to zero
__global__ void cols_group(const ColCand* __restrict__ buf, const unsigned long long* __restrict__ count, int64_t cap,
                           const unsigned long long* __restrict__ kth, const int* __restrict__ coff,
                           int* __restrict__ ccount, int* __restrict__ order) {
    const unsigned long long c = *count;
    if (c > (unsigned long long)cap) return;  // overflowed: the role-swapped sweep gives the columns
    for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < (int64_t)c; s += (int64_t)gridDim.x * blockDim.x) {
        const ColCand cc = buf[s];
        if (cc.j >= 0 && cc.v >= key_double(kth[cc.j])) order[coff[cc.j] + atomicSub(ccount + cc.j, 1) - 1] = (int)s;
    }
}

// each column's k best among its candidates (tie rule), one thread per column
template <int K>
__global__ void cols_select(const ColCand* __restrict__ buf, const unsigned long long* __restrict__ count, int64_t cap,
                            const int* __restrict__ coff, const int* __restrict__ order, int64_t n, int k,
                            double* __restrict__ out_v, int* __restrict__ out_i) {
    if (*count > (unsigned long long)cap) return;
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    double v[K];
    int id[K];
#pragma unroll
    for (int s = 0; s < K; ++s) { v[s] = -INFINITY; id[s] = -1; }
    for (int e = coff[j]; e < coff[j + 1]; ++e) {
        const ColCand c = buf[order[e]];
        put_sorted<K>(v, id, k, c.v, c.i);
    }
    for (int s = 0; s < k; ++s) { out_v[j * k + s] = v[s]; out_i[j * k + s] = id[s]; }
}

__global__ void norm_reduce_stats(const double* __restrict__ blockstats, int64_t blocks, double* __restrict__ stats,
                                  const unsigned long long* __restrict__ rowmax, int linf) {
    __shared__ double s[256][5];
    const int t = threadIdx.x;
    double v[5] = {0, 0, 0, 0, 0};
    for (int64_t b = t; b < blocks; b += 256)
        for (int e = 0; e < 5; ++e) v[e] = e >= 3 ? fmax(v[e], blockstats[b * 5 + e]) : v[e] + blockstats[b * 5 + e];
    for (int e = 0; e < 5; ++e) s[t][e] = v[e];
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if (t < w)
            for (int e = 0; e < 5; ++e) s[t][e] = e >= 3 ? fmax(s[t][e], s[t + w][e]) : s[t][e] + s[t + w][e];
        __syncthreads();
    }
    if (t == 0) {
        stats[0] = s[0][0];
        stats[1] = s[0][1];
        stats[2] = s[0][2];
        stats[3] = key_double(*rowmax);  // the exact maximum violation: the best entry of the fp64 row lists, or 0
        stats[4] = linf ? s[0][4] : 0.0;
    }
}

// seeds at float_key(-inf)
__global__ __launch_bounds__(256) void norm_fill(unsigned int* __restrict__ p, int64_t count) {
    const int64_t first = (int64_t)blockIdx.x * 1024 + threadIdx.x;
#pragma unroll
    for (int t = 0; t < 4; ++t)
        if (first + 256 * t < count) p[first + 256 * t] = 0x007fffffu;
}

__global__ void norm_zero(unsigned long long* p, int count) {
    if ((int)threadIdx.x < count) p[threadIdx.x] = 0ull;
}

constexpr int GLOBAL_FEATURES = 32;  // longest rows whose sweeps also come with lists outside LDS
// One sweep direction: S segments of seg_len columns; workgroups of T threads with R rows each.
struct NormPlan {
    int S, R, T;
    bool global;  // lists in their place in the partial lists
    int64_t seg_len;
};

inline NormPlan norm_segments(int64_t rows, int64_t cols, int64_t rows_per_block, int64_t max_s) {
    const int64_t blocks = (rows + rows_per_block - 1) / rows_per_block;
    int64_t s = (1024 + blocks - 1) / blocks;
    const int64_t tiles = (cols + NT - 1) / NT;
    if (s > tiles) s = tiles;
    if (s > max_s) s = max_s;
    if (s < 1) s = 1;
    const int64_t per = (tiles + s - 1) / s;
    NormPlan p;
    p.seg_len = per * NT;
    p.S = (int)((cols + p.seg_len - 1) / p.seg_len);
    p.R = 1;
    p.T = NB_ROWS;
    p.global = false;
    return p;
}

// The fp64 sweep: 256 threads, one row each. The fp32 sweep: two rows per thread share the loads and tests of a Y row
// where their features fit the registers beside enough waves (d <= 32) and the problem still fills the chip. Its partial
// lists take no more than those of one row per thread, or 24 MiB.
// Lists in LDS, 12 k bytes a row, leave few waves on a CU: 20 at k = 9 and 10, 12 to 16 at k = 11 to 16, 10 at k = 17 to 20
// (128 threads from 17 on), 8 and 6 beyond. In their place in the partial lists, in memory, an entry costs more and a
// pair less, so memory wins on long sides, and first where the waves in LDS are few for their k. Rows of l1, in LDS and in
// memory, d = 8:
//   k = 16: 16384^2 3.8 and 3.6 ms, 32768^2 9.1 and 8.1, 262144^2 99 and 58, 524288^2 379 and 200 (k = 11: 2.5 and 2.5,
//           5.7 and 5.3; k = 14: 3.1 and 3.5, 7.3 and 7.7, 65536^2 14.0 and 13.4); both sides of 3000^2 1.15 and 1.45
//   k = 32: 16384^2 13.4 and 9.5, 65536^2 56 and 44, 524288^2 894 and 332; both sides of 3000^2 2.2 and 2.9
//   k = 9: 65536^2 5.8 and 7.0, 131072^2 14.2 and 15.4; k = 20: 65536^2 15.2 and 23.3, 131072^2 32 and 38
//   k = 8: 65536^2 5.1 and 5.8, 131072^2 13.3 and 13.7, 180000^2 32.1 and 20.8, 524288^2 183 and, two rows a thread, 128.
// Rows of more than 32 features keep LDS.
inline bool lists_in_memory(int64_t rows, int64_t cols, int d, int k) {
    if (d > GLOBAL_FEATURES || k <= 4 || (k <= 8 && d > 8)) return false;
    const bool few_waves = (k > 10 && k <= 16) || k > 20;
    return rows > (int64_t(1) << (few_waves ? 29 : 34)) / cols;
}

inline NormPlan norm_plan(int64_t rows, int64_t cols, int d, int k, uint32_t flags) {
    const NormPlan one = norm_segments(rows, cols, NB_ROWS, 64);
    if (flags & HM_FP64) return one;
    const bool global = lists_in_memory(rows, cols, d, k);
    const int T = k > 16 && !global ? 128 : 256;
    const bool fills = ((rows + 511) / 512) * ((cols + NT - 1) / NT) >= 4096;
    const int R = d <= 32 && ((k <= 4 && fills) || (global && k <= 8 && rows >= 524288)) ? 2 : 1;
    int64_t most = (int64_t(24) << 20) / (12 * rows * k);
    if (most < one.S) most = one.S;
    NormPlan p = norm_segments(rows, cols, (int64_t)T * R, most < 64 ? most : 64);
    p.R = R;
    p.T = T;
    p.global = global;
    return p;
}

inline int kbucket(int k) { return k <= 2 ? 2 : (k <= 8 ? 8 : 32); }

// columns ride on the row sweep (k <= 2 with rows and columns requested; buffer slots in int32). Not where the rows are
// many times the columns: the workgroups that are on a column's tile at one time each append their best, which at 64
// times overflows the buffer (262144 x 4000, l2: 8.1 ms with the second sweep that follows, 6.9 ms by two sweeps).
inline bool fusable(int64_t m, int64_t n, int k, uint32_t flags) {
    return k <= 2 && m <= 32 * n && (flags & HM_ROWS) && (flags & HM_COLS) && !(flags & HM_FP64) && fused_cap(n, k) < INT32_MAX;
}

struct NormWork {
    double* pv;  // segment lists (rows, then the role-swapped columns)
    int* pi;
    double* bs;  // per-workgroup certificate partials
    unsigned long long* maxima;  // [0..1] Y side, [2..3] X side, [4] the largest row score
    float *ytail, *xtail;        // fp32 sweeps: padded copies of the sides' last rows (SweepSide)
    unsigned int *rseeds, *cseeds;  // fp32 sweeps: entry floors of the row and column lists (norm_seed); null: no room
    // fused columns
    unsigned long long* gthr;
    ColCand* buf;
    unsigned long long* count;
    int *ccount, *coff, *order;
    void* scan_tmp;
    size_t scan_bytes;
    int64_t cap;
};

inline size_t scan_tmp_bytes(int64_t n) {
    size_t bytes = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, (const int*)nullptr, (int*)nullptr, (int)(n + 1));
    return bytes;
}

// certificate partials: of the row sweep, which in a fused call takes them in any case
inline size_t blockstats_doubles(const NormPlan& rows, int64_t m, uint32_t flags, int64_t cap) {
    const int64_t per = (int64_t)rows.R * rows.T;
    return (flags & HM_STATS) || cap > 0 ? (size_t)5 * ((m + per - 1) / per) * rows.S : 1;
}

// cap > 0: the fused path with a candidate buffer of cap entries
template <class A>
void norm_layout(A& a, int64_t m, int64_t n, int d, int k, uint32_t flags, bool seeded, int64_t cap, NormWork& w) {
    const NormPlan pr = norm_plan(m, n, d, k, flags), pc = norm_plan(n, m, d, k, flags);
    size_t entries = 0;
    if (flags & (HM_ROWS | HM_STATS)) entries = (size_t)pr.S * m * k;
    if (flags & HM_COLS) {
        const size_t c = (size_t)pc.S * n * k;
        if (c > entries) entries = c;
    }
    w.pv = a.template take<double>(entries > 0 ? entries : 1);
    w.pi = a.template take<int>(entries > 0 ? entries : 1);
    w.bs = a.template take<double>(blockstats_doubles(pr, m, flags, cap));
    w.maxima = a.template take<unsigned long long>(5);
    const bool fp32 = !(flags & HM_FP64);
    w.ytail = a.template take<float>(fp32 && (flags & (HM_ROWS | HM_STATS)) ? tail_floats(n, d) : 1);
    w.xtail = a.template take<float>(fp32 && (flags & HM_COLS) ? tail_floats(m, d) : 1);
    w.rseeds = w.cseeds = nullptr;
    if (seeded && fp32) {
        if (flags & (HM_ROWS | HM_STATS)) w.rseeds = a.template take<unsigned int>((size_t)m * k);
        if (flags & HM_COLS) w.cseeds = a.template take<unsigned int>((size_t)n * k);
    }
    w.cap = cap;
    if (cap <= 0) return;
    w.gthr = a.template take<unsigned long long>(2 * n);
    w.count = a.template take<unsigned long long>(1);
    w.ccount = a.template take<int>(n + 1);
    w.coff = a.template take<int>(n + 1);
    w.order = a.template take<int>(w.cap);
    w.buf = a.template take<ColCand>(w.cap);
    w.scan_bytes = scan_tmp_bytes(n);
    w.scan_tmp = a.template take<char>(w.scan_bytes > 0 ? w.scan_bytes : 1);
}

// one sweep direction: rows of X against Y (TRANSPOSED: the roles swapped for the column lists)
struct Direction {
    const float *X, *Y;
    const float* tail;            // the padded copy of Y's last rows
    const unsigned int* seeds;    // entry floors of X's row lists, or none
    int64_t m, n;
    const double *rb, *cb;
    const unsigned long long* ymaxima;
    bool stats, transposed;
    NormPlan plan;
    double* out_v;
    int* out_i;
    ColArgs cols;                     // fused columns (cols.gthr == nullptr: none)
    const unsigned long long* gate;   // role-swapped column sweep of a fused call
    int64_t gate_cap;
};

inline void launch_merge(hipStream_t st, const Direction& D, int k, const NormWork& w) {
    int G = 1;
    while (G < D.plan.S) G *= 2;  // S <= 64
    hipLaunchKernelGGL(norm_merge, dim3((unsigned)((D.m * G + 255) / 256)), dim3(256), 0, st, w.pv, w.pi, D.m, D.plan.S,
                       G, k, D.out_v, D.out_i, D.gate, D.gate_cap, D.stats ? w.maxima + 4 : nullptr);
}

// the segment lists merged (after the sweep), and the certificate's partial sums reduced
inline int finish_direction(hipStream_t st, const Direction& D, int64_t blocks, int k, const NormWork& w,
                            double* stats_out, int linf) {
    launch_merge(st, D, k, w);
    HM_LAUNCH_CHECK("norm_merge");
    if (D.stats) {
        hipLaunchKernelGGL(norm_reduce_stats, dim3(1), dim3(256), 0, st, w.bs, blocks, stats_out, w.maxima + 4, linf);
        HM_LAUNCH_CHECK("norm_reduce_stats");
    }
    return HM_OK;
}

template <int KIND, int DR, int R, bool TAIL>
int norm_direction_t(hipStream_t st, const Direction& D, int d, int k, const NormWork& w, double* stats_out, int linf) {
    const int64_t rows = (int64_t)D.plan.T * R;
    const dim3 grid((unsigned)((D.m + rows - 1) / rows), (unsigned)D.plan.S), block((unsigned)D.plan.T);
    const size_t shmem = sweep_lds(D.plan.T, R, D.plan.global ? 0 : k, D.cols.gthr != nullptr);
    const SweepSide side{D.Y, D.tail, tail_start(D.n, d)};
    prof_begin(st, D.gate != nullptr ? "norm_sweep_swapped" : "norm_sweep");
#define HM_NORM_SWEEP(FUSED, ST, GL)                                                                                \
    hipLaunchKernelGGL((norm_sweep<KIND, DR, R, TAIL, FUSED, ST, GL>), grid, block, shmem, st, D.X, side, D.m, D.n, d, D.rb, \
                       D.cb, D.ymaxima, k, D.plan.seg_len, w.pv, w.pi, w.bs, (int)D.transposed, D.seeds, D.cols, D.gate, D.gate_cap)
    // (a fused call without the certificate takes the same kernel and leaves its sums unread)
    bool done = false;
    if constexpr (DR > 0 && DR <= GLOBAL_FEATURES) {
        if (D.plan.global) {
            if (D.stats) HM_NORM_SWEEP(false, true, true);
            else HM_NORM_SWEEP(false, false, true);
            done = true;
        }
    }
    if (done) {
    } else if (D.cols.gthr != nullptr) HM_NORM_SWEEP(true, true, false);
    else if (D.stats) HM_NORM_SWEEP(false, true, false);
    else HM_NORM_SWEEP(false, false, false);
#undef HM_NORM_SWEEP
    prof_end(st);
    HM_LAUNCH_CHECK("norm_sweep");
    return finish_direction(st, D, (int64_t)grid.x * grid.y, k, w, stats_out, linf);
}

// Entry floors of one side's lists (norm_seed) from 1/32 of the columns, at least 1024 of them: a floor then lets through
// a few times the k pairs a list keeps on a short side. Short lists find the rest of the way themselves (at most 1024
// columns: under a hundredth of the sweep on long sides); long ones take up to 4096. Split over enough workgroups to
// fill the chip with at least 32 columns each. Where the rows alone fill it (256 workgroups) the sample's own time counts:
// lists of up to 8 then take 1/16 of the columns of a short side, at least 128 (top-1 rows of l1, d = 5, 200000 x 1000 /
// 3000 / 8000: 0.71 / 0.95 / 1.53 -> 0.38 / 0.72 / 1.37 ms; top-16 would go 4.5 -> 5.3 and 3000 x 3000 0.069 -> 0.089).
constexpr int64_t SEED_FULL_ROWS = 65536;
struct Seeding {
    const float* X;
    SweepSide side;
    int64_t m, n;
    const double *rb, *cb;
    unsigned int* seeds;
};

template <int KIND, int DR, bool TAIL>
int norm_seed_t(hipStream_t st, const Seeding& s, int d, int k) {
    int64_t count = s.n / 32;
    const int64_t most = k <= 4 ? 1024 : 4096;
    int64_t least = 1024;
    if (s.m >= SEED_FULL_ROWS && k <= 8) least = s.n / 16 < 128 ? 128 : (s.n / 16 > 1024 ? 1024 : s.n / 16);
    count = count < least ? least : (count > most ? most : count);
    if (count > s.n) count = s.n;
    const int64_t blocks = (s.m + 255) / 256;
    int64_t q = (1024 + blocks - 1) / blocks;
    if (q > count / 32) q = count / 32;
    q = (q + k - 1) / k * k;
    if (q < k) q = k;
    const int64_t words = s.m * k;
    hipLaunchKernelGGL(norm_fill, dim3((unsigned)((words + 1023) / 1024)), dim3(256), 0, st, s.seeds, words);
    hipLaunchKernelGGL((norm_seed<KIND, DR, TAIL>), dim3((unsigned)blocks, (unsigned)q), dim3(256), 0, st, s.X, s.side,
                       s.m, s.n, d, s.rb, s.cb, k, (int)count, (int)q, s.seeds);
    HM_LAUNCH_CHECK("norm_seed");
    return HM_OK;
}

// Register features: F<KIND, DR, R, TAIL> at the smallest width of below() that holds d and the plan's rows per thread;
// rows past 128 features are streamed.
#define HM_NORM_WIDTH(F, DR, R, WHOLE, ...) \
    return (d % (WHOLE) != 0) ? F<KIND, DR, R, true>(__VA_ARGS__) : F<KIND, DR, R, false>(__VA_ARGS__)
#define HM_NORM_ROWS(F, DR, WHOLE, ...)                             \
    do {                                                            \
        if (rows == 2) HM_NORM_WIDTH(F, DR, 2, WHOLE, __VA_ARGS__); \
        HM_NORM_WIDTH(F, DR, 1, WHOLE, __VA_ARGS__);                \
    } while (0)
template <int KIND>
int norm_direction(hipStream_t st, const Direction& D, int d, int k, const NormWork& w, double* stats_out, int linf) {
    const int rows = D.plan.R;
#define HM_ARGS st, D, d, k, w, stats_out, linf
    if (d <= 4) HM_NORM_ROWS(norm_direction_t, 4, 4, HM_ARGS);
    if (d <= 8) HM_NORM_ROWS(norm_direction_t, 8, 8, HM_ARGS);
    if (d <= 16) HM_NORM_ROWS(norm_direction_t, 16, 8, HM_ARGS);
    if (d <= 24) HM_NORM_ROWS(norm_direction_t, 24, 8, HM_ARGS);
    if (d <= 32) HM_NORM_ROWS(norm_direction_t, 32, 8, HM_ARGS);
    if (d <= 48) HM_NORM_WIDTH(norm_direction_t, 48, 1, 8, HM_ARGS);
    if (d <= 64) HM_NORM_WIDTH(norm_direction_t, 64, 1, 8, HM_ARGS);
    if (d <= 96) HM_NORM_WIDTH(norm_direction_t, 96, 1, 8, HM_ARGS);
    if (d <= 128) HM_NORM_WIDTH(norm_direction_t, 128, 1, 8, HM_ARGS);
    return norm_direction_t<KIND, 0, 1, true>(HM_ARGS);
#undef HM_ARGS
}
#undef HM_NORM_ROWS
#undef HM_NORM_WIDTH

template <int KIND>
int norm_seeds(hipStream_t st, const Seeding& s, int d, int k) {
#define HM_SEED(DR, WHOLE) return (d % (WHOLE) != 0) ? norm_seed_t<KIND, DR, true>(st, s, d, k) : norm_seed_t<KIND, DR, false>(st, s, d, k)
    if (d <= 4) HM_SEED(4, 4);
    if (d <= 8) HM_SEED(8, 8);
    if (d <= 16) HM_SEED(16, 8);
    if (d <= 24) HM_SEED(24, 8);
    if (d <= 32) HM_SEED(32, 8);
    if (d <= 48) HM_SEED(48, 8);
    if (d <= 64) HM_SEED(64, 8);
    if (d <= 96) HM_SEED(96, 8);
    if (d <= 128) HM_SEED(128, 8);
    return norm_seed_t<KIND, 0, true>(st, s, d, k);
#undef HM_SEED
}

template <int KIND, int K, int DR>
int norm_direction64_t(hipStream_t st, const Direction& D, int d, int k, const NormWork& w, double* stats_out,
                       int linf) {
    dim3 grid((unsigned)((D.m + NB_ROWS - 1) / NB_ROWS), (unsigned)D.plan.S);
    const size_t budget = (size_t)LDS_FLOATS * sizeof(float);
    auto bytes = [d](int t) { return (size_t)t * sizeof(double) + (size_t)t * d * sizeof(float); };
    int ntile = NT;
    while (ntile > 1 && bytes(ntile) > budget) ntile >>= 1;
    if (bytes(ntile) > budget) return fail(HM_EINVAL, "fp64 norm pricing supports d <= %d", LDS_FLOATS - 2);
    prof_begin(st, D.transposed ? "norm_sweep64_swapped" : "norm_sweep64");
    hipLaunchKernelGGL((norm_sweep64<KIND, K, DR>), grid, dim3(256), bytes(ntile), st, D.X, D.Y, D.m, D.n, d, D.rb, D.cb,
                       k, D.plan.seg_len, w.pv, w.pi, w.bs, (int)D.stats, (int)D.transposed, ntile);
    prof_end(st);
    HM_LAUNCH_CHECK("norm_sweep64");
    return finish_direction(st, D, (int64_t)grid.x * grid.y, k, w, stats_out, linf);
}

template <int KIND, int K>
int norm_direction64_d(hipStream_t st, const Direction& D, int d, int k, const NormWork& w, double* stats_out, int linf) {
    if (d <= 8) return norm_direction64_t<KIND, K, 8>(st, D, d, k, w, stats_out, linf);
    if (d <= 32) return norm_direction64_t<KIND, K, 32>(st, D, d, k, w, stats_out, linf);
    if (d <= 64) return norm_direction64_t<KIND, K, 64>(st, D, d, k, w, stats_out, linf);
    return norm_direction64_t<KIND, K, 0>(st, D, d, k, w, stats_out, linf);
}

template <int KIND>
int norm_direction64(hipStream_t st, const Direction& D, int d, int k, const NormWork& w, double* stats_out, int linf) {
    switch (kbucket(k)) {
        case 2: return norm_direction64_d<KIND, 2>(st, D, d, k, w, stats_out, linf);
        case 8: return norm_direction64_d<KIND, 8>(st, D, d, k, w, stats_out, linf);
        case 32: return norm_direction64_d<KIND, 32>(st, D, d, k, w, stats_out, linf);
    }
    return fail(HM_EINVAL, "unsupported k");
}

inline size_t norm_workspace(int64_t m, int64_t n, int d, int k, uint32_t flags, bool seeded, int64_t cap) {
    Sizer s;
    NormWork w;
    norm_layout(s, m, n, d, k, flags, seeded, cap, w);
    return s.used;
}

// What a workspace of `bytes` holds beyond the two-sweep minimum: the entry floors of the lists (seeded), and the
// candidate capacity of the fused path: the full one when it fits, else (with partial) what fits (the fused path stays
// exact with any capacity: an overflow hands the columns to the role-swapped sweep); 0: two sweeps.
struct NormFit {
    bool seeded;
    int64_t cap;
};

inline NormFit norm_fit(int64_t m, int64_t n, int d, int k, uint32_t flags, size_t bytes, bool partial) {
    auto fits = [&](bool seeded, int64_t cap) { return norm_workspace(m, n, d, k, flags, seeded, cap) <= bytes; };
    if (fusable(m, n, k, flags)) {
        const int64_t full = fused_cap(n, k);
        if (fits(true, full)) return NormFit{true, full};
        if (fits(false, full)) return NormFit{false, full};
        for (int seeded = 1; partial && seeded >= 0; --seeded) {
            const size_t fixed = norm_workspace(m, n, d, k, flags, seeded != 0, 1);
            const size_t per = sizeof(ColCand) + sizeof(int);
            if (bytes < fixed + 512 + per) continue;
            int64_t cap = (int64_t)((bytes - fixed - 512) / per);  // 512: the two arrays' rounding to 256 bytes
            if (cap > full) cap = full;
            if (fits(seeded != 0, cap)) return NormFit{seeded != 0, cap};
        }
    }
    return NormFit{fits(true, 0), 0};
}

}  // namespace
}  // namespace hm

using namespace hm;

// the workspace of the fused path where it applies (a smaller workspace still runs the two-sweep path)
extern "C" size_t hm_pricing_norm_workspace_bytes(int64_t m, int64_t n, int32_t d, int32_t k, uint32_t flags) {
    if (m < 1 || n < 1 || d < 1 || k < 1 || k > 32) return 0;
    return norm_workspace(m, n, d, k, flags, true, fusable(m, n, k, flags) ? fused_cap(n, k) : 0);
}

namespace {

// the most features a scan takes
int check_features(int32_t d, uint32_t flags) {
    const int most = (flags & HM_FP64) ? LDS_FLOATS - 2 : LDS_FLOATS - 1;
    HM_CHECK_ARG(d >= 1 && d <= most, "%snorm pricing supports d <= %d", (flags & HM_FP64) ? "fp64 " : "", most);
    return HM_OK;
}

// The scan with its scratch in `workspace` (caller memory, or the static scratch array of hm_pricing_norm_noalloc).
// Everything the scratch holds is written before it is read; maxima, thresholds and counts are cleared by kernels,
// not memsets.
int norm_scan_run(void* stream, const float* X, const float* Y, const double* f, const double* g, int64_t m,
                  int64_t n, int32_t d, int32_t k, int32_t kind, uint32_t flags, double* row_val, int32_t* row_idx,
                  double* col_val, int32_t* col_idx, double* stats, void* workspace, size_t workspace_bytes,
                  bool partial_buffer) {
    HM_CHECK_ARG(X && Y && f && g, "norm pricing: feature and dual pointers are required");
    HM_CHECK_ARG(m >= 1 && n >= 1 && d >= 1 && m < INT32_MAX && n < INT32_MAX,
                 "norm pricing requires nonempty inputs with int32 dimensions");
    HM_CHECK_ARG(k >= 1 && k <= 32, "norm pricing requires 1 <= k <= 32 (k=%d)", k);
    if (int rc = check_features(d, flags)) return rc;
    HM_CHECK_ARG(kind == HM_COST_L1 || kind == HM_COST_LINF || kind == HM_COST_L2, "unsupported norm cost %d", kind);
    HM_CHECK_ARG(!(flags & HM_ROWS) || (row_val && row_idx), "HM_ROWS requires row outputs");
    HM_CHECK_ARG(!(flags & HM_COLS) || (col_val && col_idx), "HM_COLS requires column outputs");
    HM_CHECK_ARG(!(flags & HM_STATS) || stats, "HM_STATS requires a stats output");
    HM_CHECK_ARG(!(flags & HM_STATS) || (flags & HM_ROWS), "norm pricing: HM_STATS requires HM_ROWS");
    HM_CHECK_ARG(workspace != nullptr, "workspace is required");
    const size_t need = norm_workspace(m, n, d, k, flags, false, 0);
    if (workspace_bytes < need)
        return fail(HM_ENOSPC, "norm pricing workspace too small: %zu < %zu bytes", workspace_bytes, need);
    const NormFit fit = norm_fit(m, n, d, k, flags, workspace_bytes, partial_buffer);
    const bool fused = fit.cap > 0;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    Arena a(workspace, workspace_bytes);
    NormWork w;
    norm_layout(a, m, n, d, k, flags, fit.seeded, fit.cap, w);
    hipLaunchKernelGGL(norm_zero, dim3(1), dim3(64), 0, st, w.maxima, 5);
    HM_LAUNCH_CHECK("norm_zero");
    hipLaunchKernelGGL(norm_prep, dim3(prep_blocks(n)), dim3(256), 0, st, Y, n, d, g, w.maxima);
    HM_LAUNCH_CHECK("norm_prep");
    hipLaunchKernelGGL(norm_prep, dim3(prep_blocks(m)), dim3(256), 0, st, X, m, d, f, w.maxima + 2);
    HM_LAUNCH_CHECK("norm_prep");
    const int linf = (flags & HM_LINF) ? 1 : 0;
    const bool fp64 = (flags & HM_FP64) != 0;
    auto dispatch = [&](const Direction& D) {
        if (fp64) {
            if (kind == HM_COST_L1) return norm_direction64<HM_COST_L1>(st, D, d, k, w, stats, linf);
            if (kind == HM_COST_LINF) return norm_direction64<HM_COST_LINF>(st, D, d, k, w, stats, linf);
            return norm_direction64<HM_COST_L2>(st, D, d, k, w, stats, linf);
        }
        if (kind == HM_COST_L1) return norm_direction<HM_COST_L1>(st, D, d, k, w, stats, linf);
        if (kind == HM_COST_LINF) return norm_direction<HM_COST_LINF>(st, D, d, k, w, stats, linf);
        return norm_direction<HM_COST_L2>(st, D, d, k, w, stats, linf);
    };
    if (!fp64) {
        if (d <= REG_FEATURES) {
            auto tail = [&](const float* S, int64_t rows, float* out) {
                const int64_t first = tail_start(rows, d) * d, count = rows * d - first;
                hipLaunchKernelGGL(norm_tail, dim3((unsigned)((count + PAD + 255) / 256)), dim3(256), 0, st, S, first, count, out);
            };
            if (flags & HM_ROWS) tail(Y, n, w.ytail);
            if (flags & HM_COLS) tail(X, m, w.xtail);
            HM_LAUNCH_CHECK("norm_tail");
        }
        auto seeds = [&](const Seeding& s) {
            if (kind == HM_COST_L1) return norm_seeds<HM_COST_L1>(st, s, d, k);
            if (kind == HM_COST_LINF) return norm_seeds<HM_COST_LINF>(st, s, d, k);
            return norm_seeds<HM_COST_L2>(st, s, d, k);
        };
        if (w.rseeds)
            if (int rc = seeds(Seeding{X, {Y, w.ytail, tail_start(n, d)}, m, n, f, g, w.rseeds})) return rc;
        if (w.cseeds)
            if (int rc = seeds(Seeding{Y, {X, w.xtail, tail_start(m, d)}, n, m, g, f, w.cseeds})) return rc;
    }
    ColArgs none{};
    ColArgs cols{};
    if (fused) {
        cols.gthr = w.gthr;
        cols.buf = w.buf;
        cols.count = w.count;
        cols.ccount = w.ccount;
        cols.coff = w.coff;
        cols.order = w.order;
        cols.xmaxima = w.maxima + 2;
        cols.seeds = w.cseeds;
        cols.cap = w.cap;
        cols.n = n;
        hipLaunchKernelGGL(cols_clear, dim3((unsigned)((n + 256) / 256)), dim3(256), 0, st, w.gthr, w.ccount, n, w.count);
        HM_LAUNCH_CHECK("cols_clear");
    }
    if (flags & HM_ROWS) {
        const Direction D{X, Y, w.ytail, w.rseeds, m, n, f, g, w.maxima, (flags & HM_STATS) != 0, false, norm_plan(m, n, d, k, flags),
                          row_val, row_idx, fused ? cols : none, nullptr, 0};
        if (int rc = dispatch(D)) return rc;
    }
    if (fused) {
        prof_begin(st, "norm_cols");
        const unsigned long long* const kth = w.gthr + (k == 1 ? 0 : n);
        hipLaunchKernelGGL(cols_count, dim3(2048), dim3(256), 0, st, w.buf, w.count, w.cap, kth, w.ccount);
        HM_LAUNCH_CHECK("cols_count");
        HM_HIP(hipcub::DeviceScan::ExclusiveSum(w.scan_tmp, w.scan_bytes, w.ccount, w.coff, (int)(n + 1), st));
        hipLaunchKernelGGL(cols_group, dim3(2048), dim3(256), 0, st, w.buf, w.count, w.cap, kth, w.coff, w.ccount,
                           w.order);
        HM_LAUNCH_CHECK("cols_group");
        hipLaunchKernelGGL((cols_select<2>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, w.buf, w.count, w.cap,
                           w.coff, w.order, n, k, col_val, col_idx);
        HM_LAUNCH_CHECK("cols_select");
        prof_end(st);
        if (profiling()) {  // candidates appended (a count above the capacity means the buffer overflowed)
            unsigned long long c = 0;
            HM_HIP(hipMemcpyAsync(&c, w.count, sizeof(c), hipMemcpyDeviceToHost, st));
            HM_HIP(hipStreamSynchronize(st));
            prof_count("norm_cols_candidates", (int64_t)c);
            prof_count(c > (unsigned long long)w.cap ? "norm_cols_overflow" : "norm_cols_fused", 1);
        }
    }
    if (flags & HM_COLS) {
        // the role-swapped sweep; in a fused call it runs only if the candidate buffer overflowed
        const Direction D{Y, X, w.xtail, w.cseeds, n, m, g, f, w.maxima + 2, false, true, norm_plan(n, m, d, k, flags), col_val, col_idx, none,
                          fused ? w.count : nullptr, w.cap};
        if (int rc = dispatch(D)) return rc;
    }
    return HM_OK;
}

// Scratch of the allocation-free entry point: one array per GPU, for the life of the process. Host code reaches it
// only through the device address hipGetSymbolAddress returns (looked up once per device, under a lock).
constexpr size_t NORM_SCRATCH_BYTES = size_t(64) << 20;
// The lists get all of them: beyond them there is room for the padded copies of the sides' last rows, which grow with d
// alone, for the certificate partials (40 bytes a workgroup of 256 rows or 128, whose lists take at least 12 k each, k > 16
// for 128: at most 5/384 of the lists' bytes, and one workgroup more for each of 64 segments), and for alignment.
constexpr size_t NORM_ROOM_BYTES = size_t(2) * (2 * NT * REG_FEATURES + PAD) * sizeof(float) +
                                   NORM_SCRATCH_BYTES / 384 * 5 + 64 * 40 + 2048;
__device__ __align__(256) unsigned char scratch[NORM_SCRATCH_BYTES + NORM_ROOM_BYTES];
inline size_t noalloc_room(int64_t m, int64_t n, int d, int k, uint32_t flags) {
    return (tail_floats(n, d) + tail_floats(m, d)) * sizeof(float) +
           blockstats_doubles(norm_plan(m, n, d, k, flags), m, flags, 0) * sizeof(double) + 2048;
}
constexpr int SCRATCH_DEVICES = 64;
std::mutex scratch_lock;
void* scratch_address[SCRATCH_DEVICES] = {};

int scratch_for_current_device(void** out) {
    int dev = -1;
    HM_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= SCRATCH_DEVICES) return fail(HM_EINVAL, "norm pricing (no-alloc): device %d out of range", dev);
    std::lock_guard<std::mutex> hold(scratch_lock);
    if (scratch_address[dev] == nullptr) {
        void* p = nullptr;
        HM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (p == nullptr) return fail(HM_EHIP, "norm pricing (no-alloc): no device address for the scratch array");
        scratch_address[dev] = p;
    }
    *out = scratch_address[dev];
    return HM_OK;
}

}  // namespace

extern "C" int hm_pricing_norm(void* stream, const float* X, const float* Y, const double* f, const double* g,
                               int64_t m, int64_t n, int32_t d, int32_t k, int32_t kind, uint32_t flags,
                               double* row_val, int32_t* row_idx, double* col_val, int32_t* col_idx, double* stats,
                               void* workspace, size_t workspace_bytes) {
    return norm_scan_run(stream, X, Y, f, g, m, n, d, k, kind, flags, row_val, row_idx, col_val, col_idx, stats,
                         workspace, workspace_bytes, true);
}

extern "C" size_t hm_pricing_norm_noalloc_max_bytes(void) { return NORM_SCRATCH_BYTES; }

extern "C" int hm_pricing_norm_noalloc(void* stream, const float* X, const float* Y, const double* f,
                                       const double* g, int64_t m, int64_t n, int32_t d, int32_t k, int32_t kind,
                                       uint32_t flags, double* row_val, int32_t* row_idx, double* col_val,
                                       int32_t* col_idx, double* stats) {
    HM_CHECK_ARG(m >= 1 && n >= 1 && k >= 1 && k <= 32, "norm pricing requires nonempty inputs and 1 <= k <= 32");
    if (int rc = check_features(d, flags)) return rc;
    // the two-sweep path's scratch; the fused path runs when its larger scratch fits as well
    const size_t bytes = NORM_SCRATCH_BYTES + std::min(noalloc_room(m, n, d, k, flags), NORM_ROOM_BYTES);
    const size_t need = norm_workspace(m, n, d, k, flags, false, 0);
    if (need > bytes)
        return fail(HM_ENOSPC, "norm pricing (no-alloc): this call needs %zu bytes of scratch, above the %zu-byte static "
                               "scratch array; call hm_pricing_norm with a workspace instead",
                    need, NORM_SCRATCH_BYTES);
    void* scratch_ptr = nullptr;
    if (int rc = scratch_for_current_device(&scratch_ptr)) return rc;
    const ProfileOff no_events;  // timing events would be created on demand
    // the fused path only with its full candidate buffer: a partial one that overflows would cost both sweeps
    return norm_scan_run(stream, X, Y, f, g, m, n, d, k, kind, flags, row_val, row_idx, col_val, col_idx, stats,
                         scratch_ptr, bytes, false);
}
