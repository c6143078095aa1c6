// SDDMM cost evaluation on the active support (gfx950).
//
// l2^2: out[e] = (p_i + q_j) - scale*dot64(x_i, y_j)  (costs/pairs.py:394-407 association; gpu_resident/cost.py:59-71)
// norms: fp64 l1 / linf / l2 of (x_i - y_j)           (norm_cost_scan_kernel.cu:233-245, without perturbation)
//
// dot64 / norm partials use the fixed 64-lane order: lane l accumulates features l, l+64, ... sequentially
// and the lanes are combined by a halving-stride tree. For d <= G (G a power of two <= 64) a group of G
// lanes per pair produces the same bits: the missing lanes only ever add +0.0.
#include "common.h"

namespace hm {
namespace {

// Pair costs gather a row (or two) per pair: what bounds them is how much of a row a wave asks for at a time.
// Rows that are 16-byte aligned (d a multiple of 4) are read 16 bytes at a time: 16 lanes per pair, a wave four pairs,
// lane t of the 16 accumulating features 4 t .. 4 t + 3 of every 64. quad_tree finishes the fixed order: its four
// accumulators are lanes 4 t .. 4 t + 3 of the 64, so strides 32 to 4 are lane strides 8 to 1 and the last two lie
// within a lane. 1.5 million pairs of 2048 features, 12.3 GB of gathered rows: 3.25 -> 1.8 ms (6.8 TB/s, the rate of the
// last-level cache); as 64 lanes of 4 bytes each wave had one pair's rows in flight.
__device__ __forceinline__ double quad_tree_sum(double (&a)[4]) {
#pragma unroll
    for (int s = 8; s >= 1; s >>= 1)
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = a[c] + __shfl_down(a[c], s, 16);
    a[0] = a[0] + a[2];
    a[1] = a[1] + a[3];
    return a[0] + a[1];
}
__device__ __forceinline__ double quad_tree_max(double (&a)[4]) {
#pragma unroll
    for (int s = 8; s >= 1; s >>= 1)
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] = fmax(a[c], __shfl_down(a[c], s, 16));
    return fmax(fmax(a[0], a[2]), fmax(a[1], a[3]));
}

// the products are exact in fp64, so the fused form rounds like a multiply and an add
__device__ __forceinline__ void quad_fma(double (&a)[4], const float4 x, const float4 y) {
    a[0] = fma((double)x.x, (double)y.x, a[0]);
    a[1] = fma((double)x.y, (double)y.y, a[1]);
    a[2] = fma((double)x.z, (double)y.z, a[2]);
    a[3] = fma((double)x.w, (double)y.w, a[3]);
}

inline bool quad_rows(const float* X, const float* Y, int d) {
    return d % 4 == 0 && ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y)) & 15) == 0;
}

__device__ __forceinline__ double quad_dot64(const float* __restrict__ x, const float* __restrict__ y, int d, int t) {
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    for (int k = 4 * t; k < d; k += 64)
        quad_fma(a, *reinterpret_cast<const float4*>(x + k), *reinterpret_cast<const float4*>(y + k));
    return quad_tree_sum(a);
}

// CSR rows: one wave per row, four entries at a time
__global__ __launch_bounds__(256) void sddmm_quad_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                         const double* __restrict__ p, const double* __restrict__ q,
                                                         const int32_t* __restrict__ rowptr,
                                                         const int32_t* __restrict__ col, int64_t m, int d,
                                                         double scale, double* __restrict__ out) {
    const int lane = threadIdx.x & 63, t = lane & 15, g = lane >> 4;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); row < m; row += waves) {
        const uint32_t e1 = rowptr[row + 1];  // (unsigned: four past the last entry of 2^31 - 1 is still past it)
        uint32_t e = (uint32_t)rowptr[row] + g;
        int32_t next = e < e1 ? col[e] : 0;
        for (; e < e1; e += 4) {
            const int64_t j = next;
            if (e + 4 < e1) next = col[e + 4];
            const double dot = quad_dot64(X + row * (int64_t)d, Y + j * (int64_t)d, d, t);
            if (t == 0) out[e] = (p[row] + q[j]) - scale * dot;
        }
    }
}

// COO pairs
__global__ __launch_bounds__(256) void pair_costs_quad_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                              const double* __restrict__ p, const double* __restrict__ q,
                                                              const int64_t* __restrict__ rows,
                                                              const int64_t* __restrict__ cols, int64_t count, int d,
                                                              double scale, double* __restrict__ out) {
    const int t = threadIdx.x & 15;
    const int64_t quads = (int64_t)gridDim.x * 16;
    for (int64_t e = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4); e < count; e += quads) {
        const int64_t i = rows[e], j = cols[e];
        const double dot = quad_dot64(X + i * d, Y + j * d, d, t);
        if (t == 0) out[e] = (p[i] + q[j]) - scale * dot;
    }
}

// CSR rows: one wave per row, x_i cached in registers when d <= 64*XR.
template <int XR>
__global__ __launch_bounds__(256) void sddmm_l2sq_csr_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                             const double* __restrict__ p, const double* __restrict__ q,
                                                             const int32_t* __restrict__ rowptr,
                                                             const int32_t* __restrict__ col, int64_t m, int d,
                                                             double scale, double* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); row < m; row += waves) {
        const float* xr = X + row * (int64_t)d;
        const int32_t e0 = rowptr[row], e1 = rowptr[row + 1];
        if (e0 >= e1) continue;
        const double pi = p[row];
        if (XR > 0) {
            float xv[XR > 0 ? XR : 1];
#pragma unroll
            for (int t = 0; t < XR; ++t) xv[t] = (lane + 64 * t < d) ? xr[lane + 64 * t] : 0.0f;
            // U gathered Y rows in flight per step; each pair keeps the fixed lane order
            constexpr int U = 4;
            int32_t e = e0;
            for (; e1 - e >= U; e += U) {
                const float* yp[U];
                double a[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    yp[u] = Y + (int64_t)col[e + u] * d;
                    a[u] = 0.0;
                }
#pragma unroll
                for (int t = 0; t < XR; ++t) {
                    const int k = lane + 64 * t;
                    if (k < d) {
#pragma unroll
                        for (int u = 0; u < U; ++u) a[u] = a[u] + (double)xv[t] * (double)yp[u][k];
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) a[u] = wave_tree_sum(a[u]);
                if (lane < U) {
                    double mine = a[0];
#pragma unroll
                    for (int u = 1; u < U; ++u)
                        if (lane == u) mine = a[u];
                    const int64_t j = col[e + lane];
                    out[e + lane] = (pi + q[j]) - scale * mine;
                }
            }
            for (; e < e1; ++e) {
                const int64_t j0 = col[e];
                const float* y0 = Y + j0 * d;
                double a0 = 0.0;
#pragma unroll
                for (int t = 0; t < XR; ++t) {
                    const int k = lane + 64 * t;
                    if (k < d) a0 = a0 + (double)xv[t] * (double)y0[k];
                }
                a0 = wave_tree_sum(a0);
                if (lane == 0) out[e] = (pi + q[j0]) - scale * a0;
            }
        } else {
            for (int32_t e = e0; e < e1; ++e) {
                const int64_t j = col[e];
                const double dot = wave_dot64(xr, Y + j * d, d, lane);
                if (lane == 0) out[e] = (pi + q[j]) - scale * dot;
            }
        }
    }
}

template <int G>
__device__ inline double group_tree_sum(double v) {
#pragma unroll
    for (int s = G / 2; s >= 1; s >>= 1) v = v + __shfl_down(v, s, G);
    return v;
}
template <int G>
__device__ inline double group_tree_max(double v) {
#pragma unroll
    for (int s = G / 2; s >= 1; s >>= 1) v = fmax(v, __shfl_down(v, s, G));
    return v;
}

// COO pairs: groups of G lanes per pair (G = 64 handles any d; smaller G only when d <= G).
template <int G>
__global__ __launch_bounds__(256) void pair_costs_l2sq_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                              const double* __restrict__ p, const double* __restrict__ q,
                                                              const int64_t* __restrict__ rows,
                                                              const int64_t* __restrict__ cols, int64_t count, int d,
                                                              double scale, double* __restrict__ out) {
    const int g = threadIdx.x % G;
    const int64_t groups = (int64_t)gridDim.x * (blockDim.x / G);
    for (int64_t e = (int64_t)blockIdx.x * (blockDim.x / G) + threadIdx.x / G; e < count; e += groups) {
        const int64_t i = rows[e], j = cols[e];
        const float* x = X + i * d;
        const float* y = Y + j * d;
        double a = 0.0;
        for (int k = g; k < d; k += 64) a = a + (double)x[k] * (double)y[k];
        a = group_tree_sum<G>(a);
        if (g == 0) out[e] = (p[i] + q[j]) - scale * a;
    }
}

template <int KIND>
__device__ __forceinline__ double norm_term(double a, float x, float y) {
    const double z = (double)x - (double)y;
    return KIND == HM_COST_L1 ? a + fabs(z) : KIND == HM_COST_LINF ? fmax(a, fabs(z)) : a + z * z;
}

template <int KIND>
__global__ __launch_bounds__(256) void pair_costs_norm_quad_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                                   const int64_t* __restrict__ rows,
                                                                   const int64_t* __restrict__ cols, int64_t count, int d,
                                                                   double* __restrict__ out) {
    const int t = threadIdx.x & 15;
    const int64_t quads = (int64_t)gridDim.x * 16;
    for (int64_t e = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4); e < count; e += quads) {
        const float* x = X + rows[e] * d;
        const float* y = Y + cols[e] * d;
        double a[4] = {0.0, 0.0, 0.0, 0.0};
        for (int k = 4 * t; k < d; k += 64) {
            const float4 u = *reinterpret_cast<const float4*>(x + k), v = *reinterpret_cast<const float4*>(y + k);
            a[0] = norm_term<KIND>(a[0], u.x, v.x);
            a[1] = norm_term<KIND>(a[1], u.y, v.y);
            a[2] = norm_term<KIND>(a[2], u.z, v.z);
            a[3] = norm_term<KIND>(a[3], u.w, v.w);
        }
        const double r = (KIND == HM_COST_LINF) ? quad_tree_max(a) : quad_tree_sum(a);
        if (t == 0) out[e] = (KIND == HM_COST_L2) ? sqrt(r) : r;
    }
}

template <int G, int KIND>
__global__ __launch_bounds__(256) void pair_costs_norm_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                              const int64_t* __restrict__ rows,
                                                              const int64_t* __restrict__ cols, int64_t count, int d,
                                                              double* __restrict__ out) {
    const int g = threadIdx.x % G;
    const int64_t groups = (int64_t)gridDim.x * (blockDim.x / G);
    for (int64_t e = (int64_t)blockIdx.x * (blockDim.x / G) + threadIdx.x / G; e < count; e += groups) {
        const float* x = X + rows[e] * d;
        const float* y = Y + cols[e] * d;
        double a = 0.0;
        for (int k = g; k < d; k += 64) {
            const double z = (double)x[k] - (double)y[k];
            if (KIND == HM_COST_L1) a = a + fabs(z);
            else if (KIND == HM_COST_LINF) a = fmax(a, fabs(z));
            else a = a + z * z;
        }
        a = (KIND == HM_COST_LINF) ? group_tree_max<G>(a) : group_tree_sum<G>(a);
        if (g == 0) out[e] = (KIND == HM_COST_L2) ? sqrt(a) : a;
    }
}

// fp32 norm costs exactly as the pricing scan forms them: 32-feature chunks accumulated sequentially in fp32,
// chunk results combined in order, l2 = sqrt in fp64 of the fp32 sum, rounded once to fp32. G lanes per pair, one chunk
// each: the lanes read the rows side by side and each then adds the chunk results in their order.
template <int KIND, int G, bool WIDE>
__global__ __launch_bounds__(256) void pair_costs_norm32_kernel(const float* __restrict__ X, const float* __restrict__ Y,
                                                                const int64_t* __restrict__ rows,
                                                                const int64_t* __restrict__ cols, int64_t count, int d,
                                                                double* __restrict__ out) {
    const int g = threadIdx.x % G;
    const int64_t groups = (int64_t)gridDim.x * (256 / G);
    auto term = [](float part, float a, float b) {
        const float z = a - b;
        return KIND == HM_COST_L1 ? part + fabsf(z) : KIND == HM_COST_LINF ? fmaxf(part, fabsf(z)) : fmaf(z, z, part);
    };
    for (int64_t e = (int64_t)blockIdx.x * (256 / G) + threadIdx.x / G; e < count; e += groups) {
        const float* x = X + rows[e] * d;
        const float* y = Y + cols[e] * d;
        float acc = 0.0f;
        for (int first = 0; first < d; first += 32 * G) {
            const int base = first + 32 * g;
            const int end = base + 32 < d ? base + 32 : d;
            float part = 0.0f;
            if (WIDE) {
                for (int k = base; k < end; k += 4) {
                    const float4 u = *reinterpret_cast<const float4*>(x + k), v = *reinterpret_cast<const float4*>(y + k);
                    part = term(part, u.x, v.x);
                    part = term(part, u.y, v.y);
                    part = term(part, u.z, v.z);
                    part = term(part, u.w, v.w);
                }
            } else {
                for (int k = base; k < end; ++k) part = term(part, x[k], y[k]);
            }
#pragma unroll
            for (int c = 0; c < G; ++c) {
                const float other = G == 1 ? part : __shfl(part, c, G);
                if (first + 32 * c < d) acc = (KIND == HM_COST_LINF) ? fmaxf(acc, other) : acc + other;
            }
        }
        if (g == 0) out[e] = (KIND == HM_COST_L2) ? (double)(float)sqrt((double)acc) : (double)acc;
    }
}

inline int group_for(int d) { return d <= 8 ? 8 : (d <= 16 ? 16 : (d <= 32 ? 32 : 64)); }

inline unsigned grid_for(int64_t items, int per_block) {
    int64_t b = (items + per_block - 1) / per_block;
    if (b > 65536) b = 65536;
    if (b < 1) b = 1;
    return (unsigned)b;
}

}  // namespace
}  // namespace hm

using namespace hm;

extern "C" int hm_sddmm_l2sq_csr(void* stream, const float* X, const float* Y, const double* p, const double* q,
                                 const int32_t* rowptr, const int32_t* col, int64_t m, int64_t nnz, int32_t d,
                                 double scale, double* out) {
    HM_CHECK_ARG(m >= 0 && nnz >= 0 && d >= 1, "SDDMM requires m >= 0, nnz >= 0, d >= 1");
    HM_CHECK_ARG(scale == 1.0 || scale == 2.0, "dot_scale must be exactly 1 or 2");
    if (m == 0 || nnz == 0) return HM_OK;
    HM_CHECK_ARG(X && Y && p && q && rowptr && col && out, "SDDMM: null pointer argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const unsigned grid = grid_for(m, 4);
#define HM_SDDMM(XR) \
    hipLaunchKernelGGL((sddmm_l2sq_csr_kernel<XR>), dim3(grid), dim3(256), 0, st, X, Y, p, q, rowptr, col, m, d, scale, out)
    prof_begin(st, "sddmm_l2sq_csr");
    // from 129 to 512 features a wave per entry with x in registers is level or ahead (262144 rows of 16 entries, d = 256:
    // 0.74 ms and 0.75 in fours, 5.7 TB/s of gathered rows; 105 thousand rows of 20, d = 512: 0.72 and 0.81); elsewhere the
    // fours are (89 thousand rows of 20, d = 600: 1.26 -> 0.84 ms; 120 thousand rows of 20, d = 128: 0.47 -> 0.33)
    if (quad_rows(X, Y, d) && (d <= 128 || d > 512))
        hipLaunchKernelGGL(sddmm_quad_kernel, dim3(grid), dim3(256), 0, st, X, Y, p, q, rowptr, col, m, d, scale, out);
    else if (d <= 64) HM_SDDMM(1);
    else if (d <= 128) HM_SDDMM(2);
    else if (d <= 256) HM_SDDMM(4);
    else if (d <= 512) HM_SDDMM(8);
    else HM_SDDMM(0);
    prof_end(st);
#undef HM_SDDMM
    HM_LAUNCH_CHECK("sddmm_l2sq_csr");
    return HM_OK;
}

extern "C" int hm_pair_costs_l2sq(void* stream, const float* X, const float* Y, const double* p, const double* q,
                                  const int64_t* rows, const int64_t* cols, int64_t count, int32_t d, double scale,
                                  double* out) {
    HM_CHECK_ARG(count >= 0 && d >= 1, "pair costs require count >= 0 and d >= 1");
    HM_CHECK_ARG(scale == 1.0 || scale == 2.0, "dot_scale must be exactly 1 or 2");
    if (count == 0) return HM_OK;
    HM_CHECK_ARG(X && Y && p && q && rows && cols && out, "pair costs: null pointer argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int G = group_for(d);
#define HM_PAIRS(GG)                                                                                            \
    hipLaunchKernelGGL((pair_costs_l2sq_kernel<GG>), dim3(grid_for(count, 256 / GG)), dim3(256), 0, st, X, Y, p, q, \
                       rows, cols, count, d, scale, out)
    // (up to 16 features the groups below use more of their lanes: level; 2 million pairs, d = 24: 0.30 -> 0.27 ms)
    if (d > 16 && quad_rows(X, Y, d))
        hipLaunchKernelGGL(pair_costs_quad_kernel, dim3(grid_for(count, 16)), dim3(256), 0, st, X, Y, p, q, rows, cols,
                           count, d, scale, out);
    else if (G == 8) HM_PAIRS(8);
    else if (G == 16) HM_PAIRS(16);
    else if (G == 32) HM_PAIRS(32);
    else HM_PAIRS(64);
#undef HM_PAIRS
    HM_LAUNCH_CHECK("pair_costs_l2sq");
    return HM_OK;
}

extern "C" int hm_pair_costs_norm(void* stream, const float* X, const float* Y, const int64_t* rows,
                                  const int64_t* cols, int64_t count, int32_t d, int32_t kind, double* out) {
    HM_CHECK_ARG(count >= 0 && d >= 1, "pair costs require count >= 0 and d >= 1");
    HM_CHECK_ARG(kind == HM_COST_L1 || kind == HM_COST_LINF || kind == HM_COST_L2, "unsupported norm cost %d", kind);
    if (count == 0) return HM_OK;
    HM_CHECK_ARG(X && Y && rows && cols && out, "pair costs: null pointer argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int G = group_for(d);
#define HM_NORM(GG, KK)                                                                                           \
    hipLaunchKernelGGL((pair_costs_norm_kernel<GG, KK>), dim3(grid_for(count, 256 / GG)), dim3(256), 0, st, X, Y, rows, \
                       cols, count, d, out)
#define HM_NORM_K(GG)                                   \
    do {                                                \
        if (kind == HM_COST_L1) HM_NORM(GG, HM_COST_L1);     \
        else if (kind == HM_COST_LINF) HM_NORM(GG, HM_COST_LINF); \
        else HM_NORM(GG, HM_COST_L2);                        \
    } while (0)
    // (up to 32 features the groups below are ahead: 2 million pairs, l1, d = 24: 0.24 ms and 0.27 in fours; d = 40: 0.38 and 0.27)
    if (d > 32 && quad_rows(X, Y, d)) {
#define HM_NORM_QUAD(KK)                                                                                               \
    hipLaunchKernelGGL((pair_costs_norm_quad_kernel<KK>), dim3(grid_for(count, 16)), dim3(256), 0, st, X, Y, rows, cols, \
                       count, d, out)
        if (kind == HM_COST_L1) HM_NORM_QUAD(HM_COST_L1);
        else if (kind == HM_COST_LINF) HM_NORM_QUAD(HM_COST_LINF);
        else HM_NORM_QUAD(HM_COST_L2);
#undef HM_NORM_QUAD
    } else if (G == 8) HM_NORM_K(8);
    else if (G == 16) HM_NORM_K(16);
    else if (G == 32) HM_NORM_K(32);
    else HM_NORM_K(64);
#undef HM_NORM_K
#undef HM_NORM
    HM_LAUNCH_CHECK("pair_costs_norm");
    return HM_OK;
}

extern "C" int hm_pair_costs_norm_fp32(void* stream, const float* X, const float* Y, const int64_t* rows,
                                       const int64_t* cols, int64_t count, int32_t d, int32_t kind, double* out) {
    HM_CHECK_ARG(count >= 0 && d >= 1, "pair costs require count >= 0 and d >= 1");
    HM_CHECK_ARG(kind == HM_COST_L1 || kind == HM_COST_LINF || kind == HM_COST_L2, "unsupported norm cost %d", kind);
    if (count == 0) return HM_OK;
    HM_CHECK_ARG(X && Y && rows && cols && out, "pair costs: null pointer argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool wide = quad_rows(X, Y, d);
#define HM_NORM32(KK, GG)                                                                                            \
    do {                                                                                                             \
        if (wide)                                                                                                    \
            hipLaunchKernelGGL((pair_costs_norm32_kernel<KK, GG, true>), dim3(grid_for(count, 256 / GG)), dim3(256), \
                               0, st, X, Y, rows, cols, count, d, out);                                              \
        else                                                                                                         \
            hipLaunchKernelGGL((pair_costs_norm32_kernel<KK, GG, false>), dim3(grid_for(count, 256 / GG)),           \
                               dim3(256), 0, st, X, Y, rows, cols, count, d, out);                                   \
    } while (0)
#define HM_NORM32_K(GG)                                         \
    do {                                                        \
        if (kind == HM_COST_L1) HM_NORM32(HM_COST_L1, GG);      \
        else if (kind == HM_COST_LINF) HM_NORM32(HM_COST_LINF, GG); \
        else HM_NORM32(HM_COST_L2, GG);                         \
    } while (0)
    // a lane per chunk, up to 16 (a thread per pair read rows 4 bytes at a time, a line apart from its neighbours): 200
    // thousand pairs of 4096 features 12.4 -> 3.5 ms, 2 million of 64 0.71 -> 0.23
    if (d <= 32) HM_NORM32_K(1);
    else if (d <= 128) HM_NORM32_K(4);
    else HM_NORM32_K(16);
#undef HM_NORM32_K
#undef HM_NORM32
    HM_LAUNCH_CHECK("pair_costs_norm_fp32");
    return HM_OK;
}
