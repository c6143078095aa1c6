// Restricted-OT Halpern-PDHG on gfx950.
//
// Algorithm: _native/cpp/solver.cpp:39-378 (= _internal/lp/torch_restricted_ot.py:105-393; the same update
// CuPDLPx runs in cupdlpx/solver.cu:581-715): degree-sqrt constraint scaling, variable scale sqrt(2),
// constant step 0.998, reflected Halpern iterations, PID primal-weight restarts and relative L2 KKT checks
// every `evaluation_frequency` iterations.
//
// Device layout: the per-edge primal state is mirrored in two orders so that both halves of an iteration
// stream their edges contiguously and never gather per-edge values.
//   source order (position p): edges sorted by source, ascending caller edge id within a source (stable
//     sort), so source i owns [off[i], off[i+1]); perm[p] = caller edge id. Arrays: col, row, scaled cost cs,
//     iterate x, anchor ax, PDHG point px (stored only when the next iteration evaluates), checkpoint delta dx.
//   target order (slot k): edges sorted by target, ascending caller edge id within a target, so target t owns
//     [off[n+t]-e, off[n+t+1]-e). Arrays: row_t, cs_t, x_t, ax_t, px_t.
// Both copies receive identical operands in identical order and therefore stay bit-identical.
// Per node (sources then targets): scale, bs, ns, y, ay, py, dy, and dual = y / ns in several buffers: an iteration reads
// the duals of one and writes the next ones to the other.
//
// One iteration is one launch: the restatement's two loops (source nodes, then target nodes) both start from the duals
// of the previous iteration, so with the next duals going to another buffer nothing orders them, and the workgroups of
// both sides run together:
//   source side: per source node, its edges' PDHG step and reflection, their iterates (Halpern), and the node's
//                dual from the in-order sum of the reflections;
//   target side: per target node, the same steps for its edges from the mirrored state, and its dual from its
//                in-order sum.
// Each side runs in one of two shapes, chosen per solve from the side's largest degree: G-lane groups per node
// (lanes sum in edge order through shuffles) when every node fits in one chunk of the group, else node blocks
// (edge-parallel steps, then one thread per node sums its reflections in edge order from LDS). Both are
// bit-identical to a sequential sum.
// The only gathers are of duals. Scalars read back to the host only at evaluations and checkpoints. Between them, a
// problem that fits the chip runs its iterations in one launch (see "resident runs").
//
// Node numbering: on large problems (at least HELLOOT_PDHG_REORDER nodes, default 2^20, where the duals outgrow
// an XCD's L2) the nodes are renumbered inside the solve so that nodes joined by many edges get nearby numbers:
// each node's position is a few rounds of neighbour averaging from pseudo-random target values (integer arithmetic,
// so the numbering is the same on every run), then each side is sorted by it. On HELLO's supports, which join a
// point to its near neighbours, this groups the support's clusters and the dual gathers hit L2 (1.6x faster
// iterations at 1.28M x 1.28M than with shuffled numbers). A node's edges keep ascending caller ids, so every
// per-node and per-edge operation is unchanged; only the orders of the global norm sums differ.
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "common.h"

namespace hm {
namespace {

constexpr int RB = 1024;     // blocks of the fixed-shape reductions
constexpr int RT = 256;      // threads per reduction block
constexpr int RESIDENT_T = 256;        // threads per workgroup of a resident run of iterations
constexpr int RESIDENT_BLOCKS = 1024;  // its most workgroups

struct Pdhg {
    int64_t n, nt, nodes, e;
    double variable;  // the variables' scale, sqrt(2)
    // edges, source order
    int32_t *row, *col, *perm;
    double *cs, *x, *ax, *px, *dx;
    // edges, target order
    int32_t *row_t, *col_t;
    double *cs_t, *x_t, *ax_t, *px_t;
    // node-block passes: each edge's own node within its block (the low bits of row / col_t; blocks hold a power
    // of two of consecutive nodes), one byte per edge instead of the four-byte node number
    uint8_t *loc_s, *loc_t;
    // node-block passes: the other side's node each edge gathers from (col / row_t) as a 16-bit offset from its
    // block's smallest one, when the block's edges span fewer than 65536 nodes of that side (gbase = that
    // smallest node); else, up to 2^24 nodes, as one word with the own node's byte (gbase = PACKED; the words take the
    // place of keys_in, which the incidence sort has read); else gbase = -1 and the pass reads the 4-byte number and the byte
    uint16_t *g16_s, *g16_t;
    int32_t *gbase_s, *gbase_t;
    // nodes
    double *scale, *bs, *ns, *y, *ay, *py, *dy;
    double* dual[3];
    int32_t *deg, *off, *eid;
    // node numbering (map_s / map_t: internal number of a caller source / target, or null for the identity;
    // inv: caller node of an internal node, sources then targets) and its scratch
    int32_t *map_s, *map_t, *inv, *odeg;
    uint32_t* ov;
    unsigned long long *osum, *okeys_in, *okeys_out;
    void* osort_tmp;
    size_t osort_tmp_bytes;
    // sort scratch
    uint32_t *keys_in, *keys_out;
    int32_t *vals_in;
    void* sort_tmp;
    size_t sort_tmp_bytes;
    // reductions
    double* partial;   // RB * 4
    double* result;    // 4
    int* flag;         // 1
    int32_t* part;     // resident runs: first node of each workgroup
};

template <class A>
void pdhg_layout(A& a, int64_t n, int64_t nt, int64_t e, size_t sort_tmp, size_t osort_tmp, Pdhg& P) {
    const int64_t nodes = n + nt, side = n > nt ? n : nt;
    P.row = a.template take<int32_t>(e);
    P.col = a.template take<int32_t>(e);
    P.perm = a.template take<int32_t>(e);
    P.cs = a.template take<double>(e);
    P.x = a.template take<double>(e);
    P.ax = a.template take<double>(e);
    P.px = a.template take<double>(e);
    P.dx = a.template take<double>(e);
    P.row_t = a.template take<int32_t>(e);
    P.col_t = a.template take<int32_t>(e);
    P.cs_t = a.template take<double>(e);
    P.x_t = a.template take<double>(e);
    P.ax_t = a.template take<double>(e);
    P.px_t = a.template take<double>(e);
    P.loc_s = a.template take<uint8_t>(e);
    P.loc_t = a.template take<uint8_t>(e);
    P.g16_s = a.template take<uint16_t>(e);
    P.g16_t = a.template take<uint16_t>(e);
    P.gbase_s = a.template take<int32_t>(n + 1);
    P.gbase_t = a.template take<int32_t>(nt + 1);
    P.scale = a.template take<double>(nodes);
    P.bs = a.template take<double>(nodes);
    P.ns = a.template take<double>(nodes);
    P.y = a.template take<double>(nodes);
    P.ay = a.template take<double>(nodes);
    P.py = a.template take<double>(nodes);
    P.dy = a.template take<double>(nodes);
    P.dual[0] = a.template take<double>(nodes);
    P.deg = a.template take<int32_t>(nodes + 1);
    P.off = a.template take<int32_t>(nodes + 1);
    P.eid = a.template take<int32_t>(2 * e);
    P.keys_in = a.template take<uint32_t>(2 * e);
    P.keys_out = a.template take<uint32_t>(2 * e);
    P.vals_in = a.template take<int32_t>(2 * e);
    P.sort_tmp = a.template take<char>(sort_tmp > 0 ? sort_tmp : 1);
    P.sort_tmp_bytes = sort_tmp;
    P.partial = a.template take<double>((size_t)RB * 4);
    P.result = a.template take<double>(5);
    P.part = a.template take<int32_t>(RESIDENT_BLOCKS + 2);
    P.dual[2] = a.template take<double>(nodes <= (int64_t)RESIDENT_BLOCKS * RESIDENT_T ? nodes : 1);
    P.flag = a.template take<int>(4);
    P.map_s = a.template take<int32_t>(n);
    P.map_t = a.template take<int32_t>(nt);
    P.inv = a.template take<int32_t>(nodes);
    P.odeg = a.template take<int32_t>(nodes);
    P.ov = a.template take<uint32_t>(nodes);
    P.osum = a.template take<unsigned long long>(nodes);
    P.dual[1] = reinterpret_cast<double*>(P.osum);  // the numbering is done before the first iteration writes it
    P.okeys_in = a.template take<unsigned long long>(side);
    P.okeys_out = a.template take<unsigned long long>(side);
    P.osort_tmp = a.template take<char>(osort_tmp > 0 ? osort_tmp : 1);
    P.osort_tmp_bytes = osort_tmp;
}

inline int end_bit_for(int64_t nodes) {
    int b = 1;
    while (b < 32 && (int64_t(1) << b) < nodes) ++b;
    return b;
}

inline size_t sort_tmp_bytes(int64_t nodes, int64_t e) {
    size_t bytes = 0;  // a size query: it only writes `bytes`
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr,
                                             (const int32_t*)nullptr, (int32_t*)nullptr, (int)(2 * e), 0,
                                             end_bit_for(nodes));
    return bytes;
}

// key of a node in the numbering sort: position (32 bits) above the node's side-local number (31 bits)
constexpr int ORDER_KEY_BITS = 63;

inline size_t order_sort_tmp_bytes(int64_t n, int64_t nt) {
    size_t bytes = 0;  // a size query: it only writes `bytes`
    (void)hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, (const unsigned long long*)nullptr,
                                            (unsigned long long*)nullptr, (int)(n > nt ? n : nt), 0,
                                            ORDER_KEY_BITS);
    return bytes;
}

// smallest node count whose solve renumbers its nodes (HELLOOT_PDHG_REORDER: a count, or "off")
inline int64_t reorder_min_nodes() {
    const char* v = std::getenv("HELLOOT_PDHG_REORDER");
    if (v == nullptr || *v == 0) return int64_t(1) << 20;
    if (std::strcmp(v, "off") == 0) return INT64_MAX;
    char* end = nullptr;
    const long long t = std::strtoll(v, &end, 10);
    return (end && *end == 0 && t >= 0) ? (int64_t)t : (int64_t(1) << 20);
}

constexpr int ORDER_ROUNDS = 6;  // neighbour-averaging rounds (each: sources from targets, then targets)

// ---------------------------------------------------------------------------------------------------------
// setup kernels
// ---------------------------------------------------------------------------------------------------------
// Per node block (one workgroup each): the range of the other side's nodes its edges gather from, and when it spans
// fewer than 65536 nodes, each edge's gathered node as an offset from the smallest, else with `others` up to 2^24 nodes
// there the gathered node above the edge's own node in the block (Pdhg::g16_*, gbase_*). The
// block's edges are [off[b * npb] - ebase, off[min((b + 1) * npb, nodes)] - ebase).
constexpr int32_t PACKED = -2;
__global__ __launch_bounds__(256) void k_gather_base(const int32_t* __restrict__ off, int64_t nodes, int npb,
                                                     int32_t ebase, int64_t others, const int32_t* __restrict__ gidx,
                                                     const uint8_t* __restrict__ loc, int32_t* __restrict__ gbase,
                                                     uint16_t* __restrict__ g16, uint32_t* __restrict__ pack) {
    __shared__ int32_t smin[256], smax[256];
    const int64_t b = blockIdx.x;
    const int64_t n0 = b * npb, n1 = n0 + npb < nodes ? n0 + npb : nodes;
    const int32_t e0 = off[n0] - ebase, e1 = off[n1] - ebase;
    int32_t lo = INT32_MAX, hi = INT32_MIN;
    for (int32_t p = e0 + (int32_t)threadIdx.x; p < e1; p += 256) {
        const int32_t g = gidx[p];
        lo = g < lo ? g : lo;
        hi = g > hi ? g : hi;
    }
    smin[threadIdx.x] = lo;
    smax[threadIdx.x] = hi;
    __syncthreads();
    for (int w = 128; w >= 1; w >>= 1) {
        if ((int)threadIdx.x < w) {
            smin[threadIdx.x] = smin[threadIdx.x + w] < smin[threadIdx.x] ? smin[threadIdx.x + w] : smin[threadIdx.x];
            smax[threadIdx.x] = smax[threadIdx.x + w] > smax[threadIdx.x] ? smax[threadIdx.x + w] : smax[threadIdx.x];
        }
        __syncthreads();
    }
    lo = smin[0];
    hi = smax[0];
    const bool narrow = e1 > e0 && (int64_t)hi - (int64_t)lo < 65536;
    const bool packed = others <= (int64_t)1 << 24;
    if (threadIdx.x == 0) gbase[b] = narrow ? lo : packed ? PACKED : -1;
    if (narrow) {
        for (int32_t p = e0 + (int32_t)threadIdx.x; p < e1; p += 256) g16[p] = (uint16_t)(gidx[p] - lo);
    } else if (packed) {
        for (int32_t p = e0 + (int32_t)threadIdx.x; p < e1; p += 256) pack[p] = (uint32_t)gidx[p] << 8 | loc[p];
    }
}

// low bits of each edge's node number (its index within a node block of mask + 1 nodes)
__global__ void k_low_bits(const int32_t* __restrict__ node, int64_t e, int32_t mask, uint8_t* __restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = (uint8_t)(node[i] & mask);
}

__global__ void k_fill_i32(int32_t* p, int64_t count, int32_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// sums[key] += v over the wave's lanes with key >= 0, called by whole waves. Supports come with their edges in source order,
// so neighbouring lanes often hold the same key, and their atomics to one word would queue: where the wave has few runs of
// equal keys each run is summed by shuffles and added once (integers: the sums are the same). 12 million edges in source
// order, 23 to a source: 685 us with an atomic per edge.
template <typename T>
__device__ __forceinline__ void add_runs(T* __restrict__ sums, int64_t key, T v) {
    const int lane = threadIdx.x & 63;
    const int64_t left = __shfl_up(key, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || key != left);
    if (__popcll(heads) > 24) {
        if (key >= 0) atomicAdd(&sums[key], v);
        return;
    }
    const int first = 63 - __clzll(heads & (~0ull >> (63 - lane)));  // the lane where this lane's run begins
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T u = __shfl_up(v, o, 64);
        if (lane - o >= first) v += u;
    }
    const bool last = lane == 63 || ((heads >> (lane + 1)) & 1ull);
    if (last && key >= 0) atomicAdd(&sums[key], v);
}

// validation, degrees and the (node key, caller edge id) pairs of the incidence sort
__global__ void k_edges(const int64_t* __restrict__ rows, const int64_t* __restrict__ cols, int64_t e, int64_t n,
                        int64_t nt, const int32_t* __restrict__ map_s, const int32_t* __restrict__ map_t,
                        int32_t* __restrict__ deg, uint32_t* __restrict__ keys, int32_t* __restrict__ vals,
                        int* __restrict__ flag) {
    const int lane = threadIdx.x & 63;
    for (int64_t j0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; j0 < e; j0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = j0 + lane;
        int64_t ri = -1, ci = -1;
        if (j < e) {
            const int64_t r = rows[j], c = cols[j];
            if (r < 0 || r >= n || c < 0 || c >= nt) {
                atomicOr(flag, 1);
                keys[j] = 0;
                keys[e + j] = (uint32_t)n;
            } else {
                ri = map_s ? map_s[r] : r;
                ci = n + (map_t ? map_t[c] : c);
                keys[j] = (uint32_t)ri;
                keys[e + j] = (uint32_t)ci;
            }
            vals[j] = (int32_t)j;
            vals[e + j] = (int32_t)j;
        }
        add_runs(deg, ri, 1);
        add_runs(deg, ci, 1);
    }
}

// flag[1] / flag[2] = largest source / target degree (flag[1..2] start at 0)
__global__ void k_degree_max(const int32_t* __restrict__ deg, int64_t n, int64_t nodes, int* __restrict__ flag) {
    int ms = 0, mt = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nodes; i += (int64_t)gridDim.x * blockDim.x) {
        if (i < n) ms = deg[i] > ms ? deg[i] : ms;
        else mt = deg[i] > mt ? deg[i] : mt;
    }
    for (int o = 32; o >= 1; o >>= 1) {
        ms = max(ms, __shfl_xor(ms, o, 64));
        mt = max(mt, __shfl_xor(mt, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        if (ms > 0) atomicMax(&flag[1], ms);
        if (mt > 0) atomicMax(&flag[2], mt);
    }
}

// After the stable sort eid[0..e) lists caller edge ids by source and eid[e..2e) by target.
__global__ void k_source_setup(const int32_t* __restrict__ eid, int64_t e, const int64_t* __restrict__ rows,
                               const int64_t* __restrict__ cols, const double* __restrict__ c,
                               const double* __restrict__ x0, double bound, double objective, double variable,
                               Pdhg P) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < e; p += (int64_t)gridDim.x * blockDim.x) {
        const int32_t j = eid[p];
        P.perm[p] = j;
        P.row[p] = P.map_s ? P.map_s[rows[j]] : (int32_t)rows[j];
        P.col[p] = P.map_t ? P.map_t[cols[j]] : (int32_t)cols[j];
        P.cs[p] = c[j] * objective / variable;
        const double a = x0 ? fmax(x0[j], 0.0) * variable * bound : 0.0;
        P.ax[p] = a;
        P.x[p] = a;
        P.px[p] = a;
        P.dx[p] = 0.0;
    }
}

__global__ void k_target_setup(const int32_t* __restrict__ eid, int64_t e, const int64_t* __restrict__ rows,
                               const int64_t* __restrict__ cols, const double* __restrict__ c,
                               const double* __restrict__ x0, double bound, double objective, double variable,
                               Pdhg P) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < e; k += (int64_t)gridDim.x * blockDim.x) {
        const int32_t j = eid[e + k];
        P.row_t[k] = P.map_s ? P.map_s[rows[j]] : (int32_t)rows[j];
        P.col_t[k] = P.map_t ? P.map_t[cols[j]] : (int32_t)cols[j];
        P.cs_t[k] = c[j] * objective / variable;
        const double a = x0 ? fmax(x0[j], 0.0) * variable * bound : 0.0;
        P.ax_t[k] = a;
        P.x_t[k] = a;
        P.px_t[k] = a;
    }
}

// Exclusive scan of deg[0..nodes) into off[0..nodes]: each workgroup scans `per` nodes, 1024 at a time, from the total of
// the workgroups before it (part, of k_scan_sums; unused by a single workgroup). Latency bounds a scan by one workgroup
// (1.8 ms at 2^20 nodes, each thread walking a run of its own), hence many above SCAN_ONE nodes.
constexpr int SCAN_BLOCKS = 256;
constexpr int64_t SCAN_ONE = 16384;  // up to here a second launch costs more than 16 rounds of one workgroup

__global__ __launch_bounds__(1024) void k_scan_sums(const int32_t* __restrict__ deg, int64_t nodes, int64_t per,
                                                    int64_t* __restrict__ part) {
    __shared__ int64_t sums[16];
    const int64_t b0 = blockIdx.x * per, b1 = (b0 + per < nodes) ? b0 + per : nodes;
    int64_t s = 0;
    for (int64_t i = b0 + threadIdx.x; i < b1; i += 1024) s += deg[i];
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        s = 0;
        for (int w = 0; w < 16; ++w) s += sums[w];
        part[blockIdx.x] = s;
    }
}

__global__ __launch_bounds__(1024) void k_scan(const int32_t* __restrict__ deg, int64_t nodes, int64_t per,
                                               const int64_t* __restrict__ part, int32_t* __restrict__ off) {
    __shared__ int64_t sums[2][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t b0 = blockIdx.x * per, b1 = (b0 + per < nodes) ? b0 + per : nodes;
    if (b0 > 0 && b0 >= nodes) return;
    int64_t run = threadIdx.x < blockIdx.x ? part[threadIdx.x] : 0;  // (SCAN_BLOCKS <= 1024)
    for (int o = 32; o >= 1; o >>= 1) run += __shfl_xor(run, o, 64);
    if (lane == 0) sums[1][wave] = run;
    __syncthreads();
    run = 0;
    for (int w = 0; w < 16; ++w) run += sums[1][w];
    int at = 0;
    for (int64_t i0 = b0; i0 < b1; i0 += 1024, at ^= 1) {
        const int64_t i = i0 + threadIdx.x;
        const int64_t own = i < b1 ? deg[i] : 0;
        int64_t v = own;
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t u = __shfl_up(v, o, 64);
            if (lane >= o) v += u;
        }
        if (lane == 63) sums[at][wave] = v;
        __syncthreads();  // (the other set is rewritten only after the next barrier)
        int64_t before = run;
        for (int w = 0; w < 16; ++w) {
            const int64_t t = sums[at][w];
            if (w < wave) before += t;
            run += t;
        }
        if (i < b1) off[i] = (int32_t)(before + v - own);
    }
    if (b1 == nodes && threadIdx.x == 0) off[nodes] = (int32_t)run;
}

__global__ void k_node_setup(const int32_t* __restrict__ deg, const double* __restrict__ b,
                             const double* __restrict__ y0, const int32_t* __restrict__ inv, int64_t nodes,
                             double bound, double objective, double variable, double* __restrict__ scale,
                             double* __restrict__ bs, double* __restrict__ ns, double* __restrict__ y,
                             double* __restrict__ ay, double* __restrict__ py, double* __restrict__ dy,
                             double* __restrict__ dual) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nodes; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t o = inv ? inv[i] : i;  // the caller's number of internal node i
        const double sc = sqrt((double)(deg[i] > 1 ? deg[i] : 1));
        scale[i] = sc;
        bs[i] = b[o] * bound / sc;
        const double nsv = variable * sc;
        ns[i] = nsv;
        const double a = y0 ? y0[o] * sc * objective : 0.0;
        ay[i] = a;
        y[i] = a;
        py[i] = a;
        dy[i] = 0.0;
        dual[i] = a / nsv;
    }
}

// ---------------------------------------------------------------------------------------------------------
// node numbering (large problems): positions from neighbour averaging, then a sort of each side
// ---------------------------------------------------------------------------------------------------------
// validation and the caller-numbered degrees
__global__ void k_order_degrees(const int64_t* __restrict__ rows, const int64_t* __restrict__ cols, int64_t e,
                                int64_t n, int64_t nt, int32_t* __restrict__ odeg, int* __restrict__ flag) {
    const int lane = threadIdx.x & 63;
    for (int64_t j0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; j0 < e; j0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = j0 + lane;
        const int64_t r = j < e ? rows[j] : -1, c = j < e ? cols[j] : -1;
        const bool ok = r >= 0 && r < n && c >= 0 && c < nt;
        if (!ok && j < e) atomicOr(flag, 1);
        add_runs(odeg, ok ? r : -1, 1);
        add_runs(odeg, ok ? n + c : -1, 1);
    }
}

// targets start from pseudo-random 32-bit positions (a 64-bit mix of the target number), sources from 0
__global__ void k_order_seed(uint32_t* __restrict__ ov, int64_t n, int64_t nodes) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nodes; i += (int64_t)gridDim.x * blockDim.x) {
        uint64_t z = (uint64_t)(i - n) + 0x9E3779B97F4A7C15ull;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        ov[i] = i < n ? 0u : (uint32_t)(z >> 32);
    }
}

__global__ void k_order_clear(unsigned long long* __restrict__ osum, int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        osum[i] = 0ull;
}

// integer sums of the other side's positions over each node's edges (exact, so independent of the order)
__global__ void k_order_gather(const int64_t* __restrict__ rows, const int64_t* __restrict__ cols, int64_t e,
                               int64_t n, int to_sources, const uint32_t* __restrict__ ov,
                               unsigned long long* __restrict__ osum) {
    const int lane = threadIdx.x & 63;
    for (int64_t j0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x - lane; j0 < e; j0 += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = j0 + lane;
        const int64_t r = j < e ? rows[j] : -1, c = j < e ? n + cols[j] : -1;
        const int64_t from = to_sources ? c : r;
        add_runs(osum, to_sources ? r : c, from >= 0 ? (unsigned long long)ov[from] : 0ull);
    }
}

// mean position of nodes [lo, hi) (a node without edges keeps its position)
__global__ void k_order_mean(const unsigned long long* __restrict__ osum, const int32_t* __restrict__ odeg,
                             int64_t lo, int64_t hi, uint32_t* __restrict__ ov) {
    for (int64_t i = lo + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < hi; i += (int64_t)gridDim.x * blockDim.x)
        if (odeg[i] > 0) ov[i] = (uint32_t)(osum[i] / (unsigned long long)odeg[i]);
}

// sort keys of nodes [lo, lo + count): position, then side-local number
__global__ void k_order_keys(const uint32_t* __restrict__ ov, int64_t lo, int64_t count,
                             unsigned long long* __restrict__ keys) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < count; k += (int64_t)gridDim.x * blockDim.x)
        keys[k] = ((unsigned long long)ov[lo + k] << 31) | (unsigned long long)k;
}

// rank r of the sorted keys is the internal number of side-local node k: map[k] = r, inv[base + r] = base + k
__global__ void k_order_ranks(const unsigned long long* __restrict__ sorted, int64_t count, int64_t base,
                              int32_t* __restrict__ map, int32_t* __restrict__ inv) {
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < count; r += (int64_t)gridDim.x * blockDim.x) {
        const int64_t k = (int64_t)(sorted[r] & 0x7FFFFFFFull);
        map[k] = (int32_t)r;
        inv[base + r] = (int32_t)(base + k);
    }
}

// ---------------------------------------------------------------------------------------------------------
// fixed-shape reductions: grid RB x RT, grid-stride partial sums, then one block combines RB partials
// ---------------------------------------------------------------------------------------------------------
template <int Q>
__device__ inline void block_reduce_store(double (&v)[Q], double* __restrict__ partial) {
    __shared__ double s[RT / 64][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < Q; ++q)
        for (int o = 32; o >= 1; o >>= 1) v[q] = v[q] + __shfl_xor(v[q], o, 64);
    if (lane == 0)
        for (int q = 0; q < Q; ++q) s[wave][q] = v[q];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int q = 0; q < Q; ++q) {
            double t = s[0][q];
            for (int w = 1; w < RT / 64; ++w) t = t + s[w][q];
            partial[(size_t)blockIdx.x * 4 + q] = t;
        }
}

__global__ void k_combine(const double* __restrict__ partial, double* __restrict__ result, int q) {
    __shared__ double s[RT][4];
    const int t = threadIdx.x;
    double v[4] = {0, 0, 0, 0};
    for (int b = t; b < RB; b += RT)
        for (int k = 0; k < q; ++k) v[k] = v[k] + partial[(size_t)b * 4 + k];
    for (int k = 0; k < 4; ++k) s[t][k] = v[k];
    __syncthreads();
    for (int w = RT / 2; w >= 1; w >>= 1) {
        if (t < w)
            for (int k = 0; k < 4; ++k) s[t][k] = s[t][k] + s[t + w][k];
        __syncthreads();
    }
    if (t == 0)
        for (int k = 0; k < q; ++k) result[k] = s[0][k];
}

__global__ void k_sumsq(const double* __restrict__ a, int64_t count, double* __restrict__ partial) {
    double v[1] = {0.0};
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < count; i += (int64_t)RB * RT) v[0] = v[0] + a[i] * a[i];
    block_reduce_store<1>(v, partial);
}

__global__ void k_diffsq2(const double* __restrict__ a, const double* __restrict__ b, int64_t na,
                          const double* __restrict__ c, const double* __restrict__ d, int64_t nc,
                          double* __restrict__ partial) {
    double v[2] = {0.0, 0.0};
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < na; i += (int64_t)RB * RT) {
        const double t = a[i] - b[i];
        v[0] = v[0] + t * t;
    }
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < nc; i += (int64_t)RB * RT) {
        const double t = c[i] - d[i];
        v[1] = v[1] + t * t;
    }
    block_reduce_store<2>(v, partial);
}

// evaluation: [primal_sq, dobj, dual_sq, pobj]
__global__ void k_evaluate(const Pdhg P, const double* __restrict__ b, const double* __restrict__ c, double variable,
                           double bound, double objective, double* __restrict__ partial) {
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    const double vb = variable * bound;
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < P.nodes; i += (int64_t)RB * RT) {
        double sum = 0.0;
        if (i < P.n) {
            for (int32_t k = P.off[i]; k < P.off[i + 1]; ++k) sum += P.px[k] / vb;
        } else {
            for (int32_t k = P.off[i]; k < P.off[i + 1]; ++k) sum += P.px_t[k - P.e] / vb;
        }
        const double bi = b[P.inv ? P.inv[i] : i];
        const double delta = sum - bi;
        v[0] = v[0] + delta * delta;
        v[1] = v[1] + bi * (P.py[i] / (P.scale[i] * objective));
    }
    for (int64_t j = (int64_t)blockIdx.x * RT + threadIdx.x; j < P.e; j += (int64_t)RB * RT) {
        const int32_t r = P.row[j], cc = P.col[j];
        const double cj = c[P.perm[j]];
        const double score = P.py[r] / (P.scale[r] * objective) + P.py[P.n + cc] / (P.scale[P.n + cc] * objective) - cj;
        const double viol = fmax(score, 0.0);
        v[2] = v[2] + viol * viol;
        v[3] = v[3] + cj * (P.px[j] / vb);
    }
    block_reduce_store<4>(v, partial);
}

// fixed-point error pieces: [movement, dual_movement, interaction]
__global__ void k_fixed_point(const Pdhg P, double* __restrict__ partial) {
    double v[3] = {0.0, 0.0, 0.0};
    for (int64_t j = (int64_t)blockIdx.x * RT + threadIdx.x; j < P.e; j += (int64_t)RB * RT) {
        const double d = P.dx[j];
        const int32_t r = P.row[j], cc = P.col[j];
        v[0] = v[0] + d * d;
        v[2] = v[2] + (P.dy[r] / P.ns[r] + P.dy[P.n + cc] / P.ns[P.n + cc]) * d;
    }
    for (int64_t i = (int64_t)blockIdx.x * RT + threadIdx.x; i < P.nodes; i += (int64_t)RB * RT)
        v[1] = v[1] + P.dy[i] * P.dy[i];
    block_reduce_store<3>(v, partial);
}

// ---------------------------------------------------------------------------------------------------------
// iteration kernels
// ---------------------------------------------------------------------------------------------------------
// Sum of the group's per-lane values in lane order 0..count-1 (every lane of the group gets the same bits as
// a sequential loop over the group's edges).
template <int G>
__device__ inline double group_ordered_sum(double running, double value, int count) {
    if (count == G) {  // a whole group: every shuffle issued before the first add
        double t[G];
#pragma unroll
        for (int u = 0; u < G; ++u) t[u] = __shfl(value, u, G);
#pragma unroll
        for (int u = 0; u < G; ++u) running += t[u];
        return running;
    }
    for (int t = 0; t < count; ++t) running += __shfl(value, t, G);
    return running;
}

// One side of an iteration: its nodes [first, first + count) of the node arrays, its edges in its own order (the
// arrays of Pdhg's source or target half), and the first node of the other side, whose duals its edges gather.
struct Side {
    int64_t first, count, other;
    int32_t ebase;          // position of the side's first edge in off
    const int32_t* gidx;    // the other side's node of each edge
    const double *cs, *ax;
    double *x, *px, *dx;    // dx: the source side alone (the checkpoint deltas of the edges)
    const uint8_t* loc;
    const uint16_t* g16;
    const uint32_t* pack;
    const int32_t* gbase;
};

// one edge's step: the PDHG point, its reflection and the Halpern iterate (solver.cpp:210-251 order)
template <bool SOURCE, bool CHECKPOINT, bool STORE>
__device__ __forceinline__ double edge_step(const Side& sd, int32_t p, double own, double other, double primal_step,
                                            double halpern, double keep) {
    const double at = SOURCE ? own + other : other + own;
    const double xj = sd.x[p];
    const double pxj = fmax(xj - primal_step * (sd.cs[p] - at), 0.0);
    const double r = 2.0 * pxj - xj;
    if (STORE) sd.px[p] = pxj;
    if (CHECKPOINT && SOURCE) sd.dx[p] = r - xj;
    sd.x[p] = halpern * r + keep * sd.ax[p];
    return r;
}

// ns of a node of `degree` edges, as k_node_setup forms it (a square root less to wait for than a load, and 8 bytes a node
// less for the last-level cache)
__device__ __forceinline__ double node_scale(int32_t degree, double variable) {
    return variable * sqrt((double)(degree > 1 ? degree : 1));
}

// a node's update from the sum of its reflections
template <bool CHECKPOINT, bool STORE>
__device__ __forceinline__ void node_step(const Pdhg& P, int64_t i, int32_t degree, double sum, double dual_step,
                                          double halpern, double keep, double* __restrict__ next) {
    const double yi = P.y[i], nsi = node_scale(degree, P.variable);
    const double pyi = yi - dual_step * (sum / nsi - P.bs[i]);
    const double refl = 2.0 * pyi - yi;
    if (STORE) P.py[i] = pyi;
    if (CHECKPOINT) P.dy[i] = refl - yi;
    const double yn = halpern * refl + keep * P.ay[i];
    P.y[i] = yn;
    next[i] = yn / nsi;
}

constexpr int EB = 2048;  // edges per round of a node block
constexpr int PT = 256;   // threads per workgroup (also the most nodes of a node block)

// Lane groups: a G-lane group per node (block `block` of the side). A chunk covers G*U edges: lane g owns edges g, g+G,
// ..., g+(U-1)G of the chunk, all loaded before any sum.
template <int G, int U, bool SOURCE, bool CHECKPOINT, bool STORE>
__device__ __forceinline__ void group_pass(const Pdhg& P, const Side& sd, int64_t block, const double* __restrict__ cur,
                                           double* __restrict__ next, double primal_step, double dual_step,
                                           double halpern) {
    const double keep = 1.0 - halpern;
    const int g = threadIdx.x % G;
    const int64_t t = block * (PT / G) + threadIdx.x / G;
    if (t >= sd.count) return;
    const int64_t i = sd.first + t;
    const int32_t k0 = P.off[i] - sd.ebase, k1 = P.off[i + 1] - sd.ebase;
    const double own = cur[i];
    double sum = 0.0;
    for (int32_t base = k0; base < k1; base += G * U) {
        double r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t p = base + u * G + g;
            r[u] = 0.0;
            if (p < k1)
                r[u] = edge_step<SOURCE, CHECKPOINT, STORE>(sd, p, own, cur[sd.other + sd.gidx[p]], primal_step, halpern,
                                                            keep);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int32_t left = k1 - (base + u * G);
            if (left > 0) sum = group_ordered_sum<G>(sum, r[u], left < G ? left : G);
        }
    }
    if (g == 0) node_step<CHECKPOINT, STORE>(P, i, k1 - k0, sum, dual_step, halpern, keep, next);
}

// sum + v[a] + v[a+1] + ... + v[b-1], added one by one in that order; the LDS reads go out eight at a time so that
// a long node waits for one read latency per eight values rather than per value.
__device__ __forceinline__ double fold_in_order(const double* v, int a, int b, double sum) {
    int k = a;
    for (; k + 8 <= b; k += 8) {
        double t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = v[k + u];
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += t[u];
    }
    for (; k < b; ++k) sum += v[k];
    return sum;
}

struct BlockLds {
    double refl[EB];
    double dual[PT];
    int32_t off[PT + 1];
};

// Node blocks: a workgroup owns `npb` consecutive nodes of one side and their edges (contiguous in that side's order).
// Edges are processed EB at a time: every thread computes edge steps (coalesced streams, one gather of the other side's
// dual), the reflections go to LDS, and then one thread per node adds its edges' reflections in edge order from LDS,
// carrying its running sum across the rounds. Same operations, operands and order as the lane groups, so the iterates
// are bit-identical; the work per workgroup follows the edges, not the node count, and a node's fold is a run of LDS
// reads instead of lane shuffles.
template <bool SOURCE, bool CHECKPOINT, bool STORE>
__device__ __forceinline__ void block_pass(const Pdhg& P, const Side& sd, int64_t block, int npb,
                                           const double* __restrict__ cur, double* __restrict__ next,
                                           double primal_step, double dual_step, double halpern, BlockLds& lds) {
    const int tid = threadIdx.x;
    const int64_t n0 = sd.first + block * npb;
    const int64_t left = sd.count - block * npb;
    const int nn = (int)(left < npb ? left : npb);
    const double keep = 1.0 - halpern;
    const double* const other = cur + sd.other;
    if (tid < nn) lds.dual[tid] = cur[n0 + tid];
    for (int t = tid; t <= nn; t += PT) lds.off[t] = P.off[n0 + t] - sd.ebase;
    const int32_t gb = sd.gbase[block];  // uniform: 16-bit gather offsets, or -1 for 4-byte numbers
    __syncthreads();
    const int32_t e0 = lds.off[0], e1 = lds.off[nn];
    const int32_t k0 = tid < nn ? lds.off[tid] : 0, k1 = tid < nn ? lds.off[tid + 1] : 0;
    double sum = 0.0;
    for (int32_t base = e0; base < e1; base += EB) {
        const int len = e1 - base < EB ? e1 - base : EB;
        auto step = [&](int q, int l, int32_t c) {
            lds.refl[q] = edge_step<SOURCE, CHECKPOINT, STORE>(sd, base + q, lds.dual[l], other[c], primal_step, halpern, keep);
        };
        if (gb >= 0) {
            for (int q = tid; q < len; q += PT) step(q, sd.loc[base + q], gb + (int32_t)sd.g16[base + q]);
        } else if (gb == PACKED) {
            for (int q = tid; q < len; q += PT) {
                const uint32_t w = sd.pack[base + q];
                step(q, w & 255u, (int32_t)(w >> 8));
            }
        } else {
            for (int q = tid; q < len; q += PT) step(q, sd.loc[base + q], sd.gidx[base + q]);
        }
        __syncthreads();
        sum = fold_in_order(lds.refl, (k0 > base ? k0 : base) - base, (k1 < base + len ? k1 : base + len) - base, sum);
        __syncthreads();
    }
    if (tid < nn) node_step<CHECKPOINT, STORE>(P, n0 + tid, k1 - k0, sum, dual_step, halpern, keep, next);
}

// How one side runs: lane groups of U edges per lane (u > 0), or node blocks (u = 0); its workgroups.
struct SidePlan {
    int u, npb;
    int64_t blocks;
};

constexpr int GL = 8;  // lanes per group

// One PDHG iteration: workgroups [0, src.blocks) run the source side, the rest the target side; workgroup i of the launch is
// number first + step * i. Small problems are bound by the latency of a launch and of each pass's chain of dependent loads
// (offsets, edges, gathered dual, fold), which the two sides now share: 4096 nodes a side and 82 thousand edges take 10.0 us
// an iteration, as two dependent launches they took 11.3.
// Large ones stream the edge state, all of it in each iteration, and whether that fits the last-level cache (256 MB) decides:
// every other iteration runs its workgroups backward, so that it begins with what the last one left there, where a stream in
// one direction has always just lost what it needs next. The second dual buffer had taken 262144 nodes a side of degree 16
// (some 250 MB) over that edge, to 82 to 95 us by placement from 83; backward, without ns and with packed indexes 78 to 85.
// 524288 a side, 12 million edges: 325 -> 301 us, as two launches 330.
template <bool CHECKPOINT, bool STORE>
__global__ __launch_bounds__(PT) void k_iteration(const Pdhg P, SidePlan src, SidePlan tgt, int64_t first, int64_t step,
                                                  const double* __restrict__ cur, double* __restrict__ next, double ps,
                                                  double ds, double h) {
    __shared__ BlockLds lds;
    const int64_t b = first + step * (int64_t)blockIdx.x;
    if (b < src.blocks) {
        const Side sd{0, P.n, P.n, 0, P.col, P.cs, P.ax, P.x, P.px, P.dx, P.loc_s, P.g16_s, P.keys_in, P.gbase_s};
        if (src.u == 0) block_pass<true, CHECKPOINT, STORE>(P, sd, b, src.npb, cur, next, ps, ds, h, lds);
        else if (src.u == 1) group_pass<GL, 1, true, CHECKPOINT, STORE>(P, sd, b, cur, next, ps, ds, h);
        else if (src.u == 2) group_pass<GL, 2, true, CHECKPOINT, STORE>(P, sd, b, cur, next, ps, ds, h);
        else group_pass<GL, 4, true, CHECKPOINT, STORE>(P, sd, b, cur, next, ps, ds, h);
    } else {
        const int64_t bt = b - src.blocks;
        const Side sd{P.n, P.nt, 0, (int32_t)P.e, P.row_t, P.cs_t, P.ax_t, P.x_t, P.px_t, nullptr, P.loc_t, P.g16_t,
                      P.keys_in + P.e, P.gbase_t};
        if (tgt.u == 0) block_pass<false, CHECKPOINT, STORE>(P, sd, bt, tgt.npb, cur, next, ps, ds, h, lds);
        else if (tgt.u == 1) group_pass<GL, 1, false, CHECKPOINT, STORE>(P, sd, bt, cur, next, ps, ds, h);
        else if (tgt.u == 2) group_pass<GL, 2, false, CHECKPOINT, STORE>(P, sd, bt, cur, next, ps, ds, h);
        else group_pass<GL, 4, false, CHECKPOINT, STORE>(P, sd, bt, cur, next, ps, ds, h);
    }
}

// ---------------------------------------------------------------------------------------------------------
// resident runs of iterations
// ---------------------------------------------------------------------------------------------------------
// While the two mirrored copies of the edges, and 8 for each node, fit RESIDENT_BLOCKS workgroups of 2048 less the largest
// degree (resident_plan: 2 e + 8 nodes <= 1024 * (2039 - degree), some 0.6 million edges at a mean degree of 15), the whole
// iteration state fits the chip's registers, and an iteration of separate launches is bound by latency: the launch, then
// offsets, edges, gathered duals, each from memory. A resident run does
// the plain iterations between two checkpoints in one cooperative launch: each workgroup keeps the edges of a run of
// consecutive nodes of one side in registers (iterate, anchor, cost, gathered node) and its nodes' duals in LDS, and
// only the duals that other workgroups gather pass through memory.
//
// There is no grid barrier: a dual is its own signal. Iteration s reads slot s % 3 of the three dual buffers and
// publishes to slot (s + 1) % 3; a slot holds UNPUBLISHED until its node's dual arrives, and a reader repeats its load
// until it sees another value. Every edge is held by both of its ends, so once a workgroup has gathered the duals of
// iteration s, each node it reads has used this workgroup's duals of iteration s - 1: the workgroup then sets them to
// UNPUBLISHED again, waits until that store has reached memory, and publishes. A reader that has seen the new dual can
// therefore only find UNPUBLISHED or a newer dual in the slot it reads next. All loads and stores of duals inside a
// run have agent scope (they bypass the caches of the XCDs). All workgroups have to be on the chip at once: the launch is
// cooperative, and where it is refused the solve goes on with separate launches. Where workgroups wait for one that is not
// there all the same (CUs masked off the process, another process's run), a wait of ResidentSetting::wait ends the run,
// and the solve starts again with separate launches.
//
// Measured, 1000 iterations with set-up and checks, separate launches -> resident: 700 nodes a side and 6.6 thousand edges
// 6.4 -> 3.3 ms, 4096 and 82 thousand 10.1 -> 4.6, 16384 and 328 thousand 12.9 -> 9.3, 24000 and 480 thousand 17.5 -> 13.5,
// where the gathers that bypass the caches (some 50 per ns) bound it; at 4096 nodes an iteration with a grid barrier instead
// of the signals took 6 us, with a release fence that writes back L2 14.
constexpr long long UNPUBLISHED = 0x7FF85E1DE0000001ll;  // a NaN that no operation returns

// HELLOOT_PDHG_RESIDENT: "off" for separate launches alone, or the ticks of the 100 MHz clock a wait may last (default 2 s)
struct ResidentSetting {
    bool on;
    long long wait;
};
inline ResidentSetting resident_setting() {
    constexpr long long WAIT = 200000000ll;
    const char* v = std::getenv("HELLOOT_PDHG_RESIDENT");
    if (v == nullptr || *v == 0) return {true, WAIT};
    if (std::strcmp(v, "off") == 0) return {false, WAIT};
    char* end = nullptr;
    const long long t = std::strtoll(v, &end, 10);
    return {true, (end && *end == 0 && t >= 0) ? t : WAIT};
}

// part[0..ws]: first source node of each of the ws source workgroups (and n), then part[ws+1..]: the same for the
// targets. Cut at equal weights of a side's nodes in order, a node weighing its degree + k.
__global__ void k_partition(const int32_t* __restrict__ off, int64_t n, int64_t nt, int64_t e, int ws, int wt, int k,
                            int32_t* __restrict__ part) {
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < ws + wt + 2; b += gridDim.x * blockDim.x) {
        const bool source = b <= ws;
        const int64_t count = source ? n : nt, w = source ? ws : wt, j = source ? b : b - ws - 1;
        const int32_t* const o = source ? off : off + n;
        const int64_t first = source ? 0 : e;
        const int64_t goal = (e + k * count) * j / w;
        int64_t lo = 0, hi = count;  // the first node whose weight before it reaches the goal
        while (lo < hi) {
            const int64_t mid = (lo + hi) / 2;
            if ((int64_t)o[mid] - first + k * mid >= goal) hi = mid;
            else lo = mid + 1;
        }
        part[b] = (int32_t)(j == w ? count : lo);
    }
}

// no dual published yet in the two buffers that a resident run writes first
__global__ void k_unpublish(double* __restrict__ a, double* __restrict__ b, int64_t nodes) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nodes; i += (int64_t)gridDim.x * blockDim.x) {
        a[i] = __longlong_as_double(UNPUBLISHED);
        b[i] = __longlong_as_double(UNPUBLISHED);
    }
}

__device__ __forceinline__ bool unpublished(double v) { return __double_as_longlong(v) == UNPUBLISHED; }

// `steps` iterations, none of them a checkpoint, from the duals in `cur`; the last ones end up in the buffer that `steps`
// rotations of (cur, next, spare) bring to the front. Workgroups [0, ws) hold source nodes, the rest target nodes:
// at most RESIDENT_T * K edges and RESIDENT_T nodes each. Same operations, operands and order as k_iteration.
// K = 8 leaves 128 registers a thread (four workgroups on a CU), which it fills.
template <int K>
__global__ __launch_bounds__(RESIDENT_T, K > 4 ? 4 : 1) void k_resident(const Pdhg P, int ws, int steps, int64_t inner,
                                                                      double* cur, double* next, double* spare,
                                                                      double primal_step, double dual_step,
                                                                      long long wait) {
    constexpr int T = RESIDENT_T;
    __shared__ double refl[T * K];
    __shared__ double dual[T];
    __shared__ int late;
    const int tid = threadIdx.x;
    // a workgroup that starts after the others gave up has nobody to wait for
    if (tid == 0) late = __hip_atomic_load(P.result + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0.0;
    __syncthreads();
    if (late) return;
    const bool source = (int)blockIdx.x < ws;
    const int b = source ? blockIdx.x : blockIdx.x + 1;
    const int32_t p0 = P.part[b], p1 = P.part[b + 1];
    const int64_t first = (source ? 0 : P.n) + p0;
    const int nn = p1 - p0;
    const int32_t ebase = source ? 0 : (int32_t)P.e;
    const int32_t e0 = P.off[first] - ebase;
    const int len = P.off[first + nn] - ebase - e0;
    double* const xs = (source ? P.x : P.x_t) + e0;
    const double* const axs = (source ? P.ax : P.ax_t) + e0;
    const double* const css = (source ? P.cs : P.cs_t) + e0;
    const int32_t* const own = (source ? P.row : P.col_t) + e0;
    const int32_t* const far = (source ? P.col : P.row_t) + e0;
    const int32_t other = source ? (int32_t)P.n : 0;
    double x[K], ax[K], cs[K];
    int32_t gi[K], loc[K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int q = u * T + tid;
        const bool in = q < len;
        x[u] = in ? xs[q] : 0.0;
        ax[u] = in ? axs[q] : 0.0;
        cs[u] = in ? css[q] : 0.0;
        loc[u] = in ? own[q] - p0 : 0;
        gi[u] = in ? other + far[q] : 0;
    }
    double y = 0.0, ns = 1.0, bs = 0.0, ay = 0.0;
    int k0 = 0, k1 = 0;
    if (tid < nn) {
        const int64_t i = first + tid;
        y = P.y[i];
        ns = P.ns[i];
        bs = P.bs[i];
        ay = P.ay[i];
        dual[tid] = cur[i];
        k0 = P.off[i] - ebase - e0;
        k1 = P.off[i + 1] - ebase - e0;
    }
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        double g[K];
#pragma unroll
        for (int u = 0; u < K; ++u) {
            g[u] = 0.0;
            if (u * T + tid < len) g[u] = __hip_atomic_load(cur + gi[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const double halpern = double(inner + s + 1) / double(inner + s + 2);
        const double keep = 1.0 - halpern;
        if (s > 0) {
            bool miss = false;
#pragma unroll
            for (int u = 0; u < K; ++u) miss |= unpublished(g[u]);
            if (__any(miss)) {
                const long long from = wall_clock64();
                do {
                    miss = false;
#pragma unroll
                    for (int u = 0; u < K; ++u)
                        if (unpublished(g[u]))
                            g[u] = __hip_atomic_load(cur + gi[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int u = 0; u < K; ++u) miss |= unpublished(g[u]);
                    if (wall_clock64() - from > wait) {
                        late = 1;
                        break;
                    }
                } while (__any(miss));
            }
        }
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const double at = dual[loc[u]] + g[u];
            const double pxj = fmax(x[u] - primal_step * (cs[u] - at), 0.0);
            const double r = 2.0 * pxj - x[u];
            x[u] = halpern * r + keep * ax[u];
            refl[u * T + tid] = r;
        }
        __syncthreads();
        if (late) {
            if (tid == 0) __hip_atomic_store(P.result + 4, 1.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        if (tid < nn) {
            __hip_atomic_store(spare + first + tid, __longlong_as_double(UNPUBLISHED), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
            const double sum = fold_in_order(refl, k0, k1, 0.0);
            const double py = y - dual_step * (sum / ns - bs);
            const double r = 2.0 * py - y;
            y = halpern * r + keep * ay;
            const double d = y / ns;
            dual[tid] = d;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __hip_atomic_store(next + first + tid, unpublished(d) ? __builtin_nan("") : d, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        double* const t = cur;
        cur = next;
        next = spare;
        spare = t;
    }
#pragma unroll
    for (int u = 0; u < K; ++u)
        if (u * T + tid < len) xs[u * T + tid] = x[u];
    if (tid < nn) P.y[first + tid] = y;
}

struct ResidentPlan {
    int k, ws, wt;  // edges per thread (0: separate launches), workgroups of the two sides
};

// Fewest workgroups that surely hold a side. k_partition cuts at equal weights, a node weighing its degree + k, so a
// workgroup's weight stays below its share + the heaviest node; at most RESIDENT_T * k of weight means at most
// RESIDENT_T * k edges and RESIDENT_T nodes.
inline int64_t resident_blocks(int64_t e, int64_t nodes, int max_degree, int k) {
    const int64_t room = (int64_t)RESIDENT_T * k - max_degree - k - 1;
    return room < 1 ? INT32_MAX : (e + k * nodes + room - 1) / room;
}

inline const void* resident_kernel(int k) {
    return k == 2   ? reinterpret_cast<const void*>(k_resident<2>)
           : k == 4 ? reinterpret_cast<const void*>(k_resident<4>)
                    : reinterpret_cast<const void*>(k_resident<8>);
}

// Edges per thread: the fewest that need no more than a workgroup per CU (a second one on the CU shares its gather
// path: at 4096 nodes a side 213 workgroups of 4 edges a thread take 3.3 us an iteration, 433 of 2 take 4.5, 118 of 8
// take 3.8), else 8 if all fit on the chip at once. Larger problems keep the separate launches, whose gathers hit L2:
// the two are level where the chip is full.
inline ResidentPlan resident_plan(int64_t n, int64_t nt, int64_t e, int max_s, int max_t) {
    int device = 0, cus = 0, cooperative = 0, per_cu = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cooperative, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess || !cooperative ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
        return {0, 0, 0};
    for (int k = 2; k <= 8; k *= 2) {
        const int64_t ws = resident_blocks(e, n, max_s, k), wt = resident_blocks(e, nt, max_t, k);
        if (ws + wt > (k < 8 ? cus : RESIDENT_BLOCKS)) continue;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, resident_kernel(k), RESIDENT_T, 0) != hipSuccess) break;
        if (ws + wt <= (int64_t)per_cu * cus) return {k, (int)ws, (int)wt};
    }
    return {0, 0, 0};
}

// shortest run worth its two launches and the load and store of the state (some 30 us; an iteration saves 3 to 5)
constexpr int64_t RESIDENT_STEPS = 16;
constexpr int64_t RESIDENT_MOST = 4096;  // keeps a launch under some 50 ms

// REFUSED: the runtime did not take the cooperative launch; `cur` and the state are as they were.
constexpr int REFUSED = -1;
int launch_resident(hipStream_t st, const Pdhg& P, const ResidentPlan& rp, int steps, int64_t inner, double* cur,
                    double* next, double* spare, double ps, double ds, long long wait) {
    hipLaunchKernelGGL(k_unpublish, dim3(64), dim3(256), 0, st, next, spare, P.nodes);
    HM_LAUNCH_CHECK("k_unpublish");
    Pdhg p = P;
    int ws = rp.ws;
    void* args[] = {&p, &ws, &steps, &inner, &cur, &next, &spare, &ps, &ds, &wait};
    if (hipLaunchCooperativeKernel(resident_kernel(rp.k), dim3(rp.ws + rp.wt), dim3(RESIDENT_T), args, 0, st) != hipSuccess) {
        (void)hipGetLastError();
        return REFUSED;
    }
    prof_count(rp.k == 2 ? "pdhg_resident_2" : rp.k == 4 ? "pdhg_resident_4" : "pdhg_resident_8", 1);
    return HM_OK;
}

__global__ void k_restart(const Pdhg P, double* __restrict__ dual) {
    const int64_t total = P.e > P.nodes ? P.e : P.nodes;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < total; j += (int64_t)gridDim.x * blockDim.x) {
        if (j < P.e) {
            const double v = P.px[j];
            P.ax[j] = v;
            P.x[j] = v;
            const double vt = P.px_t[j];
            P.ax_t[j] = vt;
            P.x_t[j] = vt;
        }
        if (j < P.nodes) {
            const double v = P.py[j];
            P.ay[j] = v;
            P.y[j] = v;
            dual[j] = v / P.ns[j];
        }
    }
}

__global__ void k_output(const Pdhg P, double vb, double objective, double* __restrict__ xo, double* __restrict__ yo) {
    const int64_t total = P.e > P.nodes ? P.e : P.nodes;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < total; j += (int64_t)gridDim.x * blockDim.x) {
        if (j < P.e) xo[P.perm[j]] = P.px[j] / vb;
        if (j < P.nodes) yo[P.inv ? P.inv[j] : j] = P.py[j] / (P.scale[j] * objective);
    }
}

inline unsigned grid_of(int64_t items) {
    int64_t b = (items + 255) / 256;
    if (b > 8192) b = 8192;
    if (b < 1) b = 1;
    return (unsigned)b;
}

inline int edges_per_lane(int64_t e, int64_t nodes) {
    const int64_t mean = (e + nodes - 1) / nodes;
    return mean <= GL ? 1 : (mean <= 12 ? 2 : 4);
}

// nodes per workgroup of a node-block pass: about 2048 workgroups, at most PT nodes each
inline int nodes_per_block(int64_t nodes) {
    int npb = 1;
    while (npb < PT && (int64_t)npb * 2 * 2048 <= nodes) npb *= 2;
    return npb;
}

// Lane groups (U = 1, 2 or 4 from the side's mean degree) when every node of the side fits in one chunk of GL * U
// edges: each lane then holds at most U independent edges and no group waits for a longer neighbour. Otherwise node
// blocks, whose work follows the edges (on the supports of the HELLO levels, where degrees spread to several times
// their mean, they take 27-32% less time per iteration; on uniform degree 16 the lane groups are 8% faster).
inline SidePlan side_plan(int64_t e, int64_t nodes, int max_degree) {
    const int u = edges_per_lane(e, nodes);
    SidePlan sp{max_degree <= GL * u ? u : 0, nodes_per_block(nodes), 0};
    const int per = sp.u == 0 ? sp.npb : PT / GL;
    sp.blocks = (nodes + per - 1) / per;
    return sp;
}

// One PDHG iteration from the duals of `cur` to those of `next`. px / py are stored only on major iterations: they are
// read only by the evaluation that follows one.
int launch_iteration(hipStream_t st, const Pdhg& P, const SidePlan& src, const SidePlan& tgt, const double* cur,
                     double* next, bool backward, bool checkpoint, bool major, double ps, double ds, double h) {
    // (a launch of 2^32 threads or more runs some of them; the lane groups take 8 a node)
    constexpr int64_t MOST = (int64_t)UINT32_MAX / PT;
    const int64_t blocks = src.blocks + tgt.blocks;
    const int64_t step = backward ? -1 : 1;
    for (int64_t done = 0; done < blocks; done += MOST) {
        const int64_t first = backward ? blocks - 1 - done : done;
        const dim3 grid((unsigned)(blocks - done < MOST ? blocks - done : MOST)), block(PT);
        if (major)
            hipLaunchKernelGGL((k_iteration<true, true>), grid, block, 0, st, P, src, tgt, first, step, cur, next, ps, ds, h);
        else if (checkpoint)
            hipLaunchKernelGGL((k_iteration<true, false>), grid, block, 0, st, P, src, tgt, first, step, cur, next, ps, ds, h);
        else
            hipLaunchKernelGGL((k_iteration<false, false>), grid, block, 0, st, P, src, tgt, first, step, cur, next, ps, ds, h);
    }
    HM_LAUNCH_CHECK("pdhg iteration");
    return HM_OK;
}

// Internal node numbers (see the header): positions by ORDER_ROUNDS rounds of neighbour averaging, then each side
// sorted by (position, caller number). Also validates the endpoints.
int number_nodes(hipStream_t st, const int64_t* rows, const int64_t* cols, int64_t n, int64_t nt, int64_t e,
                 const Pdhg& P) {
    const int64_t nodes = n + nt;
    const unsigned ge = grid_of(e), gn = grid_of(nodes);
    hipLaunchKernelGGL(k_fill_i32, dim3(gn), dim3(256), 0, st, P.odeg, nodes, 0);
    hipLaunchKernelGGL(k_order_degrees, dim3(ge), dim3(256), 0, st, rows, cols, e, n, nt, P.odeg, P.flag);
    HM_LAUNCH_CHECK("k_order_degrees");
    int bad = 0;
    HM_HIP(hipMemcpyAsync(&bad, P.flag, sizeof(int), hipMemcpyDeviceToHost, st));
    HM_HIP(hipStreamSynchronize(st));
    if (bad) return fail(HM_EINVAL, "active-support endpoint index is out of bounds");
    hipLaunchKernelGGL(k_order_seed, dim3(gn), dim3(256), 0, st, P.ov, n, nodes);
    for (int round = 0; round < ORDER_ROUNDS; ++round) {
        for (int to_sources = 1; to_sources >= 0; --to_sources) {
            hipLaunchKernelGGL(k_order_clear, dim3(gn), dim3(256), 0, st, P.osum, nodes);
            hipLaunchKernelGGL(k_order_gather, dim3(ge), dim3(256), 0, st, rows, cols, e, n, to_sources, P.ov, P.osum);
            hipLaunchKernelGGL(k_order_mean, dim3(gn), dim3(256), 0, st, P.osum, P.odeg, to_sources ? 0 : n,
                               to_sources ? n : nodes, P.ov);
        }
    }
    HM_LAUNCH_CHECK("node numbering rounds");
    for (int side = 0; side < 2; ++side) {
        const int64_t lo = side ? n : 0, count = side ? nt : n;
        hipLaunchKernelGGL(k_order_keys, dim3(grid_of(count)), dim3(256), 0, st, P.ov, lo, count, P.okeys_in);
        size_t bytes = P.osort_tmp_bytes;
        HM_HIP(hipcub::DeviceRadixSort::SortKeys(P.osort_tmp, bytes, P.okeys_in, P.okeys_out, (int)count, 0,
                                                 ORDER_KEY_BITS, st));
        hipLaunchKernelGGL(k_order_ranks, dim3(grid_of(count)), dim3(256), 0, st, P.okeys_out, count, lo,
                           side ? P.map_t : P.map_s, P.inv);
    }
    HM_LAUNCH_CHECK("node numbering sort");
    return HM_OK;
}

constexpr int LATE = -2;  // a resident run gave up: its state is lost
int read_result(hipStream_t st, const Pdhg& P, int q, double* host) {
    hipLaunchKernelGGL(k_combine, dim3(1), dim3(RT), 0, st, P.partial, P.result, q);
    HM_LAUNCH_CHECK("k_combine");
    HM_HIP(hipMemcpyAsync(host, P.result, sizeof(double) * 5, hipMemcpyDeviceToHost, st));
    HM_HIP(hipStreamSynchronize(st));
    return host[4] != 0.0 ? LATE : HM_OK;
}

// One solve on validated arguments, from the assembly on; LATE: start again without resident runs (the outputs are
// written at the end alone).
int pdhg_solve(hipStream_t st, const int64_t* rows, const int64_t* cols, const double* costs, const double* masses,
               const double* x0, const double* y0, const hm_pdhg_params* params, double* x_out, double* y_out,
               hm_pdhg_result* result, Pdhg& P, std::chrono::steady_clock::time_point started, ResidentSetting setting) {
    const int64_t n = P.n, nt = P.nt, nodes = P.nodes, e = P.e;
    const int freq = params->evaluation_frequency;
    // ---- LP assembly: node numbers, endpoints, degrees, per-node incident edge lists (ascending edge id) ----
    hipLaunchKernelGGL(k_fill_i32, dim3(grid_of(nodes + 1)), dim3(256), 0, st, P.deg, nodes + 1, 0);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, P.flag, 4, 0);
    hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, st, reinterpret_cast<int32_t*>(P.result + 4), 2, 0);
    if (nodes >= reorder_min_nodes()) {
        if (int rc = number_nodes(st, rows, cols, n, nt, e, P)) return rc;
    } else {
        P.map_s = P.map_t = P.inv = nullptr;  // caller numbers
    }
    hipLaunchKernelGGL(k_edges, dim3(grid_of(e)), dim3(256), 0, st, rows, cols, e, n, nt, P.map_s, P.map_t, P.deg,
                       P.keys_in, P.vals_in, P.flag);
    HM_LAUNCH_CHECK("k_edges");
    hipLaunchKernelGGL(k_degree_max, dim3(grid_of(nodes)), dim3(256), 0, st, P.deg, n, nodes, P.flag);
    HM_LAUNCH_CHECK("k_degree_max");
    int flag[3] = {0, 0, 0};  // out-of-range endpoint, largest source degree, largest target degree
    HM_HIP(hipMemcpyAsync(flag, P.flag, sizeof(flag), hipMemcpyDeviceToHost, st));
    HM_HIP(hipStreamSynchronize(st));
    if (flag[0]) return fail(HM_EINVAL, "active-support endpoint index is out of bounds");
    const int scan_blocks = nodes > SCAN_ONE ? SCAN_BLOCKS : 1;
    const int64_t scan_per = (nodes + scan_blocks - 1) / scan_blocks;
    int64_t* const scan_part = reinterpret_cast<int64_t*>(P.partial);  // (RB * 4 words, free until the first norm)
    if (scan_blocks > 1)
        hipLaunchKernelGGL(k_scan_sums, dim3(scan_blocks), dim3(1024), 0, st, P.deg, nodes, scan_per, scan_part);
    hipLaunchKernelGGL(k_scan, dim3(scan_blocks), dim3(1024), 0, st, P.deg, nodes, scan_per, scan_part, P.off);
    HM_LAUNCH_CHECK("k_scan");
    size_t tmp_bytes = P.sort_tmp_bytes;
    HM_HIP(hipcub::DeviceRadixSort::SortPairs(P.sort_tmp, tmp_bytes, P.keys_in, P.keys_out, P.vals_in, P.eid,
                                              (int)(2 * e), 0, end_bit_for(nodes), st));

    // ---- scaling (solver.cpp:91-110) ----
    double host[5];
    hipLaunchKernelGGL(k_sumsq, dim3(RB), dim3(RT), 0, st, masses, nodes, P.partial);
    HM_LAUNCH_CHECK("k_sumsq");
    if (int rc = read_result(st, P, 1, host)) return rc;
    const double mass_norm = std::sqrt(host[0]);
    hipLaunchKernelGGL(k_sumsq, dim3(RB), dim3(RT), 0, st, costs, e, P.partial);
    HM_LAUNCH_CHECK("k_sumsq");
    if (int rc = read_result(st, P, 1, host)) return rc;
    const double cost_norm = std::sqrt(host[0]);
    const bool rescale = params->rescale != 0;
    const double bound = rescale ? 1.0 / std::max(1.0, mass_norm) : 1.0;
    const double objective = rescale ? 1.0 / std::max(1.0, cost_norm) : 1.0;
    const double variable = P.variable = std::sqrt(2.0);
    // source-order edge state and its target-order mirror
    hipLaunchKernelGGL(k_source_setup, dim3(grid_of(e)), dim3(256), 0, st, P.eid, e, rows, cols, costs, x0, bound,
                       objective, variable, P);
    HM_LAUNCH_CHECK("k_source_setup");
    hipLaunchKernelGGL(k_target_setup, dim3(grid_of(e)), dim3(256), 0, st, P.eid, e, rows, cols, costs, x0, bound,
                       objective, variable, P);
    HM_LAUNCH_CHECK("k_target_setup");
    hipLaunchKernelGGL(k_node_setup, dim3(grid_of(nodes)), dim3(256), 0, st, P.deg, masses, y0, P.inv, nodes, bound,
                       objective, variable, P.scale, P.bs, P.ns, P.y, P.ay, P.py, P.dy, P.dual[0]);
    HM_LAUNCH_CHECK("k_node_setup");
    double weight = 1.0;
    if (!rescale) {
        hipLaunchKernelGGL(k_sumsq, dim3(RB), dim3(RT), 0, st, P.cs, e, P.partial);
        if (int rc = read_result(st, P, 1, host)) return rc;
        const double ncs = std::sqrt(host[0]);
        hipLaunchKernelGGL(k_sumsq, dim3(RB), dim3(RT), 0, st, P.bs, nodes, P.partial);
        if (int rc = read_result(st, P, 1, host)) return rc;
        const double nbs = std::sqrt(host[0]);
        weight = std::max(ncs / std::max(nbs, 1e-16), 1e-16);
    }

    // ---- Halpern PDHG loop (solver.cpp:157-312) ----
    double best_weight = weight, error_sum = 0.0;
    const double inf = INFINITY;
    double best_balance = inf, initial_error = inf, last_trial_error = inf, fixed_error = inf;
    bool restart = false;
    int32_t reason = 0;
    int64_t count = 0, inner = 0, restarts = 0;
    double pobj = 0, dobj = 0, ap = 0, rp = 0, ad = 0, rd = 0, gap = 0;
    int64_t local_count = 0, local_inner = 0;
    int at = 0;  // the dual buffer the next iteration reads
    const unsigned gr = grid_of(e > nodes ? e : nodes);
    const SidePlan src = side_plan(e, n, flag[1]), tgt = side_plan(e, nt, flag[2]);
    static_assert(PT <= 256, "a node's index within its block fits one byte");
    if (src.u == 0) {
        hipLaunchKernelGGL(k_low_bits, dim3(grid_of(e)), dim3(256), 0, st, P.row, e, src.npb - 1, P.loc_s);
        hipLaunchKernelGGL(k_gather_base, dim3((unsigned)((n + src.npb - 1) / src.npb)), dim3(256), 0, st, P.off, n,
                           src.npb, 0, nt, P.col, P.loc_s, P.gbase_s, P.g16_s, P.keys_in);
    }
    if (tgt.u == 0) {
        hipLaunchKernelGGL(k_low_bits, dim3(grid_of(e)), dim3(256), 0, st, P.col_t, e, tgt.npb - 1, P.loc_t);
        hipLaunchKernelGGL(k_gather_base, dim3((unsigned)((nt + tgt.npb - 1) / tgt.npb)), dim3(256), 0, st, P.off + n,
                           nt, tgt.npb, (int32_t)e, n, P.row_t, P.loc_t, P.gbase_t, P.g16_t, P.keys_in + e);
    }
    HM_LAUNCH_CHECK("node-block setup");
    ResidentPlan resident{0, 0, 0};
    if (setting.on) resident = resident_plan(n, nt, e, flag[1], flag[2]);
    if (resident.k > 0) {
        hipLaunchKernelGGL(k_partition, dim3(1), dim3(256), 0, st, P.off, n, nt, e, resident.ws, resident.wt, resident.k,
                           P.part);
        HM_LAUNCH_CHECK("k_partition");
    }
    for (;;) {
        if (local_count % freq == 0) {
            hipLaunchKernelGGL(k_evaluate, dim3(RB), dim3(RT), 0, st, P, masses, costs, variable, bound, objective,
                               P.partial);
            HM_LAUNCH_CHECK("k_evaluate");
            if (int rc = read_result(st, P, 4, host)) return rc;
            count = local_count;
            inner = local_inner;
            ap = std::sqrt(host[0]);
            dobj = host[1];
            ad = std::sqrt(host[2]);
            pobj = host[3];
            rp = ap / (1.0 + mass_norm);
            rd = ad / (1.0 + cost_norm);
            gap = std::fabs(pobj - dobj) / (1.0 + std::fabs(pobj) + std::fabs(dobj));
            const bool finite = std::isfinite(pobj) && std::isfinite(dobj) && std::isfinite(ap) && std::isfinite(rp) &&
                                std::isfinite(ad) && std::isfinite(rd) && std::isfinite(gap);
            const double elapsed = std::chrono::duration<double>(std::chrono::steady_clock::now() - started).count();
            if (!finite || !std::isfinite(weight)) reason = 3;
            else if (rp < params->tol_primal && rd < params->tol_dual && gap < params->tol_objective) reason = 1;
            else if (count >= params->iteration_limit) reason = 2;
            else if (elapsed >= params->time_limit_seconds) reason = 4;
            if (reason != 0) break;
            restart = false;
            if (count == freq) restart = true;
            else if (count > freq)
                restart = inner >= 0.36 * count || fixed_error <= 0.2 * initial_error ||
                          (fixed_error <= 0.5 * initial_error && fixed_error > last_trial_error);
            last_trial_error = fixed_error;
            if (restart) {
                hipLaunchKernelGGL(k_diffsq2, dim3(RB), dim3(RT), 0, st, P.px, P.ax, e, P.py, P.ay, nodes, P.partial);
                HM_LAUNCH_CHECK("k_diffsq2");
                if (int rc = read_result(st, P, 2, host)) return rc;
                const double pd = std::sqrt(host[0]), dd = std::sqrt(host[1]);
                const double ratio = rd / std::max(rp, 1e-300);
                if (pd > 1e-16 && pd < 1e12 && dd > 1e-16 && dd < 1e12 && ratio > 1e-8 && ratio < 1e8) {
                    const double error = std::log(dd) - std::log(pd) - std::log(weight);
                    error_sum = 0.3 * error_sum + error;
                    weight *= std::exp(0.99 * error + 0.01 * error_sum);
                } else {
                    weight = best_weight;
                    error_sum = 0;
                }
                if (rp > 0 && rd > 0) {
                    const double balance = std::fabs(std::log10(rd / rp));
                    if (balance < best_balance) {
                        best_balance = balance;
                        best_weight = weight;
                    }
                }
                inner = 0;
                last_trial_error = inf;
                ++restarts;
                hipLaunchKernelGGL(k_restart, dim3(gr), dim3(256), 0, st, P, P.dual[at]);
                HM_LAUNCH_CHECK("k_restart");
                local_inner = 0;
            }
        }
        const double primal_step = 0.998 / weight;
        const double dual_step = 0.998 * weight;
        const double halpern = double(local_inner + 1) / double(local_inner + 2);
        const bool major = ((local_count + 1) % freq) == 0;
        const bool is_restart = (local_count % freq == 0) && restart;
        const bool checkpoint = major || is_restart;
        // px / py are read only by the evaluation that follows a major iteration
        prof_begin(st, "pdhg_iteration");
        const int64_t plain = freq - 1 - local_count % freq;  // iterations before the next major one
        const int64_t steps = plain < RESIDENT_MOST ? plain : RESIDENT_MOST;
        if (resident.k > 0 && !checkpoint && steps >= RESIDENT_STEPS) {
            const int rc = launch_resident(st, P, resident, (int)steps, local_inner, P.dual[at], P.dual[(at + 1) % 3],
                                           P.dual[(at + 2) % 3], primal_step, dual_step, setting.wait);
            prof_end(st);
            if (rc == REFUSED) {  // separate launches from here on
                resident.k = 0;
                continue;
            }
            if (rc) return rc;
            prof_count("pdhg_iteration", steps - 1);
            at = (int)((at + steps) % 3);
            local_count += steps;
            local_inner += steps;
            continue;
        }
        if (int rc = launch_iteration(st, P, src, tgt, P.dual[at], P.dual[at == 0], (local_count & 1) != 0, checkpoint, major,
                                      primal_step, dual_step, halpern))
            return rc;
        at = at == 0;
        prof_end(st);
        HM_LAUNCH_CHECK("pdhg iteration");
        if (checkpoint) {
            hipLaunchKernelGGL(k_fixed_point, dim3(RB), dim3(RT), 0, st, P, P.partial);
            HM_LAUNCH_CHECK("k_fixed_point");
            if (int rc = read_result(st, P, 3, host)) return rc;
            const double squared = host[0] * weight + host[1] / weight + 2.0 * 0.998 * host[2];
            fixed_error = std::sqrt(std::max(0.0, squared));
            if (is_restart) initial_error = fixed_error;
        }
        ++local_count;
        ++local_inner;
    }
    hipLaunchKernelGGL(k_output, dim3(gr), dim3(256), 0, st, P, variable * bound, objective, x_out, y_out);
    HM_LAUNCH_CHECK("k_output");
    HM_HIP(hipStreamSynchronize(st));
    result->iterations = count;
    result->restarts = restarts;
    result->reason = reason;
    result->pad = 0;
    result->primal_objective = pobj;
    result->dual_objective = dobj;
    result->abs_primal = ap;
    result->rel_primal = rp;
    result->abs_dual = ad;
    result->rel_dual = rd;
    result->rel_gap = gap;
    result->primal_weight = weight;
    result->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - started).count();
    return HM_OK;
}

}  // namespace
}  // namespace hm

using namespace hm;

extern "C" size_t hm_pdhg_workspace_bytes(int64_t n_source, int64_t n_target, int64_t e) {
    if (n_source < 1 || n_target < 1 || e < 1) return 0;
    Sizer s;
    Pdhg P;
    pdhg_layout(s, n_source, n_target, e, sort_tmp_bytes(n_source + n_target, e),
                order_sort_tmp_bytes(n_source, n_target), P);
    return s.used;
}

extern "C" int hm_pdhg_solve(void* stream, const int64_t* rows, const int64_t* cols, const double* costs,
                             const double* masses, const double* x0, const double* y0, int64_t n_source,
                             int64_t n_target, int64_t e, const hm_pdhg_params* params, double* x_out, double* y_out,
                             hm_pdhg_result* result, void* workspace, size_t workspace_bytes) {
    const auto started = std::chrono::steady_clock::now();
    HM_CHECK_ARG(params && result, "PDHG: params and result are required");
    HM_CHECK_ARG(n_source >= 1 && n_target >= 1 && e >= 1, "invalid restricted OT dimensions");
    HM_CHECK_ARG(2 * e < INT32_MAX && n_source + n_target < INT32_MAX, "restricted OT too large for int32 indexing");
    HM_CHECK_ARG(rows && cols && costs && masses && x_out && y_out, "PDHG: null pointer argument");
    const int freq = params->evaluation_frequency;
    HM_CHECK_ARG(freq >= 1 && params->iteration_limit >= 1 && params->time_limit_seconds > 0,
                 "invalid restricted OT dimensions or runtime limits");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int64_t n = n_source, nt = n_target, nodes = n + nt;
    const size_t tmp = sort_tmp_bytes(nodes, e), otmp = order_sort_tmp_bytes(n, nt);
    Sizer sz;
    Pdhg P;
    pdhg_layout(sz, n, nt, e, tmp, otmp, P);
    HM_CHECK_ARG(workspace != nullptr, "workspace is required");
    if (workspace_bytes < sz.used) return fail(HM_ENOSPC, "PDHG workspace too small: %zu < %zu", workspace_bytes, sz.used);
    Arena a(workspace, workspace_bytes);
    pdhg_layout(a, n, nt, e, tmp, otmp, P);
    P.n = n;
    P.nt = nt;
    P.nodes = nodes;
    P.e = e;
    const ResidentSetting setting = resident_setting();
    const Pdhg fresh = P;
    int rc = pdhg_solve(st, rows, cols, costs, masses, x0, y0, params, x_out, y_out, result, P, started, setting);
    if (rc == LATE) {
        prof_count("pdhg_resident_late", 1);
        P = fresh;
        rc = pdhg_solve(st, rows, cols, costs, masses, x0, y0, params, x_out, y_out, result, P, started, {false, 0});
    }
    return rc;
}
