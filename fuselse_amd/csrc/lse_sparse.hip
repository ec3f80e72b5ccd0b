// Sparse probabilistic-circuit sum-layer forward for gfx950: per sum node n
// and batch column b,
//     out[n, b] = log sum_e exp(logw_e + child[c_e, b])
// over the node's edges e, in fp32 or in the IntLSE Q16.16 arithmetic.
//
// Two edge layouts:
//   * CSR (offsets[n] .. offsets[n+1] index child ids and log-parameters);
//   * the pyjuice block layout of the reference (experiment_pyjuice/
//     sparse_float_kernel.cu:40-105, sparse_q16_kernel.cu:61-134): node block
//     j of block_size parents p shares the child ids cids[j, :]; parent p takes
//     weight params[pids[j, e] + p]; it writes node_mars[nids[j] + p, :].
// Node values are [node][batch] rows, so each edge gathers one contiguous
// child row.
//
// Mapping.  CSR layers: csr_fwd_narrow, several nodes per wave, up to 32
// columns; csr_fwd_kernel, a wave per run of nodes and tile of 64, 128 or 256
// columns, its edges one stream.  The block layout (and some Q16.16 CSR
// layers): sparse_kernel, one wave per (node, tile of 64, 128 or 256 columns);
// lane l owns 1, 2 or 4 columns (one vector when the batch is a multiple of it
// and rows are aligned, else strided scalars), edge metadata is held one
// 64-edge window at a time across the lanes and broadcast per edge with
// readlane, and child rows are loaded G = 4 edges at a time into two
// alternating register buffers.
//
// fp32: an online (max, scaled sum) per column with one rescale per group.
// Q16.16: bit-exact with the reference's reduction: ET = 1, 2, 4, 8 chains
// for fan-in <= 8, 16, 32, above (sparse_q16_kernel.cu:161-165), chain et folds
// edges e = et, et + ET, ... in order starting from the identity -0x3fffffff,
// then an xor butterfly over the ET chains; each logit is quantised as
// rne_sat(fmaxf(logw + child, -20000) * 94548.4609375) and a result at or
// below the identity becomes -inf (sparse_q16_kernel.cu:113,129-131).
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/fuselse_amd.h"
#include "fl_status.hpp"
#include "lse_blocked.hpp"
#include "lse_common.hpp"
#include "lse_pair.hpp"

namespace fl {
namespace sparse {

constexpr int kNegInfQ = -0x3fffffff;
constexpr float kConv = 1.44269504089f * 65536.0f;
constexpr float kOutScale = 0.69314718056f / 65536.0f;
constexpr int G = 4;      // edges per load group

__constant__ int kLut[64] = {
       0,  571,  907, 1282, 1634, 1745, 2054, 2592,
    2900, 2859, 2895, 3015, 3222, 3522, 3922, 4426,
    4617, 4441, 4294, 4178, 4093, 4039, 4018, 4030,
    4076, 4157, 4272, 4424, 4613, 4838, 5102, 5404,
    5399, 5068, 4746, 4435, 4134, 3843, 3562, 3291,
    3031, 2781, 2541, 2312, 2094, 1886, 1689, 1502,
    1327, 1162, 1008,  865,  732,  611,  500,  401,
     312,  235,  168,  113,   69,   35,   13,    2,
};

constexpr uint32_t kNegInfU = (uint32_t)kNegInfQ ^ kQBias;

__device__ __forceinline__ uint32_t pair(uint32_t a, uint32_t b, const int* __restrict__ lut) {
    return q16_pair<true>(a, b, lut);
}

__device__ __forceinline__ uint32_t quant(float logit) {
    const float r = __builtin_rintf(fmaxf(logit, -20000.0f) * kConv);
    int q;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));
    return (uint32_t)q ^ kQBias;
}

// Vectors of VW floats and their buffer loads.
template <int VW>
struct Vec;
template <>
struct Vec<4> {
    typedef f32x4 T;
    __device__ static __forceinline__ T load(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    }
};
template <>
struct Vec<2> {
    typedef float T __attribute__((ext_vector_type(2)));
    __device__ static __forceinline__ T load(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
    }
};
template <>
struct Vec<1> {
    typedef float T __attribute__((ext_vector_type(1)));
    __device__ static __forceinline__ T load(__amdgpu_buffer_rsrc_t r, int off) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    }
};

// The PP columns of lane l in the tile of 64*PP columns starting at b0: the
// vectors of VW columns at b0 + 64*VW*q + VW*l (q < PP/VW), each load of the
// wave covering 64*VW contiguous columns of a row.  VW > 1 needs the batch and
// the rows to be whole, aligned vectors, so that none crosses the batch's end.
template <int VW, int PP>
struct Cols {
    static_assert(PP % VW == 0, "columns come in whole vectors");
    __device__ static __forceinline__ bool ok(int64_t b0, int l, int64_t batch, int i) {
        return b0 + 64 * VW * (i / VW) + VW * l < batch;
    }
    __device__ static __forceinline__ void store(float* __restrict__ row, int64_t b0, int l, int64_t batch,
                                                 const float (&v)[PP]) {
#pragma unroll
        for (int q = 0; q < PP / VW; ++q) {
            const int64_t c = b0 + 64 * VW * q + VW * l;
            if (c < batch) {
                typename Vec<VW>::T t;
#pragma unroll
                for (int k = 0; k < VW; ++k) t[k] = v[VW * q + k];
                store_stream<typename Vec<VW>::T>(t, row + c);
            }
        }
    }
};

// Lane-held metadata of edge (window start + lane).
struct EdgeMeta {
    int64_t cid;
    float logw;
};

__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const int lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uint64_t)v);
    const int hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

__device__ __forceinline__ int64_t bcast64(int64_t v, int lane) {
    const int lo = __builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, lane);
    const int hi = __builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), lane);
    return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ float bcastf(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// ---------------------------------------------------------------------------
// Layouts: node(n) returns a wave-uniform descriptor (edge count, output row);
// meta(d, e) the metadata of edge e of that node (called per lane).
// ---------------------------------------------------------------------------
struct CsrDesc {
    int64_t e0, k, n;
};
struct CsrLayout {
    const int64_t* offsets;
    const int32_t* cids;
    const float* logp;
    float* out;
    int64_t batch;
    __device__ __forceinline__ CsrDesc node(int64_t n) const {
        const int64_t e0 = uniform64(offsets[n]);
        return {e0, uniform64(offsets[n + 1]) - e0, n};
    }
    __device__ __forceinline__ EdgeMeta meta(const CsrDesc& d, int64_t e) const {
        return {(int64_t)cids[d.e0 + e], logp[d.e0 + e]};
    }
    __device__ __forceinline__ float* out_row(const CsrDesc& d) const { return out + d.n * batch; }
};

struct BlockDesc {
    int64_t base, k, p, row;
};
template <bool LOGP>
struct BlockLayout {
    float* node_mars;
    const float* params;
    const int64_t* nids;
    const int64_t* cids;
    const int64_t* pids;
    int64_t num_edges, block_size, batch;
    __device__ __forceinline__ BlockDesc node(int64_t jp) const {
        const int64_t j = jp / block_size;
        const int64_t p = jp - j * block_size;
        return {j * num_edges, num_edges, p, uniform64(nids[j]) + p};
    }
    __device__ __forceinline__ EdgeMeta meta(const BlockDesc& d, int64_t e) const {
        const float w = params[pids[d.base + e] + d.p];
        // log of the linear weight with the reference's 1e-45 floor
        // (sparse_float_kernel.cu:76), accurate libm log once per edge
        return {cids[d.base + e], LOGP ? w : logf(fmaxf(w, 1e-45f))};
    }
    __device__ __forceinline__ float* out_row(const BlockDesc& d) const { return node_mars + d.row * batch; }
};

// ---------------------------------------------------------------------------
// Per-node reductions over one tile of 64 * PP columns.
// ---------------------------------------------------------------------------
// The columns of lane l (as Cols<VW, PP>) from the row segment starting at b0
// (`row` points at it), through a buffer resource of `rec` bytes: columns past
// the range read as zeros, without a memory access, and the load needs no
// branch.  The rows are gathered by id, and they take plain loads: with the
// nontemporal hint (which streamed dense rows read faster) the C5 layer's
// forward took 3339 us against 3139, its backward 7046 us against 6169.
template <int VW, int PP>
__device__ __forceinline__ void load_cols_buf(const float* row, int rec, int l, float (&v)[PP]) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, rec, 0x00020000);
#pragma unroll
    for (int q = 0; q < PP / VW; ++q) {
        const typename Vec<VW>::T t = Vec<VW>::load(r, (64 * VW * q + VW * l) * 4);
#pragma unroll
        for (int k = 0; k < VW; ++k) v[VW * q + k] = t[k];
    }
}

// Bytes of a row from column b0 to the batch's end, clamped to a buffer range.
__device__ __forceinline__ int cols_bytes(int64_t batch, int64_t b0) {
    const int64_t left = (batch - b0) * 4;
    return left > 0x7fffffff ? 0x7fffffff : (int)left;
}

// Loads the child rows of window edges j .. j + GS - 1 (edges at or past wn
// are left for the fold to mask).  Every load is issued: each edge's row goes
// through a buffer resource built from its wave-uniform child id, with an
// empty range for edges past wn and the range check covering the batch's end,
// so no load sits behind a branch.  A load behind a branch left the wait-count
// pass unable to count the loads in flight, and the fold of a group then
// waited for the next group's loads as well.
template <int GS, int VW, int PP>
__device__ __forceinline__ void load_group(float (&v)[GS][PP], const EdgeMeta& ew, int j, int wn,
                                           const float* __restrict__ child, int64_t batch, int64_t b0, int l) {
    const int rec = cols_bytes(batch, b0);
#pragma unroll
    for (int g = 0; g < GS; ++g)
        load_cols_buf<VW, PP>(child + bcast64(ew.cid, (j + g) & 63) * batch + b0, j + g < wn ? rec : 0, l, v[g]);
}

template <int PP>
__device__ __forceinline__ void fold_group_f32(const float (&v)[G][PP], const EdgeMeta& ew, int j, int wn,
                                               float (&m)[PP], float (&s)[PP]) {
    float lw[G];
#pragma unroll
    for (int g = 0; g < G; ++g) lw[g] = j + g < wn ? bcastf(ew.logw, j + g) : -kInf;
#pragma unroll
    for (int i = 0; i < PP; ++i) {
        float col[G];
#pragma unroll
        for (int g = 0; g < G; ++g) col[g] = j + g < wn ? v[g][i] + lw[g] : -kInf;
        lse_fold<true, G>(m[i], s[i], col);
    }
}

// Edge g of a group starting at window edge j belongs to chain (j + g) % ET.
// Windows start at multiples of 64 and groups at multiples of G = 4, so for
// ET <= 4 the chain is g % ET, and for ET = 8 it is C0 + g with C0 = j % 8,
// 0 or 4: a wave-uniform choice between two static code paths.
template <int ET, int C0, int P>
__device__ __forceinline__ void fold_group_q16_at(const float (&v)[G][P], const EdgeMeta& ew, int j, int wn,
                                                  uint32_t (&acc)[ET][P], const int* __restrict__ lut) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
        if (j + g < wn) {
            const float lw = bcastf(ew.logw, j + g);
            const int c = (C0 + g) % ET;
#pragma unroll
            for (int i = 0; i < P; ++i) acc[c][i] = pair(acc[c][i], quant(lw + v[g][i]), lut);
        }
    }
}

template <int ET, int P>
__device__ __forceinline__ void fold_group_q16(const float (&v)[G][P], const EdgeMeta& ew, int j, int wn,
                                               uint32_t (&acc)[ET][P], const int* __restrict__ lut) {
    if constexpr (ET == 8) {
        if (j & 4)
            fold_group_q16_at<ET, 4, P>(v, ew, j, wn, acc, lut);
        else
            fold_group_q16_at<ET, 0, P>(v, ew, j, wn, acc, lut);
    } else {
        fold_group_q16_at<ET, 0, P>(v, ew, j, wn, acc, lut);
    }
}

// Walks the node's edges in 64-edge windows; groups of GS edges alternate
// between two register buffers (loads of group g+1 in flight while group g
// folds).  FOLD(buf, j, wn, ew) folds group starting at window edge j.
template <int GS, int VW, int PP, typename LAYOUT, typename DESC, typename FOLD>
__device__ __forceinline__ void walk_edges(const LAYOUT& L, const DESC& d, const EdgeMeta& first,
                                           const float* __restrict__ child, int64_t batch, int64_t b0, int l,
                                           FOLD fold) {
    for (int64_t w0 = 0; w0 < d.k; w0 += 64) {
        const EdgeMeta ew = w0 == 0 ? first : (w0 + l < d.k ? L.meta(d, w0 + l) : EdgeMeta{0, 0.0f});
        const int wn = (int)(d.k - w0 < 64 ? d.k - w0 : 64);
        const int ng = (wn + GS - 1) / GS;
        float va[GS][PP], vb[GS][PP];
        load_group<GS, VW, PP>(va, ew, 0, wn, child, batch, b0, l);
        for (int gi = 0; gi < ng; gi += 2) {
            // the prefetch is unconditional (a group past the window reads
            // empty ranges), keeping every load outside a branch
            load_group<GS, VW, PP>(vb, ew, (gi + 1) * GS, wn, child, batch, b0, l);
            fold(va, gi * GS, wn, ew);
            if (gi + 1 >= ng) break;
            load_group<GS, VW, PP>(va, ew, (gi + 2) * GS, wn, child, batch, b0, l);
            fold(vb, (gi + 1) * GS, wn, ew);
        }
    }
}

template <int VW, int P, typename LAYOUT, typename DESC>
__device__ __forceinline__ void reduce_f32(const LAYOUT& L, const DESC& d, const EdgeMeta& first,
                                           const float* __restrict__ child, int64_t batch, int64_t b0, int l) {
    float m[P], s[P];
#pragma unroll
    for (int i = 0; i < P; ++i) { m[i] = -kInf; s[i] = 0.0f; }
    walk_edges<G, VW, P>(L, d, first, child, batch, b0, l,
                           [&](const float (&v)[G][P], int j, int wn, const EdgeMeta& ew) {
                               fold_group_f32<P>(v, ew, j, wn, m, s);
                           });
    float res[P];
#pragma unroll
    for (int i = 0; i < P; ++i) res[i] = lse_finish<true>(m[i], s[i]);
    Cols<VW, P>::store(L.out_row(d), b0, l, batch, res);
}

template <int ET, int VW, int P, typename LAYOUT, typename DESC>
__device__ __forceinline__ void reduce_q16_et(const LAYOUT& L, const DESC& d, const EdgeMeta& first,
                                              const float* __restrict__ child, int64_t batch, int64_t b0, int l,
                                              const int* __restrict__ lut) {
    uint32_t acc[ET][P];
#pragma unroll
    for (int c = 0; c < ET; ++c)
#pragma unroll
        for (int i = 0; i < P; ++i) acc[c][i] = kNegInfU;
    walk_edges<G, VW, P>(L, d, first, child, batch, b0, l,
                          [&](const float (&v)[G][P], int j, int wn, const EdgeMeta& ew) {
                              fold_group_q16<ET, P>(v, ew, j, wn, acc, lut);
                          });
    float res[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        // xor butterfly over the chains, distances ET/2 .. 1; chain 0 ends with the result
        if constexpr (ET >= 8) {
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[c][i] = pair(acc[c][i], acc[c + 4][i], lut);
        }
        if constexpr (ET >= 4) {
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[c][i] = pair(acc[c][i], acc[c + 2][i], lut);
        }
        if constexpr (ET >= 2) acc[0][i] = pair(acc[0][i], acc[1][i], lut);
        const int q = (int)(acc[0][i] ^ kQBias);
        res[i] = q > kNegInfQ ? (float)q * kOutScale : -kInf;
    }
    Cols<VW, P>::store(L.out_row(d), b0, l, batch, res);
}

template <int VW, int P, typename LAYOUT, typename DESC>
__device__ __forceinline__ void reduce_q16(const LAYOUT& L, const DESC& d, const EdgeMeta& first,
                                           const float* __restrict__ child, int64_t batch, int64_t b0, int l,
                                           const int* __restrict__ lut) {
    if (d.k <= 8)
        reduce_q16_et<1, VW, P>(L, d, first, child, batch, b0, l, lut);
    else if (d.k <= 16)
        reduce_q16_et<2, VW, P>(L, d, first, child, batch, b0, l, lut);
    else if (d.k <= 32)
        reduce_q16_et<4, VW, P>(L, d, first, child, batch, b0, l, lut);
    else
        reduce_q16_et<8, VW, P>(L, d, first, child, batch, b0, l, lut);
}

// One single-wave block per (node, tile of 64 * P columns) pair, pairs numbered
// tile-fastest from pair0.  A block lives exactly as long as its own node's
// edge loop: with four nodes per block, a block held its slot until the
// largest of four power-law fan-ins was done, and the Q16 table needed a block
// barrier (C5: Q16 4.70 -> 3.79 ms, fp32 3.37 -> 3.32 ms).  One wave needs no
// barrier for the table: its LDS operations retire in order.  The pair index
// is block-uniform, so the node's descriptor comes through scalar loads.
template <bool Q16, int VW, int P, typename LAYOUT>
__global__ __launch_bounds__(64) void sparse_kernel(LAYOUT L, const float* __restrict__ child, int64_t batch,
                                                    int64_t items, int64_t tiles, int64_t pair0) {
    __shared__ int lut[64];
    if constexpr (Q16) {
        lut[threadIdx.x] = kLut[threadIdx.x];
        __builtin_amdgcn_wave_barrier();
    }
    const int l = lane_id();
    const int64_t pair = pair0 + blockIdx.x;
    const int64_t item = pair / tiles;
    if (item >= items) return;
    const auto desc = L.node(item);
    const EdgeMeta first = l < desc.k ? L.meta(desc, l) : EdgeMeta{0, 0.0f};
    const int64_t b0 = (pair - item * tiles) * 64 * P;
    if constexpr (Q16)
        reduce_q16<VW, P>(L, desc, first, child, batch, b0, l, lut);
    else
        reduce_f32<VW, P>(L, desc, first, child, batch, b0, l);
}

template <bool Q16, int VW, int P, typename LAYOUT>
static void launch_cols(const LAYOUT& L, const float* child, int64_t items, int64_t batch, hipStream_t st) {
    const int64_t tiles = (batch + 64 * P - 1) / (64 * P);
    for_grid_chunks(items * tiles, 64, [&](int64_t p0, int64_t n) {
        sparse_kernel<Q16, VW, P, LAYOUT><<<dim3((unsigned)n), dim3(64), 0, st>>>(L, child, batch, items, tiles, p0);
    });
}

// Columns per lane by the batch (200000 CSR nodes through this kernel, Q16.16,
// us at 1 / 2 / 4 columns a lane: batch 64 134 / 160 / 242, 100 236 / 164 / 244,
// 256 437 / 286 / 300, 512 923 / 584 / 531).
template <bool Q16, typename LAYOUT>
static void launch(const LAYOUT& L, const float* child, const float* out_any, int64_t items, int64_t batch,
                   hipStream_t st) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(child) | reinterpret_cast<uintptr_t>(out_any);
    if (batch <= 64)
        launch_cols<Q16, 1, 1>(L, child, items, batch, st);
    else if (batch <= 128) {
        if (batch % 2 == 0 && (at & 7) == 0)
            launch_cols<Q16, 2, 2>(L, child, items, batch, st);
        else
            launch_cols<Q16, 1, 2>(L, child, items, batch, st);
    } else if (batch % 4 == 0 && (at & 15) == 0)
        launch_cols<Q16, 4, 4>(L, child, items, batch, st);
    else
        launch_cols<Q16, 1, 4>(L, child, items, batch, st);
}

// ---------------------------------------------------------------------------
// CSR forward: one wave per run of `npw` consecutive nodes and tile of 64 * P
// columns, walking the run's edges as one stream of groups of up to G edges
// (a group never spans two nodes).  The next group's rows are in flight while
// a group folds, across node boundaries too, and the group after that has its
// edge ids and weights on the way through scalar loads, so a node costs no
// round trips of its own: with a wave per node, each paid three in a row
// (offsets, ids, rows).  The tiles go one after the other over all runs, so
// that at any time the gathers stay within one column slice of the children,
// of which the 256 MB Infinity Cache holds a part: a 1M-row, 512-column layer
// (8.0M edges to random rows, fan-in k^-2 on [2, 256], 18.5 GB) went from 3140 us,
// 5.9 TB/s, to 2548 in fp32 and 2599 in Q16.16, 7.3 and 7.1 TB/s (wave per node and
// 256-column tile, tile-fastest -> this).
// ---------------------------------------------------------------------------
// Scalar loads of 4 consecutive words through a buffer resource: words past
// its range read as 0.
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
__device__ u32x4v s_buffer_load4(u32x4v rsrc, int32_t off, int32_t aux) __asm("llvm.amdgcn.s.buffer.load.v4i32");

// Group j.. of a run's node: `left` edges of the node from the run's edge e on,
// of which the group takes the first G.  All of it wave-uniform, in 32-bit
// scalars (64-bit compares and carried booleans would move to vector
// registers).  k: the node's edges.
struct Group {
    int32_t e, node, left, first, k;
};

// Lane i holds the edge at which the run's node i starts, counted from the
// run's first; lanes at and past the run's node count hold the run's end.
struct Run {
    int32_t at;
    __device__ __forceinline__ int32_t start(int node) const { return __builtin_amdgcn_readlane(at, node); }
    __device__ __forceinline__ Group next(const Group& g) const {
        const int32_t last = g.left <= G;
        const int32_t e = g.e + (last ? g.left : G), node = g.node + last;
        const int32_t left = start(node + 1) - e;
        return {e, node, left, last, last ? left : g.k};
    }
};

// Ids and weights of a group's edges; entries past the group's are those of
// following edges, or 0, and are masked by `left`.
struct GroupMeta {
    u32x4v cid, lw;
};
static_assert(G == 4, "a group's ids are one 4-word scalar load");

__device__ __forceinline__ u32x4v words_rsrc(const void* p, int64_t words) {
    const uint64_t a = reinterpret_cast<uintptr_t>(p);
    return {(uint32_t)a, (uint32_t)(a >> 32) & 0xFFFFu, words < 0x1FFFFFFF ? (uint32_t)words * 4u : 0x7FFFFFFCu,
            0x00020000u};
}

// Folds K edges into (m, s) of each column (FIRST: from nothing).  Where every
// column's new maximum is finite and below 2^24 the rescale and the
// exponentials need no special cases (a -inf term is exp2(-inf) = 0, a NaN
// stays NaN); other lanes take lse_fold's robust forms, on the same values.
template <int K, bool FIRST, int P>
__device__ __forceinline__ void fold_edges_f32(const float (&v)[G][P], const float (&lw)[G], float (&m)[P],
                                               float (&s)[P]) {
    float t[P][K], mn[P], top = 0.0f;
#pragma unroll
    for (int i = 0; i < P; ++i) {
#pragma unroll
        for (int g = 0; g < K; ++g) t[i][g] = v[g][i] + lw[g];
        float cm = t[i][0];
#pragma unroll
        for (int g = 1; g < K; ++g) cm = fmaxf(cm, t[i][g]);
        mn[i] = FIRST ? cm : fmaxf(m[i], cm);
        top = fmaxf(top, __builtin_fabsf(mn[i]));
    }
    if (top < 0x1p24f) {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const float nb = -mn[i] * kLog2e;
            float acc = 0.0f;
#pragma unroll
            for (int g = 0; g < K; ++g) acc += lse_exp_fused(t[i][g], nb);
            s[i] = FIRST ? acc : s[i] * fexp2((m[i] - mn[i]) * kLog2e) + acc;
            m[i] = mn[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            if (FIRST) {
                m[i] = -kInf;
                s[i] = 0.0f;
            }
            lse_fold<true, K>(m[i], s[i], t[i]);
        }
    }
}

template <int P>
__device__ __forceinline__ void fold_f32(const float (&v)[G][P], const GroupMeta& em, const Group& g, float (&m)[P],
                                         float (&s)[P]) {
    float lw[G];
#pragma unroll
    for (int k = 0; k < G; ++k) lw[k] = __builtin_bit_cast(float, k < g.left ? (uint32_t)em.lw[k] : 0xFF800000u);
    if (g.first) {
        if (g.left <= 2)
            fold_edges_f32<2, true, P>(v, lw, m, s);
        else
            fold_edges_f32<G, true, P>(v, lw, m, s);
    } else {
        fold_edges_f32<G, false, P>(v, lw, m, s);
    }
}

// The folds over a node's groups: begin() at its first group, add() per group,
// end() after its last.
template <int P>
struct FoldF32 {
    float m[P], s[P];
    __device__ __forceinline__ void add(const float (&v)[G][P], const GroupMeta& em, const Group& g) {
        fold_f32<P>(v, em, g, m, s);
    }
    __device__ __forceinline__ void end(const Group&, float (&res)[P]) const {
#pragma unroll
        for (int i = 0; i < P; ++i) res[i] = lse_finish<true>(m[i], s[i]);
    }
};

// The edge-thread tree of reduce_q16_et over a node's groups; chains by the
// node's fan-in.  A group starts at a multiple of G of its node's edges, so
// with 8 chains its first edge belongs to chain 0 or 4.
template <int P>
struct FoldQ16 {
    uint32_t acc[8][P];
    const int* lut;
    template <int ET, int C0>
    __device__ __forceinline__ void chains(const float (&v)[G][P], const GroupMeta& em, const Group& g) {
#pragma unroll
        for (int e = 0; e < G; ++e) {
            if (e < g.left) {
                const uint32_t w = em.lw[e];
#pragma unroll
                for (int i = 0; i < P; ++i)
                    acc[(C0 + e) % ET][i] =
                        pair(acc[(C0 + e) % ET][i], quant(__builtin_bit_cast(float, w) + v[e][i]), lut);
            }
        }
    }
    __device__ __forceinline__ void add(const float (&v)[G][P], const GroupMeta& em, const Group& g) {
        if (g.first) {
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int i = 0; i < P; ++i) acc[c][i] = kNegInfU;
        }
        if (g.k <= 8)
            chains<1, 0>(v, em, g);
        else if (g.k <= 16)
            chains<2, 0>(v, em, g);
        else if (g.k <= 32)
            chains<4, 0>(v, em, g);
        else if ((g.k - g.left) & 4)
            chains<8, 4>(v, em, g);
        else
            chains<8, 0>(v, em, g);
    }
    // xor butterfly over the chains, distances 4, 2, 1 as far as there are chains
    __device__ __forceinline__ void end(const Group& g, float (&res)[P]) {
        if (g.k > 32) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int i = 0; i < P; ++i) acc[c][i] = pair(acc[c][i], acc[c + 4][i], lut);
        }
        if (g.k > 16) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < P; ++i) acc[c][i] = pair(acc[c][i], acc[c + 2][i], lut);
        }
        if (g.k > 8) {
#pragma unroll
            for (int i = 0; i < P; ++i) acc[0][i] = pair(acc[0][i], acc[1][i], lut);
        }
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int q = (int)(acc[0][i] ^ kQBias);
            res[i] = q > kNegInfQ ? (float)q * kOutScale : -kInf;
        }
    }
};

// Edges of a run that the stream's 32-bit edge numbers and byte offsets hold;
// a run of more walks its nodes one by one with 64-bit ones (walk_edges).
constexpr int64_t kRunEdges = 1 << 20;

template <bool Q16, int P>
struct FoldPick {
    typedef FoldF32<P> T;
};
template <int P>
struct FoldPick<true, P> {
    typedef FoldQ16<P> T;
};
template <bool Q16, int P>
using FoldOf = typename FoldPick<Q16, P>::T;

// The run a block takes.  Workgroups go to the eight XCDs in turn, so of each
// 8 * kXcdRuns consecutive blocks those of one XCD take kXcdRuns consecutive
// runs: neighbouring nodes often share children (a block of parents, a banded
// structure), and each XCD's L2 is its own.  us, in block order -> this: 262144
// nodes, 32 edges, batch 512, 32 neighbours sharing their children, forward 2464
// -> 1094, Q16.16 2472 -> 1587; 8 edges to the nearest 65 children, forward 549
// -> 434, backward 1193 -> 1056; random children, 1M nodes, 7924 -> 7840 both.
// 32 and 64 runs measured the same within 1%.
constexpr int kXcdRuns = 16;
__device__ __forceinline__ int64_t xcd_unit(int64_t u, int64_t total) {
    const int64_t g = u & ~(int64_t)(8 * kXcdRuns - 1);
    const int i = (int)(u - g);
    return g + 8 * kXcdRuns > total ? u : g + (i & 7) * kXcdRuns + (i >> 3);
}

template <bool Q16, int VW, int P, bool SHORT>
__global__ __launch_bounds__(64) void csr_fwd_kernel(const float* __restrict__ child, const int64_t* __restrict__ off,
                                                     const int32_t* __restrict__ cids, const float* __restrict__ logp,
                                                     float* __restrict__ out, int64_t batch, int64_t nodes,
                                                     int npw, int64_t unit0) {
    __shared__ int lut[64];
    FoldOf<Q16, P> state;
    if constexpr (Q16) {
        // one wave needs no barrier for the table: its LDS operations retire in order
        lut[threadIdx.x] = kLut[threadIdx.x];
        __builtin_amdgcn_wave_barrier();
        state.lut = lut;
    }
    const int l = lane_id();
    const int64_t runs = (nodes + npw - 1) / npw;
    const int64_t unit = xcd_unit(unit0 + blockIdx.x, runs * ((batch + 64 * P - 1) / (64 * P)));
    const int64_t tile = unit / runs;
    const int64_t n0 = (unit - tile * runs) * npw;
    const int64_t b0 = tile * 64 * P;
    const int nn = (int)(nodes - n0 < npw ? nodes - n0 : npw);
    const int64_t at = off[n0 + (l < nn ? l : nn)];
    const int64_t e0 = uniform64(at);
    if (bcast64(at, nn) - e0 > kRunEdges) {
        const CsrLayout L{off, cids, logp, out, batch};
        for (int n = 0; n < nn; ++n) {
            const CsrDesc d = L.node(n0 + n);
            const EdgeMeta first = l < d.k ? L.meta(d, l) : EdgeMeta{0, 0.0f};
            if constexpr (Q16)
                reduce_q16<VW, P>(L, d, first, child, batch, b0, l, lut);
            else
                reduce_f32<VW, P>(L, d, first, child, batch, b0, l);
        }
        return;
    }
    const Run run{(int32_t)(at - e0)};
    const int64_t nnz = uniform64(off[nodes]);
    const u32x4v rc = words_rsrc(cids + e0, nnz - e0), rl = words_rsrc(logp + e0, nnz - e0);
    const float* child_b0 = child + b0;
    const uint32_t row_bytes = (uint32_t)batch * 4u;  // launch_csr sends larger rows elsewhere
    const int rec = cols_bytes(batch, b0);
    const auto load_meta = [&](const Group& g) {
        return GroupMeta{s_buffer_load4(rc, g.e * 4, 0), s_buffer_load4(rl, g.e * 4, 0)};
    };
    const auto load_rows = [&](float (&v)[G][P], const GroupMeta& em, const Group& g) {
#pragma unroll
        for (int k = 0; k < G; ++k)
            load_cols_buf<VW, P>(reinterpret_cast<const float*>(reinterpret_cast<const char*>(child_b0) +
                                                                (uint64_t)em.cid[k] * row_bytes),
                                 k < g.left ? rec : 0, l, v[k]);
    };
    const auto fold = [&](const float (&v)[G][P], const GroupMeta& em, const Group& g) {
        state.add(v, em, g);
        if (g.left <= G && g.node < nn) {
            float res[P];
            state.end(g, res);
            Cols<VW, P>::store(out + (n0 + g.node) * batch, b0, l, batch, res);
        }
    };
    // ga, gb: the groups whose rows are in va, vb; the second one's ids (mb)
    // are loaded while the first one's rows are awaited.  Groups past the run
    // load nothing and store nothing: with an exit after the first fold the
    // compiler sinks the ids' loads below it, next to their use.  Runs of one or
    // two groups leave before the loop instead, without its waits for the ids of
    // groups past them (8000 nodes, batch 128, 2 edges 7.9 -> 6.1 us, 5 edges 7.8 ->
    // 7.1); kernels for longer runs (SHORT false) do without the test, which took
    // 20000 nodes, batch 256, 5 edges, two nodes a run from 20.6 to 21.2.
    float va[G][P], vb[G][P];
    Group ga = {0, 0, run.start(1), 1, run.start(1)};
    GroupMeta ma = load_meta(ga);
    load_rows(va, ma, ga);
    Group gb = run.next(ga);
    if (SHORT && gb.node >= nn) {
        fold(va, ma, ga);
        return;
    }
    GroupMeta mb = load_meta(gb);
    if (SHORT && run.next(gb).node >= nn) {
        load_rows(vb, mb, gb);
        fold(va, ma, ga);
        fold(vb, mb, gb);
        return;
    }
    while (true) {
        load_rows(vb, mb, gb);
        const Group gc = run.next(gb);
        const GroupMeta mc = load_meta(gc);
        fold(va, ma, ga);
        load_rows(va, mc, gc);
        const Group gd = run.next(gc);
        const GroupMeta md = load_meta(gd);
        fold(vb, mb, gb);
        if (gc.node >= nn) return;
        ga = gc;
        ma = mc;
        gb = gd;
        mb = md;
    }
}

// ---------------------------------------------------------------------------
// Batches of up to 32 columns: LG lanes (a power of two >= the batch) per node,
// 64 / LG nodes per wave, so a narrow batch does not leave a wave's lanes idle.
// A group folds the edges of its own node, four at a time, up to kOwnEdges of
// them; the wave's groups then take each longer node together, an edge (Q16.16:
// a chain of the node's eight) per group in turn, so that a large fan-in is not
// one group's serial chain.  Loads are unconditional: ids and weights through
// buffer ranges (an edge past the node's reads as id 0), a child row 0 there
// and the last column in idle lanes, all masked after.  Against a wave per run
// of nodes (csr_fwd_kernel with 1 column a lane; us, fp32 / Q16.16 / backward):
// 300000 nodes, batch 4: 137 / 159 / 214 -> 33 / 50 / 142, batch 16 135 / 159 /
// 215 -> 64 / 78 / 167, batch 32 133 / 157 / 214 -> 103 / 126 / 171; 2000 nodes,
// batch 16, where the largest fan-in's chain is the time, 20.9 / 31.8 / 11.6 ->
// 12.4 / 13.6 / 11.8.
// ---------------------------------------------------------------------------
constexpr int64_t kNarrowBatch = 32;
constexpr int kOwnEdges = 32;  // fan-ins of one, two or four Q16.16 chains

// A value of lane (lane ^ mask).
__device__ __forceinline__ float shuffle_xor(float v, int mask) { return __shfl_xor(v, mask, 64); }
__device__ __forceinline__ uint32_t shuffle_xor(uint32_t v, int mask) { return (uint32_t)__shfl_xor((int)v, mask, 64); }

// The edges of the nodes a wave's lane groups hold.  Node: what says where a
// node's edges are; logit(node, i, ok): the lane's column of its edge i, -inf
// where !ok; of_lane(node, j): lane j's, wave-uniform.
// CSR: Node is the node's first edge's place in the wave's run of edges, and ids
// and weights have range checks.
struct CsrNarrow {
    typedef int32_t Node;
    __amdgpu_buffer_rsrc_t ids, lws;
    const float* child;
    int64_t batch;
    int col;
    __device__ __forceinline__ float logit(Node first, int32_t i, bool ok) const {
        const int at = ok ? (first + i) * 4 : 0x7FFFFFFC;
        const uint32_t id = __builtin_amdgcn_raw_buffer_load_b32(ids, at, 0, 0);
        const float lw = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(lws, at, 0, 0));
        const float t = lw + child[(int64_t)id * batch + col];
        return ok ? t : -kInf;
    }
    __device__ __forceinline__ Node of_lane(Node n, int j) const { return __builtin_amdgcn_readlane(n, j); }
};
// Block layout: Node is the parent's number (block * block_size + position); an
// edge past the node's reads the block's first.
template <bool LOGP>
struct BlockNarrow {
    typedef int64_t Node;
    BlockLayout<LOGP> L;
    const float* child;
    int col;
    __device__ __forceinline__ float logit(Node item, int32_t i, bool ok) const {
        const int64_t j = div_small(item, L.block_size);
        const EdgeMeta m = L.meta({j * L.num_edges, L.num_edges, item - j * L.block_size, 0}, ok ? i : 0);
        const float t = m.logw + child[m.cid * L.batch + col];
        return ok ? t : -kInf;
    }
    __device__ __forceinline__ Node of_lane(Node n, int j) const { return bcast64(n, j); }
    __device__ static __forceinline__ int64_t div_small(int64_t a, int64_t b) {
        return ((uint64_t)a | (uint64_t)b) >> 32 ? a / b : (int64_t)((uint32_t)a / (uint32_t)b);
    }
};

// The result of each group's node (k edges, 0 for none) in the group's lanes.
template <bool Q16, int LG, typename EDGES>
__device__ __forceinline__ float reduce_narrow(const EDGES& E, const typename EDGES::Node node, int32_t k,
                                               const int* __restrict__ lut) {
    constexpr int NG = 64 / LG;
    const int l = lane_id();
    const int grp = l / LG, b = l % LG;
    const int32_t own = k <= kOwnEdges ? k : 0;
    uint64_t longer = __ballot(k > kOwnEdges && b == 0);
    if constexpr (Q16) {
        uint32_t a0 = kNegInfU, a1 = kNegInfU, a2 = kNegInfU, a3 = kNegInfU;
        const bool two = own > 8, four = own > 16;  // two or more chains, four
        for (int32_t e = 0; __any(e < own); e += 4) {
            float t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = E.logit(node, e + u, e + u < own);
            // edge u belongs to chain u mod 1, 2 or 4; a masked one leaves its chain
            const auto step = [&](uint32_t acc, int u) {
                const uint32_t r = pair(acc, quant(t[u]), lut);
                return e + u < own ? r : acc;
            };
            a0 = step(a0, 0);
            const uint32_t r1 = step(two ? a1 : a0, 1);
            a0 = two ? a0 : r1;
            a1 = two ? r1 : a1;
            const uint32_t r2 = step(four ? a2 : a0, 2);
            a0 = four ? a0 : r2;
            a2 = four ? r2 : a2;
            const uint32_t r3 = step(four ? a3 : two ? a1 : a0, 3);
            a0 = two ? a0 : r3;
            a1 = two && !four ? r3 : a1;
            a3 = four ? r3 : a3;
        }
        const uint32_t p0 = pair(a0, a2, lut), p1 = pair(a1, a3, lut);
        a0 = four ? p0 : a0;
        a1 = four ? p1 : a1;
        const uint32_t p = pair(a0, a1, lut);
        a0 = two ? p : a0;
        // a longer node's chain grp + NC * i in acc[i]
        constexpr int NC = NG < 8 ? NG : 8, CPG = 8 / NC;
        while (longer) {
            const int j = __builtin_ctzll(longer);
            longer &= longer - 1;
            const typename EDGES::Node nj = E.of_lane(node, j);
            const int32_t kj = __builtin_amdgcn_readlane(k, j);
            uint32_t acc[CPG];
#pragma unroll
            for (int i = 0; i < CPG; ++i) acc[i] = kNegInfU;
            for (int32_t r = 0; r < kj; r += 16) {
                float t[2][CPG];
#pragma unroll
                for (int v = 0; v < 2; ++v)
#pragma unroll
                    for (int i = 0; i < CPG; ++i) {
                        const int32_t e = r + 8 * v + grp + NC * i;
                        t[v][i] = E.logit(nj, e, grp < NC && e < kj);
                    }
#pragma unroll
                for (int v = 0; v < 2; ++v)
#pragma unroll
                    for (int i = 0; i < CPG; ++i) {
                        const uint32_t p = pair(acc[i], quant(t[v][i]), lut);
                        acc[i] = r + 8 * v + grp + NC * i < kj ? p : acc[i];
                    }
            }
            // xor butterfly, distances 4, 2, 1: inside the lane while a
            // chain's partner is there, then across the groups
            if constexpr (CPG == 4) {
                acc[0] = pair(acc[0], acc[2], lut);
                acc[1] = pair(acc[1], acc[3], lut);
            }
            if constexpr (CPG >= 2) acc[0] = pair(acc[0], acc[1], lut);
            if constexpr (CPG == 1) acc[0] = pair(acc[0], shuffle_xor(acc[0], 4 * LG), lut);
            if constexpr (CPG <= 2) acc[0] = pair(acc[0], shuffle_xor(acc[0], 2 * LG), lut);
            acc[0] = pair(acc[0], shuffle_xor(acc[0], LG), lut);
            const uint32_t r = (uint32_t)__shfl((int)acc[0], b, 64);  // group 0's
            a0 = grp == j / LG ? r : a0;
        }
        const int q = (int)(a0 ^ kQBias);
        return q > kNegInfQ ? (float)q * kOutScale : -kInf;
    } else {
        float m = -kInf, s = 0.0f;
        for (int32_t e = 0; __any(e < own); e += 4) {
            float t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = E.logit(node, e + u, e + u < own);
            lse_fold<true, 4>(m, s, t);
        }
        while (longer) {
            const int j = __builtin_ctzll(longer);
            longer &= longer - 1;
            const typename EDGES::Node nj = E.of_lane(node, j);
            const int32_t kj = __builtin_amdgcn_readlane(k, j);
            float mj = -kInf, sum = 0.0f;
            for (int32_t r = 0; r < kj; r += 4 * NG) {
                float t[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) t[u] = E.logit(nj, r + u * NG + grp, r + u * NG + grp < kj);
                lse_fold<true, 4>(mj, sum, t);
            }
            for (int d = LG; d < 64; d <<= 1) {
                const float m2 = shuffle_xor(mj, d), s2 = shuffle_xor(sum, d);
                lse_merge(mj, sum, m2, s2);
            }
            m = grp == j / LG ? mj : m;
            s = grp == j / LG ? sum : s;
        }
        return lse_finish<true>(m, s);
    }
}

template <bool Q16, int LG>
__global__ __launch_bounds__(64) void csr_fwd_narrow(const float* __restrict__ child, const int64_t* __restrict__ off,
                                                     const int32_t* __restrict__ cids, const float* __restrict__ logp,
                                                     float* __restrict__ out, int64_t batch, int64_t nodes,
                                                     int64_t block0) {
    constexpr int NG = 64 / LG;
    __shared__ int lut[64];
    if constexpr (Q16) {
        lut[threadIdx.x] = kLut[threadIdx.x];
        __builtin_amdgcn_wave_barrier();
    }
    const int l = lane_id();
    const int grp = l / LG, b = l % LG;
    const int64_t n0 = (block0 + blockIdx.x) * NG;
    const int64_t n = n0 + grp;
    const int64_t nc = n < nodes ? n : nodes - 1;
    const int64_t start = off[nc], e0 = uniform64(start);
    const int64_t k64 = n < nodes ? off[nc + 1] - start : 0;
    const int64_t total = uniform64(off[n0 + NG < nodes ? n0 + NG : nodes]) - e0;
    float res = -kInf;
    if (total > kRunEdges) {  // beyond 32-bit edge numbers: one edge at a time
        const int64_t col = b < batch ? b : 0;
        if constexpr (Q16) {
            const int et = k64 <= 8 ? 1 : k64 <= 16 ? 2 : k64 <= 32 ? 4 : 8;
            uint32_t acc[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                acc[c] = kNegInfU;
                if (c < et)
                    for (int64_t e = start + c; e < start + k64; e += et)
                        acc[c] = pair(acc[c], quant(logp[e] + child[(int64_t)cids[e] * batch + col]), lut);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (et > 4) acc[c] = pair(acc[c], acc[c + 4], lut);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (et > 2) acc[c] = pair(acc[c], acc[c + 2], lut);
            if (et > 1) acc[0] = pair(acc[0], acc[1], lut);
            const int q = (int)(acc[0] ^ kQBias);
            res = q > kNegInfQ ? (float)q * kOutScale : -kInf;
        } else {
            float m = -kInf, s = 0.0f;
            for (int64_t e = start; e < start + k64; e += 4) {  // groups of four, as the other kernels' sums
                float t[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    t[u] = e + u < start + k64 ? logp[e + u] + child[(int64_t)cids[e + u] * batch + col] : -kInf;
                lse_fold<true, 4>(m, s, t);
            }
            res = lse_finish<true>(m, s);
        }
    } else if (total > 0) {
        const int64_t nnz = uniform64(off[nodes]);
        const int left = (int)(nnz - e0 < kRunEdges * 2 ? nnz - e0 : kRunEdges * 2) * 4;
        const CsrNarrow E{__builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(cids + e0), 0, left, 0x00020000),
                          __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(logp + e0), 0, left, 0x00020000), child,
                          batch, b < batch ? b : (int)batch - 1};
        res = reduce_narrow<Q16, LG>(E, (int32_t)(start - e0), (int32_t)k64, lut);
    }
    if (n < nodes && b < batch) out[n * batch + b] = res;
}

template <bool Q16, int LG, bool LOGP>
__global__ __launch_bounds__(64) void block_fwd_narrow(BlockLayout<LOGP> L, const float* __restrict__ child,
                                                       int64_t items, int per_wave, int64_t block0) {
    // per_wave: parents a wave holds, 64 / LG or, the other groups only
    // helping, 1
    __shared__ int lut[64];
    if constexpr (Q16) {
        lut[threadIdx.x] = kLut[threadIdx.x];
        __builtin_amdgcn_wave_barrier();
    }
    const int l = lane_id();
    const int b = l % LG;
    const int64_t item = (block0 + blockIdx.x) * per_wave + l / LG;
    const bool ok = l / LG < per_wave && item < items;
    const int64_t it = ok ? item : items - 1;
    const BlockNarrow<LOGP> E{L, child, b < L.batch ? b : (int)L.batch - 1};
    const float res = reduce_narrow<Q16, LG>(E, it, ok ? (int32_t)L.num_edges : 0, lut);
    const int64_t j = BlockNarrow<LOGP>::div_small(it, L.block_size);
    if (ok && b < L.batch) L.node_mars[(L.nids[j] + it - j * L.block_size) * L.batch + b] = res;
}

// -inf into the rows [j * block_size, (j + 1) * block_size) of each block j that
// does not write them itself (nids[j] elsewhere): with nids in order from 0 on, no
// rows at all.  `per` blocks to a wave, at most one a lane.  262144 rows of 512
// columns, us: in order 1.9, all elsewhere 99; a fill of all rows takes 78.
__global__ __launch_bounds__(256) void block_clear_rows(float* __restrict__ node_mars, const int64_t* __restrict__ nids,
                                                        int64_t nblocks, int64_t block_size, int64_t batch, int per,
                                                        int64_t block0) {
    const int l = lane_id();
    const int64_t j0 = ((block0 + blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * per;
    const int64_t j = j0 + l;
    uint64_t elsewhere = __ballot(l < per && j < nblocks && nids[j < nblocks ? j : 0] != j * block_size);
    const int64_t span = block_size * batch;
    while (elsewhere) {
        float* rows = node_mars + (j0 + __builtin_ctzll(elsewhere)) * span;
        elsewhere &= elsewhere - 1;
        for (int64_t i = l; i < span; i += 64) rows[i] = -kInf;
    }
}

// Q16.16, us, a wave per (parent, 64 columns) -> this: 2048 x 32 parents, 32
// edges, batch 4 237 -> 20, batch 32 238 -> 109; 1651 x 24 parents, 72 edges,
// batch 3 345 -> 75; 200 x 16 parents, 100 edges, batch 4 55 -> 9.
template <bool Q16, bool LOGP>
static void launch_block(const BlockLayout<LOGP>& L, const float* child, int64_t items, hipStream_t st) {
    if (L.batch > kNarrowBatch || L.num_edges == 0 || L.num_edges > kRunEdges) {
        launch<Q16>(L, child, L.node_mars, items, L.batch, st);
        return;
    }
    const auto go = [&](auto lg) {
        constexpr int LG = decltype(lg)::value;
        const int per = L.num_edges > kOwnEdges && items < 8192 ? 1 : 64 / LG;
        for_grid_chunks((items + per - 1) / per, 64, [&](int64_t b0, int64_t nb) {
            block_fwd_narrow<Q16, LG, LOGP><<<dim3((unsigned)nb), dim3(64), 0, st>>>(L, child, items, per, b0);
        });
    };
    // parents of more than kOwnEdges edges are taken one after the other by all
    // groups, of which Q16.16 uses eight; few enough of them take a wave each
    if (L.batch <= 4 && L.num_edges <= kOwnEdges)
        go(std::integral_constant<int, 4>{});
    else if (L.batch <= 8)
        go(std::integral_constant<int, 8>{});
    else if (L.batch <= 16)
        go(std::integral_constant<int, 16>{});
    else
        go(std::integral_constant<int, 32>{});
}

template <bool Q16, int LG>
static void launch_csr_narrow(const CsrLayout& L, const float* child, int64_t nodes, hipStream_t st) {
    constexpr int NG = 64 / LG;
    for_grid_chunks((nodes + NG - 1) / NG, 64, [&](int64_t b0, int64_t nb) {
        csr_fwd_narrow<Q16, LG><<<dim3((unsigned)nb), dim3(64), 0, st>>>(child, L.offsets, L.cids, L.logp, L.out,
                                                                         L.batch, nodes, b0);
    });
}

// Nodes per run, by the (node, column tile) pairs of the launch: longer runs
// spare more of the wave starts, shorter ones keep a small layer's waves many
// and its largest nodes apart (MI355X, fan-in k^-2 on [2, 256], us at 1 / 2 /
// 4 / 8 / 16 nodes a run: 2000 x 512 columns 26.5 / 28.0 / 28.9 / 30.5 / 34.0,
// 20000 x 512 79.7 / 66.8 / 69.9 / 80.0 / 85.6, 200000 x 512 565 / 509 / 497 /
// 506 / 514, 1M x 512 3325 / 2748 / 2619 / 2554 / 2576).
static int run_nodes(int64_t pairs) {
    return pairs < 40000 ? 1 : pairs < 160000 ? 2 : pairs < 1000000 ? 4 : 8;
}

// brief: most runs have one or two groups.
template <bool Q16, int VW, int P>
static void launch_csr_cols(const CsrLayout& L, const float* child, int64_t nodes, int npw, bool brief,
                            hipStream_t st) {
    const int64_t tiles = (L.batch + 64 * P - 1) / (64 * P);
    for_grid_chunks((nodes + npw - 1) / npw * tiles, 64, [&](int64_t u0, int64_t n) {
        const auto go = [&](auto kernel) {
            kernel<<<dim3((unsigned)n), dim3(64), 0, st>>>(child, L.offsets, L.cids, L.logp, L.out, L.batch, nodes, npw,
                                                           u0);
        };
        if (brief)
            go(csr_fwd_kernel<Q16, VW, P, true>);
        else
            go(csr_fwd_kernel<Q16, VW, P, false>);
    });
}

// Whether the batch's rows cut into 128-column slices without loss: whole
// 128-byte lines (a slice of a row that starts inside a line reads one more)
// and at most a tenth of the last slice's lanes idle over all of them.
static bool slices_fit(int64_t batch) { return batch % 32 == 0 && batch * 10 >= (batch + 127) / 128 * 128 * 9; }

// Whether 256-column tiles leave no more lanes idle than 128-column ones.
static bool wide_tiles_fit(int64_t batch) { return (batch + 127) / 128 == 2 * ((batch + 255) / 256); }

// Up to 32 columns: several nodes per wave (csr_fwd_narrow).  Columns per lane
// above: 1 up to a batch of 64, else 2 (200000 nodes, fp32, us, 1 / 2
// columns a lane: batch 64 99 / 105, 100 182 / 142, 512 515 / 497; 4 columns
// 140, 152, 519).  Large layers whose rows do not cut into such slices but fit
// tiles of 256 columns take these, in fp32 through the stream (us, 128 / 256
// columns: 1M x 200 1304 / 1143, 500000 x 500 1482 / 1349, 200000 x 130, 16 edges
// a node, 401 / 297; 100000 x 300, which does not fit, 212 / 231), in Q16.16 with
// a wave per node and tile (200000 x 500: 618 in slices, 595 through the stream,
// whose 8 chains of 4 columns leave it four waves per SIMD).
//
// From some thousand (node, 128-column tile) pairs on, the waves are more than
// the GPU holds at once, and a short node is a wave's fixed cost; up to 40000,
// where longer runs begin, half as many waves in fp32, of 256 columns or where
// these do not fit of two nodes, take less.  Below, the longest node's chain is the
// time, and a wave for it alone is fastest, as in Q16.16, whose chains are longer.
// us at 2 / 5 / 16 / power-law edges a node, one node and 128 columns a wave ->
// this: 8000 nodes, batch 512, 15.0 / 18.8 / 31.0 / 40.3 -> 10.0 / 15.9 / 27.6 / 43.4;
// 8000 x 300 12.5 / 15.5 / 24.3 / 35.6 -> 9.9 / 14.9 / 23.5 / 37.2; not 2000 x 256,
// 4.7 / 5.3 / 7.3 / 22.4 against 4.0 / 4.6 / 6.1 / 26.4 with 256 columns, nor Q16.16,
// 14000 x 256, 14.0 / 18.0 / 32.8 / 56.1 against 11.2 / 17.3 / 31.1 / 66.9 with two
// nodes.
//
// Up to 4 columns, 4 lanes a node; of fewer than 4000 nodes 8, as fan-ins past
// kOwnEdges are then the time, and 16 nodes' worth of them queue in one wave (us,
// 4 / 8 lanes, batch 4: 1000 nodes of 40 edges, fp32 14.3 / 10.7, Q16.16 21.1 /
// 12.2; 4000 nodes of 16 edges 4.3 / 4.4, 4.8 / 5.0; power law, 1000 nodes 8.8 /
// 9.3, 13.0 / 12.1).
template <bool Q16>
static void launch_csr(const CsrLayout& L, const float* child, int64_t nodes, hipStream_t st) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(child) | reinterpret_cast<uintptr_t>(L.out);
    const int64_t batch = L.batch;
    if (batch <= kNarrowBatch) {
        if (batch <= 4 && nodes >= 4000)
            launch_csr_narrow<Q16, 4>(L, child, nodes, st);
        else if (batch <= 8)
            launch_csr_narrow<Q16, 8>(L, child, nodes, st);
        else if (batch <= 16)
            launch_csr_narrow<Q16, 16>(L, child, nodes, st);
        else
            launch_csr_narrow<Q16, 32>(L, child, nodes, st);
        return;
    }
    if (batch <= 64) {
        launch_csr_cols<Q16, 1, 1>(L, child, nodes, run_nodes(nodes), nodes < 40000, st);
        return;
    }
    // rows of 4 GiB: the stream holds a row's bytes in 32 bits (in 64 the extra
    // scalar arithmetic per edge took 200000 x 100 Q16.16 from 176.9 to 178.4 us)
    if (batch >= (int64_t)1 << 30) {
        launch<Q16>(L, child, L.out, nodes, batch, st);
        return;
    }
    const int64_t pairs = nodes * ((batch + 127) / 128);
    const bool brief = pairs < 40000;
    const bool wide = batch > 128 && wide_tiles_fit(batch), slices = slices_fit(batch);
    const bool large = wide && !slices && nodes >= 40000;
    if constexpr (Q16) {
        if (large) {
            launch<true>(L, child, L.out, nodes, batch, st);
            return;
        }
    } else if (large || (wide && pairs >= 12000 && (brief || (!slices && batch <= 256)))) {
        const int npw = large ? 2 : 1;
        if (batch % 4 == 0 && (at & 15) == 0)
            launch_csr_cols<false, 4, 4>(L, child, nodes, npw, !large, st);
        else
            launch_csr_cols<false, 1, 4>(L, child, nodes, npw, !large, st);
        return;
    }
    const int npw = !Q16 && batch > 128 && brief && pairs >= 8000 ? 2 : run_nodes(pairs);
    if (batch % 2 == 0 && (at & 7) == 0)
        launch_csr_cols<Q16, 2, 2>(L, child, nodes, npw, brief, st);
    else
        launch_csr_cols<Q16, 1, 2>(L, child, nodes, npw, brief, st);
}

// ---------------------------------------------------------------------------
// CSR backward (flows).  For out[n, b] = LSE_e(lw_e + child[c_e, b]) and an
// upstream gradient gout:
//   term[e, b]       = gout[n_e, b] * exp(lw_e + child[c_e, b] - out[n_e, b])
//   grad_child[c, b] = sum of term[e, b] over the edges e with c_e = c
//   grad_lw[e]       = sum of term[e, b] over b
// A term whose out[n_e, b] is -inf is 0: nothing flows through a node of
// probability 0 (torch's autograd of logsumexp would give NaN there).
// The kernel walks the transposed structure (CSC: for child c the edges that
// point at it, each with its parent node) the way csr_fwd_kernel walks the
// nodes: a wave per run of children and column tile, tile-slowest, the two
// parent rows of each of a group's edges in flight while a group folds.
// grad_child is accumulated in registers and written once.
//
// The edges' weights and batch sums are scattered 4-byte accesses, once per
// column tile.  So with several tiles csr_bwd_weights gathers the weights into
// the walk's order first, each tile stores its sums in that order, coalesced,
// in a workspace, and csr_bwd_sums adds the tiles' sums in tile order and
// scatters them.  DIRECT, a single tile, takes them where they are and spares
// two launches.  The summation order is fixed either way.  The 1M-child,
// 8.0M-edge layer at batch 512 went from 6160 to 5270 us (two gathered rows an
// edge, 33 GB; a wave per child over whole rows -> this); 200000 x 64 columns,
// DIRECT, from 265 to 169.
// ---------------------------------------------------------------------------
// g * exp(t - o), or 0 where o is -inf or the place is not one of the batch's.
// (The product is taken before the select: inside it the compiler branches
// around the exponential, and waits for every load in flight there.)
__device__ __forceinline__ float flow(float g, float t, float o, bool ok) {
    const float x = g * fexp2((t - o) * kLog2e);
    return ok && o != -kInf ? x : 0.0f;
}

__device__ __forceinline__ float wave_sum(float v) {
    v += reduce_partner<1>(v);
    v += reduce_partner<2>(v);
    v += reduce_partner<4>(v);
    v += reduce_partner<8>(v);
    v += reduce_partner<16>(v);
    v += reduce_partner<32>(v);
    return v;
}

// Sums of four values over the wave: lane l ends with value l % 4's.
__device__ __forceinline__ float wave_sum4(const float (&v)[4], int l) {
    const bool odd = l & 1, hi = l & 2;
    const float a = (odd ? v[1] : v[0]) + reduce_partner<1>(odd ? v[0] : v[1]);
    const float b = (odd ? v[3] : v[2]) + reduce_partner<1>(odd ? v[2] : v[3]);
    float s = (hi ? b : a) + reduce_partner<2>(hi ? a : b);
    // row rotations by 4 and 8: the other quads of the row, lane for lane
    s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x124, 0xF, 0xF, false));
    s += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x128, 0xF, 0xF, false));
    s += reduce_partner<16>(s);
    return s + reduce_partner<32>(s);
}

__global__ __launch_bounds__(256) void csr_bwd_weights(const float* __restrict__ logp,
                                                       const int32_t* __restrict__ edges, float* __restrict__ lwc,
                                                       int64_t nnz, int64_t block0) {
    const int64_t k = (block0 + blockIdx.x) * 256 + threadIdx.x;
    if (k < nnz) lwc[k] = logp[edges[k]];
}

__global__ __launch_bounds__(256) void csr_bwd_sums(const float* __restrict__ part, const int32_t* __restrict__ edges,
                                                    float* __restrict__ glogp, int64_t nnz, int64_t tiles,
                                                    int64_t block0) {
    const int64_t k = (block0 + blockIdx.x) * 256 + threadIdx.x;
    if (k >= nnz) return;
    float s = part[k];
    for (int64_t t = 1; t < tiles; ++t) s += part[t * nnz + k];
    glogp[edges[k]] = s;
}

// SHORT: most runs have one or two groups, which leave before the loop, as in
// csr_fwd_kernel (20000 children, batch 64, us at 2 / 5 / 16 edges a child 20.4 /
// 22.7 / 38.5 -> 16.3 / 19.7 / 39.6).
template <bool DIRECT, int VW, int P, bool SHORT>
__global__ __launch_bounds__(64) void csr_bwd_kernel(const float* __restrict__ child, const float* __restrict__ out,
                                                     const float* __restrict__ gout, const float* __restrict__ logp,
                                                     const int64_t* __restrict__ csc_off,
                                                     const int32_t* __restrict__ csc_edge,
                                                     const int32_t* __restrict__ csc_node,
                                                     float* __restrict__ gchild, float* __restrict__ glogp,
                                                     int64_t children, int64_t batch, int npw, int64_t tiles,
                                                     int64_t unit0) {
    // logp, glogp: by edge id with DIRECT, else in the walk's order (glogp: one
    // such array per tile)
    const int l = lane_id();
    const int64_t runs = (children + npw - 1) / npw;
    const int64_t unit = xcd_unit(unit0 + blockIdx.x, DIRECT ? runs : runs * tiles);
    const int64_t tile = DIRECT ? 0 : unit / runs;
    const int64_t n0 = (unit - tile * runs) * npw;
    const int nn = (int)(children - n0 < npw ? children - n0 : npw);
    const int64_t at = csc_off[n0 + (l < nn ? l : nn)];
    const int64_t nnz = uniform64(csc_off[children]);
    const int64_t e0 = uniform64(at);
    // a layer without any edge goes the other way too: the stream reads the weight
    // of edge 0 for a masked one
    const bool streamed = nnz > 0 && bcast64(at, nn) - e0 <= kRunEdges;
    const int64_t b0 = tile * 64 * P;
    const int rec = cols_bytes(batch, b0);
    const float* child_b0 = child + b0;
    const float* gout_b0 = gout + b0;
    const float* out_b0 = out + b0;
    const uint64_t row_bytes = (uint64_t)batch * 4u;
    bool lane_ok[P];
#pragma unroll
    for (int i = 0; i < P; ++i) lane_ok[i] = Cols<VW, P>::ok(b0, l, batch, i);
    float cv[P], acc[P];
    if (streamed) {
        const Run run{(int32_t)(at - e0)};
        const u32x4v rn = words_rsrc(csc_node + e0, nnz - e0);
        const u32x4v rw = DIRECT ? words_rsrc(csc_edge + e0, nnz - e0) : words_rsrc(logp + e0, nnz - e0);
        // ids: the parents; w: the weights, or with DIRECT the edge ids
        struct Meta {
            u32x4v ids, w;
        };
        const auto load_meta = [&](const Group& g) {
            return Meta{s_buffer_load4(rn, g.e * 4, 0), s_buffer_load4(rw, g.e * 4, 0)};
        };
        struct Rows {
            float x[P], g[G][P], o[G][P], lw[G];
        };
        const auto load_rows = [&](Rows& v, const Meta& em, const Group& g) {
            load_cols_buf<VW, P>(child_b0 + (n0 + (g.node < nn ? g.node : 0)) * batch,
                                 g.first && g.node < nn ? rec : 0, l, v.x);
#pragma unroll
            for (int k = 0; k < G; ++k) {
                const uint64_t row = (uint64_t)em.ids[k] * row_bytes;
                const int r = k < g.left ? rec : 0;
                load_cols_buf<VW, P>(reinterpret_cast<const float*>(reinterpret_cast<const char*>(gout_b0) + row), r,
                                     l, v.g[k]);
                load_cols_buf<VW, P>(reinterpret_cast<const float*>(reinterpret_cast<const char*>(out_b0) + row), r,
                                     l, v.o[k]);
            }
            if constexpr (DIRECT) {
#pragma unroll
                for (int k = 0; k < G; ++k)
                    v.lw[k] = logp[k < g.left ? (uint32_t)em.w[k] : 0u];
            } else {
#pragma unroll
                for (int k = 0; k < G; ++k) v.lw[k] = __builtin_bit_cast(float, (uint32_t)em.w[k]);
            }
        };
        const auto fold = [&](const Rows& v, const Meta& em, const Group& g) {
            if (g.first) {
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    cv[i] = v.x[i];
                    acc[i] = 0.0f;
                }
            }
            float t[G];
#pragma unroll
            for (int k = 0; k < G; ++k) {
                t[k] = 0.0f;
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    const float x = flow(v.g[k][i], v.lw[k] + cv[i], v.o[k][i], lane_ok[i] && k < g.left);
                    acc[i] += x;
                    t[k] += x;
                }
            }
            const float s = wave_sum4(t, l);
            if constexpr (DIRECT) {
                const uint32_t lo = l & 1 ? em.w[1] : em.w[0], hi = l & 1 ? em.w[3] : em.w[2];
                float* dst = glogp + (l & 2 ? hi : lo);
                if (l < 4 && l < g.left) *dst = s;
            } else {
                if (l < 4 && l < g.left) glogp[tile * nnz + e0 + g.e + l] = s;
            }
            if (g.left <= G && g.node < nn) Cols<VW, P>::store(gchild + (n0 + g.node) * batch, b0, l, batch, acc);
        };
        Rows va, vb;
        Group ga = {0, 0, run.start(1), 1, 0};
        Meta ma = load_meta(ga);
        load_rows(va, ma, ga);
        Group gb = run.next(ga);
        Meta mb = load_meta(gb);
        if (SHORT && run.next(gb).node >= nn) {
            load_rows(vb, mb, gb);
            fold(va, ma, ga);
            fold(vb, mb, gb);
            return;
        }
        while (true) {
            load_rows(vb, mb, gb);
            const Group gc = run.next(gb);
            const Meta mc = load_meta(gc);
            fold(va, ma, ga);
            load_rows(va, mc, gc);
            const Group gd = run.next(gc);
            const Meta md = load_meta(gd);
            fold(vb, mb, gb);
            if (gc.node >= nn) break;
            ga = gc;
            ma = mc;
            gb = gd;
            mb = md;
        }
    } else {  // too many edges for the stream's 32-bit edge numbers: one at a time
        for (int c = 0; c < nn; ++c) {
            load_cols_buf<VW, P>(child_b0 + (n0 + c) * batch, rec, l, cv);
#pragma unroll
            for (int i = 0; i < P; ++i) acc[i] = 0.0f;
            for (int64_t k = bcast64(at, c); k < bcast64(at, c + 1); ++k) {
                float g[P], o[P], t = 0.0f;
                const int64_t row = (int64_t)csc_node[k] * batch, e = csc_edge[k];
                load_cols_buf<VW, P>(gout_b0 + row, rec, l, g);
                load_cols_buf<VW, P>(out_b0 + row, rec, l, o);
                const float lw = logp[DIRECT ? e : k];
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    const float x = flow(g[i], lw + cv[i], o[i], lane_ok[i]);
                    acc[i] += x;
                    t += x;
                }
                t = wave_sum(t);
                if (l == 0) glogp[DIRECT ? e : tile * nnz + k] = t;
            }
            Cols<VW, P>::store(gchild + (n0 + c) * batch, b0, l, batch, acc);
        }
    }
}

// The backward of a batch of up to 32 columns: csr_fwd_narrow's walk over the
// children, LG lanes per child, both of an edge's parent rows per lane group.
// An edge's sum is reduced over its group's lanes, four edges at a time.
template <int LG>
__global__ __launch_bounds__(64) void csr_bwd_narrow(const float* __restrict__ child, const float* __restrict__ out,
                                                     const float* __restrict__ gout, const float* __restrict__ logp,
                                                     const int64_t* __restrict__ csc_off,
                                                     const int32_t* __restrict__ csc_edge,
                                                     const int32_t* __restrict__ csc_node,
                                                     float* __restrict__ gchild, float* __restrict__ glogp,
                                                     int64_t children, int64_t batch, int64_t block0) {
    constexpr int NG = 64 / LG;
    const int l = lane_id();
    const int grp = l / LG, b = l % LG;
    const int64_t c0 = (block0 + blockIdx.x) * NG;
    const int64_t c = c0 + grp;
    const int64_t cc = c < children ? c : children - 1;
    const int64_t start = csc_off[cc], e0 = uniform64(start);
    const int64_t k64 = c < children ? csc_off[cc + 1] - start : 0;
    const int64_t total = uniform64(csc_off[c0 + NG < children ? c0 + NG : children]) - e0;
    const bool col_ok = b < batch;
    const int64_t col = col_ok ? b : batch - 1;
    const float x = child[cc * batch + col];
    float acc = 0.0f;
    if (total > kRunEdges) {  // beyond 32-bit edge numbers: one edge at a time
        for (int64_t k = start; __any(k < start + k64); ++k) {
            const bool ok = k < start + k64;
            const int64_t kk = ok ? k : e0, row = (int64_t)csc_node[kk] * batch + col, e = csc_edge[kk];
            float t = flow(gout[row], logp[e] + x, out[row], ok && col_ok);
            acc += t;
            for (int d = 1; d < LG; d <<= 1) t += shuffle_xor(t, d);
            if (ok && b == 0) glogp[e] = t;
        }
    } else if (total > 0) {
        const int64_t nnz = uniform64(csc_off[children]);
        const int left = (int)(nnz - e0 < kRunEdges * 2 ? nnz - e0 : kRunEdges * 2) * 4;
        const __amdgpu_buffer_rsrc_t re =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(csc_edge + e0), 0, left, 0x00020000);
        const __amdgpu_buffer_rsrc_t rn =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(csc_node + e0), 0, left, 0x00020000);
        // four edges i[u] of a child with value xv: their terms into sum,
        // their sums over the batch into glogp
        const auto four = [&](const int32_t (&i)[4], const bool (&ok)[4], float xv, float& sum) {
            uint32_t ed[4];
            float t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int at = ok[u] ? i[u] * 4 : 0x7FFFFFFC;
                ed[u] = __builtin_amdgcn_raw_buffer_load_b32(re, at, 0, 0);
                const int64_t row = (int64_t)(uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rn, at, 0, 0) * batch + col;
                t[u] = flow(gout[row], logp[ed[u]] + xv, out[row], ok[u] && col_ok);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) sum += t[u];
            const bool odd = b & 1, hi = b & 2;
            const float p = (odd ? t[1] : t[0]) + reduce_partner<1>(odd ? t[0] : t[1]);
            const float q = (odd ? t[3] : t[2]) + reduce_partner<1>(odd ? t[2] : t[3]);
            float s = (hi ? q : p) + reduce_partner<2>(hi ? p : q);  // lane b: edge b % 4 over its quad
            if constexpr (LG >= 8) s += exact_xor<4>(s);
            if constexpr (LG >= 16) s += exact_xor<8>(s);
            if constexpr (LG >= 32) s += exact_xor<16>(s);
            const uint32_t lo = odd ? ed[1] : ed[0], up = odd ? ed[3] : ed[2];
            const bool mine = hi ? (odd ? ok[3] : ok[2]) : (odd ? ok[1] : ok[0]);
            if (b < 4 && mine) glogp[hi ? up : lo] = s;
        };
        const int32_t s0 = (int32_t)(start - e0), k = (int32_t)k64;
        const int32_t own = k <= kOwnEdges ? k : 0;
        uint64_t longer = __ballot(k > kOwnEdges && b == 0);
        for (int32_t e = 0; __any(e < own); e += 4) {
            const int32_t i[4] = {s0 + e, s0 + e + 1, s0 + e + 2, s0 + e + 3};
            const bool ok[4] = {e < own, e + 1 < own, e + 2 < own, e + 3 < own};
            four(i, ok, x, acc);
        }
        while (longer) {
            const int j = __builtin_ctzll(longer);
            longer &= longer - 1;
            const int32_t sj = __builtin_amdgcn_readlane(s0, j), kj = __builtin_amdgcn_readlane(k, j);
            const float xj = child[(c0 + j / LG) * batch + col];
            float sum = 0.0f;
            for (int32_t r = grp; __any(r < kj); r += 4 * NG) {
                const int32_t i[4] = {sj + r, sj + r + NG, sj + r + 2 * NG, sj + r + 3 * NG};
                const bool ok[4] = {r < kj, r + NG < kj, r + 2 * NG < kj, r + 3 * NG < kj};
                four(i, ok, xj, sum);
            }
            for (int d = LG; d < 64; d <<= 1) sum += shuffle_xor(sum, d);
            acc = grp == j / LG ? sum : acc;
        }
    }
    if (c < children && col_ok) gchild[c * batch + b] = acc;
}

template <int LG>
static void launch_csr_bwd_narrow(const float* child, const float* out, const float* gout, const float* logp,
                                  const int64_t* off, const int32_t* edge, const int32_t* node, float* gchild,
                                  float* glogp, int64_t children, int64_t batch, hipStream_t st) {
    constexpr int NG = 64 / LG;
    for_grid_chunks((children + NG - 1) / NG, 64, [&](int64_t b0, int64_t nb) {
        csr_bwd_narrow<LG><<<dim3((unsigned)nb), dim3(64), 0, st>>>(child, out, gout, logp, off, edge, node, gchild,
                                                                    glogp, children, batch, b0);
    });
}

template <bool DIRECT, int VW, int P>
static void launch_csr_bwd_cols(const float* child, const float* out, const float* gout, const float* logp,
                                const int64_t* off, const int32_t* edge, const int32_t* node, float* gchild,
                                float* glogp, int64_t children, int64_t batch, hipStream_t st) {
    const int64_t tiles = (batch + 64 * P - 1) / (64 * P);
    const int npw = run_nodes(DIRECT ? children : children * tiles);
    const int64_t runs = (children + npw - 1) / npw;
    for_grid_chunks(DIRECT ? runs : runs * tiles, 64, [&](int64_t u0, int64_t n) {
        const auto go = [&](auto kernel) {
            kernel<<<dim3((unsigned)n), dim3(64), 0, st>>>(child, out, gout, logp, off, edge, node, gchild, glogp,
                                                           children, batch, npw, tiles, u0);
        };
        if (DIRECT && npw == 1)
            go(csr_bwd_kernel<DIRECT, VW, P, DIRECT>);
        else
            go(csr_bwd_kernel<DIRECT, VW, P, false>);
    });
}

// Columns of a tile of the backward at this batch (200000 children, us, tiles
// of 64 / 128 / 256 columns: batch 64 169 / 181 / 245, 128 281 / 264 / 273, 512
// 970 / 973 / 1039; 1M children, batch 512 5285 / 5316 / 5175 at their best run
// lengths).
static int64_t bwd_tile_cols(int64_t batch) { return batch <= 64 ? 64 : 128; }

template <bool DIRECT>
static void launch_csr_bwd(const float* child, const float* out, const float* gout, const float* logp,
                           const int64_t* off, const int32_t* edge, const int32_t* node, float* gchild, float* glogp,
                           int64_t children, int64_t batch, hipStream_t st) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(child) | reinterpret_cast<uintptr_t>(out) |
                         reinterpret_cast<uintptr_t>(gout) | reinterpret_cast<uintptr_t>(gchild);
    if (bwd_tile_cols(batch) == 64)
        launch_csr_bwd_cols<DIRECT, 1, 1>(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
    else if (batch % 2 == 0 && (at & 7) == 0)
        launch_csr_bwd_cols<DIRECT, 2, 2>(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
    else
        launch_csr_bwd_cols<DIRECT, 1, 2>(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
}

// Several column tiles without a workspace: one wave per child row (four to a
// block), every 512-column tile in turn, its parents' rows one edge ahead.  The
// first tile stores an edge's sum and the later ones add to it with a no-return
// atomic, all from lane 0 of the wave that owns the edge, in tile order.
struct ParentMeta {
    int64_t node;
    int64_t edge;
    float lw;
};

constexpr int PB = 8;  // columns per lane
// Parent edges per load group (two rows each), and columns per lane: 8 columns
// and single-edge groups measured 7.2 ms on the 1M-node layer of 8.0M edges,
// batch 512, against 7.8 ms for 4 columns and two-edge groups.
constexpr int GB = 1;

template <int VW>
__device__ __forceinline__ void load_parents(float (&gv)[GB][PB], float (&ov)[GB][PB], const ParentMeta& pw, int j,
                                             int wn, const float* __restrict__ gout, const float* __restrict__ out,
                                             int64_t batch, int64_t b0, int l) {
    // every load issued, as in load_group: parents past wn read empty ranges
    const int rec = cols_bytes(batch, b0);
#pragma unroll
    for (int g = 0; g < GB; ++g) {
        const int64_t n = bcast64(pw.node, (j + g) & 63);
        const int r = j + g < wn ? rec : 0;
        load_cols_buf<VW, PB>(gout + n * batch + b0, r, l, gv[g]);
        load_cols_buf<VW, PB>(out + n * batch + b0, r, l, ov[g]);
    }
}

template <int VW>
__device__ __forceinline__ void flow_group(const float (&gv)[GB][PB], const float (&ov)[GB][PB], const ParentMeta& pw,
                                           int j, int wn, const float (&cv)[PB], float (&acc)[PB], bool first_tile,
                                           float* __restrict__ glogp, int64_t batch, int64_t b0, int l) {
#pragma unroll
    for (int g = 0; g < GB; ++g) {
        if (j + g < wn) {
            const float lw = bcastf(pw.lw, j + g);
            float tsum = 0.0f;
#pragma unroll
            for (int i = 0; i < PB; ++i) {
                const float t = flow(gv[g][i], lw + cv[i], ov[g][i], Cols<VW, PB>::ok(b0, l, batch, i));
                acc[i] += t;
                tsum += t;
            }
            tsum = wave_sum(tsum);
            const int64_t e = bcast64(pw.edge, j + g);
            // later tiles add without reading back, so no load sits in the
            // edge loop; only this wave touches edge e, so the adds land in
            // tile order and the result is deterministic
            if (l == 0) {
                if (first_tile)
                    glogp[e] = tsum;
                else
                    __hip_atomic_fetch_add(glogp + e, tsum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

template <int VW>
__global__ __launch_bounds__(256) void csr_bwd_rows_kernel(const float* __restrict__ child, const float* __restrict__ out,
                                                      const float* __restrict__ gout, const float* __restrict__ logp,
                                                      const int64_t* __restrict__ csc_off,
                                                      const int32_t* __restrict__ csc_edge,
                                                      const int32_t* __restrict__ csc_node,
                                                      float* __restrict__ gchild, float* __restrict__ glogp,
                                                      int64_t children, int64_t batch, int64_t block0) {
    const int l = lane_id();
    const int64_t c =
        (block0 + (int64_t)blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (c >= children) return;
    const int64_t p0 = uniform64(csc_off[c]);
    const int64_t k = uniform64(csc_off[c + 1]) - p0;
    for (int64_t b0 = 0; b0 < batch; b0 += 64 * PB) {
        float cv[PB], acc[PB];
        load_cols_buf<VW, PB>(child + c * batch + b0, cols_bytes(batch, b0), l, cv);
#pragma unroll
        for (int i = 0; i < PB; ++i) acc[i] = 0.0f;
        for (int64_t w0 = 0; w0 < k; w0 += 64) {
            ParentMeta pw{0, 0, 0.0f};
            if (w0 + l < k) {
                const int64_t e = csc_edge[p0 + w0 + l];
                pw = {(int64_t)csc_node[p0 + w0 + l], e, logp[e]};
            }
            const int wn = (int)(k - w0 < 64 ? k - w0 : 64);
            const int ng = (wn + GB - 1) / GB;
            float ga[GB][PB], oa[GB][PB], gb[GB][PB], ob[GB][PB];
            load_parents<VW>(ga, oa, pw, 0, wn, gout, out, batch, b0, l);
            int gi = 0;
            for (; gi + 1 < ng; gi += 2) {
                load_parents<VW>(gb, ob, pw, (gi + 1) * GB, wn, gout, out, batch, b0, l);
                flow_group<VW>(ga, oa, pw, gi * GB, wn, cv, acc, b0 == 0, glogp, batch, b0, l);
                load_parents<VW>(ga, oa, pw, (gi + 2) * GB, wn, gout, out, batch, b0, l);
                flow_group<VW>(gb, ob, pw, (gi + 1) * GB, wn, cv, acc, b0 == 0, glogp, batch, b0, l);
            }
            if (gi < ng) flow_group<VW>(ga, oa, pw, gi * GB, wn, cv, acc, b0 == 0, glogp, batch, b0, l);
        }
        Cols<VW, PB>::store(gchild + c * batch, b0, l, batch, acc);
    }
}

static void launch_csr_bwd_rows(const float* child, const float* out, const float* gout, const float* logp,
                                const int64_t* off, const int32_t* edge, const int32_t* node, float* gchild,
                                float* glogp, int64_t children, int64_t batch, hipStream_t st) {
    const uintptr_t at = reinterpret_cast<uintptr_t>(child) | reinterpret_cast<uintptr_t>(out) |
                         reinterpret_cast<uintptr_t>(gout) | reinterpret_cast<uintptr_t>(gchild);
    for_grid_chunks((children + 3) / 4, 256, [&](int64_t b0, int64_t nb) {
        if (batch % 4 == 0 && (at & 15) == 0)
            csr_bwd_rows_kernel<4><<<dim3((unsigned)nb), dim3(256), 0, st>>>(child, out, gout, logp, off, edge, node,
                                                                            gchild, glogp, children, batch, b0);
        else
            csr_bwd_rows_kernel<1><<<dim3((unsigned)nb), dim3(256), 0, st>>>(child, out, gout, logp, off, edge, node,
                                                                            gchild, glogp, children, batch, b0);
    });
}

// Without a workspace.
static void launch_csr_bwd_plain(const float* child, const float* out, const float* gout, const float* logp,
                                 const int64_t* off, const int32_t* edge, const int32_t* node, float* gchild,
                                 float* glogp, int64_t children, int64_t batch, hipStream_t st) {
    if (batch <= kNarrowBatch) {
        const auto go = [&](auto launch) {
            launch(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
        };
        if (batch <= 4)
            go(launch_csr_bwd_narrow<4>);
        else if (batch <= 8)
            go(launch_csr_bwd_narrow<8>);
        else if (batch <= 16)
            go(launch_csr_bwd_narrow<16>);
        else
            go(launch_csr_bwd_narrow<32>);
        return;
    }
    if (batch <= bwd_tile_cols(batch))
        launch_csr_bwd<true>(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
    else
        launch_csr_bwd_rows(child, out, gout, logp, off, edge, node, gchild, glogp, children, batch, st);
}

}  // namespace sparse
}  // namespace fl

using namespace fl;

extern "C" int fl_sparse_csr_bwd(const float* child, const float* out, const float* grad_out, const float* logparams,
                                 const int64_t* csc_offsets, const int32_t* csc_edges, const int32_t* csc_nodes,
                                 float* grad_child, float* grad_logparams, int64_t num_children, int64_t batch,
                                 void* stream) {
    const char* name = "fl_sparse_csr_bwd";
    FL_CHECK(num_children >= 0 && batch >= 0, "%s: negative size", name);
    if (num_children == 0 || batch == 0) return ok();
    FL_CHECK(child && out && grad_out && logparams && csc_offsets && csc_edges && csc_nodes && grad_child &&
                 grad_logparams,
             "%s: NULL pointer argument", name);
    sparse::launch_csr_bwd_plain(child, out, grad_out, logparams, csc_offsets, csc_edges, csc_nodes, grad_child,
                                 grad_logparams, num_children, batch, reinterpret_cast<hipStream_t>(stream));
    return launch_status(name);
}

// The workspace form is for slices that fit (slices_fit; 500000 x 400 took 2540
// us in them against 2099 in whole rows) of layers of at least 64000 (child,
// column tile) pairs: it pays two more launches (us, workspace / none: 2000 x
// 512 20 / 13, 12000 x 512 58 / 53, 20000 x 512 89 / 97, 50000 x 512 227 / 265).
// And of at least 5 edges a child, as each tile of a child is a walk of its own
// (100000 x 384 at 2 / 4 / 5 / 8 edges a child 192 / 241 / 273 / 391, none 132 / 229 /
// 278 / 412).
// It grows with the edges, so above 256 MB it is taken only up to the size of
// the gradient of the children that it serves (about 100 edges a child); past
// that, whole rows (20000 children of 200 edges, batch 512, 80 MB: 1887 us
// against 2200; 16000 of 1000, 320 MB: 9156 against 9204).
constexpr size_t kBwdWorkspaceSmall = (size_t)256 << 20;

extern "C" size_t fl_sparse_csr_bwd_workspace_bytes(int64_t num_children, int64_t nnz, int64_t batch) {
    if (nnz <= 0 || batch <= 0) return 0;
    const int64_t cols = sparse::bwd_tile_cols(batch);
    const int64_t tiles = (batch + cols - 1) / cols;
    if (tiles < 2 || num_children * tiles < 64000 || nnz / 5 < num_children || !sparse::slices_fit(batch)) return 0;
    const size_t need = (size_t)nnz * (size_t)(tiles + 1) * sizeof(float);
    const size_t rows = (size_t)num_children * (size_t)batch * sizeof(float);
    return need <= kBwdWorkspaceSmall || need <= rows ? need : 0;
}

extern "C" int fl_sparse_csr_bwd_ws(const float* child, const float* out, const float* grad_out,
                                    const float* logparams, const int64_t* csc_offsets, const int32_t* csc_edges,
                                    const int32_t* csc_nodes, float* grad_child, float* grad_logparams,
                                    int64_t num_children, int64_t nnz, int64_t batch, void* workspace,
                                    size_t workspace_bytes, void* stream) {
    const char* name = "fl_sparse_csr_bwd_ws";
    FL_CHECK(num_children >= 0 && nnz >= 0 && batch >= 0, "%s: negative size", name);
    if (num_children == 0 || batch == 0) return ok();
    FL_CHECK(child && out && grad_out && logparams && csc_offsets && csc_edges && csc_nodes && grad_child &&
                 grad_logparams,
             "%s: NULL pointer argument", name);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const size_t need = fl_sparse_csr_bwd_workspace_bytes(num_children, nnz, batch);
    if (need == 0) {
        sparse::launch_csr_bwd_plain(child, out, grad_out, logparams, csc_offsets, csc_edges, csc_nodes, grad_child,
                                     grad_logparams, num_children, batch, st);
        return launch_status(name);
    }
    FL_CHECK(workspace != nullptr && workspace_bytes >= need, "%s: workspace of %llu bytes, %llu needed", name,
             (unsigned long long)workspace_bytes, (unsigned long long)need);
    FL_CHECK((reinterpret_cast<uintptr_t>(workspace) & 3u) == 0, "%s: workspace is not 4-byte aligned", name);
    const int64_t cols = sparse::bwd_tile_cols(batch);
    const int64_t tiles = (batch + cols - 1) / cols;
    float* lwc = static_cast<float*>(workspace);
    float* part = lwc + nnz;
    for_grid_chunks((nnz + 255) / 256, 256, [&](int64_t b0, int64_t nb) {
        sparse::csr_bwd_weights<<<dim3((unsigned)nb), dim3(256), 0, st>>>(logparams, csc_edges, lwc, nnz, b0);
    });
    sparse::launch_csr_bwd<false>(child, out, grad_out, lwc, csc_offsets, csc_edges, csc_nodes, grad_child, part,
                                  num_children, batch, st);
    for_grid_chunks((nnz + 255) / 256, 256, [&](int64_t b0, int64_t nb) {
        sparse::csr_bwd_sums<<<dim3((unsigned)nb), dim3(256), 0, st>>>(part, csc_edges, grad_logparams, nnz, tiles, b0);
    });
    return launch_status(name);
}

extern "C" int fl_sparse_csr_fwd(const float* child, const int64_t* offsets, const int32_t* child_ids,
                                 const float* logparams, float* out, int64_t num_nodes, int64_t batch, int q16,
                                 void* stream) {
    const char* name = "fl_sparse_csr_fwd";
    FL_CHECK(num_nodes >= 0 && batch >= 0, "%s: negative size", name);
    if (num_nodes == 0 || batch == 0) return ok();
    FL_CHECK(child && offsets && out, "%s: NULL pointer argument", name);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const sparse::CsrLayout L{offsets, child_ids, logparams, out, batch};
    if (q16)
        sparse::launch_csr<true>(L, child, num_nodes, st);
    else
        sparse::launch_csr<false>(L, child, num_nodes, st);
    return launch_status(name);
}

extern "C" int fl_sparse_blocked_fwd(float* node_mars, const float* element_mars, const float* params,
                                     const int64_t* nids, const int64_t* cids, const int64_t* pids, int64_t num_nblocks,
                                     int64_t num_edges, int64_t block_size, int64_t batch, int q16, int params_are_log,
                                     void* stream) {
    const char* name = "fl_sparse_blocked_fwd";
    FL_CHECK(num_nblocks >= 0 && num_edges >= 0 && block_size >= 0 && batch >= 0, "%s: negative size", name);
    if (num_nblocks == 0 || block_size == 0 || batch == 0) return ok();
    FL_CHECK(node_mars && element_mars && params && nids && (num_edges == 0 || (cids && pids)),
             "%s: NULL pointer argument", name);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (!q16 && sparse::blocked_mfma_eligible(num_edges, block_size)) {
        sparse::launch_blocked_mfma(node_mars, element_mars, params, nids, cids, pids, num_nblocks, num_edges,
                                    block_size, batch, params_are_log != 0, st);
        return launch_status(name);
    }
    const int64_t items = num_nblocks * block_size;
    if (params_are_log) {
        const sparse::BlockLayout<true> L{node_mars, params, nids, cids, pids, num_edges, block_size, batch};
        if (q16) sparse::launch_block<true>(L, element_mars, items, st);
        else sparse::launch_block<false>(L, element_mars, items, st);
    } else {
        const sparse::BlockLayout<false> L{node_mars, params, nids, cids, pids, num_edges, block_size, batch};
        if (q16) sparse::launch_block<true>(L, element_mars, items, st);
        else sparse::launch_block<false>(L, element_mars, items, st);
    }
    return launch_status(name);
}

extern "C" int fl_sparse_blocked_fwd_fresh(float* node_mars, const float* element_mars, const float* params,
                                           const int64_t* nids, const int64_t* cids, const int64_t* pids,
                                           int64_t num_nblocks, int64_t num_edges, int64_t block_size, int64_t batch,
                                           int q16, int params_are_log, void* stream) {
    // sizes and pointers that the forward refuses launch nothing
    if (num_nblocks > 0 && num_edges >= 0 && block_size > 0 && batch > 0 && node_mars && element_mars && params && nids &&
        (num_edges == 0 || (cids && pids))) {
        // a wave per block up to 16384 waves, then a few blocks each
        const int64_t share = (num_nblocks + 16383) / 16384;
        const int per = (int)(share < 64 ? share : 64);
        for_grid_chunks((num_nblocks + 4 * per - 1) / (4 * per), 256, [&](int64_t b0, int64_t n) {
            sparse::block_clear_rows<<<dim3((unsigned)n), dim3(256), 0, reinterpret_cast<hipStream_t>(stream)>>>(
                node_mars, nids, num_nblocks, block_size, batch, per, b0);
        });
    }
    return fl_sparse_blocked_fwd(node_mars, element_mars, params, nids, cids, pids, num_nblocks, num_edges, block_size,
                                 batch, q16, params_are_log, stream);
}
