// SpMV over the sliced ELL copy of a PSPG system (EllMat): lane r of a wavefront computes
// the NF rows of node 64 c + r of slice c.  Each rank k is one column node j (one index
// load, NF gathers of x) and NF*NF value loads, each 64 consecutive doubles per wavefront.
// Of matrices larger than the caches the values are loaded non-temporally (ELL_STREAM): they are
// read once per launch, and without the hint they evict the x entries and the results from the
// caches (516 MB matrix: 98.7 -> 90.0 us per launch; 2D 900k nodes: 104 -> 94 us).
#pragma once

#include "common.hpp"
#include "nodespmv.hpp"
#include "views.hpp"

namespace pfem {

// acc[s] = (A x) of row (64 c + lane, s) over the ranks k0, k0 + step, ... of slice c, with values
// of type VT and vectors and sums of type XT; xat(j, xv) gives the NF entries of x at node j.
// Lanes past the last node compute values that the callers drop.
template <int NF, bool STREAM, typename VT, typename XT, class X>
__device__ __forceinline__ void slice_part(const EllMatT<VT>& E, long long c, int k0, int step, X&& xat,
                                           XT (&acc)[NF]) {
    const int lane = threadIdx.x & (kEllSlice - 1);
    const long long b = E.soff[c];
    const int W = E.soff[c + 1] - (int)b;
    const VT* __restrict__ vb = E.vals + b * (NF * NF * kEllSlice) + lane;
    const int* __restrict__ ib = E.idx + b * kEllSlice + lane;
#pragma unroll
    for (int s = 0; s < NF; ++s) acc[s] = XT(0);
#pragma unroll 2
    for (int k = k0; k < W; k += step) {
        const long long j = ib[(long long)k * kEllSlice];
        XT a[NF][NF];
#pragma unroll
        for (int s = 0; s < NF; ++s)
#pragma unroll
            for (int t = 0; t < NF; ++t)
            {
                const VT* q = vb + ((long long)k * NF * NF + s * NF + t) * kEllSlice;
                a[s][t] = (XT)(STREAM ? ld_stream(q) : *q);
            }
        XT xv[NF];
        xat(j, xv);
#pragma unroll
        for (int s = 0; s < NF; ++s)
#pragma unroll
            for (int t = 0; t < NF; ++t) acc[s] += a[s][t] * xv[t];
    }
}

// Entries of a field-blocked vector x[t N + j], and of a node-blocked one x[j NF + t].
template <int NF, typename T>
__device__ __forceinline__ void at_fields(const T* __restrict__ x, long long N, long long j, T (&xv)[NF]) {
#pragma unroll
    for (int t = 0; t < NF; ++t) xv[t] = x[j + t * N];
}
template <int NF, typename T>
__device__ __forceinline__ void at_node(const T* __restrict__ x, long long j, T (&xv)[NF]) {
#pragma unroll
    for (int t = 0; t < NF; ++t) xv[t] = x[j * NF + t];
}

// y[f] without dynamic register indexing (the values are pinned in registers: a selected address
// would put the array into LDS).
template <int NF, typename T>
__device__ __forceinline__ T at_field(const T (&y)[NF], int f) {
    T a = y[0], b = y[1], c = y[2], d = y[NF - 1];
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
    const T lo = (f & 1) ? b : a, hi = (f & 1) ? d : c;
    return (f & 2) ? hi : lo;
}

// Row f of B^-1 times the node's NF values.
template <int NF, typename T>
__device__ __forceinline__ T block_row(const T (&brow)[NF], const T (&y)[NF]) {
    T acc = 0;
#pragma unroll
    for (int t = 0; t < NF; ++t) acc += brow[t] * y[t];
    return acc;
}
template <int NF, typename T>
__device__ __forceinline__ void load_block_row(const T* __restrict__ binv, long long nodes, int f, long long i,
                                               T (&brow)[NF]) {
#pragma unroll
    for (int t = 0; t < NF; ++t) brow[t] = binv[(f * NF + t) * nodes + i];
}

// A pass of products over the workgroup's slices of a matrix with `rows` row nodes:
// prod(c, k0, step, acc) leaves the product of slice c over the ranks k0, k0 + step, ...;
// pre(i, f) loads what row f of node i < rows needs besides (issued before any store), and
// fin(i, f, y, pre's result, h) finishes that row from the node's NF products y, h = 0 and then 1
// (a result per pass: the stores of one lane's fields to one vector then merge).
// ELL_SPLIT: the four wavefronts share a slice, add their parts through LDS in order and finish the
// slice's rows in the order of node-blocked vectors (thread e: node e / NF, field e % NF); else
// each wavefront takes whole slices, one lane per node.
template <int NF, int MODE, typename T, class PR, class PRE, class FI>
__device__ __forceinline__ void slice_products(const BlockTask& task, int nsl, long long rows, PR&& prod, PRE&& pre,
                                               FI&& fin) {
    const Seg sg = xcd_segment(task, nsl);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if constexpr ((MODE & ELL_SPLIT) != 0) {
        __shared__ T red[kWaves][NF][kEllSlice];
        const int n = threadIdx.x / NF, f = threadIdx.x - n * NF;
        for (int l = sg.lb; l < sg.ns; l += sg.cnt) {
            const long long c = sg.n0 + l, i = c * kEllSlice + n;
            const bool own = n < kEllSlice && i < rows;
            // clamped and not branched around: a value loaded in a branch is waited for at its end
            const auto o = pre(own ? i : rows - 1, f);
            T acc[NF];
            prod(c, wave, kWaves, acc);
#pragma unroll
            for (int t = 0; t < NF; ++t) red[wave][t][lane] = acc[t];
            __syncthreads();
            if (own) {
                T y[NF];
#pragma unroll
                for (int t = 0; t < NF; ++t) {
                    y[t] = red[0][t][n];
#pragma unroll
                    for (int w = 1; w < kWaves; ++w) y[t] += red[w][t][n];
                }
                fin(i, f, y, o, 0);
                fin(i, f, y, o, 1);
            }
            __syncthreads();
        }
    } else {
        for (int l = sg.lb * kWaves + wave; l < sg.ns; l += sg.cnt * kWaves) {
            const long long c = sg.n0 + l, i = c * kEllSlice + lane;
            T y[NF];
            decltype(pre(i, 0)) o[NF];
            const long long ic = i < rows ? i : rows - 1;
            if (sizeof(T) == 4)
#pragma unroll
                for (int f = 0; f < NF; ++f) o[f] = pre(ic, f);
            prod(c, 0, 1, y);
            if (sizeof(T) != 4)  // FP64: the registers are the product's
#pragma unroll
                for (int f = 0; f < NF; ++f) o[f] = pre(ic, f);
            if (i >= rows) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int f = 0; f < NF; ++f) fin(i, f, y, o[f], h);
        }
    }
}

// Calls BODY<NF, MODE> for a view's fields and split and the launch's STREAM.
#define PFEM_NF_MODE(BODY, STREAM, nf, split, ...)                                                      \
    do {                                                                                                \
        constexpr int kWhole = (STREAM) ? ELL_STREAM : 0;                                               \
        if ((nf) == 4) (split) ? BODY<4, kWhole | ELL_SPLIT>(__VA_ARGS__) : BODY<4, kWhole>(__VA_ARGS__); \
        else (split) ? BODY<3, kWhole | ELL_SPLIT>(__VA_ARGS__) : BODY<3, kWhole>(__VA_ARGS__);         \
    } while (0)

}  // namespace pfem
