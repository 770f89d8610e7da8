// Aggregation multigrid for the PSPG systems: per-assembly setup (Galerkin coarse
// operators, block-Jacobi inverses, dense inverse of the coarsest level) and the V-cycle
// used as BiCGSTAB's right preconditioner, each batched over cases and levels through work
// tables.  The hierarchy's structure comes from amg_hierarchy.cpp; see amg.hpp for the
// transfer.
//
// V-cycle on level l (input r_l, output z_l; level 0 reads p or s and writes ph or sh):
//   w = omega B^-1 r                      (block-Jacobi pre-smoothing: at level 0 done by the
//                                          BiCGSTAB kernel that forms r_0, on coarser levels by
//                                          the restriction above)
//   t = r - A w                           (k_amg_res; levels >= 1: k_amg_rr or k_amg_res_nodes)
//   r_{l+1} = P^T t                       (k_amg_restrict, gather over aggregate members; k_amg_rr)
//   z_{l+1} = V-cycle(l+1)  /  A_c^-1 r_c (k_amg_tail, dense inverse on the coarsest)
//   w' = w + alpha P z_{l+1}              (alpha > 1 over-corrects the piecewise-constant
//                                          interpolation)
//   z = w' + omega B^-1 (r - A w')        (k_amg_post, post-smoothing; r - A w' is formed
//       = w' + omega B^-1 (t - alpha (A P) z_{l+1})   from t with the set-up product A P)
// Every vector of the cycle is node-blocked (entry i nf + s), as BiCGSTAB's are.
// What bounds it: on level 0 the matrix's bytes (large cases), elsewhere a chain of dependent loads
// of 4-6 us per launch.  With a launch of its own for every residual, restriction and solve a
// V-cycle took 13 launches and 48 us on 20k nodes in 2D (five levels), now 8 and 37 us; on 263k nodes
// in 3D 141 -> 131 us.
// Every reduction is a fixed-order gather, so a case's V-cycle does not depend on the batch.
#include <type_traits>

#include "common.hpp"
#include "ellspmv.hpp"
#include "nodespmv.hpp"
#include "views.hpp"

namespace pfem {

namespace {

__device__ __forceinline__ bool row_full_flags(uint8_t f, int s, int D) {
    return (s < D) ? (f & (NODE_BOUND | NODE_FREE)) == 0 : (f & NODE_FREE) == 0;
}

__device__ __forceinline__ long long row_start_of(const int4& inf, int s, int D, int mom_nnz) {
    return (s < D) ? (long long)s * mom_nnz + inf.x : (long long)D * mom_nnz + inf.y;
}

constexpr int kTailBlock = 1024;
constexpr int kRrMembers = 64;  // members of an aggregate that k_amg_rr stages at a time

}  // namespace

// ---- setup --------------------------------------------------------------------------------

// Galerkin coarse operator of level l >= 1: entry block (I, J) = P^T A P = the sum over the
// members i of aggregate I of the finer level's A P block (i, J), gathered in member order
// (A P already holds the finer blocks (i, j) summed over j in J, level 0's masked to full rows
// and columns).  L lanes per coarse node, lane k owns entry k of the node's list.
template <typename T, typename ST, int L>
__device__ __forceinline__ void galerkin_body(const AmgView<T>& V, const EllMatT<ST>& F, const BlockTask& task) {
    constexpr int NPB = kBlock / L;
    const int lane = threadIdx.x % L;
    const int nf = V.A.nf, D = nf - 1, nf2 = nf * nf;
    for (long long I = (long long)task.block * NPB + threadIdx.x / L; I < V.A.N; I += (long long)task.nblocks * NPB) {
        const int4 inf = V.A.info[I];
        const int deg = inf.z;
        const int self = V.self_rank[I];
        for (int k = lane; k < deg; k += L) {
            const int mc = V.A.nbr_ptr[I] + k;
            double blk[kMaxNf][kMaxNf];
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s)
#pragma unroll
                for (int t = 0; t < kMaxNf; ++t) blk[s][t] = 0.0;
            for (int q = V.gal_ptr[mc]; q < V.gal_ptr[mc + 1]; ++q) {
                const int2 src = V.gal_src[q];
                const long long c = src.x / kEllSlice, r = src.x % kEllSlice;
                const ST* b = F.vals + ((long long)F.soff[c] + src.y) * nf2 * kEllSlice + r;
#pragma unroll
                for (int s = 0; s < kMaxNf; ++s) {
                    if (s >= nf) continue;
#pragma unroll
                    for (int t = 0; t < kMaxNf; ++t)
                        if (t < nf) blk[s][t] += (double)b[(long long)(s * nf + t) * kEllSlice];
                }
            }
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s) {
                if (s >= nf) continue;
                const long long rs = row_start_of(inf, s, D, V.A.mom_nnz) + k;
#pragma unroll
                for (int t = 0; t < kMaxNf; ++t) {
                    if (t >= nf) continue;
                    double v = blk[s][t];
                    if (k == self && s == t && v == 0.0) v = 1.0;  // DOF with no member DOF: decoupled
                    V.vals_out[rs + (long long)t * deg] = (T)v;
                }
            }
        }
    }
}

template <typename T, typename ST>
__device__ __forceinline__ void galerkin_lanes(const AmgView<T>& V, const EllMatT<ST>& F, const BlockTask& task) {
    if (V.lanes == 4) galerkin_body<T, ST, 4>(V, F, task);
    else if (V.lanes == 8) galerkin_body<T, ST, 8>(V, F, task);
    else galerkin_body<T, ST, 16>(V, F, task);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_galerkin(const AmgView<T>* __restrict__ views,
                                                         const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (V.FAPf.vals) galerkin_lanes<T, float>(V, V.FAPf, task);
    else galerkin_lanes<T, T>(V, V.FAP, task);
}

// Block-Jacobi inverse of a coarse level (the diagonal nf x nf block of each node).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_bjac(const AmgView<T>* __restrict__ views,
                                                     const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    const int nf = V.A.nf, D = nf - 1, N = V.A.N;
    for (long long I = (long long)task.block * kBlock + threadIdx.x; I < N; I += (long long)task.nblocks * kBlock) {
        const int4 inf = V.A.info[I];
        const int self = V.self_rank[I];
        double m[4][8];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < 8; ++t) m[s][t] = (t - 4 == s) ? 1.0 : 0.0;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s >= nf) {
                m[s][s] = 1.0;  // padding rows: identity
                continue;
            }
            const long long rs = row_start_of(inf, s, D, V.A.mom_nnz) + self;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (t < nf) m[s][t] = (double)V.A.vals[rs + (long long)t * inf.z];
        }
        gj_invert4<true>(m);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (s < nf && t < nf) V.binv_out[(long long)(s * nf + t) * N + I] = (T)m[s][4 + t];
    }
}

// A P of a level with a coarser one: entry block (i, J) sums the blocks (i, j) of i's
// neighbours j in aggregate J (gather list, fixed order).  Level 0 keeps only full rows
// (i, s) and full columns (j, t): P prolongates to full rows only, and a row holding only
// its diagonal has no entry off it.  Written in the sliced ELL layout, padding ranks of
// each node's slice as zeros.
template <typename T, int L>
__device__ __forceinline__ void ap_body(const AmgView<T>& V, const BlockTask& task) {
    constexpr int NPB = kBlock / L;
    const int lane = threadIdx.x % L;
    const int nf = V.A.nf, D = nf - 1;
    const NodeMat<T>& A = V.A;
    const EllMatT<T>& P = V.AP;
    for (long long i = (long long)task.block * NPB + threadIdx.x / L; i < P.N; i += (long long)task.nblocks * NPB) {
        const int e0 = V.ap_ptr[i], pdeg = V.ap_ptr[i + 1] - e0;
        const long long c = i / kEllSlice, r = i % kEllSlice;
        const long long b = P.soff[c];
        const int W = P.soff[c + 1] - (int)b;
        const int4 ainf = A.info[i];
        const int anb = A.nbr_ptr[i];
        const uint8_t fi = (uint8_t)ainf.w;
        for (int m = lane; m < W; m += L) {
            double blk[kMaxNf][kMaxNf];
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s)
#pragma unroll
                for (int t = 0; t < kMaxNf; ++t) blk[s][t] = 0.0;
            const int qe = m < pdeg ? V.ap_gptr[e0 + m + 1] : 0;
            for (int q = m < pdeg ? V.ap_gptr[e0 + m] : 0; q < qe; ++q) {
                const int k = V.ap_gsrc[q];
                const uint8_t fj = V.mask ? V.flags[A.nbr_idx[anb + k]] : (uint8_t)0;
#pragma unroll
                for (int s = 0; s < kMaxNf; ++s) {
                    if (s >= nf) continue;
                    if (V.mask && !row_full_flags(fi, s, D)) continue;
                    const long long rs = row_start_of(ainf, s, D, A.mom_nnz) + k;
#pragma unroll
                    for (int t = 0; t < kMaxNf; ++t) {
                        if (t >= nf) continue;
                        if (V.mask && !row_full_flags(fj, t, D)) continue;
                        blk[s][t] += (double)A.vals[rs + (long long)t * ainf.z];
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s)
#pragma unroll
                for (int t = 0; t < kMaxNf; ++t)
                    if (s < nf && t < nf) {
                        const long long q = ((b + m) * nf * nf + s * nf + t) * kEllSlice + r;
                        if (V.ap_out32) V.ap_out32[q] = (float)blk[s][t];
                        else V.ap_out[q] = (T)blk[s][t];
                    }
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_ap(const AmgView<T>* __restrict__ views,
                                                   const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (V.ap_lanes == 4) ap_body<T, 4>(V, task);
    else if (V.ap_lanes == 8) ap_body<T, 8>(V, task);
    else ap_body<T, 16>(V, task);
}

// Dense inverse of the coarsest level (one workgroup per case; Gauss-Jordan in LDS without
// pivoting: the coarse Galerkin operators keep positive diagonals; a vanishing pivot is
// replaced by 1, which decouples that unknown).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_dense(const AmgView<T>* __restrict__ views,
                                                      const BlockTask* __restrict__ tasks) {
    __shared__ double a[kAmgMaxDense * kAmgMaxDense];
    __shared__ double pivrow[kAmgMaxDense];
    __shared__ double colk[kAmgMaxDense];
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    const int n = V.nc, N = V.A.N, nf = V.A.nf, D = nf - 1;
    for (int e = threadIdx.x; e < n * n; e += kBlock) a[e] = 0.0;
    __syncthreads();
    // scatter the node-block values: unknown (I, s) is I nf + s
    for (int I = threadIdx.x; I < N; I += kBlock) {
        const int4 inf = V.A.info[I];
        const int nb = V.A.nbr_ptr[I];
        for (int k = 0; k < inf.z; ++k) {
            const int J = V.A.nbr_idx[nb + k];
            for (int s = 0; s < nf; ++s) {
                const long long rs = row_start_of(inf, s, D, V.A.mom_nnz) + k;
                for (int t = 0; t < nf; ++t) a[(I * nf + s) * n + (J * nf + t)] = (double)V.A.vals[rs + (long long)t * inf.z];
            }
        }
    }
    __syncthreads();
    // in-place Gauss-Jordan inversion with partial pivoting: step k brings the largest entry of
    // column k (rows >= k) to the diagonal, scales row k by its inverse and eliminates column k
    // from every other row, storing the inverse's column k in place of the eliminated one; the
    // row exchanges are undone on the inverse's columns at the end, last one first.  A column
    // that is zero on and below the diagonal (an exactly singular operator) keeps a unit pivot.
    __shared__ int perm[kAmgMaxDense];
    for (int k = 0; k < n; ++k) {
        if (threadIdx.x == 0) {
            int r = k;
            double best = fabs(a[k * n + k]);
            for (int i = k + 1; i < n; ++i) {
                const double v = fabs(a[i * n + k]);
                if (v > best) {
                    best = v;
                    r = i;
                }
            }
            perm[k] = r;
        }
        __syncthreads();
        const int r = perm[k];
        if (r != k)
            for (int j = threadIdx.x; j < n; j += kBlock) {
                const double t = a[k * n + j];
                a[k * n + j] = a[r * n + j];
                a[r * n + j] = t;
            }
        __syncthreads();
        double p = a[k * n + k];
        p = (p != 0.0) ? 1.0 / p : 1.0;
        for (int j = threadIdx.x; j < n; j += kBlock) {
            pivrow[j] = (j == k) ? p : a[k * n + j] * p;
            colk[j] = a[j * n + k];
        }
        __syncthreads();
        for (int e = threadIdx.x; e < n * n; e += kBlock) {
            const int i = e / n, j = e - i * n;
            if (i == k) a[e] = pivrow[j];
            else if (j == k) a[e] = -colk[i] * p;
            else a[e] -= colk[i] * pivrow[j];
        }
        __syncthreads();
    }
    for (int k = n - 1; k >= 0; --k) {
        const int r = perm[k];
        if (r != k)
            for (int i = threadIdx.x; i < n; i += kBlock) {
                const double t = a[i * n + k];
                a[i * n + k] = a[i * n + r];
                a[i * n + r] = t;
            }
        __syncthreads();
    }
    for (int e = threadIdx.x; e < n * n; e += kBlock) V.dense[e] = a[e];
}

// ---- V-cycle -----------------------------------------------------------------------------

// Level 0, over the system's ELL copy; an FP64 hierarchy reads the FP32 copy of the values when
// the view has one (E0f).
template <int NF, int MODE, typename T>
__device__ __forceinline__ void res_rows(const AmgView<T>& V, const BlockTask& task, int which) {
    auto xat = [&](long long j, T (&xv)[NF]) { at_node<NF>((const T*)V.w, j, xv); };
    auto prod = [&](long long c, int k0, int step, T (&acc)[NF]) {
        if (V.E0f.vals) slice_part<NF, (MODE & ELL_STREAM) != 0>(V.E0f, c, k0, step, xat, acc);
        else slice_part<NF, (MODE & ELL_STREAM) != 0>(V.E0, c, k0, step, xat, acc);
    };
    auto pre = [&](long long i, int f) { return (T)V.r0[which][i * NF + f]; };
    auto fin = [&](long long i, int f, const T (&y)[NF], T r, int h) {
        if (!h) V.t[i * NF + f] = r - at_field(y, f);
    };
    slice_products<NF, MODE, T>(task, V.E0.nsl, V.E0.N, prod, pre, fin);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_amg_res(const AmgView<T>* __restrict__ views,
                                                    const BlockTask* __restrict__ tasks, int which) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    PFEM_NF_MODE(res_rows, STREAM, V.A.nf, V.split, V, task, which);
}

// Residual of a level l >= 1 on its own, `lanes` lanes per node.
template <typename T, int L>
__device__ __forceinline__ void res_nodes(const AmgView<T>& V, const BlockTask& task) {
    constexpr int NPB = kBlock / L;
    const int lane = threadIdx.x % L, nf = V.A.nf;
    for (long long i = (long long)task.block * NPB + threadIdx.x / L; i < V.A.N; i += (long long)task.nblocks * NPB) {
        T y[kMaxNf];
        node_spmv<L, true>(V.A, (const T*)V.w, i, lane, y);
        if (lane < nf) V.t[i * nf + lane] = V.r[i * nf + lane] - pick(y, lane);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_res_nodes(const AmgView<T>* __restrict__ views,
                                                          const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    if (V.lanes == 4) res_nodes<T, 4>(V, task);
    else if (V.lanes == 8) res_nodes<T, 8>(V, task);
    else res_nodes<T, 16>(V, task);
}

// Pre-smoothing of aggregate I on level l+1 (not the coarsest), field f: it is local to I.
template <typename T>
__device__ __forceinline__ void pre_smooth(const AmgView<T>& Vn, long long I, int f, int nf, int Nc,
                                           const double (&sum)[kMaxNf]) {
    T w = 0;
#pragma unroll
    for (int t = 0; t < kMaxNf; ++t)
        if (t < nf) w = fma(Vn.binv[(long long)(f * nf + t) * Nc + I], (T)sum[t], w);
    Vn.w[I * nf + f] = (T)Vn.omega * w;
}

// Residual and restriction of a level l >= 1 in one pass, a workgroup per aggregate: its lane
// groups take the aggregate's members (every node of a coarse level has an aggregate) and form
// t = r - A w there, then kRestrictLanes lanes per field sum it in k_amg_restrict's order.  The
// launches of a large batch take k_amg_res_nodes and k_amg_restrict instead, which give the same bits.
template <typename T, int L>
__device__ __forceinline__ void rr_body(const AmgView<T>& V, const AmgView<T>& Vn, const BlockTask& task,
                                        T (&tl)[kRrMembers * kMaxNf], double (&red)[kMaxNf]) {
    constexpr int R = kRestrictLanes;
    static_assert(kRrMembers % R == 0 && R * kMaxNf <= 64, "a lane's members keep their order over the rounds");
    const int lane = threadIdx.x % L, nf = V.A.nf, Nc = V.next_N, rl = threadIdx.x % R, rf = threadIdx.x / R;
    for (int I = task.block; I < Nc; I += task.nblocks) {
        const int m1 = V.agg_ptr[I + 1];
        double acc = 0.0;
        for (int m0 = V.agg_ptr[I]; m0 < m1; m0 += kRrMembers) {
            const int cnt = min(kRrMembers, m1 - m0);
            for (int m = threadIdx.x / L; m < cnt; m += kBlock / L) {
                const long long i = V.agg_nodes[m0 + m];
                T y[kMaxNf];
                node_spmv<L, true>(V.A, (const T*)V.w, i, lane, y);
                if (lane < nf) {
                    const T t = V.r[i * nf + lane] - pick(y, lane);
                    V.t[i * nf + lane] = t;
                    tl[m * nf + lane] = t;
                }
            }
            __syncthreads();
            if (rf < nf)
                for (int m = rl; m < cnt; m += R) acc += (double)tl[m * nf + rf];
            __syncthreads();
        }
        if (rf < nf) {
            acc = group_sum<R>(acc);
            if (rl == 0) red[rf] = acc;
        }
        __syncthreads();
        if ((int)threadIdx.x < nf) {
            const int f = threadIdx.x;
            V.next_r[(long long)I * nf + f] = (T)red[f];
            if (Vn.dense == nullptr) pre_smooth(Vn, I, f, nf, Nc, red);
        }
        __syncthreads();
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_rr(const AmgView<T>* __restrict__ views,
                                                   const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    const AmgView<T>& Vn = views[task.case_id + 1];  // level l+1 (views of a case are consecutive)
    __shared__ T tl[kRrMembers * kMaxNf];
    __shared__ double red[kMaxNf];
    if (V.lanes == 4) rr_body<T, 4>(V, Vn, task, tl, red);
    else if (V.lanes == 8) rr_body<T, 8>(V, Vn, task, tl, red);
    else rr_body<T, 16>(V, Vn, task, tl, red);
}

// r_{l+1}(I, s) = sum over the members i of aggregate I of t(i, s) (level 0: full rows only);
// kRestrictLanes lanes per aggregate share its members (aggregates hold 5-30 nodes).  When
// level l+1 is not the coarsest, its pre-smoothing is applied here as well.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_amg_restrict(const AmgView<T>* __restrict__ views,
                                                         const BlockTask* __restrict__ tasks) {
    constexpr int L = kRestrictLanes, NPB = kBlock / L;
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    const AmgView<T>& Vn = views[task.case_id + 1];  // level l+1 (views of a case are consecutive)
    const int nf = V.A.nf, D = nf - 1, Nc = V.next_N;
    const int lane = threadIdx.x % L;
    for (long long I = (long long)task.block * NPB + threadIdx.x / L; I < Nc; I += (long long)task.nblocks * NPB) {
        double acc[kMaxNf] = {0.0, 0.0, 0.0, 0.0};
        for (int m = V.agg_ptr[I] + lane; m < V.agg_ptr[I + 1]; m += L) {
            const int i = V.agg_nodes[m];
            const uint8_t f = V.mask ? V.flags[i] : (uint8_t)0;
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s)
                if (s < nf && (!V.mask || row_full_flags(f, s, D))) acc[s] += (double)V.t[(long long)i * nf + s];
        }
#pragma unroll
        for (int s = 0; s < kMaxNf; ++s)
            if (s < nf) acc[s] = group_sum<L>(acc[s]);
        if (lane < nf) {
            V.next_r[I * nf + lane] = (T)pick(acc, lane);
            if (Vn.dense == nullptr) pre_smooth(Vn, I, lane, nf, Nc, acc);
        }
    }
}

// The end of the V-cycle in one workgroup per case: on the coarsest level z = A_c^-1 r (8 lanes
// per unknown), and with task.pad the level above it too (kAmgTailNodes), its residual and
// restriction before and its post-smoothing after, with t, r_c and z_c in LDS.
template <typename T, int L>
__device__ __forceinline__ void tail_down(const AmgView<T>& V, T* __restrict__ tl, double* __restrict__ rc) {
    const int lane = threadIdx.x % L, nf = V.A.nf;
    for (int i = threadIdx.x / L; i < V.A.N; i += kTailBlock / L) {
        T y[kMaxNf];
        node_spmv<L, true>(V.A, (const T*)V.w, i, lane, y);
        if (lane < nf) tl[i * nf + lane] = V.r[(long long)i * nf + lane] - pick(y, lane);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < V.next_N * nf; k += kTailBlock) {
        const int I = k / nf, f = k - I * nf;
        double acc = 0.0;
        for (int m = V.agg_ptr[I]; m < V.agg_ptr[I + 1]; ++m) acc += (double)tl[V.agg_nodes[m] * nf + f];
        rc[k] = (double)(T)acc;
    }
    __syncthreads();
}

template <typename T, int L>
__device__ __forceinline__ void tail_up(const AmgView<T>& V, const T* __restrict__ tl, const T* __restrict__ zc) {
    const int lane = threadIdx.x % L, nf = V.A.nf, N = V.A.N;
    const T om = (T)V.omega, al = (T)V.alpha;
    for (int i = threadIdx.x / L; i < N; i += kTailBlock / L) {
        const int c = i / kEllSlice, r = i % kEllSlice, b = V.AP.soff[c], W = V.AP.soff[c + 1] - b;
        T y[kMaxNf] = {T(0), T(0), T(0), T(0)};
        for (int k = lane; k < W; k += L) {
            const int J = V.AP.idx[(long long)(b + k) * kEllSlice + r];
            const T* __restrict__ a = V.AP.vals + (long long)(b + k) * nf * nf * kEllSlice + r;
#pragma unroll
            for (int s = 0; s < kMaxNf; ++s)
#pragma unroll
                for (int t = 0; t < kMaxNf; ++t)
                    if (s < nf && t < nf) y[s] += a[(long long)(s * nf + t) * kEllSlice] * zc[J * nf + t];
        }
        T d[kMaxNf];
#pragma unroll
        for (int s = 0; s < kMaxNf; ++s) d[s] = s < nf ? tl[i * nf + s] - al * group_sum<L>(y[s]) : T(0);
        if (lane < nf) {
            T acc = 0;
#pragma unroll
            for (int t = 0; t < kMaxNf; ++t)
                if (t < nf) acc += V.binv[(long long)(lane * nf + t) * N + i] * d[t];
            const long long q = (long long)i * nf + lane;
            V.z[q] = V.w[q] + al * zc[V.fine_agg[i] * nf + lane] + om * acc;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kTailBlock) void k_amg_tail(const AmgView<T>* __restrict__ views,
                                                         const BlockTask* __restrict__ tasks) {
    __shared__ T tl[kAmgTailNodes * kMaxNf];
    __shared__ double rc[kAmgMaxDense];
    __shared__ T zc[kAmgMaxDense];
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    const int n = V.nc;
    const AmgView<T>& Vf = views[task.case_id - task.pad];  // the level above
    if (task.pad) {
        if (Vf.lanes == 4) tail_down<T, 4>(Vf, tl, rc);
        else if (Vf.lanes == 8) tail_down<T, 8>(Vf, tl, rc);
        else tail_down<T, 16>(Vf, tl, rc);
    } else {
        for (int k = threadIdx.x; k < n; k += kTailBlock) rc[k] = (double)V.r[k];
        __syncthreads();
    }
    const int lane = threadIdx.x % 8;
    for (int row = threadIdx.x / 8; row < n; row += kTailBlock / 8) {
        double acc = 0.0;
        for (int j = lane; j < n; j += 8) acc += V.dense[row * n + j] * rc[j];
        acc = group_sum<8>(acc);
        if (lane == 0) {
            zc[row] = (T)acc;
            if (!task.pad) V.z[row] = (T)acc;
        }
    }
    if (!task.pad) return;
    __syncthreads();
    if (Vf.ap_lanes == 4) tail_up<T, 4>(Vf, tl, zc);
    else if (Vf.ap_lanes == 8) tail_up<T, 8>(Vf, tl, zc);
    else tail_up<T, 16>(Vf, tl, zc);
}

// z = w' + omega B^-1 (t - alpha (A P) z_{l+1}),  w' = w + alpha P z_{l+1} (level 0: full
// rows only); A P in FP32 when the view holds it so (APf).
template <int NF, int MODE, typename T>
__device__ __forceinline__ void post_rows(const AmgView<T>& V, const BlockTask& task, int which) {
    struct Pre {
        T w, z, t[NF], brow[NF];
    };
    const int N = V.A.N;
    const T om = (T)V.omega, al = (T)V.alpha;
    auto xat = [&](long long j, T (&xv)[NF]) { at_node<NF>(V.next_z.get(), j, xv); };
    auto prod = [&](long long c, int k0, int step, T (&acc)[NF]) {
        if (V.APf.vals) slice_part<NF, (MODE & ELL_STREAM) != 0>(V.APf, c, k0, step, xat, acc);
        else slice_part<NF, (MODE & ELL_STREAM) != 0>(V.AP, c, k0, step, xat, acc);
    };
    auto pre = [&](long long i, int f) {
        Pre o;
        const int I = V.fine_agg[i];
        const bool full = I >= 0 && (!V.mask || row_full_flags(V.flags[i], f, NF - 1));
        o.w = V.w[i * NF + f];
        at_node<NF>((const T*)V.t, i, o.t);
        load_block_row<NF>((const T*)V.binv, N, f, i, o.brow);
        const T z = V.next_z[(long long)max(I, 0) * NF + f];
        o.z = full ? z : T(0);
        return o;
    };
    auto fin = [&](long long i, int f, const T (&y)[NF], const Pre& o, int h) {
        if (h) return;
        T d[NF];
#pragma unroll
        for (int t = 0; t < NF; ++t) d[t] = o.t[t] - al * y[t];
        const T out = (o.w + al * o.z) + om * block_row<NF>(o.brow, d);
        if (V.level == 0) V.out0[which][i * NF + f] = (double)out;
        else V.z[i * NF + f] = out;
    };
    slice_products<NF, MODE, T>(task, V.AP.nsl, N, prod, pre, fin);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_amg_post(const AmgView<T>* __restrict__ views,
                                                     const BlockTask* __restrict__ tasks, int which) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const AmgView<T>& V = views[task.case_id];
    if (*V.done_flag) return;
    PFEM_NF_MODE(post_rows, STREAM, V.A.nf, V.split, V, task, which);
}

// ---- launchers ---------------------------------------------------------------------------
template <typename T>
void launch_amg_galerkin(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_galerkin<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_bjac(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_bjac<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_dense(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_dense<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_res(const AmgView<T>* v, const BlockTask* t, int nt, int which, bool stream, hipStream_t s) {
    if (stream) k_amg_res<T, true><<<nt, kBlock, 0, s>>>(v, t, which);
    else k_amg_res<T, false><<<nt, kBlock, 0, s>>>(v, t, which);
}
template <typename T>
void launch_amg_restrict(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_restrict<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_rr(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_rr<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_res_nodes(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_res_nodes<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_tail(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_tail<T><<<nt, kTailBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_ap(const AmgView<T>* v, const BlockTask* t, int nt, hipStream_t s) {
    k_amg_ap<T><<<nt, kBlock, 0, s>>>(v, t);
}
template <typename T>
void launch_amg_post(const AmgView<T>* v, const BlockTask* t, int nt, int which, bool stream, hipStream_t s) {
    if (stream) k_amg_post<T, true><<<nt, kBlock, 0, s>>>(v, t, which);
    else k_amg_post<T, false><<<nt, kBlock, 0, s>>>(v, t, which);
}

#define PFEM_AMG_INSTANTIATE(T)                                                                    \
    template void launch_amg_galerkin<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);   \
    template void launch_amg_bjac<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);       \
    template void launch_amg_dense<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);      \
    template void launch_amg_res<T>(const AmgView<T>*, const BlockTask*, int, int, bool, hipStream_t); \
    template void launch_amg_restrict<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);   \
    template void launch_amg_rr<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);         \
    template void launch_amg_res_nodes<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);  \
    template void launch_amg_tail<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);       \
    template void launch_amg_ap<T>(const AmgView<T>*, const BlockTask*, int, hipStream_t);         \
    template void launch_amg_post<T>(const AmgView<T>*, const BlockTask*, int, int, bool, hipStream_t);
PFEM_AMG_INSTANTIATE(double)
PFEM_AMG_INSTANTIATE(float)

}  // namespace pfem
