// Node-block SpMV and right-preconditioned BiCGSTAB for a batch of cases, plus the FP64
// iterative-refinement kernels of the mixed-precision solve.
//
// Replaces SparseLU<SparseMatrix<double>, COLAMDOrdering<int>> (analyzePattern / factorize /
// solve at MomContEquationPSPG.inl:281-290) with right-preconditioned BiCGSTAB
// (van der Vorst 1992).  The preconditioner is block Jacobi over the nf x nf diagonal
// block of each node (its velocity and pressure DOFs), or the multigrid V-cycle.
//
// The vector updates are merged into as few launches as the two reductions of an iteration
// allow.  rho is taken from the previous product as (rh, s) - omega (rh, t) (as in the improved
// BiCGSTAB of Yang and Brent 2002), so that the end of one iteration and the start of the next
// are one pass (a rho lost in rounding ends it: kWeakRho in views.hpp); and with block Jacobi the
// preconditioned vectors follow the recurrences of the plain ones (rhat = B^-1 r and vhat = B^-1 v
// are local to a node), so that the products read them from there.  One iteration is
//   block Jacobi (3 launches)                   multigrid M (4 launches and two V-cycles)
//   U: r = s - om t, s = r - al v;              U: the same, with s stored;
//      x += al ph + om (rhat - al vhat);           x += al ph + om sh;
//      rhat = B^-1 r;                              p = r + beta (p - om v)
//      ph = rhat + beta (ph - om vhat)             [V-cycle: ph = M^-1 p]
//   V: v = A ph, vhat = B^-1 v   -> (rh, v)     V: v = A ph                     -> (rh, v)
//   T: t = A (rhat - al vhat)                   S: s = r - al v                 -> (s, s), (rh, s)
//                                                  [V-cycle: sh = M^-1 s]
//       -> (s, s), (rh, s), (t, s),             T: t = A sh  -> (t, s), (t, t), (rh, t)
//          (t, t), (rh, t)
// U also sums (r, r), which the test after V reads.  (Five launches per iteration before, with
// field-blocked vectors; each is a chain of dependent loads that takes ~5 us on a small system.
// Per iteration: 1,001 nodes in 2D 29 -> 15 us, 12k nodes in 3D 59 -> 25 us, 48k Delaunay nodes
// 94 -> 61 us, 72k nodes with FP32 inner solves 68 -> 43 us, the last three with plain value loads
// (ELL_STREAM); above 100k nodes the products are bound by the matrix's bytes.)
//
// Reductions: every workgroup writes its FP64 partial sums to its own place and the next
// kernel's workgroups each re-reduce them in block order — deterministic, and ordered by
// the kernel boundary, so no device-scope fence (an L2 write-back on gfx950) is needed.
// Scalars: two slots used alternately by iteration parity (KScal in views.hpp).
//
// Work split: workgroups are dispatched round-robin over the 8 XCDs; the workgroups of a
// case that land on one XCD own one contiguous range of 64-node slices (every field of those
// nodes), so the SpMV's x gathers (neighbour nodes) and the vectors handed from one
// kernel to the next stay in that XCD's L2.  On small cases a workgroup's four wavefronts share
// a slice: they split the ranks of the product (four times the wavefronts in flight: a case of
// 12k nodes has 188 slices for 1,024 SIMDs) and add their parts through LDS.
#include <hip/hip_ext.h>

#include <type_traits>

#include "common.hpp"
#include "ellspmv.hpp"
#include "nodespmv.hpp"
#include "views.hpp"

namespace pfem {

// Sum of a case's partial sums over the producer's workgroups, in block order; valid in every
// thread.
template <int NV>
__device__ __forceinline__ void reduce_partials(const double* __restrict__ P, int nblk, const int (&slot)[NV],
                                                double (&out)[NV]) {
    __shared__ double bc[NV];
    double acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[j] = 0.0;
    for (int b = threadIdx.x; b < nblk; b += kBlock)
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] += P[slot[j] * kMaxCaseBlocks + b];
    block_sum<NV>(acc);
    if (threadIdx.x == 0)
#pragma unroll
        for (int j = 0; j < NV; ++j) bc[j] = acc[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; ++j) out[j] = bc[j];
}

// Writes this workgroup's partial sums (thread-local contributions).
template <int NV>
__device__ __forceinline__ void write_partials(double (&v)[NV], double* __restrict__ P, int block,
                                               const int (&slot)[NV]) {
    block_sum<NV>(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int j = 0; j < NV; ++j) P[slot[j] * kMaxCaseBlocks + block] = v[j];
}

// y = A x (plain node-block SpMV; pfem_spmv and the Picard paths).
template <typename T, int K>
__global__ __launch_bounds__(kBlock) void k_spmv(NodeMat<T> A, const T* __restrict__ x, T* __restrict__ y) {
    constexpr int NPB = kBlock / K;
    const int lane = threadIdx.x % K;
    for (long long i = (long long)blockIdx.x * NPB + threadIdx.x / K; i < A.N; i += (long long)gridDim.x * NPB) {
        T yv[kMaxNf];
        node_spmv<K>(A, x, i, lane, yv);
        if (lane < A.nf) y[i + (long long)lane * A.N] = pick(yv, lane);
    }
}

// (Re)start: r = b - A x (or b when x_zero), rh = r.
template <int NF, int MODE, typename T>
__device__ __forceinline__ void init_body(const KrylovView<T>& V, const BlockTask& task, double (&part)[3]) {
    const T* __restrict__ x = V.x;
    const long long N = V.nodes;
    auto prod = [&](long long c, int k0, int step, T (&acc)[NF]) {
        if (V.x_zero) {
#pragma unroll
            for (int t = 0; t < NF; ++t) acc[t] = T(0);
        } else {
            slice_part<NF, (MODE & ELL_STREAM) != 0>(V.E, c, k0, step, [&](long long j, T (&xv)[NF]) { at_fields<NF>(x, N, j, xv); }, acc);
        }
    };
    auto pre = [&](long long i, int f) { return V.b[i + f * N]; };
    auto fin = [&](long long i, int f, const T (&y)[NF], T bi, int h) {
        if (h) return;
        const T r = bi - at_field(y, f);
        V.r[i * NF + f] = r;
        V.rh[i * NF + f] = r;
        if (V.x_zero) V.x[i + f * N] = T(0);
        part[0] += (double)r * (double)r;
        part[1] += (double)r * (double)r;
        part[2] += (double)bi * (double)bi;
    };
    slice_products<NF, MODE, T>(task, V.E.nsl, N, prod, pre, fin);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_kry_init(const KrylovView<T>* __restrict__ views,
                                                     const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const KrylovView<T>& V = views[task.case_id];
    if (!V.sc->req_init) return;
    double part[3] = {0.0, 0.0, 0.0};
    PFEM_NF_MODE(init_body, STREAM, V.nf, V.split, V, task, part);
    constexpr int slots[3] = {P_RHR, P_RR, P_BB};
    write_partials<3>(part, V.partials, task.block, slots);
}

// One workgroup per listed case: finalises a (re)start and writes slot `par` as the
// "previous" slot of the next iteration (which runs with parity par ^ 1).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_kry_init_fin(const KrylovView<T>* __restrict__ views,
                                                         const BlockTask* __restrict__ ids, int count, int par) {
    for (int c = blockIdx.x; c < count; c += gridDim.x) {
        const KrylovView<T>& V = views[ids[c].case_id];
        if (!V.sc->req_init) continue;
        constexpr int slots[3] = {P_RHR, P_RR, P_BB};
        double tot[3];
        reduce_partials<3>(V.partials, V.nblk, slots, tot);
        if (threadIdx.x == 0) {
            KScal& S = *V.sc;
            S.bb = tot[2];
            S.tol2 = S.rtol * S.rtol * tot[2];
            if (S.atol2 > 0.0 && S.atol2 < S.tol2) S.tol2 = S.atol2;
            S.rr = tot[1];
            // (rh = r here)
            S.weak_rho = sizeof(T) == 8 && S.weak < kMaxWeak ? kWeakRho * sqrt(tot[1]) : -1.0;
            S.slot[par].rho = tot[0];
            S.slot[par].alpha = 1.0;
            S.slot[par].omega = 1.0;
            S.slot[par].state = K_FRESH;
            S.true_rr = 1;
            S.req_init = 0;
            if (tot[2] == 0.0 || tot[1] <= S.tol2) S.done = 1;
            else if (!isfinite(tot[1])) S.done = 2;
            else if (S.iters >= S.maxit) S.done = 3;
            else S.done = 0;
        }
        __syncthreads();
    }
}

// What U finds from the iteration's sums.
struct UScal {
    double alpha, omega, beta, rho;
    int state;
    bool sconv, stop;
};

// What thread e of a slice (node e / NF, field e % NF) needs in U.
template <int NF, typename T>
struct UOwn {
    T r, v, t, p, s, ph, sh, x, brow[NF];
};

template <int NF, bool AMG, typename T>
__device__ __forceinline__ UOwn<NF, T> u_load(const KrylovView<T>& V, long long i, int f) {
    const long long q = i * NF + f;
    UOwn<NF, T> o;
    o.r = V.r[q];
    o.v = V.v[q];
    o.t = V.t[q];
    o.p = V.p[q];
    o.s = V.s[q];
    o.ph = V.ph[q];
    o.sh = AMG ? V.sh[q] : T(0);
    o.x = V.x[i + (long long)f * V.nodes];
    load_block_row<NF>((const T*)V.binv, V.nodes, f, i, o.brow);
    return o;
}

// U over the workgroup's slices.  fresh: the first pass after a (re)start (r stands, no iteration
// to finish: what is loaded of the other vectors is dropped); scalars() reduces the iteration's
// sums, after the first slice's loads are issued (those are clamped and not branched around: a
// value loaded in a branch is waited for at its end).
template <int NF, bool AMG, typename T, class SC>
__device__ __forceinline__ void update_rows(const KrylovView<T>& V, const BlockTask& task, bool fresh, SC&& scalars,
                                            double (&part)[1]) {
    __shared__ T rs[kEllSlice * NF];
    const Seg sg = xcd_segment(task, V.E.nsl);
    const int e = threadIdx.x, n = e / NF, f = e - n * NF;
    const long long N = V.nodes;
    UScal S;
    for (int l = sg.lb; l < sg.ns; l += sg.cnt) {
        const long long i = (long long)(sg.n0 + l) * kEllSlice + n, q = i * NF + f;
        const bool own = n < kEllSlice && i < N;
        const UOwn<NF, T> o = u_load<NF, AMG>(V, own ? i : N - 1, f);
        if (l == sg.lb) S = scalars();
        const T a = (T)S.alpha, om = (T)S.omega, be = (T)S.beta;
        T r = o.r, z = T(0);
        if (own) {
            if (!fresh) {
                const T s = AMG ? o.s : r - a * o.v;       // block Jacobi: V.p holds rhat, V.s holds vhat
                const T sh = AMG ? o.sh : o.p - a * o.s;
                V.x[i + (long long)f * N] = o.x + (S.sconv ? a * o.ph : a * o.ph + om * sh);
                r = S.sconv ? s : s - om * o.t;
                V.r[q] = r;
            }
            part[0] += (double)r * (double)r;
            z = r;
            if (AMG && !S.stop) {
                z = fresh ? r : r + be * (o.p - om * o.v);
                V.p[q] = z;
            }
        }
        if (S.stop) continue;
        if (n < kEllSlice) rs[e] = z;
        __syncthreads();
        if (own) {
            T y[NF];
            at_node<NF>((const T*)rs, n, y);
            const T bz = block_row<NF>(o.brow, y);
            if (!AMG) {
                V.p[q] = bz;
                V.ph[q] = fresh ? bz : bz + be * (o.ph - om * o.s);
            } else if (V.mg_w0) {
                V.mg_w0[q] = (double)((T)V.mg_om * bz);
            } else {
                V.mg_w0f[q] = (float)((T)V.mg_om * bz);
            }
        }
        __syncthreads();
    }
}

template <int NF, typename T, class SC>
__device__ __forceinline__ void update_body(const KrylovView<T>& V, const BlockTask& task, bool fresh, SC&& scalars,
                                            double (&part)[1]) {
    if (V.amg) update_rows<NF, true>(V, task, fresh, scalars, part);
    else update_rows<NF, false>(V, task, fresh, scalars, part);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_kry_update(const KrylovView<T>* __restrict__ views,
                                                       const BlockTask* __restrict__ tasks, int par) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const KrylovView<T>& V = views[task.case_id];
    KScal& S = *V.sc;
    if (S.done) return;
    const KSlot prev = S.slot[par ^ 1];
    const bool fresh = prev.state == K_FRESH;
    UScal u{prev.alpha, 0.0, 0.0, prev.rho, K_RUN, false, false};
    auto scalars = [&] {
        if (!fresh) {
            constexpr int sl[5] = {P_SS, P_TS, P_TT, P_RHT, P_RHS};
            double tot[5];
            reduce_partials<5>(V.partials, V.nblk, sl, tot);
            u.sconv = tot[0] <= S.tol2;
            u.omega = u.sconv ? 1.0 : (tot[2] == 0.0 ? 0.0 : tot[1] / tot[2]);
            u.rho = tot[4] - u.omega * tot[3];
            u.beta = (u.rho / prev.rho) * (prev.alpha / u.omega);
            if (u.sconv) u.state = K_CONV;
            else if (u.rho == 0.0 || !isfinite(u.beta)) u.state = K_BREAK;
            u.stop = u.state != K_RUN;
        }
        return u;
    };
    double part[1] = {0.0};
    if (V.nf == 4) update_body<4>(V, task, fresh, scalars, part);
    else update_body<3>(V, task, fresh, scalars, part);
    constexpr int slots[1] = {P_RR};
    write_partials<1>(part, V.partials, task.block, slots);
    if (task.block == 0 && threadIdx.x == 0) {
        // the stop is announced through the slot: S.done would end workgroups of this launch that
        // start late before they have updated their nodes
        S.slot[par].rho = u.rho;
        S.slot[par].state = u.state;
        if (!fresh) {
            S.iters += 1;
            S.true_rr = 0;
        }
    }
}

// V: v = A ph (and vhat = B^-1 v); part = {(rh, v)}.
template <int NF, int MODE, bool AMG, typename T>
__device__ __forceinline__ void v_rows(const KrylovView<T>& V, const BlockTask& task, double (&part)[1]) {
    struct Pre {
        T rh, brow[NF];
    };
    const T* __restrict__ x = V.ph;
    auto prod = [&](long long c, int k0, int step, T (&acc)[NF]) {
        slice_part<NF, (MODE & ELL_STREAM) != 0>(V.E, c, k0, step, [&](long long j, T (&xv)[NF]) { at_node<NF>(x, j, xv); }, acc);
    };
    auto pre = [&](long long i, int f) {
        Pre o;
        o.rh = V.rh[i * NF + f];
        if (!AMG) load_block_row<NF>((const T*)V.binv, V.nodes, f, i, o.brow);
        return o;
    };
    auto fin = [&](long long i, int f, const T (&y)[NF], const Pre& o, int h) {
        if (h) {
            if (!AMG) V.s[i * NF + f] = block_row<NF>(o.brow, y);
            return;
        }
        const T v = at_field(y, f);
        V.v[i * NF + f] = v;
        part[0] += (double)o.rh * (double)v;
    };
    slice_products<NF, MODE, T>(task, V.E.nsl, V.nodes, prod, pre, fin);
}

template <int NF, int MODE, typename T>
__device__ __forceinline__ void v_body(const KrylovView<T>& V, const BlockTask& task, double (&part)[1]) {
    if (V.amg) v_rows<NF, MODE, true>(V, task, part);
    else v_rows<NF, MODE, false>(V, task, part);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_kry_v(const KrylovView<T>* __restrict__ views,
                                                  const BlockTask* __restrict__ tasks, int par) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const KrylovView<T>& V = views[task.case_id];
    KScal& S = *V.sc;
    if (S.done) return;
    double part[1] = {0.0};
    PFEM_NF_MODE(v_body, STREAM, V.nf, V.split, V, task, part);
    constexpr int slots[1] = {P_RV};
    write_partials<1>(part, V.partials, task.block, slots);
}

// Ends the solve when U found so or (r, r) says so; else alpha = rho / (rh, v) of the iteration,
// or a breakdown (every workgroup finds the same).  Tested here and not before the product: one
// more product at the end costs less than a reduction at the head of every one.
template <typename T>
__device__ __forceinline__ bool step_alpha(const KrylovView<T>& V, const BlockTask& task, int par, double& alpha) {
    KScal& S = *V.sc;
    constexpr int rs[2] = {P_RV, P_RR};
    double tot[2];
    // (loaded ahead of the reduction: loads in the tests below are waited for one by one)
    const double rho = S.slot[par].rho, tol2 = S.tol2, weak_rho = S.weak_rho;
    const int state = S.slot[par].state, iters = S.iters, maxit = S.maxit;
    reduce_partials<2>(V.partials, V.nblk, rs, tot);
    alpha = rho / tot[0];
    int stop = 0;
    if (state == K_CONV || tot[1] <= tol2) stop = 1;
    else if (state == K_BREAK || !isfinite(tot[1])) stop = 2;
    else if (iters >= maxit) stop = 3;
    else if (fabs(rho) <= weak_rho * sqrt(tot[1])) stop = 4;
    else if (tot[0] == 0.0 || !isfinite(alpha)) stop = 2;
    if (task.block == 0 && threadIdx.x == 0) {
        S.rr = tot[1];
        S.slot[par].alpha = alpha;
        if (stop) S.done = stop;
    }
    return !stop;
}

// S: s = r - alpha v and the V-cycle's pre-smoothing (multigrid cases only).
template <int NF, typename T>
__device__ __forceinline__ void s_body(const KrylovView<T>& V, const BlockTask& task, double alpha, double (&part)[2]) {
    __shared__ T rs[kEllSlice * NF];
    const Seg sg = xcd_segment(task, V.E.nsl);
    const int e = threadIdx.x, n = e / NF, f = e - n * NF;
    const T a = (T)alpha;
    for (int l = sg.lb; l < sg.ns; l += sg.cnt) {
        const long long i = (long long)(sg.n0 + l) * kEllSlice + n, q = i * NF + f;
        const bool own = n < kEllSlice && i < V.nodes;
        const long long ic = own ? i : V.nodes - 1, qc = ic * NF + f;
        T brow[NF];
        load_block_row<NF>((const T*)V.binv, V.nodes, f, ic, brow);
        const T s = V.r[qc] - a * V.v[qc], rh = V.rh[qc];
        if (own) {
            rs[e] = s;
            V.s[q] = s;
            part[0] += (double)s * (double)s;
            part[1] += (double)rh * (double)s;
        }
        __syncthreads();
        if (own) {
            T y[NF];
            at_node<NF>((const T*)rs, n, y);
            const T w = (T)V.mg_om * block_row<NF>(brow, y);
            if (V.mg_w0) V.mg_w0[q] = (double)w;
            else V.mg_w0f[q] = (float)w;
        }
        __syncthreads();
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_kry_s(const KrylovView<T>* __restrict__ views,
                                                  const BlockTask* __restrict__ tasks, int par) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const KrylovView<T>& V = views[task.case_id];
    if (!V.amg || V.sc->done) return;
    double alpha;
    if (!step_alpha(V, task, par, alpha)) return;
    double part[2] = {0.0, 0.0};
    if (V.nf == 4) s_body<4>(V, task, alpha, part);
    else s_body<3>(V, task, alpha, part);
    constexpr int slots[2] = {P_SS, P_RHS};
    write_partials<2>(part, V.partials, task.block, slots);
}

// T: part = {(t, s), (t, t), (rh, t)} and, with block Jacobi, {(s, s), (rh, s)}.
template <int NF, int MODE, bool AMG, typename T>
__device__ __forceinline__ void t_rows(const KrylovView<T>& V, const BlockTask& task, double alpha, double (&part)[5]) {
    struct Pre {
        T rh, s, r, v;
    };
    const T a = (T)alpha;
    const T* __restrict__ x = AMG ? V.sh : V.p;
    const T* __restrict__ vh = V.s;
    auto prod = [&](long long c, int k0, int step, T (&acc)[NF]) {
        auto xat = [&](long long j, T (&xv)[NF]) {
            at_node<NF>(x, j, xv);
            if (!AMG) {
                T hv[NF];
                at_node<NF>(vh, j, hv);
#pragma unroll
                for (int t = 0; t < NF; ++t) xv[t] -= a * hv[t];
            }
        };
        slice_part<NF, (MODE & ELL_STREAM) != 0>(V.E, c, k0, step, xat, acc);
    };
    auto pre = [&](long long i, int f) {
        const long long q = i * NF + f;
        Pre o{};
        o.rh = V.rh[q];
        if (AMG) {
            o.s = V.s[q];
        } else {
            o.r = V.r[q];
            o.v = V.v[q];
        }
        return o;
    };
    auto fin = [&](long long i, int f, const T (&y)[NF], const Pre& o, int h) {
        if (h) return;
        const T t = at_field(y, f), s = AMG ? o.s : o.r - a * o.v;
        V.t[i * NF + f] = t;
        part[0] += (double)t * (double)s;
        part[1] += (double)t * (double)t;
        part[2] += (double)o.rh * (double)t;
        if (!AMG) {
            part[3] += (double)s * (double)s;
            part[4] += (double)o.rh * (double)s;
        }
    };
    slice_products<NF, MODE, T>(task, V.E.nsl, V.nodes, prod, pre, fin);
}

template <int NF, int MODE, typename T>
__device__ __forceinline__ void t_body(const KrylovView<T>& V, const BlockTask& task, double alpha, double (&part)[5]) {
    if (V.amg) t_rows<NF, MODE, true>(V, task, alpha, part);
    else t_rows<NF, MODE, false>(V, task, alpha, part);
}

template <typename T, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_kry_t(const KrylovView<T>* __restrict__ views,
                                                  const BlockTask* __restrict__ tasks, int par) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const KrylovView<T>& V = views[task.case_id];
    if (V.sc->done) return;
    double part[5] = {0.0, 0.0, 0.0, 0.0, 0.0}, alpha = 0.0;
    if (!V.amg && !step_alpha(V, task, par, alpha)) return;
    PFEM_NF_MODE(t_body, STREAM, V.nf, V.split, V, task, alpha, part);
    if (V.amg) {  // S has written the other two
        double p3[3] = {part[0], part[1], part[2]};
        constexpr int slots[3] = {P_TS, P_TT, P_RHT};
        write_partials<3>(p3, V.partials, task.block, slots);
    } else {
        constexpr int slots[5] = {P_TS, P_TT, P_RHT, P_SS, P_RHS};
        write_partials<5>(part, V.partials, task.block, slots);
    }
}

// Mixed precision: r = b - A x in FP64, r32 = (float) r, ||r||^2 and ||b||^2.
template <int L>
__global__ __launch_bounds__(kBlock) void k_ir_residual(const RefineView* __restrict__ views,
                                                        const BlockTask* __restrict__ tasks) {
    constexpr int NPB = kBlock / L;
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const RefineView& V = views[task.case_id];
    const int lane = threadIdx.x % L;
    double part[2] = {0.0, 0.0};
    for (long long i = (long long)task.block * NPB + threadIdx.x / L; i < V.A.N; i += (long long)task.nblocks * NPB) {
        double ax[kMaxNf];
        node_spmv<L>(V.A, V.x.get(), i, lane, ax);
        if (lane < V.A.nf) {
            const long long row = i + (long long)lane * V.A.N;
            const double bi = V.b[row];
            const double r = bi - pick(ax, lane);
            V.r[row] = r;
            if (V.r32) V.r32[row] = (float)r;
            part[0] += r * r;
            part[1] += bi * bi;
        }
    }
    double tot[2];
    if (reduce_last_block<2>(part, V.partials, V.counters, task.block, task.nblocks, tot) && threadIdx.x == 0) {
        V.out[0] = tot[0];
        V.out[1] = tot[1];
    }
}

__global__ __launch_bounds__(kBlock) void k_ir_update(const RefineView* __restrict__ views,
                                                      const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const RefineView& V = views[task.case_id];
    for (long long i = (long long)task.block * kBlock + threadIdx.x; i < V.n; i += (long long)task.nblocks * kBlock)
        V.x[i] += (double)V.d32[i];
}

// Launchers ---------------------------------------------------------------------------

// lanes: the lanes per node of the node-block SpMV (4, 8 or 16)
#define PFEM_DISPATCH_L(lanes, CALL)                      \
    switch (lanes) {                                       \
        case 4: { constexpr int LL = 4; CALL; } break;     \
        case 8: { constexpr int LL = 8; CALL; } break;     \
        default: { constexpr int LL = 16; CALL; } break;   \
    }

template <typename T>
void launch_kry_init(const KrylovView<T>* v, const BlockTask* t, int nt, const BlockTask* ids, int nids, int par,
                     bool stream, hipStream_t s) {
    if (stream) k_kry_init<T, true><<<nt, kBlock, 0, s>>>(v, t);
    else k_kry_init<T, false><<<nt, kBlock, 0, s>>>(v, t);
    k_kry_init_fin<T><<<nids < 1024 ? nids : 1024, kBlock, 0, s>>>(v, ids, nids, par);
}

// One kernel of an iteration (phase 0 U, 1 V, 2 S, 3 T) with parity par, so that a
// preconditioner's launches can sit between them; stream: non-temporal value loads; ev
// (optional) brackets V.
template <typename T, bool STREAM>
static void kry_phase(int phase, const KrylovView<T>* v, const BlockTask* t, int nt, int par, hipStream_t s,
                      hipEvent_t* ev) {
    switch (phase) {
        case 0: k_kry_update<T><<<nt, kBlock, 0, s>>>(v, t, par); break;
        case 1:
            // timed: the events ride on the dispatch itself (start and end of the kernel,
            // as a profiler sees them), not as separate packets around it
            if (ev) hipExtLaunchKernelGGL((k_kry_v<T, STREAM>), dim3(nt), dim3(kBlock), 0, s, ev[0], ev[1], 0, v, t, par);
            else k_kry_v<T, STREAM><<<nt, kBlock, 0, s>>>(v, t, par);
            break;
        case 2: k_kry_s<T><<<nt, kBlock, 0, s>>>(v, t, par); break;
        default: k_kry_t<T, STREAM><<<nt, kBlock, 0, s>>>(v, t, par); break;
    }
}

template <typename T>
void launch_kry_phase(int phase, const KrylovView<T>* v, const BlockTask* t, int nt, int par, bool stream,
                      hipStream_t s, hipEvent_t* ev) {
    if (stream) kry_phase<T, true>(phase, v, t, nt, par, s, ev);
    else kry_phase<T, false>(phase, v, t, nt, par, s, ev);
}

// y = A x over the sliced ELL copy (one wavefront per 64-node slice), the SpMV the BiCGSTAB
// kernels run; for checking the copy against the node-block values.
template <int NF>
__global__ __launch_bounds__(kBlock) void k_spmv_ell(const EllMatT<double> E, const double* __restrict__ x,
                                                     double* __restrict__ y) {
    const int lane = threadIdx.x & (kEllSlice - 1);
    for (long long c = (long long)blockIdx.x * kWaves + (threadIdx.x >> 6); c < E.nsl; c += (long long)gridDim.x * kWaves) {
        double r[NF];
        slice_part<NF, true>(E, c, 0, 1, [&](long long j, double (&xv)[NF]) { at_fields<NF>(x, E.N, j, xv); }, r);
        const long long i = c * kEllSlice + lane;
        if (i < E.N)
#pragma unroll
            for (int s = 0; s < NF; ++s) y[i + (long long)s * E.N] = r[s];
    }
}

void launch_spmv_ell(const EllMatT<double>& E, const double* x, double* y, int nblocks, hipStream_t s) {
    if (E.nf == 3) k_spmv_ell<3><<<nblocks, kBlock, 0, s>>>(E, x, y);
    else k_spmv_ell<4><<<nblocks, kBlock, 0, s>>>(E, x, y);
}

template <typename T>
void launch_spmv(int lanes, const NodeMat<T>& A, const T* x, T* y, int nblocks, hipStream_t s) {
    PFEM_DISPATCH_L(lanes, (k_spmv<T, LL><<<nblocks, kBlock, 0, s>>>(A, x, y)));
}

void launch_ir_residual(int lanes, const RefineView* v, const BlockTask* t, int nt, hipStream_t s) {
    PFEM_DISPATCH_L(lanes, (k_ir_residual<LL><<<nt, kBlock, 0, s>>>(v, t)));
}

void launch_ir_update(const RefineView* v, const BlockTask* t, int nt, hipStream_t s) {
    k_ir_update<<<nt, kBlock, 0, s>>>(v, t);
}

template void launch_kry_init<double>(const KrylovView<double>*, const BlockTask*, int, const BlockTask*, int, int,
                                      bool, hipStream_t);
template void launch_kry_init<float>(const KrylovView<float>*, const BlockTask*, int, const BlockTask*, int, int,
                                     bool, hipStream_t);
template void launch_kry_phase<double>(int, const KrylovView<double>*, const BlockTask*, int, int, bool, hipStream_t,
                                       hipEvent_t*);
template void launch_kry_phase<float>(int, const KrylovView<float>*, const BlockTask*, int, int, bool, hipStream_t,
                                      hipEvent_t*);
template void launch_spmv<double>(int, const NodeMat<double>&, const double*, double*, int, hipStream_t);
template void launch_spmv<float>(int, const NodeMat<float>&, const float*, float*, int, hipStream_t);

}  // namespace pfem
