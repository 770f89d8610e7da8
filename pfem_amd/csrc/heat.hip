// The heat equation of the reference (HeatEqIncompNewton without phase change,
// srcs/simulation/physics/IncompNewton/HeatEquation.inl), one conduction step on the GPU:
//
//   A = M + dt L on rows that are neither Dirichlet nor free (m_buildAb, :209-280), unit rows
//   otherwise; b = sum_e M_e theta_prev; then m_applyBC (:283-364): the facet terms
//   (prescribed flux q.n, convection h (T - Tinf), radiation sigma eps (T^4 - Tinf^4), each
//   integrated with the reference's 3-point facet rule) subtracted times dt in facet order,
//   free rows b = theta_prev, Dirichlet rows b = T_bc with the column elimination; and the
//   solve of the reference's Eigen::ConjugateGradient<Lower|Upper> (diagonal preconditioner,
//   initial guess theta_prev; HeatEquation.hpp:50, HeatEquation.inl:131).
//
// Layout: a scalar CSR over the case's node graph (a full row holds the sorted neighbours,
// the node itself included, so value k of row i is node-graph entry k of i; other rows hold
// their diagonal only).  The assembly gathers, like the PSPG one: each value sums the
// contributions M_e + dt L_e of the elements holding both nodes (pair-element incidence) from one
// element record per element (gradients and measure) written by an element pass: off-diagonal
// values in element order, diagonal values and the right-hand side in a fixed order, split over
// the node's lanes.
#include "common.hpp"
#include "heat.hpp"
#include "p1geom.hpp"

namespace pfem {

namespace {

constexpr int kHeatRec = 16;  // doubles per element record: dN_i/dx_k (d (d+1)), |e| at 15

template <int D>
__global__ __launch_bounds__(kBlock) void k_heat_elem(HeatView V) {
    const int e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= V.E) return;
    int nd[D + 1];
#pragma unroll
    for (int a = 0; a <= D; ++a) nd[a] = V.conn[(size_t)a * V.E + e];
    double x[D][D + 1];
    WGeom<D> G;
    wc_geometry<D>(V.pos, V.N, nd, x, G);
    double* rec = V.erec + (size_t)kHeatRec * e;
#pragma unroll
    for (int k = 0; k < D; ++k)
#pragma unroll
        for (int a = 0; a <= D; ++a) rec[k * (D + 1) + a] = G.gN[k][a];
    rec[15] = G.vol;
}

// L lanes per node: its row of A = M + dt L (or the unit row) and, for a full row, its share of
// b = sum_e M_e theta_prev.  The lanes take the row's off-diagonal entries (each the sum over its
// pair-element list, in element order) and share the diagonal's list, which holds every element of
// the node.  One thread per node walked ~100 element records in sequence (69k nodes, 3D: 249 ->
// 83 us).
template <int D, int L>
__global__ __launch_bounds__(kBlock) void k_heat_asm(HeatView V) {
    const int i = (blockIdx.x * kBlock + threadIdx.x) / L, lane = threadIdx.x % L;
    if (i >= V.N) return;
    const uint8_t f = V.flags[i];
    const int rp = V.row_ptr[i];
    if ((f & V.dbit) || (f & NODE_FREE)) {
        if (lane == 0) V.vals[rp] = 1.0;
        return;
    }
    const double mfac = V.rho * V.cv / ((D + 1) * (D + 2));
    const int nb = V.nbr_ptr[i], deg = V.nbr_ptr[i + 1] - nb;
    auto term = [&](unsigned pe, double& vol, int& a) {  // an element's share of one entry
        const int e = (int)(pe >> 4), bb = (int)(pe & 3u);
        a = (int)((pe >> 2) & 3u);
        const double* rec = V.erec + (size_t)kHeatRec * e;
        vol = rec[15];
        double gg = 0;
#pragma unroll
        for (int c = 0; c < D; ++c) gg += rec[c * (D + 1) + a] * rec[c * (D + 1) + bb];
        return mfac * vol * (a == bb ? 2.0 : 1.0) + V.dt * (V.k * vol * gg);
    };
    double vol;
    int a;
    for (int k = lane; k < deg; k += L) {
        const int g = nb + k;
        if (V.nbr_idx[g] == i) continue;
        double acc = 0.0;
        for (int q = V.pei_ptr[g]; q < V.pei_ptr[g + 1]; ++q) acc += term(V.pei[q], vol, a);
        V.vals[rp + k] = acc;
    }
    const int kd = V.diag_pos[i] - rp, gd = nb + kd;
    double acc = 0.0, bi = 0.0;
    for (int q = V.pei_ptr[gd] + lane; q < V.pei_ptr[gd + 1]; q += L) {
        const unsigned pe = V.pei[q];
        acc += term(pe, vol, a);
        double t = 0;
#pragma unroll
        for (int jj = 0; jj <= D; ++jj)
            t += mfac * vol * (jj == a ? 2.0 : 1.0) * V.Tprev[V.conn[(size_t)jj * V.E + (int)(pe >> 4)]];
        bi += t;
    }
    acc = group_sum<L>(acc);
    bi = group_sum<L>(bi);
    if (lane == 0) {
        V.vals[rp + kd] = acc;
        V.b[i] = bi;
    }
}

// one thread per facet: getQN (MatricesBuilder.inl:247-274) and the two getSGamma
// (:358-371) with the factors of HeatEquation.inl:87-99, T = N theta_prev at each point
template <int D>
__global__ __launch_bounds__(kBlock) void k_heat_facet(HeatView V) {
    const int f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= V.F) return;
    int fn[D];
#pragma unroll
    for (int i = 0; i < D; ++i) fn[i] = V.facets[(size_t)f * D + i];
    const int out = V.fout[f];
    auto P = [&](int node, int k) { return V.pos[(size_t)k * V.N + node]; };
    double det, nrm[3] = {0, 0, 0};
    double Nq[3][D], w[3];
    double refs;
    if constexpr (D == 2) {
        const double J00 = (P(fn[1], 0) - P(fn[0], 0)) / 2, J10 = (P(fn[1], 1) - P(fn[0], 1)) / 2;
        det = sqrt(J00 * J00 + J10 * J10);
        double nx = P(fn[1], 1) - P(fn[0], 1), ny = P(fn[0], 0) - P(fn[1], 0);
        if (nx * (P(out, 0) - P(fn[0], 0)) + ny * (P(out, 1) - P(fn[0], 1)) > 0) {
            nx = -nx;
            ny = -ny;
        }
        const double nn = sqrt(nx * nx + ny * ny);
        nrm[0] = nx / nn;
        nrm[1] = ny / nn;
        const double xi[3] = {-sqrt(3.0 / 5.0), 0.0, sqrt(3.0 / 5.0)};
        w[0] = 5.0 / 18.0;
        w[1] = 8.0 / 18.0;
        w[2] = 5.0 / 18.0;
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            Nq[g][0] = (1 - xi[g]) / 2;
            Nq[g][1] = (1 + xi[g]) / 2;
        }
        refs = 2.0;
    } else {
        double a[3], b[3], v[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            a[k] = P(fn[1], k) - P(fn[0], k);
            b[k] = P(fn[2], k) - P(fn[0], k);
            v[k] = P(out, k) - P(fn[0], k);
        }
        const double g0 = a[1] * b[2] - b[1] * a[2], g1 = a[2] * b[0] - b[2] * a[0], g2 = a[0] * b[1] - b[0] * a[1];
        det = sqrt(g0 * g0 + g1 * g1 + g2 * g2);
        double n[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
        if (v[0] * n[0] + v[1] * n[1] + v[2] * n[2] > 0)
            for (int k = 0; k < 3; ++k) n[k] *= -1.0;
        const double nn = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
        for (int k = 0; k < 3; ++k) nrm[k] = n[k] / nn;
        const double gp[3][2] = {{1.0 / 6.0, 1.0 / 6.0}, {1.0 / 6.0, 2.0 / 3.0}, {2.0 / 3.0, 1.0 / 6.0}};
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            Nq[g][0] = 1 - gp[g][0] - gp[g][1];
            Nq[g][1] = gp[g][0];
            Nq[g][2] = gp[g][1];
            w[g] = 1.0 / 3.0;
        }
        refs = 0.5;
    }
    double qn[D], sgh[D], sgr[D];
#pragma unroll
    for (int i = 0; i < D; ++i) qn[i] = sgh[i] = sgr[i] = 0;
    const double sigma = 5.670374419e-8;
    const double T4inf = V.Tinf * V.Tinf * V.Tinf * V.Tinf;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
        double qv = 0;
        if (V.qgp)
#pragma unroll
            for (int k = 0; k < D; ++k) qv += V.qgp[((size_t)f * 3 + g) * D + k] * nrm[k];
        const double fact = qv * w[g];
        double Tg = 0;
#pragma unroll
        for (int j = 0; j < D; ++j) Tg += Nq[g][j] * V.Tprev[fn[j]];
        const double fh = V.h * (Tg - V.Tinf);
        const double fr = sigma * V.epsRad * (Tg * Tg * Tg * Tg - T4inf);
#pragma unroll
        for (int i = 0; i < D; ++i) {
            qn[i] += fact * Nq[g][i];
            sgh[i] += fh * Nq[g][i] * w[g];
            sgr[i] += fr * Nq[g][i] * w[g];
        }
    }
    const double s = refs * det;
#pragma unroll
    for (int i = 0; i < D; ++i) {
        double* t = V.fterm + ((size_t)f * D + i) * 3;
        t[0] = qn[i] * s;
        t[1] = sgh[i] * s;
        t[2] = sgr[i] * s;
    }
}

// one thread per node: m_applyBC's effect on its row, in the reference's order (facet terms in
// facet order, then the eliminations of the Dirichlet columns in increasing node order), and
// the diagonal inverse for the preconditioner
__global__ __launch_bounds__(kBlock) void k_heat_bc(HeatView V) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= V.N) return;
    const uint8_t f = V.flags[i];
    const int rp = V.row_ptr[i];
    if (f & V.dbit) {
        V.b[i] = V.Tbc[i];
    } else if (f & NODE_FREE) {
        V.b[i] = V.Tprev[i];
    } else {
        double bi = V.b[i];
        for (int q = V.nf_ptr[i]; q < V.nf_ptr[i + 1]; ++q) {
            const int ent = V.nf_list[q];
            const int fc = ent / V.dim;
            const uint8_t kind = V.fkind[fc];
            const double* t = V.fterm + (size_t)ent * 3;
            if (kind & 1) bi -= V.dt * t[0];
            if (kind & 2) bi -= V.dt * t[1];
            if (kind & 4) bi -= V.dt * t[2];
        }
        const int nb = V.nbr_ptr[i], deg = V.nbr_ptr[i + 1] - nb;
        for (int k = 0; k < deg; ++k) {
            const int j = V.nbr_idx[nb + k];
            if (j != i && (V.flags[j] & V.dbit)) {
                bi -= V.vals[rp + k] * V.Tbc[j];
                V.vals[rp + k] = 0.0;
            }
        }
        V.b[i] = bi;
    }
    const double dg = V.vals[V.diag_pos[i]];
    V.dinv[i] = dg != 0.0 ? 1.0 / dg : 1.0;
}

// ---- conjugate gradient, diagonal preconditioner -------------------------------------------
// Reductions are fence-free: every workgroup writes its partial sums to its own slot, and the
// next kernel's workgroups re-reduce them in workgroup order.  rz partials alternate between
// two arrays by iteration parity, so no kernel reads a slot that it also writes.
// An iteration is two launches: Q finishes the previous one (beta, p = z + beta p_old) while it
// multiplies, gathering z and p_old and adding A z + beta A p_old (the directions alternate between
// two arrays, so no workgroup overwrites what another still gathers), X updates x, r and z.  Both
// issue their loads before they sum the partials.  A group of lanes takes a row: one thread per row
// read each value from another cache line.  69k nodes in 3D: three
// launches 22 -> 14 us per iteration; what is left is the rows' values and two launches' latency.

// Sums of two arrays of partials, in every thread.
struct CgSums {
    double v[2];
    __device__ __forceinline__ void load(const double* a, int na, const double* b, int nb) {
        v[0] = v[1] = 0.0;
        for (int q = threadIdx.x; q < na; q += kBlock) v[0] += a[q];
        for (int q = threadIdx.x; q < nb; q += kBlock) v[1] += b[q];
    }
    __device__ __forceinline__ void sum() {
        __shared__ double bc[2];
        block_sum<2>(v);
        if (threadIdx.x == 0) {
            bc[0] = v[0];
            bc[1] = v[1];
        }
        __syncthreads();
        v[0] = bc[0];
        v[1] = bc[1];
    }
};

__device__ double row_dot(const HeatView& V, int i, const double* x) {
    double s = 0;
    for (int q = V.row_ptr[i]; q < V.row_ptr[i + 1]; ++q) s += V.vals[q] * x[V.col[q]];
    return s;
}

// r = b - A x, z = D^-1 r; partials of r.z (parity 0), r.r and b.b
__global__ __launch_bounds__(kBlock) void k_cg_init(HeatView V) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double v[3] = {0, 0, 0};
    if (i < V.N) {
        const double r = V.b[i] - row_dot(V, i, V.x);
        const double z = V.dinv[i] * r;
        V.r[i] = r;
        V.z[i] = z;
        v[0] = r * z;
        v[1] = r * r;
        v[2] = V.b[i] * V.b[i];
    }
    block_sum<3>(v);
    if (threadIdx.x == 0) {
        V.part[blockIdx.x] = v[0];                    // rz, parity 0
        V.part[2 * V.nb + blockIdx.x] = v[1];         // rr
        V.part[3 * V.nb + blockIdx.x] = v[2];         // bb
    }
}

// Q: beta = rz_new / rz_old, p = z + beta p_old (first: p = z), q = A p; partials of p.q
template <int L>
__global__ __launch_bounds__(kBlock) void k_cg_q(HeatView V, int par, int first) {
    constexpr int NPB = kBlock / L;
    const double* __restrict__ z = V.z;
    const double* __restrict__ po = first ? V.z : V.p + (size_t)(1 - par) * V.N;
    double* pn = V.p + (size_t)par * V.N;
    const int lane = threadIdx.x % L;
    CgSums S;
    S.load(V.part + par * V.nb, V.nb, V.part + (1 - par) * V.nb, V.nb);
    double v[1] = {0}, beta = 0.0;
    for (int i0 = blockIdx.x * NPB; i0 < V.N; i0 += gridDim.x * NPB) {
        const int i = i0 + threadIdx.x / L, ic = min(i, V.N - 1);
        double sz = 0, sp = 0;
        for (int q = V.row_ptr[ic] + lane; q < V.row_ptr[ic + 1]; q += L) {
            const int j = V.col[q];
            const double a = V.vals[q];
            sz += a * z[j];
            sp += a * po[j];
        }
        sz = group_sum<L>(sz);
        sp = group_sum<L>(sp);
        const double zi = z[ic], pi = po[ic];
        if (i0 == (int)blockIdx.x * NPB && !first) {
            S.sum();
            beta = S.v[1] != 0.0 ? S.v[0] / S.v[1] : 0.0;
        }
        if (i < V.N && lane == 0) {
            const double p = zi + beta * pi, q = sz + beta * sp;
            pn[i] = p;
            V.q[i] = q;
            v[0] += p * q;
        }
    }
    block_sum<1>(v);
    if (threadIdx.x == 0) V.part[4 * V.nb + blockIdx.x] = v[0];
}

// X: alpha = rz / pq; x += alpha p; r -= alpha q; z = D^-1 r; partials of r.z (other parity), r.r
__global__ __launch_bounds__(kBlock) void k_cg_x(HeatView V, int par) {
    const int i = blockIdx.x * kBlock + threadIdx.x, ic = min(i, V.N - 1);
    CgSums S;
    S.load(V.part + par * V.nb, V.nb, V.part + 4 * V.nb, V.nq);
    const double x = V.x[ic], p = V.p[(size_t)par * V.N + ic], q = V.q[ic], r0 = V.r[ic], di = V.dinv[ic];
    S.sum();
    const double alpha = S.v[1] != 0.0 ? S.v[0] / S.v[1] : 0.0;
    double v[2] = {0, 0};
    if (i < V.N) {
        V.x[i] = x + alpha * p;
        const double r = r0 - alpha * q;
        const double z = di * r;
        V.r[i] = r;
        V.z[i] = z;
        v[0] = r * z;
        v[1] = r * r;
    }
    block_sum<2>(v);
    if (threadIdx.x == 0) {
        V.part[(1 - par) * V.nb + blockIdx.x] = v[0];
        V.part[2 * V.nb + blockIdx.x] = v[1];
    }
}

// r.r and b.b for the host
__global__ __launch_bounds__(kBlock) void k_cg_publish(HeatView V) {
    CgSums S;
    S.load(V.part + 2 * V.nb, V.nb, V.part + 3 * V.nb, V.nb);
    S.sum();
    if (threadIdx.x == 0) {
        V.scal[0] = S.v[0];
        V.scal[1] = S.v[1];
    }
}

}  // namespace

int heat_blocks(int n) { return (n + kBlock - 1) / kBlock; }

void launch_heat_assemble(const HeatView& V, hipStream_t s) {
    const int be = heat_blocks(V.E), bn = heat_blocks(V.N), bf = heat_blocks(V.F);
    if (V.dim == 2) {
        k_heat_elem<2><<<be, kBlock, 0, s>>>(V);
        k_heat_asm<2, 8><<<heat_blocks(V.N * 8), kBlock, 0, s>>>(V);
        if (V.F > 0) k_heat_facet<2><<<bf, kBlock, 0, s>>>(V);
    } else {
        k_heat_elem<3><<<be, kBlock, 0, s>>>(V);
        k_heat_asm<3, 16><<<heat_blocks(V.N * 16), kBlock, 0, s>>>(V);
        if (V.F > 0) k_heat_facet<3><<<bf, kBlock, 0, s>>>(V);
    }
    k_heat_bc<<<bn, kBlock, 0, s>>>(V);
}

void launch_cg_init(const HeatView& V, hipStream_t s) {
    k_cg_init<<<V.nb, kBlock, 0, s>>>(V);
    launch_cg_publish(V, s);
}

void launch_cg_iteration(const HeatView& V, int it, hipStream_t s) {
    if (V.dim == 2) k_cg_q<kCgLanes[0]><<<V.nq, kBlock, 0, s>>>(V, it & 1, it == 0);
    else k_cg_q<kCgLanes[1]><<<V.nq, kBlock, 0, s>>>(V, it & 1, it == 0);
    k_cg_x<<<V.nb, kBlock, 0, s>>>(V, it & 1);
}

void launch_cg_publish(const HeatView& V, hipStream_t s) { k_cg_publish<<<1, kBlock, 0, s>>>(V); }

}  // namespace pfem
