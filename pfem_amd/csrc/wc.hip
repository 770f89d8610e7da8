// K4: weakly compressible explicit CDS_dpdt step for a batch of cases
// (WCompNewton/Solver.cpp:236-276, ContEquation.inl:123-166,304-413, MomEquation.inl:201-374)
// and the CFL time step (WCompNewton/Solver.cpp:192-234).
//
// Node state (v, a, p, rho) is stored in S (double or float); positions, element
// arithmetic and the lumped-mass / force sums are FP64.  A step is three launches: the half
// step (node pass), continuity and momentum (tile passes that sum over the elements and
// finish their nodes).  There are no atomics on sums: device-scope FP64 atomics on gfx950 ran
// at ~36 G/s; every sum is gathered per node in a fixed order.
//
// Tile passes.  A workgroup owns kWcTile consecutive nodes (small 3D cases: 16).  The nodes of
// all their elements (the tile's nodes and a halo, listed once per mesh) are staged in LDS, and
// kWcTileLanes lanes per node (2 in 2D, 4 in 3D; small 3D cases 16) walk the node's incident
// elements, finding each element's other nodes through one 32-bit word of LDS slots
// (WcView::visit).  Reading the nodes from memory at every visit
// (d x 64 bytes, 24 visits per node in 3D) was bound by the rate at which the L1 looks up
// scattered cache lines: the 3D momentum gather took the same time per visit on a mesh that
// fits the L2 as on one 20 times larger, and halving its arithmetic gained 15 %.  A tile reads
// ~7 node states per node instead of 72, mostly in runs.  On the 2.06M-node 3D tank (12M tets,
// FP32 state) the six kernels of the record gathers (half 82, continuity element pass 280 and
// gather 255, node pass 56, momentum gather 767, node pass 78 us) became half 33, continuity 379-432
// and momentum 369-410 us (over GPUs); 100k nodes in FP64: 88 -> 60 us.  What bounds the tile passes
// now, by the counters on that tank: with FP32 state vector issue (207 and 194 instructions per visit,
// 63 % of the launch at a wave per 4 cycles and SIMD) and the LDS (half of it); with FP64 state the
// LDS, three quarters of the launch, over half of it bank conflicts between lanes that read different
// nodes; not HBM (1.46 GB per step in 0.87 ms).
//
// The P1 element quantities are the reference's Gauss-rule integrals in closed form:
//   lump2(M(1))_i           = |e| / (d+1)
//   (M(1) P)_i              = |e| (P_i + sum P) / ((d+1)(d+2))
//   (D(K0 + K0' N.P) V)_i   = |e| (K0/(d+1) + K0' (P_i + sum P)/((d+1)(d+2))) div_e(V)
//   lump(M(N.rho))_i        = |e| (rho_i + sum rho) / ((d+1)(d+2))
//   F(N.rho)_(i,s)          = lump(M(N.rho))_i g_s
//   (K V)_(i,s)             = mu |e| (B^T ddev B V)_(i,s),  ddev the deviatoric operator
//   (D^T P)_(i,s)           = |e|/(d+1) d_sN_i sum P
#include "common.hpp"
#include "fst.hpp"
#include "views.hpp"

namespace pfem {

template <int D>
constexpr double kRefSize = D == 2 ? 0.5 : 0.16666666666666666666666666666667;  // |e| / det J

// An element seen from one of its nodes: c[m-1] is det J times the gradient of the m-th other
// node's shape function (3D: the cross products of the edges, area vectors of the faces through
// the node; C, their sum, is minus the own node's, the area vector of the opposite face), so a
// visit needs one division in all (1 / det J) and no gradient selection by local index.
// The products' roundings are spelled out (fma): he of one element in one node's frame must have the
// same bits in the step and in the CFL pass, whatever the compiler merges around it.
template <int D>
struct Frame {
    double c[D][D], C[D], dj;
};

template <int D>
__device__ __forceinline__ void frame_of(const double (&e)[D][D], Frame<D>& F) {
    if constexpr (D == 2) {
        F.c[0][0] = e[1][1];
        F.c[0][1] = -e[1][0];
        F.c[1][0] = -e[0][1];
        F.c[1][1] = e[0][0];
    } else {
        auto cross = [](const double (&u)[D], const double (&v)[D], double (&w)[D]) {
            w[0] = fma(u[1], v[D - 1], -(u[D - 1] * v[1]));
            w[1] = fma(u[D - 1], v[0], -(u[0] * v[D - 1]));
            w[D - 1] = fma(u[0], v[1], -(u[1] * v[0]));
        };
        cross(e[1], e[D - 1], F.c[0]);
        cross(e[D - 1], e[0], F.c[1]);
        cross(e[0], e[1], F.c[D - 1]);
    }
    F.dj = 0;
#pragma unroll
    for (int k = 0; k < D; ++k) {
        F.dj = fma(e[0][k], F.c[0][k], F.dj);
        F.C[k] = F.c[0][k];
#pragma unroll
        for (int m = 1; m < D; ++m) F.C[k] += F.c[m][k];
    }
}

// he = 2 r_in of an element (Element::getRin, Element.cpp:226-294): 2D |e| / semi-perimeter,
// 3D 3 |e| / total face area; the edges' (2D) or faces' (3D) measures are the frame's lengths.
//
// The square roots take the hardware's reciprocal square root estimate through one coupled step of
// Goldschmidt's iteration and two residual corrections (within an ulp); the library's adds range
// scaling that areas and lengths of elements do not need.  2^-1000 keeps a zero finite.
__device__ __forceinline__ double sqrt_len(double v) {
    v = fmax(v, 9.332636185032189e-302);
    const double y = __builtin_amdgcn_rsq(v);
    double g = v * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, v), h, g);
    return fma(fma(-g, g, v), h, g);
}

template <int D>
__device__ __forceinline__ double elem_he(const Frame<D>& F) {
    double s = 0;
#pragma unroll
    for (int m = 0; m <= D; ++m) {
        double q = 0;
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const double v = m < D ? F.c[m < D ? m : 0][k] : F.C[k];
            q = fma(v, v, q);
        }
        s += sqrt_len(q);
    }
    return 2.0 * F.dj / s;  // 2D: 2 (dj/2) / (s/2); 3D: 2 (3 dj/6) / (s/2)
}

// One node's share of computeNextDT (WCompNewton/Solver.cpp:192-234) through an element of
// size he: sc^2 he^2 / max(u^2, c^2, 4 alpha^2 / he^2) with c^2 = (K0 + K0' p) / rho
// (ContEquation.inl:117-121), alpha = mu / rho (MomEquation.inl:184-198).  The reference's
// element value is the smallest of its nodes' shares (x / max(a, b) = min(x / a, x / b)), and a
// share only grows with he, so a node's smallest share over its elements is the one through its
// smallest he.  The step takes the minimum over nodes of that and the CFL pass the minimum over
// every element's nodes; both evaluate he in the frame of the share's node (an element's frames
// round it differently) and agree bit for bit, so that a run restarted from saved states and
// positions takes the time steps of an uninterrupted one.
__device__ __forceinline__ double cfl_share(double sc2, double he, double u2, double p, double rho, double K0,
                                            double K0p, double mu) {
    const double c2 = fma(K0p, p, K0) / rho;
    const double alpha = mu / rho;
    const double maxS = fmax(fmax(u2, c2), 4 * alpha * alpha / (he * he));
    return sc2 * he * he / maxS;
}

// v1/2 = v + dt/2 a (all nodes); x += dt v1/2 (non-fixed).  v1/2 and p go to arrays of their
// own: the tile passes replace p and v of their nodes while other tiles still read them.
template <typename S>
__global__ __launch_bounds__(kBlock) void k_wc_half(const WcView<S>* __restrict__ views,
                                                    const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const WcView<S>& V = views[task.case_id];
    const int N = V.N;
    const double dt = V.dt;
    // the CFL minimum of the step's last pass starts from the largest double
    if (task.block == 0 && threadIdx.x == 0) *V.dt2 = 0x7fefffffffffffffULL;
    const Seg sg = xcd_segment(task, N);
    for (int l = sg.lb * kBlock + threadIdx.x; l < sg.ns; l += sg.cnt * kBlock) {
        const int i = sg.n0 + l;
        const bool fixed = V.flags[i] & NODE_FIXED;
        V.p_old[i] = V.p[i];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k >= V.dim) continue;
            const long long q = (long long)k * N + i;
            const double vh = (double)V.v[q] + 0.5 * dt * (double)V.a[q];
            V.vh[q] = (S)vh;
            if (!fixed) V.pos[q] += vh * dt;
        }
    }
}

// The staged node states of one tile in LDS: per node d words of 8 bytes with its position, then
// d + 1 (MOM: d + 2) values of type S with its velocity, pressure (and density), each part with
// constant component offsets and a record length that spreads different records over the banks
// (3D: 24 bytes and 20 or 40 in the momentum pass); then the tile's visit words.
template <int D, typename S, bool MOM>
struct TileLds {
    static constexpr int kX = D, kU = D + 1 + (MOM ? 1 : 0);
    double* x;
    S* u;
    uint32_t* words;
    int cap;
    int q0;  // first incidence entry of the tile
    __host__ __device__ static constexpr size_t bytes(int cap) {  // multiples of 8
        return (8 * (size_t)kX * cap + sizeof(S) * (size_t)kU * cap + 7) / 8 * 8 + 4 * (size_t)kWcVisits[D - 2];
    }
    __device__ __forceinline__ TileLds(double* lds, int c) : cap(c) {
        x = lds;
        u = reinterpret_cast<S*>(lds + (size_t)kX * c);
        words = reinterpret_cast<uint32_t*>(lds + (8 * (size_t)kX * c + sizeof(S) * (size_t)kU * c + 7) / 8);
        q0 = 0;
    }
    // Every thread takes all its list entries, then all their states, so that staging costs a few
    // memory latencies in all and not a few per record.
    template <int T>
    __device__ __forceinline__ void stage(const WcView<S>& V, const S* __restrict__ pin, int tile) {
        constexpr int kVis = kWcVisits[D - 2];
        constexpr int R = (kWcTileCap + kBlock - 1) / kBlock, RV = kVis / kBlock;
        static_assert(kVis % kBlock == 0, "whole rounds of visit words");
        const int* __restrict__ list = V.tile_nodes + (long long)tile * kWcTileCap;
        const long long N = V.N;
        int j[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = (int)threadIdx.x + r * kBlock;
            j[r] = r * kBlock < cap && k < kWcTileCap ? list[k] : -1;
        }
        q0 = V.elem_ptr[tile * T];
        const int q1 = V.elem_ptr[min(V.N, tile * T + T)];
        double xs[R][D];
        S vs[R][D], ps[R], rs[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r * kBlock >= cap) continue;  // (uniform: no tile of the launch stages that many)
            const int n = max(j[r], 0);
#pragma unroll
            for (int d = 0; d < D; ++d) {
                xs[r][d] = V.pos[d * N + n];
                vs[r][d] = V.vh[d * N + n];
            }
            ps[r] = pin[n];
            rs[r] = MOM ? V.rho[n] : S(0);
        }
        uint32_t w[RV];
#pragma unroll
        for (int r = 0; r < RV; ++r) {
            if (r * kBlock >= q1 - q0) continue;  // (uniform)
            const int q = q0 + (int)threadIdx.x + r * kBlock;
            w[r] = V.visit[max(min(q, q1 - 1), 0)];  // past the tile: unused
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (j[r] < 0) continue;
            const int k = (int)threadIdx.x + r * kBlock;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                x[k * kX + d] = xs[r][d];
                u[k * kU + d] = vs[r][d];
            }
            u[k * kU + D] = ps[r];
            if (MOM) u[k * kU + D + 1] = rs[r];
        }
#pragma unroll
        for (int r = 0; r < RV; ++r) {
            if (r * kBlock >= q1 - q0) continue;
            words[(int)threadIdx.x + r * kBlock] = w[r];
        }
    }
    __device__ __forceinline__ void get(int k, double (&xa)[D], double (&va)[D], double& pa, double& ra) const {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            xa[d] = x[k * kX + d];
            va[d] = (double)u[k * kU + d];
        }
        pa = (double)u[k * kU + D];
        ra = MOM ? (double)u[k * kU + D + 1] : 0.0;
    }
};

// The element of incidence entry q in the frame of node i (x0, v0): edges, velocity
// differences, and the sums of p (and rho) over its nodes.
template <int D, typename S, bool MOM>
__device__ __forceinline__ void visit_elem(const WcView<S>& V, const TileLds<D, S, MOM>& T, const S* __restrict__ pin,
                                           int q, const double (&x0)[D], const double (&v0)[D], double (&ed)[D][D],
                                           double (&w)[D][D], double& psum, double& rsum) {
    // (the asm statements here and below keep the loads from memory in their branch: merged with
    // the LDS reads of the other one they all become flat loads)
    uint32_t word;
    if (q - T.q0 < kWcVisits[D - 2]) word = T.words[q - T.q0];
    else {
        word = V.visit[q];
        asm volatile("" : "+v"(word));
    }
    double xa[D][D], va[D][D], pa[D], ra[D];
    if (word != kWcFar) {
#pragma unroll
        for (int a = 0; a < D; ++a) T.get((int)((word >> (10 * a)) & 1023u), xa[a], va[a], pa[a], ra[a]);
    } else {  // a node beyond the tile's capacity: the element's nodes from memory
        const uint32_t en = V.elem_list[q];
        const long long e = en >> 2, N = V.N;
        const int me = (int)(en & 3u);
#pragma unroll
        for (int a = 0; a < D; ++a) {
            const int j = V.conn[(long long)wc_other<D>(me, a + 1) * V.E + e];
#pragma unroll
            for (int d = 0; d < D; ++d) {
                xa[a][d] = V.pos[d * N + j];
                va[a][d] = (double)V.vh[d * N + j];
            }
            pa[a] = (double)pin[j];
            ra[a] = MOM ? (double)V.rho[j] : 0.0;
        }
#pragma unroll
        for (int a = 0; a < D; ++a) {
#pragma unroll
            for (int d = 0; d < D; ++d) asm volatile("" : "+v"(xa[a][d]), "+v"(va[a][d]));
            asm volatile("" : "+v"(pa[a]), "+v"(ra[a]));
        }
    }
#pragma unroll
    for (int a = 0; a < D; ++a) {
        psum += pa[a];
        if (MOM) rsum += ra[a];
#pragma unroll
        for (int k = 0; k < D; ++k) {
            ed[a][k] = xa[a][k] - x0[k];
            w[a][k] = va[a][k] - v0[k];
        }
    }
}

// Continuity (m_buildSystemdpdt, ContEquation.inl:353-413, 139-147, 319-350): lumped mass
// lump2(M(1)), rhs F0 = -dt D(K0 + K0' N.P) V + M(1) P (Meduri) or lump2(M(1)) P and the
// smallest he of each node, then p = M^-1 F0 (free nodes: 0) and rho from the Tait-Murnaghan law.
template <int D, typename S, int L>
__device__ __forceinline__ void wc_cont_tiles(const WcView<S>& V, const BlockTask& task, int cap, double* lds,
                                              double (&red)[2][kWcTile[D - 2]]) {
    constexpr int T = kBlock / L;  // a lane group per tile node
    const int N = V.N;
    const double dt = V.dt;
    const int lane = threadIdx.x % L, r = threadIdx.x / L;
    TileLds<D, S, false> TL(lds, cap);
    const Seg sg = xcd_segment(task, V.ntiles);
    for (int l = sg.lb; l < sg.ns; l += sg.cnt) {
        const int tile = sg.n0 + l;
        const int own = V.tile_own[tile];
        const int j = tile * T + (int)threadIdx.x;  // the node this thread finishes
        const bool fin = threadIdx.x < T && j < N;
        const uint8_t fl = fin ? V.flags[j] : (uint8_t)0;
        const int i = tile * T + r;
        const int qb = i < N ? V.elem_ptr[i] : 0, qe = i < N ? V.elem_ptr[i + 1] : 0;
        TL.template stage<T>(V, V.p_old, tile);
        __syncthreads();
        double ml = 0.0, fc = 0.0, hmin = 1.7976931348623157e308;
        if (i < N) {
            double x0[D], v0[D], p0, r0;
            TL.get(own + r, x0, v0, p0, r0);
            for (int q = qb + lane; q < qe; q += L) {
                double ed[D][D], w[D][D], psum = p0, rsum = 0;
                visit_elem<D, S, false>(V, TL, V.p_old, q, x0, v0, ed, w, psum, rsum);
                Frame<D> F;
                frame_of<D>(ed, F);
                double dv = 0;  // det J div_e(V)
#pragma unroll
                for (int a = 0; a < D; ++a)
#pragma unroll
                    for (int k = 0; k < D; ++k) dv += F.c[a][k] * w[a][k];
                hmin = fmin(hmin, elem_he<D>(F));
                const double pp = (p0 + psum) * (1.0 / (D + 2));  // in units of refSize / (d + 1)
                ml += F.dj;
                fc += F.dj * (V.meduri ? pp : p0) - dt * (V.K0 + V.K0p * pp) * dv;
            }
            ml = group_sum<L>(ml) * (kRefSize<D> / (D + 1));
            fc = group_sum<L>(fc) * (kRefSize<D> / (D + 1));
            hmin = group_min<L>(hmin);
            if (lane == 0) {
                V.hmin[i] = hmin;
                red[0][r] = ml;
                red[1][r] = fc;
            }
        }
        __syncthreads();
        if (fin) {
            double p;
            if (fl & NODE_FREE) p = 0.0;
            else p = (1.0 / red[0][threadIdx.x]) * red[1][threadIdx.x];
            V.p[j] = (S)p;
            V.rho[j] = (S)(pow((V.K0p / V.K0) * p + 1.0, 1.0 / V.K0p) * V.rho_star);
        }
        __syncthreads();
    }
}

template <int D, typename S>
__global__ __launch_bounds__(kBlock, 4) void k_wc_cont(const WcView<S>* __restrict__ views,
                                                    const BlockTask* __restrict__ tasks, int cap) {
    extern __shared__ double lds[];
    __shared__ double red[2][kWcTile[D - 2]];
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const WcView<S>& V = views[task.case_id];
    if (kWcSmallLanes[D - 2] == kWcTileLanes[D - 2] || V.lanes == kWcTileLanes[D - 2])
        wc_cont_tiles<D, S, kWcTileLanes[D - 2]>(V, task, cap, lds, red);
    else wc_cont_tiles<D, S, kWcSmallLanes[D - 2]>(V, task, cap, lds, red);
}

// The end of a step at node i: a = M^-1 F with the BC of MomEquation.inl:341-373,
// v = v1/2 + dt/2 a (:216-222), and the node's share of the next step's CFL time step from the
// final v, p, rho and its smallest incident he (free nodes belong to no element: no share).
template <typename S>
__device__ __forceinline__ double wc_finish(const WcView<S>& V, int i, uint8_t f, double hmin, double mm,
                                            const double (&fm)[3]) {
    const int N = V.N;
    const double invm = 1.0 / mm;
    double u2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (k >= V.dim) continue;
        const long long q = (long long)k * N + i;
        double acc;
        if ((f & NODE_FREE) && !(f & NODE_BOUND)) acc = V.g[k];
        else if ((f & NODE_BOUND) && (f & NODE_DIRICHLET)) acc = V.dir_vals[q];
        else acc = invm * fm[k];
        V.a[q] = (S)acc;
        const S vs = (S)((double)V.vh[q] + 0.5 * V.dt * acc);
        V.v[q] = vs;
        u2 = fma((double)vs, (double)vs, u2);
    }
    if (f & NODE_FREE) return 1.7976931348623157e308;
    return cfl_share(V.sc2, hmin, u2, (double)V.p[i], (double)V.rho[i], V.K0, V.K0p, V.mu);
}

// Momentum (m_buildSystem, MomEquation.inl:229-302): lumped mass lump(M(N.rho)) and force
// F = -K V + D^T P + F(N.rho) of each node, summed over its elements.  In the frame of node i,
// with w_a = v_a - v_i, c_a and C of Frame, grad v = sum_a w_a c_a^T / dj and grad N_i = -C / dj:
//   (K V)_i = -mu refSize / dj [ sum_a (w_a (c_a.C) + c_a (w_a.C)) - 2/3 (sum_a w_a.c_a) C ].
// Cases with surface-tension facets leave the sums for k_wc_mom_node, which adds the facet terms.
template <int D, typename S, int L>
__device__ __forceinline__ void wc_mom_tiles(const WcView<S>& V, const BlockTask& task, int cap, double* lds,
                                              double (&red)[D + 1][kWcTile[D - 2]]) {
    constexpr int T = kBlock / L;  // a lane group per tile node
    const int N = V.N;
    const double c2 = 1.0 / (double)((D + 1) * (D + 2));
    const double muf = V.mu * (D + 1);  // in units of refSize / (d + 1)
    const int lane = threadIdx.x % L, r = threadIdx.x / L;
    double best = 1.7976931348623157e308;
    TileLds<D, S, true> TL(lds, cap);
    const Seg sg = xcd_segment(task, V.ntiles);
    for (int l = sg.lb; l < sg.ns; l += sg.cnt) {
        const int tile = sg.n0 + l;
        const int own = V.tile_own[tile];
        const int j = tile * T + (int)threadIdx.x;  // the node this thread finishes
        const bool fin = threadIdx.x < T && j < N;
        const uint8_t fl = fin ? V.flags[j] : (uint8_t)0;
        const double hmin = fin ? V.hmin[j] : 0.0;
        const int i = tile * T + r;
        const int qb = i < N ? V.elem_ptr[i] : 0, qe = i < N ? V.elem_ptr[i + 1] : 0;
        TL.template stage<T>(V, V.p, tile);
        __syncthreads();
        if (i < N) {
            double x0[D], v0[D], p0, r0, mm = 0.0, fm[D];
            TL.get(own + r, x0, v0, p0, r0);
#pragma unroll
            for (int s = 0; s < D; ++s) fm[s] = 0.0;
            for (int q = qb + lane; q < qe; q += L) {
                double ed[D][D], w[D][D], psum = p0, rsum = r0;
                visit_elem<D, S, true>(V, TL, V.p, q, x0, v0, ed, w, psum, rsum);
                Frame<D> F;
                frame_of<D>(ed, F);
                double h[D], tr = 0;
#pragma unroll
                for (int k = 0; k < D; ++k) h[k] = 0;
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    double cC = 0, wC = 0;
#pragma unroll
                    for (int k = 0; k < D; ++k) {
                        cC += F.c[a][k] * F.C[k];
                        wC += w[a][k] * F.C[k];
                        tr += w[a][k] * F.c[a][k];
                    }
#pragma unroll
                    for (int k = 0; k < D; ++k) h[k] += w[a][k] * cC + F.c[a][k] * wC;
                }
                const double visc = muf / F.dj, cc = psum + visc * ((2.0 / 3.0) * tr);
                mm += F.dj * (r0 + rsum);
#pragma unroll
                for (int s = 0; s < D; ++s) fm[s] += visc * h[s] - cc * F.C[s];
            }
            // the factors common to every visit, and F(N.rho) = mass x gravity
            mm = group_sum<L>(mm) * (kRefSize<D> * c2);
#pragma unroll
            for (int s = 0; s < D; ++s) fm[s] = group_sum<L>(fm[s]) * (kRefSize<D> / (D + 1)) + mm * V.g[s];
            if (lane == 0) {
                red[0][r] = mm;
#pragma unroll
                for (int s = 0; s < D; ++s) red[s + 1][r] = fm[s];
            }
        }
        __syncthreads();
        if (fin) {
            const double m = red[0][threadIdx.x];
            double f[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < D; ++s) f[s] = red[s + 1][threadIdx.x];
            if (V.fst.F > 0) {
                V.m_mom[j] = m;
#pragma unroll
                for (int s = 0; s < D; ++s) V.f_mom[(long long)s * N + j] = f[s];
            } else {
                best = fmin(best, wc_finish<S>(V, j, fl, hmin, m, f));
            }
        }
        __syncthreads();
    }
    if (V.fst.F == 0) block_min_to(V.dt2, best);
}

template <int D, typename S>
__global__ __launch_bounds__(kBlock, 4) void k_wc_mom(const WcView<S>* __restrict__ views,
                                                    const BlockTask* __restrict__ tasks, int cap) {
    extern __shared__ double lds[];
    __shared__ double red[D + 1][kWcTile[D - 2]];
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const WcView<S>& V = views[task.case_id];
    if (kWcSmallLanes[D - 2] == kWcTileLanes[D - 2] || V.lanes == kWcTileLanes[D - 2])
        wc_mom_tiles<D, S, kWcTileLanes[D - 2]>(V, task, cap, lds, red);
    else wc_mom_tiles<D, S, kWcSmallLanes[D - 2]>(V, task, cap, lds, red);
}

// The end of the step for cases with surface-tension facets: the force with the FST entries of
// the facets whose element holds i (WCompNewton/MomEquation.inl:312-335, added before the
// boundary conditions).
template <typename S>
__global__ __launch_bounds__(kBlock) void k_wc_mom_node(const WcView<S>* __restrict__ views,
                                                        const BlockTask* __restrict__ tasks) {
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const WcView<S>& V = views[task.case_id];
    const int N = V.N;
    double best = 1.7976931348623157e308;
    for (int i = task.block * kBlock + threadIdx.x; i < N; i += task.nblocks * kBlock) {
        double fm[3] = {0.0, 0.0, 0.0};
        for (int k = 0; k < V.dim; ++k) fm[k] = V.f_mom[(long long)k * N + i];
        if (V.fst.ptr[i] < V.fst.ptr[i + 1]) {
            auto flag_of = [&](int n) { return V.flags[n]; };
            if (V.dim == 2) {
                double bb[2] = {fm[0], fm[1]};
                fst_add<2>(V.fst, V.conn, V.E, V.pos, N, i, flag_of, bb);
                fm[0] = bb[0];
                fm[1] = bb[1];
            } else {
                double bb[3] = {fm[0], fm[1], fm[2]};
                fst_add<3>(V.fst, V.conn, V.E, V.pos, N, i, flag_of, bb);
                fm[0] = bb[0];
                fm[1] = bb[1];
                fm[2] = bb[2];
            }
        }
        best = fmin(best, wc_finish<S>(V, i, V.flags[i], V.hmin[i], V.m_mom[i], fm));
    }
    block_min_to(V.dt2, best);
}

// CFL on its own (no step before it): dt^2 = min_e sc^2 he^2 / max_n(u^2, c^2, 4 alpha^2/he^2),
// he = 2 r_in (Element.cpp:226-294), as the minimum of every element node's share, through he in
// that node's frame.
template <int D, typename S>
__global__ __launch_bounds__(kBlock) void k_wc_cfl(const WcView<S>* __restrict__ views,
                                                   const BlockTask* __restrict__ tasks) {
    constexpr int NE = D + 1;
    const BlockTask task = tasks[blockIdx.x];
    if (task.case_id < 0) return;
    const WcView<S>& V = views[task.case_id];
    const int N = V.N, E = V.E;
    const double sc2 = V.sc2;
    double best = 1.7976931348623157e308;
    for (long long e = (long long)task.block * kBlock + threadIdx.x; e < E; e += (long long)task.nblocks * kBlock) {
        int nd[NE];
#pragma unroll
        for (int a = 0; a < NE; ++a) nd[a] = V.conn[(long long)a * E + e];
        double x[NE][D];
#pragma unroll
        for (int a = 0; a < NE; ++a)
#pragma unroll
            for (int k = 0; k < D; ++k) x[a][k] = V.pos[(long long)k * N + nd[a]];
#pragma unroll
        for (int a = 0; a < NE; ++a) {
            double ed[D][D];
#pragma unroll
            for (int m = 1; m < NE; ++m)
#pragma unroll
                for (int k = 0; k < D; ++k) ed[m - 1][k] = x[wc_other<D>(a, m)][k] - x[a][k];
            Frame<D> F;
            frame_of<D>(ed, F);
            const int i = nd[a];
            double u2 = 0;
#pragma unroll
            for (int k = 0; k < D; ++k) {
                const double vk = (double)V.v[(long long)k * N + i];
                u2 = fma(vk, vk, u2);
            }
            best = fmin(best, cfl_share(sc2, elem_he<D>(F), u2, (double)V.p[i], (double)V.rho[i], V.K0, V.K0p, V.mu));
        }
    }
    block_min_to(V.dt2, best);
}

// Launchers ---------------------------------------------------------------------------
template <typename S>
void launch_wc_step(const WcView<S>* v, const BlockTask* node, int n_node, const BlockTask* const (&tiles)[2],
                    const int (&n_tiles)[2], const int (&cap)[2], const BlockTask* fst, int n_fst, hipStream_t s) {
    k_wc_half<S><<<n_node, kBlock, 0, s>>>(v, node);
    const size_t c2 = TileLds<2, S, false>::bytes(cap[0]), c3 = TileLds<3, S, false>::bytes(cap[1]);
    const size_t m2 = TileLds<2, S, true>::bytes(cap[0]), m3 = TileLds<3, S, true>::bytes(cap[1]);
    if (n_tiles[0]) k_wc_cont<2, S><<<n_tiles[0], kBlock, c2, s>>>(v, tiles[0], cap[0]);
    if (n_tiles[1]) k_wc_cont<3, S><<<n_tiles[1], kBlock, c3, s>>>(v, tiles[1], cap[1]);
    if (n_tiles[0]) k_wc_mom<2, S><<<n_tiles[0], kBlock, m2, s>>>(v, tiles[0], cap[0]);
    if (n_tiles[1]) k_wc_mom<3, S><<<n_tiles[1], kBlock, m3, s>>>(v, tiles[1], cap[1]);
    if (n_fst) k_wc_mom_node<S><<<n_fst, kBlock, 0, s>>>(v, fst);
}

template <typename S>
void launch_wc_cfl(const WcView<S>* v, const BlockTask* elem2, int n_elem2, const BlockTask* elem3, int n_elem3,
                   hipStream_t s) {
    if (n_elem2) k_wc_cfl<2, S><<<n_elem2, kBlock, 0, s>>>(v, elem2);
    if (n_elem3) k_wc_cfl<3, S><<<n_elem3, kBlock, 0, s>>>(v, elem3);
}

#define PFEM_WC_INSTANTIATE(S)                                                                                      \
    template void launch_wc_step<S>(const WcView<S>*, const BlockTask*, int, const BlockTask* const (&)[2],         \
                                    const int (&)[2], const int (&)[2], const BlockTask*, int, hipStream_t);        \
    template void launch_wc_cfl<S>(const WcView<S>*, const BlockTask*, int, const BlockTask*, int, hipStream_t);
PFEM_WC_INSTANTIATE(double)
PFEM_WC_INSTANTIATE(float)

}  // namespace pfem
