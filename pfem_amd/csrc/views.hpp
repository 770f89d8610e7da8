// Plain-old-data views of one case's device arrays, passed to kernels through device
// arrays indexed by BlockTask::case_id.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace pfem {

// A device-memory pointer held in a view.  The views live in memory, so the compiler cannot see
// which address space a plain pointer loaded from one refers to and makes every access through
// it a flat one: that goes through the LDS unit as well, takes its whole 64-bit address in
// vector registers, and is waited for together with every other access in flight.  Held as a
// pointer into global memory, accesses through it are global ones.  Measured
// (same bits): steps of a 12k-node 3D column 16.65 -> 16.24 ms, of a 48k-node Delaunay mesh 66.4 ->
// 64.1 ms, of a 20k-node 2D column 27.95 -> 27.37 ms.
#if defined(__HIP_DEVICE_COMPILE__)
#define PFEM_GLOBAL __attribute__((address_space(1)))
#else
#define PFEM_GLOBAL
#endif
template <class T>
struct Gp {
    PFEM_GLOBAL T* p = nullptr;
    __host__ __device__ Gp() = default;
    __host__ __device__ Gp(T* q) : p((PFEM_GLOBAL T*)q) {}
    __host__ __device__ __forceinline__ T* get() const { return (T*)p; }
    __host__ __device__ __forceinline__ operator T*() const { return (T*)p; }
    __host__ __device__ __forceinline__ T* operator->() const { return (T*)p; }
};

// Surface-tension facets of a case (fst.hpp gathers them per node).
struct FstView {
    int F = 0;                  // facets (0: no surface tension)
    int all_nodes = 0;          // 1: a facet acts when every node is on the free surface (WC), 0: any node
    Gp<const int> nodes; // [F][dim] facet nodes (Facet::m_nodesIndexes order)
    Gp<const int> elem;  // [F] element of each facet
    Gp<const int> ptr;   // [N+1] node -> entries
    Gp<const unsigned> ent;  // f << 2 | a, a the node's local index in the facet's element
    Gp<const double> T;  // Boussinesq node temperatures (null: the factor is gamma)
    double gamma = 0, dgdT = 0, t_ref = 0;
};

// PSPG assembly + boundary conditions (MomContEquationPSPG.inl:7-235).
struct PspgView {
    int dim, N, E, mom_nnz;
    Gp<const int> conn;          // [ne][E]
    Gp<const double> pos;        // [dim][N]
    Gp<const double> q_prev;     // [(dim+1)N]  states at the start of the time step (be, free-node rhs)
    Gp<const double> q_iter;     // [(dim+1)N]  current Picard iterate (node states used by tau)
    Gp<const int4> node_info;    // [N] {mom_ptr, cont_ptr, deg, flags}
    Gp<const int> nbr_ptr;       // [N+1] node graph
    Gp<const int> nbr_idx;       // [graph_nnz]
    Gp<const int> pei_ptr;       // [graph_nnz+1] pair-element incidence
    Gp<const uint32_t> pei;      // [E*ne*ne]  e << 4 | a << 2 | b, sorted by e within each pair
    Gp<const double> dir_vals;   // [dim][N] Dirichlet velocities (read at Dirichlet nodes)
    Gp<double> vals;             // [nnz]
    Gp<double> b;                // [(dim+1)N]
    Gp<float> vals32;            // [nnz] FP32 copy for the mixed-precision inner solve (may be null)
    Gp<const int> diag_pos;      // [n]
    int ell_nsl, pad_ell;     // ELL copy of the values (EllMat): slices,
    Gp<const int> ell_soff;      // slice offsets,
    Gp<double> vals_ell;         // values written after assembly and BC (null: none)
    Gp<float> vals32_ell;        // FP32 ELL copy for an FP32 multigrid hierarchy (null: none)
    Gp<double> erec;             // [E][16] element records of the assembly (pspg.hip)
    Gp<double> esv;              // [E][4] sums of the previous-step velocities over each element
                              //        (and, with T, of the node temperatures in the 4th slot)
    Gp<double> binv;             // [(dim+1)^2][N] inverse diagonal node blocks (block Jacobi), SoA
    Gp<float> binv32;            // FP32 copy for the mixed-precision inner solve (may be null)
    long long nnz;
    double rho, mu, dt;
    double g[3];
    int problem, pad_problem;  // PFEM_PROBLEM_*
    double tau0, mreg;         // Bingham parameters
    // Boussinesq: node temperatures (null: none) scaling the body force of F by
    // 1 - alpha (T - Tr) at each Gauss point, and H by the same factor
    Gp<const double> T;
    double alpha, t_ref;
    FstView fst;  // surface tension (fst.F == 0: none)
};

// The assembled PSPG matrix seen through its node structure.  Values are the CSR values
// (pattern.hpp layout); the column structure is read from the node graph instead of the
// CSR column indices: the full rows (i, s) of node i all hold, for t = 0..nf-1, the
// columns nbr_k + t*N of i's deg neighbours at offset t*deg + k, and every other row
// holds only its diagonal.
template <typename T>
struct NodeMat {
    int N, nf, mom_nnz;
    int ncol;            // nodes of the column space when it differs from the rows' (0: N)
    Gp<const int4> info;    // [N] {mom_ptr, cont_ptr, deg, flags}
    Gp<const int> nbr_ptr;  // [N+1]
    Gp<const int> nbr_idx;  // [graph_nnz]
    Gp<const T> vals;       // [nnz]
};

// Node-major sliced ELL copy of a case's FP64 system (rebuilt from the values after every
// assembly) for the hot SpMV-type kernels: nodes in slices of 64, one wavefront lane per
// node, each slice padded to its largest node degree W_c.  A node's d+1 rows are computed
// by its own lane: no cross-lane sums, and every value load is 64 consecutive doubles.
// Rows holding only their diagonal keep it at (rank of the node itself, t = s) and zeros
// elsewhere, so every row is computed the same way.
constexpr int kEllSlice = 64;  // nodes per slice: one wavefront

template <typename VT>
struct EllMatT {
    int N, nf, nsl;       // row nodes, fields, slices
    int ncol;             // column nodes when they differ from the rows' (0: N)
    Gp<const int> soff;      // [nsl + 1] sum of the widths of the earlier slices
    Gp<const int> idx;       // [soff[nsl] * 64] column node of lane r at rank k: idx[(soff[c] + k) * 64 + r]
                          // (padding ranks: the node itself or node 0, with zero values)
    Gp<const VT> vals;       // [soff[nsl] * nf * nf * 64] value (s, t) of lane r at rank k:
                          // vals[((soff[c] + k) * nf * nf + s * nf + t) * 64 + r]; null: no copy
};
using EllMat = EllMatT<double>;

// Options of the products over such a matrix: a workgroup's four wavefronts share each slice (else
// one wavefront per slice); non-temporal value loads.
enum : int { ELL_SPLIT = 1, ELL_STREAM = 2 };

// Scalars of one BiCGSTAB solve.  The per-iteration scalars live in two slots used
// alternately (the host passes the slot parity of each iteration): a kernel only writes
// the current slot and only reads the previous one or fields written by earlier kernels,
// so no workgroup ever reads a value another workgroup of the same launch is writing.
struct KSlot {
    double rho, alpha, omega;
    int state, pad;  // K_*: what the iteration's first kernel found
};
// Slot states: an iteration follows; the slot of a (re)start; converged on ||s||; breakdown.
enum : int { K_RUN = 0, K_FRESH = 1, K_CONV = 2, K_BREAK = 3 };
struct KScal {
    KSlot slot[2];
    double rr;    // last ||r||^2
    double bb;    // ||b||^2
    double weak_rho;  // rho is lost at |rho| <= weak_rho ||r|| (set by init; negative: not tested)
    double tol2;  // absolute squared tolerance on ||r||^2
    double rtol;
    double atol2; // > 0: ||r||^2 must also fall below it (absolute cap), 0: relative only
    int done;     // 0 running, 1 converged, 2 breakdown or non-finite, 3 iteration limit, 4 rho lost
                  // in rounding (kWeakRho): the host restarts with a new shadow residual
    int iters;
    int maxit;
    int req_init;  // set by the host: the next init launch (re)starts this case
    int true_rr;   // 1 when rr is a true residual b - A x (set by init, cleared by each iteration)
    int weak;      // restarts on a lost rho so far (after kMaxWeak the solve goes on without the test)
};

// An FP64 solve's rho = (rh, r) is taken for lost at |rho| <= kWeakRho ||rh|| ||r||, the unit
// roundoff: beta and alpha are then rounding noise, and the solve wanders on a plateau for
// thousands of iterations (what ends it otherwise, rho = 0 exactly, only a dot product meets, whose
// rounding lies on a grid; the recurrence for rho never does).  Iterations per case without the
// test / at 1e-17 / 1e-16 / 1e-15, block Jacobi to a relative residual of 1e-10: 3D column fields of
// 72k nodes (two steps) 1,240 / 1,152 / 1,081 / 1,022, 250k (one) 1,549 / 1,062 / 1,011 / 882, 1.03M (one)
// 3,915 / - / 1,654 / 1,487; 8k nodes in 2D 1,981 / 1,973 / 1,873 / 1,680; a dam break of 1k nodes to
// 1e-12 838 / 838 / 838 / 849 (0.05, 0.25 and 0.5 restarts per step; one idles the rest of its launches:
// 18.5, 18.7 and 19.1 ms).  FP32 inner solves end at their own limits: with the test at 1e-11, their
// rounding, 72k nodes took 1,450 iterations instead of 1,366.
constexpr double kWeakRho = 1.1102230246251565e-16;
constexpr int kMaxWeak = 64;

// The per-workgroup partial sums: kPartStride arrays of kMaxCaseBlocks doubles per case.
enum : int { P_RR = 0, P_RV = 1, P_SS = 2, P_TS = 3, P_TT = 4, P_RHT = 5, P_RHS = 6, P_RHR = 2, P_BB = 3, kPartStride = 8 };

// BiCGSTAB workspace of one case; T is the inner arithmetic type (double or float).
// x and b are field-blocked (entry f N + i) as the assembly and the Picard loop hold them, the
// solver's own vectors node-blocked (entry i nf + f): a product gathers a neighbour's fields from
// one cache line.  Workgroups are assigned XCD-local node ranges.
template <typename T>
struct KrylovView {
    int n, x_zero;
    int nodes, nf;
    int nblk;       // workgroups of this case in the Krylov launches (partials producers)
    int amg;        // 1: ph and sh come from the multigrid V-cycle
    int split, pad_split;  // 1: the wavefronts of a workgroup share each slice of the products
    EllMatT<T> E;   // the system's values in type T
    Gp<const T> binv;  // [nf*nf][nodes] inverse of each node's diagonal (nf x nf) block, SoA
    Gp<const T> b;
    Gp<T> x;
    Gp<T> r;
    Gp<T> rh;
    Gp<T> p;   // multigrid: p; block Jacobi: rhat = B^-1 r
    Gp<T> v;
    Gp<T> s;   // multigrid: s; block Jacobi: vhat = B^-1 v
    Gp<T> t;
    Gp<T> ph;
    Gp<T> sh;  // multigrid only
    Gp<double> partials;    // [kPartStride][kMaxCaseBlocks]
    Gp<KScal> sc;
    // multigrid: U and S also write the V-cycle's level-0 pre-smoothing w = om B^-1 p (or s) from
    // the vector they hold, in the hierarchy's type
    Gp<double> mg_w0;
    Gp<float> mg_w0f;
    double mg_om;
};

// One level of a case's aggregation multigrid (amg.hpp) as seen by the setup and V-cycle
// kernels; T is the hierarchy's arithmetic type (FP64, or FP32 under FP64 BiCGSTAB: the
// preconditioner only shapes the search directions, the solve converges on the FP64 system).
constexpr int kAmgMaxDense = 88;  // coarsest-level unknowns inverted densely in LDS
// The level above the coarsest is handled with it, in one workgroup, up to these sizes: the four
// launches cost ~16 us, one workgroup 8 us on 60 nodes in 2D (4k values), 25 us on 250 (16k) and
// 26-37 us on 100-200 nodes in 3D (50-90k values).
constexpr int kAmgTailNodes = 128, kAmgTailValues = 6144;
constexpr int kRestrictLanes = 8;  // lanes per aggregate of the restriction
// Lanes per node in the PSPG assembly gathers (pair blocks, diagonal block and b).  Measured on
// the 262k-node 3D dam break / a 100k-node 2D column, off-diagonal + diagonal kernels: 16 lanes
// 767 + 370 / 41 + 44 us, 8 lanes 747 + 298 / 34 + 29 us, 4 lanes 888 + 298 / 49 + 27 us.
constexpr int kAsmLanes = 8;

template <typename T>
struct AmgView {
    NodeMat<T> A;          // this level's matrix (level 0: the system or its FP32 copy)
    EllMatT<T> E0;         // level 0: the system's ELL copy in type T (vals null: none)
    EllMatT<float> E0f;    // level 0 of an FP64 hierarchy: FP32 values read by the residual (vals null: none)
    Gp<const T> binv;         // block-Jacobi inverse, SoA [(nf*nf)][N]
    int level;
    int lanes;             // SpMV lanes per node on this level
    int split, pad2;       // 1: the wavefronts of a workgroup share each slice (level 0 and A P products)
    int mask;              // level 0: transfers and Galerkin sums use full rows only
    Gp<const uint8_t> flags;  // level 0: the nodes' flags (the masks read them; 1 byte per node)
    int nc;                // coarsest level: unknowns of the dense inverse
    double omega;          // block-Jacobi damping of the smoother
    double alpha;          // scaling of the coarse-grid correction (over-correction of the
                           // piecewise-constant prolongation)
    Gp<const int> done_flag;  // the case's BiCGSTAB done flag (finished solves skip the cycle)
    Gp<const double> r0[2];   // level 0 inputs (p, s of the FP64 BiCGSTAB)
    Gp<double> out0[2];       // level 0 outputs (ph, sh)
    Gp<T> r;                  // level >= 1 input
    Gp<T> w;                  // smoothed iterate
    Gp<T> t;                  // residual
    Gp<T> z;                  // level >= 1 output
    // transfer to the next coarser level
    int next_N;
    int pad0;
    Gp<const int> agg_ptr;    // members (nodes of this level) of each next-level aggregate
    Gp<const int> agg_nodes;
    Gp<const int> fine_agg;   // next-level aggregate of each node of this level (-1: none)
    Gp<T> next_r;
    Gp<const T> next_z;
    // A P in the sliced ELL layout: this level's rows, the next coarser level's columns; the
    // entry block (i, J) sums the blocks (i, j) of i's neighbours j in aggregate J (level 0:
    // over full rows (j, t) only; zero in rows (i, s) that hold only their diagonal)
    EllMatT<T> AP;
    int ap_lanes;          // lanes per node of the set-up kernel
    int pad1;
    Gp<const int> ap_ptr;     // [N + 1] AP entries of each node (ranks 0 .. degree-1 of its ELL row)
    Gp<const int> ap_gptr;    // [AP entries + 1] gather list of each AP entry
    Gp<const int> ap_gsrc;    // rank k in i's neighbour list of each gathered block
    Gp<T> ap_out;             // AP values (written at set-up, padding ranks included)
    EllMatT<float> APf;    // level 0 of an FP64 hierarchy: AP held in FP32 instead (vals null: none)
    Gp<float> ap_out32;       // its values (written at set-up in place of ap_out)
    // setup of this level (>= 1) from the finer level: entry block (I, J) is the sum of the
    // finer level's A P blocks (i, J) over the members i of aggregate I
    EllMatT<T> FAP;        // the finer level's A P
    EllMatT<float> FAPf;   // ... or its FP32 copy (level 1 of an FP64 hierarchy whose level 0
                           // holds A P in FP32; vals null: none)
    Gp<const int> gal_ptr;    // [entries + 1] gather list of each entry of this level
    Gp<const int2> gal_src;   // {finer node i, rank m of J in i's A P row}
    Gp<const int> self_rank;
    Gp<T> vals_out;
    Gp<T> binv_out;
    Gp<double> dense;  // coarsest: [nc * nc] inverse, row major over unknowns I nf + s (FP64 in
                    // either type: the coarse operators are the worst conditioned)
};

// Mixed-precision iterative refinement (FP64 outer residual, FP32 inner solve).
struct RefineView {
    int n, pad;
    NodeMat<double> A;   // FP64 system
    Gp<const double> b;
    Gp<double> x;           // FP64 solution
    Gp<double> r;           // FP64 residual
    Gp<float> r32;          // inner right-hand side
    Gp<const float> d32;    // inner correction
    Gp<double> partials;
    Gp<unsigned> counters;
    Gp<double> out;         // [4] {||r||^2, ||b||^2, ...}
};

// Tiles of the weakly compressible passes (2D, 3D): consecutive nodes per workgroup, lanes per
// node (a P1 node has ~6 incident triangles in 2D and ~24 tetrahedra in 3D), the nodes that one
// tile stages in LDS at most (64 bytes each in FP64, 3D momentum pass) and the visit words staged beside them:
// together with the static arrays within 64 KiB.  Tiles of a spatially ordered 3D mesh hold ~600
// nodes, of a random order up to ~1,000; elements with a node beyond the capacity are visited
// through memory (kWcFar), visit words past theirs are read from memory.
constexpr int kWcTile[2] = {128, 64};
constexpr int kWcTileLanes[2] = {2, 4};
constexpr int kWcSmallLanes[2] = {2, 16};  // of small cases (build_mesh_basic): kBlock / lanes nodes per tile
constexpr int kWcTileCap = 752;
constexpr int kWcVisits[2] = {1024, 1792};
constexpr uint32_t kWcFar = 0xffffffffu;

// Local index of the m-th other node (m = 1..D) of an element seen from its local node me,
// positively oriented with me first (3D: double transpositions, 2D: rotations).
template <int D>
__host__ __device__ constexpr int wc_other(int me, int m) {
    return D == 3 ? (me ^ m) : (me + m) % 3;
}

// Weakly compressible explicit step (WCompNewton/Solver.cpp:236-276).
template <typename S>
struct WcView {
    int dim, N, E, pad;
    Gp<const int> conn;          // [ne][E]
    Gp<const uint8_t> flags;     // [N] with NODE_FREE derived
    Gp<const int> elem_ptr;        // [N+1] node-element incidence (Pattern::elem_ptr / elem_list)
    Gp<const uint32_t> elem_list;
    int ntiles, lanes;
    Gp<const int> tile_own;      // [ntiles] LDS slot of the tile's first node
    Gp<const int> tile_nodes;    // [ntiles][kWcTileCap] staged nodes, ascending, then -1
    Gp<const uint32_t> visit;    // per incidence entry: LDS slots of the other nodes, 10 bits each, or kWcFar
    Gp<double> pos;              // [dim][N]
    Gp<S> v;                     // [dim][N]
    Gp<S> a;                     // [dim][N]
    Gp<S> p;                     // [N]
    Gp<S> rho;                   // [N]
    Gp<const double> dir_vals;   // [dim][N]
    Gp<S> vh;                    // [dim][N] half-step velocity
    Gp<S> p_old;                 // [N] pressure before the continuity pass
    Gp<double> m_mom;            // [N] lumped momentum mass (cases with surface-tension facets)
    Gp<double> f_mom;            // [dim][N] momentum force (same)
    Gp<double> hmin;             // [N] smallest he of each node's elements (CFL after the step)
    Gp<unsigned long long> dt2;  // CFL min accumulator (bits of a positive double)
    double mu, K0, K0p, rho_star;
    double g[3];
    double dt;   // time step of the current launch
    double sc2;  // securityCoeff^2 of the CFL reduction
    int meduri, pad1;
    FstView fst;  // surface tension (fst.F == 0: none)
};

// Picard loop helpers (MomContEquationPSPG.inl:293-372).
struct PicardView {
    int dim, N, n, res_kind;  // res_kind: 0 U, 1 U_P, 2 Ax_f
    double dt;
    Gp<const uint8_t> flags;
    Gp<double> pos;
    Gp<double> pos_save;
    Gp<double> q_prev;  // state at the start of the step (committed when the loop converges)
    Gp<double> x;       // Picard iterate q
    Gp<double> x_prev;  // previous iterate (U / U_P residuals)
    NodeMat<double> A;
    Gp<const double> b;
    Gp<double> partials;
    Gp<unsigned> counters;
    Gp<double> out;  // [4]
};

// Bookkeeping copies of the Picard step, one bit per copy (BlockTask::pad of the copy table).
enum : int {
    COPY_PREP = 1,     // pos_save = pos, x = q_prev, x_prev = q_prev   (prepare callback)
    COPY_SAVEIT = 2,   // x_prev = x                                   (next Picard iteration)
    COPY_COMMIT = 4,   // q_prev = x                                   (converged step)
    COPY_RESTORE = 8,  // pos = pos_save                               (Mesh::restoreNodesList)
    COPY_ZERO_X = 16,  // x = 0                                        (restart from zero)
    COPY_RESET_X = 32, // x = q_prev                                   (node states restored)
};

// Scalars of one case in an engine slot, read back by the host once per tick.
struct SlotScal {
    KScal k[2];              // FP64 solve, FP32 inner solve
    double out[4];           // residual sums (Picard residual, refinement residual)
    unsigned long long dt2;  // CFL minimum (bits of a positive double)
    double pad[3];
};

constexpr int kMaxCaseBlocks = 2048;

}  // namespace pfem
