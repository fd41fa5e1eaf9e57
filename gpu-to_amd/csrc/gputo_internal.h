// Internal declarations of libgputo: grid geometry, tiling of the node-gather
// kernels, device state of one multigrid level and of a solver handle.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/gputo.h"

namespace gputo {

// Largest halo / element box of one node-gather tile (LDS arrays are sized
// from these; the tile chooser keeps every tile inside them).
constexpr int kMaxHalo = 864;
constexpr int kMaxElemBox = 640;
constexpr int kBlock = 256;          // threads per block of the gather kernels
constexpr int kStageRows = 4;        // halo rows per wave loaded before any is stored
constexpr int kStNodes = kBlock / 8; // nodes per block of the stored-matrix operator
constexpr int kRedBlocks = 1024;     // blocks of the two-stage reductions
constexpr int kMaxLevels = 12;
constexpr int kMaxCoarseDofs = 20000;  // dense coarsest solve (mgcg9.cu:74, maxDofs0)
constexpr int kKeMaxClasses = 16;    // Ke0 entry classes passed by value to the level-0 kernels

// One structured hex grid: elements nx*ny*nz, nodes (nx+1)(ny+1)(nz+1);
// node id = nny*nnz*i + nny*k + j, element id = ny*nz*i + ny*k + j.
struct Grid {
    int nx, ny, nz;
    int nnx, nny, nnz;
    long nel, nnod, ndof;
};

Grid make_grid(int nx, int ny, int nz);

// Node tile of a gather kernel: TJ x TK x TI nodes per block.
struct Tile {
    int TJ, TK, TI;
    int ntj, ntk, nti;
    __host__ __device__ long blocks() const { return (long)ntj * ntk * nti; }
};

// XCD-aware block order.  Consecutive blocks are dealt round-robin over the
// 8 XCDs, each with its own L2; launching 8*ceil(n/8) blocks and giving XCD x
// the contiguous tile range [x*m, (x+1)*m), m = ceil(n/8), keeps
// neighbouring tiles, which share halo nodes, on one L2.
constexpr int kXcds = 8;
inline long xcd_launch(long ntiles) { return (ntiles + kXcds - 1) / kXcds * kXcds; }
__device__ __forceinline__ long xcd_tile(long b, long ntiles)
{
    const long m = (ntiles + kXcds - 1) / kXcds;
    return (b % kXcds) * m + b / kXcds;
}

// Work decomposition of the modal operator kernels (modal.hip): strips of W
// nodes along j, R = W + 1 list columns, blocks of NW waves owning M list
// entries and TI node layers.  NW = 0: the grid is past the kernel's 32-bit
// offsets.
constexpr int kMdMaxWaves = 8;
struct ModalWork {
    int flat = 0;  // one group of NW waves per element layer instead of a march
    int NW = 0, W = 0, R = 0, M = 0, TI = 0;
    int ns = 0, nch = 0, nib = 0;
    __host__ __device__ long blocks() const { return (long)ns * nch * nib; }
};
// el 0: one scale per element, 1: the level-1 element (children: 8 scales)
ModalWork modal_work(const Grid &g, int bytes, int el, int children);
bool modal_constants(const double *Ke0, double *C);      // C[8]; false: Ke0 has no isotropic modal form

Tile choose_tile(const Grid &g);   // level-0 node-gather bricks
Tile stored_tile(const Grid &g);   // stored-matrix operator (at most kStNodes nodes)

struct CgScalars;
// The residual test of a PCG iteration: the sums of r.r (n <= 256 of them) and
// the pinned progress word it is reported in.
struct CgTest {
    CgScalars *sc = nullptr;  // null: no test
    const double *rr = nullptr;
    int n = 0;
    double tol = 0.0;
    unsigned long long *prog = nullptr;
};

// Arguments of the operator kernels (T = double or float).  A kernel takes the
// smallest part that it reads: a small level's launch is short enough for the
// lines of its argument buffer to show (48 bytes more: 7.12 -> 7.26 us per FP32
// level-0 sweep at 96x48x48, 4.73 -> 4.86 per level-1 sweep).
template <class T>
struct OpStencil {  // k_stencil
    Grid g;
    const T *U;            // input vector
    const T *F;            // right-hand side (defect / Jacobi)
    T *out;                // result vector
    const T *S;            // assembled node stencils [14][3][3][stencil_ld] of the same operator, or null
    const T *AD;           // diagonal (Jacobi)
    const uint8_t *mask;   // per node: bit d set when DOF 3n+d is fixed
    const int *ctl;        // ctl[0] != 0: skip (converged)
    const T *Uc;           // OP_INTERP_JACOBI: the coarse level's correction
    T *out2;               // second result (prerelax+defect writes U and R)
    double omega, prerelax;
};
template <class T>
struct OpModal : OpStencil<T> {  // k_modal, k_modal_flat
    const T *RD;           // 1/AD for the modal kernels (null: no Jacobi or prerelaxed mode): one value per
                           // node where Ke0 has one diagonal value, per DOF for the level-1 operator
    double *partials;      // per-block partial sums (fused dot), may be null
    ModalWork mw;          // the level's tiling
    T mc[8];               // modal constants of Ke0
    double cx_floor;       // > 0: element scales below it count as 0 (mgcg9 smoother defect)
    const float *Uf;       // OP_MATVEC_UF: the input vector in FP32
};
template <class T>
struct OpArgsT : OpModal<T> {
    Tile t;
    const T *Ke;           // 24x24 row-major (level 0)
    const T *CX;           // element scale (level 0)
    const T *A;            // packed 300 x nel entry-major element matrices (levels >= 1)
    int nb;                // right-hand sides of a batched launch (0 or 1: one)
    int kc;                // Ke0 has the unit-H8 class structure: use kv
    T kv[kKeMaxClasses];   // value of each Ke0 entry class (kKeClass)
    int modal;             // Ke0 has the isotropic modal form: use mc and mw
    int per;               // modal kernels: periodic cell, the result complete on masters and images
};
using OpArgs = OpArgsT<double>;
template <class T>
struct OpTile : OpStencil<T> {  // k_gather, k_stored
    double *partials, cx_floor;
    const float *Uf;
    Tile t;
    const T *Ke, *CX, *A;
    T kv[kKeMaxClasses];
    explicit OpTile(const OpArgsT<T> &a)
        : OpStencil<T>(a), partials(a.partials), cx_floor(a.cx_floor), Uf(a.Uf), t(a.t), Ke(a.Ke), CX(a.CX), A(a.A)
    {
        for (int k = 0; k < kKeMaxClasses; ++k) kv[k] = a.kv[k];
    }
};

enum OpMode {
    OP_MATVEC = 0,      // out = K U, masked; partials = sum U.out
    OP_DEFECT = 1,      // out = F - K U, masked
    OP_JACOBI = 2,      // out = (1-w) U + w (r + AD U)/AD with r = F - K U masked; partials = sum F.out
    OP_PRE_JACOBI = 3,  // as OP_JACOBI with U = prerelax*F/AD formed on the fly
    OP_PRE_DEFECT = 4,  // U = prerelax*F/AD written to out2, out = F - K U masked
    OP_MATVEC_UF = 5,   // as OP_MATVEC with the input Uf in FP32 (level-0 node-gather, FP64)
    OP_INTERP_JACOBI = 6  // as OP_JACOBI with U + P Uc, 0 at fixed DOFs, in U's place (k_modal_flat, k_stencil)
};

// Scalars of one device-resident PCG (all on the device, one struct).
struct CgScalars {
    double rho, rho_p, alpha, beta, res0, relres, pq, rr;
    int done, nit, it, bad;
    // mixed precision: residual replacement state
    double rmax;     // largest recursive residual norm since the last replacement
    int noru;        // 0: replace the recursive residual by b - A x this iteration
    int nru;         // replacements done
};

constexpr int kMaxBatch = 6;  // the six load cases of a homogenisation

// The residual test, by one wave.  prog (pinned host memory) tells the host how
// far the iteration is: iterations tested << 1 | converged in the low half, the
// relative residual in FP32 in the high half; one 64-bit store, so the host never
// sees them apart.  The residual in FP64 is in the word kMaxBatch further on; the
// host takes it once its rounding is the one in prog (cg_wait).
constexpr int kCgBlocks = 256;  // blocks (= partial sums) of the PCG's reductions at most
__device__ __forceinline__ void cg_test(const CgTest &t)
{
    CgScalars *sc = t.sc;
    const double res0 = sc->res0;
    int done = sc->done;
    const int it = sc->it;
    double v[kCgBlocks / 64], rr = 0.0;
#pragma unroll
    for (int q = 0; q < kCgBlocks / 64; ++q) {
        const int i = 64 * q + (int)(threadIdx.x & 63);
        v[q] = i < t.n ? t.rr[i] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < kCgBlocks / 64; ++q) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off, 64);
        rr += v[q];
    }
    if (threadIdx.x) return;
    double rel = sc->relres;
    if (!done) {
        rel = sqrt(rr) / res0;
        sc->rr = rr;
        sc->relres = rel;
        if (!(rel < INFINITY)) {
            sc->bad = 1;
            done = 1;
        } else if (rel < t.tol) {
            done = 1;
        }
        if (done) {
            sc->done = 1;
            sc->nit = it;
        }
    }
    const unsigned long long w =
        ((unsigned long long)__builtin_bit_cast(unsigned, (float)rel) << 32) | ((unsigned)(it + 1) << 1) | (unsigned)done;
    __hip_atomic_store(t.prog + kMaxBatch, __builtin_bit_cast(unsigned long long, rel), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(t.prog, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Batched launches: several right-hand sides on one hierarchy, one per
// blockIdx.z.  The vectors of a batch follow each other with the level's DOF
// count (or the vector length n) as stride, each right-hand side has its own
// CgScalars, and a producer of per-block partial sums with G blocks writes
// right-hand side z's at partials + z G.  The convergence flag of right-hand
// side z is ctl[z * kCtlStride] (ctl points at CgScalars::done).  A launch
// with one right-hand side has blockIdx.z = 0 and is unchanged.
static_assert(sizeof(CgScalars) % sizeof(int) == 0, "CgScalars stride in ints");
constexpr int kCtlStride = (int)(sizeof(CgScalars) / sizeof(int));

template <class P>
__device__ __forceinline__ P *batch_ptr(P *p, long stride)
{
    return p ? p + (long)blockIdx.z * stride : p;
}
__device__ __forceinline__ const int *batch_ctl(const int *ctl) { return batch_ptr(ctl, kCtlStride); }
// DOFs of the level below a level of even element counts
__host__ __device__ inline long coarse_ndof(const Grid &g)
{
    return 3L * (g.nx / 2 + 1) * (g.ny / 2 + 1) * (g.nz / 2 + 1);
}
template <class T>
__device__ __forceinline__ void batch_shift(OpStencil<T> &a)
{
    const long st = a.g.ndof;
    a.U = batch_ptr(a.U, st);
    a.F = batch_ptr(a.F, st);
    a.Uc = batch_ptr(a.Uc, coarse_ndof(a.g));
    a.out = batch_ptr(a.out, st);
    a.out2 = batch_ptr(a.out2, st);
    a.ctl = batch_ctl(a.ctl);
}
template <class T>
__device__ __forceinline__ void batch_shift(OpModal<T> &a)
{
    batch_shift(static_cast<OpStencil<T> &>(a));
    a.partials = batch_ptr(a.partials, (long)gridDim.x);
}
template <class T>
__device__ __forceinline__ void batch_shift(OpTile<T> &a)
{
    batch_shift(static_cast<OpStencil<T> &>(a));
    a.partials = batch_ptr(a.partials, (long)gridDim.x);
}
// values of OpArgsT::RD on level l: per node, per DOF on level 1 (which may be
// the rediscretised one); it follows AD in one allocation
inline long rd_len(const Grid &g, int l) { return l == 1 ? g.ndof : g.nnod; }
inline unsigned batch_dim(int nb) { return nb > 1 ? (unsigned)nb : 1u; }

struct Level {
    Grid g;
    Tile t;
    ModalWork mw32, mw64;         // tilings of the modal operator (level 1 of REF_C: of its matrix-free operator)
    Tile tg;                      // node-gather tiling of this level (matrix-free levels)
    double *CXl = nullptr;        // element scales of a matrix-free coarse level (mgcg9)
    double *U = nullptr, *F = nullptr, *R = nullptr, *AD = nullptr, *T = nullptr;
    double *RD = nullptr;         // 1/AD of the levels the modal kernels apply (OpArgsT::RD)
    double *A = nullptr;          // packed element matrices (levels >= 1)
    double *S = nullptr;          // the level's operator as node stencils (stored levels below the coarsest)
    uint8_t *mask = nullptr;      // fixed-DOF node mask
    int *fixed_d = nullptr;       // fixed list (0-based DOF) on the device
    std::vector<int> fixed;       // fixed list (0-based DOF), reference order
};

// Order of the factored coarsest matrix (coarse_dof in coarse.hip): N entries;
// ps = 0: the DOFs in order (o2 = os = N), else two parts that end at o2 and os
// and the separator plane a.
struct CoarseMap {
    int n = 0, N = 0;
    int o2 = 0, os = 0, ps = 0, pad1 = 0, pad2 = 0;
    int p = 0, nplanes = 0, a = 0;  // DOFs of a plane, planes
    float rp = 0.0f;                // 1/p
};
// the matrices that are factored (each part followed by the separator, row
// stride = order), and the diagonal blocks of the whole factor
struct CoarseParts {
    int np;
    double *A[2], *L[2];  // L: where the factor is
    int n[2];
};
struct CoarseBlocks {
    int nblk, off[4];
    const double *L[3];
    long ld[3];
};

// Orders up to which the whole inverse is formed and applied: the product replaces
// a launch in every V-cycle (3.2-3.7 us), at the cost of N^3 operations in place of
// the transpose in every setup.  A mgcg1 call of 10 iterations: 1343 -> 1300 us at
// 525 DOFs, 1495 -> 1462 at 1008; the error against a solve in 80 bits is the same to
// two digits (up to 8e-14 at a condition of 1e15).  From there on the product
// grows faster (it is dense where the factor's inverse has its zero block).
constexpr int kCoarseFull = 1024;
struct Coarse {
    int n = 0;
    CoarseMap map;
    int *dof = nullptr;      // coarse_dof of every entry
    bool direct = true;      // factored (else smoothed: mgcg9 above 20000 DOFs)
    int bw = 0;              // lower bandwidth of the assembled matrix (node-major DOFs)
    double *AQ = nullptr;       // dense matrix (matrices of the parts, updated by the factorisation), then their factors
    double *Linv = nullptr;     // inverse of the factor used by the solves (lower, row-major)
    double *LinvT = nullptr;    // its transpose (row-major); of at most kCoarseFull entries: the whole inverse
    double *Lbuf[2] = {}, *LTbuf[2] = {};  // two inverse buffers (lagged factorisation)
    int cur = 0;                // buffer of Linv/LinvT
    int target = 0;             // buffer the factorisation in flight writes
    bool have = false;          // buffers[cur] hold a factor of an earlier setup
    bool invalid = false;       // set by a parameter or operator change: the next setup
                                // drops a lagged factor still in flight and factors exactly
    bool solve_waits = true;    // solves wait for the factorisation in flight
    double *y = nullptr;     // work vector
    int *flag = nullptr;     // SPD failure flag
    // the factorisation runs on a side stream, overlapped with the start of
    // the solve: ev_in orders it after the assembly, ev_done orders every
    // coarsest solve and the next assembly after it
    hipStream_t side = nullptr;
    hipEvent_t ev_in = nullptr, ev_done = nullptr;
    bool pending = false;  // factorisation launched, SPD flag not read yet
    mutable bool inv_pending = false;  // its inverse not enqueued yet (coarse_finish)
    mutable bool waited = false;       // the solve stream already waits for it (stream order holds after)
};

struct MixedState;
struct LearnState;

// Buffers of a batched PCG (several right-hand sides on one hierarchy):
// every vector holds nb vectors one after another, every level of the
// V-cycle has its own batched work vectors (U, F, R, Tmp; FP64 for an FP64
// solve, FP32 for the mixed one).
struct BatchState {
    int nb = 0;
    int precision = -1;
    double *R = nullptr, *P = nullptr, *Q = nullptr, *Z = nullptr;
    double *partials = nullptr;  // nb x (the most per-block partials of a launch)
    double *rr = nullptr;        // nb x (kCgBlocks residual sums), then nb x 2 kCgBlocks dots
    CgScalars *sc = nullptr, *sc_host = nullptr;
    double *v64[kMaxLevels][4] = {};
    float *v32[kMaxLevels][4] = {};
    float *r32 = nullptr, *z32 = nullptr;  // the FP32 V-cycle's right-hand side and result
};

struct HostStage;

}  // namespace gputo

struct gputo_handle {
    gputo_params prm{};
    int nl = 0;
    gputo::Level L[gputo::kMaxLevels];
    gputo::Coarse C;
    hipStream_t stream = nullptr;
    int device = 0;
    double *Ke = nullptr;         // fine element matrix (row-major, symmetric)
    int ke_classes = 0;           // Ke has the unit-H8 class structure (values in kv)
    double kv[gputo::kKeMaxClasses] = {};
    int ke_modal = 0;             // and the isotropic modal form (constants in mc)
    double mc[8] = {};
    double *Aelm = nullptr;       // level-1 Gauss-point matrices, packed [300][8]
    double *CX = nullptr;         // element scales of level 0
    double *Fv = nullptr, *Uv = nullptr, *R = nullptr, *P = nullptr, *Q = nullptr, *Z = nullptr;
    double *partials = nullptr;   // reduction partials
    gputo::CgScalars *sc = nullptr;
    gputo::CgScalars *sc_host = nullptr;  // pinned mirror
    double *rr = nullptr;         // the PCG's residual sums, then its dots (kCgBlocks + 2 kCgBlocks)
    unsigned long long *prog = nullptr;   // pinned progress words of the PCG (k_cg_check), one per right-hand side
    int *ctl_zero = nullptr;      // an always-zero control word
    long long bytes = 0;
    bool hier_ready = false;
    bool l1_built = false;        // level 1's element matrices are those of the current hierarchy
    bool per_masks = false;       // periodic cell: on every level an image is fixed where its master is
    bool masks_ready = false;     // level fixed lists and masks match L[0].fixed
    std::vector<void *> allocs;
    struct ToState *to = nullptr;
    struct ToState *to_kept = nullptr;  // an ended design loop's buffers, for the next one
    gputo::HostStage *stage = nullptr;  // pinned slots of the host copies (hostio.hip)
    gputo::MixedState *mx = nullptr;
    gputo::LearnState *ln = nullptr;  // learned level-2 correction (params.learned)
    // per-fine-element Galerkin tables of levels 1..gt_max (device, packed
    // [8^l][300]; null where the level is built from the level above)
    double *gt[gputo::kMaxLevels] = {};
    int gt_max = 0;
    int gt_preset = -1;          // preset the tables were built for (-1: none yet)
    std::vector<double> gt_ke;  // Ke they were built from (Galerkin level 1)
    double *hom = nullptr;      // periodic homogenisation: 6 load vectors and 6 fluctuations
    gputo::BatchState *bt = nullptr;  // batched PCG buffers (allocated on first use)
};

namespace gputo {

// ---- launch helpers (kernels.hip) ------------------------------------
template <class T> void launch_op0(hipStream_t s, int mode, const OpArgsT<T> &a, const CgTest *test = nullptr);
void launch_op0_uf(hipStream_t s, const OpArgs &a);  // OP_MATVEC_UF
// test: the PCG's residual test, run by a block of its own (the prerelaxed modes)
template <class T> void launch_op0_modal(hipStream_t s, int mode, const OpArgsT<T> &a, const CgTest *test = nullptr);
// whether launch_op0 takes the modal kernel for `mode`, and the blocks
// (= partial sums per right-hand side) of its launch
template <class T>
inline bool op0_is_modal(const OpArgsT<T> &a, int mode)
{
    return a.modal && a.mw.NW > 0 && (a.RD || mode == OP_MATVEC || mode == OP_MATVEC_UF || mode == OP_DEFECT);
}
template <class T>
inline int op0_blocks(const OpArgsT<T> &a, int mode)
{
    return (int)xcd_launch(op0_is_modal(a, mode) ? a.mw.blocks() : a.t.blocks());
}
template <class T> void launch_opA(hipStream_t s, int mode, const OpArgsT<T> &a);
// AD and, when RD is not null, 1/AD (launch_diag0: of the first DOF of each
// node; the diagonal entries of an isotropic Ke0 are equal)
void launch_diag0(hipStream_t s, const Grid &g, const double *Ke, const double *CX, double *AD, double *RD = nullptr);
void launch_diagA(hipStream_t s, const Grid &g, const double *A, double *AD, double *RD = nullptr);
void launch_recip(hipStream_t s, const double *AD, double *RD, long n, int stride);  // RD[i] = 1/AD[stride i]
// S = the operator of the packed element matrices A as node stencils
void launch_stencil_build(hipStream_t s, const Grid &g, const double *A, double *S);
constexpr int kStencilEntries = 126;  // the own and 13 forward 3 x 3 blocks per node (the rest by symmetry)
constexpr int kStencilNodes = 16;     // nodes of a workgroup; rows of S are whole workgroups long
__host__ __device__ inline long stencil_ld(long nnod) { return (nnod + kStencilNodes - 1) / kStencilNodes * kStencilNodes; }
template <class T>
void launch_restrict(hipStream_t s, const Grid &gc, const T *Rf, T *Fc, const uint8_t *maskc, const int *ctl,
                     int nb = 1);
template <class T>
void launch_interp(hipStream_t s, const Grid &gf, const T *Uc, T *Uf, const uint8_t *maskf, int zero_fixed,
                   const int *ctl, int nb = 1);
template <class T>  // Uout = Uin + P Uc (Uout may equal Uin)
void launch_interp_to(hipStream_t s, const Grid &gf, const T *Uc, const T *Uin, T *Uout, const uint8_t *maskf,
                      int zero_fixed, const int *ctl, int nb = 1);
template <class T> void launch_fill(hipStream_t s, T *v, long n, double val);
template <class Ta, class Tb>
void launch_dot_partial(hipStream_t s, const Ta *a, const Tb *b, long n, double *partials, const int *ctl,
                        int nb = 1);
template <class Ti, class To>
void launch_copy(hipStream_t s, const Ti *src, To *dst, long n, const int *ctl, int nb = 1);
template <class T>  // U = prerelax F / AD
void launch_prerelax(hipStream_t s, const T *F, const T *AD, T *U, long n, double prerelax, const int *ctl,
                     int nb = 1);
void launch_coarse_l1(hipStream_t s, const Grid &gc, const double *Aelm, const double *CXf, double *A);
// diagonal (and 1/AD) of the rediscretised level 1 from the child densities
void launch_diag_l1(hipStream_t s, const Grid &g, const double *Aelm, const double *CXf, double *AD, double *RD);
void launch_coarse_galerkin(hipStream_t s, const Grid &gc, const double *Af, double *Ac);
void launch_galerkin_table(hipStream_t s, const Grid &gc, int depth, const double *T, const double *CX0, double *A);
std::vector<std::vector<double>> galerkin_tables(const double *Ke, const double *base1, int maxdepth);
constexpr int kGtMaxDepth = 4;  // deepest level built from tables (8^4 x 300 doubles = 9.8 MB)
// A table product costs 300 FMA per level-0 element at every level, spread
// over nel_l/32 x 10 waves that each stream 8^l table rows.  Down to level 2
// (64 rows) it is the cheapest form at any size; deeper levels with fewer
// elements than this take the child-by-child Galerkin of the level above.
// Measured at 192x96x96: level 3 (3456 elements) 57 us from its table; level
// 4 (432 elements, 4096 rows) 24 us child by child.
constexpr long kGtMinElems = 2048;
inline bool from_table(int l, long nel) { return l <= kGtMaxDepth && (l <= 2 || nel >= kGtMinElems); }
void launch_corrcsa(hipStream_t s, const Grid &g, const int *fixed_d, int nfd, double *A, int mirrored);
// mgcg9 coarse levels: CX_c = 2 mean(children), element matrices CX Ke, and
// the zeroing of fixed rows/columns of the dense coarsest matrix
void launch_coarse_cx(hipStream_t s, const Grid &gc, const double *CXf, double *CXc);
void launch_ke_elements(hipStream_t s, const Grid &g, const double *CX, const double *Ke, double *A);
void launch_zero_rowcol(hipStream_t s, int N, const int *fixed_d, int nfd, double *AQ);
// mask: decouple the fixed DOFs (mgcg9), or null
void launch_assemble(hipStream_t s, const Grid &g, const double *A, const uint8_t *mask, const Coarse &C);
void coarse_layout(Coarse &C, const Grid &g, bool periodic);  // C.map from C.n, C.bw
std::vector<int> coarse_dofs(const Coarse &C);                // coarse_dof of every entry
CoarseParts coarse_parts(const Coarse &C);
long coarse_matrix_len(const Coarse &C);  // doubles of C.AQ
// Factor C.AQ on C.side after the work on s.  lag: when an earlier factor
// exists, write the new one into the other buffer and let the solves keep
// the earlier one (coarse_adopt switches at the next setup).
void coarse_factor(hipStream_t s, Coarse &C, bool lag);
// enqueues the inverse of a factorisation launched by coarse_factor and
// records ev_done; every wait on ev_done comes after it
void coarse_finish(const Coarse &C);
int coarse_check(Coarse &C);  // waits for an exact factorisation; GPUTO_ERR_NOT_SPD on a bad pivot
void coarse_adopt(Coarse &C);  // before a setup: take a finished lagged factor
// after a parameter or operator change: no factor of an earlier setup
// (current or still in flight) is used again
void coarse_invalidate(Coarse &C);
// mid-solve: make the solves on s wait for the factorisation in flight and
// use it from now on (no-op without a lagged factorisation)
void coarse_switch(Coarse &C, hipStream_t s);
template <class T>
void launch_coarse_solve(hipStream_t s, const Coarse &C, const T *b, T *x, const uint8_t *mask, const int *ctl,
                         int nb = 1);

// Steps of the PCG (cg.hip).  pq: npq per-block sums of p.q; rr, dots: room
// for kCgBlocks (2 kCgBlocks, flexible beta) sums per right-hand side, apart
// from pq.
constexpr int kCgFuse = 2048;   // most sums that every block of an update reads (2.4 % of a solve with 1100, 2 % with 1300)
// U = 0, R = F (R32, X0 as launch_cg_update_r) and the first residual norm
void launch_cg_start(hipStream_t s, const double *F, double *U, double *R, long n, CgScalars *sc, double *rr,
                     float *R32 = nullptr, const float *AD32 = nullptr, float *X0 = nullptr, double prerelax = 0.0);
// rho = r.z of the first direction
template <class TZ>
void launch_cg_rho(hipStream_t s, const double *r, const TZ *z, long n, CgScalars *sc, double *dots, int nb = 1);
// the first residual norm from the sums of launch_dot_partial
void launch_cg_init(hipStream_t s, CgScalars *sc, const double *partials, int nparts, int nb = 1);
// alpha, U += alpha P, R -= alpha Q, sums of R.R; R32 (if not null) gets R in FP32
void launch_cg_update_ur(hipStream_t s, double *U, double *R, const double *P, const double *Q, long n, CgScalars *sc,
                         const double *pq, int npq, double *rr, float *R32 = nullptr, int nb = 1);
// PCG with deferred u: the iterations' alphas are logged (0 once converged)
// and u += sum alpha_t p_t is applied every kCgLog iterations from the
// kept FP32 directions.
// X0 (optional): also writes X0 = prerelax R32 / AD32, the prerelaxed
// level-0 iterate of the next FP32 V-cycle (mixed_prerelax_target)
constexpr int kCgLog = 16;
void launch_cg_update_r(hipStream_t s, double *R, const double *Q, long n, CgScalars *sc, const double *pq, int npq,
                        double *rr, double *alog, float *R32, const float *AD32 = nullptr, float *X0 = nullptr,
                        double prerelax = 0.0);
void launch_cg_flush_u(hipStream_t s, double *U, const float *P, long n, const double *alog, int m);
// residual test from the sums of an update over n elements
CgTest cg_test_of(CgScalars *sc, const double *rr, long n, double tol, unsigned long long *prog);
void launch_cg_check(hipStream_t s, const CgTest &t, int nb = 1);
// dots of z and Pout = z + beta Pin (flex: Polak-Ribiere beta)
template <class TP, class TZ>
void launch_cg_direction(hipStream_t s, const double *r, const TZ *z, const double *q, TP *Pout, const TP *Pin, long n,
                         CgScalars *sc, double *dots, bool flex, int nb = 1, const double *zr = nullptr, int nzr = 0);

void check_hip(hipError_t e, const char *what);  // throws on an error
#define HIPCHK(x) ::gputo::check_hip((x), #x)
void set_ke(gputo_handle *h, const double *Ke0);  // upload Ke0 and detect its class structure

// Deterministic sum over a kBlock-thread block: fixed butterfly per wave,
// then the wave sums in order.  Every thread of the block must call it.
__device__ __forceinline__ double block_sum(double v)
{
    __shared__ double ws[kBlock / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) ws[w] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < kBlock / 64; ++i) s += ws[i];
    return s;
}


void to_release(gputo_handle *h);  // ends the design loop, its buffers stay with the handle (driver.hip)
void to_destroy(gputo_handle *h);
// ---- host arrays (hostio.hip) ------------------------------------------
// dev null: the host array is only checked.  check: FP64 values, all finite.
struct HostJob {
    void *dev;
    void *host;
    size_t bytes;
    bool check;
};
// In stream order on h->stream; the host arrays may be reused on return.
// False: a checked array holds a NaN or an infinity (what is on the device is
// then undefined).
bool host_upload(gputo_handle *h, const HostJob *jobs, int njobs);
void host_download(gputo_handle *h, const HostJob *jobs, int njobs);
void stage_destroy(gputo_handle *h);  // after the stream's work
void launch_flip_y(hipStream_t s, double *u, long nnod);

// ---- periodic unit cell (periodic.hip) --------------------------------
// A periodic vector lives on the full node grid; the nodes with i = nx,
// j = ny or k = nz are images of the master node (i mod nx, j mod ny,
// k mod nz).  Primal vectors (iterates) hold equal values on a master and
// its images; dual vectors (right-hand sides, residuals) are kept with the
// whole value on the master and zeros on the images, so that dot products
// over the full grid count every periodic DOF once.  The non-periodic
// operators applied to a primal vector give each master part of its row
// and the rest on its images: summing the images into the master (fold)
// completes the periodic operator.
// fold: master += images; images = bcast ? master : 0
template <class T> void launch_per_fold(hipStream_t s, const Grid &g, T *v, int bcast, const int *ctl, int nb = 1);
// images = master
template <class T> void launch_per_bcast(hipStream_t s, const Grid &g, T *v, const int *ctl, int nb = 1);
// pre: U = prerelax F/AD (0 on fixed DOFs); else U += omega fold(R)/AD;
// the new master value is written to the images too
template <class T>
void launch_per_jacobi(hipStream_t s, const Grid &g, T *U, const T *R, const T *F, const T *AD, const uint8_t *mask,
                       double omega, double prerelax, int pre, const int *ctl, int nb = 1);
// dense coarsest matrix of the periodic operator in the full numbering:
// master rows and columns hold the wrapped assembly, image rows are unit
void launch_assemble_per(hipStream_t s, const Grid &g, const double *A, double *AQ);

// unit-strain loads: fe[q] = Ke0 u0_q on the unit element, Q0[q][p] = u0_q.Ke0 u0_p
void homog_loads(const double *Ke0, double fe[6][24], double Q0[6][6]);
// the six load vectors (6 x ndof, master form) of the element scales CX
void launch_homog_rhs(hipStream_t s, const Grid &g, const double *CX, const double fe[6][24], const uint8_t *mask,
                      double *F);

int setup_hierarchy(gputo_handle *h, const std::vector<int> &fixed0);
// the stored element matrices of level 1 where the V-cycle applies it
// matrix-free (built on first use after a setup)
void ensure_level1(gputo_handle *h);
int run_pcg(gputo_handle *h, const double *F, double *U, double tol, int maxit, double *relres, int *nit);
// nb <= kMaxBatch right-hand sides together (F, U: nb vectors one after another)
int run_pcg_batch(gputo_handle *h, const double *F, double *U, int nb, double tol, int maxit, double *relres,
                  int *nit);

}  // namespace gputo
