// Topology-optimisation driver on the device: the design loop of
// Cantilever/omp/top3D125mod.m:105-165 (density filter with symmetric
// padding, volume-preserving Heaviside projection, SIMP interpolation,
// MGCG solve, compliance sensitivities, OC bisection), with every
// element-sized array resident in HBM.  Reductions are two-stage with a
// fixed summation order.
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "gputo_internal.h"
#include "mixed.h"

using namespace gputo;

namespace {
struct OcState;
}

// The device buffers of a design loop.  The loop's state is new with each
// gputo_to_begin; its buffers stay with the handle from one loop to the next
// (their sizes are the mesh's) and are freed with it: freeing and allocating
// 270 MB took 4.5 ms per restart at 192x96x96.
struct ToBuffers {
    double *x = nullptr, *xPhys = nullptr, *xOld = nullptr, *Hs = nullptr, *dHs = nullptr, *dsK = nullptr;
    double *dc = nullptr, *dv = nullptr, *tmp = nullptr, *ocP = nullptr, *F = nullptr, *U = nullptr;
    double *w = nullptr;     // filter weights
    double *part = nullptr;  // reduction partials [32][kRedBlocks]
    OcState *oc = nullptr;  // the bisection's state
    double *red_host = nullptr;    // pinned: sums and the bisection's result (kSum...)
    std::vector<void *> allocs;
};

struct ToState : ToBuffers {
    gputo_to_config cfg;
    long nel = 0, ndof = 0;
    std::vector<int> fixed;
    std::vector<double> Ke;
    int fw = 0;              // filter half width
    int loop = 0;
    double penal = 3, beta = 2, eta = 0.4;
};

namespace {

constexpr int kMaxFilterWeights = 15 * 15 * 15;  // rmin <= 8: half width at most 7
constexpr int kCand = 31;  // OC candidates per pass: a depth-5 bisection tree
// words of red_host: eta sums; change and volume; compliance; the bisection's done and lmid
enum { kSumEta = 0, kSumPhys = 2, kSumComp = 4, kSumOc = 5, kSumCount = 8 };

template <class T>
T *talloc(ToBuffers *t, size_t n)
{
    void *p = nullptr;
    check_hip(hipMalloc(&p, (n ? n : 1) * sizeof(T)), "hipMalloc");
    t->allocs.push_back(p);
    return static_cast<T *>(p);
}

__device__ __forceinline__ int mirror_idx(int a, int n)
{
    // 'symmetric' padding of imfilter: -1 -> 0, -2 -> 1, n -> n-1
    while (a < 0 || a >= n) a = a < 0 ? -a - 1 : 2 * n - a - 1;
    return a;
}

__device__ __forceinline__ double wsum256(double v)
{
    __shared__ double ws[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    return ws[0] + ws[1] + ws[2] + ws[3];
}

// imfilter(in, h, 'symmetric') on the (nely, nelz, nelx) array = element
// order (top3D125mod.m:96,108,140-141), divided by `div` where given.  FW > 0:
// the half width, and the loads of a plane dx (FW = 1: of all three) are in
// flight together; with a loop over the neighbours each waited for its weight
// and its value: 38 us at 192x96x96 and FW = 1, 26 now (9.4 and 4.2 us at
// 48x24x24).  FW = 0: any half width fw.  Field 0 or 1 by blockIdx.y.
struct FilterField {
    const double *in, *div;
    double *out;
};

template <int FW>
__global__ __launch_bounds__(256) void k_filter(Grid g, FilterField f0, FilterField f1, const double *__restrict__ w,
                                               int fw)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= g.nel) return;
    const FilterField f = blockIdx.y ? f1 : f0;
    const double *__restrict__ in = f.in;
    const unsigned eu = (unsigned)e, q1 = eu / (unsigned)g.ny;  // far fewer than 2^32 elements
    const int j = (int)(eu - q1 * (unsigned)g.ny), k = (int)(q1 % (unsigned)g.nz), i = (int)(q1 / (unsigned)g.nz);
    double acc = 0.0;
    if constexpr (FW > 0) {
        constexpr int D = 2 * FW + 1, P = FW == 1 ? 3 : 1;  // planes loaded together
        int jj[D];
#pragma unroll
        for (int y = 0; y < D; ++y) jj[y] = mirror_idx(j + y - FW, g.ny);
        for (int x0 = 0; x0 < D; x0 += P) {
            double v[P][D][D];
#pragma unroll
            for (int x = 0; x < P; ++x) {
                const long pi = (long)g.ny * g.nz * mirror_idx(i + x0 + x - FW, g.nx);
#pragma unroll
                for (int z = 0; z < D; ++z) {
                    const long pk = pi + (long)g.ny * mirror_idx(k + z - FW, g.nz);
#pragma unroll
                    for (int y = 0; y < D; ++y) v[x][z][y] = in[pk + jj[y]];
                }
            }
#pragma unroll
            for (int x = 0; x < P; ++x)
#pragma unroll
                for (int z = 0; z < D; ++z)
#pragma unroll
                    for (int y = 0; y < D; ++y) {
                        const double wq = w[((x0 + x) * D + z) * D + y];
                        if (wq != 0.0) acc += wq * v[x][z][y];
                    }
        }
    } else {
        int q = 0;
        for (int dx = -fw; dx <= fw; ++dx) {
            const int ii = mirror_idx(i + dx, g.nx);
            for (int dz = -fw; dz <= fw; ++dz) {
                const int kk = mirror_idx(k + dz, g.nz);
                for (int dy = -fw; dy <= fw; ++dy, ++q) {
                    const double wq = w[q];
                    if (wq == 0.0) continue;
                    acc += wq * in[(long)g.ny * g.nz * ii + (long)g.ny * kk + mirror_idx(j + dy, g.ny)];
                }
            }
        }
    }
    f.out[e] = f.div ? acc / f.div[e] : acc;
}

// nf = 1 or 2 fields
void launch_filter(hipStream_t s, const Grid &g, int nf, const FilterField &f0, const FilterField &f1, const double *w,
                   int fw)
{
    const dim3 grid((unsigned)((g.nel + 255) / 256), (unsigned)nf);
    switch (fw) {
    case 1: k_filter<1><<<grid, 256, 0, s>>>(g, f0, f1, w, fw); break;
    case 2: k_filter<2><<<grid, 256, 0, s>>>(g, f0, f1, w, fw); break;
    case 3: k_filter<3><<<grid, 256, 0, s>>>(g, f0, f1, w, fw); break;
    default: k_filter<0><<<grid, 256, 0, s>>>(g, f0, f1, w, fw); break;
    }
}

__device__ __forceinline__ double prj_d(double v, double eta, double beta)
{
    return (tanh(beta * eta) + tanh(beta * (v - eta))) / (tanh(beta * eta) + tanh(beta * (1 - eta)));
}
__device__ __forceinline__ double deta_d(double v, double eta, double beta)
{
    const double se = 1.0 / cosh(beta * (v - eta));
    return -beta / sinh(beta) * se * se * sinh(v * beta) * sinh((1 - v) * beta);
}
__device__ __forceinline__ double dprj_d(double v, double eta, double beta)
{
    const double t = tanh(beta * (v - eta));
    return beta * (1 - t * t) / (tanh(beta * eta) + tanh(beta * (1 - eta)));
}

// partial sums of prj and deta for the eta Newton step (top3D125mod.m:110-116)
__global__ __launch_bounds__(256) void k_eta_sums(const double *__restrict__ xp, long n, double eta, double beta,
                                                 double *part)
{
    double s0 = 0.0, s1 = 0.0;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long)kRedBlocks * 256) {
        s0 += prj_d(xp[e], eta, beta);
        s1 += deta_d(xp[e], eta, beta);
    }
    s0 = wsum256(s0);
    s1 = wsum256(s1);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s0;
        part[kRedBlocks + blockIdx.x] = s1;
    }
}

// one block per sum: fixed-order reduction of kRedBlocks partials
__global__ __launch_bounds__(256) void k_finalise(const double *part, int nsums, double *out)
{
    const int q = blockIdx.x;
    double s = 0.0;
    for (int i = threadIdx.x; i < kRedBlocks; i += 256) s += part[(long)q * kRedBlocks + i];
    s = wsum256(s);
    if (threadIdx.x == 0) out[q] = s;
}

// projection, SIMP and change (top3D125mod.m:117-129): dHs = Hs/dprj,
// xPhys = prj, ch partials, xOld = xPhys, CX and dsK.
__global__ __launch_bounds__(256) void k_physics(double *__restrict__ xPhys, double *__restrict__ xOld,
                                                const double *__restrict__ Hs, double *__restrict__ dHs,
                                                double *__restrict__ CX, double *__restrict__ dsK, long n, int project,
                                                double eta, double beta, double penal, double Emin, double E0,
                                                double *part)
{
    double s = 0.0, vs = 0.0;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long)kRedBlocks * 256) {
        double xp = xPhys[e];
        if (project) {
            dHs[e] = Hs[e] / dprj_d(xp, eta, beta);
            xp = prj_d(xp, eta, beta);
            xPhys[e] = xp;
        } else {
            dHs[e] = Hs[e];
        }
        const double d = xp - xOld[e];
        s += d * d;
        vs += xp;
        xOld[e] = xp;
        CX[e] = Emin + pow(xp, penal) * (E0 - Emin);
        dsK[e] = -penal * (E0 - Emin) * pow(xp, penal - 1);
    }
    s = wsum256(s);
    vs = wsum256(vs);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s;
        part[kRedBlocks + blockIdx.x] = vs;
    }
}

// Compliance density ce_e = u_e^T Ke u_e in the C frame and C local order,
// scaled into dc = dsK ce / dHs, and dv = (1/(nel volfrac)) / dHs
// (top3D125mod.m:139-141 before filtering).  The quadratic form is the same
// in the MATLAB frame with cMat because Ke is invariant under the y-mirror.
__global__ __launch_bounds__(256) void k_sens(Grid g, const double *__restrict__ Ke, const double *__restrict__ U,
                                             const double *__restrict__ dsK, const double *__restrict__ dHs,
                                             double dv0, double *__restrict__ dc, double *__restrict__ dv,
                                             double *__restrict__ ce_out)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= g.nel) return;
    const int j = (int)(e % g.ny), k = (int)((e / g.ny) % g.nz), i = (int)(e / ((long)g.ny * g.nz));
    const int ie[8] = {0, 1, 1, 0, 0, 1, 1, 0}, je[8] = {0, 0, 1, 1, 0, 0, 1, 1}, ke[8] = {0, 0, 0, 0, 1, 1, 1, 1};
    double u[24];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        const long n = (long)g.nny * g.nnz * (i + ie[a]) + (long)g.nny * (k + ke[a]) + (j + je[a]);
        u[3 * a] = U[3 * n];
        u[3 * a + 1] = U[3 * n + 1];
        u[3 * a + 2] = U[3 * n + 2];
    }
    double ce = 0.0;
#pragma unroll
    for (int r = 0; r < 24; ++r) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < 24; ++c) t += Ke[24 * r + c] * u[c];
        ce += u[r] * t;
    }
    if (ce_out) {
        ce_out[e] = ce;
        return;
    }
    dc[e] = dsK[e] * ce / dHs[e];
    dv[e] = dv0 / dHs[e];
}

// OC: ocP = x sqrt(-dc/dv) (top3D125mod.m:145)
__global__ void k_ocp(const double *__restrict__ x, const double *__restrict__ dc, const double *__restrict__ dv,
                      double *__restrict__ ocP, long n, double *part)
{
    double s = 0.0;
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long)kRedBlocks * 256) {
        const double v = x[e] * sqrt(-dc[e] / dv[e]);
        ocP[e] = v;
        s += v;
    }
    s = wsum256(s);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__device__ __forceinline__ double oc_x(double ocp, double xt, double lmid, double move)
{
    // max(max(min(min(ocP/lmid, xU), 1), xL), 0) (top3D125mod.m:149)
    double v = ocp / lmid;
    v = fmin(v, xt + move);
    v = fmin(v, 1.0);
    v = fmax(v, xt - move);
    v = fmax(v, 0.0);
    return v;
}

// The OC bisection on the device (top3D125mod.m:143-151): a pass sums the
// volumes of kCand candidate multipliers at once (the midpoints of the next
// five bisection levels in heap order: node q has children 2q+1, "volume >
// volfrac", and 2q+2), reading x once, and walks the tree.  Three passes are
// enough as a rule, so nothing but the last state returns to the host: with
// the walk on the host each pass was a copy and a round trip of 25 us.
struct OcState {
    double l1, l2, lmid;
    double l[kCand];
    int done;
};

// l1, l2 -> the candidates, one thread each: the bits of q + 1 below its
// highest are the way from the root
__device__ __forceinline__ void oc_next(OcState *s)
{
    const int q = threadIdx.x;
    if (s->done || q >= kCand) return;
    double lo = s->l1, hi = s->l2;
    for (int b = 30 - __builtin_clz(q + 1); b >= 0; --b) {
        const double mid = 0.5 * (lo + hi);
        if ((q + 1) >> b & 1)
            hi = mid;  // volume <= volfrac: l2 = lmid
        else
            lo = mid;
    }
    s->l[q] = 0.5 * (lo + hi);
}

__device__ __forceinline__ bool oc_open(double l1, double l2) { return (l2 - l1) / (l2 + l1) > 1e-4; }

// the bracket from the sum of ocP
__global__ __launch_bounds__(256) void k_oc_begin(const double *part, double ne, double volfrac, OcState *st)
{
    double v = 0.0;
    for (int i = threadIdx.x; i < kRedBlocks; i += 256) v += part[i];
    v = wsum256(v);
    if (threadIdx.x == 0) {
        st->l1 = 0.0;
        st->l2 = v / ne / volfrac;
        st->lmid = 0.0;
        st->done = !oc_open(0.0, st->l2);
    }
    __syncthreads();
    oc_next(st);
}

// Partial volumes of eight candidates (blockIdx.y); a candidate is a division
// and five comparisons per element, 31 of them in one thread took 23 us at
// 48x24x24 and 49 at 192x96x96, 7.9 and 40 now.
constexpr int kCandGroup = 8;

__global__ __launch_bounds__(256) void k_oc_volumes(const double *__restrict__ ocP, const double *__restrict__ x, long n,
                                                   const OcState *__restrict__ st, double move, double *part)
{
    __shared__ double ws[4][kCandGroup];
    if (st->done) return;
    const int c0 = blockIdx.y * kCandGroup, tid = threadIdx.x;
    double s[kCandGroup];
#pragma unroll
    for (int q = 0; q < kCandGroup; ++q) s[q] = 0.0;
    if ((long)blockIdx.x * 256 < n) {
        double l[kCandGroup];
#pragma unroll
        for (int q = 0; q < kCandGroup; ++q) l[q] = st->l[min(c0 + q, kCand - 1)];
        for (long e = (long)blockIdx.x * 256 + tid; e < n; e += (long)kRedBlocks * 256) {
            const double o = ocP[e], xt = x[e];
#pragma unroll
            for (int q = 0; q < kCandGroup; ++q) s[q] += oc_x(o, xt, l[q], move);
        }
#pragma unroll
        for (int q = 0; q < kCandGroup; ++q)
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) s[q] += __shfl_xor(s[q], off, 64);
    }
    if ((tid & 63) == 0) {
#pragma unroll
        for (int q = 0; q < kCandGroup; ++q) ws[tid >> 6][q] = s[q];
    }
    __syncthreads();
    if (tid < kCandGroup && c0 + tid < kCand)
        part[(long)(c0 + tid) * kRedBlocks + blockIdx.x] = ws[0][tid] + ws[1][tid] + ws[2][tid] + ws[3][tid];
}

// One block: the sums of the pass (in k_finalise's order; 256 threads to a sum,
// eight sums to a thread, every load in flight together), the walk, the next
// candidates.
__global__ __launch_bounds__(1024) void k_oc_walk(const double *part, double ne, double volfrac, OcState *st)
{
    constexpr int kPer = (kCand + 3) / 4, kLoads = kRedBlocks / 256;
    __shared__ double ws[kPer][16], sum[4 * kPer];
    const int tid = threadIdx.x, t = tid & 255;
    double v[kPer][kLoads];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const int q = min(4 * r + (tid >> 8), kCand - 1);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) v[r][i] = part[(long)q * kRedBlocks + t + 256 * i];
    }
    if (st->done) return;
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        double x = 0.0;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) x += v[r][i];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if ((tid & 63) == 0) ws[r][tid >> 6] = x;
    }
    __syncthreads();
    if (tid < 4 * kPer) {
        const double *w = ws[tid >> 2] + 4 * (tid & 3);
        sum[tid] = w[0] + w[1] + w[2] + w[3];
    }
    __syncthreads();
    if (tid == 0) {
        double l1 = st->l1, l2 = st->l2, lmid;
        for (int q = 0;;) {
            lmid = st->l[q];
            const bool more = sum[q] / ne > volfrac;
            if (more)
                l1 = lmid;
            else
                l2 = lmid;
            q = more ? 2 * q + 1 : 2 * q + 2;
            if (!oc_open(l1, l2) || q >= kCand) break;
        }
        st->l1 = l1;
        st->l2 = l2;
        st->lmid = lmid;
        st->done = !oc_open(l1, l2);
    }
    __syncthreads();
    oc_next(st);
}

// x of the final multiplier, and the state for the host
__global__ void k_oc_apply(const double *__restrict__ ocP, double *__restrict__ x, long n, const OcState *st,
                           double move, double *host)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const bool done = st->done;
    if (e == 0) {
        host[0] = done ? 1.0 : 0.0;
        host[1] = st->lmid;
    }
    if (done && e < n) x[e] = oc_x(ocP[e], x[e], st->lmid, move);
}

__global__ void k_edofmat(Grid g, int *cmat)
{
    // cMat (top3D125mod.m:37-41): cVec = 3*nodeNrs+1 (1-based nodes) plus
    // 24 offsets, in MATLAB local order
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= g.nel) return;
    const int j = (int)(e % g.ny), k = (int)((e / g.ny) % g.nz), i = (int)(e / ((long)g.ny * g.nz));
    const long s1 = 3L * g.nny * g.nnz, s2 = 3L * g.nny * (g.nnz + 1), s3 = 3L * g.nny;
    const long off[24] = {0,      1,      2,      s1,     s1 + 1, s1 + 2, s1 - 3, s1 - 2,
                          s1 - 1, -3,     -2,     -1,     s3,     s3 + 1, s3 + 2, s2,
                          s2 + 1, s2 + 2, s2 - 3, s2 - 2, s2 - 1, s3 - 3, s3 - 2, s3 - 1};
    const long nodeNr = (long)g.nny * g.nnz * i + (long)g.nny * k + j + 1;
    const long cvec = 3 * nodeNr + 1;
#pragma unroll
    for (int q = 0; q < 24; ++q) cmat[24 * e + q] = (int)(cvec + off[q]);
}

unsigned nb256(long n) { return (unsigned)((n + 255) / 256); }

std::vector<double> filter_weights(double rmin, int *fw)
{
    // h = max(0, rmin - dist) on offsets -ceil(rmin)+1 .. ceil(rmin)-1
    // (top3D125mod.m:92-95), ordered [dx][dz][dy]
    const int w = (int)std::ceil(rmin) - 1;
    std::vector<double> h;
    for (int dx = -w; dx <= w; ++dx)
        for (int dz = -w; dz <= w; ++dz)
            for (int dy = -w; dy <= w; ++dy) {
                const double v = rmin - std::sqrt((double)(dx * dx + dy * dy + dz * dz));
                h.push_back(v > 0 ? v : 0.0);
            }
    *fw = w;
    return h;
}

// the partial sums to the pinned words from `slot` on, without a copy
void launch_finalise(ToState *t, hipStream_t s, int nsums, int slot)
{
    k_finalise<<<nsums, 256, 0, s>>>(t->part, nsums, t->red_host + slot);
}

void reduce_host(ToState *t, hipStream_t s, int nsums, int slot)
{
    launch_finalise(t, s, nsums, slot);
    check_hip(hipStreamSynchronize(s), "sync");
}

int map_exc()
{
    try {
        throw;
    } catch (const std::exception &e) {
        std::fprintf(stderr, "gputo: %s\n", e.what());
        return GPUTO_ERR_DEVICE;
    }
}

}  // namespace

static void free_buffers(ToState *t)
{
    if (!t) return;
    for (void *p : t->allocs) hipFree(p);
    if (t->red_host) hipHostFree(t->red_host);
    delete t;
}

void gputo::to_release(gputo_handle *h)
{
    if (!h->to) return;
    h->to_kept = h->to;
    h->to = nullptr;
}

void gputo::to_destroy(gputo_handle *h)
{
    free_buffers(h->to);
    free_buffers(h->to_kept);
    h->to = h->to_kept = nullptr;
}

// the buffers for a mesh of ne elements and ndof DOFs
static void make_buffers(ToState *t, size_t ne, size_t ndof)
{
    if (!t->x) {
        double **el[] = {&t->x, &t->xPhys, &t->xOld, &t->Hs, &t->dHs, &t->dsK, &t->dc, &t->dv, &t->tmp, &t->ocP};
        for (double **p : el) *p = talloc<double>(t, ne);
        t->F = talloc<double>(t, ndof);
        t->U = talloc<double>(t, ndof);
        t->part = talloc<double>(t, (size_t)kCand * kRedBlocks);
        t->oc = talloc<OcState>(t, 1);
        t->w = talloc<double>(t, kMaxFilterWeights);
        check_hip(hipHostMalloc((void **)&t->red_host, kSumCount * sizeof(double), hipHostMallocDefault), "hostmalloc");
    }
}

extern "C" {

int gputo_edofmat(gputo_handle *h, int *cmat)
{
    if (!h || !cmat) return GPUTO_ERR_ARGUMENT;
    try {
        const Grid &g = h->L[0].g;
        int *d = nullptr;
        check_hip(hipMalloc(&d, 24 * g.nel * sizeof(int)), "hipMalloc");
        k_edofmat<<<nb256(g.nel), 256, 0, h->stream>>>(g, d);
        hipError_t e1 = hipMemcpyAsync(cmat, d, 24 * g.nel * sizeof(int), hipMemcpyDeviceToHost, h->stream);
        hipError_t e2 = hipStreamSynchronize(h->stream);
        hipFree(d);
        check_hip(e1, "copy");
        check_hip(e2, "sync");
        return 0;
    } catch (...) {
        return map_exc();
    }
}

int gputo_filter_f64(gputo_handle *h, const double *in, double rmin, double *out)
{
    if (!h || !in || !out || !(rmin > 0) || rmin > 8) return GPUTO_ERR_ARGUMENT;
    try {
        const Grid &g = h->L[0].g;
        int fw;
        std::vector<double> w = filter_weights(rmin, &fw);
        double *dw, *din, *dout;
        check_hip(hipMalloc(&dw, w.size() * sizeof(double)), "hipMalloc");
        check_hip(hipMalloc(&din, g.nel * sizeof(double)), "hipMalloc");
        check_hip(hipMalloc(&dout, g.nel * sizeof(double)), "hipMalloc");
        hipStream_t s = h->stream;
        hipMemcpyAsync(dw, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice, s);
        hipMemcpyAsync(din, in, g.nel * sizeof(double), hipMemcpyHostToDevice, s);
        launch_filter(s, g, 1, {din, nullptr, dout}, {}, dw, fw);
        hipMemcpyAsync(out, dout, g.nel * sizeof(double), hipMemcpyDeviceToHost, s);
        hipError_t e = hipStreamSynchronize(s);
        hipFree(dw);
        hipFree(din);
        hipFree(dout);
        check_hip(e, "filter");
        return 0;
    } catch (...) {
        return map_exc();
    }
}

int gputo_sens_f64(gputo_handle *h, const double *Ke0, const double *U_cframe, double *ce)
{
    if (!h || !Ke0 || !U_cframe || !ce) return GPUTO_ERR_ARGUMENT;
    try {
        const Grid &g = h->L[0].g;
        hipStream_t s = h->stream;
        set_ke(h, Ke0);
        check_hip(hipMemcpyAsync(h->P, U_cframe, g.ndof * sizeof(double), hipMemcpyHostToDevice, s), "copy");
        k_sens<<<nb256(g.nel), 256, 0, s>>>(g, h->Ke, h->P, nullptr, nullptr, 0.0, nullptr, nullptr, h->Q);
        check_hip(hipMemcpyAsync(ce, h->Q, g.nel * sizeof(double), hipMemcpyDeviceToHost, s), "copy");
        check_hip(hipStreamSynchronize(s), "sync");
        return 0;
    } catch (...) {
        return map_exc();
    }
}

int gputo_to_begin(gputo_handle *h, const double *Ke0, const double *x0, const double *F, const double *fixed, int nfd,
                   const gputo_to_config *cfg)
{
    if (!h || !Ke0 || !x0 || !F || !cfg || nfd < 0 || (nfd && !fixed)) return GPUTO_ERR_ARGUMENT;
    if (!(cfg->rmin > 0) || cfg->rmin > 8 || (cfg->ft != 1 && cfg->ft != 3)) return GPUTO_ERR_ARGUMENT;
    to_release(h);
    // the fixed list is validated (finite, 1 <= v <= ndof) before any state
    // is published: a rejected call leaves no design loop on the handle
    std::vector<int> fx((size_t)nfd);
    {
        const double ndof = (double)h->L[0].g.ndof;
        for (int n = 0; n < nfd; ++n) {
            const double v = fixed[n];
            if (!(v >= 1.0 && v <= ndof)) return GPUTO_ERR_ARGUMENT;  // NaN fails too
            fx[n] = (int)v - 1;
        }
    }
    try {
        const Grid &g = h->L[0].g;
        ToState *t = new ToState();
        if (h->to_kept) {
            static_cast<ToBuffers &>(*t) = *h->to_kept;
            delete h->to_kept;
            h->to_kept = nullptr;
        }
        h->to = t;
        t->cfg = *cfg;
        t->nel = g.nel;
        t->ndof = g.ndof;
        t->penal = cfg->penal;
        t->beta = cfg->beta;
        t->eta = cfg->eta;
        t->Ke.assign(Ke0, Ke0 + 576);
        t->fixed = std::move(fx);
        const long ne = g.nel;
        make_buffers(t, ne, g.ndof);
        std::vector<double> w = filter_weights(cfg->rmin, &t->fw);
        hipStream_t s = h->stream;
        check_hip(hipMemcpyAsync(t->w, w.data(), w.size() * sizeof(double), hipMemcpyHostToDevice, s), "copy");
        const HostJob in[2] = {{t->x, (void *)x0, ne * sizeof(double), false},
                               {t->F, (void *)F, g.ndof * sizeof(double), false}};
        host_upload(h, in, 2);
        check_hip(hipMemcpyAsync(t->xPhys, t->x, ne * sizeof(double), hipMemcpyDeviceToDevice, s), "copy");
        launch_fill(s, t->xOld, ne, 1.0);  // xOld = 1 (top3D125mod.m:102)
        launch_fill(s, t->U, g.ndof, 0.0);
        launch_fill(s, t->tmp, ne, 1.0);
        launch_filter(s, g, 1, {t->tmp, nullptr, t->Hs}, {}, t->w, t->fw);  // Hs = imfilter(ones)
        check_hip(hipGetLastError(), "launch");
        check_hip(hipStreamSynchronize(s), "sync");
        t->loop = 0;
        return 0;
    } catch (...) {
        int rc = map_exc();
        to_destroy(h);
        return rc;
    }
}

int gputo_to_iterate(gputo_handle *h, gputo_to_stats *st)
{
    if (!h || !h->to || !st) return GPUTO_ERR_ARGUMENT;
    std::memset(st, 0, sizeof(*st));
    ToState *t = h->to;
    const gputo_to_config &c = t->cfg;
    const Grid &g = h->L[0].g;
    const long ne = g.nel;
    hipStream_t s = h->stream;
    try {
        const auto t0 = std::chrono::steady_clock::now();
        t->loop += 1;
        // RL 1: filtered field and projection (top3D125mod.m:108-121)
        launch_filter(s, g, 1, {t->x, t->Hs, t->xPhys}, {}, t->w, t->fw);
        const double *sums = t->red_host;
        if (c.ft == 3) {
            k_eta_sums<<<kRedBlocks, 256, 0, s>>>(t->xPhys, ne, t->eta, t->beta, t->part);
            reduce_host(t, s, 2, kSumEta);
            double f = sums[kSumEta] / ne - c.volfrac;
            int it = 0;
            while (std::fabs(f) > 1e-6 && it < 100) {
                t->eta = t->eta - f / (sums[kSumEta + 1] / ne);
                k_eta_sums<<<kRedBlocks, 256, 0, s>>>(t->xPhys, ne, t->eta, t->beta, t->part);
                reduce_host(t, s, 2, kSumEta);
                f = sums[kSumEta] / ne - c.volfrac;
                ++it;
            }
        }
        k_physics<<<kRedBlocks, 256, 0, s>>>(t->xPhys, t->xOld, t->Hs, t->dHs, h->CX, t->dsK, ne, c.ft == 3 ? 1 : 0,
                                             t->eta, t->beta, t->penal, c.Emin, c.E0, t->part);
        launch_finalise(t, s, 2, kSumPhys);
        // RL 2: solve (top3D125mod.m:130-134)
        hipEvent_t e0, e1;
        hipEventCreate(&e0);
        hipEventCreate(&e1);
        hipEventRecord(e0, s);
        double relres = 0.0;
        int nit = 0;
        set_ke(h, t->Ke.data());
        int rc = setup_hierarchy(h, t->fixed);
        if (rc == 0) {
            rc = run_pcg(h, t->F, t->U, c.cg_tol, c.cg_maxit, &relres, &nit);
        }
        hipEventRecord(e1, s);
        hipEventSynchronize(e1);
        float ms = 0.f;
        hipEventElapsedTime(&ms, e0, e1);
        hipEventDestroy(e0);
        hipEventDestroy(e1);
        st->seconds_solve = ms * 1e-3;
        st->change = std::sqrt(sums[kSumPhys]) / ne;  // written before the solve
        st->volume = sums[kSumPhys + 1] / ne;
        st->relres = relres;
        st->cg_iters = nit;
        if (rc) {
            st->status = rc;
            return rc;
        }
        // RL 3: sensitivities (top3D125mod.m:139-141)
        k_sens<<<nb256(ne), 256, 0, s>>>(g, h->Ke, t->U, t->dsK, t->dHs, 1.0 / ne / c.volfrac, t->tmp, t->ocP,
                                          nullptr);
        launch_filter(s, g, 2, {t->tmp, nullptr, t->dc}, {t->ocP, nullptr, t->dv}, t->w, t->fw);
        // RL 4: OC bisection (top3D125mod.m:143-151)
        k_ocp<<<kRedBlocks, 256, 0, s>>>(t->x, t->dc, t->dv, t->ocP, ne, t->part);
        k_oc_begin<<<1, 256, 0, s>>>(t->part, (double)ne, c.volfrac, t->oc);
        const dim3 vols(kRedBlocks, (kCand + kCandGroup - 1) / kCandGroup);
        auto oc_passes = [&](int np) {
            for (int p = 0; p < np; ++p) {
                k_oc_volumes<<<vols, 256, 0, s>>>(t->ocP, t->x, ne, t->oc, c.move, t->part);
                k_oc_walk<<<1, 1024, 0, s>>>(t->part, (double)ne, c.volfrac, t->oc);
            }
            k_oc_apply<<<nb256(ne), 256, 0, s>>>(t->ocP, t->x, ne, t->oc, c.move, t->red_host + kSumOc);
        };
        oc_passes(3);
        // RL 5: compliance F'U (top3D125mod.m:155)
        launch_dot_partial(s, t->F, t->U, g.ndof, t->part, nullptr);
        reduce_host(t, s, 1, kSumComp);
        check_hip(hipGetLastError(), "launch");
        while (sums[kSumOc] == 0.0) {  // the bracket is not narrow enough yet
            oc_passes(2);
            check_hip(hipGetLastError(), "launch");
            check_hip(hipStreamSynchronize(s), "sync");
        }
        const double lmid = sums[kSumOc + 1];
        // continuation (top3D125mod.m:32-33,152): cnt(v,{1,1,25,d},loop)
        const int L = t->loop;
        if (L >= 1 && t->penal < 1 && L % 25 == 0) t->penal += 0.25;
        if (L >= 1 && t->beta < 1 && L % 25 == 0) t->beta += 2;
        st->compliance = sums[kSumComp];
        st->eta = t->eta;
        st->lmid = lmid;
        st->status = 0;
        st->seconds_total = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        if (h->mx) mixed_stats(h, st);
        return 0;
    } catch (...) {
        st->status = map_exc();
        return st->status;
    }
}

int gputo_to_get(gputo_handle *h, double *x, double *xPhys, double *U)
{
    if (!h || !h->to) return GPUTO_ERR_ARGUMENT;
    try {
        ToState *t = h->to;
        HostJob out[3];
        int n = 0;
        if (x) out[n++] = {t->x, x, t->nel * sizeof(double), false};
        if (xPhys) out[n++] = {t->xPhys, xPhys, t->nel * sizeof(double), false};
        if (U) out[n++] = {t->U, U, t->ndof * sizeof(double), false};
        host_download(h, out, n);
        check_hip(hipStreamSynchronize(h->stream), "sync");
        return 0;
    } catch (...) {
        return map_exc();
    }
}

int gputo_to_end(gputo_handle *h)
{
    if (!h) return GPUTO_ERR_ARGUMENT;
    if (h->stream) hipStreamSynchronize(h->stream);
    to_release(h);
    return 0;
}

}  // extern "C"
