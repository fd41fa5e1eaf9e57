// Vector and scalar steps of the device-resident PCG (the scalar arithmetic
// of Cantilever/TOP3D125MGCGCUDA/mgcg1.cu:235-275, kept on the device so the
// loop never waits on the host).
//
// One iteration is
//   q = K p                      per-block sums of p.q (the operator kernel)
//   r -= alpha q (u += alpha p)  alpha = rho / p.q, per-block sums of r.r
//   check                        one block: residual test, progress word
//   z = M r                      V-cycle
//   dots                         per-block sums of r.z (and q.z); in FP64 the
//                                V-cycle's last sweep leaves them
//   p = z + beta p               beta from rho
// alpha and beta are formed inside the update that uses them: every block
// adds the per-block sums in the same order (at most kCgFuse of them, read
// while the block's first vector loads are in flight) and block 0 records the
// scalars.  That takes two one-block launches of 2.8-4.5 us out of an
// iteration.  No block reads a field that its own kernel writes: rho (read
// for alpha) is written with beta, rho_p (read for beta) with alpha.  The
// check is a block of the V-cycle's first level-0 launch where that is a modal
// kernel in a prerelaxed mode (as a launch: 2.7 us).  Its other blocks do not
// read the flag; what they write at convergence is not read any more.
//
// Sums are two-stage with fixed grids and fixed orders, so results do not
// depend on timing; products and sums are FP64 for both vector types.  The
// reductions run on at most kCgBlocks blocks of 1024 threads (one per CU, 16
// waves), small vectors on fewer: 256 sums are quick to read back in every
// block.
#include <algorithm>

#include "gputo_internal.h"

namespace gputo {

namespace {

constexpr int kCgThreads = 1024;
constexpr int kCgUpdBlocks = 2048;  // blocks of kBlock threads of the direction update

template <int NT>
__device__ __forceinline__ double cg_block_sum(double v)
{
    __shared__ double ws[NT / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s += ws[i];
    return s;
}

// sum of p[0..n), the same order in every block of NT threads
template <int NT>
__device__ __forceinline__ double cg_partials(const double *p, int n)
{
    constexpr int kChunk = 4;
    double s = 0.0;
    for (int i0 = threadIdx.x; i0 < n; i0 += kChunk * NT) {
        double v[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) v[k] = i0 + k * NT < n ? p[i0 + k * NT] : 0.0;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) s += v[k];
    }
    return cg_block_sum<NT>(s);
}

// U = 0, R = F, the FP32 copy of R and the prerelaxed level-0 iterate of the
// first FP32 V-cycle (optional, as k_cg_update_r), sums of F.F.
__global__ __launch_bounds__(kCgThreads) void k_cg_start(const double *__restrict__ F, double *__restrict__ U,
                                                        double *__restrict__ R, long n, double *rr,
                                                        float *__restrict__ R32, const float *__restrict__ AD32,
                                                        float *__restrict__ X0, float pr)
{
    double s = 0.0;
    for (long i = (long)blockIdx.x * kCgThreads + threadIdx.x; i < n; i += (long)gridDim.x * kCgThreads) {
        const double f = F[i];
        const float f32 = (float)f;
        float x = 0.0f;
        if (X0) x = pr * f32 / AD32[i];
        U[i] = 0.0;
        R[i] = f;
        if (R32) R32[i] = f32;
        if (X0) X0[i] = x;
        s += f * f;
    }
    s = cg_block_sum<kCgThreads>(s);
    if (threadIdx.x == 0) rr[blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_cg_init(CgScalars *sc, const double *p, int n)
{
    sc += blockIdx.z;
    p += (long)blockIdx.z * n;
    const double ff = cg_partials<kBlock>(p, n);
    if (threadIdx.x == 0) {
        sc->res0 = sqrt(ff);
        sc->done = 0;
        sc->nit = 0;
        sc->it = 0;
        sc->bad = 0;
        sc->relres = 0.0;
        if (!(sc->res0 < INFINITY)) {  // NaN or Inf in F
            sc->bad = 1;
            sc->done = 1;
        } else if (sc->res0 == 0.0) {  // F = 0: U = 0 is exact
            sc->done = 1;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_cg_rho0(CgScalars *sc, const double *p, int n)
{
    sc += blockIdx.z;
    p += (long)blockIdx.z * n;
    const double rz = cg_partials<kBlock>(p, n);
    if (sc->done) return;
    if (threadIdx.x == 0) {
        sc->rho = rz;
        sc->rho_p = rz;
    }
}

// block 0's record of alpha (one thread); alog: the iteration's slot of the
// alpha log, 0 once converged
__device__ __forceinline__ void cg_record_alpha(CgScalars *sc, double rho, double pq, double al, double *alog)
{
    sc->pq = pq;
    sc->alpha = al;
    sc->rho_p = rho;
    if (alog) *alog = al;
    if (!(fabs(al) < INFINITY)) {
        sc->bad = 1;
        sc->done = 1;
        sc->nit = sc->it;
    }
}

// more per-block sums than every block should read: alpha in its own launch
__global__ __launch_bounds__(kCgThreads) void k_cg_alpha(CgScalars *sc, const double *p, int n, double *alog)
{
    sc += blockIdx.z;
    p += (long)blockIdx.z * n;
    const double rho = sc->rho;
    const int done = sc->done;
    const double pq = cg_partials<kCgThreads>(p, n);
    if (threadIdx.x) return;
    if (done) {
        if (alog) *alog = 0.0;
        return;
    }
    cg_record_alpha(sc, rho, pq, rho / pq, alog);
}

// alpha of the update kernels: from the sums, or recorded by k_cg_alpha
// (npq = 0).  Returns false when there is nothing to update (converged, or
// alpha is not finite).  Every thread of the block calls it.
__device__ __forceinline__ bool cg_alpha(CgScalars *sc, const double *pq, int npq, double *alog, double &al)
{
    const int done = sc->done;
    if (npq == 0) {
        al = sc->alpha;
        return !done;
    }
    const double rho = sc->rho;
    const double s = cg_partials<kCgThreads>(pq, npq);
    al = rho / s;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (!done)
            cg_record_alpha(sc, rho, s, al, alog);
        else if (alog)
            *alog = 0.0;
    }
    return !done && fabs(al) < INFINITY;
}

// U += alpha P, R -= alpha Q, R32 = R in FP32 (optional), sums of R.R.  Two
// elements per pass, both loaded before either is stored (the memory counter
// retires in order: a load issued after a store waits for it).
__global__ __launch_bounds__(kCgThreads) void k_cg_update_ur(double *__restrict__ U, double *__restrict__ R,
                                                            const double *__restrict__ P,
                                                            const double *__restrict__ Q, long n, CgScalars *sc,
                                                            const double *pq, int npq, double *rr,
                                                            float *__restrict__ R32)
{
    sc += blockIdx.z;
    pq += (long)blockIdx.z * npq;
    U = batch_ptr(U, n);
    R = batch_ptr(R, n);
    P = batch_ptr(P, n);
    Q = batch_ptr(Q, n);
    R32 = batch_ptr(R32, n);
    const long stride = (long)gridDim.x * kCgThreads;
    double al;
    if (!cg_alpha(sc, pq, npq, nullptr, al)) return;
    double s = 0.0;
    for (long i = (long)blockIdx.x * kCgThreads + threadIdx.x; i < n; i += 2 * stride) {
        const bool two = i + stride < n;
        const long j = two ? i + stride : i;  // in bounds; unused when !two
        const double u0 = U[i], p0 = P[i], r0 = R[i], q0 = Q[i];
        const double u1 = U[j], p1 = P[j], r1 = R[j], q1 = Q[j];
        const double ra = r0 - al * q0, rb = r1 - al * q1;
        U[i] = u0 + al * p0;
        R[i] = ra;
        if (R32) R32[i] = (float)ra;  // the FP32 V-cycle's right-hand side
        s += ra * ra;
        if (two) {
            U[j] = u1 + al * p1;
            R[j] = rb;
            if (R32) R32[j] = (float)rb;
            s += rb * rb;
        }
    }
    s = cg_block_sum<kCgThreads>(s);
    if (threadIdx.x == 0) rr[(long)blockIdx.z * gridDim.x + blockIdx.x] = s;
}

// The residual update of the PCG with deferred u (u += alpha p is applied
// later from the logged alphas and directions).  PRE: also the FP32 V-cycle's
// prerelaxed level-0 iterate X0 = pr R32 / AD32, the expression of k_prerelax
// on the same FP32 values.
template <bool PRE>
__global__ __launch_bounds__(kCgThreads) void k_cg_update_r(double *__restrict__ R, const double *__restrict__ Q,
                                                           long n, CgScalars *sc, const double *pq, int npq,
                                                           double *rr, double *alog, float *__restrict__ R32,
                                                           const float *__restrict__ AD32, float *__restrict__ X0,
                                                           float pr)
{
    const long stride = (long)gridDim.x * kCgThreads;
    double al;
    if (!cg_alpha(sc, pq, npq, alog, al)) return;
    double s = 0.0;
    for (long i = (long)blockIdx.x * kCgThreads + threadIdx.x; i < n; i += 2 * stride) {
        const bool two = i + stride < n;
        const long j = two ? i + stride : i;  // in bounds; unused when !two
        const double r0 = R[i], q0 = Q[i], r1 = R[j], q1 = Q[j];
        float d0 = 0.0f, d1 = 0.0f;
        if (PRE) {
            d0 = AD32[i];
            d1 = AD32[j];
        }
        const double ra = r0 - al * q0, rb = r1 - al * q1;
        const float fa = (float)ra, fb = (float)rb;
        R[i] = ra;
        R32[i] = fa;
        if (PRE) X0[i] = pr * fa / d0;
        s += ra * ra;
        if (two) {
            R[j] = rb;
            R32[j] = fb;
            if (PRE) X0[j] = pr * fb / d1;
            s += rb * rb;
        }
    }
    s = cg_block_sum<kCgThreads>(s);
    if (threadIdx.x == 0) rr[blockIdx.x] = s;
}

// the residual test of a launch of its own (batches, level-0 kernels without it)
__global__ __launch_bounds__(64) void k_cg_check(CgTest t)
{
    t.sc += blockIdx.z;
    t.rr += (long)blockIdx.z * t.n;
    t.prog += blockIdx.z;
    cg_test(t);
}

// sums of r.z at dots[0..blocks) and, FLEX, of q.z after them
template <class TZ, bool FLEX>
__global__ __launch_bounds__(kCgThreads) void k_cg_dots(const double *__restrict__ r, const TZ *__restrict__ z,
                                                       const double *__restrict__ q, long n, double *dots,
                                                       const int *ctl)
{
    ctl = batch_ctl(ctl);
    if (ctl && ctl[0]) return;
    r = batch_ptr(r, n);
    z = batch_ptr(z, n);
    q = batch_ptr(q, n);
    dots = batch_ptr(dots, (FLEX ? 2L : 1L) * gridDim.x);
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (long i = (long)blockIdx.x * kCgThreads + threadIdx.x; i < n; i += (long)gridDim.x * kCgThreads) {
        const double zi = (double)z[i];  // exact for an FP32 z
        a += r[i] * zi;
        if (FLEX) b += q[i] * zi;
    }
    a = cg_block_sum<kCgThreads>(a);
    if (threadIdx.x == 0) dots[blockIdx.x] = a;
    if (FLEX) {
        b = cg_block_sum<kCgThreads>(b);
        if (threadIdx.x == 0) dots[gridDim.x + blockIdx.x] = b;
    }
}

// sum of p[0..n) to out, for one value per right-hand side
__global__ __launch_bounds__(kCgThreads) void k_cg_sum(const double *p, int n, double *out, const int *ctl)
{
    ctl = batch_ctl(ctl);
    if (ctl[0]) return;
    const double s = cg_partials<kCgThreads>(p + (long)blockIdx.z * n, n);
    if (threadIdx.x == 0) out[blockIdx.z] = s;
}

// Pout = Z + beta Pin formed in FP64 and rounded once (Pout may be Pin).
// beta = <r,z>/rho_old, or for a preconditioner that varies between
// iterations the flexible (Polak-Ribiere) <z, r - r_old>/rho_old with r -
// r_old = -alpha q, i.e. -alpha <z,q>/rho_old.
template <class TP, class TZ, bool FLEX>
__global__ __launch_bounds__(kBlock) void k_cg_update_p(TP *Pout, const TP *Pin, const TZ *__restrict__ Z, long n,
                                                       CgScalars *sc, const double *dots, int nd)
{
    sc += blockIdx.z;
    Pout = batch_ptr(Pout, n);
    Pin = batch_ptr(Pin, n);
    Z = batch_ptr(Z, n);
    dots = batch_ptr(dots, (FLEX ? 2L : 1L) * nd);
    const int done = sc->done;
    const double rho_p = sc->rho_p, alpha = sc->alpha;
    const long stride = (long)gridDim.x * kBlock, i0 = (long)blockIdx.x * kBlock + threadIdx.x;
    // the first pass's loads are in flight while the sums are added
    const long f0 = i0 < n ? i0 : 0, f1 = i0 + stride < n ? i0 + stride : f0;
    TP p0 = Pin[f0], p1 = Pin[f1];
    TZ z0 = Z[f0], z1 = Z[f1];
    const double rz = cg_partials<kBlock>(dots, nd);
    const double qz = FLEX ? cg_partials<kBlock>(dots + nd, nd) : 0.0;
    if (done) return;
    const double be = FLEX ? -alpha * qz / rho_p : rz / rho_p;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->rho = rz;
        sc->beta = be;
        sc->it += 1;
    }
    for (long i = i0; i < n; i += 2 * stride) {
        const bool two = i + stride < n;
        const long j = two ? i + stride : i;
        if (i != i0) {
            p0 = Pin[i];
            p1 = Pin[j];
            z0 = Z[i];
            z1 = Z[j];
        }
        Pout[i] = (TP)fma(be, (double)p0, (double)z0);
        if (two) Pout[j] = (TP)fma(be, (double)p1, (double)z1);
    }
}

// U += alpha_0 P_0 + ... + alpha_{m-1} P_{m-1}, term by term in that order
// (the same fused multiply-adds as one update per iteration).  An iteration
// enqueued after convergence logged alpha 0 and left its slot as it was: with an
// earlier solve's direction, which may not be finite, so the term is left out.
// One element per thread, its m + 1 loads all in flight together.
__global__ __launch_bounds__(kBlock) void k_cg_flush_u(double *__restrict__ U, const float *__restrict__ P, long n,
                                                      const double *__restrict__ alog, int m)
{
    const long i = (long)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    float pv[kCgLog];
#pragma unroll
    for (int t = 0; t < kCgLog; ++t) pv[t] = t < m ? P[(long)t * n + i] : 0.0f;
    double u = U[i];
#pragma unroll
    for (int t = 0; t < kCgLog; ++t)
        if (t < m && alog[t] != 0.0) u = fma(alog[t], (double)pv[t], u);
    U[i] = u;
}

// blocks of the reductions over n elements: two elements per thread at least
int cg_blocks(long n) { return (int)std::min<long>(std::max<long>((n + 2 * kCgThreads - 1) / (2 * kCgThreads), 1), kCgBlocks); }

}  // namespace

void launch_cg_start(hipStream_t s, const double *F, double *U, double *R, long n, CgScalars *sc, double *rr,
                     float *R32, const float *AD32, float *X0, double prerelax)
{
    const int nblk = cg_blocks(n);
    k_cg_start<<<nblk, kCgThreads, 0, s>>>(F, U, R, n, rr, R32, AD32, X0, (float)prerelax);
    k_cg_init<<<1, kBlock, 0, s>>>(sc, rr, nblk);
}
template <class TZ>
void launch_cg_rho(hipStream_t s, const double *r, const TZ *z, long n, CgScalars *sc, double *dots, int nb)
{
    const int nblk = cg_blocks(n);
    k_cg_dots<TZ, false><<<dim3(nblk, 1, batch_dim(nb)), kCgThreads, 0, s>>>(r, z, nullptr, n, dots, &sc->done);
    k_cg_rho0<<<dim3(1, 1, batch_dim(nb)), kBlock, 0, s>>>(sc, dots, nblk);
}
template void launch_cg_rho<double>(hipStream_t, const double *, const double *, long, CgScalars *, double *, int);
template void launch_cg_rho<float>(hipStream_t, const double *, const float *, long, CgScalars *, double *, int);

void launch_cg_init(hipStream_t s, CgScalars *sc, const double *partials, int nparts, int nb)
{
    k_cg_init<<<dim3(1, 1, batch_dim(nb)), kBlock, 0, s>>>(sc, partials, nparts);
}
// alpha in its own launch when there are more sums than every block should
// read; returns the number the update has to read
static int alpha_launch(hipStream_t s, CgScalars *sc, const double *pq, int npq, double *alog, int nb)
{
    if (npq <= kCgFuse) return npq;
    k_cg_alpha<<<dim3(1, 1, batch_dim(nb)), kCgThreads, 0, s>>>(sc, pq, npq, alog);
    return 0;
}

void launch_cg_update_ur(hipStream_t s, double *U, double *R, const double *P, const double *Q, long n, CgScalars *sc,
                         const double *pq, int npq, double *rr, float *R32, int nb)
{
    npq = alpha_launch(s, sc, pq, npq, nullptr, nb);
    k_cg_update_ur<<<dim3(cg_blocks(n), 1, batch_dim(nb)), kCgThreads, 0, s>>>(U, R, P, Q, n, sc, pq, npq, rr, R32);
}

void launch_cg_update_r(hipStream_t s, double *R, const double *Q, long n, CgScalars *sc, const double *pq, int npq,
                        double *rr, double *alog, float *R32, const float *AD32, float *X0, double prerelax)
{
    npq = alpha_launch(s, sc, pq, npq, alog, 1);
    if (X0)
        k_cg_update_r<true><<<cg_blocks(n), kCgThreads, 0, s>>>(R, Q, n, sc, pq, npq, rr, alog, R32, AD32, X0,
                                                                (float)prerelax);
    else
        k_cg_update_r<false><<<cg_blocks(n), kCgThreads, 0, s>>>(R, Q, n, sc, pq, npq, rr, alog, R32, nullptr, nullptr,
                                                                 0.0f);
}

CgTest cg_test_of(CgScalars *sc, const double *rr, long n, double tol, unsigned long long *prog)
{
    CgTest t;
    t.sc = sc;
    t.rr = rr;
    t.n = cg_blocks(n);
    t.tol = tol;
    t.prog = prog;
    return t;
}

void launch_cg_check(hipStream_t s, const CgTest &t, int nb) { k_cg_check<<<dim3(1, 1, batch_dim(nb)), 64, 0, s>>>(t); }

template <class TP, class TZ>
void launch_cg_direction(hipStream_t s, const double *r, const TZ *z, const double *q, TP *Pout, const TP *Pin, long n,
                         CgScalars *sc, double *dots, bool flex, int nb, const double *zr, int nzr)
{
    const int nblk = cg_blocks(n);
    const dim3 gd(nblk, 1, batch_dim(nb));
    const dim3 gp((unsigned)std::min<long>((n + 2 * kBlock - 1) / (2 * kBlock), kCgUpdBlocks), 1, batch_dim(nb));
    if (zr && !flex) {  // the V-cycle's last sweep left the sums
        if (nzr > kCgFuse) {
            k_cg_sum<<<dim3(1, 1, batch_dim(nb)), kCgThreads, 0, s>>>(zr, nzr, dots, &sc->done);
            zr = dots;
            nzr = 1;
        }
        k_cg_update_p<TP, TZ, false><<<gp, kBlock, 0, s>>>(Pout, Pin, z, n, sc, zr, nzr);
    } else if (flex) {
        k_cg_dots<TZ, true><<<gd, kCgThreads, 0, s>>>(r, z, q, n, dots, &sc->done);
        k_cg_update_p<TP, TZ, true><<<gp, kBlock, 0, s>>>(Pout, Pin, z, n, sc, dots, nblk);
    } else {
        k_cg_dots<TZ, false><<<gd, kCgThreads, 0, s>>>(r, z, q, n, dots, &sc->done);
        k_cg_update_p<TP, TZ, false><<<gp, kBlock, 0, s>>>(Pout, Pin, z, n, sc, dots, nblk);
    }
}
template void launch_cg_direction<double, double>(hipStream_t, const double *, const double *, const double *, double *,
                                                  const double *, long, CgScalars *, double *, bool, int,
                                                  const double *, int);
template void launch_cg_direction<float, float>(hipStream_t, const double *, const float *, const double *, float *,
                                                const float *, long, CgScalars *, double *, bool, int,
                                                const double *, int);

void launch_cg_flush_u(hipStream_t s, double *U, const float *P, long n, const double *alog, int m)
{
    if (m > 0) k_cg_flush_u<<<(unsigned)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(U, P, n, alog, m);
}

}  // namespace gputo
