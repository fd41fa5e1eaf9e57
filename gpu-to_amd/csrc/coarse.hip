// Coarse levels of the MGCG hierarchy: level-1 rediscretisation from child
// densities, element-Galerkin operators, the coarsest-level penalty,
// dense assembly, blocked FP64 Cholesky, the explicit inverse of the
// factor (of the matrix, when small) and the products that apply it in every
// V-cycle.
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <vector>

#include "gputo_internal.h"

namespace gputo {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int lidx2(int x, int y, int z) { return 4 * z + (y ? (x ? 2 : 3) : (x ? 1 : 0)); }
__host__ __device__ constexpr int pidx2(int m, int n) { return n <= m ? m * (m + 1) / 2 + n : n * (n + 1) / 2 + m; }
__device__ constexpr int kIE[8] = {0, 1, 1, 0, 0, 1, 1, 0};
__device__ constexpr int kJE[8] = {0, 0, 1, 1, 0, 0, 1, 1};
__device__ constexpr int kKE[8] = {0, 0, 0, 0, 1, 1, 1, 1};

// ---------------------------------------------------------------------------
// Level-1 rediscretisation (coarseAe2c, mgcg1.cu:2042-2070): the packed
// coarse element matrix is sum_na CX[child(na)] * Aelm[:, na] where Aelm
// holds the h=2 Gauss-point stiffness matrices and child na = 4 iP + 2 kP
// + jP.  One thread per coarse element and kL1Entries packed entries (so that
// a small level fills the device, too: 26 us at 128 elements with all 300
// entries in one thread); Aelm is read through the scalar cache (uniform
// addresses).
// ---------------------------------------------------------------------------
constexpr int kL1Entries = 30;

__global__ __launch_bounds__(256) void k_coarse_l1(Grid gc, const double *__restrict__ Aelm,
                                                  const double *__restrict__ CXf, double *__restrict__ A)
{
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= gc.nel) return;
    const int j = (int)(e % gc.ny), k = (int)((e / gc.ny) % gc.nz), i = (int)(e / ((long)gc.ny * gc.nz));
    const int fny = 2 * gc.ny, fnz = 2 * gc.nz;
    double cx[8];
#pragma unroll
    for (int iP = 0; iP < 2; ++iP)
#pragma unroll
        for (int kP = 0; kP < 2; ++kP)
#pragma unroll
            for (int jP = 0; jP < 2; ++jP)
                cx[4 * iP + 2 * kP + jP] = CXf[(long)fny * fnz * (2 * i + iP) + (long)fny * (2 * k + kP) + 2 * j + jP];
    const int m0 = blockIdx.y * kL1Entries;
    for (int m = m0; m < m0 + kL1Entries; ++m) {
        double s = 0.0;
#pragma unroll
        for (int na = 0; na < 8; ++na) s += cx[na] * Aelm[8 * m + na];
        A[(long)m * gc.nel + e] = s;
    }
}

void launch_coarse_l1(hipStream_t s, const Grid &gc, const double *Aelm, const double *CXf, double *A)
{
    k_coarse_l1<<<dim3((unsigned)((gc.nel + 255) / 256), 300 / kL1Entries), 256, 0, s>>>(gc, Aelm, CXf, A);
}

// Diagonal of that operator from the child densities, without its element
// matrices (AD and 1/AD): sum over a node's 8 elements of sum_na CX[child(na)]
// Aelm[(m, m), na], in the element order of k_diag.
__global__ __launch_bounds__(256) void k_diag_l1(Grid g, const double *__restrict__ Aelm,
                                                const double *__restrict__ CXf, double *__restrict__ AD,
                                                double *__restrict__ RD)
{
    const long nod = (long)blockIdx.x * 256 + threadIdx.x;
    if (nod >= g.nnod) return;
    const unsigned nu = (unsigned)nod, q1 = nu / (unsigned)g.nny;
    const int j = (int)(nu - q1 * (unsigned)g.nny), k = (int)(q1 % (unsigned)g.nnz), i = (int)(q1 / (unsigned)g.nnz);
    const int fny = 2 * g.ny, fnz = 2 * g.nz;
    double d[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int ei = 0; ei < 2; ++ei)
#pragma unroll
        for (int ek = 0; ek < 2; ++ek)
#pragma unroll
            for (int ej = 0; ej < 2; ++ej) {
                const int ex = i - 1 + ei, ey = j - 1 + ej, ez = k - 1 + ek;
                if (ex < 0 || ex >= g.nx || ey < 0 || ey >= g.ny || ez < 0 || ez >= g.nz) continue;
                const int la = lidx2(1 - ei, 1 - ej, 1 - ek);
                double cx[8];
#pragma unroll
                for (int na = 0; na < 8; ++na)
                    cx[na] = CXf[(long)fny * fnz * (2 * ex + (na >> 2)) + (long)fny * (2 * ez + ((na >> 1) & 1)) + 2 * ey +
                                 (na & 1)];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int m = 3 * la + c;
                    double s = 0.0;
#pragma unroll
                    for (int na = 0; na < 8; ++na) s += cx[na] * Aelm[8 * pidx2(m, m) + na];
                    d[c] += s;
                }
            }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        AD[3 * nod + c] = d[c];
        if (RD) RD[3 * nod + c] = 1.0 / d[c];
    }
}

void launch_diag_l1(hipStream_t s, const Grid &g, const double *Aelm, const double *CXf, double *AD, double *RD)
{
    k_diag_l1<<<(unsigned)((g.nnod + 255) / 256), 256, 0, s>>>(g, Aelm, CXf, AD, RD);
}

// ---------------------------------------------------------------------------
// Element Galerkin (coarseAe3c, mgcg1.cu:1678-1743): A_c = P (sum of the 8
// children on the 27-node patch) P^T.  P is the trilinear interpolation of
// the coarse element's 8 nodes onto its 27 fine nodes, so the (a,b) node
// block of A_c is
//   sum_ch sum_{p,q} w(a, ch+p) w(b, ch+q) A_ch[p q block],
// with w(a, x) = prod_axis (1 - |2 a_axis - x_axis| / 2).  One block per
// coarse element stages its 8 children's packed matrices in LDS and forms
// T_ch = A_ch P_ch (24 x 24 each, sums over q), then the 300 entries of
// sum_ch P_ch^T T_ch (sums over ch and p).  (36 threads that
// each ran the triple sum for a 3 x 3 block took 91-95 us a launch, however
// few the elements; this form 14 us for 54 elements and 24 us for 432.)
// ---------------------------------------------------------------------------
__device__ __forceinline__ double trilin_w(int a, int x0, int x1, int x2)
{
    // coarse local node a (offsets kIE/kJE/kKE), fine patch node (x0,x1,x2) in {0,1,2}^3
    const double w0 = 1.0 - 0.5 * abs(2 * kIE[a] - x0);
    const double w1 = 1.0 - 0.5 * abs(2 * kJE[a] - x1);
    const double w2 = 1.0 - 0.5 * abs(2 * kKE[a] - x2);
    return w0 * w1 * w2;
}

constexpr int kGalThreads = 256;

__global__ __launch_bounds__(kGalThreads) void k_galerkin(Grid gc, const double *__restrict__ Af,
                                                         double *__restrict__ Ac)
{
    __shared__ double S[8][300];
    __shared__ double T[8][24][25];
    __shared__ double W[8][8][8];  // [child][child node q][coarse node b]
    const long e = blockIdx.x;
    const int j = (int)(e % gc.ny), k = (int)((e / gc.ny) % gc.nz), i = (int)(e / ((long)gc.ny * gc.nz));
    const int fny = 2 * gc.ny, fnz = 2 * gc.nz, tid = threadIdx.x;
    const long nelf = 8 * gc.nel;
    constexpr int kIt = (8 * 300 + kGalThreads - 1) / kGalThreads;
    double v[kIt];
#pragma unroll
    for (int u = 0; u < kIt; ++u) {  // child fastest: neighbouring children are neighbouring in memory
        const int q = tid + u * kGalThreads, ch = q & 7, p = min(q >> 3, 299);
        const long eP = (long)fny * fnz * (2 * i + (ch >> 2)) + (long)fny * (2 * k + ((ch >> 1) & 1)) + 2 * j + (ch & 1);
        v[u] = Af[(long)p * nelf + eP];
    }
    // children in the order (ci, ck, cj) = bits 4, 2, 1
#pragma unroll
    for (int u = 0; u < kIt; ++u) {
        const int q = tid + u * kGalThreads;
        if (q < 8 * 300) S[q & 7][q >> 3] = v[u];
    }
    for (int q = tid; q < 512; q += kGalThreads) {
        const int ch = q >> 6, n = (q >> 3) & 7, b = q & 7;
        W[ch][n][b] = trilin_w(b, (ch >> 2) + kIE[n], (ch & 1) + kJE[n], ((ch >> 1) & 1) + kKE[n]);
    }
    __syncthreads();
    for (int q = tid; q < 8 * 576; q += kGalThreads) {
        const int ch = q / 576, r = (q / 24) % 24, n = q % 24, b = n / 3, d = n - 3 * b;
        double t = 0.0;
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const int m = 3 * p + d;
            t += W[ch][p][b] * S[ch][m <= r ? r * (r + 1) / 2 + m : m * (m + 1) / 2 + r];
        }
        T[ch][r][n] = t;
    }
    __syncthreads();
    for (int q = tid; q < 300; q += kGalThreads) {
        int m = (int)((sqrtf(8.0f * q + 1.0f) - 1.0f) * 0.5f);
        m += (m + 1) * (m + 2) / 2 <= q;
        m -= m * (m + 1) / 2 > q;
        const int n = q - m * (m + 1) / 2, a = m / 3, c = m - 3 * a;
        double t = 0.0;
        for (int ch = 0; ch < 8; ++ch)
#pragma unroll
            for (int p = 0; p < 8; ++p) t += W[ch][p][a] * T[ch][3 * p + c][n];
        Ac[(long)q * gc.nel + e] = t;
    }
}

void launch_coarse_galerkin(hipStream_t s, const Grid &gc, const double *Af, double *Ac)
{
    k_galerkin<<<(unsigned)gc.nel, kGalThreads, 0, s>>>(gc, Af, Ac);
}

// ---------------------------------------------------------------------------
// Element-Galerkin operators from per-fine-element tables.  The Galerkin
// product of level l (coarseAe3c, mgcg1.cu:1653-1743: A_c = P^T (sum of the 8
// children) P with the trilinear P of mgcg1.cu:1653-1676) is linear in the
// level-0 element scales, so the level-l element matrix is
//   A_e = sum_f CX[f] T_l[f],   f over the 8^l level-0 elements inside e,
// with T_l[f] = P_chain(f)^T B(f) P_chain(f) fixed per fine position: B = Ke
// when level 1 is itself Galerkin, B = the Gauss-point matrix of f's position
// in its level-1 parent when level 1 is rediscretised (coarseAe2c,
// mgcg1.cu:2042-2070).  The tables are built once on the host; the device
// work per level is one [nel_l x 8^l] x [8^l x 300] product.  Same operator
// as the child-by-child product, summed in a different order.
// ---------------------------------------------------------------------------
// The product on the matrix cores: D[p][e] = sum_f T[f][p] CX0[fine(e, f)]
// as v_mfma_f64_16x16x4f64 tiles (operand layout at dgemm_tile32), p (the
// packed entry) along the rows and e along the columns, so the stores of a
// tile row are contiguous in A (p-major).  One wave per 32 x 32 tile of
// (p, e), four waves per workgroup; the operands come straight from L2 (the
// table is at most 1.2 MB, CX0 is read once per p tile), kGtAhead K steps
// of loads in flight.
constexpr int kGtAhead = 8;

__global__ __launch_bounds__(256) void k_galerkin_table(Grid gc, int depth, const double *__restrict__ T,
                                                       const double *__restrict__ CX0, double *__restrict__ A)
{
    const int lane = threadIdx.x & 63;
    const long wt = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const long etiles = (gc.nel + 31) / 32;
    const int p0 = (int)(wt / etiles) * 32;
    const long e0 = (wt % etiles) * 32;
    if (p0 >= 300) return;  // whole wave
    const int S = 1 << depth, nf = S * S * S;
    const long ny0 = (long)gc.ny * S, nz0 = (long)gc.nz * S;
    const int i16 = lane & 15, kq = lane >> 4;
    // B operand: element e0 + 16 b + i16 of this lane, its first fine element
    long eb[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const long e = e0 + 16 * b + i16;
        eb[b] = -1;
        if (e < gc.nel) {
            const long i = e / ((long)gc.ny * gc.nz), k = (e / gc.ny) % gc.nz, j = e % gc.ny;
            eb[b] = (i * S) * nz0 * ny0 + (k * S) * ny0 + j * S;
        }
    }
    f64x4 d[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) d[a][b] = f64x4{0.0, 0.0, 0.0, 0.0};
    for (int f0 = 0; f0 < nf; f0 += 4 * kGtAhead) {
        double fa[kGtAhead][2], fb[kGtAhead][2];
#pragma unroll
        for (int u = 0; u < kGtAhead; ++u) {
            const int f = f0 + 4 * u + kq;  // this lane's K index
            const bool fin = f < nf;
            const long fo = (long)(f / (S * S)) * nz0 * ny0 + (long)((f / S) % S) * ny0 + f % S;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int p = p0 + 16 * a + i16;
                fa[u][a] = (fin && p < 300) ? T[(long)f * 300 + p] : 0.0;
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) fb[u][b] = (fin && eb[b] >= 0) ? CX0[eb[b] + fo] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kGtAhead; ++u)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    d[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[u][a], fb[u][b], d[a][b], 0, 0, 0);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const long e = e0 + 16 * b + i16;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int p = p0 + 16 * a + 4 * v + kq;
                if (p < 300 && e < gc.nel) A[(long)p * gc.nel + e] = d[a][b][v];
            }
        }
}

void launch_galerkin_table(hipStream_t s, const Grid &gc, int depth, const double *T, const double *CX0, double *A)
{
    const long waves = 10 * ((gc.nel + 31) / 32);  // ceil(300 / 32) p tiles
    k_galerkin_table<<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(gc, depth, T, CX0, A);
}

// Host: the tables T_l for l = 1..maxdepth, packed [8^l][300] with the
// fine position f = (fi*S + fk)*S + fj, S = 2^l.  base1: the 8 full matrices
// of depth 1 (index 4 fi + 2 fk + fj), or nullptr to start from Ke at depth 0.
static void child_prolongation(int cx, int cy, int cz, double P[24][24])
{
    // P[3a+d][3b+d] = trilinear weight of parent node b at child node a
    static const int ie[8] = {0, 1, 1, 0, 0, 1, 1, 0}, je[8] = {0, 0, 1, 1, 0, 0, 1, 1}, ke[8] = {0, 0, 0, 0, 1, 1, 1, 1};
    for (int r = 0; r < 24; ++r)
        for (int c = 0; c < 24; ++c) P[r][c] = 0.0;
    for (int a = 0; a < 8; ++a)
        for (int b = 0; b < 8; ++b) {
            const double w = (1.0 - 0.5 * std::abs(cx + ie[a] - 2 * ie[b])) * (1.0 - 0.5 * std::abs(cy + je[a] - 2 * je[b])) *
                             (1.0 - 0.5 * std::abs(cz + ke[a] - 2 * ke[b]));
            for (int d = 0; d < 3; ++d) P[3 * a + d][3 * b + d] = w;
        }
}

std::vector<std::vector<double>> galerkin_tables(const double *Ke, const double *base1, int maxdepth)
{
    std::vector<std::vector<double>> out(maxdepth + 1);
    std::vector<double> cur;  // full matrices of the current depth, [S^3][576]
    int d = 0;
    if (base1) {
        cur.assign(8 * 576, 0.0);
        for (int fi = 0; fi < 2; ++fi)
            for (int fk = 0; fk < 2; ++fk)
                for (int fj = 0; fj < 2; ++fj)
                    std::copy(base1 + 576 * (4 * fi + 2 * fk + fj), base1 + 576 * (4 * fi + 2 * fk + fj) + 576,
                              cur.begin() + 576 * ((fi * 2 + fk) * 2 + fj));
        d = 1;
    } else {
        cur.assign(Ke, Ke + 576);
    }
    auto pack = [](const std::vector<double> &full, int n) {
        std::vector<double> t((size_t)n * 300);
        for (int f = 0; f < n; ++f)
            for (int m = 0; m < 24; ++m)
                for (int c = 0; c <= m; ++c) t[(size_t)f * 300 + m * (m + 1) / 2 + c] = full[(size_t)f * 576 + 24 * m + c];
        return t;
    };
    if (d >= 1 && d <= maxdepth) out[d] = pack(cur, 8);
    double P[8][24][24];
    for (int c = 0; c < 8; ++c) child_prolongation(c & 1, (c >> 1) & 1, c >> 2, P[c]);
    while (d < maxdepth) {
        const int S = 1 << d, S2 = 2 * S;
        std::vector<double> nxt((size_t)S2 * S2 * S2 * 576);
        double tmp[24][24];
        for (int fi = 0; fi < S2; ++fi)
            for (int fk = 0; fk < S2; ++fk)
                for (int fj = 0; fj < S2; ++fj) {
                    const int cx = fi / S, cy = fj / S, cz = fk / S;
                    const double(*Pc)[24] = P[cx + 2 * cy + 4 * cz];
                    const double *B = &cur[(size_t)(((fi % S) * S + (fk % S)) * S + (fj % S)) * 576];
                    // tmp = B P, then out = P^T tmp
                    for (int r = 0; r < 24; ++r)
                        for (int c = 0; c < 24; ++c) {
                            double acc = 0.0;
                            for (int q = 0; q < 24; ++q) acc += B[24 * r + q] * Pc[q][c];
                            tmp[r][c] = acc;
                        }
                    double *o = &nxt[(size_t)((fi * S2 + fk) * S2 + fj) * 576];
                    for (int r = 0; r < 24; ++r)
                        for (int c = 0; c < 24; ++c) {
                            double acc = 0.0;
                            for (int q = 0; q < 24; ++q) acc += Pc[q][r] * tmp[q][c];
                            o[24 * r + c] = acc;
                        }
                }
        cur.swap(nxt);
        ++d;
        out[d] = pack(cur, S2 * S2 * S2);
    }
    return out;
}

// ---------------------------------------------------------------------------
// mgcg9 coarse levels (Homogenization/QNC/mgcg9.cu).
// formCXc (:753-789): CX_c = 2 * mean of the 8 children, summed in the
// reference's child order.
__global__ void k_coarse_cx(Grid gc, const double *__restrict__ CXf, double *__restrict__ CXc)
{
    const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= gc.nel) return;
    const int j = (int)(e % gc.ny), k = (int)((e / gc.ny) % gc.nz), i = (int)(e / ((long)gc.ny * gc.nz));
    const long fny = 2L * gc.ny, fnz = 2L * gc.nz;
    double s = 0.0;
    for (int iP = 0; iP < 2; ++iP)
        for (int kP = 0; kP < 2; ++kP)
            for (int jP = 0; jP < 2; ++jP) s += CXf[fnz * fny * (2 * i + iP) + fny * (2 * k + kP) + 2 * j + jP];
    CXc[e] = 2.0 * (s / 8);
}

void launch_coarse_cx(hipStream_t s, const Grid &gc, const double *CXf, double *CXc)
{
    k_coarse_cx<<<(unsigned)((gc.nel + 255) / 256), 256, 0, s>>>(gc, CXf, CXc);
}

// packed element matrices CX_e Ke (assembAQc's element products, :1747-...)
__global__ void k_ke_elements(Grid g, const double *__restrict__ CX, const double *__restrict__ Ke,
                              double *__restrict__ A)
{
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= 300 * g.nel) return;
    const int p = (int)(q / g.nel);
    const long e = q % g.nel;
    int m = 0;
    while ((m + 1) * (m + 2) / 2 <= p) ++m;
    const int n = p - m * (m + 1) / 2;
    A[q] = CX[e] * Ke[24 * m + n];
}

void launch_ke_elements(hipStream_t s, const Grid &g, const double *CX, const double *Ke, double *A)
{
    k_ke_elements<<<(unsigned)((300 * g.nel + 255) / 256), 256, 0, s>>>(g, CX, Ke, A);
}

// periodic cells, CorrCsAQc (:1005-1028): zero the rows and columns of the fixed DOFs of
// the dense coarsest matrix (N x N, row-major), then 1e10 on their diagonal
__global__ void k_zero_rowcol(int N, const int *__restrict__ fixed, int nfd, double *__restrict__ AQ)
{
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long)nfd * N) return;
    const long d = fixed[q / N], i = q % N;
    AQ[d * N + i] = 0.0;
    AQ[i * N + d] = 0.0;
}

__global__ void k_fixed_diag(int N, const int *__restrict__ fixed, int nfd, double *__restrict__ AQ)
{
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f < nfd) AQ[(long)fixed[f] * N + fixed[f]] = 1e10;
}

void launch_zero_rowcol(hipStream_t s, int N, const int *fixed_d, int nfd, double *AQ)
{
    if (nfd <= 0) return;
    k_zero_rowcol<<<(unsigned)(((long)nfd * N + 255) / 256), 256, 0, s>>>(N, fixed_d, nfd, AQ);
    k_fixed_diag<<<(unsigned)((nfd + 255) / 256), 256, 0, s>>>(N, fixed_d, nfd, AQ);
}

// ---------------------------------------------------------------------------
// Coarsest-level penalty (CorrCsAc, mgcg1.cu:1368-1402): the diagonal of
// every incident element matrix is set to 1e10 for each fixed DOF.  The
// reference's table {5,6,1,2,4,7,0,3} is the y-mirror of the node's own
// local index {6,5,2,1,7,4,3,0}; `mirrored` selects it.  Threads that hit
// the same entry store the same value.
// ---------------------------------------------------------------------------
__global__ void k_corrcsa(Grid g, const int *__restrict__ fixed, int nfd, double *__restrict__ A, int mirrored)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nfd) return;
    const int tmir[8] = {5, 6, 1, 2, 4, 7, 0, 3};
    const int town[8] = {6, 5, 2, 1, 7, 4, 3, 0};
    const int dof = fixed[n];
    const int idof = dof % 3, nod = dof / 3;
    const int i = nod / (g.nnz * g.nny);
    const int k = (nod - g.nnz * g.nny * i) / g.nny;
    const int j = nod - g.nnz * g.nny * i - g.nny * k;
    for (int di = -1; di <= 0; di++)
        for (int dk = -1; dk <= 0; dk++)
            for (int dj = -1; dj <= 0; dj++) {
                const int iP = i + di, jP = j + dj, kP = k + dk;
                if (iP < 0 || iP > g.nx - 1 || jP < 0 || jP > g.ny - 1 || kP < 0 || kP > g.nz - 1) continue;
                const long e = (long)g.ny * g.nz * iP + (long)g.ny * kP + jP;
                const int t = 4 * (di + 1) + 2 * (dk + 1) + dj + 1;
                const int n1 = mirrored ? tmir[t] : town[t];
                const int m = 3 * n1 + idof;
                A[(long)pidx2(m, m) * g.nel + e] = 1e10;
            }
}

void launch_corrcsa(hipStream_t s, const Grid &g, const int *fixed_d, int nfd, double *A, int mirrored)
{
    if (nfd > 0) k_corrcsa<<<(nfd + 255) / 256, 256, 0, s>>>(g, fixed_d, nfd, A, mirrored);
}

// ---------------------------------------------------------------------------
// Order of the factored coarsest matrix.  The steps of a band matrix eliminated
// from one end are a chain.  The node planes i = const are therefore split at the middle plane a: part 1
// holds planes 0 .. a-1 in order, part 2 planes nnx-1 .. a+1 in reverse, and
// the separator, plane a, comes last.  Each part followed by the separator is
// a band matrix of its own (the parts do not couple), so both are eliminated at
// once, the chain is half as long, and the inverse of the factor has a zero
// block between the parts.  Parts are padded to whole
// 32 x 32 tiles in front, the separator behind, with identity rows.
// The factorisation takes 265 us at 13 x 7 x 7 nodes (1911 DOFs; 840 in one
// workgroup as one band) and 430 at 12 x 8 x 10 (2880; 2200 as one band by three
// launches per block column).
//
// coarse_dof: the DOF of entry c of that order (-1: padding).  part_dof: of
// row r of part q followed by the separator.
// ---------------------------------------------------------------------------
constexpr int NB = 32;

__host__ __device__ inline int coarse_dof(const CoarseMap &m, int c)
{
    if (m.ps == 0) return c < m.n ? c : -1;  // one part
    if (c < m.o2) return c >= m.pad1 ? c - m.pad1 : -1;
    if (c < m.os) {
        c -= m.o2 + m.pad2;
        if (c < 0) return -1;
        const int q = (int)(((float)c + 0.5f) * m.rp);  // c / p: exact below 2^20
        return (m.nplanes - 1 - q) * m.p + (c - q * m.p);
    }
    c -= m.os;
    return c < m.p ? m.a * m.p + c : -1;
}

__device__ __forceinline__ int part_dof(const CoarseMap &m, int q, int r)
{
    const int len = q == 0 ? m.o2 : m.os - m.o2;
    return coarse_dof(m, r < len ? (q == 0 ? r : m.o2 + r) : m.os + r - len);
}

// Dense coarsest assembly (assembAc, mgcg1.cu:1747-1806) of each part with the
// separator.  One block per row writes its columns from `back` tiles before
// its own tile to the end of that (zeros included: nothing beyond is read),
// each thread one column: the entry sums the elements that hold both nodes, up
// to 8.  The separator's own block goes to part 1 (part 2: zeros).  mask (may
// be null): the rows and columns of fixed DOFs are decoupled, 1e10 on their
// diagonal (CorrCsAQc, Homogenization/QNC/mgcg9.cu:1005-1028).  (One thread
// per row that added its 192 element entries to zeroed memory one by one took
// 29-60 us after a fill of the whole matrix; 5-8 us now, and no fill.)
__global__ __launch_bounds__(256) void k_assemble(Grid g, CoarseMap m, const double *__restrict__ A,
                                                 const uint8_t *__restrict__ mask, CoarseParts P, int back)
{
    int q = 0, r = blockIdx.x;
    if (P.np > 1 && r >= P.n[0]) {
        q = 1;
        r -= P.n[0];
    }
    const int c0 = max(0, r / NB - back) * NB, c1 = (r / NB + 1) * NB;
    const int len = q == 0 ? m.o2 : m.os - m.o2;
    const int dr = part_dof(m, q, r);
    const int nr = dr / 3, cr = dr - 3 * nr;
    const int j = nr % g.nny, k = (nr / g.nny) % g.nnz, i = nr / (g.nny * g.nnz);
    const bool rfix = mask && dr >= 0 && ((mask[nr] >> cr) & 1u);
    for (int c = c0 + (int)threadIdx.x; c < c1; c += 256) {
        double v = 0.0;
        const int dc = part_dof(m, q, c);
        const bool second = q == 1 && r >= len && c >= len;  // the separator's block of part 2
        if (dr < 0 || dc < 0) {
            v = r == c && !second ? 1.0 : 0.0;
        } else if (!second) {
            const int nc = dc / 3, cc = dc - 3 * nc;
            const int dj = nc % g.nny - j, dk = (nc / g.nny) % g.nnz - k, di = nc / (g.nny * g.nnz) - i;
            if (mask && (rfix || ((mask[nc] >> cc) & 1u))) {
                v = dr == dc ? 1e10 : 0.0;
            } else if (abs(di) <= 1 && abs(dk) <= 1 && abs(dj) <= 1) {
                for (int ei = 0; ei < 2; ++ei)
                    for (int ek = 0; ek < 2; ++ek)
                        for (int ej = 0; ej < 2; ++ej) {
                            const int ex = i - 1 + ei, ey = j - 1 + ej, ez = k - 1 + ek;
                            const int bx = di + 1 - ei, bz = dk + 1 - ek, by = dj + 1 - ej;
                            if (ex < 0 || ex >= g.nx || ey < 0 || ey >= g.ny || ez < 0 || ez >= g.nz) continue;
                            if (bx < 0 || bx > 1 || by < 0 || by > 1 || bz < 0 || bz > 1) continue;
                            const long e = (long)g.ny * g.nz * ex + (long)g.ny * ez + ey;
                            const int mm = 3 * lidx2(1 - ei, 1 - ej, 1 - ek) + cr, nn = 3 * lidx2(bx, by, bz) + cc;
                            v += A[(long)pidx2(mm, nn) * g.nel + e];
                        }
            }
        }
        P.A[q][(long)r * P.n[q] + c] = v;
    }
}

// The factorisation reads up to nbt = (bw + 2 NB - 2) / NB tiles before a
// row's own, the corners of the inverse's products up to 2 nbt - 1.
void launch_assemble(hipStream_t s, const Grid &g, const double *A, const uint8_t *mask, const Coarse &C)
{
    const CoarseParts P = coarse_parts(C);
    k_assemble<<<P.n[0] + (P.np > 1 ? P.n[1] : 0), 256, 0, s>>>(g, C.map, A, mask, P, 2 * ((C.bw + 2 * NB - 2) / NB));
}

// ---------------------------------------------------------------------------
// Blocked right-looking Cholesky A = L L^T on a row-major matrix (lower triangle
// used), NB = 32: factor the diagonal tile, solve the panel below it, update the
// trailing lower triangle.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Columns J0..J1-1 of the tile factorisation in one wave, lane r < NB
// holding row r in L (r >= NB: a row below the tile): at step jj the pivot comes from lane jj and each
// multiplier L[c][jj] from lane c by v_readlane (scalar operands of the
// updates), so no memory round trip is on the chain of pivots.  Only
// columns below J1 are updated.  Entries right of the diagonal (c > r) take
// garbage that is never read: lj = 0 on rows above the column, and only
// c <= r is stored.
template <int J0, int J1>
__device__ __forceinline__ void potrf_cols(double (&L)[NB], int r, bool &bad)
{
#pragma unroll
    for (int jj = J0; jj < J1; ++jj) {
        double d = readlane_f64(L[jj], jj);  // updated A[jj][jj]
        if (!(d > 0.0)) {  // not positive definite (or NaN)
            bad = true;
            d = 1.0;
        }
        // y = 1/sqrt(d): v_rsq_f64 (2^-29 relative) and one Newton step;
        // the pivot is d y and the column is scaled by y, so the chain of a
        // column has no square root or division in it
        double y = __builtin_amdgcn_rsq(d);
        y = y * fma(-0.5 * d * y, y, 1.5);
        const double lj = r == jj ? d * y : (r > jj ? L[jj] * y : 0.0);
        L[jj] = lj;
#pragma unroll
        for (int c = jj + 1; c < J1; ++c) L[c] -= lj * readlane_f64(lj, c);  // L[c][jj]
    }
}

__device__ __forceinline__ void wave_lds_sync()
{
    // LDS operations of one wave complete in order; the fences keep the
    // compiler from moving them across
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void tri_index(int b, int &ti, int &tj)
{
    // b-th tile of a lower-triangular tile set: (ti, tj) with tj <= ti
    int t = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while ((t + 1) * (t + 2) / 2 <= b) ++t;
    while (t * (t + 1) / 2 > b) --t;
    ti = t;
    tj = b - t * (t + 1) / 2;
}

// Inverse of each 32x32 diagonal factor tile, written into Linv (one wave per
// tile of the whole order): lane c < 32 solves column c of the inverse of its
// 16x16 half, then X10 = -X11 L10 X00 on the matrix cores.  (32 rows in turn
// with a division each: 14 us; 7 us.)
__global__ __launch_bounds__(64) void k_trtri_diag(CoarseBlocks B, double *Linv, int N)
{
    __shared__ double L[NB][NB + 1], X[NB][NB + 1], P[16][17], rd[NB];
    const int k0 = blockIdx.x * NB, lane = threadIdx.x;
    int q = 0;
    while (q + 1 < B.nblk && k0 >= B.off[q + 1]) ++q;
    const double *A = B.L[q];
    const long ld = B.ld[q];
    const int l0 = k0 - B.off[q];
    double v[NB * NB / 64];
#pragma unroll
    for (int u = 0; u < NB * NB / 64; ++u) {
        const int r = (lane + 64 * u) / NB, c = lane % NB;
        v[u] = c <= r ? A[(l0 + r) * ld + l0 + c] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < NB * NB / 64; ++u) {
        const int r = (lane + 64 * u) / NB, c = lane % NB;
        L[r][c] = v[u];
        X[r][c] = 0.0;
        if (r == c) rd[r] = 1.0 / v[u];
    }
    __syncthreads();
    if (lane < NB) {
        const int h = lane & 16, col = lane & 15;
        double x[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            double t = r == col ? 1.0 : 0.0;
#pragma unroll
            for (int m = 0; m < r; ++m) t -= L[h + r][h + m] * x[m];
            x[r] = r < col ? 0.0 : t * rd[h + r];
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) X[h + r][lane] = x[r];
    }
    __syncthreads();
    const int i = lane & 15, kq = lane >> 4;
    f64x4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4)  // L10 X00
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(L[16 + i][kk + kq], X[kk + kq][i], d, 0, 0, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) P[4 * u + kq][i] = d[u];
    __syncthreads();
    d = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4)
        d = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 + i][16 + kk + kq], P[kk + kq][i], d, 0, 0, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) X[16 + 4 * u + kq][i] = -d[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NB * NB / 64; ++u) {
        const int r = (lane + 64 * u) / NB, c = lane % NB;
        Linv[(long)(k0 + r) * N + k0 + c] = X[r][c];
    }
}

// of the tiles on and below the diagonal: the others are neither written nor read
__global__ void k_transpose(const double *__restrict__ In, double *__restrict__ Out, int N)
{
    __shared__ double T[NB][NB + 1];
    if (blockIdx.x > blockIdx.y) return;
    const int bi = blockIdx.y * NB, bj = blockIdx.x * NB;
    for (int q = threadIdx.x; q < NB * NB; q += blockDim.x) T[q / NB][q % NB] = In[(long)(bi + q / NB) * N + bj + q % NB];
    __syncthreads();
    for (int q = threadIdx.x; q < NB * NB; q += blockDim.x) Out[(long)(bj + q / NB) * N + bi + q % NB] = T[q % NB][q / NB];
}

// sum_m A[i][m] B[j][m] for a 16x16 block, D layout of the MFMA;
// every operand is read from LDS before the chain starts, so the matrix
// core does not wait on each pair of reads
typedef double CholTile[NB][NB + 1];
__device__ __forceinline__ f64x4 panel_product(const double (*A)[NB + 1], const double (*B)[NB + 1], int lane)
{
    const int i = lane & 15, k = lane >> 4;
    double fa[NB / 4], fb[NB / 4];
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
        fa[s] = A[i][4 * s + k];
        fb[s] = B[i][4 * s + k];
    }
    f64x4 d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) d = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s], fb[s], d, 0, 0, 0);
    return d;
}

// One wave: D = L L^T in place (lower triangle) and P <- P L^-T.  Lane r < NB
// holds row r of D, the others a row of P: the column operations that factor the
// one solve the other.  In two halves of 16 columns, the second updated by the
// first on the matrix cores.
__device__ __forceinline__ bool factor_solve(CholTile &D, CholTile &P, int lane)
{
    double L[NB];
    bool bad = false;
    const int r = lane < NB ? lane : 2 * NB;  // below every column
    double *V = lane < NB ? D[lane] : P[lane - NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) L[c] = c <= r ? V[c] : 0.0;
    potrf_cols<0, 16>(L, r, bad);
    wave_lds_sync();  // every lane has read its row
#pragma unroll
    for (int c = 0; c < 16; ++c) V[c] = L[c];
    wave_lds_sync();
    f64x4 v[3];
#pragma unroll
    for (int rb = 0; rb < 3; ++rb) {
        const double(*R)[NB + 1] = rb == 0 ? D + 16 : P + 16 * (rb - 1);
        v[rb] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4)
            v[rb] = __builtin_amdgcn_mfma_f64_16x16x4f64(R[lane & 15][kk + (lane >> 4)],
                                                         D[16 + (lane & 15)][kk + (lane >> 4)], v[rb], 0, 0, 0);
    }
#pragma unroll
    for (int rb = 0; rb < 3; ++rb) {
        double(*R)[NB + 1] = rb == 0 ? D + 16 : P + 16 * (rb - 1);
#pragma unroll
        for (int u = 0; u < 4; ++u) R[4 * u + (lane >> 4)][16 + (lane & 15)] = v[rb][u];
    }
    wave_lds_sync();
    if (lane >= 16) {
#pragma unroll
        for (int c = 16; c < NB; ++c) L[c] -= V[c];
    }
    potrf_cols<16, NB>(L, r, bad);
    wave_lds_sync();
#pragma unroll
    for (int c = 16; c < NB; ++c) V[c] = L[c];
    return bad;
}

// ---------------------------------------------------------------------------
// Cholesky A = L L^T of the lower band, one launch per two block columns of 32 (a
// step; a last odd one alone) while the tiles of a step fit the chip.  Every
// workgroup owns one 32x32 tile (ti, tj) of the trailing band and does all it needs
// for it: it factors the step's diagonal tiles, solves the panel tiles of its rows
// and columns and subtracts their products.  The repeated work costs nothing where
// the CUs would idle, and nothing waits for another workgroup.  The factor goes to
// its own matrix, since other workgroups of the launch still read the panel as it
// was.  A step of one block column takes 8.7 us, of which the launch 2.7, the loads
// 1 and the chain of 32 pivots most of the rest; of two 15.7.  (In one workgroup
// with a look-ahead, the FP64 rate of one CU and barriers: 7 us per block column at
// a band of 65 rows, 13 at 173 and 25 at 269; with three launches per block
// column, tile, panel and update, 25 us.)
// A step of more than kCholFit tiles would repeat the chain in several rounds: it
// solves its panel once per row tile, and a second launch updates the trailing
// band.  The set-up of a periodic cell takes 28.2 ms at 6591 DOFs and 307 at 14739
// with the first form alone, 8.2 and 82 with both (three launches per block column:
// 17.3 and 152); a plate of 5x33x33 coarsest nodes (band 3371) 58.4, 23.8 (53.5).
// ---------------------------------------------------------------------------
struct CholStep {
    double *A[2], *L[2];
    long ld[2];
    int n[2], steps[2];
    int nt;  // tiles of the band below the diagonal tile
    int *flag;
};

__global__ __launch_bounds__(256) void k_chol_step(CholStep a)
{
    __shared__ CholTile W[4];  // the diagonal tile and a panel tile, for wave 0 and for wave 1
    const int q = blockIdx.y, k = a.steps[q] - 1;
    if (!(a.steps[q] & 1)) return;  // the last block column, where their number is odd
    const long ld = a.ld[q], k0 = (long)k * NB;
    const int nt = min(a.nt, a.n[q] / NB - k - 1);
    int ti, tj;
    tri_index(blockIdx.x, ti, tj);
    const bool tile = ti < nt;
    if (!tile && blockIdx.x > 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const double *Ak = a.A[q] + k0 * ld + k0;
    const long ri = (long)(ti + 1) * NB, rj = (long)(tj + 1) * NB;
    // this wave's quadrant of the tile, in the MFMA's result layout
    double *Tq = a.A[q] + (k0 + ri + 16 * (wave >> 1) + (lane >> 4)) * ld + k0 + rj + 16 * (wave & 1) + (lane & 15);
    double d[4], pi[4] = {}, pj[4] = {}, old[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        d[u] = Ak[r * ld + c];
        if (tile) {
            pi[u] = Ak[(ri + r) * ld + c];
            pj[u] = Ak[(rj + r) * ld + c];
            old[u] = Tq[4 * u * ld];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        W[0][r][c] = d[u];
        W[1][r][c] = pi[u];
        W[2][r][c] = d[u];
        W[3][r][c] = pj[u];
    }
    __syncthreads();
    if (wave < 2 && factor_solve(W[2 * wave], W[2 * wave + 1], lane) && blockIdx.x == 0 && tid == 0) a.flag[0] = 1;
    __syncthreads();
    if (tile) {
        const f64x4 v = panel_product(W[1] + 16 * (wave >> 1), W[3] + 16 * (wave & 1), lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) Tq[4 * u * ld] = old[u] - v[u];
    }
    if (tj > 0) return;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        if (blockIdx.x == 0 && c <= r) a.L[q][(k0 + r) * ld + k0 + c] = W[0][r][c];
        if (tile) a.L[q][(k0 + ri + r) * ld + k0 + c] = W[1][r][c];
    }
}

// Block columns k and k + 1 of every part that has both.  Wave 0 solves the tile
// between the two diagonal tiles, waves 1 and 2 the panel tiles of the workgroup's
// rows and columns, each with its own copy of the first diagonal tile; the second
// diagonal tile and the second panel tiles are updated on the matrix cores
// (quadrant w of each by wave w), then waves 1 and 2 go on with those.
// PANEL: one workgroup per row tile, which leaves the trailing band to
// k_chol_update.
template <bool PANEL>
__global__ __launch_bounds__(256) void k_chol_step2(CholStep a, int k)
{
    constexpr int NP = PANEL ? 1 : 2;
    __shared__ CholTile D[1 + NP], X, P[NP], Q[NP];  // diagonal tile (a copy per wave), the tile below it, panel tiles
    const int q = blockIdx.y;
    if (k + 1 >= a.steps[q]) return;
    const long ld = a.ld[q], k0 = (long)k * NB;
    const int nt = min(a.nt, a.n[q] / NB - k - 2);
    int ti = blockIdx.x, tj = 0;
    if (!PANEL) tri_index(blockIdx.x, ti, tj);
    const bool tile = ti < nt;
    if (!tile && blockIdx.x > 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qr = 16 * (wave >> 1), qc = 16 * (wave & 1);  // this wave's quadrant
    double *Ak = a.A[q] + k0 * ld + k0;
    const long ri = (long)(ti + 2) * NB, rj = (long)(tj + 2) * NB;
    // quadrants in the MFMA's result layout
    const long qo = (qr + (lane >> 4)) * ld + qc + (lane & 15);
    double *Tq = Ak + ri * ld + rj + qo;
    const double *Eq = Ak + NB * ld + NB + qo, *Pq = Ak + ri * ld + NB + qo, *Jq = Ak + rj * ld + NB + qo;
    double d[4], x[4], pi[4] = {}, pj[4] = {}, e[4], oi[4] = {}, oj[4] = {}, old[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        d[u] = Ak[r * ld + c];
        x[u] = Ak[(NB + r) * ld + c];
        e[u] = Eq[4 * u * ld];
        if (tile) {
            pi[u] = Ak[(ri + r) * ld + c];
            oi[u] = Pq[4 * u * ld];
            if (!PANEL) {
                pj[u] = Ak[(rj + r) * ld + c];
                oj[u] = Jq[4 * u * ld];
                old[u] = Tq[4 * u * ld];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
#pragma unroll
        for (int w = 0; w <= NP; ++w) D[w][r][c] = d[u];
        X[r][c] = x[u];
        P[0][r][c] = pi[u];
        if (!PANEL) P[NP - 1][r][c] = pj[u];
    }
    __syncthreads();
    bool bad = false;
    if (wave == 0) bad = factor_solve(D[0], X, lane);
    if (wave >= 1 && wave <= NP) factor_solve(D[wave], P[wave - 1], lane);
    __syncthreads();
    {
        const f64x4 ve = panel_product(X + qr, X + qc, lane), vi = panel_product(P[0] + qr, X + qc, lane);
        f64x4 vj = {0.0, 0.0, 0.0, 0.0};
        if (!PANEL) vj = panel_product(P[NP - 1] + qr, X + qc, lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int r = qr + 4 * u + (lane >> 4), c = qc + (lane & 15);
#pragma unroll
            for (int w = 1; w <= NP; ++w) D[w][r][c] = e[u] - ve[u];
            Q[0][r][c] = oi[u] - vi[u];
            if (!PANEL) Q[NP - 1][r][c] = oj[u] - vj[u];
        }
    }
    __syncthreads();
    if (wave >= 1 && wave <= NP) bad = factor_solve(D[wave], Q[wave - 1], lane);
    if (bad && blockIdx.x == 0 && lane == 0 && wave < 2) a.flag[0] = 1;
    __syncthreads();
    if (!PANEL && tile) {
        const f64x4 v = panel_product(P[0] + qr, P[NP - 1] + qc, lane), w = panel_product(Q[0] + qr, Q[NP - 1] + qc, lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) Tq[4 * u * ld] = (old[u] - v[u]) - w[u];
    }
    if (tj > 0) return;
    double *Lk = a.L[q] + k0 * ld + k0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        if (blockIdx.x == 0) {
            Lk[(NB + r) * ld + c] = X[r][c];
            if (c <= r) {
                Lk[r * ld + c] = D[0][r][c];
                Lk[(NB + r) * ld + NB + c] = D[1][r][c];
            }
        }
        if (tile) {
            Lk[(ri + r) * ld + c] = P[0][r][c];
            Lk[(ri + r) * ld + NB + c] = Q[0][r][c];
        }
    }
}

// The trailing band after k_chol_step2<true>: A -= L L^T over block columns k and
// k + 1, two by two tiles per workgroup, one per wave.  Both operands are rows of
// the factor; a lane of group g = lane / 16 holds columns 2g and 2g + 1 of eight (as
// in dgemm_tile32), and the loads are two batches of eight ahead.
__global__ __launch_bounds__(256) void k_chol_update(CholStep a, int k)
{
    typedef double f64x2 __attribute__((ext_vector_type(2)));
    const int q = blockIdx.y;
    if (k + 1 >= a.steps[q]) return;
    const int nt = min(a.nt, a.n[q] / NB - k - 2);
    int ti, tj;
    tri_index(blockIdx.x, ti, tj);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ti = 2 * ti + (wave >> 1);
    tj = 2 * tj + (wave & 1);
    if (ti >= nt || tj > ti) return;
    const long ld = a.ld[q], k0 = (long)k * NB, r0 = k0 + 2 * NB;
    const int i = lane & 15, g = lane >> 4;
    const double *Li = a.L[q] + (r0 + (long)ti * NB + i) * ld + k0 + 2 * g;
    const double *Lj = a.L[q] + (r0 + (long)tj * NB + i) * ld + k0 + 2 * g;
    double *T = a.A[q] + (r0 + (long)ti * NB + g) * ld + r0 + (long)tj * NB + i;
    constexpr int kBatches = 2 * NB / 8, kAhead = 2;
    f64x2 fa[kAhead + 1][2], fb[kAhead + 1][2];
    auto load = [&](int s) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            fa[s % (kAhead + 1)][h] = *reinterpret_cast<const f64x2 *>(Li + 16 * h * ld + 8 * s);
            fb[s % (kAhead + 1)][h] = *reinterpret_cast<const f64x2 *>(Lj + 16 * h * ld + 8 * s);
        }
    };
#pragma unroll
    for (int s = 0; s < kAhead; ++s) load(s);
    double old[2][2][4];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) old[p][h][v] = T[(16 * p + 4 * v) * ld + 16 * h];
    f64x4 d[2][2] = {};
#pragma unroll
    for (int s = 0; s < kBatches; ++s) {
        if (s + kAhead < kBatches) load(s + kAhead);
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    d[p][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s % (kAhead + 1)][p][e], fb[s % (kAhead + 1)][h][e],
                                                                   d[p][h], 0, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) T[(16 * p + 4 * v) * ld + 16 * h] = old[p][h][v] - d[p][h][v];
}

// row blockIdx.x of the lower triangle: A += B (the two parts' updates of the
// separator's block)
__global__ __launch_bounds__(256) void k_add_lower(int n, const double *__restrict__ B, long ldb,
                                                  double *__restrict__ A, long lda)
{
    const long r = blockIdx.x;
    for (int c = threadIdx.x; c <= r && c < n; c += 256) A[r * lda + c] += B[r * ldb + c];
}

// ---------------------------------------------------------------------------
// L^-1 by recursive halving.  With the block rows of a group of g tiles
// split in halves, L = [L11 0; L21 L22] and inv(L) = [X11 0; X21 X22] with
//   X21 = -X22 L21 X11,
// where X11 and X22, the inverses of the halves, come from the level below
// (g/2; level 1 is the 32x32 diagonal tile inverses of k_trtri_diag).  L21
// has nonzero tiles only in its top-right nbt x nbt corner (the band), so
//   W   = L21[0:r, n1-c:n1] X11[n1-c:n1, 0:n1]      (r x n1 tiles)
//   X21 = -X22[0:n2, 0:r] W                          (n2 x n1 tiles)
// with n1 = g/2, n2 <= n1 the tiles of the second half, r = min(nbt, n2)
// and c = min(nbt, n1).  The groups of a level are independent: each level
// is two batched products (blockIdx.z = group), so the inverse takes
// 2 ceil(log2 nb) launches instead of a march down nb dependent block rows.
// ---------------------------------------------------------------------------
struct LinvLevel {
    int g, nbt;      // group size in tiles, band in tiles
    int groups;      // groups per diagonal block
    long wstride;    // doubles of W per group
};

// A 32x32 tile of C = alpha A B over K columns of A (a multiple of 32), all
// row-major, 16-byte aligned rows: i0, j0 its first row and column.  The four
// waves take a quarter of K each, as 2 x 2 v_mfma_f64_16x16x4f64 tiles, and meet
// in LDS.  Operands go straight from memory into registers, one batch of eight
// columns ahead: a lane of group g = lane / 16 holds columns 2g and 2g + 1 of
// the eight (one 16-byte load of A; the order of a sum's terms is free as long
// as both operands use the same).  Operand layout of that instruction: A[i][k]
// in lane i + 16k, B[k][j] in lane j + 16k, D[4v + q][j] in element v of lane
// j + 16q.  (64x64 tiles staged through LDS 32 columns at a time had few
// workgroups, two barriers and a round trip per 32 columns: a launch took 12 us
// at 1911 DOFs, 5.1 now; 15 to 30 with the whole of K in one wave.)
typedef double f64x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void dgemm_tile32(const double *__restrict__ A, long lda, const double *__restrict__ B,
                                             long ldb, double *__restrict__ C, long ldc, int i0, int j0, int K,
                                             double alpha)
{
    __shared__ double red[4][NB][NB + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15;
    const int steps = K / 32;  // of 8 columns, per wave
    const int k0 = w * (K / 4) + 2 * (lane >> 4);
    const double *a0 = A + (long)(i0 + i) * lda + k0, *a1 = a0 + 16 * lda;
    const double *b0 = B + (long)k0 * ldb + j0 + i;
    f64x4 d[2][2] = {};
    struct Ops {
        f64x2 a[2];
        double b[2][2];
    } x, y;
    auto load = [&](int s, Ops &o) {
        o.a[0] = *reinterpret_cast<const f64x2 *>(a0 + 8 * s);
        o.a[1] = *reinterpret_cast<const f64x2 *>(a1 + 8 * s);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            o.b[e][0] = b0[(8 * s + e) * ldb];
            o.b[e][1] = b0[(8 * s + e) * ldb + 16];
        }
    };
    auto multiply = [&](const Ops &o) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    d[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[p][e], o.b[e][q], d[p][q], 0, 0, 0);
    };
    load(0, x);
    int s = 0;
    for (; s + 2 < steps; s += 2) {
        load(s + 1, y);
        multiply(x);
        load(s + 2, x);
        multiply(y);
    }
    if (s + 1 < steps) load(s + 1, y);
    multiply(x);
    if (s + 1 < steps) multiply(y);
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[w][16 * p + 4 * v + (lane >> 4)][16 * q + i] = d[p][q][v];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        C[(long)(i0 + r) * ldc + j0 + c] = alpha * ((red[0][r][c] + red[1][r][c]) + (red[2][r][c] + red[3][r][c]));
    }
}

// A^-1 = X^T X, X the inverse of the factor, of a small matrix (kCoarseFull), one
// 32x32 tile per workgroup, in the place of the transpose: a solve is then one
// product instead of two.  Rows of X before the tile's later column are zero,
// rows of the other part and what couples the parts are neither stored nor read:
// the rows of X that count are up to two ranges, one after the other for the four
// waves, which split them as in dgemm_tile32.  Both triangles are formed, the sums
// of (i, j) and (j, i) in the same order: A^-1 is symmetric bit for bit.
__global__ __launch_bounds__(256) void k_inverse_product(CoarseMap m, const double *__restrict__ X,
                                                         double *__restrict__ Out)
{
    __shared__ double red[4][NB][NB + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15;
    const int i0 = blockIdx.y * NB, j0 = blockIdx.x * NB, from = max(i0, j0);
    // rows from .. from + n1 - 1 (none when the columns are of different parts),
    // then the separator's
    int n1 = m.N - from, sep = 0;
    if (m.ps > 0 && from < m.os) {
        const bool same = (i0 < m.o2) == (j0 < m.o2);
        n1 = same ? (from < m.o2 ? m.o2 : m.os) - from : 0;
        sep = m.ps;
    }
    const int steps = (n1 + sep) / 32;  // of 8 rows, per wave
    struct Ops {
        double a[2][2], b[2][2];
    } x, y;
    auto load = [&](int s, Ops &o) {
        const int r = 8 * (w * steps + s);
        const double *p = X + (long)((r < n1 ? from + r : m.os + r - n1) + 2 * (lane >> 4)) * m.N + i;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                o.a[e][h] = p[(long)e * m.N + i0 + 16 * h];
                o.b[e][h] = p[(long)e * m.N + j0 + 16 * h];
            }
    };
    f64x4 d[2][2] = {};
    auto multiply = [&](const Ops &o) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    d[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(o.a[e][p], o.b[e][q], d[p][q], 0, 0, 0);
    };
    load(0, x);
    int s = 0;
    for (; s + 2 < steps; s += 2) {
        load(s + 1, y);
        multiply(x);
        load(s + 2, x);
        multiply(y);
    }
    if (s + 1 < steps) load(s + 1, y);
    multiply(x);
    if (s + 1 < steps) multiply(y);
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[w][16 * p + 4 * v + (lane >> 4)][16 * q + i] = d[p][q][v];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = (tid >> 5) + 8 * u, c = tid & 31;
        Out[(long)(i0 + r) * m.N + j0 + c] = (red[0][r][c] + red[1][r][c]) + (red[2][r][c] + red[3][r][c]);
    }
}

// blockIdx.z: diagonal block x group.  Tiles above the diagonal of X are
// neither read nor written.
template <int STEP>
__global__ __launch_bounds__(256) void k_linv_level(CoarseBlocks B, double *Li, double *W, int N, LinvLevel lv)
{
    const int q = blockIdx.z / lv.groups, z = blockIdx.z - q * lv.groups;
    const int nb = (B.off[q + 1] - B.off[q]) / NB, n1 = lv.g / 2, s = z * lv.g, h = s + n1;
    if (h >= nb) return;
    const int n2 = min(lv.g, nb - s) - n1;
    const int r = min(lv.nbt, n2), c = min(lv.nbt, n1);
    const int ti = blockIdx.y, tj = blockIdx.x;
    if (ti >= (STEP == 0 ? r : n2)) return;
    const double *L = B.L[q];
    const long ldl = B.ld[q];
    double *X = Li + (long)B.off[q] * N + B.off[q];
    double *Wz = W + blockIdx.z * lv.wstride;
    const long ldw = (long)n1 * NB;
    if (STEP == 0) {  // W = L21[0:r, n1-c:n1] X11[n1-c:n1, 0:n1], rows of X11 from tile tj on
        const int k = max(n1 - c, tj);
        dgemm_tile32(L + (long)h * NB * ldl + (long)(s + k) * NB, ldl, X + (long)(s + k) * NB * N + (long)s * NB,
                             N, Wz, ldw, ti * NB, tj * NB, (n1 - k) * NB, 1.0);
    } else {  // X21 = -X22[0:n2, 0:r] W, columns of X22 up to tile ti
        dgemm_tile32(X + (long)h * NB * N + (long)h * NB, N, Wz, ldw, X + (long)h * NB * N + (long)s * NB, N,
                             ti * NB, tj * NB, min(r, ti + 1) * NB, -1.0);
    }
}

// The separator's rows of the inverse, blockIdx.z = part q: W = X_q L_qq^-1
// with X_q the separator's rows of the part's factor (nonzero in the last nbt
// tiles), then -L_ss^-1 W.
template <int STEP>
__global__ __launch_bounds__(256) void k_linv_sep(CoarseBlocks B, double *Li, double *W, int N, int nbt)
{
    const int q = blockIdx.z, o = B.off[q], nq = B.off[q + 1] - o, os = B.off[2], ps = B.off[3] - os;
    const int ti = blockIdx.y, tj = blockIdx.x;
    if (tj * NB >= nq) return;
    double *Wz = W + (long)q * ps * N;
    if (STEP == 0) {
        const int k = max(nq / NB - nbt, tj) * NB;
        dgemm_tile32(B.L[q] + (long)nq * B.ld[q] + k, B.ld[q], Li + (long)(o + k) * N + o, N, Wz, nq, ti * NB,
                             tj * NB, nq - k, 1.0);
    } else {
        dgemm_tile32(Li + (long)os * N + os, N, Wz, nq, Li + (long)os * N + o, N, ti * NB, tj * NB,
                             (ti + 1) * NB, -1.0);
    }
}

// Levels 2, 4, ... of the halving on every diagonal block at once; Li holds
// the diagonal tile inverses, W has room for wcap doubles.
static void launch_linv_levels(hipStream_t s, const CoarseBlocks &B, double *Li, double *W, long wcap, int N, int nbt)
{
    int nb = 0;
    for (int q = 0; q < B.nblk; ++q) nb = std::max(nb, (B.off[q + 1] - B.off[q]) / NB);
    for (int g = 2; g / 2 < nb; g *= 2) {
        const int n1 = g / 2;
        const int groups = (nb - n1 + g - 1) / g;
        const int rmax = std::min(nbt, n1);
        const LinvLevel lv{g, nbt, groups, (long)rmax * NB * n1 * NB};
        if (lv.wstride * groups * B.nblk > wcap) throw std::runtime_error("coarsest inverse: work buffer too small");
        const unsigned tn = (unsigned)n1, tz = (unsigned)(groups * B.nblk);
        k_linv_level<0><<<dim3(tn, (unsigned)rmax, tz), 256, 0, s>>>(B, Li, W, N, lv);
        k_linv_level<1><<<dim3(tn, tn, tz), 256, 0, s>>>(B, Li, W, N, lv);
    }
    if (B.nblk == 3) {
        const int ps = B.off[3] - B.off[2], nq = std::max(B.off[1], B.off[2] - B.off[1]);
        if (2L * ps * N > wcap) throw std::runtime_error("coarsest inverse: work buffer too small");
        const dim3 grid((unsigned)(nq / NB), (unsigned)(ps / NB), 2);
        k_linv_sep<0><<<grid, 256, 0, s>>>(B, Li, W, N, nbt);
        k_linv_sep<1><<<grid, 256, 0, s>>>(B, Li, W, N, nbt);
    }
}

// The split takes one pair of block columns (15.7 us), the sum of the updates (4.7)
// and a last one (8.7) at 5x3x3 nodes already, for two pairs and a last one
// without it; it needs two planes per part.
void coarse_layout(Coarse &C, const Grid &g, bool periodic)
{
    CoarseMap &m = C.map;
    m = CoarseMap();
    m.n = C.n;
    m.p = 3 * g.nny * g.nnz;
    m.nplanes = g.nnx;
    m.rp = 1.0f / (float)m.p;
    auto up = [](int v) { return (v + NB - 1) / NB * NB; };
    const int N1 = up(C.n);
    m.o2 = m.os = m.N = N1;
    if (periodic || g.nnx < 5 || N1 / NB < 4) return;
    m.a = g.nnx / 2;
    const int p1 = m.a * m.p, p2 = (g.nnx - 1 - m.a) * m.p;
    m.o2 = up(p1);
    m.pad1 = m.o2 - p1;
    m.os = m.o2 + up(p2);
    m.pad2 = up(p2) - p2;
    m.ps = up(m.p);
    m.N = m.os + m.ps;
}

std::vector<int> coarse_dofs(const Coarse &C)
{
    std::vector<int> d(C.map.N);
    for (int c = 0; c < C.map.N; ++c) d[c] = coarse_dof(C.map, c);
    return d;
}

CoarseParts coarse_parts(const Coarse &C)
{
    const CoarseMap &m = C.map;
    CoarseParts P{};
    P.np = m.ps ? 2 : 1;
    P.A[0] = C.AQ;
    P.n[0] = m.o2 + m.ps;
    if (m.ps) {
        P.A[1] = C.AQ + (long)P.n[0] * P.n[0];
        P.n[1] = m.os - m.o2 + m.ps;
    }
    // the factor goes to matrices of its own behind these
    const long half = (long)P.n[0] * P.n[0] + (long)P.n[1] * P.n[1];
    for (int q = 0; q < P.np; ++q) P.L[q] = P.A[q] + half;
    return P;
}

long coarse_matrix_len(const Coarse &C)
{
    const CoarseParts P = coarse_parts(C);
    return 2 * ((long)P.n[0] * P.n[0] + (long)P.n[1] * P.n[1]);
}

// Tiles of a step that are resident together: two workgroups per CU (their LDS).
// Up to there both forms take the same time or the one launch less (4x32x32 at two
// levels, 406 tiles: 1.30 ms both; 1029 periodic DOFs, up to 496: 0.64 against 0.68).
constexpr int kCholFit = 512;

static void launch_chol_steps(hipStream_t s, const CholStep &a, int np)
{
    auto blocks = [&](int nt) { return dim3((unsigned)std::max(1, nt * (nt + 1) / 2), (unsigned)np); };
    int last = -1;  // most trailing tiles after an odd last block column
    for (int q = 0; q < np; ++q)
        if (a.steps[q] & 1) last = std::max(last, std::min(a.nt, a.n[q] / NB - a.steps[q]));
    for (int k = 0;; k += 2) {
        int nt = -1;
        for (int q = 0; q < np; ++q)
            if (k + 1 < a.steps[q]) nt = std::max(nt, std::min(a.nt, a.n[q] / NB - k - 2));
        if (nt < 0) break;
        const int n2 = (nt + 1) / 2;
        if (nt * (nt + 1) / 2 * np > kCholFit) {
            k_chol_step2<true><<<dim3((unsigned)nt, (unsigned)np), 256, 0, s>>>(a, k);
            k_chol_update<<<dim3((unsigned)(n2 * (n2 + 1) / 2), (unsigned)np), 256, 0, s>>>(a, k);
        } else {
            k_chol_step2<false><<<blocks(nt), 256, 0, s>>>(a, k);
        }
    }
    if (last >= 0) k_chol_step<<<blocks(last), 256, 0, s>>>(a);
}

void coarse_factor(hipStream_t s0, Coarse &C, bool lag)
{
    C.target = (lag && C.have) ? 1 - C.cur : C.cur;
    C.solve_waits = C.target == C.cur;
    C.Linv = C.Lbuf[C.cur];
    C.LinvT = C.LTbuf[C.cur];
    const int N = C.map.N, ps = C.map.ps;
    // the factor of a banded matrix keeps its band: panel rows and trailing
    // tiles beyond it are exact zeros and are skipped
    const int bw = std::max(1, std::min(C.bw, N));
    hipStream_t s = C.side;
    HIPCHK(hipEventRecord(C.ev_in, s0));
    HIPCHK(hipStreamWaitEvent(s, C.ev_in, 0));
    HIPCHK(hipMemsetAsync(C.flag, 0, sizeof(int), s));
    const CoarseParts P = coarse_parts(C);
    CholStep a{};
    a.flag = C.flag;
    for (int q = 0; q < P.np; ++q) {
        a.A[q] = P.A[q];
        a.L[q] = P.L[q];
        a.ld[q] = a.n[q] = P.n[q];
        a.steps[q] = (P.n[q] - ps) / NB;
    }
    a.nt = (bw + NB - 1) / NB;
    launch_chol_steps(s, a, P.np);
    if (ps) {
        const long l0 = P.n[0] - ps, l1 = P.n[1] - ps;
        a.A[0] += l0 * (P.n[0] + 1);
        a.L[0] += l0 * (P.n[0] + 1);
        k_add_lower<<<ps, 256, 0, s>>>(ps, P.A[1] + l1 * (P.n[1] + 1), P.n[1], a.A[0], P.n[0]);
        a.n[0] = ps;
        a.steps[0] = ps / NB;
        a.nt = ps / NB;  // dense
        launch_chol_steps(s, a, 1);
    }
    HIPCHK(hipGetLastError());
    // the inverse's launches are enqueued by coarse_finish, when the host
    // has enqueued the start of the solve on the main stream
    C.inv_pending = true;
    C.waited = false;
    C.pending = true;
}

void coarse_finish(const Coarse &C)
{
    if (!C.inv_pending) return;
    C.inv_pending = false;
    const CoarseMap &m = C.map;
    const int N = m.N, nb = N / NB;
    const int bw = std::max(1, std::min(C.bw, N));
    double *Li = C.Lbuf[C.target], *LiT = C.LTbuf[C.target];
    hipStream_t s = C.side;
    const CoarseParts P = coarse_parts(C);
    CoarseBlocks B{};
    B.nblk = m.ps ? 3 : 1;
    B.off[0] = 0;
    B.L[0] = P.L[0];
    B.ld[0] = P.n[0];
    B.off[1] = m.ps ? m.o2 : N;
    if (m.ps) {
        B.L[1] = P.L[1];
        B.ld[1] = P.n[1];
        B.off[2] = m.os;
        B.L[2] = P.L[0] + (long)m.o2 * P.n[0] + m.o2;
        B.ld[2] = P.n[0];
        B.off[3] = N;
    }
    k_trtri_diag<<<nb, 64, 0, s>>>(B, Li, N);
    // the last step's buffer is free until then: it holds W
    launch_linv_levels(s, B, Li, LiT, (long)N * N, N, (bw + 2 * NB - 2) / NB);
    if (N <= kCoarseFull)
        k_inverse_product<<<dim3(nb, nb), 256, 0, s>>>(m, Li, LiT);
    else
        k_transpose<<<dim3(nb, nb), 256, 0, s>>>(Li, LiT, N);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(C.ev_done, s));
}

int coarse_check(Coarse &C)
{
    if (!C.pending || !C.solve_waits) return 0;  // a lagged factor is checked when adopted
    coarse_finish(C);
    int flag = 0;
    HIPCHK(hipMemcpyAsync(&flag, C.flag, sizeof(int), hipMemcpyDeviceToHost, C.side));
    HIPCHK(hipStreamSynchronize(C.side));
    C.pending = false;
    C.have = flag == 0;
    return flag ? GPUTO_ERR_NOT_SPD : 0;
}

void coarse_invalidate(Coarse &C)
{
    C.have = false;
    C.invalid = true;
}

void coarse_adopt(Coarse &C)
{
    const bool invalid = C.invalid;
    C.invalid = false;
    if (!C.pending) {
        if (invalid) C.have = false;
        return;
    }
    coarse_finish(C);
    int flag = 0;
    HIPCHK(hipMemcpyAsync(&flag, C.flag, sizeof(int), hipMemcpyDeviceToHost, C.side));
    HIPCHK(hipStreamSynchronize(C.side));  // launched a solve ago: normally finished
    C.pending = false;
    if (flag || invalid) {
        // a failed factor, or one of an earlier configuration: factor
        // again, exactly, at this setup
        C.have = false;
        return;
    }
    C.cur = C.target;
    C.have = true;
}

void coarse_switch(Coarse &C, hipStream_t s)
{
    if (!C.pending || C.solve_waits) return;  // no lagged factorisation in flight
    coarse_finish(C);
    HIPCHK(hipStreamWaitEvent(s, C.ev_done, 0));
    C.waited = true;
    C.cur = C.target;
    C.Linv = C.Lbuf[C.cur];
    C.LinvT = C.LTbuf[C.cur];
    C.solve_waits = true;  // coarse_check reads its SPD flag when the solve ends
}

// ---------------------------------------------------------------------------
// Coarsest solve x = L^-T L^-1 b as two row-parallel triangular products, or
// one with the whole inverse (kCoarseFull), then x[fixed] = 0
// (mgcg1.c:431-432).  One wave per row and, for a batch, all its
// right-hand sides: a row is read once, two entries per load, kTrmvLoads of
// them (and of b) in flight before the first product; the longest rows come
// first.  Rows start and end at whole tiles (the diagonal tiles are stored with
// their zeros).  Rows and columns are in the factor's order (coarse_dof, from a
// table: the arithmetic for every column of a row took 2 to 3 us), the
// right-hand side and the solution in the level's; a row of one part skips the
// other's columns, which halves the bytes.  (A workgroup per row with single
// loads and a sum through LDS: 7.1 + 6.3 us at 1911 DOFs and 10.6 + 8.2 at
// 2880, 5.6 + 5.0 and 8.1 + 6.4 now; six right-hand sides at 1029 DOFs, each with
// its own pass over the matrix: 14 + 13, 13 + 8.7 now.)
// ---------------------------------------------------------------------------
constexpr int kTrmvThreads = 256, kTrmvLoads = 8;

enum TrmvKind { TRMV_LOWER, TRMV_UPPER, TRMV_FULL };

template <TrmvKind KIND, int MAXB, class Ti, class To>
__global__ __launch_bounds__(kTrmvThreads) void k_trmv(CoarseMap m, const int *__restrict__ dof,
                                                      const double *__restrict__ M,
                                                      const Ti *__restrict__ b, To *__restrict__ x,
                                                      const uint8_t *__restrict__ mask, const int *ctl, int nb)
{
    // lower: b has n entries, x has N (the padded y); upper: the reverse; full: both n
    constexpr bool UPPER = KIND == TRMV_UPPER, FULL = KIND == TRMV_FULL, LOWER = KIND == TRMV_LOWER;
    const long sb = UPPER ? m.N : m.n, sx = LOWER ? m.N : m.n;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int idx = blockIdx.x * (kTrmvThreads / 64) + wave;  // < N
    const int row = LOWER ? m.N - 1 - idx : idx;
    // columns lo .. lo + cnt - 1, those from `cut` on shifted by `skip` (the
    // separator's columns of a row of part 1)
    const int tile = row / NB * NB;
    int lo, cnt, cut = m.N, skip = 0;
    if (FULL) {
        lo = 0;
        cnt = m.N;
    } else if (LOWER) {
        lo = m.ps > 0 && row >= m.o2 && row < m.os ? m.o2 : 0;
        cnt = tile + NB - lo;
    } else {
        lo = tile;
        cnt = m.N - tile;
        if (m.ps > 0 && row < m.o2) {
            cut = m.o2;
            skip = m.os - m.o2;
            cnt -= skip;
        }
    }
    const double *__restrict__ Mr = M + (long)row * m.N;
    double s[MAXB];
#pragma unroll
    for (int q = 0; q < MAXB; ++q) s[q] = 0.0;
    for (int t0 = 2 * lane; t0 < cnt; t0 += 128 * kTrmvLoads) {
        f64x2 mv[kTrmvLoads];
        int d0[kTrmvLoads], d1[kTrmvLoads];
#pragma unroll
        for (int u = 0; u < kTrmvLoads; ++u) {
            const int t = t0 + 128 * u;
            int c = lo + (t < cnt ? t : t0);  // in the row
            c += c >= cut ? skip : 0;
            mv[u] = *reinterpret_cast<const f64x2 *>(Mr + c);
            if (t >= cnt) mv[u] = f64x2{0.0, 0.0};
            if (UPPER) {
                d0[u] = c;
                d1[u] = c + 1;
            } else {  // padding: an identity row's entry, times nothing
                const int2 d = *reinterpret_cast<const int2 *>(dof + c);
                d0[u] = d.x;
                d1[u] = d.y;
                if (d0[u] < 0) d0[u] = 0, mv[u][0] = 0.0;
                if (d1[u] < 0) d1[u] = 0, mv[u][1] = 0.0;
            }
        }
        if (MAXB == 1 && ctl && ctl[0]) return;  // converged: read with the loads above
#pragma unroll
        for (int q = 0; q < MAXB; ++q) {
            if (MAXB > 1 && q >= nb) break;
            double bv[kTrmvLoads][2];
#pragma unroll
            for (int u = 0; u < kTrmvLoads; ++u) {
                bv[u][0] = (double)b[q * sb + d0[u]];
                bv[u][1] = (double)b[q * sb + d1[u]];
            }
#pragma unroll
            for (int u = 0; u < kTrmvLoads; ++u) s[q] = fma(mv[u][1], bv[u][1], fma(mv[u][0], bv[u][0], s[q]));
        }
    }
    const int d = LOWER ? row : dof[row];
    const bool fixed = !LOWER && mask && d >= 0 && ((mask[d / 3] >> (d % 3)) & 1u);
#pragma unroll
    for (int q = 0; q < MAXB; ++q) {
        if (MAXB > 1 && q >= nb) break;
        double v = s[q];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        const bool done = ctl && ctl[q * kCtlStride];
        if (lane == 0 && d >= 0 && !done) x[q * sx + d] = (To)(fixed ? 0.0 : v);  // lower, padding rows: 0
    }
}

// The solve is FP64 for both vector types: the right-hand side is widened,
// the result rounded once on output.
template <class T>
void launch_coarse_solve(hipStream_t s, const Coarse &C, const T *b, T *x, const uint8_t *mask, const int *ctl, int nb)
{
    coarse_finish(C);  // also a lagged factorisation's, which runs meanwhile
    if (C.solve_waits && !C.waited) {  // the factorisation of this hierarchy, once per stream order
        HIPCHK(hipStreamWaitEvent(s, C.ev_done, 0));
        C.waited = true;
    }
    // C.y has room for kMaxBatch right-hand sides; N is a multiple of the rows of a workgroup
    const unsigned grid = (unsigned)(C.map.N / (kTrmvThreads / 64));
    auto run = [&](auto maxb) {
        constexpr int MB = decltype(maxb)::value;
        if (C.map.N <= kCoarseFull) {
            k_trmv<TRMV_FULL, MB, T, T><<<grid, kTrmvThreads, 0, s>>>(C.map, C.dof, C.LinvT, b, x, mask, ctl, nb);
            return;
        }
        k_trmv<TRMV_LOWER, MB, T, double><<<grid, kTrmvThreads, 0, s>>>(C.map, C.dof, C.Linv, b, C.y, nullptr, ctl, nb);
        k_trmv<TRMV_UPPER, MB, double, T><<<grid, kTrmvThreads, 0, s>>>(C.map, C.dof, C.LinvT, C.y, x, mask, ctl, nb);
    };
    if (nb > 1)
        run(std::integral_constant<int, kMaxBatch>());
    else
        run(std::integral_constant<int, 1>());
}
template void launch_coarse_solve<double>(hipStream_t, const Coarse &, const double *, double *, const uint8_t *,
                                          const int *, int);
template void launch_coarse_solve<float>(hipStream_t, const Coarse &, const float *, float *, const uint8_t *,
                                         const int *, int);

}  // namespace gputo
