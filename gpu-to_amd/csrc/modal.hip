// Matrix-free hex operators in the element's modal basis: the level-0
// operator of a unit-H8 Ke0 (multAV0c / defect0c, Cantilever/TOP3D125MGCGCUDA/
// mgcg1.cu:941-997,1208-1264), the same operator on every level of the mgcg9
// engine, and the rediscretised level-1 operator of the REF_C hierarchy
// (coarseAe2c applied with defectc, mgcg1.cu:2042-2070,1266-1324) from the
// child densities.
//
// Modal basis.  Along each direction a node pair (u0, u1) becomes the sum
// u0 + u1 (index 0) and the difference u1 - u0 (index 1); the 8 values of one
// displacement component become 8 modes m(a, b, c).  The three reflections of
// the cube leave an isotropic element unchanged, so its matrix couples only
// modes of equal parity, and the 24 x 24 products shrink to 33 operations:
//   m(1,0,0) of u, m(0,1,0) of v, m(0,0,1) of w   normal strains (full 3 x 3)
//   u(0,1,0) + v(1,0,0) and its two rotations      shears (rank one)
//   v(1,1,0), w(1,0,1) and their two rotations     bending pairs (2 x 2)
//   u(0,1,1), v(1,0,1), w(1,1,0)                   twist (full 3 x 3)
//   u(1,1,1), v(1,1,1), w(1,1,1)                   one value each
// and the three translations to nothing.  Sums and differences are formed
// once per node pair along j, once per face along k and i.  Per element that
// is about 190 operations in place of 576 multiply-adds, and the differences
// are taken between neighbouring nodes first, so a smooth field loses no
// digits in the products.  The level-1 operator uses the same basis: the
// displacement gradient at the 2 x 2 x 2 Gauss points is a sum and difference
// transform of the modes again (a derivative along x does not depend on x).
//
// Work of a block.  The nodes of a plane i = const are cut into strips of W
// nodes along j; the strip's rows follow each other in one list of R = W + 1
// columns each (column c holds element column and node j0 - 1 + c), and a
// block owns M consecutive entries of that list and TI node layers.  Entry t
// of a block is thread column t; element t reaches nodes t, t + 1, t + R and
// t + R + 1, so the block works on R + 1 entries before its own, too.  It
// marches along i, one element layer per step:
//   * each lane loads the node pairs (k, j..j+1) and (k+1, j..j+1) of the next
//     layer (48 contiguous bytes each in FP64) while it works on this one (as
//     few loads as possible: an FP32 pair as three 8-byte loads instead of a
//     16-byte and an 8-byte one made mixed solves 3 % slower);
//   * sums and differences along j, k and i, the modal products, and back:
//     the i direction meets in the lane's registers;
//   * along j the neighbour's share comes by a one-lane shift (consecutive
//     waves overlap by one entry, so no lane lacks its neighbour);
//   * along k it goes through LDS, R entries further, one barrier per layer
//     (two buffers).
// No atomics and one fixed order of every sum: results are bitwise
// deterministic.  Elements outside the mesh take loads past the buffer's
// range, which return 0, so nothing of a neighbouring row enters a sum.
//
// Periodic cells (PER).  An iterate is equal on a master node and its images,
// a residual lives on the masters and is 0 on the images.  The list's entries
// before the first column, row and layer hold the last elements of their row
// instead of none, a block owns masters only, and the epilogue writes the
// images too: the whole periodic row, its Jacobi update and both node copies
// come from one launch.  (The operator without the wrap, then a pass that
// folds the images into the masters, updates and copies back, took 22.9 +
// 10.4 us per level-0 sweep of six right-hand sides at 48x48x48; 25.8 us now.)
//
// Measured on MI355X at 192x96x96 (matvecs back to back; before: node-gather,
// split-BF16 MFMA and Gauss point by Gauss point kernels): FP64 level 0
// 75 -> 27.4 us (101 MB of operands, 3.7 TB/s; 87 % of the VALU operations are
// the transforms and products above), FP32 level 0 66 (node-gather) and 23
// (MFMA) -> 17.1 us, FP64 level 1 34 -> 12.4 us, FP32 level 1 24 -> 8.8 us;
// an FP64 Jacobi sweep in the solve 65 -> 37 us, an FP32 one 34 (MFMA) ->
// 25 us.  At 16x8x8 a launch takes 3.5 us against 8-10 us: 27 x 24 dependent
// products per node are gone.  Level 0 is bound by memory and by the two
// waves per SIMD that cover its latency.
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>

#include "vcycle.h"

namespace gputo {

namespace {

typedef float f32x2m __attribute__((ext_vector_type(2)));
typedef float f32x4m __attribute__((ext_vector_type(4)));
typedef double f64x2m __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t MdBuf;

constexpr int kMdOut = 0x7f000000;  // a byte offset past every buffer (vectors are below it)

__device__ __forceinline__ MdBuf md_buf(const void *p, long bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ f64x2m md_ld2d(MdBuf b, int off, int soff)
{
    return __builtin_bit_cast(f64x2m, __builtin_amdgcn_raw_buffer_load_b128(b, off, soff, 0));
}
__device__ __forceinline__ f32x4m md_ld4f(MdBuf b, int off, int soff)
{
    return __builtin_bit_cast(f32x4m, __builtin_amdgcn_raw_buffer_load_b128(b, off, soff, 0));
}
__device__ __forceinline__ f32x2m md_ld2f(MdBuf b, int off, int soff)
{
    return __builtin_bit_cast(f32x2m, __builtin_amdgcn_raw_buffer_load_b64(b, off, soff, 0));
}
template <class T>
__device__ __forceinline__ T md_ld1(MdBuf b, int off, int soff);
template <>
__device__ __forceinline__ double md_ld1<double>(MdBuf b, int off, int soff)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, off, soff, 0));
}
template <>
__device__ __forceinline__ float md_ld1<float>(MdBuf b, int off, int soff)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(b, off, soff, 0));
}

// six consecutive values: a node pair along j
__device__ __forceinline__ void md_ld6(MdBuf b, int off, int soff, double (&v)[6])
{
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const f64x2m x = md_ld2d(b, off + 16 * q, soff);
        v[2 * q] = x[0];
        v[2 * q + 1] = x[1];
    }
}
__device__ __forceinline__ void md_ld6(MdBuf b, int off, int soff, float (&v)[6])
{
    const f32x4m x = md_ld4f(b, off, soff);
    const f32x2m y = md_ld2f(b, off + 16, soff);
    v[0] = x[0];
    v[1] = x[1];
    v[2] = x[2];
    v[3] = x[3];
    v[4] = y[0];
    v[5] = y[1];
}
// two consecutive values
__device__ __forceinline__ void md_ld2(MdBuf b, int off, int soff, double (&v)[2])
{
    const f64x2m x = md_ld2d(b, off, soff);
    v[0] = x[0];
    v[1] = x[1];
}
__device__ __forceinline__ void md_ld2(MdBuf b, int off, int soff, float (&v)[2])
{
    const f32x2m x = md_ld2f(b, off, soff);
    v[0] = x[0];
    v[1] = x[1];
}
// three consecutive values: one node
__device__ __forceinline__ void md_ld3(MdBuf b, int off, int soff, double (&v)[3])
{
    const f64x2m x = md_ld2d(b, off, soff);
    v[0] = x[0];
    v[1] = x[1];
    v[2] = md_ld1<double>(b, off + 16, soff);
}
__device__ __forceinline__ void md_ld3(MdBuf b, int off, int soff, float (&v)[3])
{
    const f32x2m x = md_ld2f(b, off, soff);
    v[0] = x[0];
    v[1] = x[1];
    v[2] = md_ld1<float>(b, off + 8, soff);
}

// the value of the lane below (lane 0: 0), a DPP wave shift
__device__ __forceinline__ float md_below(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ double md_below(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, 0x138, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), 0x138, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Values of one node layer at an element column: [component][b][d], b the
// mode along j, d the mode along k.
template <class T>
struct Jk {
    T v[3][2][2];
};

template <class T>
__device__ __forceinline__ void md_jk(const T (&lo)[6], const T (&hi)[6], Jk<T> &o)
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const T s0 = lo[c] + lo[3 + c], d0 = lo[3 + c] - lo[c];
        const T s1 = hi[c] + hi[3 + c], d1 = hi[3 + c] - hi[c];
        o.v[c][0][0] = s0 + s1;
        o.v[c][0][1] = s1 - s0;
        o.v[c][1][0] = d0 + d1;
        o.v[c][1][1] = d1 - d0;
    }
}

// Modes m[c][a][b][d] (a along i) to modal forces in place, one scale E for
// the element (C: the 8 modal constants of Ke0, md_constants).
template <class T>
__device__ __forceinline__ void md_element(T (&m)[3][2][2][2], const T *C, T E)
{
    {
        const T t = (C[1] * E) * (m[0][1][0][0] + m[1][0][1][0] + m[2][0][0][1]);
        const T c0 = C[0] * E;
        m[0][1][0][0] = fma(c0, m[0][1][0][0], t);
        m[1][0][1][0] = fma(c0, m[1][0][1][0], t);
        m[2][0][0][1] = fma(c0, m[2][0][0][1], t);
    }
    {
        const T c2 = C[2] * E;
        m[0][0][1][0] = m[1][1][0][0] = c2 * (m[0][0][1][0] + m[1][1][0][0]);
        m[1][0][0][1] = m[2][0][1][0] = c2 * (m[1][0][0][1] + m[2][0][1][0]);
        m[0][0][0][1] = m[2][1][0][0] = c2 * (m[0][0][0][1] + m[2][1][0][0]);
    }
    {
        const T c3 = C[3] * E;
#pragma unroll
        for (int c = 0; c < 3; ++c) m[c][1][1][1] *= c3;
    }
    {
        const T c4 = C[4] * E, c5 = C[5] * E;
        T p, q;
        p = m[1][1][1][0], q = m[2][1][0][1];
        m[1][1][1][0] = fma(c4, p, c5 * q);
        m[2][1][0][1] = fma(c4, q, c5 * p);
        p = m[0][1][1][0], q = m[2][0][1][1];
        m[0][1][1][0] = fma(c4, p, c5 * q);
        m[2][0][1][1] = fma(c4, q, c5 * p);
        p = m[0][1][0][1], q = m[1][0][1][1];
        m[0][1][0][1] = fma(c4, p, c5 * q);
        m[1][0][1][1] = fma(c4, q, c5 * p);
    }
    {
        const T t = (C[7] * E) * (m[0][0][1][1] + m[1][1][0][1] + m[2][1][1][0]);
        const T c6 = C[6] * E;
        m[0][0][1][1] = fma(c6, m[0][0][1][1], t);
        m[1][1][0][1] = fma(c6, m[1][1][0][1], t);
        m[2][1][1][0] = fma(c6, m[2][1][1][0], t);
    }
}

// Sum and difference transform of four values over two directions.
template <class T>
__device__ __forceinline__ void md_had4(T (&g)[2][2])
{
    const T a = g[0][0] + g[1][0], b = g[0][1] + g[1][1], c = g[0][0] - g[1][0], d = g[0][1] - g[1][1];
    g[0][0] = a + b;
    g[0][1] = a - b;
    g[1][0] = c + d;
    g[1][1] = c - d;
}

// The same with one scale per Gauss point (the level-1 operator: the scale
// of the child at that point), cx[sx][sy][sz], s = 1 the point at +1/sqrt3.
// C[0] = lam, C[1] = 2 mu, C[2] = mu, each times the 1/64 of the two
// transforms; C[3] = 1/sqrt3.  A mode of order n enters its derivatives with
// (1/sqrt3)^(n - 1) and its force collects them with the same weight.
template <class T>
__device__ __forceinline__ void md_element_gp(T (&m)[3][2][2][2], const T *C, const T (&cx)[2][2][2])
{
    const T g1 = C[3], g2 = C[3] * C[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        m[c][1][1][0] *= g1;
        m[c][1][0][1] *= g1;
        m[c][0][1][1] *= g1;
        m[c][1][1][1] *= g2;
    }
    // gradients G[c][x] at (sy, sz), G[c][y] at (sx, sz), G[c][z] at (sx, sy);
    // index 0 of a transform's result is the point at +1/sqrt3
    T gx[3][2][2], gy[3][2][2], gz[3][2][2];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                gx[c][p][q] = m[c][1][p][q];
                gy[c][p][q] = m[c][p][1][q];
                gz[c][p][q] = m[c][p][q][1];
            }
        md_had4(gx[c]);
        md_had4(gy[c]);
        md_had4(gz[c]);
    }
    // stresses, summed over the direction of the test function's derivative
    T px[3][2][2], py[3][2][2], pz[3][2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int z = 0; z < 2; ++z) {
                const T e = cx[1 - x][1 - y][1 - z];
                const T exx = gx[0][y][z], eyy = gy[1][x][z], ezz = gz[2][x][y];
                const T t = (C[0] * e) * (exx + eyy + ezz);
                const T c2 = C[1] * e, cm = C[2] * e;
                const T sxx = fma(c2, exx, t), syy = fma(c2, eyy, t), szz = fma(c2, ezz, t);
                const T sxy = cm * (gy[0][x][z] + gx[1][y][z]);
                const T syz = cm * (gz[1][x][y] + gy[2][x][z]);
                const T szx = cm * (gx[2][y][z] + gz[0][x][y]);
                const T sx[3] = {sxx, sxy, szx}, sy[3] = {sxy, syy, syz}, sz[3] = {szx, syz, szz};
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    px[c][y][z] = x == 0 ? sx[c] : px[c][y][z] + sx[c];
                    py[c][x][z] = y == 0 ? sy[c] : py[c][x][z] + sy[c];
                    pz[c][x][y] = z == 0 ? sz[c] : pz[c][x][y] + sz[c];
                }
            }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        md_had4(px[c]);
        md_had4(py[c]);
        md_had4(pz[c]);
        m[c][1][0][0] = px[c][0][0];
        m[c][0][1][0] = py[c][0][0];
        m[c][0][0][1] = pz[c][0][0];
        m[c][1][1][0] = g1 * (px[c][1][0] + py[c][1][0]);
        m[c][1][0][1] = g1 * (px[c][0][1] + pz[c][1][0]);
        m[c][0][1][1] = g1 * (py[c][0][1] + pz[c][0][1]);
        m[c][1][1][1] = g2 * (px[c][1][1] + py[c][1][1] + pz[c][1][1]);
    }
}

// P Uc at the 4 nodes (k, j), (k, j + 1), (k + 1, j), (k + 1, j + 1) of a node
// layer, added to the node rows lo and hi; fixed DOFs become 0.  The nodes of a
// fine element lie in one coarse element: c holds its node pairs along j, rows
// K and K + 1 (K = k / 2), already averaged over the coarse layers; ko, jo: k,
// j odd; m: the nodes' fixed bits.
template <class T>
__device__ __forceinline__ void md_prolong(const T (&c)[2][6], bool ko, bool jo, const unsigned (&m)[4], T (&lo)[6],
                                          T (&hi)[6])
{
    const T h = T(0.5);
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        // rows k and k + 1 at the coarse columns
        const T m0 = h * (c[0][x] + c[1][x]), m1 = h * (c[0][3 + x] + c[1][3 + x]);
        const T l0 = ko ? m0 : c[0][x], l1 = ko ? m1 : c[0][3 + x];
        const T h0 = ko ? c[1][x] : m0, h1 = ko ? c[1][3 + x] : m1;
        const T lm = h * (l0 + l1), hm = h * (h0 + h1);
        lo[x] = (m[0] >> x) & 1u ? T(0) : lo[x] + (jo ? lm : l0);
        lo[3 + x] = (m[1] >> x) & 1u ? T(0) : lo[3 + x] + (jo ? l1 : lm);
        hi[x] = (m[2] >> x) & 1u ? T(0) : hi[x] + (jo ? hm : h0);
        hi[3 + x] = (m[3] >> x) & 1u ? T(0) : hi[3 + x] + (jo ? h1 : hm);
    }
}

// Element scales of one element layer at a column: one (level 0) or one per
// child (level 1).
template <class T, int EL>
struct MdScale {
    T e[EL == 0 ? 1 : 8];
};

// Waves per SIMD that the registers allow.  A lane holds the modes of the
// previous layer, of this one and the pending sums (36 values), the next
// layer's operands (13) and the epilogue's (10): 202-212 registers in FP64
// and 108-118 in FP32 at level 0; the Gauss points of level 1 add up to 72
// values, and FP64 takes the whole register file with one wave per SIMD
// (12.4 us per matvec at 192x96x96; 21.0 us with two waves and 80-230 bytes
// of scratch per lane).
template <class T, int EL>
constexpr int md_min_waves()
{
    return sizeof(T) == 8 ? (EL == 0 ? 2 : 1) : (EL == 0 ? 4 : 3);
}

// Whether a launch may carry the PCG's residual test: the prerelaxed modes, which
// start a V-cycle.  (The FP32 cycle of a mixed solve starts with a plain sweep;
// with the test in that kernel too its solves were 1 to 1.5 % slower.)  The
// test goes first, and seven idle blocks behind it keep the tiles on their XCDs.
// The other blocks of such a launch do not look at the flag, which it may set
// while they run: waves of one block could see different values and part at a
// barrier.  What they write once it is set is not read any more.
constexpr unsigned kMdTestBlocks = 8;
template <int MODE, int EL, bool PER>
constexpr bool md_tests()
{
    return EL == 0 && !PER && (MODE == OP_PRE_JACOBI || MODE == OP_PRE_DEFECT);
}
struct MdNoTest {};
template <int MODE, int EL, bool PER>
using MdTest = std::conditional_t<md_tests<MODE, EL, PER>(), CgTest, MdNoTest>;

// waves of a block at most
template <class T, int EL>
constexpr int md_max_waves()
{
    return sizeof(T) == 8 && EL == 1 ? 4 : kMdMaxWaves;
}

template <class T, class TU, int MODE, int EL, bool PER>
__global__ __launch_bounds__((md_max_waves<T, EL>() * 64)) __attribute__((amdgpu_waves_per_eu(md_min_waves<T, EL>())))
void k_modal(OpModal<T> a, const T *__restrict__ CX, MdTest<MODE, EL, PER> test)
{
    const ModalWork &w = a.mw;
    constexpr bool PRE = MODE == OP_PRE_JACOBI || MODE == OP_PRE_DEFECT;
    constexpr bool JAC = MODE == OP_JACOBI || MODE == OP_PRE_JACOBI;
    constexpr bool MV = MODE == OP_MATVEC || MODE == OP_MATVEC_UF;
    // fused dots: of a matvec u.(K u), of a sweep F.(its result)
    constexpr bool DOT = MV || (MODE == OP_JACOBI && EL == 0 && sizeof(T) == 8);
    // the next layer's operands are loaded a layer ahead where the registers
    // allow it
    constexpr bool AHEAD = sizeof(T) == 4 ? !PRE : (EL == 0 && !PRE);
    constexpr int SU = (int)sizeof(TU), S = (int)sizeof(T);
    unsigned bx = blockIdx.x;
    bool tested = false;  // the launch sets the flag
    if constexpr (md_tests<MODE, EL, PER>()) {
        if (test.sc) {
            tested = true;
            if (bx < kMdTestBlocks) {
                if (bx == 0 && threadIdx.x < 64) cg_test(test);
                return;
            }
            bx -= kMdTestBlocks;
        }
    }
    batch_shift(a);
    if (MODE == OP_MATVEC_UF) a.Uf = batch_ptr(a.Uf, a.g.ndof);
    extern __shared__ double md_lds[];
    T *ex = reinterpret_cast<T *>(md_lds);  // [2][3][ne]
    const int ne = 63 * w.NW + 1;
    const Grid &g = a.g;
    const unsigned nb = (unsigned)w.blocks();
    const unsigned tb = (unsigned)xcd_tile(bx, nb);
    if (tb >= nb) {  // padding block of the XCD order
        if (a.partials && threadIdx.x == 0) a.partials[bx] = 0.0;
        return;
    }
    const int ch = (int)(tb % (unsigned)w.nch);
    const unsigned r1 = tb / (unsigned)w.nch;
    const int s = (int)(r1 % (unsigned)w.ns), ib = (int)(r1 / (unsigned)w.ns);
    // owned node layers (PER: masters only)
    const int i0 = ib * w.TI, i1 = min(i0 + w.TI, PER ? g.nx : g.nnx);
    if (PER && i0 >= i1) {
        if (a.partials && threadIdx.x == 0) a.partials[bx] = 0.0;
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = wave * 63 + lane;  // the block's entry (a wave's last is the next one's first)
    // list entry q = ch M - (R + 1) + t -> row k, column c
    const unsigned qs = (unsigned)(ch * w.M + t + w.R - 1);  // q + 2R >= 0
    const int kq = (int)(qs / (unsigned)w.R), c = (int)(qs - (unsigned)(kq * w.R));
    const int k = kq - 2, j = s * w.W - 1 + c;
    // the entry's element; PER: element -1 is the last one of its row
    const int ke = PER && k == -1 ? g.nz - 1 : k, je = PER && j == -1 ? g.ny - 1 : j;
    const bool el_ok = ke >= 0 && ke < g.nz && je >= 0 && je < g.ny;
    const bool own = lane > 0 && t > w.R && t <= w.R + w.M && c > 0 && k >= 0 && k < (PER ? g.nz : g.nnz) &&
                     j < (PER ? g.ny : g.nny);
    const int plane = g.nny * g.nnz;
    const int nod0 = k * g.nny + j;    // own node in its plane
    // A sweep's and a matvec's own value comes with the operands: the pair of row k
    // holds the own node, also where no element follows it along k or j (there as
    // its second node).  Two loads less per layer: the no-allocation matvec at
    // 192x96x96 40.1 -> 37.4 us, an FP64 solve 1 % and a mixed one 1.7 % faster.
    constexpr bool OWN = !PRE && MODE != OP_DEFECT;
    const bool nod_ok = el_ok || (OWN && own), jlast = OWN && own && j == g.ny;
    const int enod = ke * g.nny + je - (int)jlast;  // the element's first node
    // byte offsets in a plane of the element's two node rows, of its scale(s)
    // and of the own node
    const int ulo = nod_ok ? 3 * SU * enod : kMdOut, uhi = el_ok ? 3 * SU * (enod + g.nny) : kMdOut;
    const int flo = el_ok ? 3 * S * enod : kMdOut, fhi = el_ok ? 3 * S * (enod + g.nny) : kMdOut;
    const int eo = el_ok ? (EL == 0 ? S * (ke * g.ny + je) : S * (4 * ke * g.ny + 2 * je)) : kMdOut;
    const int oo = own ? 3 * S * nod0 : kMdOut;
    const long vb = (long)S * g.ndof;
    const MdBuf BU = PRE ? md_buf(a.F, vb)
                         : (MODE == OP_MATVEC_UF ? md_buf(a.Uf, (long)SU * g.ndof) : md_buf(a.U, vb));
    const MdBuf BF = md_buf(a.F, MV ? 0 : vb), BD = md_buf(a.RD, (JAC || PRE) ? (EL == 0 ? vb / 3 : vb) : 0);
    const MdBuf BE = md_buf(CX, (long)S * (EL == 0 ? 1 : 8) * g.nel), BM = md_buf(a.mask, a.mask ? g.nnod : 0);  // no mask: reads 0
    const int up = 3 * SU * plane, fp = 3 * S * plane;         // bytes of a node layer
    const int dp = S * plane, dlo = el_ok ? S * enod : kMdOut, dhi = el_ok ? S * (enod + g.nny) : kMdOut;
    const int ep = (EL == 0 ? 1 : 4) * S * g.ny * g.nz;        // bytes of a scale layer
    const T pr = T(a.prerelax), om = T(a.omega);

    struct Raw {
        TU lo[6], hi[6];
        T dlo[EL == 0 ? 2 : 6], dhi[EL == 0 ? 2 : 6];  // PRE: 1/AD of the same nodes
    };
    auto load = [&](int pl, Raw &x) {
        md_ld6(BU, PRE ? flo : ulo, pl * (PRE ? fp : up), x.lo);
        md_ld6(BU, PRE ? fhi : uhi, pl * (PRE ? fp : up), x.hi);
        if constexpr (PRE && EL == 0) {
            md_ld2(BD, dlo, pl * dp, x.dlo);
            md_ld2(BD, dhi, pl * dp, x.dhi);
        } else if constexpr (PRE) {
            md_ld6(BD, flo, pl * fp, x.dlo);
            md_ld6(BD, fhi, pl * fp, x.dhi);
        }
    };
    auto load_e = [&](int ie, MdScale<T, EL> &x) {
        if (EL == 0) {
            x.e[0] = md_ld1<T>(BE, eo, ie * ep);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // children (is, iz): the pair along j
                const int off = eo + (q & 1) * 2 * S * g.ny, soff = (2 * ie + (q >> 1)) * ep;
                if (S == 8) {
                    const f64x2m v = md_ld2d(BE, off, soff);
                    x.e[2 * q] = (T)v[0];
                    x.e[2 * q + 1] = (T)v[1];
                } else {
                    const f32x2m v = md_ld2f(BE, off, soff);
                    x.e[2 * q] = (T)v[0];
                    x.e[2 * q + 1] = (T)v[1];
                }
            }
        }
    };
    T own_u[3] = {T(0), T(0), T(0)};  // OWN: the own node of the layer last transformed
    auto jk = [&](const Raw &x, Jk<T> &o) {
        T lo[6], hi[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            lo[q] = PRE ? pr * (T(x.lo[q]) * x.dlo[EL == 0 ? q / 3 : q]) : T(x.lo[q]);
            hi[q] = PRE ? pr * (T(x.hi[q]) * x.dhi[EL == 0 ? q / 3 : q]) : T(x.hi[q]);
        }
        if (OWN) {
#pragma unroll
            for (int q = 0; q < 3; ++q) own_u[q] = jlast ? lo[3 + q] : lo[q];
        }
        md_jk(lo, hi, o);
    };

    double part = 0.0;
    // node layer pl is complete in sum: the k and j directions, the
    // neighbours' shares and the epilogue
    struct Epi {
        T f[3], d[3], u[3];
        unsigned m;
    };
    auto load_epi = [&](int pl, Epi &e) {
        e.m = __builtin_amdgcn_raw_buffer_load_b8(BM, own ? nod0 : kMdOut, pl * plane, 0);
        if (!MV) md_ld3(BF, oo, pl * fp, e.f);
        if constexpr (EL == 0) {
            if (JAC || PRE) e.d[0] = e.d[1] = e.d[2] = md_ld1<T>(BD, own ? S * nod0 : kMdOut, pl * dp);
        } else {
            if (JAC || PRE) md_ld3(BD, oo, pl * fp, e.d);
        }
    };
    auto finish = [&](int pl, const Jk<T> &sum, const Epi &e) {
        T y[3];
        T *buf = ex + (pl & 1) * 3 * ne;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            const T l0 = sum.v[cc][0][0] - sum.v[cc][0][1], l1 = sum.v[cc][1][0] - sum.v[cc][1][1];  // row k
            const T h0 = sum.v[cc][0][0] + sum.v[cc][0][1], h1 = sum.v[cc][1][0] + sum.v[cc][1][1];  // row k + 1
            y[cc] = (l0 - l1) + md_below(l0 + l1);
            const T yh = (h0 - h1) + md_below(h0 + h1);
            if (lane > 0) buf[cc * ne + t] = yh;
        }
        __syncthreads();
        if (!own) return;
        const long dof = 3 * ((long)pl * plane + nod0);
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            const T yc = y[cc] + buf[cc * ne + t - w.R];
            const bool fixed = (e.m >> cc) & 1u;
            T v;
            if (MV) {
                v = fixed ? T(0) : yc;
                part += (double)e.u[cc] * (double)v;
            } else if (!JAC) {
                v = fixed ? T(0) : e.f[cc] - yc;
                if (PRE) a.out2[dof + cc] = pr * (e.f[cc] * e.d[cc]);
            } else {
                // U = (1-w) U + w (R + AD U)/AD = U + w R/AD  (mgcg1.cu:1199-1206)
                const T u = PRE ? pr * (e.f[cc] * e.d[cc]) : e.u[cc];
                const T rv = fixed ? T(0) : e.f[cc] - yc;
                v = fma(om * e.d[cc], rv, u);
                if (DOT) part += (double)e.f[cc] * (double)v;
            }
            a.out[dof + cc] = v;
            if (PER) {
                // the images: an iterate's value, 0 for a residual
                const bool bi = pl == 0, bk = k == 0, bj = j == 0;
                if (bi || bk || bj) {
                    const T im = JAC ? v : T(0);
                    const long di = 3L * plane * g.nx, dk = 3L * g.nny * g.nz, dj = 3L * g.ny;
#pragma unroll
                    for (int q = 1; q < 8; ++q)
                        if ((!(q & 4) || bi) && (!(q & 2) || bk) && (!(q & 1) || bj))
                            a.out[dof + cc + (q & 4 ? di : 0) + (q & 2 ? dk : 0) + (q & 1 ? dj : 0)] = im;
                }
            }
        }
    };

    // node layers read (PER: layer -1 is layer nx - 1)
    const int lo = PER ? i0 - 1 : max(i0 - 1, 0), hi = min(i1, g.nnx - 1), first = PER && i0 == 0 ? g.nx - 1 : lo;
    Raw xa, xb;
    MdScale<T, EL> ea, eb;
    load(first, xa);
    load(lo + 1, xb);
    load_e(first, ea);
    if (!tested && a.ctl && a.ctl[0]) return;  // converged: read with the loads above
    Jk<T> pa, pb, pend;
    jk(xa, pa);
#pragma unroll
    for (int cc = 0; cc < 3; ++cc)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int d = 0; d < 2; ++d) pend.v[cc][b][d] = T(0);
    // element layer ie = pl - 1 between node layers pl - 1 (modes in prev) and
    // pl (raw values in x, modes to cur); its loads for the next layer go to
    // xn, en.  Node layer pl - 1 is complete after it.
    auto step = [&](int pl, const Jk<T> &prev, Jk<T> &cur, Raw &x, Raw &xn, MdScale<T, EL> &e,
                    MdScale<T, EL> &en) {
        const bool emit = pl - 1 >= i0;
        // loads complete in order for the wait counter: the epilogue's
        // operands go before the prefetch
        Epi epi;
        if (emit && AHEAD) load_epi(pl - 1, epi);
        const T below_u[3] = {own_u[0], own_u[1], own_u[2]};  // of layer pl - 1
        if (AHEAD) {
            if (pl < hi) {
                load(pl + 1, xn);
                load_e(pl, en);
            }
        } else if (pl > lo + 1) {
            load(pl, x);
            load_e(pl - 1, e);
        }
        jk(x, cur);
        T m[3][2][2][2];
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    m[cc][0][b][d] = prev.v[cc][b][d] + cur.v[cc][b][d];
                    m[cc][1][b][d] = cur.v[cc][b][d] - prev.v[cc][b][d];
                }
        if constexpr (EL == 0) {
            T E = e.e[0];
            if (a.cx_floor > 0.0 && E < T(a.cx_floor)) E = T(0);  // mgcg9 defect0c skip
            md_element(m, a.mc, E);
        } else {
            const T cx[2][2][2] = {{{e.e[0], e.e[2]}, {e.e[1], e.e[3]}}, {{e.e[4], e.e[6]}, {e.e[5], e.e[7]}}};
            md_element_gp(m, a.mc, cx);
        }
        if (emit && !AHEAD) load_epi(pl - 1, epi);
        if (OWN) {
#pragma unroll
            for (int cc = 0; cc < 3; ++cc) epi.u[cc] = below_u[cc];
        }
        Jk<T> sum;
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const T r1v = m[cc][1][b][d];
                    if (b == 0 && d == 0) {  // no force from a translation
                        sum.v[cc][b][d] = pend.v[cc][b][d] - r1v;
                        pend.v[cc][b][d] = r1v;
                    } else {
                        const T r0v = m[cc][0][b][d];
                        sum.v[cc][b][d] = pend.v[cc][b][d] + (r0v - r1v);
                        pend.v[cc][b][d] = r0v + r1v;
                    }
                }
        if (emit) finish(pl - 1, sum, epi);
    };
    for (int pl = lo + 1; pl <= hi; pl += 2) {
        step(pl, pa, pb, xb, AHEAD ? xa : xb, ea, AHEAD ? eb : ea);
        if (pl + 1 <= hi) step(pl + 1, pb, pa, AHEAD ? xa : xb, xb, AHEAD ? eb : ea, ea);
    }
    if (!PER && i1 == g.nnx) {  // the last node layer of the mesh ends with what is pending
        Epi epi;
        load_epi(g.nnx - 1, epi);
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) epi.u[cc] = own_u[cc];
        finish(g.nnx - 1, pend, epi);
    }
    if (DOT && a.partials) {
        // fixed butterfly per wave, then the waves in order
        __shared__ double ws[kMdMaxWaves];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
        if (lane == 0) ws[wave] = part;
        __syncthreads();
        if (threadIdx.x == 0) {
            double v = 0.0;
            for (int q = 0; q < w.NW; ++q) v += ws[q];
            a.partials[bx] = v;
        }
    }
}

// The level-1 operator on small meshes: one group of NW waves per element
// layer, TI + 1 of them, where a march of TI + 1 layers takes as many layer
// times (about 0.9 us each, the Gauss points of one element in one lane).
// Group q owns element layer i0 - 1 + q and, from the second on, finishes the
// node layer below it: its own share of row k stays in registers, its share of
// row k + 1 and both of the group below's come through LDS, one barrier in all.
// It holds one layer's modes (160-172 registers in FP64, 78-86 in FP32).
// A sweep in the solve at 225 nodes FP64 4.9 -> 4.4 us, 4225 nodes 5.3 -> 4.6,
// 15625 nodes of six right-hand sides (periodic) 15.5 -> 13.1, 30625 nodes FP32
// 5.2 -> 4.7 us.  Level 0's layer is a third of that: no gain at any size.
// OP_INTERP_JACOBI: a group reads its coarse element with the rest and adds the
// correction to its 8 nodes, 5.8-6.0 us where the interpolation (3.1) and the
// sweep took 7.7 (225 to 4225 nodes FP64).  A march would wait for the coarse
// nodes in every layer: its level-0 sweep went from 35 to 64 us at 192x96x96 and
// from 4.8 to 8.4 at 48x24x24, more than the interpolation.
constexpr int kMdFlatWaves = 8;

template <class T, int MODE, bool PER>
__global__ __launch_bounds__(kMdFlatWaves * 64) void k_modal_flat(OpModal<T> a, const T *__restrict__ CX)
{
    const ModalWork &w = a.mw;
    constexpr bool PRE = MODE == OP_PRE_JACOBI || MODE == OP_PRE_DEFECT;
    constexpr bool INT = MODE == OP_INTERP_JACOBI;
    constexpr bool JAC = MODE == OP_JACOBI || MODE == OP_PRE_JACOBI || INT;
    constexpr bool MV = MODE == OP_MATVEC;
    constexpr int S = (int)sizeof(T);
    batch_shift(a);
    extern __shared__ double md_lds[];
    const int ne = 63 * w.NW + 1;
    const Grid &g = a.g;
    const unsigned nb = (unsigned)w.blocks();
    const unsigned tb = (unsigned)xcd_tile(blockIdx.x, nb);
    if (tb >= nb) return;  // padding block of the XCD order
    const int ch = (int)(tb % (unsigned)w.nch);
    const unsigned r1 = tb / (unsigned)w.nch;
    const int s = (int)(r1 % (unsigned)w.ns), i0 = (int)(r1 / (unsigned)w.ns) * w.TI;
    const int i1 = min(i0 + w.TI, PER ? g.nx : g.nnx);  // owned node layers (PER: masters only)
    if (PER && i0 >= i1) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave / w.NW, t = (wave - q * w.NW) * 63 + lane;
    // [group][9][ne]: own share of row k + 1, of the layer above rows k, k + 1
    T *ex = reinterpret_cast<T *>(md_lds) + 9 * q * ne + t;
    // entry, element and own node as in k_modal
    const unsigned qs = (unsigned)(ch * w.M + t + w.R - 1);
    const int kq = (int)(qs / (unsigned)w.R), c = (int)(qs - (unsigned)(kq * w.R));
    const int k = kq - 2, j = s * w.W - 1 + c;
    const int ke = PER && k == -1 ? g.nz - 1 : k, je = PER && j == -1 ? g.ny - 1 : j;
    const bool el_ok = ke >= 0 && ke < g.nz && je >= 0 && je < g.ny;
    const bool own = lane > 0 && t > w.R && t <= w.R + w.M && c > 0 && k >= 0 && k < (PER ? g.nz : g.nnz) &&
                     j < (PER ? g.ny : g.nny);
    // INT: the pair of row k holds the own node, also where no element follows it
    // along j (then as its second) or k
    const bool nod_ok = INT ? ke >= 0 && ke < g.nnz && je >= 0 && je < g.nny : el_ok;
    const bool jlast = INT && je == g.ny;
    const int jp = jlast ? je - 1 : je;
    const int plane = g.nny * g.nnz, nod0 = k * g.nny + j, enod = ke * g.nny + jp;
    const int lo = nod_ok ? 3 * S * enod : kMdOut, hi = el_ok ? 3 * S * (enod + g.nny) : kMdOut;
    const int eo = el_ok ? S * (4 * ke * g.ny + 2 * je) : kMdOut, oo = own ? 3 * S * nod0 : kMdOut;
    const long vb = (long)S * g.ndof;
    const MdBuf BU = md_buf(PRE ? a.F : a.U, vb), BF = md_buf(a.F, MV ? 0 : vb);
    const MdBuf BD = md_buf(a.RD, JAC || PRE ? vb : 0), BE = md_buf(CX, 8L * S * g.nel);
    const MdBuf BM = md_buf(a.mask, a.mask ? g.nnod : 0);  // no mask: reads 0
    const int fp = 3 * S * plane, ep = 4 * S * g.ny * g.nz;  // bytes of a node layer, of a layer of scales
    const T pr = T(a.prerelax), om = T(a.omega);

    const int il = i0 - 1 + q;  // the group's element layer, and the node layer below it
    const int ie = PER && il < 0 ? g.nx - 1 : il;
    const bool el = ie >= 0 && ie < g.nx && il < i1, emit = q > 0 && il < i1;
    T u[4][6], d[4][6], e[8], f[3], de[3], ue[3];  // node rows: lower layer k, k + 1, upper layer k, k + 1
    unsigned m8 = 0;
    T cv[INT ? 4 : 1][6];  // INT: the coarse element's node pairs, rows K, K + 1 of its two layers
    unsigned mk[2][4];
    if constexpr (INT) {
        const int cny = g.ny / 2 + 1, cp = 3 * S * cny * (g.nz / 2 + 1);
        const MdBuf BC = md_buf(a.Uc, (long)S * coarse_ndof(g));
        const int clo = nod_ok ? 3 * S * ((ke >> 1) * cny + (jp >> 1)) : kMdOut;
        const int chi = nod_ok && ke < g.nz ? clo + 3 * S * cny : kMdOut;
        const int mlo = nod_ok ? enod : kMdOut, mhi = el_ok ? enod + g.nny : kMdOut;
        if (el || emit) {
            md_ld6(BC, clo, (il >> 1) * cp, cv[0]);
            md_ld6(BC, chi, (il >> 1) * cp, cv[1]);
            if (el) {
                md_ld6(BC, clo, ((il >> 1) + 1) * cp, cv[2]);
                md_ld6(BC, chi, ((il >> 1) + 1) * cp, cv[3]);
            }
#pragma unroll
            for (int p = 0; p < 2; ++p)
                if (p == 0 || el) {
                    const int so = (il + p) * plane;
                    mk[p][0] = __builtin_amdgcn_raw_buffer_load_b8(BM, mlo, so, 0);
                    mk[p][1] = __builtin_amdgcn_raw_buffer_load_b8(BM, mlo + 1, so, 0);
                    mk[p][2] = __builtin_amdgcn_raw_buffer_load_b8(BM, mhi, so, 0);
                    mk[p][3] = __builtin_amdgcn_raw_buffer_load_b8(BM, mhi + 1, so, 0);
                }
            if (!el) {  // the mesh's last node layer: its own node alone
                md_ld6(BU, lo, il * fp, u[0]);
                md_ld6(BU, hi, il * fp, u[1]);
            }
        }
    }
    if (el) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int so = (p < 2 ? ie : il + 1) * fp;
            md_ld6(BU, p & 1 ? hi : lo, so, u[p]);
            if (PRE) md_ld6(BD, p & 1 ? hi : lo, so, d[p]);
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {  // children (is, iz): the pair along j
            T v[2];
            md_ld2(BE, eo + (p & 1) * 2 * S * g.ny, (2 * ie + (p >> 1)) * ep, v);
            e[2 * p] = v[0];
            e[2 * p + 1] = v[1];
        }
    }
    if (emit) {
        m8 = __builtin_amdgcn_raw_buffer_load_b8(BM, own ? nod0 : kMdOut, il * plane, 0);
        if (!MV) md_ld3(BF, oo, il * fp, f);
        if (JAC || PRE) md_ld3(BD, oo, il * fp, de);
        if (!PRE && !INT && MODE != OP_DEFECT) md_ld3(BU, oo, il * fp, ue);
    }
    if (a.ctl && a.ctl[0]) return;  // converged: read with the loads above
    T y[3] = {T(0), T(0), T(0)};
    if constexpr (INT) {
        if (el || emit) {
            T cc[2][2][6];  // the lower and the upper layer
            const bool odd = il & 1;
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int x = 0; x < 6; ++x) {
                    const T mean = el ? T(0.5) * (cv[r][x] + cv[2 + r][x]) : T(0);
                    cc[0][r][x] = odd ? mean : cv[r][x];
                    cc[1][r][x] = odd ? cv[2 + r][x] : mean;
                }
            md_prolong(cc[0], ke & 1, jp & 1, mk[0], u[0], u[1]);
            if (el) md_prolong(cc[1], ke & 1, jp & 1, mk[1], u[2], u[3]);
#pragma unroll
            for (int x = 0; x < 3; ++x) ue[x] = jlast ? u[0][3 + x] : u[0][x];
        }
    }
    if (el) {
        if (PRE) {
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int x = 0; x < 6; ++x) u[p][x] = pr * (u[p][x] * d[p][x]);
        }
        Jk<T> pa, pb;
        md_jk(u[0], u[1], pa);
        md_jk(u[2], u[3], pb);
        T m[3][2][2][2];
#pragma unroll
        for (int cc = 0; cc < 3; ++cc)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    m[cc][0][b][x] = pa.v[cc][b][x] + pb.v[cc][b][x];
                    m[cc][1][b][x] = pb.v[cc][b][x] - pa.v[cc][b][x];
                }
        const T cx[2][2][2] = {{{e[0], e[2]}, {e[1], e[3]}}, {{e[4], e[6]}, {e[5], e[7]}}};
        md_element_gp(m, a.mc, cx);
        // forces of one layer to its rows: v for row k, vh for row k + 1
        auto rows = [&](const T (&s4)[2][2], T &v, T &vh) {
            const T l0 = s4[0][0] - s4[0][1], l1 = s4[1][0] - s4[1][1];
            const T h0 = s4[0][0] + s4[0][1], h1 = s4[1][0] + s4[1][1];
            v = (l0 - l1) + md_below(l0 + l1);
            vh = (h0 - h1) + md_below(h0 + h1);
        };
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) {
            T below[2][2], above[2][2], yh, z, zh;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const T r1v = m[cc][1][b][x], r0v = b == 0 && x == 0 ? T(0) : m[cc][0][b][x];  // no force from a translation
                    below[b][x] = r0v - r1v;
                    above[b][x] = r0v + r1v;
                }
            rows(below, y[cc], yh);
            rows(above, z, zh);
            if (lane > 0) {
                ex[cc * ne] = yh;
                ex[(3 + cc) * ne] = z;
                ex[(6 + cc) * ne] = zh;
            }
        }
    }
    __syncthreads();
    if (!emit || !own) return;
    const T *ey = ex - 9 * ne;  // the group below
    const long dof = 3 * ((long)il * plane + nod0);
#pragma unroll
    for (int cc = 0; cc < 3; ++cc) {
        T yc = y[cc];
        if (el) yc += ex[cc * ne - w.R];
        if (PER || il > 0) yc += ey[(3 + cc) * ne] + ey[(6 + cc) * ne - w.R];
        const bool fixed = (m8 >> cc) & 1u;
        T v;
        if (MV) {
            v = fixed ? T(0) : yc;
        } else if (!JAC) {
            v = fixed ? T(0) : f[cc] - yc;
            if (PRE) a.out2[dof + cc] = pr * (f[cc] * de[cc]);
        } else {
            const T uo = PRE ? pr * (f[cc] * de[cc]) : ue[cc];
            v = fma(om * de[cc], fixed ? T(0) : f[cc] - yc, uo);
        }
        a.out[dof + cc] = v;
        if (PER) {
            // the images: an iterate's value, 0 for a residual
            const bool bi = il == 0, bk = k == 0, bj = j == 0;
            if (bi || bk || bj) {
                const T im = JAC ? v : T(0);
                const long di = 3L * plane * g.nx, dk = 3L * g.nny * g.nz, dj = 3L * g.ny;
#pragma unroll
                for (int p = 1; p < 8; ++p)
                    if ((!(p & 4) || bi) && (!(p & 2) || bk) && (!(p & 1) || bj))
                        a.out[dof + cc + (p & 4 ? di : 0) + (p & 2 ? dk : 0) + (p & 1 ? dj : 0)] = im;
            }
        }
    }
}

template <class T, int MODE, bool PER>
void launch_flat(hipStream_t s, const OpArgsT<T> &a, const T *CX)
{
    const ModalWork &w = a.mw;
    const dim3 grid((unsigned)xcd_launch(w.blocks()), 1, batch_dim(a.nb));
    const unsigned ne = 63u * w.NW + 1u;
    k_modal_flat<T, MODE, PER><<<grid, 64 * w.NW * (w.TI + 1), 9u * (w.TI + 1) * ne * sizeof(T), s>>>(a, CX);
}

template <class T, class TU, int MODE, int EL, bool PER>
void launch_mode(hipStream_t s, const OpArgsT<T> &a, const T *CX, const CgTest *tst = nullptr)
{
    const ModalWork &w = a.mw;
    MdTest<MODE, EL, PER> test{};
    unsigned tests = 0;
    if constexpr (md_tests<MODE, EL, PER>()) {
        if (tst && tst->sc) {
            test = *tst;
            tests = kMdTestBlocks;
        }
    }
    const dim3 grid((unsigned)xcd_launch(w.blocks()) + tests, 1, batch_dim(a.nb));
    const unsigned ne = 63u * w.NW + 1u;
    if constexpr (EL == 1) {
        if (w.flat && !a.partials) {
            launch_flat<T, MODE, PER>(s, a, CX);
            return;
        }
    }
    if (w.NW > md_max_waves<T, EL>()) throw std::runtime_error("modal operator: tiling of another element");
    k_modal<T, TU, MODE, EL, PER><<<grid, 64 * w.NW, 6u * ne * sizeof(T), s>>>(a, CX, test);
}

template <class T, int EL>
void launch(hipStream_t s, int mode, const OpArgsT<T> &a, const T *CX, const CgTest *test = nullptr)
{
    if (a.per) {
        switch (mode) {
        case OP_MATVEC: launch_mode<T, T, OP_MATVEC, EL, true>(s, a, CX); break;
        case OP_DEFECT: launch_mode<T, T, OP_DEFECT, EL, true>(s, a, CX); break;
        case OP_JACOBI: launch_mode<T, T, OP_JACOBI, EL, true>(s, a, CX); break;
        default: throw std::runtime_error("periodic operator: mode");  // the prerelaxed modes read F on images
        }
        return;
    }
    switch (mode) {
    case OP_MATVEC: launch_mode<T, T, OP_MATVEC, EL, false>(s, a, CX); break;
    case OP_DEFECT: launch_mode<T, T, OP_DEFECT, EL, false>(s, a, CX); break;
    case OP_JACOBI: launch_mode<T, T, OP_JACOBI, EL, false>(s, a, CX); break;
    case OP_PRE_JACOBI: launch_mode<T, T, OP_PRE_JACOBI, EL, false>(s, a, CX, test); break;
    case OP_PRE_DEFECT: launch_mode<T, T, OP_PRE_DEFECT, EL, false>(s, a, CX, test); break;
    case OP_INTERP_JACOBI:
        // interp_fused (vcycle.h) asks for it only here
        if (EL != 1 || !a.mw.flat || a.partials) throw std::runtime_error("fused interpolation: tiling");
        launch_flat<T, OP_INTERP_JACOBI, false>(s, a, CX);
        break;
    case OP_MATVEC_UF:
        if constexpr (EL == 0 && std::is_same<T, double>::value)
            launch_mode<double, float, OP_MATVEC_UF, 0, false>(s, a, CX);
        break;
    default: break;
    }
}

}  // namespace

template <class T>
void launch_op0_modal(hipStream_t s, int mode, const OpArgsT<T> &a, const CgTest *test)
{
    launch<T, 0>(s, mode, a, a.CX, test);
}
template void launch_op0_modal<double>(hipStream_t, int, const OpArgsT<double> &, const CgTest *);
template void launch_op0_modal<float>(hipStream_t, int, const OpArgsT<float> &, const CgTest *);

template <class T>
void launch_op1_mf(hipStream_t s, int mode, OpArgsT<T> a, const T *CXf, double nu)
{
    // Lame constants of D (E = 1), the 1/8 of each transform and the element
    // of side h = 2: |J| w_g = 1, a derivative is half a node difference
    const double c1 = 1.0 / ((1 + nu) * (1 - 2 * nu)) / 64.0;
    a.mc[0] = T(c1 * nu);
    a.mc[1] = T(c1 * (1 - 2 * nu));
    a.mc[2] = T(c1 * (1 - 2 * nu) / 2);
    a.mc[3] = T(1.0 / std::sqrt(3.0));
    launch<T, 1>(s, mode, a, CXf);
}
template void launch_op1_mf<double>(hipStream_t, int, OpArgsT<double>, const double *, double);
template void launch_op1_mf<float>(hipStream_t, int, OpArgsT<float>, const float *, double);

// Sums and differences of the 8 nodes of out[q][72], in modal order, in place:
// q = 4a + 2b + d.
static void modal_transform(double (*out)[72])
{
    for (int h = 1; h < 8; h *= 2)
        for (int q = 0; q < 8; ++q)
            if (!(q & h)) {
                double *__restrict x = out[q], *__restrict y = out[q + h];
                for (int i = 0; i < 72; ++i) {
                    const double a = x[i], b = y[i];
                    x[i] = a + b;
                    y[i] = b - a;
                }
            }
}

// The modal matrix of an isotropic element: entry (r, c) is constant id; every
// other entry is 0.
struct ModalPattern {
    struct Entry {
        int r, c, id;
    };
    int n = 0;
    Entry e[64];
    ModalPattern()
    {
        // mode q = 4a + 2b + d of component c: 3q + c
        const int n0[3] = {3 * 4 + 0, 3 * 2 + 1, 3 * 1 + 2};  // u100, v010, w001
        const int tw[3] = {3 * 3 + 0, 3 * 5 + 1, 3 * 6 + 2};  // u011, v101, w110
        const int sh[3][2] = {{3 * 2 + 0, 3 * 4 + 1}, {3 * 1 + 1, 3 * 2 + 2}, {3 * 1 + 0, 3 * 4 + 2}};
        const int bd[3][2] = {{3 * 6 + 1, 3 * 5 + 2}, {3 * 6 + 0, 3 * 3 + 2}, {3 * 5 + 0, 3 * 3 + 1}};
        auto add = [&](int r, int c, int id) { e[n++] = {r, c, id}; };
        for (int p = 0; p < 3; ++p) {
            for (int q = 0; q < 3; ++q) {
                add(n0[p], n0[q], p == q ? 1 : 2);
                add(tw[p], tw[q], p == q ? 7 : 8);
            }
            for (int x = 0; x < 2; ++x)
                for (int y = 0; y < 2; ++y) {
                    add(sh[p][x], sh[p][y], 3);
                    add(bd[p][x], bd[p][y], x == y ? 5 : 6);
                }
            add(3 * 7 + p, 3 * 7 + p, 4);
        }
        // by rows: the order in which the constants are averaged
        std::sort(e, e + n, [](const Entry &x, const Entry &y) { return x.r != y.r ? x.r < y.r : x.c < y.c; });
    }
};

// The 8 modal constants of Ke0; false when its modal matrix is not of the
// isotropic form above to rounding (1e-14 of its largest entry).  Part of every
// call that takes a Ke0, so both transforms run over 72 contiguous values and most
// others are told apart at once (1.2 and 0.07 us; 2.4 and 2.0 value by value).
bool modal_constants(const double *Ke0, double *C)
{
    static const ModalPattern pat;
    // node order ie = {0,1,1,0,0,1,1,0}, je = {0,0,1,1,0,0,1,1}, ke = {0,0,0,0,1,1,1,1}
    static const int node[8] = {0, 4, 3, 7, 1, 5, 2, 6};  // of 4 x + 2 y + z
    // a quick no, for what is clearly something else: the shear of the three planes
    {
        static const double x[8] = {-1, 1, 1, -1, -1, 1, 1, -1}, y[8] = {-1, -1, 1, 1, -1, -1, 1, 1},
                            z[8] = {-1, -1, -1, -1, 1, 1, 1, 1};
        double g[4] = {};  // (u010, u010), (v001, v001), (u001, u001), (u010, v100)
        for (int a = 0; a < 8; ++a) {
            const double *u = Ke0 + 72 * a, *v = u + 24;
            for (int b = 0; b < 8; ++b) {
                g[0] += y[a] * y[b] * u[3 * b];
                g[1] += z[a] * z[b] * v[3 * b + 1];
                g[2] += z[a] * z[b] * u[3 * b];
                g[3] += y[a] * x[b] * u[3 * b + 1];
            }
        }
        for (int k = 1; k < 4; ++k)
            if (std::fabs(g[k] - g[0]) > 1e-12 * std::fabs(g[0])) return false;
    }
    double W[8][72], V[8][72];  // W[q][24c + col], then V[p][24d + row], row = 3q + c: M[row][3p + d]
    for (int q = 0; q < 8; ++q)
        for (int i = 0; i < 72; ++i) W[q][i] = 0.125 * Ke0[72 * node[q] + i];
    modal_transform(W);
    for (int p = 0; p < 8; ++p)
        for (int d = 0; d < 3; ++d)
            for (int q = 0; q < 8; ++q)
                for (int c = 0; c < 3; ++c) V[p][24 * d + 3 * q + c] = 0.125 * W[q][24 * c + 3 * node[p] + d];
    modal_transform(V);
    auto at = [&](int r, int c) -> double & { return V[c / 3][24 * (c % 3) + r]; };
    double m[72] = {}, big = 0.0;
    for (int p = 0; p < 8; ++p)
        for (int i = 0; i < 72; ++i) m[i] = std::max(m[i], std::fabs(V[p][i]));
    for (double x : m) big = std::max(big, x);
    double v[9] = {};
    int cnt[9] = {};
    for (int k = 0; k < pat.n; ++k) {
        v[pat.e[k].id] += at(pat.e[k].r, pat.e[k].c);
        ++cnt[pat.e[k].id];
    }
    for (int q = 1; q < 9; ++q) v[q] /= cnt[q];
    for (int k = 0; k < pat.n; ++k) at(pat.e[k].r, pat.e[k].c) -= v[pat.e[k].id];
    for (int p = 0; p < 8; ++p)
        for (int i = 0; i < 72; ++i)
            if (!(std::fabs(V[p][i]) <= 1e-14 * big)) return false;  // NaN fails too
    C[0] = v[1] - v[2];
    C[1] = v[2];
    C[2] = v[3];
    C[3] = v[4];
    C[4] = v[5];
    C[5] = v[6];
    C[6] = v[7] - v[8];
    C[7] = v[8];
    return true;
}

// Tiling of grid g for values of `bytes` bytes (el: the level-1 element;
// children: element scales per element at most).
// Among waves per block NW, strips along j and the layers TI that fill one,
// two or three rounds of resident blocks, the smallest modelled time: rounds
// times the layers a block marches (its first needs the layer before it, and
// a block takes about two layers' time to start and to end), times the work
// of a layer, which is bound by the waves that share a SIMD or, when there
// are few, by one layer's latency.
ModalWork modal_work(const Grid &g, int bytes, int el, int children)
{
    ModalWork best;
    // 32-bit byte offsets
    if ((long)bytes * g.ndof >= kMdOut || (long)bytes * children * g.nel >= kMdOut) return best;
    if (el) {
        // k_modal_flat where one block per CU covers the mesh, with one wave
        // per SIMD in FP64 (TI <= 3; two share its double rate: 7.2 against
        // 7.2 us at 64x32x32 elements) and two in FP32 (4.8 against 5.4 us;
        // beyond, with two blocks per CU, 9.5 against 8.7 us at 96x48x48), the
        // fewest layers first: a block of two layers starts and ends sooner
        for (int TI = 1; TI <= (bytes == 8 ? 3 : 7); ++TI)
            for (int ns = 1; ns <= 8; ++ns) {
                const int W = (g.nny + ns - 1) / ns, R = W + 1, M = std::min(63 - R, R * g.nnz);
                if (M < 16 || (ns > 1 && W < 4)) continue;
                const int nsr = (g.nny + W - 1) / W, nch = (R * g.nnz + M - 1) / M, nib = (g.nnx + TI - 1) / TI;
                if ((long)nsr * nch * nib > 256) continue;
                best.flat = 1;
                best.NW = 1, best.W = W, best.R = R, best.M = M;
                best.ns = nsr, best.nch = nch, best.TI = TI, best.nib = nib;
                return best;
            }
    }
    const int waves = bytes == 8 ? (el ? 1 : 2) : (el ? 3 : 4);  // resident per SIMD (md_min_waves)
    const double per_wave = el ? 0.9 : 0.38;                     // a wave's layer with its SIMD alone, in us
    const double latency = 1.2;
    // Eight strips at most, more where even those are longer than two waves: a block
    // works on R + 1 entries before its own, and 8 strips of 3801 nodes left 27 of
    // 504 entries to it (20 mgcg9 iterations at 8x3800x8 9.8 -> 11.4 ms against the
    // node-gather, 7.4 now), or none.
    constexpr int kMdLongStrip = 126;
    double cost = 0.0;
    for (int NW = 1; NW <= (bytes == 8 && el ? 4 : kMdMaxWaves); NW *= 2)
        for (int ns = 1;; ++ns) {
            const int W = (g.nny + ns - 1) / ns, R = W + 1;
            if (ns > 1 && W < 12) break;
            if (ns > 8 && W <= kMdLongStrip) break;
            if (63 * NW - R < 16) continue;
            const int M = std::min(63 * NW - R, R * g.nnz);
            const int nsr = (g.nny + W - 1) / W, nch = (R * g.nnz + M - 1) / M;
            const long per_cu = std::max(1, 4 * waves / NW), slots = 256 * per_cu;
            for (int round = 1; round <= 3; ++round) {
                const long fit = std::max(1L, round * slots / ((long)nsr * nch));
                const int TI = (int)((g.nnx + fit - 1) / fit), nib = (g.nnx + TI - 1) / TI;
                const long blocks = (long)nsr * nch * nib;
                const long rounds = (blocks + slots - 1) / slots, on_cu = std::min(per_cu, (blocks + 255) / 256);
                const double c = rounds * (TI + 3) * std::max(latency, per_wave * (double)(on_cu * NW) / 4.0);
                if (best.NW == 0 || c < 0.999 * cost) {
                    cost = c;
                    best.NW = NW;
                    best.W = W;
                    best.R = R;
                    best.M = M;
                    best.ns = nsr;
                    best.nch = nch;
                    best.TI = TI;
                    best.nib = nib;
                }
            }
        }
    return best;
}

}  // namespace gputo
