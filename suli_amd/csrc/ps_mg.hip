// Multigrid-preconditioned CG, batched over problems.
//
// The scaled system A e = b (unit diagonal, ps_cg.hip) has a condition number
// that grows with the square of the grid's longest side, so plain CG takes
// about a thousand iterations on a 256x128x96 two-phase tank.  Here one
// iteration applies a V-cycle M to the residual first (z = M r, p = z + beta
// p, beta and alpha from r.z) and takes 10 to 25 on cells of about equal sides.
//
// The smoother works on points and the coarsening joins 2x2x2 cells whatever
// their sides are, so flat and tall cells take more: 40x32x24, mixed from
// prd1 = 0 to 1e-12, with dx = dy = 1/16, 1/8, 1/4, 1, 2, 4, 8, 16 dz: 231,
// 132, 77, 14, 24, 73, 143, 212 iterations and 9.9, 5.8, 3.4, 0.82, 1.25, 3.2,
// 6.2, 9.1 ms (plain CG 2584, 1024, 656, 416, 560, 1024, 2184, 10000 and 21.6,
// 8.9, 5.9, 4.0, 5.1, 8.9, 18.4, 82.6 ms; at 256x128x96 185 to 72 ms at 1/16,
// 218 to 61 at 16).  No grid tried, from 4096 cells to 3 million and from 1/32 to
// 32, was faster by plain CG (FP64 at 4096 cells and 1/32: 7.4 and 5.9 ms).
//
// Mixed solves: everything is FP32 inside FP64 residual replacement, as the CG
// step: dot products, alpha and beta are FP64 and convergence is judged on
// the FP64 true residual.  FP64 solves by the relative rule: the iterate, the
// residual, the directions, the operator and the stop test are FP64 as in
// plain CG (ps_cg.hip), and only the V-cycle works on an FP32 copy of the
// residual (scaled by a power of two, mg_shift); which z it returns changes the
// number of iterations, not what r = A e - b reaches.
//
// The V-cycle smooths with a Chebyshev polynomial of degree two before and
// after the coarse correction on every level.  A coarse cell joins 2x2x2
// cells; restriction sums the children's residuals, prolongation copies the
// parent's value, and a coarse face's coefficient is half the sum of the fine
// faces it covers (twice the distance).  The cycle is symmetric positive
// definite for any face coefficients >= 0, solid cells and periodic sides
// included.  In the scaled variables of this solver a cell's value is w p
// with w = sqrt(d): restriction weighs with w, prolongation too, and each
// coarse level is scaled to a unit diagonal in the same way (its own w).
//
// Degree two against one Jacobi sweep (weight 0.85): 15 iterations to 1e-12
// on the 256x128x96 tank instead of 49, for five passes over the fine grid
// instead of three.  Degree two on the coarse levels alone gives 24.
//
// With the polynomial s(A) = c0 + c1 A, a level's steps are
//   t = A r                      rho = r - A s(A) r = r - c0 t - c1 A t
//   (coarse: restrict rho, correct by e)
//   r0 = rho - A (w e)           z = s(A) r + w e + s(A) r0
// each a single pass with one application of A on the fine grid; below it the
// two on either side of the coarser levels are one pass.
//
// Measured at 256x128x96 from prd1 = 0 to 1e-12 relative: plain CG 37.8 ms
// (1992 iterations of one 18.5 us launch), this 3.3 ms (18 iterations); the
// stretched masked cylinder at 384x192x128 238.4 and 10.4 ms, SuLi-IT's
// 256x128x48 19.4 and 3.0 ms, twelve uneven tanks in a batch 67.7 and 6.1 ms.
//
// One iteration n (lbot: the first level of the bottom kernel):
//   A1      r_{n-1} = r_{n-2} - alpha q (formed where needed), t; partials r.r
//   A2      rho, restricted to level 1
//   D       the same on levels 1 .. lbot-1
//   bottom  levels lbot and coarser, one workgroup per problem, in LDS
//   U       coarse correction and post-smoothing on levels lbot-1 .. 1
//   B1, B2  the same on level 0: z_n; partials r.z
//   dir     beta, c -= alpha_{n-1} p_{n-1}, p_n = z + beta p, q = A p;
//           partials p.q
// or, in a step whose A2 finds r_{n-1} small enough, instead of D .. dir the
// residual replacement: dir folds c and alpha p into e, then
//   k_true_residual, k_mg_decide: converged, or on with the replaced residual
// FP64: before A1, upd64 (r -= alpha q, its FP32 copy, partials r.r); instead
// of dir, dir64 (ps_cg.hip; e -= alpha p), which ends the solve when A2 found
// r.r at the threshold.  Problems in bricks (pd.brick): A1 and A2 in one launch
// (down), r.r judged by the bottom kernel, B1 and B2 in one (up).
// Each total is summed by the kernel that needs it from the partials of an
// earlier launch, as in ps_cg.hip.
#include <algorithm>
#include <climits>

#include "ps_device.h"

namespace sps {
namespace {

// Chebyshev polynomial of degree two on [kLmax / 6, kLmax], kLmax = 2 above
// the scaled operator's spectrum (0, 2): s(x) = kC0 + kC1 x, positive there,
// as 1 - x s(x) stays within (-1, 1).
constexpr float kLmax = 2.0f, kLmin = kLmax / 6.0f;
constexpr float kTheta = 0.5f * (kLmax + kLmin), kDelta = 0.5f * (kLmax - kLmin);
constexpr float kRho1 = 1.0f / (2.0f * kTheta / kDelta - kDelta / kTheta);
constexpr float kC0 = (1.0f + kRho1 * kDelta / kTheta) / kTheta + 2.0f * kRho1 / kDelta;
constexpr float kC1 = -2.0f * kRho1 / (kDelta * kTheta);
constexpr int kBotThreads = 1024;
constexpr int kBotPer = kMgBottomCells / kBotThreads;

enum { kA1 = 0, kA2 = 1, kB1 = 2, kB2 = 3, kDir = 4 };

__device__ __forceinline__ TileRef tile_of(const MgStep &st, const TileRef *tab, int t)
{
    return st.one >= 0 ? TileRef{st.one, t} : tab[t];
}

struct Run {
    int begin, end;
};
__device__ __forceinline__ Run my_run(int ntab, int block, int G)
{
    const long long L = xcd_tile(block, G);
    Run r;
    r.begin = (int)(L * ntab / G);
    r.end = (int)((L + 1) * ntab / G);
    return r;
}

__device__ __forceinline__ Run my_run(int ntab) { return my_run(ntab, blockIdx.x, gridDim.x); }

// Per-workgroup cache of a problem's partial-sum total.
struct TotalCache {
    int prob = -1;
    double value = 0.0;
    __device__ __forceinline__ double get(int p, const double *partial, int n)
    {
        if (p != prob) {
            value = block_total_of(partial, n);
            prob = p;
        }
        return value;
    }
};

// Partial sums of a problem's fine kernels (ntm tiles): p.q, r.z, r.r.
__device__ __forceinline__ double *part_pq(const ProbDev &pd) { return pd.P.m4; }
__device__ __forceinline__ double *part_rz(const ProbDev &pd) { return pd.P.m4 + pd.ntm; }
__device__ __forceinline__ double *part_rr(const ProbDev &pd) { return pd.P.m4 + 2 * pd.ntm; }
// r_k alternates between two buffers, as p_k does.
__device__ __forceinline__ float *rbuf(const ProbDev &pd, int k) { return (k & 1) ? pd.r32b : pd.r32; }
__device__ __forceinline__ float *mpbuf(const ProbDev &pd, int k) { return pd.p32 + (k & 1) * pd.pslot; }


typedef float vf4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float vf2 __attribute__((ext_vector_type(2), aligned(4)));

// Four (two) floats `off` floats into a plane that starts at `base`: base is
// the same in every lane, so the load takes a scalar base and a 32-bit offset.
__device__ __forceinline__ void ld4(gptr<const float> base, unsigned off, float (&o)[4])
{
    const vf4 t = *(gptr<const vf4>)((gptr<const char>)base + (unsigned)(off * 4u));
#pragma unroll
    for (int m = 0; m < 4; ++m) o[m] = t[m];
}
__device__ __forceinline__ void ld2(gptr<const float> base, unsigned off, float (&o)[2])
{
    const vf2 t = *(gptr<const vf2>)((gptr<const char>)base + (unsigned)(off * 4u));
    o[0] = t[0];
    o[1] = t[1];
}
__device__ __forceinline__ float ld1(gptr<const float> base, unsigned off)
{
    return *(gptr<const float>)((gptr<const char>)base + (unsigned)(off * 4u));
}
__device__ __forceinline__ void st4(gptr<float> base, unsigned off, const float (&v)[4], int nv)
{
    if (nv == 4) {
        vf4 t;
#pragma unroll
        for (int m = 0; m < 4; ++m) t[m] = v[m];
        *(gptr<vf4>)((gptr<char>)base + (unsigned)(off * 4u)) = t;
    } else {
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if (m < nv) *(gptr<float>)((gptr<char>)base + (unsigned)((off + m) * 4u)) = v[m];
    }
}
__device__ __forceinline__ void fld4(gptr<const float> p, float (&o)[4])
{
    const vf4 t = *(gptr<const vf4>)p;
#pragma unroll
    for (int m = 0; m < 4; ++m) o[m] = t[m];
}

// Lane shifts by one within the wave (DPP): lane l gets lane l - 1's (l + 1's)
// value; the first (last) lane keeps its own, which the callers replace.
__device__ __forceinline__ float from_lower(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float from_upper(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x130, 0xf, 0xf, false));
}

// One tile of a fine kernel.  A wave holds 64 / lr pairs of rows (j, j + 1),
// each lane four x cells of both, and marches the tile's planes with the
// values at k - 1, k and k + 1 in registers; a workgroup's four waves take
// consecutive pairs.  Two rows per lane halve the y-neighbour loads and put
// the 2x2x2 cells of a coarse cell into one lane.  Rows up to 64 (128) cells
// take 16 (32) lanes, so that short rows share a wave.
//
// The stencil value v is formed where it is needed, y = (A v), and on the
// tile's cells
//   A1   v = a - s b   a = r_{n-2}, b = q (fresh: v = a)   r = v, t = y
//   A2   v = a         a = t       rho = r - c0 t - c1 y, summed into coarse cells
//   B1   v = w e       e = the parent's correction         r0 = rho - y
//   B2   v = a         a = r0      z = c0 r + c1 t + w e + c0 r0 + c1 y
//   dir  v = a + s b   a = z, b = p_{n-1} (fresh: v = a)   p = v, q = y, c -= s2 b
// EDGE: rows whose ends need a loaded neighbour (x periodic, or more than one
// segment of 4 lr cells) or whose length is no multiple of four.
struct FineArgs {
    gptr<const float> a, b;       // stencil operands
    gptr<const float> r, t;       // at the cell: r, t (A2, B2), rho as r (B1)
    gptr<float> o1, o2, x;        // outputs; x: c (dir)
    bool fresh, do_x;
    float s, s2;
};

template <int KIND, bool EDGE>
__device__ __forceinline__ double mg_tile(const ProbDev &pd, int tile, const FineArgs &F)
{
    constexpr bool kTwo = KIND == kA1 || KIND == kDir;   // two operands a, b
    constexpr bool kW = KIND == kA2 || KIND == kB2;      // w at the cell
    const gptr<const float> a_ = F.a, b_ = F.b;
    const bool fresh = F.fresh;
    const float s = F.s;
    const int nx = pd.g.nx, ny = pd.g.ny, nz = pd.g.nz;
    const int px = pd.g.px, py = pd.g.py;
    const int lrs = pd.mlrs, lr = 1 << lrs;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sl = lane & (lr - 1), grp = lane >> lrs;
    const int tx = tile % pd.mtx, rest = tile / pd.mtx, ty = rest % pd.mty, tz = rest / pd.mty;
    const int i0 = tx * (lr * 4), i = i0 + 4 * sl;
    const int jw = 2 * ((ty * 4 + wv) << (6 - lrs));
    double acc = 0.0;
    if (jw >= ny) return acc;   // the whole wave
    const int j = jw + 2 * grp;
    const int k0 = tz * pd.mkz, k1 = min(k0 + pd.mkz, nz);
    const bool rowa = j < ny, rowb = j + 1 < ny;
    const int nva = (rowa && i < nx) ? min(nx - i, 4) : 0, nvb = rowb ? nva : 0;
    const int ci = i < nx ? i : 0;
    const int ja = rowa ? j : ny - 1;
    // row b's place holds row a's north neighbour where row b does not exist
    const int jb = rowb ? j + 1 : nb_hi(ja, ny, py);
    const int js = nb_lo(ja, ny, py), jn = rowb ? nb_hi(j + 1, ny, py) : jb;
    const unsigned oa = (unsigned)ja * nx + ci, ob = (unsigned)jb * nx + ci;
    const unsigned os = (unsigned)js * nx + ci, on = (unsigned)jn * nx + ci;
    const long long plane = (long long)nx * ny;
    // parents (smooth), and this lane's coarse cells (resid)
    const MgLevel &C = pd.lv[1];
    const int ncx = C.nx;
    const long long cplane = (long long)C.nx * C.ny;
    const unsigned ca = (unsigned)(ja >> 1) * ncx + (ci >> 1), cb = (unsigned)(jb >> 1) * ncx + (ci >> 1);
    const unsigned cs = (unsigned)(js >> 1) * ncx + (ci >> 1), cn = (unsigned)(jn >> 1) * ncx + (ci >> 1);
    const gptr<const float> e1 = glob((const float *)C.t), w_ = glob((const float *)pd.w32);
    // cells beyond the segment's ends
    const bool ise = i < nx && (i + 4 >= nx || sl == lr - 1);
    const bool ldw = EDGE && sl == 0 && (i0 > 0 || px), lde = EDGE && ise && (i + 4 < nx || px);
    const int xw = i0 > 0 ? i0 - 1 : nx - 1, xe = i + 4 < nx ? i + 4 : 0;

    auto v_of = [&](float a, float b) -> float {
        if (KIND == kB1) return a * b;
        if (KIND == kA1) return fresh ? a : a - s * b;
        if (KIND == kDir) return fresh ? a : a + s * b;
        return a;
    };
    // four values of a row at plane kk, with the second operand
    auto row = [&](int kk, unsigned o, unsigned c, float (&v)[4], float (&b)[4]) {
        float a[4], e[2];
        if (KIND == kB1) {
            ld4(w_ + kk * plane, o, a);
            ld2(e1 + (kk >> 1) * cplane, c, e);
        } else {
            ld4(a_ + kk * plane, o, a);
            if (kTwo) ld4(b_ + kk * plane, o, b);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) v[m] = v_of(a[m], KIND == kB1 ? e[m >> 1] : kTwo ? b[m] : 0.f);
    };
    auto one = [&](int kk, int jj, int x) -> float {
        const unsigned o = (unsigned)jj * nx + x;
        if (KIND == kB1)
            return ld1(w_ + kk * plane, o) * ld1(e1 + (kk >> 1) * cplane, (unsigned)(jj >> 1) * ncx + (x >> 1));
        return v_of(ld1(a_ + kk * plane, o), kTwo ? ld1(b_ + kk * plane, o) : 0.f);
    };

    // the rows' table bits for the tile's planes (planes past 32, which mg_plan's
    // tiles of at most 8 do not have, would read the arrays)
    unsigned bita = 0, bitb = 0;
    if (pd.rowreg) {
        const gptr<const unsigned> rr = glob((const unsigned *)pd.rowreg);
        const int wpp = (ny + 31) / 32;
        const int ke = min(k1, k0 + 32);
        for (int k = k0; k < ke; ++k) {
            const unsigned word = rr[(long long)k * wpp + (ja >> 5)] >> (ja & 31);
            bita |= (word & 1u) << (k - k0);
            if (rowb) bitb |= ((word >> 1) & 1u) << (k - k0);
        }
    }
    const gptr<const float> SX = glob(pd.sx32), SY = glob(pd.sy32), SZ = glob(pd.sz32);
    const gptr<const float> RX = glob(pd.rx32), RY = glob(pd.ry32), RZ = glob(pd.rz32);
    const int jb1 = min(ja + 1, ny - 1);   // row b for face addresses
    const int jy2 = min(ja + 2, ny);       // y face north of row b

    float vb[2][4], vc[2][4], bc[2][4];
    row(k0, oa, ca, vc[0], bc[0]);
    row(k0, ob, cb, vc[1], bc[1]);
    if (k0 > 0) {
        float t1[4];
        row(k0 - 1, oa, ca, vb[0], t1);
        row(k0 - 1, ob, cb, vb[1], t1);
    } else {
#pragma unroll
        for (int m = 0; m < 4; ++m) vb[0][m] = vc[0][m], vb[1][m] = vc[1][m];
    }
    float szb[2][4];
    {
        const bool ra = bita & 1u, rb = bitb & 1u;
        fld4(ra ? RZ + 4 * k0 : SZ + (long long)k0 * plane + (unsigned)ja * nx + ci, szb[0]);
        fld4(rb ? RZ + 4 * k0 : SZ + (long long)k0 * plane + (unsigned)jb1 * nx + ci, szb[1]);
    }
    float sum[2] = {0.f, 0.f};
    for (int k = k0; k < k1; ++k) {
        const int ku = k < nz - 1 ? k + 1 : k;
        const bool ra = (k - k0) < 32 && ((bita >> (k - k0)) & 1u), rb = (k - k0) < 32 && ((bitb >> (k - k0)) & 1u);
        float vt[2][4], bt[2][4], vs[4], vn[4], t1[4];
        row(ku, oa, ca, vt[0], bt[0]);
        row(ku, ob, cb, vt[1], bt[1]);
        row(k, os, cs, vs, t1);
        row(k, on, cn, vn, t1);
        float sx[2][5], sy0[4], sy1[4], sy2[4], szt[2][4];
        {
            const gptr<const float> xa = ra ? RX + 8 * k : SX + ((long long)k * ny + ja) * (nx + 1) + ci;
            const gptr<const float> xb = rb ? RX + 8 * k : SX + ((long long)k * ny + jb1) * (nx + 1) + ci;
            float t[4];
            fld4(xa, t);
#pragma unroll
            for (int m = 0; m < 4; ++m) sx[0][m] = t[m];
            sx[0][4] = xa[4];
            fld4(xb, t);
#pragma unroll
            for (int m = 0; m < 4; ++m) sx[1][m] = t[m];
            sx[1][4] = xb[4];
            const long long fy = (long long)k * (ny + 1);
            fld4(ra ? RY + 4 * k : SY + (fy + ja) * nx + ci, sy0);
            fld4(ra ? RY + 4 * k : SY + (fy + ja + 1) * nx + ci, sy1);
            fld4(rb ? RY + 4 * k : SY + (fy + jy2) * nx + ci, sy2);
            fld4(ra ? RZ + 4 * (k + 1) : SZ + (long long)(k + 1) * plane + (unsigned)ja * nx + ci, szt[0]);
            fld4(rb ? RZ + 4 * (k + 1) : SZ + (long long)(k + 1) * plane + (unsigned)jb1 * nx + ci, szt[1]);
        }
        // operands of the outputs
        float wx[2][4], rc[2][4], tc[2][4], ec[2][2];
        if (kW) {
            ld4(w_ + k * plane, oa, wx[0]);
            ld4(w_ + k * plane, ob, wx[1]);
        }
        if (KIND == kDir) {
            ld4((gptr<const float>)F.x + k * plane, oa, wx[0]);
            ld4((gptr<const float>)F.x + k * plane, ob, wx[1]);
        }
        if (KIND == kA2 || KIND == kB1 || KIND == kB2) {
            ld4(F.r + k * plane, oa, rc[0]);
            ld4(F.r + k * plane, ob, rc[1]);
        }
        if (KIND == kB2) {
            ld4(F.t + k * plane, oa, tc[0]);
            ld4(F.t + k * plane, ob, tc[1]);
            ld2(e1 + (k >> 1) * cplane, ca, ec[0]);
            ld2(e1 + (k >> 1) * cplane, cb, ec[1]);
        }
        float ew[2] = {vc[0][0], vc[1][0]}, ee[2];
        if (EDGE) {
            if (ldw) {
                ew[0] = one(k, ja, xw);
                ew[1] = one(k, jb, xw);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r)   // mirror ghost: the row's last cell
                ee[r] = nva == 1 ? vc[r][0] : nva == 2 ? vc[r][1] : nva == 3 ? vc[r][2] : vc[r][3];
            if (lde) {
                ee[0] = one(k, ja, xe);
                ee[1] = one(k, jb, xe);
            }
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int m = 1; m < 4; ++m)
                    if (nva == m) vc[r][m] = ee[r];
        } else {
            ee[0] = vc[0][3];
            ee[1] = vc[1][3];
        }
        if (k == nz - 1) {
            const float sg = pd.g.dtop ? -1.f : 1.f;   // Dirichlet lid: ghost = -cell
#pragma unroll
            for (int m = 0; m < 4; ++m) vt[0][m] = sg * vc[0][m], vt[1][m] = sg * vc[1][m];
        }
        float y[2][4];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float lo = from_lower(vc[r][3]), hi = from_upper(vc[r][0]);
            const float pw = sl == 0 ? ew[r] : lo;
            const float pe = ise ? ee[r] : hi;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const float east = m == 3 ? pe : vc[r][m + 1];
                const float west = m == 0 ? pw : vc[r][m - 1];
                const float north = r == 0 ? vc[1][m] : vn[m], south = r == 0 ? vs[m] : vc[0][m];
                const float sn = r == 0 ? sy1[m] : sy2[m], ss = r == 0 ? sy0[m] : sy1[m];
                y[r][m] = vc[r][m] - sx[r][m + 1] * east - sx[r][m] * west - sn * north - ss * south -
                          szt[r][m] * vt[r][m] - szb[r][m] * vb[r][m];
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int nv = r == 0 ? nva : nvb;
            const unsigned o = r == 0 ? oa : ob;
            float o1[4], o2[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const bool in = EDGE ? m < nv : nv > 0;
                const float v = vc[r][m], av = y[r][m];
                o1[m] = v;
                o2[m] = av;
                if (KIND == kA1) {
                    acc += in ? (double)v * (double)v : 0.0;
                } else if (KIND == kA2) {
                    o1[m] = rc[r][m] - kC0 * v - kC1 * av;
                    sum[m >> 1] += in ? wx[r][m] * o1[m] : 0.f;
                } else if (KIND == kB1) {
                    o1[m] = rc[r][m] - av;
                } else if (KIND == kB2) {
                    o1[m] = kC0 * (rc[r][m] + v) + kC1 * (tc[r][m] + av) + wx[r][m] * ec[r][m >> 1];
                    acc += in ? (double)rc[r][m] * (double)o1[m] : 0.0;
                } else {
                    acc += in ? (double)v * (double)av : 0.0;
                    wx[r][m] = wx[r][m] - F.s2 * bc[r][m];
                }
            }
            if (!(KIND == kA1 && fresh)) st4(F.o1 + k * plane, o, o1, nv);
            if (KIND == kA1 || KIND == kDir) st4(F.o2 + k * plane, o, o2, nv);
            if (KIND == kDir && F.do_x) st4(F.x + k * plane, o, wx[r], nv);
        }
        if (KIND == kA2 && ((k & 1) || k == nz - 1)) {
            // the coarse cells are complete: scaled residual of level 1
            const unsigned cc = (unsigned)(ja >> 1) * ncx + (ci >> 1);
            const gptr<float> rc = glob(C.r) + (k >> 1) * cplane;
            const gptr<const float> wc = glob((const float *)C.w) + (k >> 1) * cplane;
#pragma unroll
            for (int m = 0; m < 2; ++m)
                if (2 * m < nva) {
                    const float w1 = wc[cc + m];
                    rc[cc + m] = w1 > 0.f ? sum[m] / w1 : 0.f;
                }
            sum[0] = sum[1] = 0.f;
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                vb[r][m] = vc[r][m];
                vc[r][m] = vt[r][m];
                if (KIND == kDir) bc[r][m] = bt[r][m];
                szb[r][m] = szt[r][m];
            }
    }
    return acc;
}

// A tile's share of e += c - al p, c = 0 (all arrays, 16 or 32 bytes a lane).
__device__ __forceinline__ void fold_correction(const ProbDev &pd, int tile, gptr<float> c, gptr<const float> p,
                                                float al)
{
    typedef double vd4 __attribute__((ext_vector_type(4)));
    typedef float va4 __attribute__((ext_vector_type(4)));
    const gptr<double> e = glob(pd.e);
    const long long len = pd.g.n, nv = len / 4, stride = (long long)pd.ntm * kThreads;
    for (long long v = (long long)tile * kThreads + threadIdx.x; v < nv; v += stride) {
        const va4 cv = ((gptr<const va4>)c)[v], pv = ((gptr<const va4>)p)[v];
        vd4 ev = ((gptr<const vd4>)e)[v];
#pragma unroll
        for (int m = 0; m < 4; ++m) ev[m] += (double)(cv[m] - al * pv[m]);
        ((gptr<vd4>)e)[v] = ev;
        ((gptr<va4>)c)[v] = va4{0.f, 0.f, 0.f, 0.f};
    }
    if (tile == 0) {
        const long long x = nv * 4 + threadIdx.x;
        if (x < len) {
            e[x] += (double)(c[x] - al * p[x]);
            c[x] = 0.f;
        }
    }
}

// The total r.r entering iteration n is known: whether the step ends otherwise
// (S->next_refresh = n, stored by one thread).  Mixed: a replacement instead of
// iteration n once r.r (the FP32 recurrence's) has reached the threshold, or
// fallen as far as FP32 carries one cycle, or at the cap; FP64: the end.
__device__ __forceinline__ bool judge(gptr<CgScalars> S, bool mixed, bool fresh, int n, double rr, bool store)
{
    const double thresh = S->thresh, base = S->refreshes ? S->rr_after : S->rr0;
    const int iters = S->iters, max_iter = S->max_iter;
    int prev = S->prev_iters;
    bool due;
    if (!mixed) {
        const bool below = n > 1 && rr <= thresh;
        if (below && prev == 0) {
            prev = n;
            if (store) S->prev_iters = n;
        }
        due = n > 1 && (rr <= kMgMargin * thresh || iters >= max_iter || (below && n - prev >= kMgMarginIters));
    } else {
        due = !fresh && (rr <= kMgMargin * thresh || rr <= kMgCycleDrop * base || iters - prev >= kMgMaxGap ||
                         iters >= max_iter);
    }
    if (store) {
        S->rr[n & 1] = rr;
        if (due) S->next_refresh = n;
    }
    return due;
}

// alpha and beta of a mixed problem's direction step; false at a breakdown:
// r.z and p.q are positive for every operator the V-cycle is definite for,
// unless a value left FP32's range (upwards: infinities and NaN; downwards: a
// sum of 0 with r.r above its threshold).  A replacement starts the directions
// afresh: the replaced residual is no longer r - alpha q, and directions
// conjugate to it went on at a third of the rate.
__device__ __forceinline__ bool direction(gptr<CgScalars> S, bool fresh, bool due, int n, double rz, bool store,
                                          double &alpha, double &beta)
{
    const double rz_prev = S->rz[(n - 1) & 1];
    alpha = S->alpha;
    const bool bad = mg_breakdown(fresh, due, rz, alpha);
    beta = fresh || !(rz_prev > 0.0) ? 0.0 : rz / rz_prev;
    if (store) {
        if (bad) {
            S->giveup = 1;
            S->final_ = 1;
            S->done_at = n;
        } else if (!due) {
            S->rz[n & 1] = rz;
            S->iters = S->iters + 1;
        }
    }
    return !bad;
}

template <int KIND>
__device__ __forceinline__ void fine_tiles(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab, Run run,
                                           const MgStep &st, int *ran)
{
    const int step = st.step;
    TotalCache tot;
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tile_of(st, tab, t);
        const ProbDev &pd = P[tr.prob];
        const gptr<CgScalars> S = glob(st.S + tr.prob);
        const int n = step - pd.n0 + 1;
        const int done_at = S->done_at, skip_e_at = S->skip_e_at;
        const bool due = KIND != kA1 && KIND != kA2 && S->next_refresh == n;   // set by A2
        if (n < 1 || n > done_at || (due && KIND != kDir)) continue;
        const bool mixed = pd.mixed != 0;
        if (KIND == kDir && !mixed) continue;
        // r_{n-1} stands in its buffer (FP64: always the one FP32 copy)
        const bool fresh = n == 1 || step == skip_e_at || !mixed;
        const gptr<float> r = glob(mixed ? rbuf(pd, n - 1) : pd.r32), r0 = glob(mixed ? rbuf(pd, n) : pd.r32b);
        const gptr<float> tt = glob(pd.t32), rho = glob(pd.q32b), z = rho, q = glob(pd.q32);
        FineArgs F{};
        if (KIND == kA1) {
            double alpha = 0.0;
            if (mixed) {
                const double rz = S->rz[(n - 1) & 1];
                const double pq = tot.get(tr.prob, part_pq(pd), pd.ntm);
                alpha = fresh || !(pq != 0.0) ? 0.0 : rz / pq;   // 0 / 0 once the residual is 0
                if (tr.tile == 0 && threadIdx.x == 0) S->alpha = alpha;
            }
            // (the second operand is loaded whether used or not)
            F = FineArgs{fresh ? r : r0, mixed ? q : r, nullptr, nullptr, r, tt, nullptr, fresh, false, (float)alpha, 0.f};
        } else if (KIND == kA2) {
            if (tr.tile == 0) {
                const double rr = mixed ? block_total_of(part_rr(pd), pd.ntm) : block_total_of(pd.P.upd, pd.nt1);
                judge(S, mixed, fresh, n, rr, threadIdx.x == 0);
            }
            F = FineArgs{tt, nullptr, r, nullptr, rho, nullptr, nullptr, false, false, 0.f, 0.f};
        } else if (KIND == kB1) {
            F = FineArgs{nullptr, nullptr, rho, nullptr, r0, nullptr, nullptr, false, false, 0.f, 0.f};
        } else if (KIND == kB2) {
            F = FineArgs{r0, nullptr, r, tt, z, nullptr, nullptr, false, false, 0.f, 0.f};
        } else {
            const double rz = due ? 0.0 : tot.get(tr.prob, part_rz(pd), pd.ntm);
            double alpha, beta;
            if (!direction(S, fresh, due, n, rz, tr.tile == 0 && threadIdx.x == 0, alpha, beta)) continue;
            if (ran && !due && tr.tile == 0 && threadIdx.x == 0 && tr.prob == 0) *ran = 1;
            const gptr<float> po = glob(mpbuf(pd, n - 1));
            const gptr<float> x = glob(pd.c32);
            if (due) {
                // e += c - alpha_{n-1} p_{n-1}, c = 0
                fold_correction(pd, tr.tile, x, po, (float)alpha);
                continue;
            }
            F = FineArgs{z, po, nullptr, nullptr, glob(mpbuf(pd, n)), q, x, fresh, !fresh, (float)beta, (float)alpha};
        }
        const double acc = pd.medge ? mg_tile<KIND, true>(pd, tr.tile, F) : mg_tile<KIND, false>(pd, tr.tile, F);
        if (KIND == kA2 || KIND == kB1) continue;
        const double sres = block_sum(acc);
        if (threadIdx.x == 0) (KIND == kA1 ? part_rr(pd) : KIND == kB2 ? part_rz(pd) : part_pq(pd))[tr.tile] = sres;
    }
}

// Waves per SIMD: the kinds with one operand fit three, those with two
// operands need the registers of two.
constexpr int fine_waves(int kind) { return kind == kA1 || kind == kDir ? 2 : 3; }
template <int KIND>
__global__ __launch_bounds__(kThreads, fine_waves(KIND)) void k_mg_fine(const ProbDev *__restrict__ P,
                                                                        const TileRef *__restrict__ tab, int ntab,
                                                                        MgStep st, int *ran)
{
    fine_tiles<KIND>(P, tab, my_run(ntab), st, ran);
}

// FP64: r_{n-1} = r_{n-2} - alpha_{n-1} q_{n-1} and its scaled FP32 copy for the
// V-cycle, r.r partials (1-D tiles).
__global__ __launch_bounds__(kThreads) void k_mg_upd64(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab,
                                                       int ntab, MgStep st)
{
    typedef double vd4 __attribute__((ext_vector_type(4)));
    typedef float va4 __attribute__((ext_vector_type(4)));
    const Run run = my_run(ntab);
    const int step = st.step;
    TotalCache tot;
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tile_of(st, tab, t);
        const ProbDev &pd = P[tr.prob];
        const gptr<CgScalars> S = glob(st.S + tr.prob);
        const int n = step - pd.n0 + 1;
        if (n < 1 || n > S->done_at) continue;
        const bool first = n == 1;
        const double rz = S->rz[(n - 1) & 1], rr = S->rr[(n - 1) & 1];
        const double pq = first ? 0.0 : tot.get(tr.prob, pd.P.spmv, pd.nt3);
        const double scale = ldexp(1.0, -mg_shift(rr));
        const double alpha = pq != 0.0 ? rz / pq : 0.0;
        if (tr.tile == 0 && threadIdx.x == 0) S->alpha = alpha;
        const gptr<double> r = glob(pd.r);
        const gptr<const double> q = glob((const double *)pd.q);
        const gptr<float> r32 = glob(pd.r32);
        const long long len = pd.g.n, nv = len / 4, stride = (long long)pd.nt1 * kThreads;
        double acc = 0.0;
        for (long long v = (long long)tr.tile * kThreads + threadIdx.x; v < nv; v += stride) {
            vd4 rv = ((gptr<const vd4>)r)[v];
            va4 f;
            if (!first) {
                const vd4 qv = ((gptr<const vd4>)q)[v];
#pragma unroll
                for (int m = 0; m < 4; ++m) rv[m] = rv[m] - alpha * qv[m];
                ((gptr<vd4>)r)[v] = rv;
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                acc += rv[m] * rv[m];
                f[m] = (float)(scale * rv[m]);
            }
            ((gptr<va4>)r32)[v] = f;
        }
        if (tr.tile == 0) {
            const long long c = nv * 4 + threadIdx.x;
            if (c < len) {
                const double rv = first ? r[c] : r[c] - alpha * q[c];
                r[c] = rv;
                r32[c] = (float)(scale * rv);
                acc += rv * rv;
            }
        }
        const double s = block_sum(acc);
        if (threadIdx.x == 0) pd.P.upd[tr.tile] = s;
    }
}

// ---- coarse levels (l >= 1) -------------------------------------------------

__device__ __forceinline__ bool running(const ProbDev &pd, const MgStep &st, int prob)
{
    const gptr<const CgScalars> S = glob((const CgScalars *)st.S + prob);
    const int n = st.step - pd.n0 + 1;
    return n >= 1 && n <= S->done_at && n != S->next_refresh;
}

// Bricks of 16x8x8 cells, one workgroup each; a brick holds whole coarse cells.
// With two cells around, a brick's vectors are in LDS, and both matrix products
// of a half of the cycle are done there: the first on the brick and its face
// neighbours, the second on the brick.  A thread loads one column of the box and
// owns kOwn cells in z, so that a cell's place is worked out once for its column.
//
// On the coarse levels and on small grids a pass waits on its launch and on
// memory's latency, not its rate, so two products a launch pay: on the coarse
// levels two launches took 4.9 us each over 128x64x48 cells and 4.0 over
// 64x32x24, one takes 8.5 to 9.1 and 5.4 to 6.6 (a 64x64x32 solve 1.20 -> 1.14 ms,
// 256x128x96 3.52 -> 3.44, 384x192x128 11.33 -> 11.09).
//
// The brick's shape weighs latency (more, smaller bricks) against the halo: 16x4x4
// took 0.72 ms for a 32x24x20 solve and 28.4 ms for 128 problems of 40 to 50 cells
// a side, 16x8x4 0.75 and 26.2, 16x8x8 0.78 and 24.2 (marched tiles on the fine
// level: 1.00 and 23.1).
constexpr int kBx = 16, kBy = 8, kBz = 8;
constexpr int kHx = kBx + 4, kHy = kBy + 4, kHz = kBz + 4;   // the box
constexpr int kOwn = kBx * kBy * kBz / kThreads;
constexpr int kCols = kBx * kBy;
static_assert(kThreads % kCols == 0 && kOwn * (kThreads / kCols) == kBz && kHx * kHy <= kThreads && kOwn > 0, "brick");
__host__ __device__ inline int bricks(const MgLevel &L)
{
    return ((L.nx + kBx - 1) / kBx) * ((L.ny + kBy - 1) / kBy) * ((L.nz + kBz - 1) / kBz);
}

// A box column's or plane's place in the grid: wrapped around periodic sides;
// beyond a wall it is the mirror image inside (the coarse levels' faces there
// are 0), at box position + shift, and above the top its values count sg times
// (the p = 0 lid: -1).
struct Col {
    int i, j, shift;
};
struct Plane {
    int k, shift;
    float sg;
};
struct Brick {
    int x0, y0, z0;      // cell (0, 0, 0) of the box
    int nx, ny, nz;
    bool px, py;
    float top;
    __device__ __forceinline__ Brick(const MgLevel &L, int tile, float lid)
        : nx(L.nx), ny(L.ny), nz(L.nz), px(L.px), py(L.py), top(lid)
    {
        const int bx = (nx + kBx - 1) / kBx, by = (ny + kBy - 1) / kBy;
        const int rest = tile / bx;
        x0 = (tile % bx) * kBx - 2;
        y0 = (rest % by) * kBy - 2;
        z0 = (rest / by) * kBz - 2;
    }
    __device__ __forceinline__ Col col(int a, int b) const
    {
        int i = x0 + a, j = y0 + b;
        if (px) i += i < 0 ? nx : i >= nx ? -nx : 0;
        if (py) j += j < 0 ? ny : j >= ny ? -ny : 0;
        Col c;
        c.i = min(max(i, 0), nx - 1);
        c.j = min(max(j, 0), ny - 1);
        c.shift = (c.i - i) + (c.j - j) * kHx;
        return c;
    }
    __device__ __forceinline__ Plane plane(int d) const
    {
        const int k = z0 + d;
        Plane p;
        p.k = min(max(k, 0), nz - 1);
        p.shift = (p.k - k) * (kHx * kHy);
        p.sg = k >= nz ? top : 1.f;
        return p;
    }
    __device__ __forceinline__ int index(const Col &c, const Plane &p) const { return (p.k * ny + c.j) * nx + c.i; }
    static __device__ __forceinline__ int pos(int a, int b, int d) { return (d * kHy + b) * kHx + a; }
};
struct Faces {
    float e, w, n, s, t, b;
    __device__ __forceinline__ void load(const MgLevel &L, int c, int j, int k)
    {
        const gptr<const float> sx = glob((const float *)L.sx) + (c + (k * L.ny + j));
        const gptr<const float> sy = glob((const float *)L.sy) + (c + k * L.nx);
        const gptr<const float> sz = glob((const float *)L.sz) + c;
        e = sx[1];
        w = sx[0];
        n = sy[L.nx];
        s = sy[0];
        t = sz[L.nx * L.ny];
        b = sz[0];
    }
    // the six neighbours' share of A v at box position x
    __device__ __forceinline__ float sum(const float *v, int x) const
    {
        return e * v[x + 1] + w * v[x - 1] + n * v[x + kHx] + s * v[x - kHx] + t * v[x + kHx * kHy] +
               b * v[x - kHx * kHy];
    }
};
// f(box position (a, b, d)) for the brick's face neighbours, below and above,
// south and north, west and east
template <class F>
__device__ __forceinline__ void each_shell(F &&f)
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int h = 0; h < 2 * kCols; h += kThreads) {
        const int u = h + tid;
        if (2 * kCols % kThreads == 0 || u < 2 * kCols)
            f(2 + (u & 15), 2 + (u >> 4) % kBy, u < kCols ? 1 : 2 + kBz);
    }
#pragma unroll
    for (int h = 0; h < 2 * kBx * kBz; h += kThreads) {
        const int u = h + tid;
        if (2 * kBx * kBz % kThreads == 0 || u < 2 * kBx * kBz)
            f(2 + (u & 15), u < kBx * kBz ? 1 : 2 + kBy, 2 + (u >> 4) % kBz);
    }
    if (tid < 2 * kBy * kBz) f(tid < kBy * kBz ? 1 : 2 + kBx, 2 + tid % kBy, 2 + tid / kBy % kBz);
}
// The thread's own cells of a brick: (a, b, d + q), q < kOwn.
struct Own {
    int a, b, d;
    Col col;
    Plane pl[kOwn];
    int c[kOwn];
    bool in[kOwn];   // a cell of the grid, and this brick's
    __device__ __forceinline__ explicit Own(const Brick &B)
    {
        const int tid = threadIdx.x;
        a = 2 + (tid & 15);
        b = 2 + (tid >> 4) % kBy;
        d = 2 + tid / kCols * kOwn;
        col = B.col(a, b);
        const bool inc = B.x0 + a < B.nx && B.y0 + b < B.ny;
#pragma unroll
        for (int q = 0; q < kOwn; ++q) {
            pl[q] = B.plane(d + q);
            c[q] = B.index(col, pl[q]);
            in[q] = inc && B.z0 + d + q < B.nz;
        }
    }
    __device__ __forceinline__ int pos(int q) const { return Brick::pos(a, b, d + q); }
};
// The thread's column of the box.
struct BoxCol {
    bool any;
    int pos;
    Col col;
    __device__ __forceinline__ explicit BoxCol(const Brick &B)
    {
        const int tid = threadIdx.x;
        any = tid < kHx * kHy;
        pos = tid;
        col = B.col(tid % kHx, any ? tid / kHx : 0);
    }
};

struct HalfBox {
    float va[kHx * kHy * kHz], vb[kHx * kHy * kHz];
};
// Both products of a half cycle, from the box column's values v0:
//   down  v = r:    u = A v,        y = A u
//   up    v = w e:  u = rho - A v,  y = A u
template <bool UP>
__device__ __forceinline__ void half_cycle(const MgLevel &L, const Brick &B, const Own &o, const BoxCol &bc,
                                           HalfBox &s, const float (&v0)[kHz], gptr<const float> rho,
                                           float (&v)[kOwn], float (&u)[kOwn], float (&y)[kOwn])
{
    Faces f0[kOwn];
    float rho0[kOwn];
#pragma unroll
    for (int q = 0; q < kOwn; ++q) {
        f0[q].load(L, o.c[q], o.col.j, o.pl[q].k);
        rho0[q] = UP ? rho[o.c[q]] : 0.f;
    }
    __syncthreads();   // reads of the last tile
    if (bc.any) {
#pragma unroll
        for (int d = 0; d < kHz; ++d) s.va[bc.pos + d * kHx * kHy] = v0[d];
    }
    __syncthreads();
    // u at a box cell: its mirror image's, times sg
    auto first = [&](const Faces &f, int x, float sg, float rh) {
        const float av = s.va[x] - f.sum(s.va, x);
        return sg * (UP ? rh - av : av);
    };
#pragma unroll
    for (int q = 0; q < kOwn; ++q) {
        const int x = o.pos(q);
        v[q] = s.va[x];
        u[q] = first(f0[q], x + o.col.shift + o.pl[q].shift, o.pl[q].sg, rho0[q]);
        s.vb[x] = u[q];
    }
    each_shell([&](int a, int b, int d) {
        const Col col = B.col(a, b);
        const Plane p = B.plane(d);
        const int c = B.index(col, p), x = Brick::pos(a, b, d);
        Faces f;
        f.load(L, c, col.j, p.k);
        s.vb[x] = first(f, x + col.shift + p.shift, p.sg, UP ? rho[c] : 0.f);
    });
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kOwn; ++q) y[q] = u[q] - f0[q].sum(s.vb, o.pos(q));
}

// The brick's coarse cells: the restricted residual, scaled, from w rho at the
// own cells.  (va is read no more.)
__device__ __forceinline__ void restrict_brick(const MgLevel &C, const Brick &B, const Own &o, float *va,
                                               const float (&wr)[kOwn])
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int q = 0; q < kOwn; ++q) va[o.pos(q)] = wr[q];
    __syncthreads();
    if (tid < kOwn * kThreads / 8) {
        const int I = tid % (kBx / 2), J = tid / (kBx / 2) % (kBy / 2), K = tid / (kBx / 2 * kBy / 2);
        const float *x = va + Brick::pos(2 + 2 * I, 2 + 2 * J, 2 + 2 * K);
        const float *z = x + kHx * kHy;
        const float sum = ((x[0] + x[1]) + (x[kHx] + x[kHx + 1])) + ((z[0] + z[1]) + (z[kHx] + z[kHx + 1]));
        const int ic = (B.x0 + 2) / 2 + I, jc = (B.y0 + 2) / 2 + J, kc = (B.z0 + 2) / 2 + K;
        if (ic < C.nx && jc < C.ny && kc < C.nz) {
            const int c = (kc * C.ny + jc) * C.nx + ic;
            const float wc = C.w[c];
            glob(C.r)[c] = wc > 0.f ? sum / wc : 0.f;
        }
    }
}

// Half a cycle on level l (1 <= l < lbot): down (A1 and A2 of the fine
// kernels) or up (B1 and B2); no partial sums, and up leaves the un-scaled
// correction.
template <bool UP>
__global__ __launch_bounds__(kThreads) void k_mg_level(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab,
                                                       int ntab, int l, MgStep st)
{
    __shared__ HalfBox box;
    const Run run = my_run(ntab);
    for (int tt = run.begin; tt < run.end; ++tt) {
        const TileRef tr = tile_of(st, tab, tt);
        const ProbDev &pd = P[tr.prob];
        if (!running(pd, st, tr.prob)) continue;
        const MgLevel &L = pd.lv[l], &C = pd.lv[l + 1];
        const Brick B(L, tr.tile, 1.f);
        const Own o(B);
        const BoxCol bc(B);
        const gptr<float> t = glob(L.t), rho = glob(L.rho);
        const gptr<const float> r = glob((const float *)L.r), w = glob((const float *)L.w),
                                e = glob((const float *)C.t);
        float v0[kHz], wc[kOwn], rc[kOwn], tc[kOwn];
#pragma unroll
        for (int d = 0; d < kHz; ++d) {
            const Plane p = B.plane(d);
            const int c = B.index(bc.col, p);
            v0[d] = UP ? w[c] * e[((p.k >> 1) * C.ny + (bc.col.j >> 1)) * C.nx + (bc.col.i >> 1)] : r[c];
        }
#pragma unroll
        for (int q = 0; q < kOwn; ++q) {
            wc[q] = w[o.c[q]];
            rc[q] = UP ? r[o.c[q]] : 0.f;
            tc[q] = UP ? t[o.c[q]] : 0.f;
        }
        float v[kOwn], u[kOwn], y[kOwn];
        half_cycle<UP>(L, B, o, bc, box, v0, rho, v, u, y);
#pragma unroll
        for (int q = 0; q < kOwn; ++q) {
            const int c = o.c[q];
            if (UP) {
                const float z = kC0 * (rc[q] + u[q]) + kC1 * (tc[q] + y[q]) + v[q];
                if (o.in[q]) t[c] = wc[q] > 0.f ? z / wc[q] : 0.f;
            } else {
                const float rh = v[q] - kC0 * u[q] - kC1 * y[q];
                if (o.in[q]) {
                    t[c] = u[q];
                    rho[c] = rh;
                }
                wc[q] = o.in[q] ? wc[q] * rh : 0.f;
            }
        }
        if (!UP) restrict_brick(C, B, o, box.va, wc);
    }
}

// The fine level of a problem with pd.brick set, the same way.
//   down  A1 and A2 (r_{n-1}, t, rho, the restriction; partials r.r)
//   up    B1 and B2 (z in the place of r0; partials r.z)
//   dir   as in k_mg_fine
// r.r is judged by the bottom kernel.
enum { kDown = 0, kUp = 1, kDirB = 2 };
template <int KIND>
__device__ __forceinline__ void brick_tiles(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab, Run run,
                                            const MgStep &st, int *ran)
{
    __shared__ HalfBox box;
    const int step = st.step;
    TotalCache tot;
    for (int tt = run.begin; tt < run.end; ++tt) {
        const TileRef tr = tile_of(st, tab, tt);
        const ProbDev &pd = P[tr.prob];
        const gptr<CgScalars> S = glob(st.S + tr.prob);
        const int n = step - pd.n0 + 1;
        const int done_at = S->done_at, skip_e_at = S->skip_e_at;
        const bool due = KIND != kDown && S->next_refresh == n;   // set by the bottom kernel
        if (n < 1 || n > done_at || (due && KIND != kDirB)) continue;
        const bool mixed = pd.mixed != 0;
        if (KIND == kDirB && !mixed) continue;
        const bool fresh = n == 1 || step == skip_e_at || !mixed;
        const bool lead = tr.tile == 0 && threadIdx.x == 0;
        const MgLevel &L = pd.lv[0], &C = pd.lv[1];
        const Brick B(L, tr.tile, pd.g.dtop ? -1.f : 1.f);
        const Own o(B);
        const gptr<float> r = glob(mixed ? rbuf(pd, n - 1) : pd.r32), r0 = glob(mixed ? rbuf(pd, n) : pd.r32b);
        const gptr<float> t = glob(pd.t32), rho = glob(pd.q32b), z = r0, qv = glob(pd.q32);
        const gptr<const float> w = glob((const float *)pd.w32);
        double acc = 0.0;
        float v[kOwn], u[kOwn], y[kOwn];
        if (KIND == kDown) {
            const BoxCol bc(B);
            // the second operand is loaded whether used or not
            const gptr<const float> a_ = fresh ? r : r0, b_ = mixed ? qv : r;
            float v0[kHz], b0[kHz], wc[kOwn];
#pragma unroll
            for (int d = 0; d < kHz; ++d) {
                const int c = B.index(bc.col, B.plane(d));
                v0[d] = a_[c];
                b0[d] = b_[c];
            }
#pragma unroll
            for (int q = 0; q < kOwn; ++q) wc[q] = w[o.c[q]];
            double alpha = 0.0;
            if (mixed) {
                const double rz = S->rz[(n - 1) & 1];
                const double pq = tot.get(tr.prob, part_pq(pd), pd.ntm);
                alpha = fresh || !(pq != 0.0) ? 0.0 : rz / pq;   // 0 / 0 once the residual is 0
                if (lead) S->alpha = alpha;
            }
#pragma unroll
            for (int d = 0; d < kHz; ++d) v0[d] = B.plane(d).sg * (fresh ? v0[d] : v0[d] - (float)alpha * b0[d]);
            half_cycle<false>(L, B, o, bc, box, v0, nullptr, v, u, y);
#pragma unroll
            for (int q = 0; q < kOwn; ++q) {
                const int c = o.c[q];
                const float rh = v[q] - kC0 * u[q] - kC1 * y[q];
                if (o.in[q]) {
                    if (!fresh) r[c] = v[q];
                    t[c] = u[q];
                    rho[c] = rh;
                    acc += (double)v[q] * (double)v[q];
                }
                wc[q] = o.in[q] ? wc[q] * rh : 0.f;
            }
            restrict_brick(C, B, o, box.va, wc);
        } else if (KIND == kUp) {
            const BoxCol bc(B);
            const gptr<const float> e = glob((const float *)C.t);
            float v0[kHz], rc[kOwn], tc[kOwn];
#pragma unroll
            for (int d = 0; d < kHz; ++d) {
                const Plane p = B.plane(d);
                v0[d] = p.sg * (w[B.index(bc.col, p)] *
                                e[((p.k >> 1) * C.ny + (bc.col.j >> 1)) * C.nx + (bc.col.i >> 1)]);
            }
#pragma unroll
            for (int q = 0; q < kOwn; ++q) {
                rc[q] = r[o.c[q]];
                tc[q] = t[o.c[q]];
            }
            half_cycle<true>(L, B, o, bc, box, v0, rho, v, u, y);
#pragma unroll
            for (int q = 0; q < kOwn; ++q) {
                const float zc = kC0 * (rc[q] + u[q]) + kC1 * (tc[q] + y[q]) + v[q];
                if (o.in[q]) {
                    z[o.c[q]] = zc;
                    acc += (double)rc[q] * (double)zc;
                }
            }
        } else {
            const gptr<const float> po = glob(mpbuf(pd, n - 1));
            const gptr<float> x = glob(pd.c32);
            float zc[kOwn], pc[kOwn], xc[kOwn];
            Faces f[kOwn];
#pragma unroll
            for (int q = 0; q < kOwn; ++q) {
                const int c = o.c[q];
                zc[q] = z[c];
                pc[q] = po[c];
                xc[q] = x[c];
                f[q].load(L, c, o.col.j, o.pl[q].k);
            }
            const double rz = due ? 0.0 : tot.get(tr.prob, part_rz(pd), pd.ntm);
            double alpha, beta;
            if (!direction(S, fresh, due, n, rz, lead, alpha, beta)) continue;
            if (ran && !due && lead && tr.prob == 0) *ran = 1;
            if (due) {
                // e += c - alpha_{n-1} p_{n-1}, c = 0
                fold_correction(pd, tr.tile, x, po, (float)alpha);
                continue;
            }
            auto p_of = [&](float zv, float pv) { return fresh ? zv : zv + (float)beta * pv; };
            __syncthreads();   // reads of the last tile
            each_shell([&](int a, int b, int d) {
                const Plane p = B.plane(d);
                const int c = B.index(B.col(a, b), p);
                box.va[Brick::pos(a, b, d)] = p.sg * p_of(z[c], po[c]);
            });
            // (beyond the grid, the own cells' places hold mirror images too)
#pragma unroll
            for (int q = 0; q < kOwn; ++q) {
                v[q] = p_of(zc[q], pc[q]);
                box.va[o.pos(q)] = o.pl[q].sg * v[q];
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kOwn; ++q)
                if (o.in[q]) {
                    const int c = o.c[q];
                    const float av = v[q] - f[q].sum(box.va, o.pos(q));
                    glob(mpbuf(pd, n))[c] = v[q];
                    qv[c] = av;
                    if (!fresh) x[c] = xc[q] - (float)alpha * pc[q];
                    acc += (double)v[q] * (double)av;
                }
        }
        if (KIND == kDown && !mixed) continue;
        const double sres = block_sum(acc);
        if (threadIdx.x == 0) (KIND == kDown ? part_rr(pd) : KIND == kUp ? part_rz(pd) : part_pq(pd))[tr.tile] = sres;
    }
}

template <int KIND>
__global__ __launch_bounds__(kThreads) void k_mg_brick(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab,
                                                       int ntab, MgStep st, int *ran)
{
    brick_tiles<KIND>(P, tab, my_run(ntab), st, ran);
}

// Both kinds of problems in the tables: the first gb workgroups take the
// bricks, the others the marched tiles, in one launch.
template <int KIND, int BRICK>
__global__ __launch_bounds__(kThreads, fine_waves(KIND)) void k_mg_both(const ProbDev *__restrict__ P,
                                                                        const TileRef *__restrict__ fine, int nfine,
                                                                        int gb, const TileRef *__restrict__ brick,
                                                                        int nbrick, MgStep st, int *ran)
{
    const int b = blockIdx.x;
    if (b < gb)
        brick_tiles<BRICK>(P, brick, my_run(nbrick, b, gb), st, ran);
    else
        fine_tiles<KIND>(P, fine, my_run(nfine, b - gb, gridDim.x - gb), st, ran);
}

// Sums over the bottom kernel's workgroup, to every thread.
template <int N>
__device__ __forceinline__ void bot_sum(double (&v)[N])
{
    __shared__ double red[N][kBotThreads / 64];
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_sum(v[i]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i)
        if ((threadIdx.x & 63) == 0) red[i][threadIdx.x >> 6] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = red[i][0];
#pragma unroll
        for (int w = 1; w < kBotThreads / 64; ++w) v[i] += red[i][w];
    }
}

// One cell of a bottom level: its faces (E, W, N, S, T, B), w, and its parent
// (bits 6 up) and the sides it is on (bits 0 .. 5).  The set-up packs the
// cells of all bottom levels one after another.
struct BotCell {
    float s[6], w;
    unsigned bits;
    __device__ __forceinline__ float iw() const { return w > 0.f ? 1.f / w : 0.f; }
};
static_assert(sizeof(BotCell) == 32, "two 16-byte loads");
__device__ __forceinline__ BotCell packed_cell(gptr<const float> pack, int c)
{
    typedef float va4 __attribute__((ext_vector_type(4)));
    const va4 u = ((gptr<const va4>)pack)[2 * c], v = ((gptr<const va4>)pack)[2 * c + 1];
    return BotCell{{u[0], u[1], u[2], u[3], v[0], v[1]}, v[2], __float_as_uint(v[3])};
}
__device__ __forceinline__ BotCell bot_cell(const MgLevel &L, int c)
{
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int i = c % nx, r0 = c / nx, j = r0 % ny, k = r0 / ny;
    const float *sx = L.sx + (c + (k * ny + j)), *sy = L.sy + (c + k * nx), *sz = L.sz + c;
    BotCell b;
    b.s[0] = sx[1];
    b.s[1] = sx[0];
    b.s[2] = sy[nx];
    b.s[3] = sy[0];
    b.s[4] = sz[nx * ny];
    b.s[5] = sz[0];
    b.w = L.w[c];
    b.bits = (i == nx - 1) | (i == 0) << 1 | (j == ny - 1) << 2 | (j == 0) << 3 |
             (unsigned)((i >> 1) + (((nx + 1) >> 1) * ((j >> 1) + ((ny + 1) >> 1) * (k >> 1)))) << 6;
    return b;
}
// The six neighbours' share of A v.  Neighbours across a wall are the next
// cells in memory: their face is 0, and everything around is finite.  Only
// periodic sides need the wrapped index.
struct BotDim {
    int nx, pl;
    bool per;
};
__device__ __forceinline__ float bot_nb(const BotDim &d, const BotCell &b, int c, const float *v)
{
    const int nx = d.nx, pl = d.pl;
    const float z = b.s[4] * v[c + pl] + b.s[5] * v[c - pl];
    if (!d.per) return b.s[0] * v[c + 1] + b.s[1] * v[c - 1] + b.s[2] * v[c + nx] + b.s[3] * v[c - nx] + z;
    const int ny1 = pl - nx;
    return b.s[0] * v[c + ((b.bits & 1u) ? 1 - nx : 1)] + b.s[1] * v[c + ((b.bits & 2u) ? nx - 1 : -1)] +
           b.s[2] * v[c + ((b.bits & 4u) ? -ny1 : nx)] + b.s[3] * v[c + ((b.bits & 8u) ? ny1 : -nx)] + z;
}

// Levels lbot .. nlev - 1 of one problem in one workgroup.  Vectors live in
// LDS; the coefficients of level lbot in registers (kBotPer cells per thread)
// and the smaller levels' in LDS, all loaded at the start, so that the passes
// wait on memory once.  Levels of at most kBotWave cells are one wave's, whose
// LDS accesses need no barrier.
//
// The constant-pressure component is taken out of level lbot's residual and
// correction where the operator has that null space: the coarse levels would
// amplify the residual's about fourfold each, and leave one in the correction
// that is 99 % of z at a density ratio of 1000; the FP32 operator is not exactly
// (nor surely not negatively) singular on it, and p.q or r.z then went
// negative at small residuals.  Taken out of both sides, the cycle stays
// symmetric.
constexpr int kBotWave = 128;
__global__ __launch_bounds__(kBotThreads) void k_mg_bottom(const ProbDev *__restrict__ P,
                                                           const int *__restrict__ probs, MgStep st)
{
    __shared__ __align__(16) float lds[kMgBottomLds];
    __shared__ int lnx[kMgLevels], lny[kMgLevels], lnz[kMgLevels];
    const int prob = st.one >= 0 ? st.one : probs[blockIdx.x];
    const ProbDev &pd = P[prob];
    if (!running(pd, st, prob)) return;
    const int tid = threadIdx.x, lb = pd.lbot, nl = pd.nlev;
    const gptr<CgScalars> S = glob(st.S + prob);
    const bool project = S->project != 0, judged = pd.brick != 0;
    const MgLevel &L0 = pd.lv[lb];
    const int m0 = L0.nx * L0.ny * L0.nz, total = pd.nbot;
    const gptr<const float> pack = glob((const float *)pd.bot);
    const gptr<const float> r0 = glob((const float *)L0.r);
    const bool per = L0.px | L0.py;
    // the coefficients of the levels below lbot, then R, A, B, D (a value
    // per cell of all levels) with a guard of one plane on both sides
    const int guard = L0.nx * L0.ny;
    BotCell *const low = reinterpret_cast<BotCell *>(lds);
    float *const R = lds + 8 * (total - m0) + guard, *const A = R + total, *const B = A + total, *const D = B + total;
    BotCell top[kBotPer];
    double pr[3] = {0.0, 0.0, 0.0};   // w.r, w.w, and r.r of the fine grid
    if (judged) {
        const gptr<const double> part = glob((const double *)(pd.mixed ? part_rr(pd) : pd.P.upd));
        const int np = pd.mixed ? pd.ntm : pd.nt1;
        for (int i = tid; i < np; i += kBotThreads) pr[2] += part[i];
    }
#pragma unroll
    for (int q = 0; q < kBotPer; ++q) {
        const int c = tid + q * kBotThreads;
        if (c < m0) {
            top[q] = packed_cell(pack, c);
            const float r = r0[c];
            R[c] = r;
            pr[0] += (double)top[q].w * (double)r;
            pr[1] += (double)top[q].w * (double)top[q].w;
        }
    }
    for (int c = tid; c < total - m0; c += kBotThreads) low[c] = packed_cell(pack, m0 + c);
    if (tid < nl - lb) {
        lnx[tid] = pd.lv[lb + tid].nx;
        lny[tid] = pd.lv[lb + tid].ny;
        lnz[tid] = pd.lv[lb + tid].nz;
    }
    // every value that a wall's neighbour index can reach is finite
    for (int c = tid; c < guard; c += kBotThreads) R[c - guard] = D[total + c] = 0.f;
    for (int c = tid; c < total - m0; c += kBotThreads) R[m0 + c] = 0.f;
    for (int c = tid; c < 3 * total; c += kBotThreads) A[c] = 0.f;
    if (project || judged) bot_sum(pr);
    if (judged) {
        const int n = st.step - pd.n0 + 1;
        if (judge(S, pd.mixed != 0, n == 1 || st.step == S->skip_e_at || !pd.mixed, n, pr[2], tid == 0)) return;
    }
    if (project) {
        const double f = pr[1] > 0.0 ? pr[0] / pr[1] : 0.0;
#pragma unroll
        for (int q = 0; q < kBotPer; ++q) {
            const int c = tid + q * kBotThreads;
            if (c < m0) R[c] = (float)((double)R[c] - f * (double)top[q].w);
        }
    }
    __syncthreads();
    // f(cell, index in the level) for the cells of level lb + l at off, by
    // all threads or by the first wave's
    auto each = [&](bool wave, int l, int off, int m, auto &&f) {
        if (l == 0) {
#pragma unroll
            for (int q = 0; q < kBotPer; ++q) {
                const int c = tid + q * kBotThreads;
                if (c < m0) f(top[q], c);
            }
        } else {
            for (int c = tid; c < m; c += wave ? 64 : kBotThreads) f(low[off - m0 + c], c);
        }
    };
    auto sync = [&](bool wave) {
        if (wave)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        else
            __syncthreads();
    };
    auto dim = [&](int l) {
        const int nx = lnx[l], ny = lny[l];
        // a side of a single cell is not periodic (mg_plan), its faces are 0
        return BotDim{nx, nx * ny, per};
    };
    auto down = [&](bool wave, int l, int off) {
        const BotDim d = dim(l);
        const int nx = d.nx, ny = lny[l], nz = lnz[l], m = d.pl * nz;
        float *const r = R + off, *const a = A + off, *const b = B + off, *const w = D + off;
        each(wave, l, off, m, [&](const BotCell &x, int c) { a[c] = r[c] - bot_nb(d, x, c, r); });
        sync(wave);
        each(wave, l, off, m, [&](const BotCell &x, int c) {
            b[c] = r[c] - kC0 * a[c] - kC1 * (a[c] - bot_nb(d, x, c, a));
            w[c] = x.w * b[c];
        });
        sync(wave);
        const int cx = lnx[l + 1], cy = lny[l + 1], mc = cx * cy * lnz[l + 1];
        for (int c = tid; c < mc; c += wave ? 64 : kBotThreads) {
            const int I = c % cx, q0 = c / cx, J = q0 % cy, K = q0 / cy;
            const float *x = w + ((2 * K * ny + 2 * J) * nx + 2 * I);
            const bool i1 = 2 * I + 1 < nx, j1 = 2 * J + 1 < ny, k1 = 2 * K + 1 < nz;
            float sum = x[0] + (i1 ? x[1] : 0.f);
            if (j1) sum += x[nx] + (i1 ? x[nx + 1] : 0.f);
            if (k1) {
                x += d.pl;
                sum += x[0] + (i1 ? x[1] : 0.f);
                if (j1) sum += x[nx] + (i1 ? x[nx + 1] : 0.f);
            }
            R[off + m + c] = sum * low[off + m - m0 + c].iw();
        }
        sync(wave);
        return off + m;
    };
    auto up = [&](bool wave, int l, int off, int m) {
        const BotDim dd = dim(l);
        const float *const e = A + off + m;
        float *const r = R + off, *const a = A + off, *const b = B + off, *const d = D + off;
        each(wave, l, off, m, [&](const BotCell &x, int c) { d[c] = x.w * e[x.bits >> 6]; });
        sync(wave);
        each(wave, l, off, m, [&](const BotCell &x, int c) { b[c] = b[c] - d[c] + bot_nb(dd, x, c, d); });
        sync(wave);
        each(wave, l, off, m, [&](const BotCell &x, int c) {
            const float y = b[c] - bot_nb(dd, x, c, b);
            a[c] = (kC0 * (r[c] + b[c]) + kC1 * (a[c] + y) + d[c]) * x.iw();
        });
        sync(wave);
    };
    const int nb = nl - lb;
    auto size = [&](int l) { return lnx[l] * lny[l] * lnz[l]; };
    int l = 0, off = 0;
    for (; l < nb - 1 && (l == 0 || size(l) > kBotWave); ++l) off = down(false, l, off);
    const int lw = l, offw = off;
    if (tid < 64) {
        for (; l < nb - 1; ++l) off = down(true, l, off);
        {
            // the coarsest level (at most 64 cells): Chebyshev semi-iteration
            // from zero on [kCoarsestMin, kLmax]
            constexpr float theta = 0.5f * (kLmax + kCoarsestMin), delta = 0.5f * (kLmax - kCoarsestMin);
            const BotDim d = dim(l);
            const int m = size(l);
            const BotCell x = nb == 1 ? top[0] : low[off - m0 + min(tid, m - 1)];
            float *const a = A + off;
            const float r = tid < m ? R[off + tid] : 0.f;
            float v = r / theta, dv = v, rho = delta / theta;
#pragma unroll
            for (int it = 1; it < kMgCoarsestDegree; ++it) {
                if (tid < m) a[tid] = v;
                sync(true);
                const float rho1 = 1.f / (2.f * theta / delta - rho);
                if (tid < m) dv = rho1 * rho * dv + 2.f * rho1 / delta * (r - v + bot_nb(d, x, tid, a));
                v += dv;
                rho = rho1;
                sync(true);
            }
            if (tid < m) a[tid] = v * x.iw();
            sync(true);
        }
        for (--l; l >= lw; --l) {
            const int m = size(l);
            off -= m;
            up(true, l, off, m);
        }
    }
    __syncthreads();
    off = offw;
    for (l = lw - 1; l >= 0; --l) {
        const int m = size(l);
        off -= m;
        up(false, l, off, m);
    }
    double f = 0.0;
    if (project) {
        double ew[1] = {0.0};
#pragma unroll
        for (int q = 0; q < kBotPer; ++q) {
            const int c = tid + q * kBotThreads;
            if (c < m0) ew[0] += (double)top[q].w * (double)top[q].w * (double)A[c];
        }
        bot_sum(ew);
        f = pr[1] > 0.0 ? ew[0] / pr[1] : 0.0;
    }
    const gptr<float> e = glob(L0.t);
#pragma unroll
    for (int q = 0; q < kBotPer; ++q) {
        const int c = tid + q * kBotThreads;
        if (c < m0) e[c] = (float)((double)A[c] - f);
    }
}

// ---- residual replacement ---------------------------------------------------

// After k_true_residual: converged, capped, given up, or on.
__global__ __launch_bounds__(kThreads) void k_mg_decide(const ProbDev *__restrict__ P, const int *__restrict__ probs,
                                                        MgStep st)
{
    const int step = st.step;
    const int prob = st.one >= 0 ? st.one : probs[blockIdx.x];
    const ProbDev &pd = P[prob];
    CgScalars *S = st.S + prob;
    const int n = step - pd.n0 + 1;
    if (n < 1 || S->final_ || n != S->next_refresh || !pd.mixed) return;
    const double rrt = block_total_of(pd.P.tres, pd.nt3);
    const double rrs = block_total_of(pd.P.tres + pd.nt3, pd.nt3);
    if (threadIdx.x == 0) {
        const bool finite = rrt >= 0.0 && rrt < 1e300;
        const double before = S->refreshes ? S->prev_rr : S->rr0;
        const bool cap = S->iters >= S->max_iter;
        // one more cycle when only the margin is missing
        const bool conv = finite && (rrt <= kMgMargin * S->thresh ||
                                     (rrt <= S->thresh && (before <= S->thresh || cap)));
        // a cycle that did not halve r.r: counted, and after three in a row
        // the solve goes back to CG from the start
        S->stalls = rrt < 0.5 * before ? 0 : S->stalls + 1;
        S->rr_true = rrt;
        S->refreshes += 1;
        if (!conv && (!finite || S->stalls >= 3)) {
            S->giveup = 1;
            S->final_ = 1;
            S->done_at = n;
        } else if (conv || cap) {
            S->final_ = 1;
            S->status = conv ? 0 : 1;
            S->done_at = n;
        } else {
            S->skip_e_at = step + 1;
            S->rr_after = rrs;
            S->prev_iters = S->iters;
            S->prev_rr = rrt;
            S->next_refresh = kNotDone;
        }
    }
}

// ---- set-up of the hierarchy -------------------------------------------------

__global__ __launch_bounds__(kThreads) void k_mg_weights(long long n, const double *d, const uint8_t *solid, float *w)
{
    const long long stride = (long long)gridDim.x * kThreads;
    for (long long c = (long long)blockIdx.x * kThreads + threadIdx.x; c < n; c += stride)
        w[c] = (solid && solid[c]) ? 0.f : (float)sqrt(d[c]);
}

// ---- connectivity of a masked problem's fluid ---------------------------------
//
// A solid mask can cut the fluid into parts that share no face.  Each part's
// pressure is then known up to a constant of its own, which plain CG keeps at
// the initial guess's; a V-cycle would move it (a coarse cell may join two
// parts).  So the parts are counted, by union-find on the cells with the
// smallest index as the root, and a problem of several goes to plain CG.
// Labels are read and joined with device-scope atomics.
constexpr int kFindLimit = 1 << 20;   // far beyond any path; bounds the loops

__device__ __forceinline__ int label(const int *p, int c)
{
    return __hip_atomic_load(p + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int find_root(int *p, int c)
{
    int a = label(p, c);
    for (int it = 0; it < kFindLimit && a != c; ++it) {
        const int b = label(p, a);
        if (b == a) return a;
        // path halving: c's label moves up (labels only ever decrease)
        __hip_atomic_store(p + c, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        c = a;
        a = b;
    }
    return a;
}

__device__ __forceinline__ void join(int *p, int a, int b)
{
    a = find_root(p, a);
    b = find_root(p, b);
    for (int it = 0; it < kFindLimit && a != b; ++it) {
        const int hi = max(a, b), lo = min(a, b);
        int expect = hi;
        if (__hip_atomic_compare_exchange_strong(p + hi, &expect, lo, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
        a = find_root(p, expect);   // hi was no root any more
        b = lo;
    }
}

// Strip labels: one wave goes through the rows of a strip, 64 cells of x in one
// plane.  A run of fluid cells takes the least label that the row before it
// holds next to it, or else its own first index (solid cells: -1), so labels
// point at the strip's root at once; where a run finds two, they are joined.
// With runs joined row by row instead, the paths grew as long as the grid is
// wide: 444 us over 384x192x128, this and k_mg_join 103 and 67.
__global__ __launch_bounds__(kThreads) void k_mg_label(Geo g, const uint8_t *__restrict__ solid, int *__restrict__ p,
                                                       int *count)
{
    const int nx = g.nx, ny = g.ny, parts = (nx + 63) / 64, lane = threadIdx.x & 63;
    const int t = blockIdx.x * (kThreads / 64) + threadIdx.x / 64;
    if (t == 0 && lane == 0) *count = 0;   // for k_mg_roots
    if (t >= parts * g.nz) return;         // the whole wave
    const int i = t % parts * 64 + lane;
    const long long base = (long long)(t / parts) * ny * nx + i;
    const bool col = i < nx;
    int lab = INT_MAX;               // of the row before; INT_MAX: solid
    unsigned long long before = 0;   // its fluid cells
    constexpr int kRows = 8;         // loaded at a time
    for (int j0 = 0; j0 < ny; j0 += kRows) {
        bool fluids[kRows];
#pragma unroll
        for (int q = 0; q < kRows; ++q) fluids[q] = col && !solid[base + (long long)min(j0 + q, ny - 1) * nx];
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
            if (j0 + q >= ny) break;
            const int c = (int)(base + (long long)(j0 + q) * nx);
            const bool fluid = fluids[q];
            const unsigned long long fl = __ballot(fluid);
            bool two = false;
            int cand = INT_MAX, first = 0;
            if (fl != before) {      // else every run goes on with its label
                const unsigned long long below = ~fl & ((1ull << lane) - 1), above = ~fl >> lane;
                first = below ? 64 - __clzll((long long)below) : 0;
                const int last = fluid ? (above ? lane + __ffsll(above) - 2 : 63) : lane;
                cand = fluid ? lab : INT_MAX;
                int m = cand;
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(m, o);
                    if (lane - o >= first) m = min(m, v);
                }
                m = __shfl(m, last);
                lab = !fluid ? INT_MAX : m == INT_MAX ? c - lane + first : m;
                two = fluid && cand != INT_MAX && cand != lab;
                before = fl;
            }
            if (col) __hip_atomic_store(p + c, fluid ? lab : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__ballot(two)) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
                const int west = __shfl_up(cand, 1);
                if (two && (lane == first || west != cand)) join(p, cand, lab);
            }
        }
    }
}

// Joins the strips with their neighbours on the low side (the first column and
// row also across a periodic side), once for each stretch over which the same
// two labels meet.
__global__ __launch_bounds__(kThreads) void k_mg_join(Geo g, int *p)
{
    const int nx = g.nx, ny = g.ny, parts = (nx + 63) / 64, lane = threadIdx.x & 63;
    const int t = blockIdx.x * (kThreads / 64) + threadIdx.x / 64;
    if (t >= parts * g.nz) return;
    const int i = t % parts * 64 + lane, k = t / parts;
    const long long base = (long long)k * ny * nx + i, plane = (long long)nx * ny;
    const bool col = i < nx;
    int za = -1, zb = -1, xa = -1, xb = -1;   // the last two labels met
    constexpr int kRows = 8;
    for (int j0 = 0; j0 < ny; j0 += kRows) {
        int a[kRows], z[kRows], x[kRows];
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
            const long long c = base + (long long)min(j0 + q, ny - 1) * nx;
            a[q] = col ? label(p, (int)c) : -1;
            z[q] = col && k > 0 ? label(p, (int)(c - plane)) : -1;
            const bool side = lane == 0 && (i > 0 || g.px);
            x[q] = side ? label(p, (int)(i > 0 ? c - 1 : c + nx - 1)) : -1;
        }
#pragma unroll
        for (int q = 0; q < kRows; ++q) {
            if (j0 + q >= ny) break;
            const int aw = __shfl_up(a[q], 1), zw = __shfl_up(z[q], 1);
            if (a[q] >= 0 && z[q] >= 0 && (a[q] != za || z[q] != zb) && (lane == 0 || a[q] != aw || z[q] != zw))
                join(p, a[q], z[q]);
            za = a[q];
            zb = z[q];
            if (a[q] >= 0 && x[q] >= 0 && (a[q] != xa || x[q] != xb)) {
                join(p, a[q], x[q]);
                xa = a[q];
                xb = x[q];
            }
        }
    }
    if (g.py && col) {
        const int a = label(p, (int)base), b = label(p, (int)(base + (long long)(ny - 1) * nx));
        if (a >= 0 && b >= 0) join(p, a, b);
    }
}

__global__ __launch_bounds__(kThreads) void k_mg_roots(long long n, const int *p, int *count)
{
    const long long stride = (long long)gridDim.x * kThreads;
    int roots = 0;
    for (long long c = (long long)blockIdx.x * kThreads + threadIdx.x; c < n; c += stride) roots += p[c] == (int)c;
    if (roots) atomicAdd(count, roots);
}

// One coarse cell: its un-scaled low faces (and the far ones of the last
// column, row and plane), w = sqrt(diagonal) and, on the top plane, the
// diagonal's extra term.  top: un-scaled extra diagonal of a fine top cell
// when the fine level has no array of them: the lid's 2 s_top (lid) or a
// constant (SuLi-IT's free surface).
__device__ __forceinline__ void coarse_cell(const MgLevel &F, const MgLevel &C, int c, int lid, float top)
{
    const int I = c % C.nx, r0 = c / C.nx, J = r0 % C.ny, K = r0 / C.ny;
    const int nx = F.nx, ny = F.ny, nz = F.nz;
    auto at = [&](int i, int j, int k) { return (k * ny + j) * nx + i; };
    // un-scaled fine faces
    auto fx = [&](int f, int j, int k) {
        const int a = f < nx ? f : 0, b = f > 0 ? f - 1 : nx - 1;
        return F.sx[(k * ny + j) * (nx + 1) + f] * F.w[at(a, j, k)] * F.w[at(b, j, k)];
    };
    auto fy = [&](int i, int f, int k) {
        const int a = f < ny ? f : 0, b = f > 0 ? f - 1 : ny - 1;
        return F.sy[(k * (ny + 1) + f) * nx + i] * F.w[at(i, a, k)] * F.w[at(i, b, k)];
    };
    auto fz = [&](int i, int j, int f) {
        return F.sz[(f * ny + j) * nx + i] * F.w[at(i, j, f)] * F.w[at(i, j, max(f - 1, 0))];
    };
    // the two fine cells of a coarse one in each direction; a side of odd
    // length repeats its last, which then does not count.  No load waits for
    // another: with loops over the cells that are there each waited for the one
    // before (a level of 16384 cells 9.3 us, of 2048 8.2; so 5.4 and 5.6).
    const int is[2] = {2 * I, min(2 * I + 1, nx - 1)}, js[2] = {2 * J, min(2 * J + 1, ny - 1)};
    const int ks[2] = {2 * K, min(2 * K + 1, nz - 1)};
    const bool i2 = 2 * I + 1 < nx, j2 = 2 * J + 1 < ny, k2 = 2 * K + 1 < nz;
    // sum of f(0 .. 1, 0 .. 1), second index fastest
    auto quad = [](bool a2, bool b2, auto &&f) {
        const float v00 = f(0, 0), v01 = f(0, 1), v10 = f(1, 0), v11 = f(1, 1);
        float s = v00;
        if (b2) s += v01;
        if (a2) s += v10;
        if (a2 && b2) s += v11;
        return s;
    };
    auto SX = [&](int If) -> float {   // coarse x face If (0 .. C.nx)
        const bool wall = If == 0 || If == C.nx;
        const int f = If == C.nx ? nx : 2 * If;
        const float s = quad(k2, j2, [&](int k, int j) { return fx(f, js[j], ks[k]); });
        return wall && !C.px ? 0.f : 0.5f * s;
    };
    auto SY = [&](int Jf) -> float {
        const bool wall = Jf == 0 || Jf == C.ny;
        const int f = Jf == C.ny ? ny : 2 * Jf;
        const float s = quad(k2, i2, [&](int k, int i) { return fy(is[i], f, ks[k]); });
        return wall && !C.py ? 0.f : 0.5f * s;
    };
    auto SZ = [&](int Kf) -> float {
        const bool wall = Kf == 0 || Kf == C.nz;
        const int f = wall ? 0 : 2 * Kf;
        const float s = quad(j2, i2, [&](int j, int i) { return fz(is[i], js[j], f); });
        return wall ? 0.f : 0.5f * s;
    };
    const float x0 = SX(I), x1 = SX(I + 1), y0 = SY(J), y1 = SY(J + 1), z0 = SZ(K), z1 = SZ(K + 1);
    float ex = 0.f;
    if (K == C.nz - 1) {
        for (int j = 2 * J; j < min(2 * J + 2, ny); ++j)
            for (int i = 2 * I; i < min(2 * I + 2, nx); ++i) {
                if (F.ex) {
                    ex += F.ex[j * nx + i];
                } else if (lid) {
                    const float w = F.w[at(i, j, nz - 1)];
                    ex += 2.f * F.sz[(nz * ny + j) * nx + i] * w * w;
                } else {
                    ex += top;
                }
            }
        C.ex[J * C.nx + I] = ex;
    }
    C.sx[(K * C.ny + J) * (C.nx + 1) + I] = x0;
    if (I == C.nx - 1) C.sx[(K * C.ny + J) * (C.nx + 1) + C.nx] = x1;
    C.sy[(K * (C.ny + 1) + J) * C.nx + I] = y0;
    if (J == C.ny - 1) C.sy[(K * (C.ny + 1) + C.ny) * C.nx + I] = y1;
    C.sz[c] = z0;
    if (K == C.nz - 1) C.sz[c + C.nx * C.ny] = 0.f;
    C.w[c] = sqrtf(x0 + x1 + y0 + y1 + z0 + z1 + ex);
}

// The same cell's faces scaled by the weights on both sides.
__device__ __forceinline__ void scale_cell(const MgLevel &C, int c)
{
    const int nx = C.nx, ny = C.ny;
    const int i = c % nx, r0 = c / nx, j = r0 % ny, k = r0 / ny;
    const float w = C.w[c];
    auto div = [&](float s, float wn) { return s != 0.f ? s / (w * wn) : 0.f; };
    const int fx = (k * ny + j) * (nx + 1) + i, fy = (k * (ny + 1) + j) * nx + i;
    C.sx[fx] = div(C.sx[fx], C.w[i > 0 ? c - 1 : c + nx - 1]);
    if (i == nx - 1) C.sx[fx + 1] = div(C.sx[fx + 1], C.w[c - i]);
    C.sy[fy] = div(C.sy[fy], C.w[j > 0 ? c - nx : c + (ny - 1) * nx]);
    if (j == ny - 1) C.sy[fy + nx] = div(C.sy[fy + nx], C.w[c - j * nx]);
    if (k > 0) C.sz[c] = div(C.sz[c], C.w[c - nx * ny]);
}

__global__ __launch_bounds__(kThreads) void k_mg_coarse(MgLevel F, MgLevel C, int lid, float top)
{
    const int c = blockIdx.x * kThreads + threadIdx.x;
    if (c < C.nx * C.ny * C.nz) coarse_cell(F, C, c, lid, top);
}

__global__ __launch_bounds__(kThreads) void k_mg_scale(MgLevel C)
{
    const int c = blockIdx.x * kThreads + threadIdx.x;
    if (c < C.nx * C.ny * C.nz) scale_cell(C, c);
}

// Levels l0 .. nlev - 1 in one workgroup (each from the one before), and the
// bottom levels' cells packed.
__global__ __launch_bounds__(kBotThreads) void k_mg_coarse_bottom(const ProbDev *__restrict__ P, int l0, int lid, float top)
{
    const ProbDev &pd = *P;
    for (int l = l0; l < pd.nlev; ++l) {
        const MgLevel F = pd.lv[l - 1], C = pd.lv[l];
        const int m = C.nx * C.ny * C.nz;
        for (int c = threadIdx.x; c < m; c += kBotThreads) coarse_cell(F, C, c, lid, top);
        __threadfence_block();
        __syncthreads();
        for (int c = threadIdx.x; c < m; c += kBotThreads) scale_cell(C, c);
        __threadfence_block();
        __syncthreads();
    }
    // the bottom kernel's pack
    int off = 0;
    for (int l = pd.lbot; l < pd.nlev; ++l) {
        const MgLevel L = pd.lv[l];
        const int m = L.nx * L.ny * L.nz;
        BotCell *const out = reinterpret_cast<BotCell *>(pd.bot) + off;
        constexpr int kAhead = 3;   // cells whose loads go together
        for (int c = threadIdx.x; c < m; c += kAhead * kBotThreads) {
            BotCell b[kAhead];
#pragma unroll
            for (int q = 0; q < kAhead; ++q) b[q] = bot_cell(L, min(c + q * kBotThreads, m - 1));
#pragma unroll
            for (int q = 0; q < kAhead; ++q)
                if (c + q * kBotThreads < m) out[c + q * kBotThreads] = b[q];
        }
        off += m;
    }
}

int cells(const MgLevel &L) { return L.nx * L.ny * L.nz; }
int blocks(long long n) { return (int)((n + kThreads - 1) / kThreads); }

}  // namespace

bool mg_plan(const Geo &g, float *w32, float *space, size_t floats, float *scratch, ProbDev &pd, size_t *used)
{
    if (g.n < kMgMinCells || (long long)g.nx * g.ny >= (1LL << 29)) return false;
    // 256-byte aligned; short reads past a row's end stay inside
    struct Take {
        float *p;
        size_t off = 0;
        float *operator()(size_t count)
        {
            float *q = p + off;
            off += (count + 63) / 64 * 64 + 64;
            return q;
        }
    } keep{space}, setup{scratch};
    pd.w32 = w32;
    MgLevel &L0 = pd.lv[0];
    L0 = MgLevel{};
    L0.nx = g.nx;
    L0.ny = g.ny;
    L0.nz = g.nz;
    L0.px = g.px;
    L0.py = g.py;
    L0.sx = const_cast<float *>(pd.sx32);
    L0.sy = const_cast<float *>(pd.sy32);
    L0.sz = const_cast<float *>(pd.sz32);
    L0.w = pd.w32;
    int l = 0, lbot = 0;
    auto coarsest = [&](const MgLevel &L) {
        return cells(L) <= kMgCoarsestCells && std::max({L.nx, L.ny, L.nz}) <= kMgCoarsestSide;
    };
    while (!coarsest(pd.lv[l])) {
        if (l + 1 >= kMgLevels) return false;
        const MgLevel &F = pd.lv[l];
        MgLevel &C = pd.lv[++l];
        C = MgLevel{};
        C.nx = (F.nx + 1) / 2;
        C.ny = (F.ny + 1) / 2;
        C.nz = (F.nz + 1) / 2;
        // a single cell around has no neighbour but itself
        C.px = F.px && C.nx > 1;
        C.py = F.py && C.ny > 1;
    }
    // the bottom kernel starts at the first level whose cells its threads hold
    // and whose hierarchy fits its LDS (four floats per cell, the coefficients
    // of the levels below, two guards)
    for (int b = 1; b <= l && !lbot; ++b) {
        size_t low = 0;
        for (int q = b + 1; q <= l; ++q) low += cells(pd.lv[q]);
        const size_t n = cells(pd.lv[b]);
        if (n <= (size_t)kMgBottomCells &&
            4 * (n + low) + 8 * low + 2 * (size_t)pd.lv[b].nx * pd.lv[b].ny <= (size_t)kMgBottomLds) {
            lbot = b;
            pd.nbot = (int)(n + low);
        }
    }
    if (!lbot) return false;
    // faces and weights of the bottom levels are packed at the end of the
    // set-up: only w of level lbot, its r and its t are read again
    for (int q = 1; q <= l; ++q) {
        MgLevel &C = pd.lv[q];
        const size_t n = (size_t)cells(C);
        Take &t = q < lbot ? keep : setup;
        C.sx = t((size_t)(C.nx + 1) * C.ny * C.nz);
        C.sy = t((size_t)C.nx * (C.ny + 1) * C.nz);
        C.sz = t(n + (size_t)C.nx * C.ny);
        C.ex = t((size_t)C.nx * C.ny);
        C.w = q <= lbot ? keep(n) : setup(n);
        if (q <= lbot) {
            C.r = keep(n);
            C.t = keep(n);
        }
        if (q < lbot) {
            C.rho = keep(n);
        }
    }
    static_assert(sizeof(BotCell) == 8 * sizeof(float), "the pack's size");
    pd.bot = keep(8 * (size_t)pd.nbot);
    // bricks on the fine level (ps_mg.hip: k_mg_brick)
    const int nb = g.n <= kMgBrickCells ? bricks(L0) : 0;
    pd.brick = nb && keep.off + 6 * (size_t)nb + 128 <= 2 * (size_t)g.n;
    if (pd.brick) pd.P.m4 = reinterpret_cast<double *>(keep(6 * (size_t)nb));
    if (used) *used = keep.off;
    if (keep.off > floats || setup.off > (size_t)g.n) return false;
    pd.nlev = l + 1;
    pd.lbot = lbot;
    // rows: 16, 32 or 64 lanes of four cells
    pd.mlrs = g.nx <= 64 ? 4 : g.nx <= 128 ? 5 : 6;
    const int lr = 1 << pd.mlrs;
    pd.mtx = (g.nx + 4 * lr - 1) / (4 * lr);
    const int rows = 8 << (6 - pd.mlrs);   // rows per workgroup
    pd.mty = (g.ny + rows - 1) / rows;
    // planes per tile (even, so that coarse cells are whole): 4, or 8 where
    // that still leaves 512 workgroups, two per CU (a third less z halo: the
    // passes over 384x192x128 took 258 us against 273), or 2 where 4 would
    // leave fewer workgroups than CUs
    const long long cols = (long long)pd.mtx * pd.mty;
    auto tiles = [&](int kz) { return cols * ((g.nz + kz - 1) / kz); };
    const int kz = tiles(8) >= 512 ? 8 : tiles(4) >= 256 ? 4 : 2;
    pd.mkz = kz;
    pd.ntm = pd.brick ? nb : (int)tiles(kz);
    pd.medge = g.px || pd.mtx > 1 || g.nx % 4 != 0;
    pd.mg = 1;
    return true;
}

int mg_level_tiles(const ProbDev &pd, int l) { return l < pd.lbot && (l || pd.brick) ? bricks(pd.lv[l]) : 0; }

void launch_mg_parts(const Geo &g, const uint8_t *solid, int *lab, int *count, hipStream_t s)
{
    const int strips = (g.nx + 63) / 64 * g.nz, grid = (strips + kThreads / 64 - 1) / (kThreads / 64);
    hipLaunchKernelGGL(k_mg_label, dim3(grid), dim3(kThreads), 0, s, g, solid, lab, count);
    hipLaunchKernelGGL(k_mg_join, dim3(grid), dim3(kThreads), 0, s, g, lab);
    hipLaunchKernelGGL(k_mg_roots, dim3(std::min(blocks(g.n), 2048)), dim3(kThreads), 0, s, g.n, lab, count);
}

void launch_mg_setup(const ProbDev &pd, const ProbDev *dev, const SetupIn &in, hipStream_t s)
{
    const long long n = pd.g.n;
    const float top = in.it ? (float)(1.0 / (in.gz * in.tetah * in.dt)) : 0.f;
    hipLaunchKernelGGL(k_mg_weights, dim3(std::min(blocks(n), 4096)), dim3(kThreads), 0, s, n, pd.d, in.solid, pd.w32);
    for (int l = 1; l <= pd.lbot; ++l) {
        const int b = blocks(cells(pd.lv[l]));
        hipLaunchKernelGGL(k_mg_coarse, dim3(b), dim3(kThreads), 0, s, pd.lv[l - 1], pd.lv[l], pd.g.dtop, top);
        hipLaunchKernelGGL(k_mg_scale, dim3(b), dim3(kThreads), 0, s, pd.lv[l]);
    }
    hipLaunchKernelGGL(k_mg_coarse_bottom, dim3(1), dim3(kBotThreads), 0, s, dev, pd.lbot + 1, pd.g.dtop, top);
}

void launch_mg_step(const ProbDev *P, const MgTables &T, int maxgrid, const MgStep &step, int *ran, hipStream_t s)
{
    const int gf = std::min(T.nfine, maxgrid), nb = T.nlev[0], gb = std::min(nb, 4 * maxgrid);
#define MG_FINE(KIND) \
    hipLaunchKernelGGL(k_mg_fine<KIND>, dim3(gf), dim3(kThreads), 0, s, P, T.fine, T.nfine, step, ran)
#define MG_BRICK(KIND) \
    hipLaunchKernelGGL(k_mg_brick<KIND>, dim3(gb), dim3(kThreads), 0, s, P, T.lev[0], nb, step, ran)
#define MG_BOTH(KIND, BRICK)                                                                                        \
    if (gf && gb)                                                                                                   \
        hipLaunchKernelGGL((k_mg_both<KIND, BRICK>), dim3(gf + gb), dim3(kThreads), 0, s, P, T.fine, T.nfine, gb,   \
                           T.lev[0], nb, step, ran);                                                                \
    else if (gf)                                                                                                    \
        MG_FINE(KIND);                                                                                              \
    else                                                                                                            \
        MG_BRICK(BRICK)
#define MG_LEVEL(UP, l)                                                                                           \
    hipLaunchKernelGGL(k_mg_level<UP>, dim3(std::min(T.nlev[l], 4 * maxgrid)), dim3(kThreads), 0, s, P, T.lev[l], \
                       T.nlev[l], l, step)
    if (T.nt1_64)
        hipLaunchKernelGGL(k_mg_upd64, dim3(std::min(T.nt1_64, maxgrid)), dim3(kThreads), 0, s, P, T.t1_64, T.nt1_64,
                           step);
    MG_BOTH(kA1, kDown);
    if (gf) MG_FINE(kA2);
    for (int l = 1; l < kMgLevels; ++l)
        if (T.nlev[l]) MG_LEVEL(false, l);
    hipLaunchKernelGGL(k_mg_bottom, dim3(T.nprobs), dim3(kBotThreads), 0, s, P, T.probs, step);
    for (int l = kMgLevels - 1; l >= 1; --l)
        if (T.nlev[l]) MG_LEVEL(true, l);
    if (gf) MG_FINE(kB1);
    MG_BOTH(kB2, kUp);
    if (T.nt3) {
        MG_BOTH(kDir, kDirB);
        launch_true_residual(P, T.t3, T.nt3, maxgrid, StepRef{nullptr, step.step, nullptr}, s);
        hipLaunchKernelGGL(k_mg_decide, dim3(T.nprobs), dim3(kThreads), 0, s, P, T.probs, step);
    }
    if (T.nt3_64) launch_mg_dir64(P, T.t3_64, T.nt3_64, maxgrid, step, ran, s);
#undef MG_FINE
#undef MG_BRICK
#undef MG_BOTH
#undef MG_LEVEL
}

}  // namespace sps
