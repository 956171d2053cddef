// Multigrid-preconditioned CG of the mixed-precision solver, batched over
// problems.
//
// The scaled system A e = b (unit diagonal, ps_cg.hip) has a condition number
// that grows with the square of the grid's longest side, so plain CG takes
// about a thousand iterations on a 256x128x96 two-phase tank.  Here one
// iteration applies a V-cycle M to the residual first (z = M r, p = z + beta
// p, beta and alpha from r.z) and takes 25 to 50 on any grid.  Everything is
// FP32 inside FP64 residual replacement, as the CG step: dot products, alpha
// and beta are FP64 and convergence is judged on the FP64 true residual.
//
// The V-cycle: a weighted Jacobi sweep before (from z = 0, so z = omega r)
// and after the coarse correction on every level.  A coarse cell joins 2x2x2
// cells; restriction sums the children's residuals, prolongation copies the
// parent's value, and a coarse face's coefficient is half the sum of the fine
// faces it covers (twice the distance).  The cycle is symmetric positive
// definite for any face coefficients >= 0, solid cells and periodic sides
// included.  In the scaled variables of this solver a cell's value is w p
// with w = sqrt(d): restriction weighs with w, prolongation too, and each
// coarse level is scaled to a unit diagonal in the same way (its own w).
//
// Measured at 256x128x96 from prd1 = 0 to 1e-12 relative: plain CG 37.8 ms
// (1992 iterations of one 18.5 us launch), this 7.70 ms (54 iterations); the
// stretched masked cylinder at 384x192x128 248.7 and 24.3 ms, SuLi-IT's
// 256x128x48 19.9 and 6.0 ms, twelve uneven tanks in a batch 72.1 and 11.7 ms.
//
// One iteration n is 4 + 2 lbot launches (lbot levels before the ones the
// bottom kernel takes whole):
//   resid   r_{n-1} = r_{n-2} - alpha q (formed where needed), the residual
//           left by z = omega r restricted to level 1; partials r.r
//   down    the same on levels 1 .. lbot-1
//   bottom  levels lbot and coarser, one workgroup per problem, in LDS
//   up      coarse correction and post-smoothing on levels lbot-1 .. 1
//   smooth  the same on level 0: z_n; partials r.z
//   dir     beta, c -= alpha_{n-1} p_{n-1}, p_n = z + beta p, q = A p;
//           partials p.q
// Each total is summed by the kernel that needs it from the partials of an
// earlier launch, as in ps_cg.hip.
#include <algorithm>

#include "ps_device.h"

namespace sps {
namespace {

// Weight of the Jacobi sweeps.  The scaled operator's spectrum lies in
// (0, 2), so any weight below 1 keeps the V-cycle positive definite.
constexpr float kOmega = 0.85f;
constexpr int kBotThreads = 1024;
constexpr int kBotPer = kMgBottomCells / kBotThreads;

enum { kResid = 0, kSmooth = 1, kDir = 2 };

__device__ __forceinline__ int step_of(StepRef s) { return s.base ? *s.base + s.off : s.off; }

struct Run {
    int begin, end;
};
__device__ __forceinline__ Run my_run(int ntab)
{
    const int G = gridDim.x;
    const long long L = xcd_tile(blockIdx.x, G);
    Run r;
    r.begin = (int)(L * ntab / G);
    r.end = (int)((L + 1) * ntab / G);
    return r;
}

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
// The stencil value v is formed where it is needed from two operands:
//   resid   v = a - s b       a = r_{n-2}, b = q          (fresh: v = a)
//   smooth  v = omega a + w e a = r_{n-1}, e = the parent's correction
//   dir     v = a + s b       a = z, b = p_{n-1}          (fresh: v = a)
// then y = (A v) and, on the tile's cells,
//   resid   r_{n-1} = v; sums w (v - omega y) into the coarse cells
//   smooth  z = v + omega (a - y)
//   dir     p_n = v, q = y, c -= s2 b
// EDGE: rows whose ends need a loaded neighbour (x periodic, or more than one
// segment of 4 lr cells) or whose length is no multiple of four.
template <int KIND, bool EDGE>
__device__ __forceinline__ double mg_tile(const ProbDev &pd, int tile, gptr<const float> __restrict__ a_,
                                          gptr<const float> __restrict__ b_, gptr<float> __restrict__ o1,
                                          gptr<float> __restrict__ o2, gptr<float> __restrict__ x_, bool fresh, float s,
                                          float s2, bool do_x)
{
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
    const gptr<const float> e1 = glob((const float *)C.e), w_ = glob((const float *)pd.w32);
    // cells beyond the segment's ends
    const bool ise = i < nx && (i + 4 >= nx || sl == lr - 1);
    const bool ldw = EDGE && sl == 0 && (i0 > 0 || px), lde = EDGE && ise && (i + 4 < nx || px);
    const int xw = i0 > 0 ? i0 - 1 : nx - 1, xe = i + 4 < nx ? i + 4 : 0;

    auto v_of = [&](float a, float b, float e) -> float {
        if (KIND == kSmooth) return kOmega * a + b * e;
        if (KIND == kResid) return fresh ? a : a - s * b;
        return fresh ? a : a + s * b;
    };
    // four values of a row at plane kk, with their operands
    auto row = [&](int kk, unsigned o, unsigned c, float (&v)[4], float (&a)[4], float (&b)[4]) {
        const gptr<const float> ap = a_ + kk * plane;
        ld4(ap, o, a);
        float e[2] = {0.f, 0.f};
        if (KIND == kSmooth) {
            ld4(w_ + kk * plane, o, b);
            ld2(e1 + (kk >> 1) * cplane, c, e);
        } else {
            ld4(b_ + kk * plane, o, b);
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) v[m] = v_of(a[m], b[m], e[m >> 1]);
    };
    auto one = [&](int kk, int jj, int x) -> float {
        const unsigned o = (unsigned)jj * nx + x;
        const float a = ld1(a_ + kk * plane, o);
        if (KIND == kSmooth)
            return v_of(a, ld1(w_ + kk * plane, o), ld1(e1 + (kk >> 1) * cplane, (unsigned)(jj >> 1) * ncx + (x >> 1)));
        return v_of(a, ld1(b_ + kk * plane, o), 0.f);
    };

    // the rows' table bits for the tile's planes (planes past 32 read the arrays)
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

    float vb[2][4], vc[2][4], ac[2][4], bc[2][4];
    row(k0, oa, ca, vc[0], ac[0], bc[0]);
    row(k0, ob, cb, vc[1], ac[1], bc[1]);
    if (k0 > 0) {
        float t0[4], t1[4];
        row(k0 - 1, oa, ca, vb[0], t0, t1);
        row(k0 - 1, ob, cb, vb[1], t0, t1);
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
        float vt[2][4], at[2][4], bt[2][4], vs[4], vn[4], t0[4], t1[4];
        row(ku, oa, ca, vt[0], at[0], bt[0]);
        row(ku, ob, cb, vt[1], at[1], bt[1]);
        row(k, os, cs, vs, t0, t1);
        row(k, on, cn, vn, t0, t1);
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
        float wx[2][4];
        if (KIND == kResid) {
            ld4(w_ + k * plane, oa, wx[0]);
            ld4(w_ + k * plane, ob, wx[1]);
        }
        if (KIND == kDir) {
            ld4(x_ + k * plane, oa, wx[0]);
            ld4(x_ + k * plane, ob, wx[1]);
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
            if (KIND == kResid) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const bool in = EDGE ? m < nv : nv > 0;
                    const float v = in ? vc[r][m] : 0.f;
                    const float rho = vc[r][m] - kOmega * y[r][m];
                    acc += (double)v * (double)v;
                    sum[m >> 1] += in ? wx[r][m] * rho : 0.f;
                }
                if (!fresh) st4(o1 + k * plane, o, vc[r], nv);
            } else if (KIND == kSmooth) {
                float z[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const bool in = EDGE ? m < nv : nv > 0;
                    z[m] = vc[r][m] + kOmega * (ac[r][m] - y[r][m]);
                    acc += in ? (double)ac[r][m] * (double)z[m] : 0.0;
                }
                st4(o1 + k * plane, o, z, nv);
            } else {
                float c[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const bool in = EDGE ? m < nv : nv > 0;
                    acc += in ? (double)vc[r][m] * (double)y[r][m] : 0.0;
                    c[m] = wx[r][m] - s2 * bc[r][m];
                }
                st4(o1 + k * plane, o, vc[r], nv);
                st4(o2 + k * plane, o, y[r], nv);
                if (do_x) st4(x_ + k * plane, o, c, nv);
            }
        }
        if (KIND == kResid && ((k & 1) || k == nz - 1)) {
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
                ac[r][m] = at[r][m];
                bc[r][m] = bt[r][m];
                szb[r][m] = szt[r][m];
            }
    }
    return acc;
}

template <int KIND>
__global__ __launch_bounds__(kThreads, 2) void k_mg_fine(const ProbDev *__restrict__ P,
                                                         const TileRef *__restrict__ tab, int ntab, StepRef sref,
                                                         int *ran)
{
    const Run run = my_run(ntab);
    const int step = step_of(sref);
    TotalCache tot;
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tab[t];
        const ProbDev &pd = P[tr.prob];
        const gptr<CgScalars> S = glob(pd.S);
        const int n = step - pd.n0 + 1;
        const int done_at = S->done_at, skip_e_at = S->skip_e_at;
        if (n < 1 || n > done_at) continue;
        const bool fresh = n == 1 || step == skip_e_at;   // r_{n-1} stands in its buffer
        double acc = 0.0;
        const bool edge = pd.medge != 0;
        if (KIND == kResid) {
            const double rz = S->rz[(n - 1) & 1];
            const double pq = tot.get(tr.prob, part_pq(pd), pd.ntm);
            const double alpha = fresh || !(pq != 0.0) ? 0.0 : rz / pq;   // 0 / 0 once the residual is 0
            if (tr.tile == 0 && threadIdx.x == 0) S->alpha = alpha;
            const gptr<const float> a = glob((const float *)rbuf(pd, fresh ? n - 1 : n));
            const gptr<const float> b = glob((const float *)pd.q32);
            const gptr<float> o = glob(rbuf(pd, n - 1));
            acc = edge ? mg_tile<KIND, true>(pd, tr.tile, a, b, o, o, o, fresh, (float)alpha, 0.f, false)
                       : mg_tile<KIND, false>(pd, tr.tile, a, b, o, o, o, fresh, (float)alpha, 0.f, false);
        } else if (KIND == kSmooth) {
            const gptr<const float> a = glob((const float *)rbuf(pd, n - 1));
            const gptr<float> o = glob(pd.q32b);
            acc = edge ? mg_tile<KIND, true>(pd, tr.tile, a, a, o, o, o, false, 0.f, 0.f, false)
                       : mg_tile<KIND, false>(pd, tr.tile, a, a, o, o, o, false, 0.f, 0.f, false);
        } else {
            const double rz_prev = S->rz[(n - 1) & 1], alpha = S->alpha;
            const int max_iter = S->max_iter;
            const double rz = tot.get(tr.prob, part_rz(pd), pd.ntm);
            // a breakdown: r.z and p.q are positive for every operator the
            // V-cycle is definite for, unless a value left FP32's range
            const bool bad = !(rz >= 0.0 && rz < 1e300) || !(alpha >= 0.0 && alpha < 1e300);
            const bool cap = n - 1 >= max_iter;
            const double beta = n == 1 || !(rz_prev > 0.0) ? 0.0 : rz / rz_prev;
            if (tr.tile == 0) {
                const double rr = block_total_of(part_rr(pd), pd.ntm);
                if (threadIdx.x == 0) {
                    S->rz[n & 1] = rz;
                    S->rr[n & 1] = rr;
                    S->iters = n - 1;
                    if (bad) {
                        S->giveup = 1;
                        S->final_ = 1;
                        S->done_at = n;
                    } else if (cap) {
                        S->done_at = n;
                    } else if (S->next_refresh == kNotDone) {
                        // r.r (FP32 recurrence) has reached the threshold,
                        // or as far as FP32 carries one cycle
                        const double base = S->refreshes ? S->rr_after : S->rr0;
                        if (rr <= S->thresh || rr <= kMgCycleDrop * base || n - S->prev_iters >= kMgMaxGap)
                            S->next_refresh = n + (n & 1);
                    }
                    if (ran && tr.prob == 0 && !bad && !cap) *ran = 1;
                }
            }
            if (bad) continue;
            const gptr<const float> z = glob((const float *)pd.q32b), po = glob((const float *)mpbuf(pd, n - 1));
            const gptr<float> x = glob(pd.c32);
            if (cap) {
                // finish iteration n - 1 only: c -= alpha p
                if (!fresh) {
                    const float al = (float)alpha;
                    for (long long c = (long long)tr.tile * kThreads + threadIdx.x; c < pd.g.n;
                         c += (long long)pd.ntm * kThreads)
                        x[c] = x[c] - al * po[c];
                }
                continue;
            }
            const gptr<float> pn = glob(mpbuf(pd, n)), q = glob(pd.q32);
            acc = edge ? mg_tile<KIND, true>(pd, tr.tile, z, po, pn, q, x, n == 1, (float)beta, (float)alpha, !fresh)
                       : mg_tile<KIND, false>(pd, tr.tile, z, po, pn, q, x, n == 1, (float)beta, (float)alpha, !fresh);
        }
        const double sres = block_sum(acc);
        if (threadIdx.x == 0) (KIND == kResid ? part_rr(pd) : KIND == kSmooth ? part_rz(pd) : part_pq(pd))[tr.tile] = sres;
    }
}

// ---- coarse levels (l >= 1) -------------------------------------------------

// sum over the six neighbours of s_face f(neighbour); faces at walls hold 0,
// so a clamped neighbour index only has to be valid
template <class F>
__device__ __forceinline__ float nb_sum(const MgLevel &L, int i, int j, int k, F &&f)
{
    const int nx = L.nx, ny = L.ny;
    const int c = (k * ny + j) * nx + i;
    const gptr<const float> sx = glob((const float *)L.sx) + ((k * ny + j) * (nx + 1) + i);
    const gptr<const float> sy = glob((const float *)L.sy) + ((k * (ny + 1) + j) * nx + i);
    const gptr<const float> sz = glob((const float *)L.sz) + c;
    const int cw = c + nb_lo(i, nx, L.px) - i, ce = c + nb_hi(i, nx, L.px) - i;
    const int cs = c + (nb_lo(j, ny, L.py) - j) * nx, cn = c + (nb_hi(j, ny, L.py) - j) * nx;
    const int pl = nx * ny, cb = k > 0 ? c - pl : c, ct = k < L.nz - 1 ? c + pl : c;
    return sx[1] * f(ce, i < nx - 1 ? i + 1 : 0, j, k) + sx[0] * f(cw, i > 0 ? i - 1 : nx - 1, j, k) +
           sy[nx] * f(cn, i, j < ny - 1 ? j + 1 : 0, k) + sy[0] * f(cs, i, j > 0 ? j - 1 : ny - 1, k) +
           sz[pl] * f(ct, i, j, k < L.nz - 1 ? k + 1 : k) + sz[0] * f(cb, i, j, k > 0 ? k - 1 : k);
}

__device__ __forceinline__ bool running(const ProbDev &pd, int step)
{
    const gptr<const CgScalars> S = glob((const CgScalars *)pd.S);
    const int n = step - pd.n0 + 1;
    return n >= 1 && n <= S->done_at;
}

// Level l -> l + 1: a thread per coarse cell sums its children's weighted
// residuals after z = omega r.
__global__ __launch_bounds__(kThreads) void k_mg_down(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab,
                                                      int ntab, int l, StepRef sref)
{
    const Run run = my_run(ntab);
    const int step = step_of(sref);
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tab[t];
        const ProbDev &pd = P[tr.prob];
        if (!running(pd, step)) continue;
        const MgLevel &L = pd.lv[l], &C = pd.lv[l + 1];
        const int c = tr.tile * kThreads + threadIdx.x;
        const int I = c % C.nx, r0 = c / C.nx, J = r0 % C.ny, K = r0 / C.ny;
        if (K >= C.nz) continue;
        const gptr<const float> r = glob((const float *)L.r), w = glob((const float *)L.w);
        float sum = 0.f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int i = 2 * I + (m & 1), j = 2 * J + ((m >> 1) & 1), k = 2 * K + (m >> 2);
            if (i < L.nx && j < L.ny && k < L.nz) {
                const int x = (k * L.ny + j) * L.nx + i;
                const float nb = nb_sum(L, i, j, k, [&](int y, int, int, int) { return r[y]; });
                sum += w[x] * ((1.f - kOmega) * r[x] + kOmega * nb);
            }
        }
        const float wc = C.w[c];
        glob(C.r)[c] = wc > 0.f ? sum / wc : 0.f;
    }
}

// Level l: v = omega r + w (parent's correction), one Jacobi sweep, and the
// correction un-scaled for the level below in the hierarchy.
__global__ __launch_bounds__(kThreads) void k_mg_up(const ProbDev *__restrict__ P, const TileRef *__restrict__ tab,
                                                    int ntab, int l, StepRef sref)
{
    const Run run = my_run(ntab);
    const int step = step_of(sref);
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tab[t];
        const ProbDev &pd = P[tr.prob];
        if (!running(pd, step)) continue;
        const MgLevel &L = pd.lv[l], &C = pd.lv[l + 1];
        const int c = tr.tile * kThreads + threadIdx.x;
        const int i = c % L.nx, r0 = c / L.nx, j = r0 % L.ny, k = r0 / L.ny;
        if (k >= L.nz) continue;
        const gptr<const float> r = glob((const float *)L.r), w = glob((const float *)L.w), e = glob((const float *)C.e);
        auto v = [&](int x, int a, int b, int d) {
            return kOmega * r[x] + w[x] * e[((d >> 1) * C.ny + (b >> 1)) * C.nx + (a >> 1)];
        };
        const float vc = v(c, i, j, k);
        const float nb = nb_sum(L, i, j, k, v);
        const float z = vc + kOmega * (r[c] - vc + nb);
        const float wc = w[c];
        glob(L.e)[c] = wc > 0.f ? z / wc : 0.f;
    }
}

// Sum over the bottom kernel's workgroup, to every thread.
__device__ __forceinline__ double bot_sum(double v)
{
    __shared__ double red[kBotThreads / 64];
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = red[0];
#pragma unroll
    for (int w = 1; w < kBotThreads / 64; ++w) s += red[w];
    return s;
}

// Takes the constant-pressure component out of a level's scaled residual (v
// -= (v.w / w.w) w) or un-scaled correction (v -= (v.w^2 / w.w)).  Where the
// operator has that null space, the coarse levels would amplify the
// component about fourfold each, and the FP32 operator is not exactly (nor
// surely not negatively) singular on it: p.q then went negative at 1e-11
// relative residuals.  Taken out of both sides, the cycle stays symmetric.
__device__ __forceinline__ void drop_null(const MgLevel &L, float *v, bool unscaled)
{
    const int m = L.nx * L.ny * L.nz;
    const gptr<const float> w = glob((const float *)L.w);
    double vw = 0.0, ww = 0.0;
    for (int c = threadIdx.x; c < m; c += kBotThreads) {
        const double wc = w[c];
        vw += (unscaled ? wc * wc : wc) * (double)v[c];
        ww += wc * wc;
    }
    vw = bot_sum(vw);
    ww = bot_sum(ww);
    const double f = ww > 0.0 ? vw / ww : 0.0;
    for (int c = threadIdx.x; c < m; c += kBotThreads) v[c] = (float)((double)v[c] - f * (unscaled ? 1.0 : (double)w[c]));
    __syncthreads();
}

// Levels lbot .. nlev - 1 of one problem in one workgroup: residuals and
// corrections in LDS, coefficients from L2.  zs holds a level's weighted
// residuals on the way down and its corrections on the way up.
__global__ __launch_bounds__(kBotThreads) void k_mg_bottom(const ProbDev *__restrict__ P,
                                                           const int *__restrict__ probs, StepRef sref)
{
    __shared__ float rs[kMgBottomLds], zs[kMgBottomLds];
    const ProbDev &pd = P[probs[blockIdx.x]];
    if (!running(pd, step_of(sref))) return;
    const int tid = threadIdx.x, lb = pd.lbot, nl = pd.nlev;
    {
        const MgLevel &L = pd.lv[lb];
        const int m = L.nx * L.ny * L.nz;
        const gptr<const float> r = glob((const float *)L.r);
        for (int c = tid; c < m; c += kBotThreads) rs[c] = r[c];
    }
    __syncthreads();
    if (pd.S->project) drop_null(pd.lv[lb], rs, false);
    int off = 0;
    for (int l = lb; l < nl - 1; ++l) {
        const MgLevel &L = pd.lv[l], &C = pd.lv[l + 1];
        const int m = L.nx * L.ny * L.nz, mc = C.nx * C.ny * C.nz;
        const float *r = rs + off;
        float *z = zs + off;
        for (int c = tid; c < m; c += kBotThreads) {
            const int i = c % L.nx, r0 = c / L.nx, j = r0 % L.ny, k = r0 / L.ny;
            const float nb = nb_sum(L, i, j, k, [&](int y, int, int, int) { return r[y]; });
            z[c] = L.w[c] * ((1.f - kOmega) * r[c] + kOmega * nb);
        }
        __syncthreads();
        for (int c = tid; c < mc; c += kBotThreads) {
            const int I = c % C.nx, r0 = c / C.nx, J = r0 % C.ny, K = r0 / C.ny;
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = 2 * I + (q & 1), j = 2 * J + ((q >> 1) & 1), k = 2 * K + (q >> 2);
                if (i < L.nx && j < L.ny && k < L.nz) sum += z[(k * L.ny + j) * L.nx + i];
            }
            const float wc = C.w[c];
            rs[off + m + c] = wc > 0.f ? sum / wc : 0.f;
        }
        __syncthreads();
        off += m;
    }
    {
        // the coarsest level: Jacobi sweeps from zero
        const MgLevel &L = pd.lv[nl - 1];
        const int m = L.nx * L.ny * L.nz;   // <= kBotThreads
        const int i = tid % L.nx, r0 = tid / L.nx, j = r0 % L.ny, k = r0 / L.ny;
        const float *r = rs + off;
        float *z = zs + off;
        float v = 0.f;
        if (tid < m) z[tid] = v = kOmega * r[tid];
        __syncthreads();
        for (int it = 1; it < kMgCoarsestSweeps; ++it) {
            if (tid < m) {
                const float nb = nb_sum(L, i, j, k, [&](int y, int, int, int) { return z[y]; });
                v = v + kOmega * (r[tid] - v + nb);
            }
            __syncthreads();
            if (tid < m) z[tid] = v;
            __syncthreads();
        }
        if (tid < m) {
            const float wc = L.w[tid];
            z[tid] = wc > 0.f ? v / wc : 0.f;
        }
        __syncthreads();
    }
    for (int l = nl - 2; l >= lb; --l) {
        const MgLevel &L = pd.lv[l], &C = pd.lv[l + 1];
        const int m = L.nx * L.ny * L.nz;
        const float *ec = zs + off;
        off -= m;
        const float *r = rs + off;
        float *z = zs + off;
        for (int c = tid; c < m; c += kBotThreads) {
            const int i = c % L.nx, r0 = c / L.nx, j = r0 % L.ny, k = r0 / L.ny;
            z[c] = kOmega * r[c] + L.w[c] * ec[((k >> 1) * C.ny + (j >> 1)) * C.nx + (i >> 1)];
        }
        __syncthreads();
        float v[kBotPer];
#pragma unroll
        for (int q = 0; q < kBotPer; ++q) {
            const int c = tid + q * kBotThreads;
            v[q] = 0.f;
            if (c < m) {
                const int i = c % L.nx, r0 = c / L.nx, j = r0 % L.ny, k = r0 / L.ny;
                const float nb = nb_sum(L, i, j, k, [&](int y, int, int, int) { return z[y]; });
                const float wc = L.w[c];
                v[q] = wc > 0.f ? (z[c] + kOmega * (r[c] - z[c] + nb)) / wc : 0.f;
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kBotPer; ++q) {
            const int c = tid + q * kBotThreads;
            if (c < m) z[c] = v[q];
        }
        __syncthreads();
    }
    if (pd.S->project) drop_null(pd.lv[lb], zs, true);
    {
        const MgLevel &L = pd.lv[lb];
        const int m = L.nx * L.ny * L.nz;
        const gptr<float> e = glob(L.e);
        for (int c = tid; c < m; c += kBotThreads) e[c] = zs[c];
    }
}

// ---- residual replacement ---------------------------------------------------

// As refresh_due in ps_cg.hip.
__device__ __forceinline__ bool mg_due(const ProbDev &pd, int step)
{
    const gptr<const CgScalars> S = glob((const CgScalars *)pd.S);
    const int n = step - pd.n0 + 1;
    return n >= 1 && !S->final_ && (n == S->next_refresh || S->done_at != kNotDone);
}

// e += c - alpha_n p_n (alpha_n from the partials of iteration n's kernels), c = 0.
__global__ __launch_bounds__(kThreads) void k_mg_refresh_e(const ProbDev *__restrict__ P,
                                                           const TileRef *__restrict__ tab, int ntab, StepRef sref)
{
    const Run run = my_run(ntab);
    const int step = step_of(sref);
    TotalCache tot;
    for (int t = run.begin; t < run.end; ++t) {
        const TileRef tr = tab[t];
        const ProbDev &pd = P[tr.prob];
        if (!mg_due(pd, step)) continue;
        const gptr<const CgScalars> S = glob((const CgScalars *)pd.S);
        const int n = step - pd.n0 + 1;
        const bool pending = S->done_at == kNotDone;
        const double pq = tot.get(tr.prob, part_pq(pd), pd.ntm);
        const float al = pending && pq != 0.0 ? (float)(S->rz[n & 1] / pq) : 0.f;
        const gptr<const float> p = glob((const float *)mpbuf(pd, n));
        const gptr<double> e = glob(pd.e);
        const gptr<float> c = glob(pd.c32);
        typedef double vd4 __attribute__((ext_vector_type(4)));
        typedef float va4 __attribute__((ext_vector_type(4)));
        const long long len = pd.g.n, nv = len / 4, stride = (long long)pd.nt1 * kThreads;
        for (long long v = (long long)tr.tile * kThreads + threadIdx.x; v < nv; v += stride) {
            va4 cv = ((gptr<const va4>)c)[v];
            const va4 pv = ((gptr<const va4>)p)[v];
            vd4 ev = ((gptr<const vd4>)e)[v];
#pragma unroll
            for (int m = 0; m < 4; ++m) ev[m] += (double)(pending ? cv[m] - al * pv[m] : cv[m]);
            ((gptr<vd4>)e)[v] = ev;
            ((gptr<va4>)c)[v] = va4{0.f, 0.f, 0.f, 0.f};
        }
        if (tr.tile == 0) {
            const long long x = nv * 4 + threadIdx.x;
            if (x < len) {
                e[x] += (double)(pending ? c[x] - al * p[x] : c[x]);
                c[x] = 0.f;
            }
        }
    }
}

// After k_true_residual: converged, capped, given up, or on.
__global__ __launch_bounds__(kThreads) void k_mg_decide(const ProbDev *__restrict__ P, const int *__restrict__ probs,
                                                        StepRef sref)
{
    const int step = step_of(sref);
    const ProbDev &pd = P[probs[blockIdx.x]];
    CgScalars *S = pd.S;
    if (!mg_due(pd, step)) return;
    const int n = step - pd.n0 + 1;
    const double rrt = block_total_of(pd.P.tres, pd.nt3);
    const double rrs = block_total_of(pd.P.tres + pd.nt3, pd.nt3);
    if (threadIdx.x == 0) {
        const bool pending = S->done_at == kNotDone;
        const int iters = pending ? n : S->iters;
        const bool finite = rrt >= 0.0 && rrt < 1e300;
        const bool conv = finite && !(rrt > S->thresh);
        const bool cap = iters >= S->max_iter;
        // a cycle that did not halve r.r: counted, and after three in a row
        // the solve goes back to CG from the start
        const double before = S->refreshes ? S->prev_rr : S->rr0;
        S->stalls = rrt < 0.5 * before ? 0 : S->stalls + 1;
        S->rr_true = rrt;
        S->refreshes += 1;
        S->iters = iters;
        if (!conv && (!finite || S->stalls >= 3)) {
            S->giveup = 1;
            S->final_ = 1;
            if (pending) S->done_at = n;
        } else if (conv || cap) {
            S->final_ = 1;
            S->status = conv ? 0 : 1;
            if (pending) S->done_at = n;
        } else {
            S->skip_e_at = step + 1;
            S->rr_after = rrs;
            S->prev_iters = n;
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

// Label: the start of the cell's run of fluid cells within its 64-cell part
// of the row (-1: solid).  One wave per part.
__global__ __launch_bounds__(kThreads) void k_mg_label(Geo g, const uint8_t *solid, int *p)
{
    const int parts = (g.nx + 63) / 64, lane = threadIdx.x & 63;
    const long long nw = (long long)parts * g.ny * g.nz;
    const long long stride = (long long)gridDim.x * (kThreads / 64);
    for (long long t = (long long)blockIdx.x * (kThreads / 64) + threadIdx.x / 64; t < nw; t += stride) {
        const int i = (int)(t % parts) * 64 + lane;
        const long long row = t / parts * g.nx;
        const bool fluid = i < g.nx && !solid[row + i];
        const unsigned long long fl = __ballot(fluid);
        if (i >= g.nx) continue;
        const unsigned long long below = ~fl & ((1ull << lane) - 1);   // solid lanes below this one
        const int first = below ? 64 - __clzll((long long)below) : 0;
        p[row + i] = fluid ? (int)(row + i) - (lane - first) : -1;
    }
}

// Joins each cell with its neighbours on the low side (the first column and
// row also across a periodic side); within a 64-cell part of a row the
// labels are joined already.
__global__ __launch_bounds__(kThreads) void k_mg_join(Geo g, int *p)
{
    const int nx = g.nx, ny = g.ny;
    const long long stride = (long long)gridDim.x * kThreads;
    for (long long c = (long long)blockIdx.x * kThreads + threadIdx.x; c < g.n; c += stride) {
        if (label(p, (int)c) < 0) continue;
        const int i = (int)(c % nx);
        const long long jk = c / nx;
        const int j = (int)(jk % ny), k = (int)(jk / ny);
        auto with = [&](long long d) {
            if (label(p, (int)d) >= 0) join(p, (int)c, (int)d);
        };
        // one join per run: where the cell to the west and its neighbour are
        // fluid too, they have joined the two runs
        auto run = [&](long long d) {
            const bool west = i > 0 && (i & 63) != 0 && label(p, (int)c - 1) >= 0 && label(p, (int)d - 1) >= 0;
            if (!west) with(d);
        };
        if (i > 0 && (i & 63) == 0) with(c - 1);
        if (i == 0 && g.px) with(c + nx - 1);
        if (j > 0) run(c - nx);
        if (j == 0 && g.py) run(c + (long long)(ny - 1) * nx);
        if (k > 0) run(c - (long long)nx * ny);
    }
}

__global__ __launch_bounds__(kThreads) void k_mg_roots(long long n, const int *p, int *count)
{
    const long long stride = (long long)gridDim.x * kThreads;
    int roots = 0;
    for (long long c = (long long)blockIdx.x * kThreads + threadIdx.x; c < n; c += stride) roots += p[c] == (int)c;
    if (roots) atomicAdd(count, roots);
}

// More than one part: the solve ends here and is set up again as plain CG.
__global__ void k_mg_parts(CgScalars *S)
{
    if (threadIdx.x == 0 && S->parts > 1 && !S->final_) {
        S->giveup = 1;
        S->final_ = 1;
        S->done_at = 0;
    }
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
        return F.sz[(f * ny + j) * nx + i] * F.w[at(i, j, f)] * F.w[at(i, j, f - 1)];
    };
    const int j1 = min(2 * J + 2, ny), k1 = min(2 * K + 2, nz), i1 = min(2 * I + 2, nx);
    auto SX = [&](int If) -> float {   // coarse x face If (0 .. C.nx)
        const bool wall = If == 0 || If == C.nx;
        if (wall && !C.px) return 0.f;
        const int f = If == C.nx ? nx : 2 * If;
        float s = 0.f;
        for (int k = 2 * K; k < k1; ++k)
            for (int j = 2 * J; j < j1; ++j) s += fx(f, j, k);
        return 0.5f * s;
    };
    auto SY = [&](int Jf) -> float {
        const bool wall = Jf == 0 || Jf == C.ny;
        if (wall && !C.py) return 0.f;
        const int f = Jf == C.ny ? ny : 2 * Jf;
        float s = 0.f;
        for (int k = 2 * K; k < k1; ++k)
            for (int i = 2 * I; i < i1; ++i) s += fy(i, f, k);
        return 0.5f * s;
    };
    auto SZ = [&](int Kf) -> float {
        if (Kf == 0 || Kf == C.nz) return 0.f;
        float s = 0.f;
        for (int j = 2 * J; j < j1; ++j)
            for (int i = 2 * I; i < i1; ++i) s += fz(i, j, 2 * Kf);
        return 0.5f * s;
    };
    const float x0 = SX(I), x1 = SX(I + 1), y0 = SY(J), y1 = SY(J + 1), z0 = SZ(K), z1 = SZ(K + 1);
    float ex = 0.f;
    if (K == C.nz - 1) {
        for (int j = 2 * J; j < j1; ++j)
            for (int i = 2 * I; i < i1; ++i) {
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

// Levels lbot .. nlev - 1 in one workgroup (each from the one before).
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
}

int cells(const MgLevel &L) { return L.nx * L.ny * L.nz; }
int blocks(long long n) { return (int)((n + kThreads - 1) / kThreads); }

}  // namespace

bool mg_plan(const Geo &g, bool mixed, float *w32, float *space, size_t floats, ProbDev &pd)
{
    if (!mixed || g.n < kMgMinCells || (long long)g.nx * g.ny >= (1LL << 29)) return false;
    size_t off = 0;
    auto take = [&](size_t count) {
        float *p = space + off;
        off += (count + 63) / 64 * 64 + 64;   // 256-byte aligned; short reads past a row's end stay inside
        return p;
    };
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
    while (cells(pd.lv[l]) > kMgCoarsestCells) {
        if (l + 1 >= kMgLevels) return false;
        const MgLevel &F = pd.lv[l];
        MgLevel &C = pd.lv[l + 1];
        C = MgLevel{};
        C.nx = (F.nx + 1) / 2;
        C.ny = (F.ny + 1) / 2;
        C.nz = (F.nz + 1) / 2;
        // a single cell around has no neighbour but itself
        C.px = F.px && C.nx > 1;
        C.py = F.py && C.ny > 1;
        const size_t n = (size_t)cells(C);
        C.sx = take((size_t)(C.nx + 1) * C.ny * C.nz);
        C.sy = take((size_t)C.nx * (C.ny + 1) * C.nz);
        C.sz = take(n + (size_t)C.nx * C.ny);
        C.w = take(n);
        C.r = take(n);
        C.e = take(n);
        C.ex = take((size_t)C.nx * C.ny);
        ++l;
        if (!lbot && n <= (size_t)kMgBottomCells) lbot = l;
    }
    if (!lbot || off > floats) return false;
    size_t lds = 0;
    for (int q = lbot; q <= l; ++q) lds += cells(pd.lv[q]);
    if (lds > (size_t)kMgBottomLds) return false;
    pd.nlev = l + 1;
    pd.lbot = lbot;
    // rows: 16, 32 or 64 lanes of four cells
    pd.mlrs = g.nx <= 64 ? 4 : g.nx <= 128 ? 5 : 6;
    const int lr = 1 << pd.mlrs;
    pd.mtx = (g.nx + 4 * lr - 1) / (4 * lr);
    const int rows = 8 << (6 - pd.mlrs);   // rows per workgroup
    pd.mty = (g.ny + rows - 1) / rows;
    // planes per tile (even, so that coarse cells are whole): thin while that
    // leaves fewer than kMgTiles workgroups
    const long long cols = (long long)pd.mtx * pd.mty;
    long long kz = cols * g.nz / kMgTiles / 2 * 2;
    kz = std::max<long long>(2, std::min<long long>(kz, 16));
    pd.mkz = (int)kz;
    pd.ntm = (int)(cols * ((g.nz + kz - 1) / kz));
    pd.medge = g.px || pd.mtx > 1 || g.nx % 4 != 0;
    pd.mg = 1;
    return true;
}

int mg_down_tiles(const ProbDev &pd, int l) { return l >= 1 && l < pd.lbot ? blocks(cells(pd.lv[l + 1])) : 0; }
int mg_up_tiles(const ProbDev &pd, int l) { return l >= 1 && l < pd.lbot ? blocks(cells(pd.lv[l])) : 0; }

void launch_mg_setup(const ProbDev &pd, const ProbDev *dev, const SetupIn &in, hipStream_t s)
{
    const long long n = pd.g.n;
    const float top = in.it ? (float)(1.0 / (in.gz * in.tetah * in.dt)) : 0.f;
    if (in.solid) {
        int *lab = reinterpret_cast<int *>(pd.q32b);
        hipLaunchKernelGGL(k_mg_label, dim3(std::min(blocks(n), 4096)), dim3(kThreads), 0, s, pd.g, in.solid, lab);
        hipLaunchKernelGGL(k_mg_join, dim3(std::min(blocks(n), 16384)), dim3(kThreads), 0, s, pd.g, lab);
        hipLaunchKernelGGL(k_mg_roots, dim3(std::min(blocks(n), 2048)), dim3(kThreads), 0, s, n, lab, &pd.S->parts);
        hipLaunchKernelGGL(k_mg_parts, dim3(1), dim3(64), 0, s, pd.S);
    }
    hipLaunchKernelGGL(k_mg_weights, dim3(std::min(blocks(n), 4096)), dim3(kThreads), 0, s, n, pd.d, in.solid, pd.w32);
    for (int l = 1; l < pd.lbot; ++l) {
        const int b = blocks(cells(pd.lv[l]));
        hipLaunchKernelGGL(k_mg_coarse, dim3(b), dim3(kThreads), 0, s, pd.lv[l - 1], pd.lv[l], pd.g.dtop, top);
        hipLaunchKernelGGL(k_mg_scale, dim3(b), dim3(kThreads), 0, s, pd.lv[l]);
    }
    hipLaunchKernelGGL(k_mg_coarse_bottom, dim3(1), dim3(kBotThreads), 0, s, dev, pd.lbot, pd.g.dtop, top);
}

void launch_mg_step(const ProbDev *P, const MgTables &T, int maxgrid, StepRef step, int *ran, hipStream_t s)
{
    const int grid = std::min(T.nfine, maxgrid);
    hipLaunchKernelGGL(k_mg_fine<kResid>, dim3(grid), dim3(kThreads), 0, s, P, T.fine, T.nfine, step, nullptr);
    for (int l = 1; l < kMgLevels; ++l)
        if (T.ndown[l])
            hipLaunchKernelGGL(k_mg_down, dim3(std::min(T.ndown[l], maxgrid)), dim3(kThreads), 0, s, P, T.down[l],
                               T.ndown[l], l, step);
    hipLaunchKernelGGL(k_mg_bottom, dim3(T.nprobs), dim3(kBotThreads), 0, s, P, T.probs, step);
    for (int l = kMgLevels - 1; l >= 1; --l)
        if (T.nup[l])
            hipLaunchKernelGGL(k_mg_up, dim3(std::min(T.nup[l], maxgrid)), dim3(kThreads), 0, s, P, T.up[l], T.nup[l],
                               l, step);
    hipLaunchKernelGGL(k_mg_fine<kSmooth>, dim3(grid), dim3(kThreads), 0, s, P, T.fine, T.nfine, step, nullptr);
    hipLaunchKernelGGL(k_mg_fine<kDir>, dim3(grid), dim3(kThreads), 0, s, P, T.fine, T.nfine, step, ran);
}

void launch_mg_refresh(const ProbDev *P, const TileRef *t1, int nt1, const TileRef *t3, int nt3, const int *probs,
                       int nprobs, int maxgrid, StepRef step, hipStream_t s)
{
    hipLaunchKernelGGL(k_mg_refresh_e, dim3(std::min(maxgrid, nt1)), dim3(kThreads), 0, s, P, t1, nt1, step);
    launch_true_residual(P, t3, nt3, maxgrid, step, s);
    hipLaunchKernelGGL(k_mg_decide, dim3(nprobs), dim3(kThreads), 0, s, P, probs, step);
}

}  // namespace sps
