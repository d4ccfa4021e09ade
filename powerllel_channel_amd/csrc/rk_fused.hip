// RK1 and RK2 of one time step in one pass over the velocity (gfx950).
//
// Restates timeIntVelRK1/RK2 (src/mod_calcVel.f90:52-426) with the boundary
// fill of the RK1 stage in between (src/mod_updateBound.f90:30-108), in the
// roundings of the separate kernels (step_kernels.hip); compiled with
// -ffp-contract=off like them.  The RK1 stage lives in LDS only: each
// workgroup computes it one cell beyond its tile on every side (the halo
// cells twice or more over the grid), so a step reads the velocity once and
// writes it once, to other arrays (a neighbour's input must not be
// overwritten).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mom_rhs.h"
#include "pll_internal.h"

namespace {

using pll::G;
using pll::make_g;
using pll::zm;

// periodic index in 1..n of any haloed index
__device__ __forceinline__ int wrapn(int i, int n)
{
    const int r = (i - 1) % n;
    return (r < 0 ? r + n : r) + 1;
}

// element at a byte offset from a uniform base (scalar base, 32-bit offset)
__device__ __forceinline__ double at(const double *b, unsigned o)
{
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(b) + o);
}
__device__ __forceinline__ void set(double *b, unsigned o, double x)
{
    *reinterpret_cast<double *>(reinterpret_cast<char *>(b) + o) = x;
}

struct Body {
    const double *u, *v, *w;
};

// Projection of the input as it is read: correctVel with the forcing shift
// and the boundary fill.
struct Proj {
    const double *p;
    double dtdxi, dtdyi;
    int fmask;
    double vfu, vfv;
    const double *mean;
};

struct Tiles {
    int ntx, nty, nkc, kc;
    int xcd;
    // Mean_h partials are those of the RK2 kernel: one per 64 x 4 x kc4 tile
    // (kc a multiple of kc4), at that kernel's workgroup index
    int nty4, nkc4, kc4, xcd4;
};

// Fluxes through the upper z face of a cell, carried from plane k to plane
// k + 1, where they are the lower face's: products and differences commute
// bit for bit with the ones mom_rhs forms there.
struct ZFlux {
    double cu, cv, cw;  // ut wt, wt vt, wt wt
    double du, dv, dw;  // dqt of u, v, w
};

struct ZMet {
    double f_k, f_kp, fi_k, fi_kp, ci_k;
};
__device__ __forceinline__ ZMet zmet(const G &g, int k)
{
    return ZMet{zm(g.dzf, k), zm(g.dzf, k + 1), zm(g.dzf_inv, k), zm(g.dzf_inv, k + 1),
                zm(g.dzc_inv, k)};
}

// plane k in cu, cv, cw and plane k + 1 in nu, nv, nw at cell c
__device__ __forceinline__ ZFlux zflux(const ZMet &z, const double *cu, const double *cv,
                                       const double *cw, const double *nu, const double *nv,
                                       const double *nw, int c, int sx, int sy)
{
    ZFlux f;
    const double u = cu[c], v = cv[c], w = cw[c], un = nu[c], vn = nv[c], wn = nw[c];
    f.cu = ((u * z.f_kp + un * z.f_k) * z.ci_k) * (w + cw[c + sx]);
    f.cv = (w + cw[c + sy]) * ((v * z.f_kp + vn * z.f_k) * z.ci_k);
    f.cw = (w + wn) * (w + wn);
    f.du = (un - u) * z.ci_k;
    f.dv = (vn - v) * z.ci_k;
    f.dw = (wn - w) * z.fi_kp;
    return f;
}

// mom_rhs (mom_rhs.h) at cell c with the lower z fluxes given in b; returns
// the upper ones.
__device__ __forceinline__ ZFlux rhs_tile(const G &g, const ZMet &z, const double *cu,
                                          const double *cv, const double *cw, const double *nu,
                                          const double *nv, const double *nw, int c, int sx,
                                          int sy, const ZFlux &b, double &fu,
                                          double &fv, double &fw)
{
    const double dx_inv = g.dx_inv, dy_inv = g.dy_inv, re_inv = g.re_inv, u_crf = g.u_crf;
    const double u000 = cu[c], up00 = cu[c + sx], um00 = cu[c - sx], u0p0 = cu[c + sy],
                 u0m0 = cu[c - sy], ump0 = cu[c - sx + sy], u00p = nu[c], um0p = nu[c - sx];
    const double v000 = cv[c], vp00 = cv[c + sx], vm00 = cv[c - sx], v0p0 = cv[c + sy],
                 v0m0 = cv[c - sy], vpm0 = cv[c + sx - sy], v00p = nv[c], v0mp = nv[c - sy];
    const double w000 = cw[c], wp00 = cw[c + sx], wm00 = cw[c - sx], w0p0 = cw[c + sy],
                 w0m0 = cw[c - sy], w00p = nw[c];
    ZFlux t;
    double conv, visc;
    // u
    const double ue = u000 + up00, uw = um00 + u000, un = u000 + u0p0, us = u0m0 + u000;
    const double ut = (u000 * z.f_kp + u00p * z.f_k) * z.ci_k;
    const double vn1 = v000 + vp00, vs1 = v0m0 + vpm0;
    const double wt1 = w000 + wp00;
    t.cu = ut * wt1;
    t.du = (u00p - u000) * z.ci_k;
    double dqe = (up00 - u000) * dx_inv, dqw = (u000 - um00) * dx_inv;
    double dqn = (u0p0 - u000) * dy_inv, dqs = (u000 - u0m0) * dy_inv;
    conv = 0.25 * ((ue * ue - uw * uw) * dx_inv + (un * vn1 - us * vs1) * dy_inv +
                   (t.cu - b.cu) * z.fi_k);
    conv = conv + 0.5 * u_crf * (ue - uw) * dx_inv;
    visc = ((dqe - dqw) * dx_inv + (dqn - dqs) * dy_inv + (t.du - b.du) * z.fi_k) * re_inv;
    fu = visc - conv;
    __builtin_amdgcn_sched_barrier(0);  // one equation's operands in registers at a time
    // v
    const double vw2 = vm00 + v000, vn2 = v000 + v0p0, vs2 = v0m0 + v000;
    const double vt = (v000 * z.f_kp + v00p * z.f_k) * z.ci_k;
    const double uw2 = um00 + ump0;
    const double wt2 = w000 + w0p0;
    t.cv = wt2 * vt;
    t.dv = (v00p - v000) * z.ci_k;
    dqe = (vp00 - v000) * dx_inv;
    dqw = (v000 - vm00) * dx_inv;
    dqn = (v0p0 - v000) * dy_inv;
    dqs = (v000 - v0m0) * dy_inv;
    conv = 0.25 * ((un * vn1 - uw2 * vw2) * dx_inv + (vn2 * vn2 - vs2 * vs2) * dy_inv +
                   (t.cv - b.cv) * z.fi_k);
    conv = conv + 0.5 * u_crf * (vn1 - vw2) * dx_inv;
    visc = ((dqe - dqw) * dx_inv + (dqn - dqs) * dy_inv + (t.dv - b.dv) * z.fi_k) * re_inv;
    fv = visc - conv;
    __builtin_amdgcn_sched_barrier(0);
    // w
    const double ww3 = wm00 + w000, ws3 = w0m0 + w000;
    const double wt3 = w000 + w00p;
    const double uw3 = (um00 * z.f_kp + um0p * z.f_k) * z.ci_k;
    const double vs3 = (v0m0 * z.f_kp + v0mp * z.f_k) * z.ci_k;
    t.cw = wt3 * wt3;
    t.dw = (w00p - w000) * z.fi_kp;
    dqe = (wp00 - w000) * dx_inv;
    dqw = (w000 - wm00) * dx_inv;
    dqn = (w0p0 - w000) * dy_inv;
    dqs = (w000 - w0m0) * dy_inv;
    conv = 0.25 * ((ut * wt1 - uw3 * ww3) * dx_inv + (vt * wt2 - vs3 * ws3) * dy_inv +
                   (t.cw - b.cw) * z.ci_k);
    conv = conv + 0.5 * u_crf * (wt1 - ww3) * dx_inv;
    visc = ((dqe - dqw) * dx_inv + (dqn - dqs) * dy_inv + (t.dw - b.dw) * z.ci_k) * re_inv;
    fw = visc - conv;
    return t;
}

// A workgroup owns 64 x TY columns and marches over a chunk of k:
//   A  the input velocity of plane k + 2 (tile plus two cells on every side)
//      is loaded into registers while plane k is computed, then projected
//      (PROJ) and written to LDS; two planes live there;
//   B  the RK1 stage of plane k on the tile plus one cell, from LDS to LDS
//      (two planes);
//   C  RK2 of plane k - 1 on the tile, to memory.
// The z fluxes of B and C are carried in registers from plane to plane, and
// so is the old velocity RK2 averages with.  No lane is masked except in the
// second round of B: indices wrap periodically, so lanes beyond the grid
// compute and store copies of the values their owners store.
//
// Per cell 56 bytes (PROJ: u, v, w, p read, u, v, w written), where the
// separate projecting kernels moved 136; about 350 FP64 operations, the RK1
// stage's halo included, and 80 eight-byte LDS accesses.  Each of the three
// (HBM, FP64 issue, LDS) takes 0.6 to 0.9 ms of the 1.6 at 768x384x256 (2.5 ms
// before), the two barriers per plane keep them from overlapping further.
// 64 x 12 columns because the RK1 halo costs by the wave: 924 cells are 15
// waves for 12 (x 8: 11 for 8, x 4: 7 for 4), and 168 registers allow 12 waves
// per CU; five steps at 768x384x256 take 16.5 ms with 64 x 12, 17.2 with
// 64 x 8 (8 waves), 17.9 with 64 x 4, and 25 to 28 with 64 x 8 or 64 x 16 held
// at 128 registers for 16 waves, which spills.
constexpr int TY = 12;

// SUB: the chunk holds several of the partials' chunks (kc > kc4).
template <bool PROJ, bool MEAN, bool SUB, bool BODY = !PROJ>
__global__ void __launch_bounds__(64 * TY, 3)
k_rk12(G g, Tiles t, const double *__restrict__ qu, const double *__restrict__ qv,
       const double *__restrict__ qw, double *__restrict__ ou, double *__restrict__ ov,
       double *__restrict__ ow, double *__restrict__ mpart, int fmask, Body fb, Proj pr)
{
    constexpr int NT = 64 * TY;
    constexpr int QX = 68, QY = TY + 4, NQ = QX * QY;            // input tile
    constexpr int PX = PROJ ? QX + 1 : QX, PY = PROJ ? QY + 1 : QY, NP = PX * PY;  // loads
    constexpr int BX = 66, BY = TY + 2, NB = BX * BY;            // RK1 tile
    constexpr int NR = (NP + NT - 1) / NT, NBR = (NB + NT - 1) / NT;
    __shared__ double tq[2][3][NQ + 1];  // the last slot takes lanes outside the tile
    __shared__ double tb[2][3][NB];
    __shared__ double tp[PROJ ? NP : 1];
    __shared__ double red[MEAN ? 2 * NT : 1];  // Mean_h sums of each lane (kept out of registers)

    int lb = blockIdx.x;
    if (t.xcd) lb = (lb & 7) * (int)(gridDim.x >> 3) + (lb >> 3);
    const int tx = lb % t.ntx;
    lb /= t.ntx;
    const int ty = lb % t.nty, kc = lb / t.nty;
    const int tid = threadIdx.x, lx = tid & 63, ly = tid >> 6;
    const int i0 = tx * 64, j0 = ty * TY;
    const int k0 = kc * t.kc + 1, k1 = min(k0 + t.kc - 1, g.nz);
    const int sy = (int)g.sy, nz = g.nz;
    const long long sz = g.sz;
    const double bcu = 0.0 - g.u_crf;

    unsigned off[NR];  // byte offset in a plane
    int sl[NR];  // LDS slots: input tile, pressure tile << 16
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int c = min(tid + r * NT, NP - 1), row = c / PX, col = c - row * PX;
        const bool in = col < QX && row < QY;
        off[r] = 8u * (unsigned)(wrapn(i0 - 1 + col, g.nx) + sy * wrapn(j0 - 1 + row, g.ny));
        sl[r] = in ? (row * QX + col) | (c << 16) : NQ;
    }
    double pu[NR], pv[NR], pw[NR], pn[NR];
    auto fetch = [&](int kp) {
        // PROJ: the plane that kp's values are formed from (the first or last
        // interior plane for the walls' ghosts), and p of the next such plane
        const int ks = PROJ ? min(max(kp, 1), nz) : min(kp, nz + 1);
        const double *bu = qu + sz * ks, *bv = qv + sz * ks, *bw = qw + sz * ks;
        // the lane offsets are opaque here, or the compiler would hoist a
        // 64-bit lane address per array out of the k loop (22 registers)
#pragma unroll
        for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(off[r]));
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            pu[r] = at(bu, off[r]);
            pv[r] = at(bv, off[r]);
            pw[r] = at(bw, off[r]);
        }
        if (PROJ) {
            const double *bp = pr.p + sz * min(max(kp + 1, 1), nz);
#pragma unroll
            for (int r = 0; r < NR; ++r) pn[r] = at(bp, off[r]);
        }
    };
    auto put_p = [&]() {
        if (PROJ) {
#pragma unroll
            for (int r = 0; r < NR; ++r) tp[min(tid + r * NT, NP - 1)] = pn[r];
        }
    };
    const double shu = (PROJ && (pr.fmask & 1)) ? pr.vfu - pr.mean[0] : 0.0;
    const double shv = (PROJ && (pr.fmask & 2)) ? pr.vfv - pr.mean[1] : 0.0;
    const bool fu_on = PROJ && (pr.fmask & 1), fv_on = PROJ && (pr.fmask & 2);
    // plane kp (fetched last) into LDS; tp holds p of its source plane
    auto put = [&](int kp, int b) {
        const bool wall = kp <= 0 || kp > nz;
        const int ks = min(max(kp, 1), nz);
        const double dzi = PROJ ? zm(g.dzc_inv, ks) : 0.0;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            double un = pu[r], vn = pv[r], wn = pw[r];
            if (PROJ) {
                const double *P = tp + (sl[r] >> 16);
                const double pc = P[0];
                un = un - (P[1] - pc) * pr.dtdxi;
                vn = vn - (P[PX] - pc) * pr.dtdyi;
                un = fu_on ? un + shu : un;
                vn = fv_on ? vn + shv : vn;
                wn = wn - (pn[r] - pc) * g.dt * dzi;
                un = wall ? 2.0 * bcu - un : un;
                vn = wall ? 2.0 * 0.0 - vn : vn;
                wn = (wall || kp == nz) ? 0.0 : wn;
            }
            const int l = sl[r] & 0xffff;
            tq[b][0][l] = un;
            tq[b][1][l] = vn;
            tq[b][2][l] = wn;
        }
    };

    int bc[NBR];
    unsigned bo[NBR];  // B cells: centre in the input tile, offset in a plane
#pragma unroll
    for (int r = 0; r < NBR; ++r) {
        const int c = min(tid + r * NT, NB - 1), row = c / BX, col = c - row * BX;
        bc[r] = (row + 1) * QX + col + 1;
        if (BODY) bo[r] = 8u * (unsigned)(wrapn(i0 + col, g.nx) + sy * wrapn(j0 + row, g.ny));
    }
    const int cc = (ly + 1) * BX + lx + 1, cq = (ly + 2) * QX + lx + 2;
    unsigned eo = 8u * (unsigned)(wrapn(i0 + lx + 1, g.nx) + sy * wrapn(j0 + ly + 1, g.ny));

    // plane k of the input and of the RK1 stage lives in slot (k - k0) & 1
    const int kbs = k0 == 1 ? 1 : k0 - 1;  // first plane of the RK1 stage
    const int sb = k0 == 1 ? 0 : 1;        // its slot
    if (PROJ) fetch(kbs - 2);  // its p: the source plane of plane kbs - 1
    put_p();
    fetch(kbs - 1);
    __syncthreads();
    put(kbs - 1, sb ^ 1);
    __syncthreads();
    put_p();
    fetch(kbs);
    __syncthreads();
    put(kbs, sb);
    __syncthreads();
    put_p();
    fetch(kbs + 1);
    ZFlux zb[NBR], zc{};
    {
        const int a = sb ^ 1;
        const ZMet z = zmet(g, kbs - 1);
#pragma unroll
        for (int r = 0; r < NBR; ++r)
            zb[r] = zflux(z, tq[a][0], tq[a][1], tq[a][2], tq[a ^ 1][0], tq[a ^ 1][1], tq[a ^ 1][2],
                          bc[r], 1, QX);
    }
    __syncthreads();
    put(kbs + 1, sb ^ 1);
    __syncthreads();
    double oldu = 0.0, oldv = 0.0, oldw = 0.0;
    if (MEAN) red[tid] = red[NT + tid] = 0.0;

    const bool own = i0 + lx + 1 <= g.nx && j0 + ly + 1 <= g.ny;
    // the partials of a chunk of kc4 planes that ends with plane k, in the order
    // of the RK2 kernel's reduction
    auto emit = [&](int k) {
        if (!own) red[tid] = red[NT + tid] = 0.0;
        __syncthreads();
        const int q = tid & 255, base = tid - q;
        for (int h = 128; h > 0; h >>= 1) {
            if (q < h) {
                red[base + q] += red[base + q + h];
                red[NT + base + q] += red[NT + base + q + h];
            }
            __syncthreads();
        }
        const int ty4 = ty * (TY / 4) + (tid >> 8);
        if (q == 0 && ty4 < t.nty4) {
            const int nb = t.ntx * t.nty4 * t.nkc4;
            int b4 = ((k - 1) / t.kc4 * t.nty4 + ty4) * t.ntx + tx;
            if (t.xcd4) b4 = (b4 % (nb >> 3)) * 8 + b4 / (nb >> 3);
            mpart[b4] = (fmask & 1) ? red[base] : 0.0;
            mpart[nb + b4] = (fmask & 2) ? red[NT + base] : 0.0;
        }
        if (SUB) red[tid] = red[NT + tid] = 0.0;
    };

    // RK1 stage of plane kb (slot PAR) into LDS; MODE 2: then RK2 of plane kb - 1,
    // 1: its lower z fluxes, 0: neither; 3: as 2 with kb the wall's ghost plane
    // nz + 1.  Loads of plane kb + 2 throughout.
    auto iter = [&](int kv, auto MODE, auto PAR) {
        constexpr int mode = decltype(MODE)::value, a = decltype(PAR)::value;
        const int kb = __builtin_amdgcn_readfirstlane(kv);
        asm volatile("" : "+v"(eo));
        double fbu[NBR], fbv[NBR], fbw[NBR], cbu = 0.0, cbv = 0.0, cbw = 0.0;
        if (BODY) {
            const long long e = sz * min(kb, nz), ec = sz * (kb - 1);
#pragma unroll
            for (int r = 0; r < NBR; ++r) {
                asm volatile("" : "+v"(bo[r]));
                fbu[r] = at(fb.u + e, bo[r]);
                fbv[r] = at(fb.v + e, bo[r]);
                fbw[r] = at(fb.w + e, bo[r]);
            }
            if (mode >= 2) {
                cbu = at(fb.u + ec, eo);
                cbv = at(fb.v + ec, eo);
                cbw = at(fb.w + ec, eo);
            }
        }
        put_p();
        fetch(min(kb + 2, k1 + 2));
        // keep the loads ahead of the arithmetic
        __builtin_amdgcn_sched_barrier(0);
        // B
        if constexpr (mode != 3) {
            const ZMet z = zmet(g, kb);
#pragma unroll
            for (int r = 0; r < NBR; ++r) {
                const int c = tid + r * NT;
                if (r == 0 || c < NB) {
                    double f0, f1, f2;
                    zb[r] = rhs_tile(g, z, tq[a][0], tq[a][1], tq[a][2], tq[a ^ 1][0],
                                     tq[a ^ 1][1], tq[a ^ 1][2], bc[r], 1, QX, zb[r], f0, f1, f2);
                    if (BODY) {
                        f0 = f0 + fbu[r];
                        f1 = f1 + fbv[r];
                        f2 = f2 + fbw[r];
                    }
                    tb[a][0][c] = tq[a][0][bc[r]] + g.dt * f0;
                    tb[a][1][c] = tq[a][1][bc[r]] + g.dt * f1;
                    tb[a][2][c] = kb == nz ? 0.0 : tq[a][2][bc[r]] + g.dt * f2;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < NBR; ++r) {
                const int c = tid + r * NT;
                if (r == 0 || c < NB) {
                    tb[a][0][c] = 2.0 * bcu - tb[a ^ 1][0][c];
                    tb[a][1][c] = 2.0 * 0.0 - tb[a ^ 1][1][c];
                    tb[a][2][c] = 0.0;
                }
            }
        }
        const double nou = tq[a][0][cq], nov = tq[a][1][cq], now = tq[a][2][cq];
        __syncthreads();
        // C
        if (mode == 1) {
            if (kb == 1) {
                // below the first plane: the wall's ghosts of the RK1 stage
                const ZMet z = zmet(g, 0);
                const double u = tb[a][0][cc], v = tb[a][1][cc], w = tb[a][2][cc];
                const double um = 2.0 * bcu - u, vm = 2.0 * 0.0 - v;
                zc.cu = ((um * z.f_kp + u * z.f_k) * z.ci_k) * 0.0;
                zc.cv = 0.0 * ((vm * z.f_kp + v * z.f_k) * z.ci_k);
                zc.cw = w * w;
                zc.du = (u - um) * z.ci_k;
                zc.dv = (v - vm) * z.ci_k;
                zc.dw = w * z.fi_kp;
            } else {
                zc = zflux(zmet(g, kb - 1), tb[a ^ 1][0], tb[a ^ 1][1], tb[a ^ 1][2], tb[a][0],
                           tb[a][1], tb[a][2], cc, 1, BX);
            }
        }
        if (mode >= 2) {
            const ZMet z = zmet(g, kb - 1);
            double f0, f1, f2;
            zc = rhs_tile(g, z, tb[a ^ 1][0], tb[a ^ 1][1], tb[a ^ 1][2], tb[a][0], tb[a][1],
                          tb[a][2], cc, 1, BX, zc, f0, f1, f2);
            if (BODY) {
                f0 = f0 + cbu;
                f1 = f1 + cbv;
                f2 = f2 + cbw;
            }
            const double un = (tb[a ^ 1][0][cc] + g.dt * f0 + oldu) * 0.5;
            const double vn = (tb[a ^ 1][1][cc] + g.dt * f1 + oldv) * 0.5;
            const long long e = sz * (kb - 1);
            set(ou + e, eo, un);
            set(ov + e, eo, vn);
            set(ow + e, eo, (tb[a ^ 1][2][cc] + g.dt * f2 + oldw) * 0.5);
            if (MEAN) {
                const double wk = zm(g.dzflzi, kb - 1);
                red[tid] = red[tid] + un * wk;
                red[NT + tid] = red[NT + tid] + vn * wk;
            }
        }
        oldu = nou;
        oldv = nov;
        oldw = now;
        put(kb + 2, a);
        __syncthreads();
        if (SUB && mode >= 2 && ((kb - 1) % t.kc4 == 0 || kb - 1 == nz)) emit(kb - 1);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if (k0 > 1) iter(k0 - 1, I0{}, I1{});
    iter(k0, I1{}, I0{});
    using I3 = std::integral_constant<int, 3>;
    const int kl = min(k1 + 1, nz);
    int kb = k0 + 1;
#pragma unroll 1
    for (; kb < kl; kb += 2) {
        iter(kb, I2{}, I1{});
        iter(kb + 1, I2{}, I0{});
    }
    if (kb == kl) {
        iter(kb, I2{}, I1{});
        ++kb;
    }
    if (k1 == nz) {
        if ((kb - k0) & 1)
            iter(kb, I3{}, I1{});
        else
            iter(kb, I3{}, I0{});
    }
    if (MEAN && !SUB) emit(k1);
}

inline int ok() { return hipGetLastError() == hipSuccess ? 0 : -3; }

}  // namespace

extern "C" int pll_launch_rk12(const pll_grid_dev *gd, const double *const q[3],
                               double *const o[3], const double *p, double *mpart, int fmask,
                               double vfu, double vfv, const double *mean,
                               const double *const *body, hipStream_t s)
{
    const G g = make_g(gd);
    int rk[5];
    pll_rk_tiling(gd, rk);
    Tiles t;
    t.ntx = rk[0];
    t.nty4 = rk[1];
    t.nkc4 = rk[2];
    t.kc4 = rk[3];
    t.xcd4 = rk[4];
    t.nty = (g.ny + TY - 1) / TY;
    // Planes per workgroup: kc4, or the multiple of it with the least rounds of
    // the 256 CUs (one workgroup each) times planes per round, a chunk costing
    // three planes more than it has (the RK1 stage below and above it, two
    // planes of loads before the first), if that saves a tenth: small grids,
    // whose RK2 chunks are a few planes.  Per step of a run, kc4 planes against
    // this: 240x140x90 (4, 20 planes) 275 -> 244 us, 96x96x96 (2, 6) 126 -> 109,
    // 64x64x64 (1, 2) 65 -> 58.  SUB's partial sums inside the loop spill, so
    // smaller gains are none (192x192x128, 384x384x192: 2 to 4% slower).
    const long long cols = (long long)t.ntx * t.nty;
    auto cost = [&](int kc) { return (cols * ((g.nz + kc - 1) / kc) + 255) / 256 * (kc + 3); };
    const bool m = mpart && fmask;
    t.kc = t.kc4;
    for (int kc = 2 * t.kc4; kc < g.nz + t.kc4; kc += t.kc4)
        if (cost(kc) < cost(t.kc)) t.kc = kc;
    if (10 * cost(t.kc) > 9 * cost(t.kc4)) t.kc = t.kc4;
    const bool sub = m && t.kc > t.kc4;
    t.nkc = (g.nz + t.kc - 1) / t.kc;
    const long long nb = cols * t.nkc;
    if (nb > 0x7fffffffLL || g.sz > 0x1fffffffLL || (p != nullptr) == (body != nullptr)) return -1;
    t.xcd = nb % 8 == 0;
    const Body fb = body ? Body{body[0], body[1], body[2]} : Body{nullptr, nullptr, nullptr};
    const Proj pr{p, g.dt * g.dx_inv, g.dt * g.dy_inv, (p && mean) ? fmask : 0, vfu, vfv, mean};
#define PLL_RK12(P_, M_, S_)                                                                      \
    hipLaunchKernelGGL((k_rk12<P_, M_, S_>), dim3((unsigned)nb), dim3(64 * TY), 0, s, g, t, q[0], \
                       q[1], q[2], o[0], o[1], o[2], mpart, m ? fmask : 0, fb, pr)
    if (p && sub) PLL_RK12(true, true, true);
    else if (p && m) PLL_RK12(true, true, false);
    else if (p) PLL_RK12(true, false, false);
    else if (sub) PLL_RK12(false, true, true);
    else if (m) PLL_RK12(false, true, false);
    else PLL_RK12(false, false, false);
#undef PLL_RK12
    return ok();
}
