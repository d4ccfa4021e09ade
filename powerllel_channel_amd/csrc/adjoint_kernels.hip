// Transposes of the step's linear(ised) pieces, for the adjoint of the RK2
// projection step (no counterpart in the reference, which has no adjoint).
//
// Every kernel here writes each output element from one thread (gathers, no
// atomics), so results are deterministic.  The directional derivative of the
// momentum right-hand side evaluates the step kernels' own mom_rhs on dual
// numbers; its transpose is written out flux by flux.
//
// Layout: all fields are the haloed arrays f(0:nx+1, 0:ny+1, 0:nz+1).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mom_rhs.h"
#include "pll_internal.h"

namespace {

using pll::G;
using pll::make_g;
using pll::mom_rhs;
using pll::NbT;

// Dual number with one tangent (directional derivative).
struct D1 {
    double v, d;
};
__device__ __forceinline__ D1 operator+(const D1 &a, const D1 &b) { return D1{a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ D1 operator-(const D1 &a, const D1 &b) { return D1{a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ D1 operator*(const D1 &a, const D1 &b)
{
    return D1{a.v * b.v, a.d * b.v + a.v * b.d};
}
__device__ __forceinline__ D1 operator*(const D1 &a, double s) { return D1{a.v * s, a.d * s}; }
__device__ __forceinline__ D1 operator*(double s, const D1 &a) { return a * s; }

__device__ __forceinline__ bool interior(const G &g, int i, int j, int k)
{
    return i >= 1 && i <= g.nx && j >= 1 && j <= g.ny && k >= 1 && k <= g.nz;
}

__device__ __forceinline__ bool cell_of(const G &g, long long t, int &i, int &j, int &k)
{
    const long long nxh = g.nx + 2, nyh = g.ny + 2;
    if (t >= nxh * nyh * (g.nz + 2)) return false;
    i = (int)(t % nxh);
    t /= nxh;
    j = (int)(t % nyh);
    k = (int)(t / nyh);
    return true;
}

// ------------------------------------------------------------ momentum RHS
// The momentum right-hand side f = visc - conv (mom_rhs.h) is a sum of face
// and edge fluxes; with l on its three outputs, each flux P carries one
// weight S, a difference of l across the face, and the transpose adds
// dP/dq S to the values q the flux is made of:
//   xx  E = u_i + u_{i+1}               -(E^2)/4     u_crf E/2     diffusion of u
//   yy  (v_j + v_{j+1})^2, zz (w_k + w_{k+1})^2 likewise
//   xy  (u_j + u_{j+1})(v_i + v_{i+1})  in the u and the v equation
//   xz  ut (w_i + w_{i+1}), ut = u at the upper z face; yz likewise
// A cell gathers the fluxes it belongs to (no atomics, so the result does not
// depend on the order of workgroups).
struct JMet {
    double f_k, f_p, fi_k, fi_p, c_k, c_p;
};
__device__ __forceinline__ JMet jmet(const G &g, int k)
{
    const int p = min(k + 1, g.nz + 1);
    return JMet{pll::zm(g.dzf, k),     pll::zm(g.dzf, p),     pll::zm(g.dzf_inv, k),
                pll::zm(g.dzf_inv, p), pll::zm(g.dzc_inv, k), pll::zm(g.dzc_inv, p)};
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

// periodic index in 1..n of any haloed index
__device__ __forceinline__ int wrapn(int i, int n)
{
    const int r = (i - 1) % n;
    return (r < 0 ? r + n : r) + 1;
}

struct JTiles {
    int ntx, nty, nkc, kc, xcd;
};
constexpr int JTX = 64, JTY = 4, JQX = JTX + 2, JNQ = JQX * (JTY + 2);

// Fluxes through the upper z face of plane k at tile cell c (planes k and
// k + 1 in Q, L and Qn, Ln): their terms for plane k into lo, for k + 1 into up.
__device__ __forceinline__ void jt_face(const G &g, const JMet &z, const double (*Q)[JNQ],
                                        const double (*L)[JNQ], const double (*Qn)[JNQ],
                                        const double (*Ln)[JNQ], int c, double lo[3],
                                        double up[3])
{
    const double re = g.re_inv;
    const double lw = L[2][c], X = (lw - L[2][c + 1]) * g.dx_inv, Xm = (L[2][c - 1] - lw) * g.dx_inv;
    const double Y = (lw - L[2][c + JQX]) * g.dy_inv, Ym = (L[2][c - JQX] - lw) * g.dy_inv;
    const double w = Q[2][c];
    const double ut = (Q[0][c] * z.f_p + Qn[0][c] * z.f_k) * z.c_k;
    const double utm = (Q[0][c - 1] * z.f_p + Qn[0][c - 1] * z.f_k) * z.c_k;
    const double Vu = L[0][c] * z.fi_k - Ln[0][c] * z.fi_p;
    const double Vum = L[0][c - 1] * z.fi_k - Ln[0][c - 1] * z.fi_p;
    const double Su = Vu + X, Gu = -0.25 * (w + Q[2][c + 1]) * Su;
    lo[0] += z.c_k * (Gu * z.f_p - re * Vu);
    up[0] = z.c_k * (Gu * z.f_k + re * Vu);
    const double vt = (Q[1][c] * z.f_p + Qn[1][c] * z.f_k) * z.c_k;
    const double vtm = (Q[1][c - JQX] * z.f_p + Qn[1][c - JQX] * z.f_k) * z.c_k;
    const double Vv = L[1][c] * z.fi_k - Ln[1][c] * z.fi_p;
    const double Vvm = L[1][c - JQX] * z.fi_k - Ln[1][c - JQX] * z.fi_p;
    const double Sv = Vv + Y, Gv = -0.25 * (w + Q[2][c + JQX]) * Sv;
    lo[1] += z.c_k * (Gv * z.f_p - re * Vv);
    up[1] = z.c_k * (Gv * z.f_k + re * Vv);
    const double Sz = lw * z.c_k - Ln[2][c] * z.c_p, Gw = -0.5 * (w + Qn[2][c]) * Sz;
    lo[2] += Gw - re * z.fi_p * Sz - 0.25 * (ut * Su + utm * (Vum + Xm)) -
             0.25 * (vt * Sv + vtm * (Vvm + Ym));
    up[2] = Gw + re * z.fi_p * Sz;
}

// Fluxes within plane k at tile cell c.
__device__ __forceinline__ void jt_plane(const G &g, const double (*Q)[JNQ],
                                         const double (*L)[JNQ], int c, double a[3])
{
    const double re = g.re_inv, dx = g.dx_inv, dy = g.dy_inv, cr = g.u_crf;
    const double *U = Q[0] + c, *V = Q[1] + c;
    const double *A = L[0] + c, *B = L[1] + c, *W = L[2] + c;
    {
        const double S = (A[0] - A[1]) * dx, Sm = (A[-1] - A[0]) * dx;
        a[0] = re * dx * (Sm - S) - 0.5 * ((U[0] + U[1] + cr) * S + (U[-1] + U[0] + cr) * Sm);
    }
    const double T = (A[0] - A[JQX]) * dy, Tm = (A[-JQX] - A[0]) * dy;
    const double P = (B[0] - B[1]) * dx, Pm = (B[-1] - B[0]) * dx;
    // edges (i, j), (i, j - 1), (i - 1, j)
    const double S0 = T + P, Sy = Tm + (B[-JQX] - B[1 - JQX]) * dx,
                 Sx = (A[-1] - A[JQX - 1]) * dy + Pm;
    a[0] += re * dy * (Tm - T) - 0.25 * ((V[0] + V[1]) * S0 + (V[-JQX] + V[1 - JQX]) * Sy);
    a[1] = re * dx * (Pm - P) - 0.25 * ((U[0] + U[JQX]) * S0 + (U[-1] + U[JQX - 1]) * Sx) -
           0.5 * cr * (P + Pm);
    {
        const double S = (B[0] - B[JQX]) * dy, Sm = (B[-JQX] - B[0]) * dy;
        a[1] += re * dy * (Sm - S) - 0.5 * ((V[0] + V[JQX]) * S + (V[-JQX] + V[0]) * Sm);
    }
    const double X = (W[0] - W[1]) * dx, Xm = (W[-1] - W[0]) * dx;
    const double Y = (W[0] - W[JQX]) * dy, Ym = (W[-JQX] - W[0]) * dy;
    a[2] = re * (dx * (Xm - X) + dy * (Ym - Y)) - 0.5 * cr * (X + Xm);
}

// o_F(c) = beta x_F(c) + a0 l_F(c) [c interior] + alpha (J_f(q)^T l)_F(c)
// over every cell c of the haloed arrays; l is read on the interior only.
// FOLD: followed by the transposed boundary fill, on the interior alone.  The
// fill copies periodically in x and y, so l and q wrap there; at the walls u
// and v ghosts are 2 bc - the first or last plane, so what a ghost gathers
// goes to that plane with a minus sign, and w's ghosts and wall row k = nz are
// set to 0, so they pass nothing on.  q's own boundary values are formed from
// its interior the same way (its fill need not be made).
// GRAD: also gr += ga l + gb x, u's planes k = 1 and k = nz of o += cb and ct,
// and the sums of o over the workgroup's cells into part (3 x workgroups).
// A workgroup owns 64 x 4 columns and marches over a chunk of k with planes k
// and k + 1 of q and l in LDS (tile plus one cell) and plane k + 2 on its way
// into registers; what a z face adds to the plane above is carried there in
// registers.  72 bytes and about 135 FP64 operations per cell, bound by the
// latency of a plane's loads at 12 waves per CU (162 registers): 256x192x128
// 145 us, 3.1 TB/s; evaluating mom_rhs on dual numbers at the 13 outputs that
// read a cell took 460 us.  Tiles of 64 x 8 and 64 x 12 (fewer workgroups per
// CU) take 163 and 176 us, 64 x 8 at 16 waves (128 registers, spills) 255 us.
// x may be o itself (each cell is read and written by the same lane).
struct JGrad {
    double *gu, *gv, *gw;
    double ga, gb, cb, ct;
    double *part;
};

template <bool FOLD, bool GRAD>
__global__ void __launch_bounds__(JTX *JTY, 3)
k_jtv(G g, JTiles t, const double *__restrict__ qu, const double *__restrict__ qv,
      const double *__restrict__ qw, const double *__restrict__ lu, const double *__restrict__ lv,
      const double *__restrict__ lw, double *ou, double *ov, double *ow, const double *xu,
      const double *xv, const double *xw, double alpha, double a0, double beta, JGrad J)
{
    constexpr int NT = JTX * JTY, NR = (JNQ + NT - 1) / NT;
    __shared__ double tq[2][3][JNQ], tl[2][3][JNQ];
    int lb = blockIdx.x;
    if (t.xcd) lb = (lb & 7) * (int)(gridDim.x >> 3) + (lb >> 3);
    const int tx = lb % t.ntx;
    lb /= t.ntx;
    const int ty = lb % t.nty, kc = lb / t.nty;
    const int tid = threadIdx.x, lx = tid & (JTX - 1), ly = tid / JTX;
    constexpr int H = FOLD ? 1 : 0;  // first haloed index of the box
    const int i0 = tx * JTX + H, j0 = ty * JTY + H;  // of the tile's first cell
    const int k0 = kc * t.kc + H, k1 = min(k0 + t.kc - 1, g.nz + 1 - H);
    const int sy = (int)g.sy;
    unsigned off[NR];
    bool in[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int q = min(tid + r * NT, JNQ - 1), row = q / JQX, col = q - row * JQX;
        const int i = i0 - 1 + col, j = j0 - 1 + row;
        in[r] = FOLD || (i >= 1 && i <= g.nx && j >= 1 && j <= g.ny);
        const int ii = FOLD ? wrapn(i, g.nx) : min(max(i, 0), g.nx + 1);
        const int jj = FOLD ? wrapn(j, g.ny) : min(max(j, 0), g.ny + 1);
        off[r] = 8u * (unsigned)(ii + sy * jj);
    }
    double pq[3][NR], pl[3][NR];
    int kpre = 0;  // the plane fetched
    auto fetch = [&](int kp) {
        const long long e = g.sz * min(max(kp, H), g.nz + 1 - H);
        // opaque offsets: no 64-bit lane address per array hoisted out of the loop
#pragma unroll
        for (int r = 0; r < NR; ++r) asm volatile("" : "+v"(off[r]));
        const double *b0 = qu + e, *b1 = qv + e, *b2 = qw + e;
        const double *m0 = lu + e, *m1 = lv + e, *m2 = lw + e;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            pq[0][r] = at(b0, off[r]);
            pq[1][r] = at(b1, off[r]);
            pq[2][r] = at(b2, off[r]);
            pl[0][r] = at(m0, off[r]);
            pl[1][r] = at(m1, off[r]);
            pl[2][r] = at(m2, off[r]);
        }
        kpre = kp;
    };
    auto put = [&](int b) {
        const bool wall = kpre < 1 || kpre > g.nz;
        const double bcu = 0.0 - g.u_crf;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int q = min(tid + r * NT, JNQ - 1);
            double u = pq[0][r], v = pq[1][r], w = pq[2][r];
            if (FOLD) {
                u = wall ? 2.0 * bcu - u : u;
                v = wall ? 2.0 * 0.0 - v : v;
                w = wall || kpre == g.nz ? 0.0 : w;
            }
            tq[b][0][q] = u;
            tq[b][1][q] = v;
            tq[b][2][q] = w;
#pragma unroll
            for (int f = 0; f < 3; ++f) tl[b][f][q] = !wall && in[r] ? pl[f][r] : 0.0;
        }
    };
    const int c = (ly + 1) * JQX + lx + 1;
    const int i = i0 + lx, j = j0 + ly;
    const bool own = i <= g.nx + 1 - H && j <= g.ny + 1 - H;
    unsigned eo = 8u * (unsigned)(i + sy * j);
    double up[3] = {0.0, 0.0, 0.0};
    // plane k lives in slot (k - k0) & 1
    fetch(k0 - 1);
    put(1);
    fetch(k0);
    put(0);
    fetch(k0 + 1);
    __syncthreads();
    if (k0 > 0) {
        double lo[3] = {0.0, 0.0, 0.0};
        jt_face(g, jmet(g, k0 - 1), tq[1], tl[1], tq[0], tl[0], c, lo, up);
        if (FOLD && k0 == 1) {  // the ghost plane's share goes to the first plane
            up[0] -= lo[0];
            up[1] -= lo[1];
        }
    }
    double sum[3] = {0.0, 0.0, 0.0};
    __syncthreads();
    put(1);
    __syncthreads();
    auto plane = [&](int kv, auto SLOT) {
        constexpr int b = decltype(SLOT)::value;
        const int k = __builtin_amdgcn_readfirstlane(kv);
        asm volatile("" : "+v"(eo));
        fetch(min(k + 2, k1 + 1));
        __builtin_amdgcn_sched_barrier(0);
        double a[3], nup[3];
        jt_plane(g, tq[b], tl[b], c, a);
        jt_face(g, jmet(g, k), tq[b], tl[b], tq[b ^ 1], tl[b ^ 1], c, a, nup);
        if (FOLD && k == g.nz) {
            a[0] -= nup[0];
            a[1] -= nup[1];
        }
        if (own) {
            const long long e = g.sz * k;
            double *const o[3] = {ou + e, ov + e, ow + e};
            const double *const x[3] = {xu + e, xv + e, xw + e};
            double *const gr[3] = {J.gu + e, J.gv + e, J.gw + e};
            const double cw = k == 1 ? J.cb : (k == g.nz ? J.ct : 0.0);
#pragma unroll
            for (int f = 0; f < 3; ++f) {
                const double lc = tl[b][f][c];
                const double xv = beta != 0.0 ? at(x[f], eo) : 0.0;
                double r = alpha * (a[f] + up[f]) + a0 * lc + beta * xv;
                if (FOLD && f == 2 && k == g.nz) r = 0.0;
                if (GRAD) {
                    if (f == 0) r += cw;
                    set(gr[f], eo, at(gr[f], eo) + (J.ga * lc + J.gb * xv));
                    sum[f] += r;
                }
                set(o[f], eo, r);
            }
        }
#pragma unroll
        for (int f = 0; f < 3; ++f) up[f] = nup[f];
        __syncthreads();
        put(b);
        __syncthreads();
    };
    int k = k0;
#pragma unroll 1
    for (; k < k1; k += 2) {
        plane(k, std::integral_constant<int, 0>{});
        plane(k + 1, std::integral_constant<int, 1>{});
    }
    if (k == k1) plane(k, std::integral_constant<int, 0>{});
    if (GRAD) {
        double *red = &tq[0][0][0];
#pragma unroll
        for (int f = 0; f < 3; ++f) red[f * NT + tid] = sum[f];
        __syncthreads();
        for (int h = NT / 2; h > 0; h >>= 1) {
            if (tid < h)
#pragma unroll
                for (int f = 0; f < 3; ++f) red[f * NT + tid] += red[f * NT + tid + h];
            __syncthreads();
        }
        if (tid < 3) J.part[(size_t)tid * gridDim.x + blockIdx.x] = red[tid * NT];
    }
}

// o = J_f(q) dq on the interior (directional derivative of the momentum
// right-hand side), for checks of the transpose.
__global__ void __launch_bounds__(256) k_jvp(G g, const double *__restrict__ qu,
                                             const double *__restrict__ qv,
                                             const double *__restrict__ qw,
                                             const double *__restrict__ du,
                                             const double *__restrict__ dv,
                                             const double *__restrict__ dw,
                                             double *__restrict__ ou, double *__restrict__ ov,
                                             double *__restrict__ ow)
{
    int i, j, k;
    if (!cell_of(g, (long long)blockIdx.x * blockDim.x + threadIdx.x, i, j, k)) return;
    if (!interior(g, i, j, k)) return;
    const long long sy = g.sy, sz = g.sz;
    const long long e = i + sy * j + sz * k;
#define S(name, arr, darr, a, b, c)                               \
    do {                                                          \
        const long long x_ = e + (a) + sy * (b) + sz * (c);       \
        n.name = D1{arr[x_], darr[x_]};                           \
    } while (0)
    NbT<D1> n;
    S(u000, qu, du, 0, 0, 0); S(up00, qu, du, 1, 0, 0); S(um00, qu, du, -1, 0, 0);
    S(u0p0, qu, du, 0, 1, 0); S(u0m0, qu, du, 0, -1, 0); S(u00p, qu, du, 0, 0, 1);
    S(u00m, qu, du, 0, 0, -1); S(ump0, qu, du, -1, 1, 0); S(um0p, qu, du, -1, 0, 1);
    S(v000, qv, dv, 0, 0, 0); S(vp00, qv, dv, 1, 0, 0); S(vm00, qv, dv, -1, 0, 0);
    S(v0p0, qv, dv, 0, 1, 0); S(v0m0, qv, dv, 0, -1, 0); S(v00p, qv, dv, 0, 0, 1);
    S(v00m, qv, dv, 0, 0, -1); S(vpm0, qv, dv, 1, -1, 0); S(v0mp, qv, dv, 0, -1, 1);
    S(w000, qw, dw, 0, 0, 0); S(wp00, qw, dw, 1, 0, 0); S(wm00, qw, dw, -1, 0, 0);
    S(w0p0, qw, dw, 0, 1, 0); S(w0m0, qw, dw, 0, -1, 0); S(w00p, qw, dw, 0, 0, 1);
    S(w00m, qw, dw, 0, 0, -1); S(wp0m, qw, dw, 1, 0, -1); S(w0pm, qw, dw, 0, 1, -1);
#undef S
    D1 fu, fv, fw;
    mom_rhs(g, n, k, fu, fv, fw);
    ou[e] = fu.d;
    ov[e] = fv.d;
    ow[e] = fw.d;
}

// ------------------------------------------------------------ boundary fills
// The forward fills set every ghost from interior values (periodic copies in
// x and y; at the walls u,v ghost = 2 bc - interior of the first/last plane,
// w ghost = 0; w's top wall row k = nz := 0; p ghost = periodic copy or the
// first/last plane).  The transpose adds each ghost's adjoint to the interior
// value it was made from and clears the ghosts.  Pass 1 (interior cells next
// to a face) gathers; pass 2 clears the ghost shell.
__device__ __forceinline__ int images(int i, int n, int out[3])
{
    int m = 0;
    out[m++] = i;
    if (i == n) out[m++] = 0;
    if (i == 1) out[m++] = n + 1;
    return m;
}

// kind 0: velocity (3 fields), kind 1: pressure (field 0 only).
template <int KIND>
__global__ void __launch_bounds__(256) k_fold(G g, double *__restrict__ f0,
                                              double *__restrict__ f1,
                                              double *__restrict__ f2)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)g.nx * g.ny * g.nz) return;
    const int i = (int)(t % g.nx) + 1, j = (int)((t / g.nx) % g.ny) + 1,
              k = (int)(t / ((long long)g.nx * g.ny)) + 1;
    const bool face = i == 1 || i == g.nx || j == 1 || j == g.ny || k == 1 || k == g.nz;
    if (!face) return;
    int ia[3], ja[3];
    const int ni = images(i, g.nx, ia), nj = images(j, g.ny, ja);
    const long long sy = g.sy, sz = g.sz;
    const long long e = i + sy * j + sz * k;
    double *F[3] = {f0, f1, f2};
    const int nf = KIND == 0 ? 3 : 1;
    for (int f = 0; f < nf; ++f) {
        double *q = F[f];
        if (KIND == 0 && f == 2 && k == g.nz) {  // w's wall row is overwritten with 0
            q[e] = 0.0;
            continue;
        }
        double s = q[e];
        for (int a = 0; a < ni; ++a)
            for (int b = 0; b < nj; ++b)
                if (a != 0 || b != 0) s += q[ia[a] + sy * ja[b] + sz * k];
        // wall ghost planes: p copies (+1), u and v mirror (-1), w is set to 0
        const double wc = KIND == 1 ? 1.0 : (f == 2 ? 0.0 : -1.0);
        if (wc != 0.0) {
            for (int side = 0; side < 2; ++side) {
                if (side == 0 ? k != 1 : k != g.nz) continue;
                const int kg = side == 0 ? 0 : g.nz + 1;
                for (int a = 0; a < ni; ++a)
                    for (int b = 0; b < nj; ++b) s += wc * q[ia[a] + sy * ja[b] + sz * kg];
            }
        }
        q[e] = s;
    }
}

__global__ void __launch_bounds__(256) k_clear_ghosts(G g, double *__restrict__ f0,
                                                      double *__restrict__ f1,
                                                      double *__restrict__ f2, int nf)
{
    int i, j, k;
    if (!cell_of(g, (long long)blockIdx.x * blockDim.x + threadIdx.x, i, j, k)) return;
    if (interior(g, i, j, k)) return;
    const long long e = i + g.sy * j + g.sz * k;
    f0[e] = 0.0;
    if (nf > 1) {
        f1[e] = 0.0;
        f2[e] = 0.0;
    }
}

// ------------------------------------------------------------ projection
// correctVel: u -= (p_{i+1} - p_i) dtdxi, v -= (p_{j+1} - p_j) dtdyi,
// w -= (p_{k+1} - p_k) dt dzc_inv(k) on the interior.  Transpose: for every
// p cell c (interior or halo), lp(c) = sum of the coefficients times the
// adjoints of the interior velocities that read it.
__global__ void __launch_bounds__(256) k_correct_adj(G g, const double *__restrict__ lu,
                                                     const double *__restrict__ lv,
                                                     const double *__restrict__ lw,
                                                     double *__restrict__ lp, double dtdxi,
                                                     double dtdyi)
{
    int i, j, k;
    if (!cell_of(g, (long long)blockIdx.x * blockDim.x + threadIdx.x, i, j, k)) return;
    const long long sy = g.sy, sz = g.sz;
    const long long e = i + sy * j + sz * k;
    double s = 0.0;
    if (interior(g, i, j, k)) {
        s += dtdxi * lu[e] + dtdyi * lv[e] + g.dt * g.dzc_inv[k] * lw[e];
    }
    if (interior(g, i - 1, j, k)) s -= dtdxi * lu[e - 1];
    if (interior(g, i, j - 1, k)) s -= dtdyi * lv[e - sy];
    if (interior(g, i, j, k - 1)) s -= g.dt * g.dzc_inv[k - 1] * lw[e - sz];
    lp[e] = s;
}

// calcRHS: rhs = (u_i - u_{i-1}) dtidxi + (v_j - v_{j-1}) dtidyi
//              + (w_k - w_{k-1}) dti dzf_inv(k) on the interior.
// Transpose, accumulated: l_u(c) += dtidxi (lr(c) - lr(c+x)) etc., over every
// velocity cell c, with lr read on the interior only.
__global__ void __launch_bounds__(256) k_rhs_adj(G g, const double *__restrict__ lr,
                                                 double *__restrict__ lu, double *__restrict__ lv,
                                                 double *__restrict__ lw, double dti,
                                                 double dtidxi, double dtidyi)
{
    int i, j, k;
    if (!cell_of(g, (long long)blockIdx.x * blockDim.x + threadIdx.x, i, j, k)) return;
    const long long sy = g.sy, sz = g.sz;
    const long long e = i + sy * j + sz * k;
    const double rc = interior(g, i, j, k) ? lr[e] : 0.0;
    const double rx = interior(g, i + 1, j, k) ? lr[e + 1] : 0.0;
    const double ry = interior(g, i, j + 1, k) ? lr[e + sy] : 0.0;
    const double rz = interior(g, i, j, k + 1) ? lr[e + sz] : 0.0;
    lu[e] += dtidxi * (rc - rx);
    lv[e] += dtidyi * (rc - ry);
    double wz = 0.0;
    if (k >= 1 && k <= g.nz) wz += dti * g.dzf_inv[k] * rc;
    if (k + 1 >= 1 && k + 1 <= g.nz) wz -= dti * g.dzf_inv[k + 1] * rz;
    lw[e] += wz;
}

// The same two transposes between transposed fills, on the interior alone: l
// and the result are folded (periodic in x and y, no ghosts at the walls, w = 0
// on its wall row), and the transposed forcing l -= dzflzi(k) tot of the
// components in fmask is applied as l is read (tot: sum of l over the interior
// / (nx ny)).  In the pressure gradient it cancels for u and v.
// A workgroup's column of cells: planes blockIdx.z + 1, + gridDim.z, ... (a grid's
// z extent ends at 65535).
#define PLL_COLUMN                                                 \
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;       \
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;       \
    if (i > g.nx || j > g.ny) return;                              \
    const long long sy = g.sy, sz = g.sz;                          \
    for (int k = blockIdx.z + 1; k <= g.nz; k += gridDim.z)

__global__ void __launch_bounds__(256) k_correct_adj_fold(G g, const double *__restrict__ lu,
                                                          const double *__restrict__ lv,
                                                          const double *__restrict__ lw,
                                                          double *__restrict__ lp, double dtdxi,
                                                          double dtdyi, int fmask,
                                                          const double *__restrict__ tot)
{
    const double sw = (fmask & 4) ? tot[2] : 0.0;
    PLL_COLUMN
    {
        const long long e = i + sy * j + sz * k;
        const double um = lu[i == 1 ? e - 1 + g.nx : e - 1],
                     vm = lv[j == 1 ? e + sy * (g.ny - 1) : e - sy];
        const double wt = k < g.nz ? g.dzc_inv[k] * (lw[e] - g.dzflzi[k] * sw) : 0.0;
        const double wb = k > 1 ? g.dzc_inv[k - 1] * (lw[e - sz] - g.dzflzi[k - 1] * sw) : 0.0;
        lp[e] = dtdxi * (lu[e] - um) + dtdyi * (lv[e] - vm) + g.dt * (wt - wb);
    }
}

__global__ void __launch_bounds__(256) k_rhs_adj_fold(G g, const double *__restrict__ lr,
                                                      double *__restrict__ lu,
                                                      double *__restrict__ lv,
                                                      double *__restrict__ lw, double dti,
                                                      double dtidxi, double dtidyi, int fmask,
                                                      const double *__restrict__ tot)
{
    PLL_COLUMN
    {
        const long long e = i + sy * j + sz * k;
        const double wk = g.dzflzi[k];
        const double rc = lr[e], rx = lr[i == g.nx ? e + 1 - g.nx : e + 1];
        const double ry = lr[j == g.ny ? e - sy * (g.ny - 1) : e + sy],
                     rz = k < g.nz ? lr[e + sz] : 0.0;
        const double tu = (fmask & 1) ? wk * tot[0] : 0.0, tv = (fmask & 2) ? wk * tot[1] : 0.0,
                     tw = (fmask & 4) ? wk * tot[2] : 0.0;
        lu[e] = (lu[e] - tu) + dtidxi * (rc - rx);
        lv[e] = (lv[e] - tv) + dtidyi * (rc - ry);
        lw[e] = k == g.nz ? 0.0 : (lw[e] - tw) + dti * (g.dzf_inv[k] * rc - g.dzf_inv[k + 1] * rz);
    }
}

inline dim3 column_grid(const G &g)
{
    return dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz < 65535 ? g.nz : 65535);
}

// ------------------------------------------------------------ forcing
// forceVel: q += vel_force - sum_c q_c dzflzi(k_c) / (nx ny).  Transpose:
// l(c) -= dzflzi(k_c) / (nx ny) * sum_interior l.  Pass 1: per-(j,k)-row
// sums; the final sum and the shift in pass 2.
__global__ void __launch_bounds__(256) k_rowsum(G g, const double *__restrict__ q,
                                                double *__restrict__ part)
{
    __shared__ double sh[256];
    const int j = blockIdx.x % g.ny + 1, k = blockIdx.x / g.ny + 1;
    const long long base = g.sy * j + g.sz * k;
    double s = 0.0;
    for (int i = threadIdx.x + 1; i <= g.nx; i += blockDim.x) s += q[base + i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// one workgroup per sum: out[b] = scale * sum of part[b n .. b n + n)
__global__ void __launch_bounds__(1024) k_sum(int n, const double *__restrict__ part,
                                              double *__restrict__ out, double scale)
{
    __shared__ double sh[1024];
    double s = 0.0;
    part += (size_t)blockIdx.x * n;
    for (int t = threadIdx.x; t < n; t += blockDim.x) s += part[t];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = sh[0] * scale;
}

__global__ void __launch_bounds__(256) k_force_adj(G g, double *__restrict__ q,
                                                   const double *__restrict__ total)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)g.nx * g.ny * g.nz) return;
    const int i = (int)(t % g.nx) + 1, j = (int)((t / g.nx) % g.ny) + 1,
              k = (int)(t / ((long long)g.nx * g.ny)) + 1;
    const long long e = i + g.sy * j + g.sz * k;
    q[e] -= g.dzflzi[k] * total[0];
}

// ------------------------------------------------------------ wall shear
// sum over (i,j) of q(i,j,kw) for the bottom (kw = 1) and top (kw = nz)
// interior planes: per-row partials part[w * ny + j - 1].
__global__ void __launch_bounds__(256) k_wall_rows(G g, const double *__restrict__ q,
                                                   double *__restrict__ part)
{
    __shared__ double sh[256];
    const int w = blockIdx.x / g.ny, j = blockIdx.x % g.ny + 1;
    const int k = w == 0 ? 1 : g.nz;
    const long long base = g.sy * j + g.sz * k;
    double s = 0.0;
    for (int i = threadIdx.x + 1; i <= g.nx; i += blockDim.x) s += q[base + i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// l_u += c_w on the interior planes k = 1 (c_bot) and k = nz (c_top).
__global__ void __launch_bounds__(256) k_wall_seed(G g, double *__restrict__ lu, double c_bot,
                                                   double c_top)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 2LL * g.nx * g.ny) return;
    const int w = (int)(t / ((long long)g.nx * g.ny));
    const long long r = t % ((long long)g.nx * g.ny);
    const int i = (int)(r % g.nx) + 1, j = (int)(r / g.nx) + 1;
    const int k = w == 0 ? 1 : g.nz;
    if (g.nz == 1 && w == 1) {  // one plane: both walls are that plane
        lu[i + g.sy * j + g.sz * k] += c_top;
        return;
    }
    lu[i + g.sy * j + g.sz * k] += (w == 0 ? c_bot : c_top);
}

// y += a x + b z over every cell of the haloed arrays (three fields).
struct Axpy3 {
    const double *x[3], *z[3];
    double *y[3];
};
__global__ void __launch_bounds__(256) k_axpy3(long long n, double a, double b, Axpy3 v)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
#pragma unroll
    for (int f = 0; f < 3; ++f) v.y[f][t] += a * v.x[f][t] + b * v.z[f][t];
}

inline int ok() { return hipGetLastError() == hipSuccess ? 0 : -3; }
inline long long ncell(const G &g) { return (long long)(g.nx + 2) * (g.ny + 2) * (g.nz + 2); }
inline unsigned nblk(long long n) { return (unsigned)((n + 255) / 256); }

// Tiles of an nx x ny x nz box: k chunks of up to 32 planes, shorter on small
// boxes so that 1536 workgroups run (two rounds of the three that fit a CU):
// 256x192x128 145 us with 16 planes, 161 with 32, 148 with 8; 512x384x256
// 974 us with 32, 985 with 16.  Then even chunks, as the stencil tiles.
JTiles jt_tiles(int nx, int ny, int nz, int kc)
{
    JTiles t;
    t.ntx = (nx + JTX - 1) / JTX;
    t.nty = (ny + JTY - 1) / JTY;
    const long long cols = (long long)t.ntx * t.nty;
    t.kc = 32;
    while (t.kc > 1 && cols * ((nz + t.kc - 1) / t.kc) < 1536) t.kc >>= 1;
    const int n = (nz + t.kc - 1) / t.kc;
    t.kc = kc > 0 ? kc : (nz + n - 1) / n;
    t.nkc = (nz + t.kc - 1) / t.kc;
    t.xcd = (cols * t.nkc) % 8 == 0;
    return t;
}

}  // namespace

extern "C" int pll_launch_jtv(const pll_grid_dev *gd, const double *const q[3],
                              const double *const l[3], double *const o[3], double alpha,
                              double a0, double beta, hipStream_t s)
{
    const G g = make_g(gd);
    if (g.sz > 0x1fffffffLL) return -1;
    const JTiles t = jt_tiles(g.nx + 2, g.ny + 2, g.nz + 2, g.kc);
    hipLaunchKernelGGL((k_jtv<false, false>), dim3((unsigned)(t.ntx * t.nty * t.nkc)),
                       dim3(JTX * JTY), 0, s, g, t, q[0], q[1], q[2], l[0], l[1], l[2], o[0], o[1],
                       o[2], o[0], o[1], o[2], alpha, a0, beta, JGrad{});
    return ok();
}

extern "C" int pll_jtv_fold_blocks(const pll_grid_dev *gd)
{
    const G g = make_g(gd);
    const JTiles t = jt_tiles(g.nx, g.ny, g.nz, g.kc);
    return t.ntx * t.nty * t.nkc;
}

extern "C" int pll_launch_jtv_fold(const pll_grid_dev *gd, const double *const q[3],
                                   const double *const l[3], double *const o[3],
                                   const double *const x[3], double alpha, double a0, double beta,
                                   double *const gr[3], double ga, double gb, double cb, double ct,
                                   double *part, hipStream_t s)
{
    const G g = make_g(gd);
    if (g.sz > 0x1fffffffLL) return -1;
    const JTiles t = jt_tiles(g.nx, g.ny, g.nz, g.kc);
    const dim3 grid((unsigned)(t.ntx * t.nty * t.nkc)), blk(JTX * JTY);
    const double *const *y = x ? x : l;
    if (gr) {
        const JGrad J{gr[0], gr[1], gr[2], ga, gb, cb, ct, part};
        hipLaunchKernelGGL((k_jtv<true, true>), grid, blk, 0, s, g, t, q[0], q[1], q[2], l[0], l[1],
                           l[2], o[0], o[1], o[2], y[0], y[1], y[2], alpha, a0, x ? beta : 0.0, J);
    } else {
        hipLaunchKernelGGL((k_jtv<true, false>), grid, blk, 0, s, g, t, q[0], q[1], q[2], l[0],
                           l[1], l[2], o[0], o[1], o[2], y[0], y[1], y[2], alpha, a0,
                           x ? beta : 0.0, JGrad{});
    }
    return ok();
}

extern "C" int pll_launch_jvp(const pll_grid_dev *gd, const double *const q[3],
                              const double *const dq[3], double *const o[3], hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_jvp, dim3(nblk(ncell(g))), dim3(256), 0, s, g, q[0], q[1], q[2], dq[0],
                       dq[1], dq[2], o[0], o[1], o[2]);
    return ok();
}

extern "C" int pll_launch_bc_vel_adj(const pll_grid_dev *gd, double *lu, double *lv, double *lw,
                                     hipStream_t s)
{
    const G g = make_g(gd);
    const long long n = (long long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(k_fold<0>, dim3(nblk(n)), dim3(256), 0, s, g, lu, lv, lw);
    if (ok()) return -3;
    hipLaunchKernelGGL(k_clear_ghosts, dim3(nblk(ncell(g))), dim3(256), 0, s, g, lu, lv, lw, 3);
    return ok();
}

extern "C" int pll_launch_bc_p_adj(const pll_grid_dev *gd, double *lp, hipStream_t s)
{
    const G g = make_g(gd);
    const long long n = (long long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(k_fold<1>, dim3(nblk(n)), dim3(256), 0, s, g, lp, lp, lp);
    if (ok()) return -3;
    hipLaunchKernelGGL(k_clear_ghosts, dim3(nblk(ncell(g))), dim3(256), 0, s, g, lp, lp, lp, 1);
    return ok();
}

extern "C" int pll_launch_correct_adj(const pll_grid_dev *gd, const double *lu, const double *lv,
                                      const double *lw, double *lp, hipStream_t s)
{
    const G g = make_g(gd);
    const double dtdxi = g.dt * g.dx_inv, dtdyi = g.dt * g.dy_inv;
    hipLaunchKernelGGL(k_correct_adj, dim3(nblk(ncell(g))), dim3(256), 0, s, g, lu, lv, lw, lp,
                       dtdxi, dtdyi);
    return ok();
}

extern "C" int pll_launch_rhs_adj(const pll_grid_dev *gd, const double *lr, double *lu,
                                  double *lv, double *lw, hipStream_t s)
{
    const G g = make_g(gd);
    const double dti = 1.0 / g.dt;
    hipLaunchKernelGGL(k_rhs_adj, dim3(nblk(ncell(g))), dim3(256), 0, s, g, lr, lu, lv, lw, dti,
                       dti * g.dx_inv, dti * g.dy_inv);
    return ok();
}

extern "C" int pll_launch_force_adj(const pll_grid_dev *gd, double *q, double *part,
                                    double *total, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_rowsum, dim3(g.ny * g.nz), dim3(256), 0, s, g, q, part);
    if (ok()) return -3;
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, s, g.ny * g.nz, part, total,
                       1.0 / ((double)g.nx * g.ny));
    if (ok()) return -3;
    const long long n = (long long)g.nx * g.ny * g.nz;
    hipLaunchKernelGGL(k_force_adj, dim3(nblk(n)), dim3(256), 0, s, g, q, total);
    return ok();
}

extern "C" int pll_launch_wall_sum(const pll_grid_dev *gd, const double *u, double *part,
                                   double *out, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_wall_rows, dim3(2 * g.ny), dim3(256), 0, s, g, u, part);
    if (ok()) return -3;
    hipLaunchKernelGGL(k_sum, dim3(2), dim3(1024), 0, s, g.ny, part, out, 1.0);
    return ok();
}

extern "C" int pll_launch_wall_seed(const pll_grid_dev *gd, double *lu, double c_bot,
                                    double c_top, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_wall_seed, dim3(nblk(2LL * g.nx * g.ny)), dim3(256), 0, s, g, lu, c_bot,
                       c_top);
    return ok();
}

extern "C" int pll_launch_axpy3(const pll_grid_dev *gd, double a, const double *const x[3],
                                double b, const double *const z[3], double *const y[3],
                                hipStream_t s)
{
    const G g = make_g(gd);
    const long long n = ncell(g);
    const Axpy3 v{{x[0], x[1], x[2]}, {z[0], z[1], z[2]}, {y[0], y[1], y[2]}};
    hipLaunchKernelGGL(k_axpy3, dim3(nblk(n)), dim3(256), 0, s, n, a, b, v);
    return ok();
}

extern "C" int pll_launch_correct_adj_fold(const pll_grid_dev *gd, const double *const l[3],
                                           double *lp, int fmask, const double *tot, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_correct_adj_fold, column_grid(g), dim3(64, 4, 1), 0, s, g, l[0], l[1],
                       l[2], lp, g.dt * g.dx_inv, g.dt * g.dy_inv, fmask, tot);
    return ok();
}

extern "C" int pll_launch_rhs_adj_fold(const pll_grid_dev *gd, const double *lr,
                                       double *const l[3], int fmask, const double *tot,
                                       hipStream_t s)
{
    const G g = make_g(gd);
    const double dti = 1.0 / g.dt;
    hipLaunchKernelGGL(k_rhs_adj_fold, column_grid(g), dim3(64, 4, 1), 0, s, g, lr, l[0], l[1],
                       l[2], dti, dti * g.dx_inv, dti * g.dy_inv, fmask, tot);
    return ok();
}

extern "C" int pll_launch_sum3(int n, const double *part, double *out, double scale, hipStream_t s)
{
    hipLaunchKernelGGL(k_sum, dim3(3), dim3(1024), 0, s, n, part, out, scale);
    return ok();
}
