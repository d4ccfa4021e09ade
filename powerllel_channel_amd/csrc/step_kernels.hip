// RK2 projection step kernels for gfx950.
//
// Each kernel restates one Fortran routine of the reference's step, with the
// same operation order; the file is compiled with -ffp-contract=off so every
// product and sum is rounded on its own, as in the reference's source:
//   RK1 / RK2 stencils  src/mod_calcVel.f90:52-146, :240-334
//   calcRHS             src/mod_calcRHS.f90:11-37
//   correctVel          src/mod_calcVel.f90:428-453
//   forceVel + Mean_h   src/mod_calcVel.f90:455-509, src/mod_utils.f90:105-131
//   updateBoundVel/P    src/mod_updateBound.f90:30-108, :186-362 (one rank)
//   calcMaxDiv          src/mod_utils.f90:257-318
// Fields are the reference's haloed arrays f(0:nx+1,0:ny+1,0:nz+1), x fastest.
#include <hip/hip_runtime.h>

#include <stdlib.h>

#include <type_traits>

#include "mom_rhs.h"
#include "pll_internal.h"

namespace {

using pll::G;
using pll::Nb;
using pll::make_g;
using pll::mom_rhs;


// RK stencils march over a chunk of k per thread: the values of plane k+1
// that become plane k (and then k-1) at the next step stay in registers, so
// each plane of the three fields is fetched once per chunk; x and y
// neighbours come through the caches.  Workgroups are numbered so that each
// of the 8 XCDs (which take workgroups round-robin) gets one contiguous run
// of tiles: y-adjacent tiles of one k-chunk then share that XCD's L2.
constexpr int RK_TX = 64, RK_TY = 4;
struct Tiles {
    int ntx, nty, nkc, kc;
    int xcd;  // 1: remap workgroup ids per XCD (tile count divisible by 8)
};

__device__ __forceinline__ void rk_tile(const Tiles &t, int &tx, int &ty, int &kc)
{
    const int nb = t.ntx * t.nty * t.nkc;
    int lb = blockIdx.x;
    if (t.xcd) lb = (lb & 7) * (nb >> 3) + (lb >> 3);
    tx = lb % t.ntx;
    lb /= t.ntx;
    ty = lb % t.nty;
    kc = lb / t.nty;
}

// SECOND = false: o := q + dt f(q)                  (RK1, o = u1, q = u)
// SECOND = true:  o := (q + dt f(q) + o) * 0.5      (RK2, o = u,  q = u1)
// MEAN (RK2 only): also the Mean_h partial sums of the new u (fmask bit 0)
// and v (bit 1), sum of o * dzflzi(k) over the block's cells, into
// mpart[blockIdx.x] and mpart[nblocks + blockIdx.x].
//
// 2.5-D blocking: a workgroup owns a 64 x 4 column tile and marches over a
// k chunk.  Planes k and k+1 of the three fields sit in LDS as 66 x 6 tiles
// (tile plus one-cell halo), loaded with coalesced row reads; plane k+2 is
// fetched into registers while plane k is computed and written over plane
// k's buffer afterwards.  The few plane k-1 values the stencil reads are
// carried in registers from the previous step.  Every stencil read is then
// an LDS read, and each field value is loaded from memory about 1.5 times
// (the halo) instead of once per neighbour that reads it.
// BODY: a body force b (haloed layout, interior read) is added to the
// right-hand side, f := f(q) + b, in both stages.
struct Body {
    const double *u, *v, *w;
};

__device__ __forceinline__ int wrap(int i, int n) { return i == 0 ? n : (i == n + 1 ? 1 : i); }

constexpr int LTX = RK_TX + 2;

// FILL: q's boundary fill has not been made; the values it would leave
// (k_bc_vel) are read from the interior instead of the ghost cells.
// FULL: every tile lies inside the grid (nx % 64 == 0, ny % TY == 0).  Then no
// lane is masked: every lane loads its plane share (lanes past the halo tile
// load and store its last element again) and the last planes of a chunk are
// fetched again instead of skipped, so the loop has no divergent branch and
// each wait covers only the loads it needs: the prefetch is waited for when it
// is written to LDS (the plane's stores may stay in flight), and RK2's old
// values of plane k are loaded before the prefetch of plane k+2, so that
// waiting for them leaves the prefetch in flight.
// Occupancy hints: the FULL RK1 kernels at 4 waves per SIMD; the general RK2
// kernels without a body force at 5 (96 VGPRs, no spills: 100 and 4 waves
// without it; step 4.365 -> 4.350 ms at 768x384x256).
template <bool SECOND, bool MEAN, bool BODY, bool FILL, bool FULL>
__global__ void __launch_bounds__(RK_TX *RK_TY, (FULL && !SECOND ? 4 : (SECOND && !FULL && !BODY ? 5 : 1))) k_rk(G g, Tiles t, const double *__restrict__ qu,
                                                     const double *__restrict__ qv,
                                                     const double *__restrict__ qw,
                                                     double *__restrict__ ou,
                                                     double *__restrict__ ov,
                                                     double *__restrict__ ow,
                                                     double *__restrict__ mpart, int fmask,
                                                     Body fb)
{
    constexpr int TY = RK_TY, LTY = TY + 2, LPL = LTX * LTY, NT = RK_TX * TY;
    constexpr int NLD = (LPL + NT - 1) / NT;
    __shared__ double tl[2][3][LPL];
    int tx, ty, kc;
    rk_tile(t, tx, ty, kc);
    const int tid = threadIdx.x;
    const int lx = tid % RK_TX, ly = tid / RK_TX;
    const int i0 = tx * RK_TX, j0 = ty * TY;  // haloed index of the tile's halo corner
    const int i = i0 + lx + 1, j = j0 + ly + 1;
    const bool valid = FULL || (i <= g.nx && j <= g.ny);
    const int k0 = kc * t.kc + 1, k1 = min(k0 + t.kc - 1, g.nz);
    const long long sy = g.sy, sz = g.sz;
    const double *__restrict__ Q[3] = {qu, qv, qw};
    // this thread's share of a plane tile: element q = tid + r * 256
    long long go[NLD];
    bool gk[NLD];
    int gii[NLD], gjj[NLD];
#pragma unroll
    for (int r = 0; r < NLD; ++r) {
        const int q = FULL ? min(tid + r * NT, LPL - 1) : tid + r * NT;
        const int row = q / LTX, col = q - row * LTX;
        const int gi = i0 + col, gj = j0 + row;
        gk[r] = FULL || (q < LPL && gi <= g.nx + 1 && gj <= g.ny + 1);
        go[r] = gi + sy * gj;
        gii[r] = gk[r] ? wrap(gi, g.nx) : 1;
        gjj[r] = gk[r] ? wrap(gj, g.ny) : 1;
    }
    double pre[3][NLD];
    int kpre = 0;
    // interior: 1 <= kp <= nz - 1 is known (no wall rule applies to the plane)
    auto fetch = [&](int kp, bool interior = false) {
        kpre = kp;
        if (FILL) {
            const int ks = kp == 0 ? 1 : (kp == g.nz + 1 ? g.nz : kp);
#pragma unroll
            for (int f = 0; f < 3; ++f)
#pragma unroll
                for (int r = 0; r < NLD; ++r)
                    pre[f][r] = gk[r] ? Q[f][gii[r] + sy * gjj[r] + sz * ks] : 0.0;
        } else {
#pragma unroll
            for (int f = 0; f < 3; ++f)
#pragma unroll
                for (int r = 0; r < NLD; ++r) pre[f][r] = gk[r] ? Q[f][go[r] + sz * kp] : 0.0;
        }
    };
    // interior: the plane put lies strictly inside (1 <= kp <= nz - 1), so no
    // wall rule of the fill applies (the FULL loop's planes but the last two)
    auto put = [&](int b, bool interior = false) {
        if (FILL && !interior) {
            const int kp = kpre;
            if (kp == 0 || kp == g.nz + 1) {
                const double bcu = 0.0 - g.u_crf;
#pragma unroll
                for (int r = 0; r < NLD; ++r) {
                    pre[0][r] = 2.0 * bcu - pre[0][r];
                    pre[1][r] = 2.0 * 0.0 - pre[1][r];
                    pre[2][r] = 0.0;
                }
            } else if (kp == g.nz) {
#pragma unroll
                for (int r = 0; r < NLD; ++r) pre[2][r] = 0.0;
            }
        }
#pragma unroll
        for (int f = 0; f < 3; ++f)
#pragma unroll
            for (int r = 0; r < NLD; ++r) {
                const int q = FULL ? min(tid + r * NT, LPL - 1) : tid + r * NT;
                if (FULL || q < LPL) tl[b][f][q] = pre[f][r];
            }
    };
    fetch(k0);
    put(0);
    fetch(k0 + 1);
    put(1);
    long long e = i + sy * j + sz * k0;
    double u00m = 0.0, v00m = 0.0, w00m = 0.0, wp0m = 0.0, w0pm = 0.0;
    if (valid) {
        if (FILL) {
            // plane k0 - 1 as the fill leaves it: a wall plane for k0 = 1
            auto fq = [&](const double *q, int f, int ii, int jj) -> double {
                const int kk = k0 - 1;
                if (kk == 0) {
                    if (f == 2) return 0.0;
                    const double bc = f == 0 ? 0.0 - g.u_crf : 0.0;
                    return 2.0 * bc - q[ii + sy * jj + sz * 1];
                }
                return q[ii + sy * jj + sz * kk];  // kk < nz: no wall row here
            };
            u00m = fq(qu, 0, i, j);
            v00m = fq(qv, 1, i, j);
            w00m = fq(qw, 2, i, j);
            wp0m = fq(qw, 2, wrap(i + 1, g.nx), j);
            w0pm = fq(qw, 2, i, wrap(j + 1, g.ny));
        } else {
            u00m = qu[e - sz];
            v00m = qv[e - sz];
            w00m = qw[e - sz];
            wp0m = qw[e - sz + 1];
            w0pm = qw[e - sz + sy];
        }
    }
    __syncthreads();
    double su = 0.0, sv = 0.0;
    const int c0 = (ly + 1) * LTX + lx + 1;  // this cell in a tile
    // plane k from LDS buffer b (plane k+1 in b ^ 1); old: RK2's previous
    // values of plane k when loaded ahead (FULL), else read here
    auto compute = [&](int kv, int b, long long ek, const double *old) {
        // k is the same for the whole workgroup: the z metrics come through
        // the scalar unit (scalar loads wait on their own counter)
        const int k = __builtin_amdgcn_readfirstlane(kv);
        const double *cu = tl[b][0], *cv = tl[b][1], *cw = tl[b][2];
        const double *nu = tl[b ^ 1][0], *nv = tl[b ^ 1][1], *nw = tl[b ^ 1][2];
        Nb n;
        n.u000 = cu[c0]; n.up00 = cu[c0 + 1]; n.um00 = cu[c0 - 1];
        n.u0p0 = cu[c0 + LTX]; n.u0m0 = cu[c0 - LTX]; n.ump0 = cu[c0 - 1 + LTX];
        n.u00p = nu[c0]; n.um0p = nu[c0 - 1]; n.u00m = u00m;
        n.v000 = cv[c0]; n.vp00 = cv[c0 + 1]; n.vm00 = cv[c0 - 1];
        n.v0p0 = cv[c0 + LTX]; n.v0m0 = cv[c0 - LTX]; n.vpm0 = cv[c0 + 1 - LTX];
        n.v00p = nv[c0]; n.v0mp = nv[c0 - LTX]; n.v00m = v00m;
        n.w000 = cw[c0]; n.wp00 = cw[c0 + 1]; n.wm00 = cw[c0 - 1];
        n.w0p0 = cw[c0 + LTX]; n.w0m0 = cw[c0 - LTX]; n.w00p = nw[c0];
        n.w00m = w00m; n.wp0m = wp0m; n.w0pm = w0pm;
        double fu, fv, fw;
        mom_rhs(g, n, k, fu, fv, fw);
        if (BODY) {
            fu = fu + fb.u[ek];
            fv = fv + fb.v[ek];
            fw = fw + fb.w[ek];
        }
        if (SECOND) {
            const double ou0 = old ? old[0] : ou[ek], ov0 = old ? old[1] : ov[ek],
                         ow0 = old ? old[2] : ow[ek];
            const double un = (n.u000 + g.dt * fu + ou0) * 0.5;
            const double vn = (n.v000 + g.dt * fv + ov0) * 0.5;
            ou[ek] = un;
            ov[ek] = vn;
            ow[ek] = (n.w000 + g.dt * fw + ow0) * 0.5;
            if (MEAN) {
                // both sums are formed (no branch in the loop); a component
                // not in fmask reports 0
                const double wk = pll::zm(g.dzflzi, k);
                su = su + un * wk;
                sv = sv + vn * wk;
            }
        } else {
            ou[ek] = n.u000 + g.dt * fu;
            ov[ek] = n.v000 + g.dt * fv;
            ow[ek] = n.w000 + g.dt * fw;
        }
        u00m = n.u000;
        v00m = n.v000;
        w00m = n.w000;
        wp0m = n.wp00;
        w0pm = n.w0p0;
    };
    if constexpr (FULL) {
        double oldc[3] = {0.0, 0.0, 0.0};
        // every load of the prologue has arrived before the loop starts, so that
        // no wait inside the loop (which covers its first iteration too) has
        // to include the loads in flight at that point
        asm volatile("" : : "v"(u00m), "v"(v00m), "v"(w00m), "v"(wp0m), "v"(w0pm));
        auto step = [&](int k, auto INTERIOR) {
            const int b = (k - k0) & 1;
            if (SECOND) {
                // RK2's old values of plane k, issued before the prefetch so
                // that waiting for them leaves the prefetch in flight
                oldc[0] = ou[e];
                oldc[1] = ov[e];
                oldc[2] = ow[e];
            }
            fetch(min(k + 2, k1 + 1), decltype(INTERIOR)::value);
            // keep the prefetch ahead of the arithmetic (the scheduler would
            // otherwise sink part of it next to its use)
            __builtin_amdgcn_sched_barrier(0);
            compute(k, b, e, SECOND ? oldc : nullptr);
            __syncthreads();                      // plane k's buffer is free
            put(b, decltype(INTERIOR)::value);    // it becomes plane k+2 (the last
            __syncthreads();                      // two: a plane not read)
            e += sz;
        };
        // planes whose plane k+2 lies inside take the put without the wall
        // rules: a wall rule in the loop would let the compiler move the w
        // prefetch into its branch, next to its use
        const int kin = min(k1, g.nz - 3);
        int k = k0;
#pragma unroll 1
        for (; k <= kin; ++k) step(k, std::true_type{});
#pragma unroll 1
        for (; k <= k1; ++k) step(k, std::false_type{});
    } else {
        for (int k = k0; k <= k1; ++k, e += sz) {
            const int b = (k - k0) & 1;
            const bool more = k + 2 <= k1 + 1;
            if (more) fetch(k + 2);
            if (valid) compute(k, b, e, nullptr);
            __syncthreads();  // plane k's buffer is free
            if (more) put(b);  // it becomes plane k+2
            __syncthreads();
        }
    }
    if (MEAN) {
        __shared__ double red[2][NT];
        red[0][tid] = su;
        red[1][tid] = sv;
        __syncthreads();
        for (int h = NT / 2; h > 0; h >>= 1) {
            if (tid < h) {
                red[0][tid] += red[0][tid + h];
                red[1][tid] += red[1][tid + h];
            }
            __syncthreads();
        }
        if (tid == 0) {
            mpart[blockIdx.x] = (fmask & 1) ? red[0][0] : 0.0;
            mpart[gridDim.x + blockIdx.x] = (fmask & 2) ? red[1][0] : 0.0;
        }
    }
}

// correctVel (mod_calcVel.f90:428-453) marching over a k chunk (p(k+1) is the
// next step's p(k)).  FORCE: then forceVel's shift q += vel_force - mean for
// the components in fmask (bit 0 u, bit 1 v), with the means in mean[0..1],
// in the same two roundings as correctVel followed by forceVel.
// Reads (qu, qv, qw) and writes (u, v, w), which may be the same arrays.
// FILL: then the boundary fill of the result (k_bc_vel, which every ghost value
// is a copy or reflection of one corrected cell in): a cell next to a face
// stores its images too, and w's wall row is zero.  Bound by its memory traffic
// (4.6 TB/s at 768x384x256; the next plane loaded ahead: 2% slower).  Against a
// fill of its own, whose few threads wait for one strided load and store each:
// 64x64x64 6.4 + 11.9 -> 8.2 us, 256x192x128 70 + 18 -> 72, 768x384x256 917 + 59
// -> 980.  At 1536x1024x384 the images cost more than the pass (7.3 + 0.15 ms,
// together 7.9), so grids above 2^27 cells take the two.
template <bool FORCE, bool FILL>
__global__ void __launch_bounds__(RK_TX *RK_TY) k_correct(G g, Tiles t, const double *__restrict__ p,
                                                          const double *qu, const double *qv,
                                                          const double *qw, double *u, double *v,
                                                          double *w, double dtdxi, double dtdyi,
                                                          int fmask, double vfu, double vfv,
                                                          const double *__restrict__ mean)
{
    int tx, ty, kc;
    rk_tile(t, tx, ty, kc);
    const int i = tx * RK_TX + (int)(threadIdx.x % RK_TX) + 1;
    const int j = ty * RK_TY + (int)(threadIdx.x / RK_TX) + 1;
    if (i > g.nx || j > g.ny) return;
    const int k0 = kc * t.kc + 1, k1 = min(k0 + t.kc - 1, g.nz);
    const long long sy = g.sy, sz = g.sz;
    long long e = i + sy * j + sz * k0;
    double fu = 0.0, fv = 0.0;
    if (FORCE) {
        if (fmask & 1) fu = vfu - mean[0];
        if (fmask & 2) fv = vfv - mean[1];
    }
    // (un, vn, wn) at e and at the cell's images across the periodic faces
    // (nx, ny >= 2: at most one in each direction)
    const long long ox = i == 1 ? g.nx : (i == g.nx ? -g.nx : 0);
    const long long oy = (j == 1 ? g.ny : (j == g.ny ? -g.ny : 0)) * sy;
    auto put = [&](long long a, double un, double vn, double wn) {
        u[a] = un;
        v[a] = vn;
        w[a] = wn;
    };
    auto store = [&](long long a, double un, double vn, double wn) {
        put(a, un, vn, wn);
        if (FILL && ox) put(a + ox, un, vn, wn);
        if (FILL && oy) {
            put(a + oy, un, vn, wn);
            if (ox) put(a + oy + ox, un, vn, wn);
        }
    };
    const double bcu = 0.0 - g.u_crf;
    double pc = p[e];
    for (int k = k0; k <= k1; ++k, e += sz) {
        if (FILL) asm volatile("" : "+v"(e));  // no kept address per field and image
        const double pz = p[e + sz];
        double un = qu[e] - (p[e + 1] - pc) * dtdxi;
        double vn = qv[e] - (p[e + sy] - pc) * dtdyi;
        const double wn = qw[e] - (pz - pc) * g.dt * g.dzc_inv[k];
        if (FORCE && (fmask & 1)) un = un + fu;
        if (FORCE && (fmask & 2)) vn = vn + fv;
        store(e, un, vn, FILL && k == g.nz ? 0.0 : wn);
        if (FILL && k == 1) store(e - sz, 2.0 * bcu - un, 2.0 * 0.0 - vn, 0.0);
        if (FILL && k == g.nz) store(e + sz, 2.0 * bcu - un, 2.0 * 0.0 - vn, 0.0);
        pc = pz;
    }
}

#define CELL_IDX                                                   \
    const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;       \
    const int j = blockIdx.y * blockDim.y + threadIdx.y + 1;       \
    const int k = blockIdx.z + 1;                                  \
    if (i > g.nx || j > g.ny) return;                              \
    const long long e = i + g.sy * j + g.sz * k;

__global__ void __launch_bounds__(256) k_calc_rhs(G g, const double *__restrict__ u,
                                                   const double *__restrict__ v,
                                                   const double *__restrict__ w,
                                                   double *__restrict__ rhs, double dti,
                                                   double dtidxi, double dtidyi)
{
    CELL_IDX
    rhs[e] = (u[e] - u[e - 1]) * dtidxi + (v[e] - v[e - g.sy]) * dtidyi +
             (w[e] - w[e - g.sz]) * dti * g.dzf_inv[k];
}

// One workgroup per interior (j,k) row: sum_i q(i,j,k)*dzflzi(k).
__global__ void __launch_bounds__(256) k_mean_part(G g, const double *__restrict__ q,
                                                    double *__restrict__ part)
{
    __shared__ double sh[256];
    const int j = blockIdx.x % g.ny + 1, k = blockIdx.x / g.ny + 1;
    const long long base = g.sy * j + g.sz * k;
    const double wk = g.dzflzi[k];
    double s = 0.0;
    for (int i = threadIdx.x + 1; i <= g.nx; i += blockDim.x) s = s + q[base + i] * wk;
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < 128) sh[threadIdx.x] += sh[threadIdx.x + 128];
    __syncthreads();
    if (threadIdx.x < 64) {
        double r = sh[threadIdx.x] + sh[threadIdx.x + 64];
        for (int h = 32; h > 0; h >>= 1) r += __shfl_down(r, h);
        if (threadIdx.x == 0) part[blockIdx.x] = r;
    }
}

__global__ void __launch_bounds__(1024) k_mean_final(int n, const double *__restrict__ part,
                                                      double *__restrict__ out, double nx,
                                                      double ny)
{
    __shared__ double sh[1024];
    double s = 0.0;
    // eight partials in flight per thread, added in order (98304 partials, one
    // at a time: 38 us)
    const int nb = blockDim.x;
    int t = threadIdx.x;
    for (; t + 7 * nb < n; t += 8 * nb) {
        double o[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) o[q] = part[t + q * nb];
#pragma unroll
        for (int q = 0; q < 8; ++q) s += o[q];
    }
    for (; t < n; t += nb) s += part[t];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 32; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < 64) {
        double r = sh[threadIdx.x];
        r = threadIdx.x < 32 ? r + sh[threadIdx.x + 32] : r;
        for (int h = 16; h > 0; h >>= 1) r += __shfl_down(r, h);
        if (threadIdx.x == 0) out[0] = r / nx / ny;
    }
}

__global__ void __launch_bounds__(256) k_force_shift(G g, double *__restrict__ q, double vel_force,
                                                      const double *__restrict__ mean)
{
    CELL_IDX
    const double force = vel_force - mean[0];
    q[e] = q[e] + force;
}

// Ghost cells after updateHalo (y periodic, full x/z range), imposePeriodicBC
// in x (full y/z range) and the wall conditions, in that order.  Every ghost
// value is a function of interior values only:
//   1 <= k <= nz:  q(wrap i, wrap j, k)        (w: 0 on the wall row k = nz)
//   k = 0, nz+1:   u,v: 2*bc - q(wrap i, wrap j, 1 | nz);  w: 0
// Work items: the two z planes (plus w's wall row k = nz), then the y faces
// and x faces of the interior k range.
__device__ __forceinline__ bool shell_pos(const G &g, long long t, int &i, int &j, int &k,
                                          int nplanes, const int *planes)
{
    const long long nxh = g.nx + 2, nyh = g.ny + 2;
    const long long nzp = nxh * nyh * nplanes;
    if (t < nzp) {
        const int pl = (int)(t / (nxh * nyh));
        const long long r = t % (nxh * nyh);
        i = (int)(r % nxh);
        j = (int)(r / nxh);
        k = planes[pl];
        return true;
    }
    t -= nzp;
    const long long nyf = 2 * nxh * g.nz;
    if (t < nyf) {
        const int side = (int)(t / (nxh * g.nz));
        const long long r = t % (nxh * g.nz);
        i = (int)(r % nxh);
        k = (int)(r / nxh) + 1;
        j = side ? g.ny + 1 : 0;
        return true;
    }
    t -= nyf;
    const long long nxf = 2LL * g.ny * g.nz;
    if (t < nxf) {
        const int side = (int)(t / ((long long)g.ny * g.nz));
        const long long r = t % ((long long)g.ny * g.nz);
        j = (int)(r % g.ny) + 1;
        k = (int)(r / g.ny) + 1;
        i = side ? g.nx + 1 : 0;
        return true;
    }
    return false;
}

__global__ void __launch_bounds__(256) k_bc_vel(G g, double *__restrict__ u, double *__restrict__ v,
                                                 double *__restrict__ w, long long total)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int planes[3] = {0, g.nz + 1, g.nz};
    int i, j, k;
    if (!shell_pos(g, t, i, j, k, 3, planes)) return;
    const long long e = i + g.sy * j + g.sz * k;
    const int ii = wrap(i, g.nx), jj = wrap(j, g.ny);
    const double bcu = 0.0 - g.u_crf;
    if (k == 0 || k == g.nz + 1) {
        const int ks = k == 0 ? 1 : g.nz;
        const long long s = ii + g.sy * jj + g.sz * ks;
        u[e] = 2.0 * bcu - u[s];
        v[e] = 2.0 * 0.0 - v[s];
        w[e] = 0.0;
    } else if (k == g.nz && t < 3LL * (g.nx + 2) * (g.ny + 2)) {
        // w's wall row, every (i,j); u and v there are ordinary cells.
        w[e] = 0.0;
        if (i != ii || j != jj) {
            const long long s = ii + g.sy * jj + g.sz * k;
            u[e] = u[s];
            v[e] = v[s];
        }
    } else {
        const long long s = ii + g.sy * jj + g.sz * k;
        u[e] = u[s];
        v[e] = v[s];
        w[e] = (k == g.nz) ? 0.0 : w[s];
    }
}

__global__ void __launch_bounds__(256) k_bc_p(G g, double *__restrict__ p, long long total)
{
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int planes[2] = {0, g.nz + 1};
    int i, j, k;
    if (!shell_pos(g, t, i, j, k, 2, planes)) return;
    const long long e = i + g.sy * j + g.sz * k;
    const int ii = wrap(i, g.nx), jj = wrap(j, g.ny);
    const int ks = k == 0 ? 1 : (k == g.nz + 1 ? g.nz : k);
    p[e] = p[ii + g.sy * jj + g.sz * ks];
}

// One workgroup per interior (j,k) row: max |div| and the smallest linear
// index (k-1)*nx*ny + (j-1)*nx + (i-1) attaining it.
// KIND 0: |div u| (calcMaxDiv, mod_utils.f90:286-288);
// KIND 1: the CFL sum before the factor dt (calcMaxCFL, mod_utils.f90:224-226)
//   |(u_i + u_{i-1})/2| dx_inv + |(v_j + v_{j-1})/2| dy_inv + |(w_k + w_{k-1})/2| dzf_inv(k).
// NaN cells never win (every comparison with NaN is false), as in the
// reference's `if (x > max)` loops.
template <int KIND>
__global__ void __launch_bounds__(256) k_maxloc_part(G g, const double *__restrict__ u,
                                                      const double *__restrict__ v,
                                                      const double *__restrict__ w,
                                                      double *__restrict__ pval,
                                                      long long *__restrict__ pidx)
{
    __shared__ double sv[256];
    __shared__ long long si[256];
    // Rows go to the 8 XCDs (which take workgroups round-robin) as y slabs:
    // XCD x works through rows j in [x ny/8, (x+1) ny/8) of one plane after
    // the other, so the rows j-1 and k-1 that a row reads were fetched into
    // the same L2 shortly before (ny % 8 == 0; plain row order otherwise).
    // The partials are reduced with ties to the lowest cell index, so the
    // result does not depend on the order.
    int j, k;
    if (g.ny % 8 == 0) {
        const int sl = g.ny >> 3, p = (int)(blockIdx.x >> 3);
        j = (int)(blockIdx.x & 7) * sl + p % sl + 1;
        k = p / sl + 1;
    } else {
        j = blockIdx.x % g.ny + 1;
        k = blockIdx.x / g.ny + 1;
    }
    const long long base = g.sy * j + g.sz * k;
    double best = -1.0;
    long long bi = 0;
    for (int i = threadIdx.x + 1; i <= g.nx; i += blockDim.x) {
        const long long e = base + i;
        double d;
        if (KIND == 0)
            d = fabs((u[e] - u[e - 1]) * g.dx_inv + (v[e] - v[e - g.sy]) * g.dy_inv +
                     (w[e] - w[e - g.sz]) * g.dzf_inv[k]);
        else
            d = fabs((u[e] + u[e - 1]) * 0.5) * g.dx_inv + fabs((v[e] + v[e - g.sy]) * 0.5) * g.dy_inv +
                fabs((w[e] + w[e - g.sz]) * 0.5) * g.dzf_inv[k];
        if (d > best) {
            best = d;
            bi = (long long)(k - 1) * g.nx * g.ny + (long long)(j - 1) * g.nx + (i - 1);
        }
    }
    sv[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            const double o = sv[threadIdx.x + h];
            const long long oi = si[threadIdx.x + h];
            if (o > sv[threadIdx.x] || (o == sv[threadIdx.x] && oi < si[threadIdx.x])) {
                sv[threadIdx.x] = o;
                si[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        pval[blockIdx.x] = sv[0];
        pidx[blockIdx.x] = si[0];
    }
}

__global__ void __launch_bounds__(1024) k_maxdiv_final(int n, const double *__restrict__ pval,
                                                        const long long *__restrict__ pidx,
                                                        double *__restrict__ oval,
                                                        long long *__restrict__ oidx)
{
    __shared__ double sv[1024];
    __shared__ long long si[1024];
    double best = -1.0;
    long long bi = 0;
    // eight partials in flight per thread (one at a time leaves the loop
    // waiting on memory latency: 54 us for 98304 partials)
    const int nb = blockDim.x;
    int t = threadIdx.x;
    for (; t + 7 * nb < n; t += 8 * nb) {
        double o[8];
        long long oi[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            o[q] = pval[t + q * nb];
            oi[q] = pidx[t + q * nb];
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (o[q] > best || (o[q] == best && oi[q] < bi)) {
                best = o[q];
                bi = oi[q];
            }
    }
    for (; t < n; t += nb) {
        const double o = pval[t];
        const long long oi = pidx[t];
        if (o > best || (o == best && oi < bi)) {
            best = o;
            bi = oi;
        }
    }
    sv[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) {
            const double o = sv[threadIdx.x + h];
            const long long oi = si[threadIdx.x + h];
            if (o > sv[threadIdx.x] || (o == sv[threadIdx.x] && oi < si[threadIdx.x])) {
                sv[threadIdx.x] = o;
                si[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        oval[0] = sv[0];
        oidx[0] = si[0];
    }
}

// The run-time checks in one pass over u, v, w: calcMaxCFL's sum (value 0),
// calcMaxDiv's (value 1), both with location as k_maxloc_part, and checkNaN of
// u (ghost cells included).  Up to CHK workgroups share the rows, in y slabs per XCD
// as there; each leaves one partial of either maximum (pval, pidx: value 0 of
// every workgroup, then value 1) and a NaN flag (after both locations).
// Bound by HBM: 24 N bytes for the 56 N of the three separate passes;
// 768x384x256 0.40 ms (4.6 TB/s) for 0.34 + 0.34 + 0.17 and their final passes.
constexpr int CHK = PLL_CHECK_BLOCKS;

struct MaxLoc {
    double v;
    long long i;
};
__device__ __forceinline__ void take(MaxLoc &a, double v, long long i)
{
    if (v > a.v || (v == a.v && i < a.i)) {
        a.v = v;
        a.i = i;
    }
}
__device__ __forceinline__ void take_wave(MaxLoc &a)
{
    for (int h = 32; h > 0; h >>= 1) {
        const double v = __shfl_xor(a.v, h);
        const long long i = __shfl_xor(a.i, h);
        take(a, v, i);
    }
}

__global__ void __launch_bounds__(256) k_check_part(G g, const double *__restrict__ u,
                                                    const double *__restrict__ v,
                                                    const double *__restrict__ w, long long nshell,
                                                    double *__restrict__ pval,
                                                    long long *__restrict__ pidx)
{
    MaxLoc c{-1.0, 0}, d{-1.0, 0};
    int bad = 0;
    const bool slab = g.ny % 8 == 0;
    const int sl = g.ny >> 3, x = blockIdx.x & 7;
    const long long rows = slab ? (long long)sl * g.nz : (long long)g.ny * g.nz;
    const long long r0 = slab ? blockIdx.x >> 3 : blockIdx.x, dr = slab ? gridDim.x >> 3 : gridDim.x;
    for (long long r = r0; r < rows; r += dr) {
        const int k = (int)(r / (slab ? sl : g.ny)) + 1;
        const int j = slab ? x * sl + (int)(r % sl) + 1 : (int)(r % g.ny) + 1;
        const long long base = g.sy * j + g.sz * k;
        const double dzi = g.dzf_inv[k];
        for (int i = threadIdx.x + 1; i <= g.nx; i += 256) {
            const long long e = base + i;
            const double uc = u[e], um = u[e - 1], vc = v[e], vm = v[e - g.sy], wc = w[e],
                         wm = w[e - g.sz];
            bad |= uc != uc;
            const double cfl = fabs((uc + um) * 0.5) * g.dx_inv + fabs((vc + vm) * 0.5) * g.dy_inv +
                               fabs((wc + wm) * 0.5) * dzi;
            const double div = fabs((uc - um) * g.dx_inv + (vc - vm) * g.dy_inv + (wc - wm) * dzi);
            const long long at = ((long long)(k - 1) * g.ny + (j - 1)) * g.nx + (i - 1);
            take(c, cfl, at);
            take(d, div, at);
        }
    }
    const int planes[2] = {0, g.nz + 1};
    for (long long t = (long long)blockIdx.x * 256 + threadIdx.x; t < nshell;
         t += gridDim.x * 256LL) {
        int i, j, k;
        if (shell_pos(g, t, i, j, k, 2, planes)) {
            const double q = u[i + g.sy * j + g.sz * k];
            bad |= q != q;
        }
    }
    __shared__ MaxLoc red[2][4];
    take_wave(c);
    take_wave(d);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = c;
        red[1][threadIdx.x >> 6] = d;
    }
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q) {
            take(c, red[0][q].v, red[0][q].i);
            take(d, red[1][q].v, red[1][q].i);
        }
        pval[blockIdx.x] = c.v;
        pidx[blockIdx.x] = c.i;
        pval[gridDim.x + blockIdx.x] = d.v;
        pidx[gridDim.x + blockIdx.x] = d.i;
        pidx[2 * gridDim.x + blockIdx.x] = bad;
    }
}

// res: two maxima, then their locations and the NaN flag (8 bytes each)
__global__ void __launch_bounds__(1024) k_check_final(int n, const double *__restrict__ pval,
                                                      const long long *__restrict__ pidx,
                                                      double *__restrict__ res)
{
    MaxLoc m[2] = {{-1.0, 0}, {-1.0, 0}};
    int bad = 0;
#pragma unroll 4
    for (int t = threadIdx.x; t < n; t += 1024) {
        take(m[0], pval[t], pidx[t]);
        take(m[1], pval[n + t], pidx[n + t]);
        bad |= pidx[2 * n + t] != 0;
    }
    __shared__ MaxLoc red[2][16];
    for (int f = 0; f < 2; ++f) {
        take_wave(m[f]);
        if ((threadIdx.x & 63) == 0) red[f][threadIdx.x >> 6] = m[f];
    }
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
        long long *ri = reinterpret_cast<long long *>(res);
        for (int f = 0; f < 2; ++f) {
            for (int q = 1; q < 16; ++q) take(m[f], red[f][q].v, red[f][q].i);
            res[f] = m[f].v;
            ri[2 + f] = m[f].i;
        }
        ri[4] = bad;
    }
}

inline dim3 cell_grid(const G &g) { return dim3((g.nx + 63) / 64, (g.ny + 3) / 4, g.nz); }
// checkNaN (mod_utils.f90:352-394) over every element of a haloed field:
// flags[block] = 1 if the block's stride of elements holds a NaN.
__global__ void __launch_bounds__(256) k_nan_part(const double *__restrict__ q, long long n,
                                                  long long *__restrict__ flags)
{
    int bad = 0;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x)
        bad |= q[t] != q[t];
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) flags[blockIdx.x] = bad;
}

inline int ok() { return hipGetLastError() == hipSuccess ? 0 : -3; }

// Planes per k chunk (PLL_RK_KC overrides): at first the largest power of two up
// to 64 that leaves at least 2048 workgroups.  A chunk costs two planes of loads
// before its first result, so long chunks are cheaper per plane; but the chip
// holds 4 workgroups per CU, 1024, and with fewer than two rounds of them it
// idles (a 64-plane chunk of a 64x64x64 grid makes 16 workgroups).  Measured,
// 64-plane chunks against the rule: step at 64x64x64 219 -> 75 us; per step
// of a run, 96x96x96 312 -> 121 us (2 planes), 192x192x128 432 -> 317 us (8),
// 240x140x90 492 -> 347 us (4), 384x384x192 1.81 -> 1.51 ms (32; 64 leaves
// 1728 workgroups); at 512x384x256 the rule keeps 64 (2.61 ms, 32: 2.62,
// 16: 2.64), and one size up or down from its choice is 0 to 20% slower.
// The planes are then spread evenly over as many chunks: with the XCD numbering
// an XCD runs the tiles of one or two chunks, and short ones leave it idle (step
// at 768x384x39 as 32 + 7 planes 884 us, as 20 + 19 726, as one chunk 728).
constexpr int RK_WG_MIN = 2048, RK_KC_MAX = 64;

Tiles rk_tiles(const G &g)
{
    Tiles t;
    t.ntx = (g.nx + RK_TX - 1) / RK_TX;
    t.nty = (g.ny + RK_TY - 1) / RK_TY;
    const long long cols = (long long)t.ntx * t.nty;
    t.kc = RK_KC_MAX;
    while (t.kc > 1 && cols * ((g.nz + t.kc - 1) / t.kc) < RK_WG_MIN) t.kc >>= 1;
    const int n = (g.nz + t.kc - 1) / t.kc;
    t.kc = g.kc > 0 ? g.kc : (g.nz + n - 1) / n;
    t.nkc = (g.nz + t.kc - 1) / t.kc;
    t.xcd = (cols * t.nkc) % 8 == 0;
    return t;
}

}  // namespace

extern "C" void pll_rk_tiling(const pll_grid_dev *gd, int rk[5])
{
    const Tiles t = rk_tiles(make_g(gd));
    rk[0] = t.ntx;
    rk[1] = t.nty;
    rk[2] = t.nkc;
    rk[3] = t.kc;
    rk[4] = t.xcd;
}

extern "C" int pll_rk_blocks(const pll_grid_dev *gd)
{
    const Tiles t = rk_tiles(make_g(gd));
    return t.ntx * t.nty * t.nkc;
}

// runtime flags -> template instantiation
template <typename F>
int with_flags(bool a, bool b, bool c, F &&f)
{
#define PLL_B3(A, B, C) \
    if (a == A && b == B && c == C) return f(std::integral_constant<bool, A>{}, std::integral_constant<bool, B>{}, std::integral_constant<bool, C>{});
    PLL_B3(false, false, false) PLL_B3(false, false, true) PLL_B3(false, true, false)
    PLL_B3(false, true, true) PLL_B3(true, false, false) PLL_B3(true, false, true)
    PLL_B3(true, true, false) PLL_B3(true, true, true)
#undef PLL_B3
    return -1;
}

// Grids whose RK tiles all lie inside take the FULL kernel for RK1
// (768x384x256: 0.94 ms either way); RK2's FULL form needs 145 VGPRs (3 waves per SIMD
// against 4) and runs 1.314 ms against 1.304, so RK2 keeps the general form
// unless PLL_RK2_FULL=1.  PLL_RK_FULL=0 takes the general kernels everywhere.
// (read at every launch, so that one process can time both forms)
bool full_tiles(const G &g, int ty, bool second = false)
{
    const char *e = getenv("PLL_RK_FULL");
    const char *e2 = getenv("PLL_RK2_FULL");
    const bool allow = !(e && atoi(e) == 0), allow2 = e2 && atoi(e2) != 0;
    return allow && (!second || allow2) && g.nx % RK_TX == 0 && g.ny % ty == 0;
}

extern "C" int pll_launch_rk1(const pll_grid_dev *gd, const double *u, const double *v,
                              const double *w, double *u1, double *v1, double *w1,
                              const double *const *body, hipStream_t s)
{
    const G g = make_g(gd);
    const Tiles t = rk_tiles(g);
    const dim3 grid((unsigned)(t.ntx * t.nty * t.nkc)), blk(RK_TX * RK_TY);
    const Body fb = body ? Body{body[0], body[1], body[2]} : Body{nullptr, nullptr, nullptr};
    return with_flags(false, body != nullptr, full_tiles(g, RK_TY), [&](auto, auto B, auto F) {
        hipLaunchKernelGGL((k_rk<false, false, decltype(B)::value, false, decltype(F)::value>),
                           grid, blk, 0, s, g, t, u, v, w, u1, v1, w1, nullptr, 0, fb);
        return ok();
    });
}

extern "C" int pll_launch_rk2(const pll_grid_dev *gd, double *u, double *v, double *w,
                              const double *u1, const double *v1, const double *w1,
                              double *mpart, int fmask, const double *const *body, int fill,
                              hipStream_t s)
{
    const G g = make_g(gd);
    const Tiles t = rk_tiles(g);
    const dim3 grid((unsigned)(t.ntx * t.nty * t.nkc)), blk(RK_TX * RK_TY);
    const Body fb = body ? Body{body[0], body[1], body[2]} : Body{nullptr, nullptr, nullptr};
    const bool mean = mpart && fmask;
    return with_flags(mean, body != nullptr, fill != 0, [&](auto M, auto B, auto F) {
        if (full_tiles(g, RK_TY, true))
            hipLaunchKernelGGL((k_rk<true, decltype(M)::value, decltype(B)::value, decltype(F)::value, true>),
                               grid, blk, 0, s, g, t, u1, v1, w1, u, v, w, mean ? mpart : nullptr,
                               mean ? fmask : 0, fb);
        else
            hipLaunchKernelGGL((k_rk<true, decltype(M)::value, decltype(B)::value, decltype(F)::value, false>),
                               grid, blk, 0, s, g, t, u1, v1, w1, u, v, w, mean ? mpart : nullptr,
                               mean ? fmask : 0, fb);
        return ok();
    });
}

extern "C" int pll_launch_calc_rhs(const pll_grid_dev *gd, const double *u, const double *v,
                                   const double *w, double *p, hipStream_t s)
{
    const G g = make_g(gd);
    const double dti = 1.0 / g.dt;  // mod_calcRHS.f90:21-23
    const double dtidxi = dti * g.dx_inv, dtidyi = dti * g.dy_inv;
    hipLaunchKernelGGL(k_calc_rhs, cell_grid(g), dim3(64, 4, 1), 0, s, g, u, v, w, p, dti, dtidxi,
                       dtidyi);
    return ok();
}

extern "C" int pll_launch_correct_vel(const pll_grid_dev *gd, const double *p,
                                      const double *const q[3], double *u, double *v,
                                      double *w, int fmask, double vfu, double vfv,
                                      const double *mean, int fill, hipStream_t s)
{
    const G g = make_g(gd);
    const Tiles t = rk_tiles(g);
    const double dtdxi = g.dt * g.dx_inv, dtdyi = g.dt * g.dy_inv;  // mod_calcVel.f90:436-437
    const dim3 grid((unsigned)(t.ntx * t.nty * t.nkc));
    const bool force = mean && fmask;
    const bool in = fill && (long long)g.nx * g.ny * g.nz <= 1LL << 27;
    const int rc = with_flags(force, in, false, [&](auto Fo, auto Fi, auto) {
        hipLaunchKernelGGL((k_correct<decltype(Fo)::value, decltype(Fi)::value>), grid,
                           dim3(RK_TX * RK_TY), 0, s, g, t, p, q[0], q[1], q[2], u, v, w, dtdxi,
                           dtdyi, force ? fmask : 0, vfu, vfv, force ? mean : nullptr);
        return ok();
    });
    return rc || !fill || in ? rc : pll_launch_bc_vel(gd, u, v, w, s);
}

extern "C" int pll_launch_mean_partials(const pll_grid_dev *gd, const double *q, double *part,
                                        hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_mean_part, dim3(g.ny * g.nz), dim3(256), 0, s, g, q, part);
    return ok();
}

extern "C" int pll_launch_mean_final(int n, const double *part, double *out, int nx, int ny,
                                      hipStream_t s)
{
    hipLaunchKernelGGL(k_mean_final, dim3(1), dim3(1024), 0, s, n, part, out, (double)nx,
                       (double)ny);
    return ok();
}

extern "C" int pll_launch_force_shift(const pll_grid_dev *gd, double *q, double vel_force,
                                      const double *mean, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_force_shift, cell_grid(g), dim3(64, 4, 1), 0, s, g, q, vel_force, mean);
    return ok();
}

extern "C" int pll_launch_bc_vel(const pll_grid_dev *gd, double *u, double *v, double *w,
                                 hipStream_t s)
{
    const G g = make_g(gd);
    const long long total = 3LL * (g.nx + 2) * (g.ny + 2) + 2LL * (g.nx + 2) * g.nz +
                            2LL * g.ny * g.nz;
    hipLaunchKernelGGL(k_bc_vel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, g, u, v,
                       w, total);
    return ok();
}

extern "C" int pll_launch_bc_p(const pll_grid_dev *gd, double *p, hipStream_t s)
{
    const G g = make_g(gd);
    const long long total = 2LL * (g.nx + 2) * (g.ny + 2) + 2LL * (g.nx + 2) * g.nz +
                            2LL * g.ny * g.nz;
    hipLaunchKernelGGL(k_bc_p, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, g, p, total);
    return ok();
}

extern "C" int pll_launch_maxdiv_partials(const pll_grid_dev *gd, const double *u,
                                          const double *v, const double *w, double *pval,
                                          long long *pidx, hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_maxloc_part<0>, dim3(g.ny * g.nz), dim3(256), 0, s, g, u, v, w, pval, pidx);
    return ok();
}

extern "C" int pll_launch_maxcfl_partials(const pll_grid_dev *gd, const double *u, const double *v,
                                          const double *w, double *pval, long long *pidx,
                                          hipStream_t s)
{
    const G g = make_g(gd);
    hipLaunchKernelGGL(k_maxloc_part<1>, dim3(g.ny * g.nz), dim3(256), 0, s, g, u, v, w, pval, pidx);
    return ok();
}

extern "C" int pll_launch_nan_partials(const pll_grid_dev *gd, const double *q, long long *flags,
                                       int nblocks, hipStream_t s)
{
    const G g = make_g(gd);
    const long long n = (long long)(g.nx + 2) * (g.ny + 2) * (g.nz + 2);
    hipLaunchKernelGGL(k_nan_part, dim3(nblocks), dim3(256), 0, s, q, n, flags);
    return ok();
}

extern "C" int pll_launch_maxdiv_final(int n, const double *pval, const long long *pidx,
                                       double *oval, long long *oidx, hipStream_t s)
{
    hipLaunchKernelGGL(k_maxdiv_final, dim3(1), dim3(1024), 0, s, n, pval, pidx, oval, oidx);
    return ok();
}

extern "C" int pll_launch_check(const pll_grid_dev *gd, const double *u, const double *v,
                                const double *w, double *pval, long long *pidx, double *res,
                                hipStream_t s)
{
    const G g = make_g(gd);
    const long long shell = 2LL * (g.nx + 2) * (g.ny + 2) + 2LL * (g.nx + 2) * g.nz +
                            2LL * g.ny * g.nz;
    const long long rows = (long long)g.ny * g.nz;
    // about twelve rows per workgroup, 2048 to 8192 of them (768x384x256 643 us per
    // check with 2048, 619 with 8192, 684 with 65536; 192x192x128 137, 159, 202:
    // more workgroups drift apart less, which keeps the neighbour rows in the
    // L2, but leave more partials and start-up)
    long long n8 = rows / 12;
    n8 = n8 < 2048 ? 2048 : (n8 > CHK ? CHK : n8);
    n8 = n8 < rows ? n8 : rows;
    const int n = (int)((n8 + 7) / 8 * 8);
    hipLaunchKernelGGL(k_check_part, dim3(n), dim3(256), 0, s, g, u, v, w, shell, pval, pidx);
    if (ok()) return -3;
    hipLaunchKernelGGL(k_check_final, dim3(1), dim3(1024), 0, s, n, pval, pidx, res);
    return ok();
}
