/*
 * Adjoint of the RK2 projection step over a window of steps (no counterpart
 * in the reference, which has no adjoint or body force).
 *
 * Objective: J = (1/nsteps) sum_{n=1..nsteps} tau_w(u^n), tau_w the wall
 * shear averaged over both walls (src/mod_monitor.f90:225-258).  Control: a
 * body force b = (bu, bv, bw) added to the momentum right-hand side of both
 * RK stages of every step (pll_channel_step_body).
 *
 * Forward: the steps run with checkpoints of (u,v,w) every `ckpt_every`
 * steps and leave the last segment's states in place.  Backward: per segment,
 * the states of the segment are recomputed from its checkpoint, then the steps
 * are reversed; each reversed step recomputes its RK1 stage (stage
 * recomputation).  One reversed step is the
 * transpose of the forward step's linearisation, in reverse order:
 *   boundary fill, forcing, correctVel, updateBoundP, PPE (transposed solve),
 *   calcRHS, boundary fill, RK2 (Jacobian at u1), boundary fill, RK1
 *   (Jacobian at u),
 * with grad b += dt/2 l* (RK2) + dt l1 (RK1).
 */
#include <stdlib.h>
#include <string.h>

#include "../../include/powerllel.h"
#include "pll_internal.h"

struct pll_adjoint {
    pll_channel *ch;
    pll_ppe *ppe;
    int nsteps, every, nck;
    size_t fbytes;           /* bytes of one haloed field */
    double *ck;              /* nck checkpoints x 3 fields */
    double *seg;             /* every states x 3 fields: see state() */
    double *u1, *p;          /* 3 fields, 1 field */
    double *lam, *lam1, *lamp, *body; /* 3, 3, 1, 3 fields */
    double *jpart, *tot;     /* device: partial sums of lam, the 3 sums */
    double *wsum;            /* device: 2 nsteps wall sums */
    double *part;            /* device: partials for the wall sums */
    double *hsum;            /* host: 2 nsteps */
    int have_forward;
    int held;                /* segment whose states are in seg (-1: none) */
    size_t dev_bytes;
};

static int hipchk(hipError_t e, const char *what)
{
    if (e == hipSuccess) return PLL_OK;
    return pll_set_error(PLL_EHIP, "%s: %s", what, hipGetErrorString(e));
}

static int launch(int rc, const char *what)
{
    if (rc == 0) return PLL_OK;
    return pll_set_error(PLL_EHIP, "%s: kernel launch failed: %s", what,
                         hipGetErrorString(hipGetLastError()));
}

int pll_adjoint_destroy(pll_adjoint *a)
{
    if (!a) return PLL_OK;
    void *bufs[] = {a->ck, a->seg, a->u1, a->p, a->lam, a->lam1, a->lamp, a->body,
                    a->wsum, a->part, a->jpart, a->tot};
    for (size_t i = 0; i < sizeof bufs / sizeof bufs[0]; i++)
        if (bufs[i]) hipFree(bufs[i]);
    free(a->hsum);
    free(a);
    return PLL_OK;
}

static int dalloc(pll_adjoint *a, double **p, size_t bytes)
{
    hipError_t e = hipMalloc((void **)p, bytes);
    if (e != hipSuccess) {
        *p = NULL;
        return pll_set_error(PLL_ENOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    }
    a->dev_bytes += bytes;
    return PLL_OK;
}

int pll_adjoint_create(pll_adjoint **out, pll_channel *ch, pll_ppe *ppe, int nsteps,
                       int ckpt_every)
{
    if (!out) return pll_set_error(PLL_EINVAL, "out is NULL");
    *out = NULL;
    if (!ch || !ppe) return pll_set_error(PLL_ESTATE, "channel or PPE handle is NULL");
    if (nsteps < 1 || ckpt_every < 1)
        return pll_set_error(PLL_EINVAL, "nsteps (%d) and ckpt_every (%d) must be >= 1", nsteps,
                             ckpt_every);
    if (pll_ppe_refinement(ppe) >= 0)
        return pll_set_error(PLL_EUNSUP, "the adjoint uses the FP64 solve (refinement is on)");
    const pll_grid_dev *g = pll_channel_grid(ch);
    pll_adjoint *a = (pll_adjoint *)calloc(1, sizeof *a);
    if (!a) return pll_set_error(PLL_ENOMEM, "calloc failed");
    a->ch = ch;
    a->ppe = ppe;
    a->nsteps = nsteps;
    a->every = ckpt_every < nsteps ? ckpt_every : nsteps;
    a->nck = (nsteps + a->every - 1) / a->every;
    const size_t nf = (size_t)(g->nx + 2) * (g->ny + 2) * (g->nz + 2);
    a->fbytes = nf * sizeof(double);
    int rc;
    if ((rc = dalloc(a, &a->ck, 3 * a->fbytes * (size_t)a->nck)) ||
        (rc = dalloc(a, &a->seg, 3 * a->fbytes * (size_t)a->every)) ||
        (rc = dalloc(a, &a->u1, 3 * a->fbytes)) || (rc = dalloc(a, &a->p, a->fbytes)) ||
        (rc = dalloc(a, &a->lam, 3 * a->fbytes)) || (rc = dalloc(a, &a->lam1, 3 * a->fbytes)) ||
        (rc = dalloc(a, &a->lamp, a->fbytes)) ||
        (rc = dalloc(a, &a->jpart, sizeof(double) * 3 * (size_t)pll_jtv_fold_blocks(g))) ||
        (rc = dalloc(a, &a->tot, sizeof(double) * 3)) ||
        (rc = dalloc(a, &a->body, 3 * a->fbytes)) ||
        (rc = dalloc(a, &a->wsum, sizeof(double) * 2 * (size_t)nsteps)) ||
        (rc = dalloc(a, &a->part, sizeof(double) * 2 * (size_t)g->ny))) {
        pll_adjoint_destroy(a);
        return rc;
    }
    a->hsum = (double *)malloc(sizeof(double) * 2 * (size_t)nsteps);
    if (!a->hsum) {
        pll_adjoint_destroy(a);
        return pll_set_error(PLL_ENOMEM, "malloc failed");
    }
    *out = a;
    return PLL_OK;
}

size_t pll_adjoint_device_bytes(const pll_adjoint *a) { return a ? a->dev_bytes : 0; }

/* field f (0..2) of the 3-field block at base */
static double *fld(const pll_adjoint *a, double *base, int f)
{
    return base + (size_t)f * (a->fbytes / sizeof(double));
}

static int copy3(const pll_adjoint *a, double *dst, const double *const src[3], hipStream_t s)
{
    for (int f = 0; f < 3; f++) {
        int rc = hipchk(hipMemcpyAsync(fld(a, dst, f), src[f], a->fbytes,
                                       hipMemcpyDeviceToDevice, s),
                        "copy");
        if (rc) return rc;
    }
    return PLL_OK;
}

/* Where state n of the window lives: the states at multiples of `every` are
 * the checkpoints (but the window's last state), the others go to slot
 * n mod every of seg, which holds one segment at a time. */
static double *state(const pll_adjoint *a, int n)
{
    const size_t f3 = 3 * (a->fbytes / sizeof(double));
    return n % a->every == 0 && n < a->nsteps ? a->ck + (size_t)(n / a->every) * f3
                                              : a->seg + (size_t)(n % a->every) * f3;
}

/* state n -> state n + 1; the ghosts of state 0 are the caller's */
static int step_fwd(pll_adjoint *a, int n, hipStream_t s)
{
    double *S = state(a, n), *D = state(a, n + 1);
    const double *src[3] = {fld(a, S, 0), fld(a, S, 1), fld(a, S, 2)};
    double *dst[3] = {fld(a, D, 0), fld(a, D, 1), fld(a, D, 2)};
    double *tmp[3] = {fld(a, a->u1, 0), fld(a, a->u1, 1), fld(a, a->u1, 2)};
    const double *body[3] = {fld(a, a->body, 0), fld(a, a->body, 1), fld(a, a->body, 2)};
    return pll_channel_step_from(a->ch, a->ppe, src, dst, tmp, a->p, body, n > 0, s);
}

int pll_adjoint_forward(pll_adjoint *a, const double *u0, const double *v0, const double *w0,
                        const double *bu, const double *bv, const double *bw, double *J,
                        void *stream)
{
    if (!a) return pll_set_error(PLL_ESTATE, "adjoint handle is NULL");
    if (!u0 || !v0 || !w0 || !bu || !bv || !bw || !J)
        return pll_set_error(PLL_EINVAL, "NULL argument");
    hipStream_t s = (hipStream_t)stream;
    const pll_grid_dev *g = pll_channel_grid(a->ch);
    const double *U0[3] = {u0, v0, w0}, *B[3] = {bu, bv, bw};
    int rc;
    if ((rc = copy3(a, a->body, B, s))) return rc;
    if ((rc = copy3(a, a->ck, U0, s))) return rc;
    a->held = -1;
    for (int n = 0; n < a->nsteps; n++) {
        if ((rc = step_fwd(a, n, s))) return rc;
        if ((rc = launch(pll_launch_wall_sum(g, state(a, n + 1), a->part, a->wsum + 2 * n, s),
                         "wall shear")))
            return rc;
    }
    a->held = a->nck - 1;
    if ((rc = hipchk(hipMemcpyAsync(a->hsum, a->wsum, sizeof(double) * 2 * (size_t)a->nsteps,
                                    hipMemcpyDeviceToHost, s),
                     "copy of wall sums")))
        return rc;
    if ((rc = hipchk(hipStreamSynchronize(s), "synchronise"))) return rc;
    double acc = 0.0;
    for (int n = 0; n < a->nsteps; n++) acc += pll_wall_shear_from_sums(a->ch, a->hsum + 2 * n);
    *J = acc / a->nsteps;
    a->have_forward = 1;
    return PLL_OK;
}

/* dJ/du on the wall planes for one state: (1/nsteps) * 1/2 * re_inv /
 * (nx ny dzf(kw)/2) */
static void seed(const pll_adjoint *a, double *cb, double *ct)
{
    const pll_grid_dev *g = pll_channel_grid(a->ch);
    const double *dzf = pll_channel_dzf_host(a->ch);
    const double nxy = (double)g->nx * g->ny;
    *cb = g->re_inv / (a->nsteps * nxy * dzf[1]);
    *ct = g->re_inv / (a->nsteps * nxy * dzf[g->nz]);
}

/* lam (adjoint of the state U_{n+1}, folded) -> adjoint of the state U_n
 * with J's reading of U_n added; U is U_n, its RK1 stage is recomputed into
 * u1.  Every adjoint field lives on the interior: the transposed boundary
 * fills are part of the passes on either side of them.
 *   lamp = transposed correctVel of lam, solved
 *   lam* = lam (forcing transposed) + transposed calcRHS of lamp
 *   RK2, u* = (u1 + dt (f(u1) + b) + u) / 2:  l1 = lam* / 2 + dt/2 J(u1)^T lam*
 *   RK1, u1 = u + dt (f(u) + b):  lam = lam* / 2 + l1 + dt J(u)^T l1 + dJ/dU_n
 *   grad += dt/2 lam* + dt l1
 * The sums of the new lam (for its transposed forcing) come out of the last
 * pass; fmask 0: lam has had its forcing transposed already.  last: the
 * adjoint of U_n is not wanted. */
static int step_adj(pll_adjoint *a, const double *U, double *const Gr[3], int fmask, int last,
                    hipStream_t s)
{
    pll_channel *ch = a->ch;
    const pll_grid_dev *g = pll_channel_grid(ch);
    const size_t nf = a->fbytes / sizeof(double);
    double *L[3] = {fld(a, a->lam, 0), fld(a, a->lam, 1), fld(a, a->lam, 2)};
    double *L1[3] = {fld(a, a->lam1, 0), fld(a, a->lam1, 1), fld(a, a->lam1, 2)};
    const double *Lc[3] = {L[0], L[1], L[2]}, *L1c[3] = {L1[0], L1[1], L1[2]};
    const double *Uc[3] = {U, U + nf, U + 2 * nf};
    double *U1[3] = {fld(a, a->u1, 0), fld(a, a->u1, 1), fld(a, a->u1, 2)};
    const double *U1c[3] = {U1[0], U1[1], U1[2]};
    const double *B[3] = {fld(a, a->body, 0), fld(a, a->body, 1), fld(a, a->body, 2)};
    const double h = 0.5 * g->dt;
    double cb, ct;
    int rc;
    seed(a, &cb, &ct);
    if ((rc = launch(pll_launch_rk1(g, Uc[0], Uc[1], Uc[2], U1[0], U1[1], U1[2], B, s), "rk1")) ||
        (rc = launch(pll_launch_correct_adj_fold(g, Lc, a->lamp, fmask, a->tot, s),
                     "correct_vel adjoint")) ||
        (rc = pll_ppe_solve_adjoint(a->ppe, a->lamp, s)) ||
        (rc = launch(pll_launch_rhs_adj_fold(g, a->lamp, L, fmask, a->tot, s),
                     "calc_rhs adjoint")) ||
        (rc = launch(pll_launch_jtv_fold(g, U1c, Lc, L1, NULL, h, 0.5, 0.0, NULL, 0.0, 0.0, 0.0,
                                         0.0, NULL, s),
                     "rk2 adjoint")))
        return rc;
    if (last) return launch(pll_launch_axpy3(g, g->dt, L1c, h, Lc, Gr, s), "gradient");
    if ((rc = launch(pll_launch_jtv_fold(g, Uc, L1c, L, Lc, g->dt, 1.0, 0.5, Gr, g->dt, h, cb, ct,
                                         a->jpart, s),
                     "rk1 adjoint")))
        return rc;
    return launch(pll_launch_sum3(pll_jtv_fold_blocks(g), a->jpart, a->tot,
                                  1.0 / ((double)g->nx * g->ny), s),
                  "forcing sums");
}

int pll_adjoint_backward(pll_adjoint *a, double *gu, double *gv, double *gw, void *stream)
{
    if (!a) return pll_set_error(PLL_ESTATE, "adjoint handle is NULL");
    if (!a->have_forward) return pll_set_error(PLL_ESTATE, "pll_adjoint_forward not run");
    if (!gu || !gv || !gw) return pll_set_error(PLL_EINVAL, "NULL gradient field");
    hipStream_t s = (hipStream_t)stream;
    const pll_grid_dev *g = pll_channel_grid(a->ch);
    double *const Gr[3] = {gu, gv, gw};
    double *L[3] = {fld(a, a->lam, 0), fld(a, a->lam, 1), fld(a, a->lam, 2)};
    int rc, forced[3], fmask = 0;
    if ((rc = pll_channel_forcing(a->ch, forced, NULL))) return rc;
    for (int d = 0; d < 3; d++) fmask |= forced[d] ? 1 << d : 0;
    for (int d = 0; d < 3; d++)
        if ((rc = hipchk(hipMemsetAsync(Gr[d], 0, a->fbytes, s), "clear"))) return rc;
    if ((rc = hipchk(hipMemsetAsync(a->lam, 0, 3 * a->fbytes, s), "clear")) ||
        (rc = hipchk(hipMemsetAsync(a->lam1, 0, 3 * a->fbytes, s), "clear")))
        return rc;
    /* state after the last step: J's reading of it, forcing transposed */
    double cb, ct;
    seed(a, &cb, &ct);
    if ((rc = launch(pll_launch_wall_seed(g, L[0], cb, ct, s), "wall seed")) ||
        (rc = pll_channel_force_vel_adj(a->ch, L[0], L[1], L[2], s)))
        return rc;
    for (int m = a->nck - 1; m >= 0; m--) {
        const int n0 = m * a->every;
        const int n1 = n0 + a->every < a->nsteps ? n0 + a->every : a->nsteps;
        /* the segment's states after its checkpoint, unless seg holds them
         * (the last segment's after a forward, the first one's after a
         * backward) */
        if (a->held != m) {
            a->held = -1;
            for (int n = n0; n < n1 - 1; n++)
                if ((rc = step_fwd(a, n, s))) return rc;
            a->held = m;
        }
        for (int n = n1 - 1; n >= n0; n--)
            if ((rc = step_adj(a, state(a, n), Gr,
                               n == a->nsteps - 1 ? 0 : fmask, n == 0, s)))
                return rc;
    }
    return PLL_OK;
}
