/*
 * tp_bs.hip -- adaptive Bulirsch-Stoer tracking on gfx950.
 *
 * Algorithm: the reference's StepperBS (src/unused/StepperBS.c:103-435, NR3
 * ch. 17 without dense output), with per-particle controller state and the
 * relativistic ODE in (x, u).  The CPU oracle (tpref_bs_track) runs the same
 * operations as plain nested loops; this file reorganises them for a GPU:
 *
 *  - Every loop iteration of the kernel performs exactly one right-hand-side
 *    evaluation on every active lane.  A lane's position inside a BS step
 *    (which extrapolation row k, which midpoint substep, whether the next
 *    evaluation is the derivative at an accepted point) is a small state
 *    machine, so lanes at different rows and orders still evaluate the field
 *    together and the expensive field sum (1000 cosines for the multi-mode
 *    field) never diverges across a wavefront; the mode sum runs on the
 *    matrix cores over the active lanes' points only (modes_wave64).  Only
 *    the tableau and controller bookkeeping between evaluations is divergent;
 *    its parts are run once an iteration for all lanes that need them.
 *  - The kernel is persistent: a fixed number of waves per compute unit pull
 *    particles from a global work queue.  Lanes whose particle reached its
 *    end time are refilled together: one atomic per wavefront hands out as
 *    many particle indices as there are idle lanes.
 *  - The counter reset and the kernel are captured once into a hipGraph and
 *    replayed (the reset is a small kernel, not a memset node).
 *  - Launch shape (lanes per block, waves per CU) comes from an autotuner
 *    that times short runs of the same kernel and caches its choice.
 *
 * The controller's pow() is tp_pow (shared with the oracle), so step-size
 * decisions and therefore trajectories are bitwise those of the oracle.
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "tp_ctx.h"

#define BS_N 6
#define BS_STEPFAC1 0.65
#define BS_STEPFAC2 0.94
#define BS_STEPFAC3 0.02
#define BS_STEPFAC4 4.0
#define BS_KFAC1 0.8
#define BS_KFAC2 0.9

enum { PH_INIT = 0, PH_MID = 1, PH_ACCEPT = 2, PH_DROW = 3, PH_PREP = 4, PH_OUT = 5 };

/* What a lane does at the end of an iteration.  The parts of a step that
 * several phases lead to are run once there, for all lanes that came to them
 * (bs_tail), instead of in a copy per phase: one copy of the code, lanes from
 * different phases in it together, and half the registers. */
enum { NX_NONE = 0, NX_ACCEPT = 1, NX_START = 2, NX_ATTEMPT = 3, NX_SEQ = 4, NX_FAIL = 5,
       NX_DONE = 6 };

/* Dense form: a lane whose step was accepted waits (PH_PREP, evaluating no
 * point, like an idle lane) until BS_PREP lanes of its wavefront wait, or a
 * quarter of those that take particles where that is fewer, or no other lane is
 * busy, and then their interpolants are formed together, a lane per component
 * (bs_prepare_dense): the wavefront waits for the rows in memory and the chain
 * of divisions once for all of them.  Each step's arithmetic is the same
 * whichever others it shares the batch with. */
enum { Q_HEAD = 0, Q_ACC = 1, Q_REJ = 2, Q_RHS = 3, Q_FAIL = 4, Q_N = 8 };

struct BsConsts {
    int kmax, ktarg0;
    int cost[10];
    double coeff[10][10];
    double errfac[19];
    double facmin[10];           /* STEPFAC3^(1 / (2k + 1)) */
};

/* largest kmax */
#define BS_KMAX 8
/* dense output: per lane, in HBM, rows of the six components: ysave (9
 * rows), fsave (162: every substep derivative of sequences 0..8, sequence k
 * from row 2 k^2 on) and the interpolation coefficients (23); row r of lane g at
 * ds[(r * nl + g) * 6] */
#define DS_YSAVE 0
#define DS_FSAVE 9
#define DS_DENS (DS_FSAVE + 162)
#define DS_ROWS (DS_DENS + 2 * 9 + 5)

struct BsArgs {
    FieldDev f;
    BsConsts c;
    int n, cap;
    int lanes;                   /* lanes of a wavefront that take particles */
    int lds_quads;               /* mode groups copied to LDS (0: none) */
    double qm, rtol, atol, t_end, t_end_gyro, b_ref, h0;
    double *x, *y, *z, *ux, *uy, *uz, *t;
    int *nsteps, *flag;
    unsigned long long *ctr;
    /* the dense form with the fixed-step loop's diagnostics */
    double *ds;                  /* dense-output scratch, DS_ROWS x 6 per lane */
    long nl;                     /* lanes of the launch that take particles */
    double dt;                   /* output grid: times t0 + j dt */
    int estep, ei, di, nd, nframes, nbins, nt_out, bc, fix_stale;
    double lo[3], hi[3], logemin, logde;
    double *xs, *ys, *zs;        /* periodic shifts */
    const double *x0, *y0, *z0, *ux0, *uy0, *uz0, *g0, *mu0, *th0;
    double *st;                  /* 5 stale D terms per particle (SoA) */
    unsigned *espect, *espect_esc;
    double *dbuf;                /* D terms [row][8][n] */
    int *outhist;                /* particles counted out from row r, [nd] */
    /* trajectory diagnostics (traj != null): the particle at the output
     * steps j = k traj_nout into traj[traj_accum[i-1] + traj_pts[i]++]
     * while that slot is the particle's; qm from stage[i] */
    tp_particle *traj;
    const int *traj_accum;
    int *traj_pts;
    int traj_nout;
    const tp_particle *stage;
};

/* StepperBase (src/unused/StepperBS.c:103-149): the step-size sequence
 * (dense output: 4k+2, else 2(k+1); bs_nseq in the kernels), costs, k_targ
 * from rtol, the extrapolation coefficients and the dense interpolation error
 * factors */
static void bs_consts(int kmax, double rtol, int dense, BsConsts *c)
{
    memset(c, 0, sizeof(*c));
    c->kmax = kmax;
    int nseq[BS_KMAX + 1];
    for (int i = 0; i <= kmax; i++) nseq[i] = dense ? 4 * i + 2 : 2 * (i + 1);
    c->cost[0] = nseq[0] + 1;
    for (int k = 0; k < kmax; k++) c->cost[k + 1] = c->cost[k] + nseq[k + 1];
    double logfact = -log10(rtol > 1.0e-12 ? rtol : 1.0e-12) * 0.6 + 0.5;
    int kt = (int)logfact;
    if (kt > kmax - 1) kt = kmax - 1;
    if (kt < 1) kt = 1;
    c->ktarg0 = kt;
    for (int k = 0; k <= kmax; k++)
        for (int l = 0; l < k; l++) {
            double ratio = (double)nseq[k] / nseq[l];
            c->coeff[k][l] = 1.0 / (ratio * ratio - 1.0);
        }
    for (int i = 0; i < 2 * (kmax + 1) + 1; i++) {
        int ip5 = i + 5;
        c->errfac[i] = 1.0 / (ip5 * ip5);
        double e = 0.5 * sqrt(((double)(i + 1)) / ip5);
        for (int j = 0; j <= i; j++) c->errfac[i] *= e / (j + 1);
    }
    for (int k = 0; k <= kmax; k++) c->facmin[k] = tp_pow(BS_STEPFAC3, 1.0 / (2 * k + 1));
}

/* the right-hand side from the field e at the point y */
__device__ __forceinline__ void bs_deriv(const Emf &e, double qm, const double *y, double *dy)
{
    double g = sqrt(1.0 + y[3] * y[3] + y[4] * y[4] + y[5] * y[5]);
    double ig = 1.0 / g;
    double vx = y[3] * ig, vy = y[4] * ig, vz = y[5] * ig;
    dy[0] = vx;
    dy[1] = vy;
    dy[2] = vz;
    dy[3] = qm * (e.ex + (vy * e.bz - vz * e.by));
    dy[4] = qm * (e.ey + (vz * e.bx - vx * e.bz));
    dy[5] = qm * (e.ez + (vx * e.by - vy * e.bx));
}

/* per-lane state of one particle's integration */
struct BsLane {
    long pi;                    /* particle, -1 idle, -2 retired */
    int phase, k, nn, nstep, ktarg, attempts, acc, rej;
    int first, last, reject, prev_reject;
    double t, tend, h, hnew, hnext, hsub, xe;
    /* yv: the last accepted state, which is also the start of the step being
     * attempted (the reference's ysav) */
    double yv[BS_N], ycur[BS_N], dydx[BS_N], ym[BS_N], yn[BS_N];
    int rhs;
    /* dense form: next fsave row, the polynomial's step (start, size), the
     * step-size cap of the interpolation error, the output-time grid (t0,
     * next frame, next D row), periodic shifts, the escape and end flags */
    int ipt, nf, nr, esc, ending;
    int jt;                     /* next trajectory output step */
    double told, hd, hopt_int, t0;
    double xs[3];
};

/* The extrapolation tableau of a lane, at constant indices only (bs_end_seq),
 * and its rows' step sizes and costs, which are indexed by the lane's own row
 * numbers.  Each is a variable of its own beside BsLane: the compiler keeps a
 * variable with one such access in private memory as a whole. */
struct BsTab {
    double t[BS_KMAX][BS_N];
};

struct BsCost {
    double hopt[BS_KMAX + 1], work[BS_KMAX + 1];
};

/* component i of row r of this lane's dense-output scratch */
#define DSR(a, r, i) ((a).ds[((size_t)(r) * (a).nl + gl) * BS_N + (i)])

__device__ __forceinline__ double bs_time(const BsArgs &a, const BsLane &L, long j)
{
    return L.t0 + (double)j * a.dt;
}

/* particle_bc, src/tracking.c:1172-1221, on the lane's state */
__device__ __forceinline__ void bs_particle_bc(const BsArgs &a, BsLane &L)
{
    if (a.bc == 0) {
        double d0 = a.hi[0] - a.lo[0], d1 = a.hi[1] - a.lo[1], d2 = a.hi[2] - a.lo[2];
        if (L.yv[0] > a.hi[0]) { L.yv[0] -= d0; L.xs[0] += d0; }
        if (L.yv[1] > a.hi[1]) { L.yv[1] -= d1; L.xs[1] += d1; }
        if (L.yv[2] > a.hi[2]) { L.yv[2] -= d2; L.xs[2] += d2; }
        if (L.yv[0] < a.lo[0]) { L.yv[0] += d0; L.xs[0] -= d0; }
        if (L.yv[1] < a.lo[1]) { L.yv[1] += d1; L.xs[1] -= d1; }
        if (L.yv[2] < a.lo[2]) { L.yv[2] += d2; L.xs[2] -= d2; }
    } else if (a.bc == 1) {
        if (L.yv[0] > a.hi[0] || L.yv[1] > a.hi[1] || L.yv[2] > a.hi[2] || L.yv[0] < a.lo[0] ||
            L.yv[1] < a.lo[1] || L.yv[2] < a.lo[2])
            L.esc = 1;
    }
}

/* ptl_energy_fixed's bin, src/diagnostics.c:187-205 */
__device__ __forceinline__ int bs_energy_bin(const BsArgs &a, double ux, double uy, double uz)
{
    double gama = sqrt(1.0 + ux * ux + uy * uy + uz * uz);
    double v = floor((log10(gama - 1.0) - a.logemin) / a.logde);
    if (!(v > -2147483649.0 && v < 2147483648.0)) return 0;
    int ib = (int)v;
    if (ib < 0) ib = 0;
    else if (ib > a.nbins - 1) ib = a.nbins - 1;
    return ib;
}

/* calc_diff_coeff's eight terms (src/diagnostics.c:659-705) of state y at
 * time tt with shifts xs and field e into row r, or, escaped, the stale
 * terms (src/tracking.c:334-336) */
__device__ __forceinline__ void bs_dterms(const BsArgs &a, long i, int r, int escaped,
                                          const double *y, double tt, const double *xs,
                                          const Emf &e)
{
    const long n = a.n;
    double *st = a.st;
    double dxx = st[i], dyy = st[n + i], dzz = st[2 * n + i];
    double daa = st[3 * n + i], dee = st[4 * n + i];
    double drr = 0.0, dpp = 0.0, duu = 0.0;
    if (escaped) {
        if (a.fix_stale) dxx = dyy = dzz = daa = dee = 0.0;
    } else {
        double t = tt * 2 + a.dt;
        double q;
        q = a.x0[i] - (y[0] + xs[0]); dxx = q * q / t;
        q = a.y0[i] - (y[1] + xs[1]); dyy = q * q / t;
        q = a.z0[i] - (y[2] + xs[2]); dzz = q * q / t;
        drr = dxx + dyy + dzz;
        double ax = a.ux0[i] - y[3], ay = a.uy0[i] - y[4], az = a.uz0[i] - y[5];
        dpp = (ax * ax + ay * ay + az * az) / t;
        double g = sqrt(1.0 + y[3] * y[3] + y[4] * y[4] + y[5] * y[5]);
        q = g - a.g0[i]; dee = q * q / t;
        double ab = sqrt(e.bx * e.bx + e.by * e.by + e.bz * e.bz);
        double au = sqrt(y[3] * y[3] + y[4] * y[4] + y[5] * y[5]);
        double mu = (e.bx * y[3] + e.by * y[4] + e.bz * y[5]) / (ab * au);
        q = mu - a.mu0[i]; duu = q * q / t;
        double th = acos(mu) * 180 / TP_PI;
        q = th - a.th0[i]; daa = q * q / t;
    }
    st[i] = dxx; st[n + i] = dyy; st[2 * n + i] = dzz;
    st[3 * n + i] = daa; st[4 * n + i] = dee;
    double *o = a.dbuf + (size_t)r * 8 * n + i;
    o[0] = drr; o[n] = dxx; o[2 * n] = dyy; o[3 * n] = dzz;
    o[4 * n] = dpp; o[5 * n] = duu; o[6 * n] = daa; o[7 * n] = dee;
}

template <bool DENSE>
__device__ __forceinline__ void bs_finish(const BsArgs &a, BsLane &L, int failed, long gl)
{
    const long i = L.pi;
    a.x[i] = L.yv[0]; a.y[i] = L.yv[1]; a.z[i] = L.yv[2];
    a.ux[i] = L.yv[3]; a.uy[i] = L.yv[4]; a.uz[i] = L.yv[5];
    a.t[i] = L.t;
    a.nsteps[i] = L.acc;
    if (DENSE) {
        /* rows from nr on: the particle has left (or failed); it is counted
         * out from row 1 if it started outside, else from the row after its
         * first stale row (the fixed-step loop's count, src/tracking.c:366-369) */
        const Emf e = {};
        for (int r = L.nr; r < a.nd; r++) bs_dterms(a, i, r, 1, L.yv, 0.0, L.xs, e);
        if (L.esc) {
            const int from = L.ending < 0 ? 1 : L.nr + 1;
            if (from < a.nd) atomicAdd(&a.outhist[from], 1);
        }
        a.xs[i] = L.xs[0]; a.ys[i] = L.xs[1]; a.zs[i] = L.xs[2];
        a.flag[i] = L.esc ? 2 : failed;
    } else {
        a.flag[i] = failed;
    }
    atomicAdd(&a.ctr[Q_ACC], (unsigned long long)L.acc);
    atomicAdd(&a.ctr[Q_REJ], (unsigned long long)L.rej);
    atomicAdd(&a.ctr[Q_RHS], (unsigned long long)L.rhs);
    if (failed) atomicAdd(&a.ctr[Q_FAIL], 1ull);
    L.pi = -1;
}

/* step number of row k */
template <bool DENSE>
__device__ __forceinline__ int bs_nseq(int k)
{
    return DENSE ? 4 * k + 2 : 2 * (k + 1);
}

template <bool DENSE>
__device__ __forceinline__ void bs_begin_seq(BsLane &L)
{
    L.nstep = bs_nseq<DENSE>(L.k);
    L.hsub = L.h / L.nstep;
    for (int i = 0; i < BS_N; i++) {
        L.ym[i] = L.yv[i];
        L.yn[i] = L.yv[i] + L.hsub * L.dydx[i];
    }
    L.xe = L.t + L.hsub;
    L.nn = 1;
    L.phase = PH_MID;
}

/* one trajectory point of the lane's particle: state y at time t with the
 * lane's shifts, folded into the box for periodic boundaries as particle_bc
 * folds the fixed-step loop's records (src/tracking.c:440-447, 1172-1221) */
__device__ __forceinline__ void bs_traj_record(const BsArgs &a, const BsLane &L, const double *y,
                                               double t)
{
    const long i = L.pi;
    const int toff = i > 0 ? a.traj_accum[i - 1] : 0;
    const int k = a.traj_pts[i];
    if (k < a.traj_accum[i] - toff) {
        tp_particle r;
        r.x = y[0]; r.y = y[1]; r.z = y[2]; r.qm = a.stage[i].qm;
        r.ux = y[3]; r.uy = y[4]; r.uz = y[5]; r.t = t;
        r.xshift = L.xs[0]; r.yshift = L.xs[1]; r.zshift = L.xs[2];
        if (a.bc == 0) {
            const double d0 = a.hi[0] - a.lo[0], d1 = a.hi[1] - a.lo[1], d2 = a.hi[2] - a.lo[2];
            if (r.x > a.hi[0]) { r.x -= d0; r.xshift += d0; }
            if (r.y > a.hi[1]) { r.y -= d1; r.yshift += d1; }
            if (r.z > a.hi[2]) { r.z -= d2; r.zshift += d2; }
            if (r.x < a.lo[0]) { r.x += d0; r.xshift -= d0; }
            if (r.y < a.lo[1]) { r.y += d1; r.yshift -= d1; }
            if (r.z < a.lo[2]) { r.z += d2; r.zshift -= d2; }
        }
        a.traj[toff + k] = r;
    }
    a.traj_pts[i] = k + 1;
}

/* the output times at the end time: the remaining frames from the final
 * state; the remaining D rows each need the field there (PH_DROW) */
template <bool DENSE>
__device__ __forceinline__ int bs_begin_end_outputs(const BsArgs &a, BsLane &L, long gl)
{
    for (; L.nf < a.nframes; L.nf++)
        atomicAdd(&a.espect[L.nf * a.nbins + bs_energy_bin(a, L.yv[3], L.yv[4], L.yv[5])], 1u);
    if (a.traj)
        for (; L.jt <= a.estep; L.jt += a.traj_nout) bs_traj_record(a, L, L.yv, bs_time(a, L, L.jt));
    if (L.nr < a.nd) {
        L.ending = 1;
        for (int i = 0; i < BS_N; i++) L.yn[i] = L.yv[i];
        L.xe = bs_time(a, L, (long)L.nr * a.di);
        L.phase = PH_DROW;
        return NX_NONE;
    }
    return NX_DONE;
}

/* top of step(): src/unused/StepperBS.c:173-191 */
template <bool DENSE>
__device__ __forceinline__ int bs_start_step(const BsArgs &a, BsLane &L, BsCost &W, long gl)
{
    if (!(L.t < L.tend - 1e-13 * fabs(L.tend)))
        return DENSE ? bs_begin_end_outputs<DENSE>(a, L, gl) : NX_DONE;
    double h = L.hnext;
    if (L.t + h > L.tend) h = L.tend - L.t;
    W.work[0] = 0.0;
    if (h != L.hnext && !L.first) L.last = 1;
    if (L.reject) {
        L.prev_reject = 1;
        L.last = 0;
    }
    L.reject = 0;
    L.hnew = fabs(h);
    return NX_ATTEMPT;
}

/* after row k's midpoint sequence: extrapolation, error and the
 * convergence/rejection tests of src/unused/StepperBS.c:206-272.  The
 * tableau is read at once, updated at constant indices (rows a lane does not
 * have keep their values) and written back: one wait for private memory
 * instead of one per element.  C: the constants in LDS, indexed by the
 * lane's own k. */
template <bool DENSE>
__device__ __forceinline__ int bs_end_seq(const BsArgs &a, const BsConsts &C, BsLane &L,
                                          BsTab &T, BsCost &W, const double *yseq)
{
    const int k = L.k;
    if (k == 0) {
#pragma unroll
        for (int i = 0; i < BS_N; i++) L.ycur[i] = yseq[i];
        L.k = 1;
        return NX_SEQ;
    }
    /* the lane's coefficients; rows from k - 1 on take no part */
    double cf[BS_KMAX], d[BS_N];
#pragma unroll
    for (int j = 0; j < BS_KMAX; j++) cf[j] = C.coeff[k][j];
#pragma unroll
    for (int i = 0; i < BS_N; i++) {
        double t[BS_KMAX];
#pragma unroll
        for (int r = 0; r < BS_KMAX; r++) t[r] = r == k - 1 ? yseq[i] : T.t[r][i];
#pragma unroll
        for (int j = BS_KMAX - 1; j > 0; j--) {
            const double v = t[j] + cf[j] * (t[j] - t[j - 1]);
            t[j - 1] = j <= k - 1 ? v : t[j - 1];
        }
#pragma unroll
        for (int r = 0; r < BS_KMAX; r++) T.t[r][i] = t[r];
        L.ycur[i] = t[0] + cf[0] * (t[0] - L.ycur[i]);
        d[i] = L.ycur[i] - t[0];
        if (i % 2) __builtin_amdgcn_sched_barrier(0);
    }
    double err = 0.0;
#pragma unroll
    for (int i = 0; i < BS_N; i++) {
        double p = fabs(L.yv[i]), q = fabs(L.ycur[i]);
        double scale = a.atol + a.rtol * (p > q ? p : q);
        double r = d[i] / scale;
        err += r * r;
    }
    err = sqrt(err / BS_N);
    double expo = 1.0 / (2 * k + 1);
    double facmin = C.facmin[k];
    double fac;
    if (err == 0.0) {
        fac = 1.0 / facmin;
    } else {
        fac = BS_STEPFAC2 / tp_pow(err / BS_STEPFAC1, expo);
        double lo = facmin / BS_STEPFAC4, hi = 1.0 / facmin;
        fac = fac < hi ? fac : hi;
        fac = lo > fac ? lo : fac;
    }
    const double hk = fabs(L.h * fac), wk = C.cost[k] / hk;
    W.hopt[k] = hk;
    W.work[k] = wk;
    bool brk = false;
    /* every rejection below lowers ktarg (to k, or to itself) by one more
     * when the row before cost less, and takes that row's step size */
    bool rej = false;
    int kt = L.ktarg;
    if ((L.first || L.last) && err <= 1.0) brk = true;
    if (!brk && k == L.ktarg - 1 && !L.prev_reject && !L.first && !L.last) {
        if (err <= 1.0) {
            brk = true;
        } else {
            double r = (double)(bs_nseq<DENSE>(L.ktarg) * bs_nseq<DENSE>(L.ktarg + 1) /
                                (bs_nseq<DENSE>(0) * bs_nseq<DENSE>(0)));
            if (err > r * r) {
                rej = true;
                kt = k;
                brk = true;
            }
        }
    }
    if (!brk && k == L.ktarg) {
        if (err <= 1.0) {
            brk = true;
        } else {
            double r = (double)bs_nseq<DENSE>(k + 1) / bs_nseq<DENSE>(0);
            if (err > r * r) {
                rej = true;
                brk = true;
            }
        }
    }
    if (!brk && k == L.ktarg + 1) {
        if (err > 1.0) rej = true;
        brk = true;
    }
    if (!brk) {
        L.k = k + 1;
        return NX_SEQ;
    }
    if (rej) {
        /* kt is k or ktarg: at k = ktarg + 1 the rows compared are ktarg - 1
         * and ktarg, otherwise k - 1 and k */
        if (kt > 1 && W.work[kt - 1] < BS_KFAC1 * W.work[kt]) kt--;
        L.ktarg = kt;
        L.hnew = W.hopt[kt];
        L.reject = 1;
        L.prev_reject = 1;
        L.rej++;
        return NX_ATTEMPT;
    }
    /* accepted: the derivative at the new point comes next */
    L.xe = L.t + L.h;
    L.phase = PH_ACCEPT;
    return NX_NONE;
}

/* ------------------------------------------------------------------ */
/* dense output: a lane per component                                   */
/* ------------------------------------------------------------------ */
/* prepare_dense (src/unused/StepperBS.c:526-615) treats the six components
 * of a step separately, so a wavefront forms the interpolants of up to
 * BS_PREP steps at once with lane 6 p + i on component i of the p-th.  The
 * reference updates its ysave and fsave arrays in place, order by order; here
 * a component goes through the same operations in registers, a sequence KK at
 * a time: its rows are read together, their differences formed order by
 * order, and each order's value (times (n_KK / 2)^(order - 1)) enters that
 * order's extrapolation as soon as it is known:
 *   y[l-1] = y[l] + (y[l] - y[l-1]) / ((n_KK / n_{l-1})^2 - 1), l = KK..KB+1,
 * KB = (order - 1) / 2 (src/unused/StepperBS.c:545-553, 564-572).  Same
 * operations on the same operands: the oracle's bits.
 * Bound: k + 2 waits for the scratch rows (from HBM) and the chain of
 * divisions.  A lane per step, with the values of an order passing through
 * scratch, took 367,000 cycles for the 8 steps of a batch (30,000 particles,
 * 200 modes, one wavefront per SIMD); a lane per component takes 48,000. */
#define BS_PREP 10
#define BS_PREP_IN (4 * BS_N + 1)    /* doubles a lane hands over: y, y', ends, h */

/* n / d - n and d the sequences' step numbers, known at compile time */
template <int J, int L1>
struct BsFactor {
    static __device__ __forceinline__ double get()
    {
        const double r = (double)(4 * J + 2) / (double)(4 * L1 + 2);
        return r * r - 1.0;
    }
};

/* y[KB .. J-1] extrapolated with sequence J's value v */
template <int KB, int J, int LL>
__device__ __forceinline__ void bs_extrap_step(double (&y)[BS_KMAX + 1])
{
    if constexpr (LL >= KB + 1) {
        y[LL - 1] = y[LL] + (y[LL] - y[LL - 1]) / BsFactor<J, LL - 1>::get();
        bs_extrap_step<KB, J, LL - 1>(y);
    }
}

template <int KB, int J>
__device__ __forceinline__ void bs_extrap(double (&y)[BS_KMAX + 1], double v)
{
    y[J] = v;
    bs_extrap_step<KB, J, J>(y);
}

constexpr double bs_const_pow(double x, int e)
{
    double r = 1.0;
    for (int i = 0; i < e; i++) r = r * x;
    return r;
}

/* sequence KK's derivative rows (offsets o in the sequence; row 0 of the
 * sequence is row 2 KK^2 of fsave), from order KMI
 * on: the value order KMI takes, then the differences between orders
 * (src/unused/StepperBS.c:558-601) */
template <int KK, int KMI>
__device__ __forceinline__ void bs_dense_orders(int mu, double dydx_i, double (&row)[4 * KK + 2],
                                                double (&Y)[2 * BS_KMAX][BS_KMAX + 1])
{
    constexpr int R = 4 * KK + 2, KB = (KMI - 1) / 2;
    if constexpr (KMI <= 2 * BS_KMAX - 1 && KK >= KB) {
        if (KMI > mu) return;
        constexpr double scale = bs_const_pow((4 * KK + 2) / 2.0, KMI - 1);
        bs_extrap<KB, KK>(Y[KMI], row[2 * KK + KMI - 1] * scale);
        if (KMI == mu) return;
        if constexpr (KK >= KMI / 2) {
#pragma unroll
            for (int o = R - 1; o >= (KMI == 1 ? 2 : KMI); o--) row[o] = row[o] - row[o - 2];
            if constexpr (KMI == 1) row[1] = row[1] - dydx_i;
        }
        bs_dense_orders<KK, KMI + 1>(mu, dydx_i, row, Y);
    }
}

template <int KK>
__device__ __forceinline__ void bs_dense_seqs(const BsArgs &a, long gl, int i, int k, int mu,
                                              double dydx_i,
                                              double (&Y)[2 * BS_KMAX][BS_KMAX + 1])
{
    if constexpr (KK <= BS_KMAX) {
        if (KK <= k) {
            double row[4 * KK + 2];
            const double ys = DSR(a, DS_YSAVE + KK, i);
#pragma unroll
            for (int o = 0; o < 4 * KK + 2; o++) row[o] = DSR(a, DS_FSAVE + 2 * KK * KK + o, i);
            bs_extrap<0, KK>(Y[0], ys);
            bs_dense_orders<KK, 1>(mu, dydx_i, row, Y);
            bs_dense_seqs<KK + 1>(a, gl, i, k, mu, dydx_i, Y);
        }
    }
}

/* component i of a step of size h with ends y0, y1 and derivatives yp0, yp1
 * there (times h): prepare_dense and dense_interp (src/unused/StepperBS.c:
 * 478-524) into the lane's dens rows; returns the last coefficient, which
 * estimates the interpolation error */
__device__ __forceinline__ double bs_dense_component(const BsArgs &a, long gl, int i, int k,
                                                     double h, double y0, double y1, double f0,
                                                     double f1)
{
    const int mu = 2 * k - 1;
    double Y[2 * BS_KMAX][BS_KMAX + 1];
    bs_dense_seqs<0>(a, gl, i, k, mu, f0, Y);
    const double yp0 = h * f0, yp1 = f1 * h;
    const double ydiff = y1 - y0;
    const double aspl = -yp1 + ydiff;
    const double bspl = yp0 - ydiff;
    DSR(a, DS_DENS + 0, i) = y0;
    DSR(a, DS_DENS + 1, i) = ydiff;
    DSR(a, DS_DENS + 2, i) = aspl;
    DSR(a, DS_DENS + 3, i) = bspl;
    const double ph0 = (y0 + y1) * 0.5 + 0.125 * (aspl + bspl);
    const double ph1 = ydiff + (aspl - bspl) * 0.25;
    const double ph2 = -(yp0 - yp1);
    const double ph3 = 6.0 * (bspl - aspl);
    /* order m's coefficient before dense_interp: Y[m][KB] h */
    double av[2 * BS_KMAX];
    av[0] = (Y[0][0] - ph0) * 16.0;
    double last = av[0];
    DSR(a, DS_DENS + 4, i) = av[0];
#pragma unroll
    for (int im = 1; im <= 2 * BS_KMAX - 1; im++) {
        if (im <= mu) {
            const double d = Y[im][(im - 1) / 2] * h;
            if (im == 1) {
                av[1] = 16.0 * (d - ph1);
            } else if (im == 2) {
                av[2] = (d - ph2 + av[0]) * 16.0;
            } else if (im == 3) {
                av[3] = 16.0 * (d - ph3 + 3 * av[1]);
            } else {
                const double fac1 = im * (im - 1) / 2.0;
                const double fac2 = im % 2 ? fac1 * (im - 2) * (im - 3) * 2.0
                                           : (double)(im * (im - 1) * (im - 2) * (im - 3));
                av[im] = 16.0 * (d + fac1 * av[im - 2] - fac2 * av[im - 4]);
            }
            DSR(a, DS_DENS + im + 4, i) = av[im];
            last = av[im];
        }
    }
    return last;
}

/* The interpolants of the lanes with `pend`, whose steps were accepted with
 * the derivatives dydxnew in ym; every lane of the wavefront calls it.  Returns
 * the interpolation error estimate of the lane's own step.  xp: the
 * wavefront's MODES_WAVE_LDS doubles of LDS. */
__device__ __forceinline__ double bs_prepare_dense(const BsArgs &a, const BsConsts &C,
                                                   const BsLane &L, bool pend, long gl,
                                                   double *xp)
{
    const int lane = threadIdx.x & 63;
    const unsigned long long mask = __ballot(pend);
    const int total = __popcll(mask);
    const int rank = __popcll(mask & ((1ull << lane) - 1ull));
    double error = 0.0;
    for (int base = 0; base < total; base += BS_PREP) {
        const int cnt = total - base < BS_PREP ? total - base : BS_PREP;
        const bool mine = pend && rank >= base && rank < base + BS_PREP;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (mine) {
            double *o = xp + BS_PREP_IN * (rank - base);
#pragma unroll
            for (int i = 0; i < BS_N; i++) {
                o[i] = L.yv[i];
                o[BS_N + i] = L.ycur[i];
                o[2 * BS_N + i] = L.dydx[i];
                o[3 * BS_N + i] = L.ym[i];
            }
            o[4 * BS_N] = L.h;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        /* the lane of the p-th step of this batch */
        const int p = lane / BS_N, i = lane - BS_N * p;
        int src = 0;
        {
            unsigned long long m = mask;
            for (int q = 0; q < base; q++) m &= m - 1;
            for (int q = 0; q < BS_PREP; q++) {
                if (q == p) src = __ffsll((long long)m) - 1;
                m &= m - 1;
            }
        }
        const bool work = p < cnt;
        src = work ? src : 0;
        const int k = __shfl(L.k, src, 64);
        double v2 = 0.0;
        if (work) {
            const double *o = xp + BS_PREP_IN * p;
            const double y0 = o[i], y1 = o[BS_N + i];
            const double v = bs_dense_component(a, gl - lane + src, i, k, o[4 * BS_N], y0, y1,
                                                o[2 * BS_N + i], o[3 * BS_N + i]);
            const double q0 = fabs(y0), q1 = fabs(y1);
            const double scale = a.atol + a.rtol * (q0 > q1 ? q0 : q1);
            const double r = v / scale;
            v2 = r * r;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (work) xp[lane] = v2;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        if (mine) {
            double e = 0.0;
#pragma unroll
            for (int q = 0; q < BS_N; q++) e += xp[BS_N * (rank - base) + q];
            const int mu = 2 * L.k - 1;
            error = mu >= 1 ? sqrt(e / BS_N) * C.errfac[mu - 1] : 0.0;
        }
    }
    return error;
}

/* dense_out, src/unused/StepperBS.c:617-644: component i at time x of the
 * lane's last accepted step (its rows read together) */
__device__ __forceinline__ double bs_dense_out(const BsArgs &a, const BsLane &L, long gl, int i,
                                               double x)
{
    const int mu = 2 * L.k - 1;
    double d[2 * BS_KMAX + 4];
#pragma unroll
    for (int r = 0; r < 2 * BS_KMAX + 4; r++) d[r] = DSR(a, DS_DENS + r, i);
    double theta = (x - L.told) / L.hd;
    double theta1 = 1.0 - theta;
    double yinterp = d[0] + theta * (d[1] + theta1 * (d[2] * theta + d[3] * theta1));
    if (mu < 0) return yinterp;
    double theta05 = theta - 0.5;
    double tt = theta * theta1;
    double t4 = tt * tt;
    double cc = 0.0;
#pragma unroll
    for (int j = 2 * BS_KMAX - 1; j >= 0; j--) {
        if (j == mu) cc = d[j + 4];
        if (j < mu) cc = d[j + 4] + cc * theta05 / (j + 1);
    }
    return yinterp + t4 * cc;
}

/* the step's own output times (strictly before its end) next: a D row
 * needs the field at its point, evaluated in the next iteration */
__device__ __forceinline__ bool bs_next_drow(const BsArgs &a, BsLane &L, long gl)
{
    if (L.nr >= a.nd) return false;
    const double tr = bs_time(a, L, (long)L.nr * a.di);
    if (!(tr < L.told + L.hd)) return false;
#pragma unroll
    for (int i = 0; i < BS_N; i++) L.yn[i] = bs_dense_out(a, L, gl, i, tr);
    L.xe = tr;
    L.phase = PH_DROW;
    return true;
}

/* the accepted step's bookkeeping after its derivative f at the new point:
 * order and step-size choice of src/unused/StepperBS.c:296-347, then (dense
 * form) the boundary and the escape */
template <bool DENSE>
__device__ __forceinline__ int bs_accept_finish(const BsArgs &a, const BsConsts &C, BsLane &L,
                                                const BsCost &W)
{
#pragma unroll
    for (int i = 0; i < BS_N; i++) {
        L.dydx[i] = L.ym[i];
        L.yv[i] = L.ycur[i];
    }
    L.t += L.h;
    L.first = 0;
    L.acc++;
    const int k = L.k, KM1 = C.kmax - 1;
    const double wk = W.work[k], wk1 = W.work[k - 1];
    int kopt;
    if (k == 1) {
        kopt = 2;
    } else if (k <= L.ktarg) {
        kopt = k;
        if (wk1 < BS_KFAC1 * wk) kopt = k - 1;
        else if (wk < BS_KFAC2 * wk1) kopt = (k + 1 < KM1) ? k + 1 : KM1;
    } else {
        kopt = k - 1;
        if (k > 2 && W.work[k - 2] < BS_KFAC1 * wk1) kopt = k - 2;
        if (wk < BS_KFAC2 * W.work[kopt]) kopt = (k < KM1) ? k : KM1;
    }
    double hnew;
    if (L.prev_reject) {
        L.ktarg = kopt < k ? kopt : k;
        double p = fabs(L.h), q = W.hopt[L.ktarg];
        hnew = p < q ? p : q;
        L.prev_reject = 0;
    } else {
        if (kopt <= k) {
            hnew = W.hopt[kopt];
        } else {
            const int num = k < L.ktarg && wk < BS_KFAC2 * wk1 ? kopt + 1 : kopt;
            hnew = W.hopt[k] * C.cost[num] / C.cost[k];
        }
        L.ktarg = kopt;
    }
    L.hnext = hnew;
    if (DENSE) {
        double hi = fabs(L.hopt_int);
        L.hnext = hnew < hi ? hnew : hi;
        bs_particle_bc(a, L);
        if (L.esc) {
            /* escape spectrum at the frame of the next output time */
            if (L.nf < a.nt_out)
                atomicAdd(&a.espect_esc[L.nf * a.nbins +
                                        bs_energy_bin(a, L.yv[3], L.yv[4], L.yv[5])], 1u);
            return NX_DONE;
        }
    }
    return NX_START;
}

/* the dense form's part of an accepted step before its bookkeeping, with the
 * interpolation error err: above 10 the step is redone with the step size it
 * suggests; otherwise the frames and trajectory points inside the step are
 * taken from its interpolant and its D rows queued */
__device__ __forceinline__ int bs_prep(const BsArgs &a, BsLane &L, double err, long gl)
{
    const double pe = tp_pow(err, 1.0 / (2 * L.k + 3));
    L.hopt_int = L.h / (pe > 0.01 ? pe : 0.01);
    if (err > 10.0) {
        L.hnew = fabs(L.hopt_int);
        L.reject = 1;
        L.prev_reject = 1;
        L.rej++;
        return NX_ATTEMPT;
    }
    L.told = L.t;
    L.hd = L.h;
    const double tnew = L.t + L.h;
    for (; L.nf < a.nframes; L.nf++) {
        const double tf = bs_time(a, L, (long)(L.nf + 1) * a.ei);
        if (!(tf < tnew)) break;
        const double ux = bs_dense_out(a, L, gl, 3, tf);
        const double uy = bs_dense_out(a, L, gl, 4, tf);
        const double uz = bs_dense_out(a, L, gl, 5, tf);
        atomicAdd(&a.espect[L.nf * a.nbins + bs_energy_bin(a, ux, uy, uz)], 1u);
    }
    /* trajectory points strictly inside the step, from the polynomial */
    if (a.traj) {
        for (; L.jt <= a.estep; L.jt += a.traj_nout) {
            const double tj = bs_time(a, L, L.jt);
            if (!(tj < tnew)) break;
            double yj[BS_N];
#pragma unroll
            for (int m = 0; m < BS_N; m++) yj[m] = bs_dense_out(a, L, gl, m, tj);
            bs_traj_record(a, L, yj, tj);
        }
    }
    /* ym keeps dydxnew while the D rows run */
    return bs_next_drow(a, L, gl) ? NX_NONE : NX_ACCEPT;
}

/* after the field e at a D row's point: its terms, then the next row or
 * the rest of the step (or, at the end time, of the particle) */
__device__ __forceinline__ int bs_drow(const BsArgs &a, BsLane &L, const Emf &e, long gl)
{
    bs_dterms(a, L.pi, L.nr, 0, L.yn, L.xe, L.xs, e);
    L.nr++;
    if (L.ending) {
        if (L.nr < a.nd) {
            L.xe = bs_time(a, L, (long)L.nr * a.di);
            return NX_NONE;                            /* same point, next row */
        }
        return NX_DONE;
    }
    return bs_next_drow(a, L, gl) ? NX_NONE : NX_ACCEPT;
}

/* the rest of a lane's iteration, from `next` on */
template <bool DENSE>
__device__ __forceinline__ void bs_tail(const BsArgs &a, const BsConsts &C, BsLane &L, BsCost &W,
                                        int next, long gl)
{
    if (next == NX_ACCEPT) next = bs_accept_finish<DENSE>(a, C, L, W);
    if (next == NX_START) next = bs_start_step<DENSE>(a, L, W, gl);
    if (next == NX_ATTEMPT) {
        L.h = L.hnew;
        L.reject = 0;
        L.k = 0;
        L.ipt = 0;
        next = ++L.attempts > a.cap ? NX_FAIL : NX_SEQ;
    }
    if (next == NX_SEQ) bs_begin_seq<DENSE>(L);
    if (next >= NX_FAIL) bs_finish<DENSE>(a, L, next == NX_FAIL ? 1 : 0, gl);
}

template <int FK, bool DENSE>
__device__ __forceinline__ void bs_body(const BsArgs &a)
{
    extern __shared__ double modes_lds[];
    const int lane = threadIdx.x & 63;
    /* scratch index of a lane that takes particles */
    const long gl = ((long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * a.lanes + lane;
    const int batch = a.lanes >> 2 < BS_PREP ? a.lanes >> 2 : BS_PREP;
    __shared__ double points[FK == FK_MODES || DENSE ? 4 * MODES_WAVE_LDS : 1];
    double *xp = points + (FK == FK_MODES || DENSE ? (threadIdx.x >> 6) * MODES_WAVE_LDS : 0);
    __shared__ BsConsts C;
    if (FK == FK_MODES && a.lds_quads) {
        for (int q = threadIdx.x; q < 32 * a.lds_quads; q += blockDim.x)
            modes_lds[q] = a.f.modesx[q];
    }
    for (unsigned q = threadIdx.x; q < sizeof(BsConsts) / 4; q += blockDim.x)
        ((int *)&C)[q] = ((const int *)&a.c)[q];
    __syncthreads();
    BsLane L;
    BsTab T;
    BsCost W;
    L.pi = lane < a.lanes ? -1 : -2;
    while (true) {
        /* refill idle lanes: one atomic per wavefront */
        unsigned long long need = __ballot(L.pi == -1);
        if (need) {
            int leader = __ffsll((long long)need) - 1;
            unsigned cnt = (unsigned)__popcll(need);
            unsigned long long base = 0;
            if (lane == leader) base = atomicAdd(&a.ctr[Q_HEAD], (unsigned long long)cnt);
            unsigned lo = __shfl((unsigned)(base & 0xffffffffull), leader, 64);
            unsigned hi = __shfl((unsigned)(base >> 32), leader, 64);
            base = ((unsigned long long)hi << 32) | lo;
            if (L.pi == -1) {
                unsigned long long below = lane ? (need & ((1ull << lane) - 1ull)) : 0ull;
                unsigned long long idx = base + (unsigned long long)__popcll(below);
                if (idx < (unsigned long long)a.n) {
                    const long i = (long)idx;
                    L.pi = i;
                    L.yv[0] = a.x[i]; L.yv[1] = a.y[i]; L.yv[2] = a.z[i];
                    L.yv[3] = a.ux[i]; L.yv[4] = a.uy[i]; L.yv[5] = a.uz[i];
                    L.t = a.t[i];
                    double g0 = sqrt(1.0 + L.yv[3] * L.yv[3] + L.yv[4] * L.yv[4] +
                                     L.yv[5] * L.yv[5]);
                    double T = 2.0 * TP_PI * g0 / (fabs(a.qm) * a.b_ref);
                    L.tend = a.t_end_gyro > 0.0 ? L.t + a.t_end_gyro * T : a.t_end;
                    L.hnext = a.h0 > 0.0 ? a.h0 : 0.01 * T;
                    L.ktarg = C.ktarg0;
                    L.first = 1;
                    L.last = L.reject = L.prev_reject = 0;
                    L.attempts = L.acc = L.rej = 0;
                    L.rhs = 0;
                    L.xe = L.t;
                    L.phase = PH_INIT;
                    if (DENSE) {
                        L.t0 = L.t;
                        L.tend = L.t + a.estep * a.dt;
                        L.nf = 0; L.nr = 1; L.esc = 0; L.ending = 0;
                        L.jt = a.traj_nout;
                        L.xs[0] = a.xs[i]; L.xs[1] = a.ys[i]; L.xs[2] = a.zs[i];
                        /* initial wrap and escape check, src/tracking.c:314-332 */
                        bs_particle_bc(a, L);
                        if (L.esc) {
                            L.ending = -1;
                            L.phase = PH_OUT;
                        }
                    }
                } else {
                    L.pi = -2;
                }
            }
        }
        if (__ballot(L.pi >= 0) == 0ull) break;
        /* the one field evaluation of this iteration, executed by the whole
         * wavefront: the mode sum packs the points of the lanes that need
         * one; for the other fields the rest evaluate a dummy point */
        const bool act = L.pi >= 0 && !(DENSE && L.phase >= PH_PREP);
        double ze[BS_N];
        for (int i = 0; i < BS_N; i++)
            ze[i] = !act ? 0.0
                         : (L.phase == PH_INIT ? L.yv[i]
                                               : (L.phase == PH_ACCEPT ? L.ycur[i] : L.yn[i]));
        Emf e;
        if constexpr (FK == FK_MODES) {
            if (a.lds_quads)
                modes_wave64(a.f, (lds_tab)modes_lds, act, ze[0], ze[1], ze[2], xp, e);
            else
                modes_wave64(a.f, a.f.modesx, act, ze[0], ze[1], ze[2], xp, e);
            /* here, out of the sum's way: inside it, the same test made the
             * adaptive form 4 % slower by moving the loops' code */
            if (__builtin_expect(modes_far(a.f, ze[0], ze[1], ze[2]), 0))
                modes_sum_far(a.f, ze[0], ze[1], ze[2], e);
        } else
            get_emf64<FK>(a.f, ze[0], ze[1], ze[2], act ? L.xe : 0.0, e);
        int next = DENSE && L.pi >= 0 && L.phase == PH_OUT ? NX_DONE : NX_NONE;
        if (act && DENSE && L.phase == PH_DROW) {
            next = bs_drow(a, L, e, gl);
        } else if (act) {
            double f[BS_N];
            bs_deriv(e, a.qm, ze, f);
            L.rhs++;
            if (L.phase == PH_MID) {
                if (DENSE) {
                    if (L.nn == L.nstep / 2 && L.nn < L.nstep)
#pragma unroll
                        for (int i = 0; i < BS_N; i++) DSR(a, DS_YSAVE + L.k, i) = L.yn[i];
                    if (abs(L.nn - L.nstep / 2) <= 2 * L.k + 1) {
#pragma unroll
                        for (int i = 0; i < BS_N; i++) DSR(a, DS_FSAVE + L.ipt, i) = f[i];
                        L.ipt++;
                    }
                }
                if (L.nn < L.nstep) {
                    double h2 = 2.0 * L.hsub;
#pragma unroll
                    for (int i = 0; i < BS_N; i++) {
                        double swap = L.ym[i] + h2 * f[i];
                        L.ym[i] = L.yn[i];
                        L.yn[i] = swap;
                    }
                    L.xe += L.hsub;
                    L.nn++;
                } else {
                    double yseq[BS_N];
#pragma unroll
                    for (int i = 0; i < BS_N; i++)
                        yseq[i] = 0.5 * (L.ym[i] + L.yn[i] + L.hsub * f[i]);
                    next = bs_end_seq<DENSE>(a, C, L, T, W, yseq);
                }
            } else if (L.phase == PH_INIT) {
#pragma unroll
                for (int i = 0; i < BS_N; i++) L.dydx[i] = f[i];
                next = NX_START;
            } else {
                /* the derivative at the accepted point goes to ym (free after
                 * the step), where the dense form's lanes keep it until their
                 * interpolant is formed */
#pragma unroll
                for (int i = 0; i < BS_N; i++) L.ym[i] = f[i];
                if (DENSE) L.phase = PH_PREP;
                else next = NX_ACCEPT;
            }
        }
        if (DENSE) {
            const unsigned long long pend = __ballot(L.pi >= 0 && L.phase == PH_PREP);
            if (pend) {
                const unsigned long long busy = __ballot(L.pi >= 0 && L.phase < PH_PREP);
                if (__popcll(pend) >= batch || busy == 0ull) {
                    const bool mine = L.pi >= 0 && L.phase == PH_PREP;
                    const double err = bs_prepare_dense(a, C, L, mine, gl, xp);
                    if (mine) next = bs_prep(a, L, err, gl);
                }
            }
        }
        bs_tail<DENSE>(a, C, L, W, next, gl);
    }
}

template <int FK, bool DENSE>
__global__ void __launch_bounds__(256) k_bs(BsArgs a)
{
    bs_body<FK, DENSE>(a);
}

/* counter reset as a kernel (graph-safe, no memset node) */
__global__ void k_bs_reset(unsigned long long *ctr)
{
    if (threadIdx.x < Q_N) ctr[threadIdx.x] = 0ull;
}

typedef void (*bs_fn)(dim3, dim3, size_t, hipStream_t, const BsArgs &);

template <int FK, bool DENSE>
static void launch_bs(dim3 g, dim3 b, size_t sh, hipStream_t s, const BsArgs &a)
{
    hipLaunchKernelGGL((k_bs<FK, DENSE>), g, b, sh, s, a);
}

template <bool DENSE>
static bs_fn pick_bs_t(int fk)
{
    switch (fk) {
    case FK_TEST: return launch_bs<FK_TEST, DENSE>;
    case FK_ABC: return launch_bs<FK_ABC, DENSE>;
    case FK_ABCV: return launch_bs<FK_ABCV, DENSE>;
    case FK_GRID_REF: return launch_bs<FK_GRID_REF, DENSE>;
    case FK_GRID_TB: return launch_bs<FK_GRID_TB, DENSE>;
    case FK_MODES: return launch_bs<FK_MODES, DENSE>;
    case FK_WLCS: return launch_bs<FK_WLCS, DENSE>;
    case FK_MHD_REF: return launch_bs<FK_MHD_REF, DENSE>;
    case FK_GRIDD_REF: return launch_bs<FK_GRIDD_REF, DENSE>;
    }
    return nullptr;
}

static bs_fn pick_bs(int fk) { return pick_bs_t<false>(fk); }

/* D sums of the dense form: column (component q, row r) of the per-particle
 * terms summed over the particles in a fixed order (strided partial sums,
 * then an LDS tree), one block per column; row 0 stays 0 */
__global__ void __launch_bounds__(256) k_bs_dsum(const double *dbuf, long n, int nd,
                                                 double *dco)
{
    __shared__ double sh[256];
    const int q = blockIdx.x % 8, r = blockIdx.x / 8;
    const double *col = dbuf + ((size_t)r * 8 + q) * n;
    double s = 0.0;
    if (r > 0)
        for (long i = threadIdx.x; i < n; i += 256) s += col[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) dco[(size_t)q * nd + r] = sh[0];
}

/* escapes counted against each row: the particles counted out from row k
 * or before (outhist[k] counts those counted out from row k) */
__global__ void k_bs_rdec(const int *outhist, int nd, int *rdec)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int run = 0;
    for (int k = 0; k < nd; k++) {
        run += outhist[k];
        rdec[k] = run;
    }
}

__global__ void __launch_bounds__(256) k_bs_zero_u32(unsigned *p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        p[i] = 0u;
}

void tp_bs_release(tp_ctx *c)
{
    if (c->bs_graph) {
        (void)hipGraphExecDestroy(c->bs_graph);
        c->bs_graph = nullptr;
    }
    (void)hipFree(c->bs_ctr);
    c->bs_ctr = nullptr;
    c->bs_graph_key = 0;
    (void)hipFree(c->bs_ds);
    (void)hipFree(c->bs_dbuf);
    (void)hipFree(c->bs_outhist);
    c->bs_ds = c->bs_dbuf = nullptr;
    c->bs_outhist = nullptr;
    c->bs_ds_cap = c->bs_dbuf_cap = c->bs_outhist_cap = 0;
}

static unsigned long long fnv(unsigned long long h, const void *p, size_t n)
{
    const unsigned char *b = (const unsigned char *)p;
    for (size_t i = 0; i < n; i++) {
        h ^= b[i];
        h *= 1099511628211ull;
    }
    return h;
}

static int bs_check(const tp_ctx *c, const tp_bs_params *p)
{
    if (!p || !(p->rtol > 0.0) || !(p->atol >= 0.0) || p->kmax < 3 || p->kmax > 8 ||
        !(p->qm != 0.0) || p->max_attempts < 0)
        return TP_E_ARG;
    if (p->t_end_gyro > 0.0 && !(p->b_ref > 0.0)) return TP_E_ARG;
    if (p->block != 0 && p->block != 64 && p->block != 128 && p->block != 256) return TP_E_ARG;
    if (p->waves_per_cu < 0 || p->waves_per_cu > 32) return TP_E_ARG;
    if (!c->have_field) return TP_E_STATE;
    return TP_OK;
}

static void bs_fill_args(const tp_ctx *c, const tp_bs_params *p, BsArgs &a, int n, double *x,
                         double *y, double *z, double *ux, double *uy, double *uz, double *t,
                         int *nsteps, int *flag, unsigned long long *ctr, int cap, int dense = 0)
{
    memset(&a, 0, sizeof(a));
    a.f = c->f;
    bs_consts(p->kmax, p->rtol, dense, &a.c);
    a.n = n;
    a.cap = cap;
    a.lanes = 64;
    a.qm = p->qm; a.rtol = p->rtol; a.atol = p->atol;
    a.t_end = p->t_end; a.t_end_gyro = p->t_end_gyro; a.b_ref = p->b_ref; a.h0 = p->h0;
    a.x = x; a.y = y; a.z = z; a.ux = ux; a.uy = uy; a.uz = uz; a.t = t;
    a.nsteps = nsteps; a.flag = flag; a.ctr = ctr;
}

static int bs_ensure_ctr(tp_ctx *c)
{
    if (!c->bs_ctr && hipMalloc(&c->bs_ctr, sizeof(unsigned long long) * Q_N) != hipSuccess) {
        c->bs_ctr = nullptr;
        return TP_E_NOMEM;
    }
    return TP_OK;
}

/* Lanes of a wavefront that take particles.  The mode sum's cost follows a
 * wavefront's particles in steps of 16 (modes_wave64), so wavefronts take 32
 * or 16 as long as that still leaves at most one for each SIMD, which is what
 * the kernels' registers allow to run at a time: 30,000 particles, 200 modes,
 * dense form, 64 / 32 / 16 lanes: 32.0 / 23.1 / 28.8 ms of kernels (16 lanes take
 * two rounds).  The other fields cost a wavefront the same however many of its
 * lanes are in use. */
static int bs_lanes(const tp_ctx *c, int wpc, int n)
{
    if (c->f.kind != FK_MODES) return 64;
    const long waves = (long)(c->num_cu > 0 ? c->num_cu : 256) * (wpc < 4 ? wpc : 4);
    int lanes = 64;
    while (lanes > 16 && ((long)n + lanes / 2 - 1) / (lanes / 2) <= waves) lanes /= 2;
    return lanes;
}

/* What the tuner's choice depends on besides field and tolerance: how many
 * particles a wavefront takes in an ensemble of n. */
static int bs_class(const tp_ctx *c, int n) { return bs_lanes(c, 4, n); }

/* the launch shape: the caller's, else the tuner's for ensembles of this
 * class, else the default */
static void bs_shape(const tp_ctx *c, const tp_bs_params *p, int n, int *block, int *wpc)
{
    *block = c->f.kind == FK_MODES ? 256 : 64;
    *wpc = 8;
    if (c->bs_tuned[0] && c->bs_tuned[2] == bs_class(c, n)) {
        *block = c->bs_tuned[0];
        *wpc = c->bs_tuned[1];
    }
    if (p->block) *block = p->block;
    if (p->waves_per_cu) *wpc = p->waves_per_cu;
}

static dim3 bs_grid(const tp_ctx *c, int block, int wpc, int n, int lanes)
{
    int cu = c->num_cu > 0 ? c->num_cu : 256;
    long waves = (long)cu * wpc;
    long need = ((long)n + lanes - 1) / lanes;  /* no more than the particles fill */
    if (waves > need) waves = need;
    long blocks = (waves * 64 + block - 1) / block;
    if (blocks < 1) blocks = 1;
    return dim3((unsigned)blocks);
}

/* The mode table goes to LDS when the copies of the blocks that share a
 * compute unit fit: its reads then take some 100 cycles instead of those of an
 * L2 hit, which a wavefront alone on its SIMD waits for (131,072 particles, 1000
 * modes, 0.3 gyroperiods: 11 % of the kernel's time).  The kernels' registers
 * leave room for four wavefronts a compute unit, whatever is launched, and a
 * block has the constants and the points of four wavefronts beside its copy.  A
 * block's copy is at most 64 KiB (1008 modes).  Returns the launch's dynamic
 * LDS. */
static size_t bs_lds(const tp_ctx *c, int block, int wpc, BsArgs &a)
{
    a.lds_quads = 0;
    if (c->f.kind != FK_MODES) return 0;
    const int quads = c->f.nquads + MODES_PAD_QUADS;
    const size_t bytes = (size_t)32 * sizeof(double) * quads;
    const size_t per_cu = (size_t)((wpc < 4 ? wpc : 4) * 64 + block - 1) / block;
    const size_t fixed = 4 * MODES_WAVE_LDS * sizeof(double) + sizeof(BsConsts);
    if (bytes > 64 * 1024 || (bytes + fixed) * per_cu > 160 * 1024) return 0;
    a.lds_quads = quads;
    return bytes;
}

/* grow a device buffer of a context to at least `need` elements */
template <typename T>
static int bs_grow(T **buf, size_t *cap, size_t need)
{
    if (need <= *cap) return TP_OK;
    (void)hipFree(*buf);
    *buf = nullptr;
    *cap = 0;
    if (hipMalloc(buf, need * sizeof(T)) != hipSuccess) {
        *buf = nullptr;
        return TP_E_NOMEM;
    }
    *cap = need;
    return TP_OK;
}

extern "C" {

int tp_gpu_run_adaptive(tp_ctx *c, const tp_bs_params *p, tp_bs_stats *stats)
{
    if (!c) return TP_E_ARG;
    int rc = bs_check(c, p);
    if (rc) return rc;
    if (!c->s.derived && c->s.n > 0) return TP_E_STATE;
    bs_fn fn = pick_bs(c->f.kind);
    if (!fn) return TP_E_ARG;
    HIPCHK(hipSetDevice(c->device));
    if ((rc = bs_ensure_ctr(c))) return rc;
    const int n = c->s.n;
    int block, wpc;
    bs_shape(c, p, n, &block, &wpc);
    const int cap = p->max_attempts > 0 ? p->max_attempts : 10000000;
    BsArgs a;
    State &S = c->s;
    bs_fill_args(c, p, a, n, S.x, S.y, S.z, S.ux, S.uy, S.uz, S.t, S.nsteps, S.esc, c->bs_ctr,
                 cap);
    a.lanes = bs_lanes(c, wpc, n);
    dim3 grid = bs_grid(c, block, wpc, n, a.lanes);
    const size_t lds = bs_lds(c, block, wpc, a);
    if (n > 0) {
        if (p->use_graph) {
            unsigned long long key = 1469598103934665603ull;
            key = fnv(key, &a, sizeof(a));
            key = fnv(key, &grid, sizeof(grid));
            key = fnv(key, &block, sizeof(block));
            if (!c->bs_graph || c->bs_graph_key != key) {
                if (c->bs_graph) {
                    (void)hipGraphExecDestroy(c->bs_graph);
                    c->bs_graph = nullptr;
                }
                hipGraph_t g;
                HIPCHK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
                hipLaunchKernelGGL(k_bs_reset, dim3(1), dim3(64), 0, c->stream, c->bs_ctr);
                fn(grid, dim3(block), lds, c->stream, a);
                HIPCHK(hipStreamEndCapture(c->stream, &g));
                hipError_t e = hipGraphInstantiate(&c->bs_graph, g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                if (e != hipSuccess) {
                    c->bs_graph = nullptr;
                    return TP_E_HIP;
                }
                c->bs_graph_key = key;
            }
            HIPCHK(hipEventRecord(c->ev0, c->stream));
            HIPCHK(hipGraphLaunch(c->bs_graph, c->stream));
            HIPCHK(hipEventRecord(c->ev1, c->stream));
        } else {
            hipLaunchKernelGGL(k_bs_reset, dim3(1), dim3(64), 0, c->stream, c->bs_ctr);
            HIPCHK(hipGetLastError());
            HIPCHK(hipEventRecord(c->ev0, c->stream));
            fn(grid, dim3(block), lds, c->stream, a);
            HIPCHK(hipGetLastError());
            HIPCHK(hipEventRecord(c->ev1, c->stream));
        }
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    if (stats) {
        memset(stats, 0, sizeof(*stats));
        if (n > 0) {
            unsigned long long h[Q_N];
            HIPCHK(hipMemcpy(h, c->bs_ctr, sizeof(h), hipMemcpyDeviceToHost));
            float ms = 0.f;
            HIPCHK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
            stats->accepted = (long long)h[Q_ACC];
            stats->rejected = (long long)h[Q_REJ];
            stats->rhs_evals = (long long)h[Q_RHS];
            stats->failed = (int)h[Q_FAIL];
            stats->launches = 1;
            stats->kernel_ms = ms;
        }
    }
    return TP_OK;
}

int tp_gpu_run_adaptive_diag(tp_ctx *c, const tp_bs_params *p, const tp_track_params *q,
                             tp_bs_stats *stats)
{
    if (!c || !q) return TP_E_ARG;
    int rc = bs_check(c, p);
    if (rc) return rc;
    if (q->sstep != 1 || q->estep < 1 || q->einterval_t <= 0 || q->dcoeff_interval <= 0 ||
        q->nbins < 1 || q->nt_out < 1 || !(q->dt > 0.0) || q->bc_flag < 0 || q->bc_flag > 2 ||
        q->precision != TP_FP64)
        return TP_E_ARG;
    if ((size_t)q->nbins * sizeof(unsigned) > 64 * 1024) return TP_E_ARG;
    if (!c->s.derived) return TP_E_STATE;
    bs_fn fn = pick_bs_t<true>(c->f.kind);
    if (!fn) return TP_E_ARG;
    HIPCHK(hipSetDevice(c->device));
    if ((rc = bs_ensure_ctr(c))) return rc;
    const int n = c->s.n;
    const int nd = q->estep / q->dcoeff_interval + 1;
    int nframes = q->estep / q->einterval_t;
    if (nframes > q->nt_out) nframes = q->nt_out;
    int block, wpc;
    bs_shape(c, p, n, &block, &wpc);
    const int lanes = bs_lanes(c, wpc, n);
    const dim3 grid = bs_grid(c, block, wpc, n, lanes);
    const long nl = (long)grid.x * (block / 64) * lanes;
    /* the run's outputs in the context's diagnostics buffers (read back by
     * tp_gpu_read_diagnostics), the scratch of the dense form */
    const size_t need = (size_t)q->nbins * q->nt_out;
    if (need > c->diag_cap) {
        (void)hipFree(c->espect); (void)hipFree(c->espect_esc);
        c->espect = nullptr; c->espect_esc = nullptr; c->diag_cap = 0;
        if (hipMalloc(&c->espect, need * sizeof(unsigned)) != hipSuccess ||
            hipMalloc(&c->espect_esc, need * sizeof(unsigned)) != hipSuccess)
            return TP_E_NOMEM;
        c->diag_cap = need;
    }
    if ((size_t)nd > c->dco_cap) {
        (void)hipFree(c->dco); (void)hipFree(c->rdec);
        c->dco = nullptr; c->rdec = nullptr; c->dco_cap = 0;
        if (hipMalloc(&c->dco, sizeof(double) * 8 * nd) != hipSuccess ||
            hipMalloc(&c->rdec, sizeof(int) * (nd + 1)) != hipSuccess)
            return TP_E_NOMEM;
        c->dco_cap = nd;
    }
    const size_t dneed = (size_t)nd * 8 * (n > 0 ? n : 1);
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) == hipSuccess &&
        (dneed + (size_t)nl * DS_ROWS * BS_N) * sizeof(double) > fr / 2 + c->bs_dbuf_cap * sizeof(double))
        return TP_E_NOMEM;
    if ((rc = bs_grow(&c->bs_dbuf, &c->bs_dbuf_cap, dneed)) ||
        (rc = bs_grow(&c->bs_ds, &c->bs_ds_cap, (size_t)nl * DS_ROWS * BS_N)) ||
        (rc = bs_grow(&c->bs_outhist, &c->bs_outhist_cap, (size_t)nd)))
        return rc;
    hipLaunchKernelGGL(k_bs_zero_u32, dim3(256), dim3(256), 0, c->stream, c->espect, need);
    hipLaunchKernelGGL(k_bs_zero_u32, dim3(256), dim3(256), 0, c->stream, c->espect_esc, need);
    hipLaunchKernelGGL(k_bs_zero_u32, dim3(64), dim3(256), 0, c->stream,
                       (unsigned *)c->bs_outhist, (size_t)nd);
    HIPCHK(hipGetLastError());
    c->nb = q->nbins; c->nt = q->nt_out; c->nd = nd; c->last_n = n;
    const int cap = p->max_attempts > 0 ? p->max_attempts : 10000000;
    BsArgs a;
    State &S = c->s;
    bs_fill_args(c, p, a, n, S.x, S.y, S.z, S.ux, S.uy, S.uz, S.t, S.nsteps, S.esc, c->bs_ctr,
                 cap, 1);
    a.lanes = lanes;
    const size_t lds = bs_lds(c, block, wpc, a);
    a.ds = c->bs_ds; a.nl = nl;
    a.dt = q->dt; a.estep = q->estep; a.ei = q->einterval_t; a.di = q->dcoeff_interval;
    a.nd = nd; a.nframes = nframes; a.nbins = q->nbins; a.nt_out = q->nt_out;
    a.bc = q->bc_flag; a.fix_stale = (q->flags & TP_FLAG_FIX_STALE_DCOEFF) ? 1 : 0;
    a.lo[0] = q->xmin; a.lo[1] = q->ymin; a.lo[2] = q->zmin;
    a.hi[0] = q->xmax; a.hi[1] = q->ymax; a.hi[2] = q->zmax;
    a.logemin = q->logemin; a.logde = q->logde;
    a.xs = S.xs; a.ys = S.ys; a.zs = S.zs;
    a.x0 = S.x0; a.y0 = S.y0; a.z0 = S.z0; a.ux0 = S.ux0; a.uy0 = S.uy0; a.uz0 = S.uz0;
    a.g0 = S.g0; a.mu0 = S.mu0; a.th0 = S.th0; a.st = S.st;
    a.espect = c->espect; a.espect_esc = c->espect_esc;
    a.dbuf = c->bs_dbuf; a.outhist = c->bs_outhist;
    if (c->traj_nout > 0) {
        /* armed by tp_gpu_track_adaptive_diag_traj */
        a.traj = c->traj; a.traj_accum = c->traj_accum; a.traj_pts = c->traj_pts;
        a.traj_nout = c->traj_nout; a.stage = S.stage;
    }
    hipLaunchKernelGGL(k_bs_reset, dim3(1), dim3(64), 0, c->stream, c->bs_ctr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev0, c->stream));
    if (n > 0) fn(grid, dim3(block), lds, c->stream, a);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->ev1, c->stream));
    hipLaunchKernelGGL(k_bs_dsum, dim3(8 * nd), dim3(256), 0, c->stream,
                       (const double *)c->bs_dbuf, (long)n, nd, c->dco);
    hipLaunchKernelGGL(k_bs_rdec, dim3(1), dim3(64), 0, c->stream,
                       (const int *)c->bs_outhist, nd, c->rdec);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    unsigned long long h[Q_N];
    HIPCHK(hipMemcpy(h, c->bs_ctr, sizeof(h), hipMemcpyDeviceToHost));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    c->last_launches = 1;
    if (stats) {
        memset(stats, 0, sizeof(*stats));
        stats->accepted = (long long)h[Q_ACC];
        stats->rejected = (long long)h[Q_REJ];
        stats->rhs_evals = (long long)h[Q_RHS];
        stats->failed = (int)h[Q_FAIL];
        stats->launches = 1;
        stats->kernel_ms = ms;
    }
    return TP_OK;
}

int tp_gpu_track_adaptive(tp_ctx *c, const tp_bs_params *p, int n, tp_particle *ptl,
                          int *nsteps, tp_bs_stats *stats)
{
    if (!c || !p || n < 0 || (n > 0 && !ptl)) return TP_E_ARG;
    int rc = bs_check(c, p);
    if (rc) return rc;
    if ((rc = tp_gpu_load_particles(c, n, ptl, ptl))) return rc;
    if ((rc = tp_gpu_run_adaptive(c, p, stats))) return rc;
    return tp_gpu_store_particles(c, ptl, nsteps);
}

int tp_gpu_tune_adaptive(tp_ctx *c, const tp_bs_params *p, const char *cache_path, int *block,
                         int *waves_per_cu)
{
    if (!c) return TP_E_ARG;
    int rc = bs_check(c, p);
    if (rc) return rc;
    if (!c->s.derived || c->s.n <= 0) return TP_E_STATE;
    bs_fn fn = pick_bs(c->f.kind);
    if (!fn) return TP_E_ARG;
    HIPCHK(hipSetDevice(c->device));
    /* "k2": timed on the present kernels; entries of others do not count */
    char key[160];
    snprintf(key, sizeof(key), "k2 fk=%d modes=%d lanes=%d rtol=%.3g kmax=%d cu=%d", c->f.kind,
             c->f.nmodes, bs_class(c, c->s.n), p->rtol, p->kmax, c->num_cu);
    int best_b = 0, best_w = 0;
    if (cache_path) {
        FILE *fp = fopen(cache_path, "r");
        if (fp) {
            char line[256];
            while (fgets(line, sizeof(line), fp)) {
                int b, w;
                double r;
                char k2[160];
                if (sscanf(line, "%d %d %lf %159[^\n]", &b, &w, &r, k2) == 4 &&
                    strcmp(k2, key) == 0) {
                    best_b = b;
                    best_w = w;
                }
            }
            fclose(fp);
        }
    }
    double best_rate = -1.0;
    if (!best_b) {
        if ((rc = bs_ensure_ctr(c))) return rc;
        const int nt = c->s.n < 65536 ? c->s.n : 65536;
        /* scratch copy of the first nt particles: 7 state arrays + 2 int */
        double *buf = nullptr;
        int *ib = nullptr;
        if (hipMalloc(&buf, sizeof(double) * 7 * nt) != hipSuccess) return TP_E_NOMEM;
        if (hipMalloc(&ib, sizeof(int) * 2 * nt) != hipSuccess) {
            (void)hipFree(buf);
            return TP_E_NOMEM;
        }
        const double *src[7] = {c->s.x, c->s.y, c->s.z, c->s.ux, c->s.uy, c->s.uz, c->s.t};
        const int blocks[3] = {64, 128, 256};
        const int wpcs[4] = {4, 8, 16, 24};
        for (int bi = 0; bi < 3 && rc == TP_OK; bi++) {
            for (int wi = 0; wi < 4 && rc == TP_OK; wi++) {
                for (int k = 0; k < 7; k++) {
                    if (hipMemcpyAsync(buf + (size_t)k * nt, src[k], sizeof(double) * nt,
                                       hipMemcpyDeviceToDevice, c->stream) != hipSuccess)
                        rc = TP_E_HIP;
                }
                BsArgs a;
                /* bounded trial: 24 step attempts per particle */
                bs_fill_args(c, p, a, nt, buf, buf + nt, buf + 2 * (size_t)nt,
                             buf + 3 * (size_t)nt, buf + 4 * (size_t)nt, buf + 5 * (size_t)nt,
                             buf + 6 * (size_t)nt, ib, ib + nt, c->bs_ctr, 24);
                a.lanes = bs_lanes(c, wpcs[wi], nt);
                const size_t lds = bs_lds(c, blocks[bi], wpcs[wi], a);
                hipLaunchKernelGGL(k_bs_reset, dim3(1), dim3(64), 0, c->stream, c->bs_ctr);
                (void)hipEventRecord(c->ev0, c->stream);
                fn(bs_grid(c, blocks[bi], wpcs[wi], nt, a.lanes), dim3(blocks[bi]), lds,
                   c->stream, a);
                (void)hipEventRecord(c->ev1, c->stream);
                if (hipGetLastError() != hipSuccess || hipStreamSynchronize(c->stream) != hipSuccess)
                    rc = TP_E_HIP;
                unsigned long long h[Q_N];
                float ms = 0.f;
                if (rc == TP_OK &&
                    (hipMemcpy(h, c->bs_ctr, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess ||
                     hipEventElapsedTime(&ms, c->ev0, c->ev1) != hipSuccess))
                    rc = TP_E_HIP;
                if (rc == TP_OK && ms > 0.f) {
                    double rate = (double)h[Q_RHS] / ms;
                    if (rate > best_rate) {
                        best_rate = rate;
                        best_b = blocks[bi];
                        best_w = wpcs[wi];
                    }
                }
            }
        }
        (void)hipFree(buf);
        (void)hipFree(ib);
        if (rc) return rc;
        if (cache_path && best_b) {
            FILE *fp = fopen(cache_path, "a");
            if (fp) {
                fprintf(fp, "%d %d %.6g %s\n", best_b, best_w, best_rate, key);
                fclose(fp);
            }
        }
    }
    if (!best_b) return TP_E_HIP;
    c->bs_tuned[0] = best_b;
    c->bs_tuned[1] = best_w;
    c->bs_tuned[2] = bs_class(c, c->s.n);
    if (block) *block = best_b;
    if (waves_per_cu) *waves_per_cu = best_w;
    return TP_OK;
}

} /* extern "C" */
