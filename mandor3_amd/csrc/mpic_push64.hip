/*
 * mpic_push64.hip -- FP64 plain-form marker push and current deposit.
 *
 * Per marker: trilinear gather of E and H on the staggered Yee
 * grid (source/misc_PIC.h:18-126), relativistic Boris rotation
 * (source/core/plasma.c:115-171), charge-conserving deposit of the straight
 * trajectory split at cell faces (source/core/plasma_currentKernel.c:20-279)
 * and the particle walls (source/core/plasma_walls.c:27-104).  Built with
 * -ffp-contract=off so each marker's arithmetic is the reference's, bit for
 * bit; J is accumulated with FP64 atomics, so only the summation order of J
 * differs from the CPU path.
 *
 * Two kernels: the tiled push (the default; one workgroup per tile of
 * sorted markers, fields and J staged in LDS) and the untiled one (one thread
 * per marker, everything straight from and to HBM), whose general marker
 * push also takes the markers the tiled one leaves.
 *
 * Roofline: HBM-bound.  Algorithmic bytes per marker-step: 128 B (read the
 * order's index, 56 B of state and the id; write state, id and new key), plus
 * per cell 48 B of E/H reads and 48 B of J read-modify-write divided by the
 * markers per cell.
 */
#include "mpic_internal.h"
#include "mpic_launch.h"
#include "mpic_tiles.h"

#define TPB 256

#define DBL_TO_INT(x) ((int)((x) + 128.0) - 128)

struct F64View {
    const double *E[3], *H[3];
    double *J[3];
    Grid g;
};

__device__ static inline double gather(const double *F, const Grid &g, int i, double sx, int j,
                                       double sy, int k, double sz)
{
    return F[gidx(g, i, j, k)] * (1 - sx) * ((1 - sy) * (1 - sz)) +
           F[gidx(g, i + 1, j, k)] * sx * ((1 - sy) * (1 - sz)) +
           F[gidx(g, i, j + 1, k)] * (1 - sx) * (sy * (1 - sz)) +
           F[gidx(g, i + 1, j + 1, k)] * sx * (sy * (1 - sz)) +
           F[gidx(g, i, j, k + 1)] * (1 - sx) * ((1 - sy) * sz) +
           F[gidx(g, i + 1, j, k + 1)] * sx * ((1 - sy) * sz) +
           F[gidx(g, i, j + 1, k + 1)] * (1 - sx) * (sy * sz) +
           F[gidx(g, i + 1, j + 1, k + 1)] * sx * (sy * sz);
}

/* Deposit target of the untiled push: J in HBM, by FP64 atomics. */
struct GlobalSink {
    double *J[3];
    Grid g;
    __device__ void seg(int i, int j, int k, const double vx[4], const double vy[4],
                        const double vz[4]) const
    {
        unsafeAtomicAdd(J[0] + gidx(g, i + 1, j, k), vx[0]);
        unsafeAtomicAdd(J[0] + gidx(g, i + 1, j + 1, k), vx[1]);
        unsafeAtomicAdd(J[0] + gidx(g, i + 1, j, k + 1), vx[2]);
        unsafeAtomicAdd(J[0] + gidx(g, i + 1, j + 1, k + 1), vx[3]);
        unsafeAtomicAdd(J[1] + gidx(g, i, j + 1, k), vy[0]);
        unsafeAtomicAdd(J[1] + gidx(g, i + 1, j + 1, k), vy[1]);
        unsafeAtomicAdd(J[1] + gidx(g, i, j + 1, k + 1), vy[2]);
        unsafeAtomicAdd(J[1] + gidx(g, i + 1, j + 1, k + 1), vy[3]);
        unsafeAtomicAdd(J[2] + gidx(g, i, j, k + 1), vz[0]);
        unsafeAtomicAdd(J[2] + gidx(g, i + 1, j, k + 1), vz[1]);
        unsafeAtomicAdd(J[2] + gidx(g, i, j + 1, k + 1), vz[2]);
        unsafeAtomicAdd(J[2] + gidx(g, i + 1, j + 1, k + 1), vz[3]);
    }
};

/* The 12 current values of one straight segment inside cell (i,j,k). */
__device__ static inline void seg_values(const Grid &g, int i, int j, int k, double x1, double x2,
                                         double y1, double y2, double z1, double z2, double rp,
                                         double vx[4], double vy[4], double vz[4])
{
    const double h1 = g.h[0], h2 = g.h[1], h3 = g.h[2], tau = g.tau;
    const double dX = x2 - x1, dY = y2 - y1, dZ = z2 - z1;
    const double tX = 0.5 * (x1 + x2) - i * h1;
    const double tY = 0.5 * (y1 + y2) - j * h2;
    const double tZ = 0.5 * (z1 + z2) - k * h3;
    const double yz = dY * dZ / 12, xz = dX * dZ / 12, xy = dX * dY / 12;
    const double ax = rp * dX / (tau * h2 * h3);
    const double ay = rp * dY / (tau * h1 * h3);
    const double az = rp * dZ / (tau * h1 * h2);
    vx[0] = ax * ((h2 - tY) * (h3 - tZ) + yz);
    vx[1] = ax * (tY * (h3 - tZ) - yz);
    vx[2] = ax * ((h2 - tY) * tZ - yz);
    vx[3] = ax * (tY * tZ + yz);
    vy[0] = ay * ((h1 - tX) * (h3 - tZ) + xz);
    vy[1] = ay * (tX * (h3 - tZ) - xz);
    vy[2] = ay * ((h1 - tX) * tZ - xz);
    vy[3] = ay * (tX * tZ + xz);
    vz[0] = az * ((h1 - tX) * (h2 - tY) + xy);
    vz[1] = az * (tX * (h2 - tY) - xy);
    vz[2] = az * ((h1 - tX) * tY - xy);
    vz[3] = az * (tX * tY + xy);
}

/* Deposit of one straight segment inside cell (i,j,k). */
__device__ static void deposit_seg(const GlobalSink &v, const Grid &g, int i, int j, int k, double x1,
                                   double x2, double y1, double y2, double z1, double z2,
                                   double rp)
{
    double vx[4], vy[4], vz[4];
    seg_values(g, i, j, k, x1, x2, y1, y2, z1, z2, rp, vx, vy, vz);
    v.seg(i, j, k, vx, vy, vz);
}

/* Two or three face crossings, source/core/plasma_currentKernel.c:156-279. */
__device__ static void deposit_multi(const GlobalSink &v, const Grid &g, int i1, int j1, int k1,
                                     int i2, int j2, int k2, double x1, double y1, double z1,
                                     double x2, double y2, double z2, double rp)
{
    const double h1 = g.h[0], h2 = g.h[1], h3 = g.h[2];
    const int di = abs(i2 - i1), dj = abs(j2 - j1), dk = abs(k2 - k1);
    if (di + dj + dk == 2) {
        int i = i1, j = j1, k = k1;
        const double sgX = di * ((i1 + i2 + 1) * 0.5 * h1 - x1) / (x2 - x1 + ((1 - di) << 16));
        const double sgY = dj * ((j1 + j2 + 1) * 0.5 * h2 - y1) / (y2 - y1 + ((1 - dj) << 16));
        const double sgZ = dk * ((k1 + k2 + 1) * 0.5 * h3 - z1) / (z2 - z1 + ((1 - dk) << 16));
        double k1s = sgX + (1 - di) * sgY;
        double k2s = sgZ + (1 - dk) * sgY;
        /* the two crossings' cell steps, in the order they happen (selected
         * by value: an array picked by pointer would live in scratch) */
        const int dI0[3] = {di * (i2 - i1), (1 - di) * (j2 - j1), 0};
        const int dI1[3] = {0, (1 - dk) * (j2 - j1), dk * (k2 - k1)};
        int st = 0;
        if (k1s > k2s) {
            double t = k1s;
            k1s = k2s;
            k2s = t;
            st = 1;
        }
        const double xA = x1 + k1s * (x2 - x1), yA = y1 + k1s * (y2 - y1), zA = z1 + k1s * (z2 - z1);
        const double xB = x1 + k2s * (x2 - x1), yB = y1 + k2s * (y2 - y1), zB = z1 + k2s * (z2 - z1);
        deposit_seg(v, g, i, j, k, x1, xA, y1, yA, z1, zA, rp);
        i += st ? dI1[0] : dI0[0];
        j += st ? dI1[1] : dI0[1];
        k += st ? dI1[2] : dI0[2];
        deposit_seg(v, g, i, j, k, xA, xB, yA, yB, zA, zB, rp);
        i += st ? dI0[0] : dI1[0];
        j += st ? dI0[1] : dI1[1];
        k += st ? dI0[2] : dI1[2];
        deposit_seg(v, g, i, j, k, xB, x2, yB, y2, zB, z2, rp);
        return;
    }
    const double xC = (i1 + i2 + 1) * 0.5 * h1, yC = (j1 + j2 + 1) * 0.5 * h2,
                 zC = (k1 + k2 + 1) * 0.5 * h3;
    double sg[3] = {(xC - x1) / (x2 - x1), (yC - y1) / (y2 - y1), (zC - z1) / (z2 - z1)};
    double rc[3][3];
    rc[0][0] = xC;
    rc[0][1] = y1 + sg[0] * (y2 - y1);
    rc[0][2] = z1 + sg[0] * (z2 - z1);
    rc[1][0] = x1 + sg[1] * (x2 - x1);
    rc[1][1] = yC;
    rc[1][2] = z1 + sg[1] * (z2 - z1);
    rc[2][0] = x1 + sg[2] * (x2 - x1);
    rc[2][1] = y1 + sg[2] * (y2 - y1);
    rc[2][2] = zC;
    const int dI[3] = {i2 - i1, j2 - j1, k2 - k1};
    int s1 = 0, s2 = 1, s3 = 2;
    double a1 = sg[0], a2 = sg[1], a3 = sg[2];
    if (a1 > a2) { int t = s1; s1 = s2; s2 = t; double d = a1; a1 = a2; a2 = d; }
    if (a1 > a3) { int t = s1; s1 = s3; s3 = t; double d = a1; a1 = a3; a3 = d; }
    if (a2 > a3) { int t = s2; s2 = s3; s3 = t; double d = a2; a2 = a3; a3 = d; }
    int ii[3] = {i1, j1, k1};
    deposit_seg(v, g, ii[0], ii[1], ii[2], x1, rc[s1][0], y1, rc[s1][1], z1, rc[s1][2], rp);
    ii[s1] += dI[s1];
    deposit_seg(v, g, ii[0], ii[1], ii[2], rc[s1][0], rc[s2][0], rc[s1][1], rc[s2][1], rc[s1][2],
                rc[s2][2], rp);
    ii[s2] += dI[s2];
    deposit_seg(v, g, ii[0], ii[1], ii[2], rc[s2][0], rc[s3][0], rc[s2][1], rc[s3][1], rc[s2][2],
                rc[s3][2], rp);
    deposit_seg(v, g, i2, j2, k2, rc[s3][0], x2, rc[s3][1], y2, rc[s3][2], z2, rp);
}

/* Particle walls in the reference order xMin yMin zMin xMax yMax zMax.
 * Returns 0 when an open wall deletes the marker. */
__device__ static inline int walls(const PushConsts &c, double *r, double *u)
{
    for (int b = 0; b < 6; ++b) {
        const int ax = b % 3, top = b / 3, bc = c.bc[b];
        const double bnd = top ? c.shell2[ax] : c.shell1[ax];
        if (bc == MPIC_BC_PERIODIC) {
            if (top ? (r[ax] >= bnd) : (r[ax] <= bnd)) r[ax] += top ? -c.L[ax] : c.L[ax];
        } else if (bc == MPIC_BC_MIRROR) {
            if (top ? (r[ax] >= bnd) : (r[ax] <= bnd)) {
                r[ax] = 2 * bnd - r[ax];
                u[ax] *= -1;
            }
        } else if (bc == MPIC_BC_OPEN) {
            const double lim = top ? bnd - c.h[ax] : bnd + c.h[ax];
            if (top ? (r[ax] >= lim) : (r[ax] <= lim)) return 0;
        }
    }
    return 1;
}

/* Gather, Boris and deposit of one live marker; returns 0 for a marker off
 * the grid (deleted and flagged), else applies the walls and returns
 * whether the marker survives.  r/u are in/out. */
__device__ static int push_marker(const GlobalSink &sink, const F64View &v, const PushConsts &c,
                                  double r[3], double u[3], float rhof, float qmf, double w3[3],
                                  unsigned *err)
{
    const Grid &g = v.g;
    const double h1 = g.h[0], h2 = g.h[1], h3 = g.h[2], tau = g.tau;
    const double x1 = r[0], y1 = r[1], z1 = r[2];
    if (!(x1 / h1 > -1.0 && x1 / h1 < g.n[0] + 1.0 && y1 / h2 > -1.0 &&
          y1 / h2 < g.n[1] + 1.0 && z1 / h3 > -1.0 && z1 / h3 < g.n[2] + 1.0)) {
        atomicOr(err, 1u);
        return 0;
    }
    double sx, sy, sz, sx_, sy_, sz_;
    int i, j, k, i_, j_, k_;
    sx = x1 / h1; sx_ = sx + 0.5; i = DBL_TO_INT(sx); i_ = DBL_TO_INT(sx_); sx -= i; sx_ -= i_;
    sy = y1 / h2; sy_ = sy + 0.5; j = DBL_TO_INT(sy); j_ = DBL_TO_INT(sy_); sy -= j; sy_ -= j_;
    sz = z1 / h3; sz_ = sz + 0.5; k = DBL_TO_INT(sz); k_ = DBL_TO_INT(sz_); sz -= k; sz_ -= k_;
    const double Ex = gather(v.E[0], g, i_, sx_, j, sy, k, sz),
                 Ey = gather(v.E[1], g, i, sx, j_, sy_, k, sz),
                 Ez = gather(v.E[2], g, i, sx, j, sy, k_, sz_),
                 Hx = gather(v.H[0], g, i, sx, j_, sy_, k_, sz_),
                 Hy = gather(v.H[1], g, i_, sx_, j, sy, k_, sz_),
                 Hz = gather(v.H[2], g, i_, sx_, j_, sy_, k, sz);
    const double tauMass = 0.5 * tau * qmf, px = u[0] + tauMass * Ex, py = u[1] + tauMass * Ey,
                 pz = u[2] + tauMass * Ez, gamma = sqrt(1 + px * px + py * py + pz * pz);
    const double W = (gamma - 1.0) * rhof / (px * px + py * py + pz * pz + 1e-19) * h1 * h2 * h3 / qmf;
    w3[0] += W * px * px;
    w3[1] += W * py * py;
    w3[2] += W * pz * pz;
    const double tauGamma = tauMass / gamma;
    const double aHx = tauGamma * Hx, aHy = tauGamma * Hy, aHz = tauGamma * Hz;
    const double uu = px + py * aHz - pz * aHy, vv = py + pz * aHx - px * aHz,
                 ww = pz + px * aHy - py * aHx;
    const double bxx = aHx * aHx, byy = aHy * aHy, bzz = aHz * aHz, bxy = aHx * aHy,
                 byz = aHy * aHz, bxz = aHz * aHx;
    const double delta = 1.0 / (1 + bxx + byy + bzz);
    u[0] = tauMass * Ex + ((1 + bxx) * uu + (bxy + aHz) * vv + (bxz - aHy) * ww) * delta;
    u[1] = tauMass * Ey + ((bxy - aHz) * uu + (1 + byy) * vv + (byz + aHx) * ww) * delta;
    u[2] = tauMass * Ez + ((bxz + aHy) * uu + (byz - aHx) * vv + (1 + bzz) * ww) * delta;
    const double tg = tau / sqrt(1 + u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
    const double x2 = x1 + u[0] * tg, y2 = y1 + u[1] * tg, z2 = z1 + u[2] * tg;
    int i2 = DBL_TO_INT(x2 / h1), j2 = DBL_TO_INT(y2 / h2), k2 = DBL_TO_INT(z2 / h3);
    int di = abs(i2 - i), dj = abs(j2 - j), dk = abs(k2 - k);
    if (fabs(x2 - x1) < 1e-10 * h1) { di = 0; i2 = i; }
    if (fabs(y2 - y1) < 1e-10 * h2) { dj = 0; j2 = j; }
    if (fabs(z2 - z1) < 1e-10 * h3) { dk = 0; k2 = k; }
    const double rp = rhof;
    if (di + dj + dk == 0) {
        deposit_seg(sink, g, i, j, k, x1, x2, y1, y2, z1, z2, rp);
    } else if (di + dj + dk == 1) {
        const double alpha = dk * ((k + k2 + 1) * 0.5 * h3 - z1) / (z2 - z1 + ((1 - dk) << 16))
                           + dj * ((j + j2 + 1) * 0.5 * h2 - y1) / (y2 - y1 + ((1 - dj) << 16))
                           + di * ((i + i2 + 1) * 0.5 * h1 - x1) / (x2 - x1 + ((1 - di) << 16));
        const double xC = x1 + alpha * (x2 - x1), yC = y1 + alpha * (y2 - y1),
                     zC = z1 + alpha * (z2 - z1);
        deposit_seg(sink, g, i, j, k, x1, xC, y1, yC, z1, zC, rp);
        deposit_seg(sink, g, i2, j2, k2, xC, x2, yC, y2, zC, z2, rp);
    } else {
        deposit_multi(sink, g, i, j, k, i2, j2, k2, x1, y1, z1, x2, y2, z2, rp);
    }
    r[0] = x2;
    r[1] = y2;
    r[2] = z2;
    return walls(c, r, u);
}

__device__ static void block_sum3(double w3[3], double *ks)
{
    __shared__ double sw[3][TPB];
    sw[0][threadIdx.x] = w3[0];
    sw[1][threadIdx.x] = w3[1];
    sw[2][threadIdx.x] = w3[2];
    __syncthreads();
    for (int s = TPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sw[0][threadIdx.x] += sw[0][threadIdx.x + s];
            sw[1][threadIdx.x] += sw[1][threadIdx.x + s];
            sw[2][threadIdx.x] += sw[2][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicAdd(ks + 0, sw[0][0]);
        atomicAdd(ks + 1, sw[1][0]);
        atomicAdd(ks + 2, sw[2][0]);
    }
}

/* Untiled push: one thread per marker, J straight to HBM.  mode 1 applies
 * the walls only (plasma_init).  A marker whose cell lies outside [-1, n]
 * (a state the reference never produces) is deleted and flagged in *err
 * instead of touching memory off the grid. */
struct Push64Args {
    Markers64  m;
    long       n;
    F64View    v;
    PushConsts c;
    double    *kin;
    int        mode;
    unsigned  *err;
};

__device__ __forceinline__ static void push64(const Markers64 &m, long n, const F64View &v,
                                     const PushConsts &c, double *kin, int mode, unsigned *err,
                                     long p)
{
    double w3[3] = {0, 0, 0};
    if (p < n && m.qm[p] != 0.0f) {
        double r[3] = {m.x[p], m.y[p], m.z[p]};
        double u[3] = {m.ux[p], m.uy[p], m.uz[p]};
        GlobalSink gs;
        for (int a = 0; a < 3; ++a) gs.J[a] = v.J[a];
        gs.g = v.g;
        int alive = (mode == 0) ? push_marker(gs, v, c, r, u, m.w[p], m.qm[p], w3, err)
                                : walls(c, r, u);
        if (!alive) {
            m.qm[p] = 0.0f;
            m.w[p] = 0.0f;
        } else {
            m.x[p] = r[0];
            m.y[p] = r[1];
            m.z[p] = r[2];
            m.ux[p] = u[0];
            m.uy[p] = u[1];
            m.uz[p] = u[2];
        }
    }
    if (mode != 0) return;
    block_sum3(w3, kin_slot(kin, (unsigned)(p / TPB)));
}

template <> struct KernelDef<Push64Args> {
    static constexpr int kBlock = TPB;
    __device__ __forceinline__ static void body(const Push64Args &a, VBlock b, VBlock)
    {
        push64(a.m, a.n, a.v, a.c, a.kin, a.mode, a.err, (long)b.x * TPB + threadIdx.x);
    }
};

int launch_push64(hipStream_t s, const Markers64 &m, long n, const Fields64 &f, const Grid &g,
                  const PushConsts &c, double *kin, int mode, unsigned *err)
{
    if (n <= 0) return MPIC_OK;
    F64View v;
    for (int a = 0; a < 3; ++a) {
        v.E[a] = f.E[a];
        v.H[a] = f.H[a];
        v.J[a] = f.J[a];
    }
    v.g = g;
    Push64Args a = {m, n, v, c, kin, mode, err};
    return launch_def(s, a, (unsigned)((n + TPB - 1) / TPB));
}

/* ---------------- tiled push ---------------- */
#define TW 64                  /* wavefront width */
#define TILE 4
#define TFN (TILE + 2)         /* E/H nodes per axis staged for a tile's gathers */
#define TFN3 (TFN * TFN * TFN)

struct Push64Consts {
    PushConsts pc;
    double     yh[3], yl[3];   /* 1/h as the sum of two doubles */
    double     cj[3];          /* h/tau: J of a segment per unit charge density and cell */
    double     vol;            /* h1*h2*h3 */
};

/* a / b, correctly rounded, from b's reciprocal yh + yl (yh = RN(1/b), yl
 * the rounded rest): q is within one unit in the last place of a/b, the
 * remainder a - q b is exact, and one correction with yh = RN(1/b) then
 * rounds correctly (P. W. Markstein, "Computation of elementary functions on
 * the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990).  Four
 * instructions instead of the eleven of a division; a zero's sign may differ. */
__device__ static inline double div_by(double a, double b, double yh, double yl)
{
    const double q = __builtin_fma(a, yh, a * yl);
    return __builtin_fma(__builtin_fma(-b, q, a), yh, q);
}

/* 1/x to about one unit in the last place: the hardware's estimate and two
 * Newton steps.  Used where the reference's rounding does not matter (the
 * crossing fraction of a segment, the energy sums). */
__device__ static inline double rcp64(double x)
{
    double y = __builtin_amdgcn_rcp(x);
    y = __builtin_fma(__builtin_fma(-x, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-x, y, 1.0), y, y);
}

__device__ static inline void cswap(double &a, int &ia, double &b, int &ib)
{
    if (b < a) {
        const double t = a; a = b; b = t;
        const int u = ia; ia = ib; ib = u;
    }
}

/* Marker state held in registers between the prefetch and the push, and
 * between the push and the stores. */
struct Marker64 {
    double  r[3], u[3];
    float   w, qm;
    int32_t id;
};

/* Records are read once and written once per step: nontemporal, so that they
 * do not push the fields out of the caches. */
__device__ static inline void load_marker(const Markers64 &m, unsigned s, Marker64 &k)
{
    k.r[0] = __builtin_nontemporal_load(m.x + s);
    k.r[1] = __builtin_nontemporal_load(m.y + s);
    k.r[2] = __builtin_nontemporal_load(m.z + s);
    k.u[0] = __builtin_nontemporal_load(m.ux + s);
    k.u[1] = __builtin_nontemporal_load(m.uy + s);
    k.u[2] = __builtin_nontemporal_load(m.uz + s);
    k.w = __builtin_nontemporal_load(m.w + s);
    k.qm = __builtin_nontemporal_load(m.qm + s);
    k.id = __builtin_nontemporal_load(m.id + s);
}

/* Results of one batch, written back at the start of the next (after its
 * prefetch is issued), so that no wait for the prefetch also waits for
 * fresh stores. */
struct Pending64 {
    Marker64 k;
    unsigned p;
    int      key;              /* new key, -1 deleted */
    bool     valid;            /* lane holds a marker of the order */
    int      ckey, clen;       /* count run head: key (-1 none), length */
};

__device__ static inline void write_back(const Markers64 &d, const TileView &tv,
                                         const Pending64 &q)
{
    if (q.valid) {
        if (q.key >= 0) {
            __builtin_nontemporal_store(q.k.r[0], d.x + q.p);
            __builtin_nontemporal_store(q.k.r[1], d.y + q.p);
            __builtin_nontemporal_store(q.k.r[2], d.z + q.p);
            __builtin_nontemporal_store(q.k.u[0], d.ux + q.p);
            __builtin_nontemporal_store(q.k.u[1], d.uy + q.p);
            __builtin_nontemporal_store(q.k.u[2], d.uz + q.p);
        }
        __builtin_nontemporal_store(q.key >= 0 ? q.k.w : 0.0f, d.w + q.p);
        __builtin_nontemporal_store(q.key >= 0 ? q.k.qm : 0.0f, d.qm + q.p);
        __builtin_nontemporal_store(q.k.id, d.id + q.p);
        tv.key[q.p] = q.key;                               /* read by the rank pass next */
    }
    if (q.ckey >= 0) atomicAdd(tv.count + q.ckey, q.clen);
}

/* The reference's trilinear sum over eight values, in its order. */
__device__ static inline double lgather(const double *F, int a, double sx, int b, double sy,
                                        int c, double sz)
{
    const double *p = F + (a * TFN + b) * TFN + c;
    const int dj = TFN, di = TFN * TFN;
    return p[0] * (1 - sx) * ((1 - sy) * (1 - sz)) + p[di] * sx * ((1 - sy) * (1 - sz)) +
           p[dj] * (1 - sx) * (sy * (1 - sz)) + p[di + dj] * sx * (sy * (1 - sz)) +
           p[1] * (1 - sx) * ((1 - sy) * sz) + p[di + 1] * sx * ((1 - sy) * sz) +
           p[dj + 1] * (1 - sx) * (sy * sz) + p[di + dj + 1] * sx * (sy * sz);
}

/* 12 J values of one straight segment inside a cell, in cell units: start
 * q1, end q2 relative to the cell's origin, w3[a] = rho h_a / tau.  The
 * deposit's sums are rounded in any order anyway, so its arithmetic may fuse
 * multiply and add. */
__device__ static inline void seg_cell(const double q1[3], const double q2[3], const double w3[3],
                                       double v[12])
{
#pragma clang fp contract(fast)
    const double dx = q2[0] - q1[0], dy = q2[1] - q1[1], dz = q2[2] - q1[2];
    const double tx = 0.5 * (q1[0] + q2[0]), ty = 0.5 * (q1[1] + q2[1]), tz = 0.5 * (q1[2] + q2[2]);
    const double yz = dy * dz * (1.0 / 12), xz = dx * dz * (1.0 / 12), xy = dx * dy * (1.0 / 12);
    const double ax = w3[0] * dx, ay = w3[1] * dy, az = w3[2] * dz;
    v[0] = ax * ((1 - ty) * (1 - tz) + yz);
    v[1] = ax * (ty * (1 - tz) - yz);
    v[2] = ax * ((1 - ty) * tz - yz);
    v[3] = ax * (ty * tz + yz);
    v[4] = ay * ((1 - tx) * (1 - tz) + xz);
    v[5] = ay * (tx * (1 - tz) - xz);
    v[6] = ay * ((1 - tx) * tz - xz);
    v[7] = ay * (tx * tz + xz);
    v[8] = az * ((1 - tx) * (1 - ty) + xy);
    v[9] = az * (tx * (1 - ty) - xy);
    v[10] = az * ((1 - tx) * ty - xy);
    v[11] = az * (tx * ty + xy);
}

/* Offset of node (+da,+db,+dc), component comp, from a node of the LDS J block. */
#define LJO(da, db, dc, comp) (3 * (((da) * TJN + (db)) * TJN + (dc)) + (comp))

/* A segment of the LDS block's cell (a, b, c), 0 to TJN - 2 each: a marker of
 * the tile starts in block cells 1 to 4 and crosses at most one face per axis. */
__device__ static inline void seg_add(double *lj, int a, int b, int c, const double s[12])
{
    double *p = lj + 3 * ((a * TJN + b) * TJN + c);
    atomicAdd(p + LJO(1, 0, 0, 0), s[0]);
    atomicAdd(p + LJO(1, 1, 0, 0), s[1]);
    atomicAdd(p + LJO(1, 0, 1, 0), s[2]);
    atomicAdd(p + LJO(1, 1, 1, 0), s[3]);
    atomicAdd(p + LJO(0, 1, 0, 1), s[4]);
    atomicAdd(p + LJO(1, 1, 0, 1), s[5]);
    atomicAdd(p + LJO(0, 1, 1, 1), s[6]);
    atomicAdd(p + LJO(1, 1, 1, 1), s[7]);
    atomicAdd(p + LJO(0, 0, 1, 2), s[8]);
    atomicAdd(p + LJO(1, 0, 1, 2), s[9]);
    atomicAdd(p + LJO(0, 1, 1, 2), s[10]);
    atomicAdd(p + LJO(1, 1, 1, 2), s[11]);
}

/* The tile being pushed: its index, first cell, neighbour strides (in tiles)
 * and whether a wall lies within reach of its markers (they move less than a
 * cell per step, so a tile one tile or more from every face is out of
 * reach). */
struct Tile64 {
    int  t, c[3], s0, s1;
    bool edge;
};

/* First segment of a lane's marker: the block cell that holds it (a << 8 | b
 * << 4 | c), -1 when there is none to sum over the wavefront. */
struct First64 {
    int    cell;
    double v[12];
};

/* Push of one marker: gather, Boris and move with the reference's arithmetic
 * (bit for bit), deposit of every segment but the first into the tile's
 * block.  Returns the new key (-1: deleted); k holds the new state.  A marker
 * whose cell is not the tile's (its quotient rounds onto the box's far face,
 * where its key was clamped, or it lies off the grid) is left untouched:
 * OFF_TILE. */
#define OFF_TILE -2
__device__ static inline int push64_marker(Marker64 &k, const F64View &v, const Push64Consts &c,
                                           const TileView &tv, const Tile64 &tl, const double *lf,
                                           double *lj, First64 &first, double w3[3])
{
    const Grid &g = v.g;
    const double tau = c.pc.tau;
    double s[3], f[3], fh[3];
    int ic[3], ih[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s[a] = div_by(k.r[a], c.pc.h[a], c.yh[a], c.yl[a]);
        const double sh = s[a] + 0.5;
        ic[a] = DBL_TO_INT(s[a]);
        ih[a] = DBL_TO_INT(sh);
        f[a] = s[a] - ic[a];
        fh[a] = sh - ih[a];
    }
    const int l[3] = {ic[0] - tl.c[0], ic[1] - tl.c[1], ic[2] - tl.c[2]};
    if ((unsigned)l[0] >= TILE || (unsigned)l[1] >= TILE || (unsigned)l[2] >= TILE) return OFF_TILE;
    const int m[3] = {ih[0] - tl.c[0], ih[1] - tl.c[1], ih[2] - tl.c[2]};
    const double Ex = lgather(lf + 0 * TFN3, m[0], fh[0], l[1], f[1], l[2], f[2]),
                 Ey = lgather(lf + 1 * TFN3, l[0], f[0], m[1], fh[1], l[2], f[2]),
                 Ez = lgather(lf + 2 * TFN3, l[0], f[0], l[1], f[1], m[2], fh[2]),
                 Hx = lgather(lf + 3 * TFN3, l[0], f[0], m[1], fh[1], m[2], fh[2]),
                 Hy = lgather(lf + 4 * TFN3, m[0], fh[0], l[1], f[1], m[2], fh[2]),
                 Hz = lgather(lf + 5 * TFN3, m[0], fh[0], m[1], fh[1], l[2], f[2]);
    const double tauMass = 0.5 * tau * k.qm, px = k.u[0] + tauMass * Ex,
                 py = k.u[1] + tauMass * Ey, pz = k.u[2] + tauMass * Ez,
                 gamma = sqrt(1 + px * px + py * py + pz * pz);
    {
#pragma clang fp contract(fast)
        const double p2 = px * px + py * py + pz * pz;
        const double W = (gamma - 1.0) * k.w * c.vol * rcp64((p2 + 1e-19) * k.qm);
        w3[0] += W * px * px;
        w3[1] += W * py * py;
        w3[2] += W * pz * pz;
    }
    const double tauGamma = tauMass / gamma;
    const double aHx = tauGamma * Hx, aHy = tauGamma * Hy, aHz = tauGamma * Hz;
    const double uu = px + py * aHz - pz * aHy, vv = py + pz * aHx - px * aHz,
                 ww = pz + px * aHy - py * aHx;
    const double bxx = aHx * aHx, byy = aHy * aHy, bzz = aHz * aHz, bxy = aHx * aHy,
                 byz = aHy * aHz, bxz = aHz * aHx;
    const double delta = 1.0 / (1 + bxx + byy + bzz);
    k.u[0] = tauMass * Ex + ((1 + bxx) * uu + (bxy + aHz) * vv + (bxz - aHy) * ww) * delta;
    k.u[1] = tauMass * Ey + ((bxy - aHz) * uu + (1 + byy) * vv + (byz + aHx) * ww) * delta;
    k.u[2] = tauMass * Ez + ((bxz + aHy) * uu + (byz - aHx) * vv + (1 + bzz) * ww) * delta;
    const double tg = tau / sqrt(1 + k.u[0] * k.u[0] + k.u[1] * k.u[1] + k.u[2] * k.u[2]);
    /* the move: cells crossed per axis (-1, 0, 1) and the displacement in cells */
    double d[3], rho3[3];
    int to[3], fc[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double x1 = k.r[a], x2 = x1 + k.u[a] * tg;
        /* (a marker moves less than a cell: the clamp only keeps one that is
         * not a number inside the block) */
        to[a] = DBL_TO_INT(div_by(x2, c.pc.h[a], c.yh[a], c.yl[a])) - ic[a];
        to[a] = to[a] < -1 ? -1 : (to[a] > 1 ? 1 : to[a]);
        fc[a] = fabs(x2 - x1) < 1e-10 * c.pc.h[a] ? 0 : to[a];
        d[a] = (x2 - x1) * c.yh[a];
        rho3[a] = k.w * c.cj[a];
        k.r[a] = x2;
    }
    /* Segments: from the start to the first face crossing (or the end), then
     * one per crossed face.  Crossing fractions ascend; an axis that is not
     * crossed gets 2 and sorts last. */
    const int nc = (fc[0] != 0) + (fc[1] != 0) + (fc[2] != 0);
    double a0 = 2.0, a1 = 2.0, a2 = 2.0, q[3] = {f[0] + d[0], f[1] + d[1], f[2] + d[2]};
    const double e[3] = {q[0], q[1], q[2]};
    int x0 = 0, x1 = 1, x2i = 2;
    if (nc) {
        if (fc[0]) a0 = ((fc[0] > 0 ? 1.0 : 0.0) - f[0]) * rcp64(d[0]);
        if (fc[1]) a1 = ((fc[1] > 0 ? 1.0 : 0.0) - f[1]) * rcp64(d[1]);
        if (fc[2]) a2 = ((fc[2] > 0 ? 1.0 : 0.0) - f[2]) * rcp64(d[2]);
        cswap(a0, x0, a1, x1);
        cswap(a1, x1, a2, x2i);
        cswap(a0, x0, a1, x1);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            q[a] = x0 == a ? (fc[a] > 0 ? 1.0 : 0.0) : __builtin_fma(a0, d[a], f[a]);
    }
    const double qf[3] = {q[0], q[1], q[2]};     /* the first segment's end */
    if (nc) {
        int sh[3] = {0, 0, 0}, axs = x0;
#pragma unroll 1
        for (int n = 1; n <= nc; ++n) {
            double b[3], en[3], sv[12];
            a0 = a1;
            x0 = x1;
            a1 = a2;
            x1 = x2i;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                sh[a] += axs == a ? fc[a] : 0;
                const double at = x0 == a ? (fc[a] > 0 ? 1.0 : 0.0) : __builtin_fma(a0, d[a], f[a]);
                const double nx = n < nc ? at : e[a];
                b[a] = q[a] - sh[a];
                en[a] = nx - sh[a];
                q[a] = nx;
            }
            seg_cell(b, en, rho3, sv);
            seg_add(lj, l[0] + 1 + sh[0], l[1] + 1 + sh[1], l[2] + 1 + sh[2], sv);
            axs = x0;
        }
    }
    /* after the loop, so that its twelve values are not live through it */
    seg_cell(f, qf, rho3, first.v);
    first.cell = (l[0] + 1) << 8 | (l[1] + 1) << 4 | (l[2] + 1);
    if (!tl.edge) {
        /* no wall within reach: the new cell is within one cell of the tile,
         * so its key follows from the tile's neighbour strides */
        const int u0 = l[0] + to[0], u1 = l[1] + to[1], u2 = l[2] + to[2];
        const int nt = tl.t + __mul24(u0 >> 2, tl.s0) + __mul24(u1 >> 2, tl.s1) + (u2 >> 2);
        return nt * TILE_CELLS + (((u0 & 3) * TILE + (u1 & 3)) * TILE + (u2 & 3));
    }
    if (!walls(c.pc, k.r, k.u)) return -1;
    return cell_key_of(tv, g, k.r);
}

/* The first segments of a batch (one marker per lane, lanes in cell
 * order): summed over each run of lanes in one cell within each row of 16
 * lanes, then added to LDS by the run's last lane in the row (at most 4
 * atomics per value and run instead of one per marker: LDS atomics to one
 * address serialise).  Called by every lane of the wavefront. */
__device__ static inline void first_run_add(double *lj, First64 &fs)
{
    if (fs.cell < 0)
        for (int q = 0; q < 12; ++q) fs.v[q] = 0.0;
    int start, len;
    bool head;
    wave_run(fs.cell, start, len, head);
    run_sums<12>(fs.v, start);
    if (run_tail(start, len) && fs.cell >= 0) seg_add(lj, fs.cell >> 8, fs.cell >> 4 & 15, fs.cell & 15, fs.v);
}

/* Tiled push: a workgroup of W wavefronts takes work items (a tile's markers
 * in the order, read through its permutation) with stride = grid size,
 * stages the tile's E/H nodes in LDS, accumulates the tile's J in an LDS block
 * and flushes it to HBM once; every marker is written, with its id and new
 * cell key, to the output buffer at its position in the order, and the
 * per-cell counts of the new positions are kept for the next sort.
 *
 * Laser-foil (8.57 M markers) 600 -> 327 us, 3.4 TB/s of the 128 B per marker
 * against 4.8 TB/s of a plain copy; 64^3 full box 469 -> 246 us, 64^3 foil
 * 98 -> 39, 32^3 box 59 -> 39.  The 600 us were gathers from L2 with one batch
 * in flight, 31 IEEE divisions per marker of which 27 had a divisor known
 * before (h, 12, tau h h) and a branch per number of face crossings, each
 * with its own segment code.  Two wavefronts per SIMD (231 VGPRs) measured
 * 339 us, four (116 spilled) 381; the run sums take 24 us of it, the
 * flush 4, the crossing loop 2. */
struct Push64TArgs {
    Markers64    m, d;         /* current buffer (read through tv.perm), output buffer */
    F64View      v;
    Push64Consts c;
    TileView     tv;
    double      *kin;
    unsigned    *err;
};

/* Position min(p, last) of the order: unconditional, so that the loads of a
 * batch are issued on every path (lanes past the end carry a duplicate). */
__device__ static inline unsigned perm_at(const int *perm, unsigned p, unsigned last)
{
    return (unsigned)perm[p < last ? p : last];
}

/* The markers the tile's loop left: pushed straight from and to HBM by the
 * general path, after the loop so that its registers are not the loop's. */
__device__ static inline void push_off_tile(const Push64TArgs &A, const Tile64 &tl, unsigned p,
                                            unsigned end, double w3[3])
{
    if (p >= end) return;
    const TileView &tv = A.tv;
    Pending64 q;
    load_marker(A.m, (unsigned)tv.perm[p], q.k);
    if (q.k.qm == 0.0f) return;
    bool on = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int l = DBL_TO_INT(div_by(q.k.r[a], A.c.pc.h[a], A.c.yh[a], A.c.yl[a])) - tl.c[a];
        on = on && (unsigned)l < TILE;
    }
    if (on) return;
    GlobalSink gs;
    for (int a = 0; a < 3; ++a) gs.J[a] = A.v.J[a];
    gs.g = A.v.g;
    q.p = p;
    q.valid = true;
    q.key = -1;
    if (push_marker(gs, A.v, A.c.pc, q.k.r, q.k.u, q.k.w, q.k.qm, w3, A.err))
        q.key = cell_key_of(tv, A.v.g, q.k.r);
    q.ckey = q.key;
    q.clen = 1;
    write_back(A.d, tv, q);
}

template <int W>
__device__ __forceinline__ static void push64_tiles(const Push64TArgs &A, const VBlock &bk,
                                                    const VBlock &gd)
{
    constexpr int BS = TW * W;                       /* threads of the workgroup */
    constexpr int NSTG = (TFN3 + BS - 1) / BS;       /* staged nodes per thread and component */
    __shared__ double lj[TJB];
    __shared__ double lf[6 * TFN3];
    const TileView &tv = A.tv;
    const F64View &v = A.v;
    const Grid &g = v.g;
    const int nitems = *tv.nitems;
    double w3[3] = {0, 0, 0};
    int4 work = tv.item[bk.x];            /* not behind the load of nitems: the grid is at
                                           * most the item capacity */
    for (int it = (int)bk.x; it < nitems; it += (int)gd.x) {
        if (it != (int)bk.x) work = tv.item[it];
        const unsigned beg = work.y, end = work.z;
        const unsigned s0 = perm_at(tv.perm, beg + threadIdx.x, end - 1);
        unsigned snx = perm_at(tv.perm, beg + BS + threadIdx.x, end - 1);
        Tile64 tl;
        tl.t = work.x;
        int t0, t1, t2;
        tile_coords(tv, tl.t, t0, t1, t2);
        tl.c[0] = TILE * t0;
        tl.c[1] = TILE * t1;
        tl.c[2] = TILE * t2;
        tl.s0 = tv.nt[1] * tv.nt[2];
        tl.s1 = tv.nt[2];
        tl.edge = false;
        for (int a = 0; a < 3; ++a) {
            tl.edge = tl.edge || tl.c[a] < TILE || tl.c[a] + 2 * TILE > g.n[a];
        }
        __syncthreads();                  /* the previous tile's LDS reads are done */
        for (int q = threadIdx.x; q < TJB; q += BS) lj[q] = 0.0;
        Marker64 cur;
        {
            /* nodes [c, c + TFN) per axis; those past the last ghost layer
             * are never read by a gather and are staged as 0 */
            const long base = gidx(g, tl.c[0], tl.c[1], tl.c[2]);
            unsigned offs[NSTG];
            bool ok[NSTG];
#pragma unroll
            for (int r = 0; r < NSTG; ++r) {
                const int rr = (int)threadIdx.x + BS * r;
                const int a = rr / (TFN * TFN), b = (rr / TFN) % TFN, cc = rr % TFN;
                ok[r] = rr < TFN3 && tl.c[0] + a <= g.n[0] + 2 && tl.c[1] + b <= g.n[1] + 2 &&
                        tl.c[2] + cc <= g.n[2] + 2;
                offs[r] = ok[r] ? (unsigned)((a * g.GY + b) * g.GZ + cc) : 0u;
            }
            double st[6][NSTG];
#pragma unroll
            for (int comp = 0; comp < 6; ++comp) {
                const double *F = (comp < 3 ? v.E[comp] : v.H[comp - 3]) + base;
#pragma unroll
                for (int r = 0; r < NSTG; ++r) st[comp][r] = F[offs[r]];
            }
            load_marker(A.m, s0, cur);
#pragma unroll
            for (int comp = 0; comp < 6; ++comp)
#pragma unroll
                for (int r = 0; r < NSTG; ++r) {
                    const int rr = (int)threadIdx.x + BS * r;
                    if (rr < TFN3) lf[comp * TFN3 + rr] = ok[r] ? st[comp][r] : 0.0;
                }
        }
        /* everything outstanding completes here, so that the loop's waits
         * only ever concern the prefetch of the batch in flight */
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        unsigned long long off_tile = 0;  /* lanes that met a marker of another cell */
        Pending64 pend;
        pend.valid = false;
        pend.ckey = -1;
        for (unsigned base = beg; base < end; base += BS) {
            const unsigned p = base + threadIdx.x;
            Marker64 nxt;
            load_marker(A.m, snx, nxt);
            snx = perm_at(tv.perm, p + 2 * BS, end - 1);
            write_back(A.d, tv, pend);
            First64 fs;
            fs.cell = -1;
            pend.k = cur;
            pend.p = p;
            pend.valid = p < end;
            pend.key = -1;
            if (pend.valid && cur.qm != 0.0f)
                pend.key = push64_marker(pend.k, v, A.c, tv, tl, lf, lj, fs, w3);
            const bool off = pend.key == OFF_TILE;
            off_tile |= __ballot(off);
            if (off) {
                pend.key = -1;
                pend.valid = false;
            }
            first_run_add(lj, fs);
            /* count[new key] += run length, once per run of equal new keys */
            int start, len;
            bool head;
            wave_run(pend.key, start, len, head);
            pend.ckey = head ? pend.key : -1;
            pend.clen = len;
            cur = nxt;
        }
        write_back(A.d, tv, pend);
        if (off_tile)
            for (unsigned base = beg; base < end; base += BS)
                push_off_tile(A, tl, base + threadIdx.x, end, w3);
        __syncthreads();
        /* flush the tile's J block: one HBM atomic per non-zero node value */
        for (int q = threadIdx.x; q < TJB; q += BS) {
            const double val = lj[q];
            if (val == 0.0) continue;
            const int comp = q % 3, node = q / 3;
            const int cc = node % TJN, bb = (node / TJN) % TJN, aa = node / (TJN * TJN);
            const int i = tl.c[0] - 1 + aa, j = tl.c[1] - 1 + bb, k = tl.c[2] - 1 + cc;
            if (i < -2 || j < -2 || k < -2 || i > g.n[0] + 2 || j > g.n[1] + 2 || k > g.n[2] + 2)
                continue;
            unsafeAtomicAdd(v.J[comp] + gidx(g, i, j, k), val);
        }
    }
    for (int d = 32; d > 0; d >>= 1)
        for (int a = 0; a < 3; ++a) w3[a] += __shfl_down(w3[a], d, 64);
    if ((threadIdx.x & 63) == 0 && (w3[0] != 0.0 || w3[1] != 0.0 || w3[2] != 0.0)) {
        double *ks = kin_slot(A.kin, bk.x);
        for (int a = 0; a < 3; ++a) atomicAdd(ks + a, w3[a]);
    }
}

/* W wavefronts per workgroup, a distinct argument type per W. */
template <int W> struct Push64TArgsW : Push64TArgs {
};

template <int W> struct KernelDef<Push64TArgsW<W>> {
    static constexpr int kBlock = TW * W;
    static constexpr int kWaves = 3;   /* register budget for 3 wavefronts per SIMD */
    __device__ __forceinline__ static void body(const Push64TArgsW<W> &a, VBlock b, VBlock gd)
    {
        push64_tiles<W>(a, b, gd);
    }
};

int launch_push64_tiled(hipStream_t s, const Markers64 &m, const Markers64 &dst,
                        const Fields64 &f, const Grid &g, const PushConsts &pc,
                        const TileView &tv, double *kin, unsigned *err, int nblocks, int waves)
{
    F64View v;
    for (int a = 0; a < 3; ++a) {
        v.E[a] = f.E[a];
        v.H[a] = f.H[a];
        v.J[a] = f.J[a];
    }
    v.g = g;
    Push64Consts c;
    c.pc = pc;
    for (int a = 0; a < 3; ++a) {
        c.yh[a] = 1.0 / g.h[a];
        c.yl[a] = fma(-g.h[a], c.yh[a], 1.0) / g.h[a];
        c.cj[a] = g.h[a] / g.tau;
    }
    c.vol = g.h[0] * g.h[1] * g.h[2];
    const Push64TArgs a = {m, dst, v, c, tv, kin, err};
    if (waves == 8) return launch_def(s, Push64TArgsW<8>{a}, (unsigned)nblocks);
    return launch_def(s, Push64TArgsW<4>{a}, (unsigned)nblocks);
}

/* CIC charge density of the live markers, source/core/plasma_rho.c:160-173:
 * the order's markers through its permutation (perm non-null: the first
 * nmark[parity] entries), else the first n records. */
__global__ void __launch_bounds__(TPB) k_rho64(Markers64 m, long n, double *rho, Grid g,
                                               const int *perm, const int *nmark, int parity)
{
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long p = q < n && (!perm || q < nmark[parity]) ? (perm ? perm[q] : q) : -1;
    double v[8] = {};
    long cell = -1;
    if (p >= 0 && m.qm[p] != 0.0f) {
        int i, j, k;
        double sx, sy, sz;
        sx = m.x[p] / g.h[0]; i = DBL_TO_INT(sx); sx -= i;
        sy = m.y[p] / g.h[1]; j = DBL_TO_INT(sy); sy -= j;
        sz = m.z[p] / g.h[2]; k = DBL_TO_INT(sz); sz -= k;
        cell = gidx(g, i, j, k);
        cic_weights(sx, sy, sz, m.w[p], v);
    }
    rho_run_add(rho, g, cell, v);
}

int launch_rho64(hipStream_t s, const Markers64 &m, long n, double *rho, const Grid &g,
                 const int *perm, const int *nmark, int parity)
{
    if (n <= 0) return MPIC_OK;
    k_rho64<<<(unsigned)((n + TPB - 1) / TPB), TPB, 0, s>>>(m, n, rho, g, perm, nmark, parity);
    MPIC_CHECK(hipGetLastError());
    return MPIC_OK;
}

/* Linear cell index of floor(x/h) for every marker of the order (through
 * its permutation when perm is non-null; -1 for deleted ones). */
__global__ void k_cells64(Markers64 m, long n, Grid g, const int *perm, const int *nmark,
                          int parity, int32_t *cell)
{
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const long p = perm ? (q < nmark[parity] ? perm[q] : -1) : q;
    if (p < 0 || m.qm[p] == 0.0f) {
        cell[q] = -1;
        return;
    }
    int i = DBL_TO_INT(m.x[p] / g.h[0]), j = DBL_TO_INT(m.y[p] / g.h[1]),
        k = DBL_TO_INT(m.z[p] / g.h[2]);
    cell[q] = (i * g.n[1] + j) * g.n[2] + k;
}

int launch_cells64(hipStream_t s, const Markers64 &m, long n, const Grid &g, const int *perm,
                   const int *nmark, int parity, int32_t *cell)
{
    if (n <= 0) return MPIC_OK;
    k_cells64<<<(unsigned)((n + TPB - 1) / TPB), TPB, 0, s>>>(m, n, g, perm, nmark, parity, cell);
    MPIC_CHECK(hipGetLastError());
    return MPIC_OK;
}
