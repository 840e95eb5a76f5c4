// ffddadi.hip — the DDADI implicit stage (BLKS%LUSGS = 0, IMPS imps3.f:321-373) on the
// device.  Included at the end of ffhip.hip (it uses the context and launch helpers
// defined there).
//
// DDADI replaces the LU-SGS sweeps by three direction-split sweeps, K, I and J, each a
// backward pass PRED (imps4.f:788-905; k-omega PREDKE imps4.f:2084-2229), a pointwise
// diagonal DIAG (imps4.f:911-971; DIAGKE imps4.f:2235-2309) and a forward pass CORR
// (imps4.f:671-787; CORRKE imps4.f:1939-2078).  Each pass is a recurrence along one grid
// line only, so the lines are independent.
// The reference sorts its arrays so that the swept direction runs slowest (SORT38, SORTZZ
// of multi.f: IJK for K, JKI for I, KIJ for J) and loops over the entries of its sorted
// (a, b) plane from entry IN+1 of the first interior row to the end of the last (DO I =
// IN+1, JMAX*ISTRID: ghost entries of the fast index a included, every 2*IN+1-th when the
// fast dimension is 1).  The kernels address the unsorted IJK arrays through the strides of
// that order and take the same plane entries, so every line does the reference's
// operations on the reference's operands.  IDI = all cells viscous (CDIFF = 2), UROT = 0,
// DTURB = 1.

struct DdDir {
    int sa, sb, sm;               // strides of the sorted fast, middle and swept indices
    int na, nb, nm;               // their interior sizes
    const double *A, *AX, *AY, *AZ;   // the face arrays of the swept direction
};

static DdDir dd_dir(const Blk &b, int dir)
{
    DdDir r;
    if (dir == 0) {          // K sweep: IJK
        r.sa = 1; r.na = b.imax; r.sb = b.is; r.nb = b.jmax; r.sm = b.il; r.nm = b.kmax;
        r.A = b.f[FF_A3]; r.AX = b.f[FF_A3X]; r.AY = b.f[FF_A3Y]; r.AZ = b.f[FF_A3Z];
    } else if (dir == 1) {   // I sweep: JKI
        r.sa = b.is; r.na = b.jmax; r.sb = b.il; r.nb = b.kmax; r.sm = 1; r.nm = b.imax;
        r.A = b.f[FF_A1]; r.AX = b.f[FF_A1X]; r.AY = b.f[FF_A1Y]; r.AZ = b.f[FF_A1Z];
    } else {                 // J sweep: KIJ
        r.sa = b.il; r.na = b.kmax; r.sb = 1; r.nb = b.imax; r.sm = b.is; r.nm = b.jmax;
        r.A = b.f[FF_A2]; r.AX = b.f[FF_A2X]; r.AY = b.f[FF_A2Y]; r.AZ = b.f[FF_A2Z];
    }
    return r;
}

// the number of plane entries (lines) of a direction
static int dd_lines(const DdDir &r)
{
    const int ist = r.na + 2 * FF_GHOST, step = r.na == 1 ? 2 * FF_GHOST + 1 : 1;
    return (r.nb * ist - FF_GHOST + step - 1) / step;
}

// SYIKE imps4.f:982-1035 (its DRH and DRP are formed but unused there)
__device__ __forceinline__ void syike(double w[7], const double x[7], double c, double ro,
                                      double a2x, double a2y, double a2z, double &a21,
                                      double &a22, double &a23, double &a31, double &a32,
                                      double &a33)
{
    const double z1 = x[0], z5 = x[4], z6 = x[5], z7 = x[6];
    surfvects(a2x, a2y, a2z, a21, a22, a23, a31, a32, a33);
    const double z2 = a2x * x[1] + a2y * x[2] + a2z * x[3];
    const double z3 = a21 * x[1] + a22 * x[2] + a23 * x[3];
    const double z4 = a31 * x[1] + a32 * x[2] + a33 * x[3];
    const double roc = ro * c;
    const double pc2 = 1. / ro;
    const double dpres = z5;
    w[0] = z1 - pc2 * dpres;
    w[1] = roc * z2 + dpres;
    w[2] = z3;
    w[3] = z4;
    w[5] = z6;
    w[6] = z7;
    w[4] = -roc * z2 + dpres;
}

// SYM1KE imps4.f:1041-1072
__device__ __forceinline__ void sym1ke(double x[7], const double w[7], double rk, double c,
                                       double ro, double drdp, double drdh, double a2x,
                                       double a2y, double a2z, double a21, double a22,
                                       double a23, double a31, double a32, double a33)
{
    const double ypro = 1. / ro;
    const double pc2 = .5 * ypro;
    const double proc = pc2 / c;
    const double drh = .667 * rk * (ypro * ypro) * drdh;
    const double ydrp = 1. / (1. + .667 * rk * ypro * drdp);
    const double dh = w[0] + pc2 * (w[1] + w[4]);
    x[0] = dh;
    const double x2i = proc * (w[1] - w[4]);
    const double x3i = w[2], x4i = w[3];
    const double x5 = .5 * (w[1] + w[4]);
    x[4] = ydrp * (x5 - drh * ro * dh - .667 * ro * w[5]);
    x[5] = w[5];
    x[6] = w[6];
    x[1] = a2x * x2i + a21 * x3i + a31 * x4i;
    x[2] = a2y * x2i + a22 * x3i + a32 * x4i;
    x[3] = a2z * x2i + a23 * x3i + a33 * x4i;
}

// The sweep's line t, as the flat offset of its cell m = 1 minus one step: the reference's
// plane entry f = IN + t*step on the K and I sweeps (consecutive lines are neighbouring I
// columns on the K sweep, rows on the I sweep); on the J sweep the entries are renumbered with the middle index b (= I)
// fastest so that consecutive lines again take neighbouring I columns.  The set of
// entries is the reference's: f = a + b*(NA+4) >= IN, every 2*IN+1-th with NA = 1.  a0: the
// line's fast index.
__device__ __forceinline__ bool dd_line(const DdDir &r, int dir, int t, int &base, int &a0)
{
    const int ist = r.na + 2 * FF_GHOST;
    int b0;
    if (dir == 2) {
        b0 = t % r.nb;
        a0 = t / r.nb;
        if (a0 >= ist || (b0 == 0 && a0 < FF_GHOST) || (r.na == 1 && a0 != FF_GHOST)) return false;
    } else {
        const int step = r.na == 1 ? 2 * FF_GHOST + 1 : 1;
        const int f = FF_GHOST + t * step;
        if (f >= r.nb * ist) return false;
        a0 = f % ist;
        b0 = f / ist;
    }
    base = a0 * r.sa + (b0 + FF_GHOST) * r.sb + (FF_GHOST - 1) * r.sm;
    return true;
}

// line numbers of a sweep launch
static int dd_threads(const DdDir &r, int dir)
{
    return dir == 2 ? (r.na + 2 * FF_GHOST) * r.nb : dd_lines(r);
}

// What a PRED (FWD = false) or CORR (FWD = true) step reads of its cell: the neighbour nn
// across the face whose viscous term T and diagonal it forms (the lower neighbour in PRED,
// the upper one in CORR), the area of the face the carried flux crosses (PRED: the upper
// face, CORR: the lower face) and of the diagonal's face, and the normal of the face whose
// characteristic variables it uses (PRED: the lower face, CORR: the upper face).
struct DdIn {
    double dt1, vol, voln, u, v, w, c, ro, ron, vis, vist, visn, vistn;
    double aflux, adiag, fx, fy, fz, lx, ly, lz;   // l: the other face's normal (DIAG)
    double d[7], rk, drdp, drdh;
};

template <bool KE, bool FWD>
__device__ __forceinline__ void dd_load(const Prm &p, const Blk &b, const DdDir &r, int n, DdIn &x)
{
    const int nu = n + r.sm, nn = FWD ? nu : n - r.sm, nf = FWD ? nu : n;
    x.dt1 = p.theta * FLD(b, FF_DTL)[n];
    x.vol = FLD(b, FF_VOL)[n];
    x.voln = FLD(b, FF_VOL)[nn];
    x.u = FLD(b, FF_U)[n];
    x.v = FLD(b, FF_V)[n];
    x.w = FLD(b, FF_W)[n];
    x.c = FLD(b, FF_C)[n];
    x.ro = FLD(b, FF_RO)[n];
    x.ron = FLD(b, FF_RO)[nn];
    x.vis = FLD(b, FF_VIS)[n];
    x.vist = FLD(b, FF_VIST)[n];
    x.visn = FLD(b, FF_VIS)[nn];
    x.vistn = FLD(b, FF_VIST)[nn];
    x.aflux = FWD ? r.A[n] : r.A[nu];
    x.adiag = FWD ? r.A[nu] : r.A[n];
    x.fx = r.AX[nf];
    x.fy = r.AY[nf];
    x.fz = r.AZ[nf];
    if (FWD) {
        x.lx = r.AX[n];
        x.ly = r.AY[n];
        x.lz = r.AZ[n];
    }
#pragma unroll
    for (int q = 0; q < (KE ? 7 : 5); q++) x.d[q] = FLD(b, FF_DRO + q)[n];
    if (KE) {
        x.rk = FLD(b, FF_RK)[n];
        x.drdp = FLD(b, FF_DRDP)[n];
        x.drdh = FLD(b, FF_DRDH)[n];
    }
}

// DIAG (DIAGKE) of a cell, on the operands CORR reads of it
template <bool KE>
__device__ __forceinline__ void dd_diag(const DdIn &x, double d[7])
{
    const double dturb = 1.;
    double y[7], a21, a22, a23, a31, a32, a33;
    if (KE)
        syike(y, x.d, x.c, x.ro, x.fx, x.fy, x.fz, a21, a22, a23, a31, a32, a33);
    else
        syi(y[0], y[1], y[2], y[3], y[4], x.d[0], x.d[1], x.d[2], x.d[3], x.d[4], x.c, x.ro, x.fx, x.fy,
            x.fz, a21, a22, a23, a31, a32, a33);
    double ucon = x.fx * x.u + x.fy * x.v + x.fz * x.w - 0.;
    const double rl2n = dmax(-(ucon + x.c), 0.), rl5n = dmax(-(ucon - x.c), 0.);
    const double rl1n = dmax(-ucon, 0.);
    ucon = x.lx * x.u + x.ly * x.v + x.lz * x.w - 0.;
    const double rl2p = dmax(ucon + x.c, 0.), rl5p = dmax(ucon - x.c, 0.);
    const double rl1p = dmax(ucon, 0.);
    const double dt = KE ? x.dt1 / (x.vol + 1.E-21) : x.dt1 / x.vol;
    const double s1 = x.aflux * rl1p + x.adiag * rl1n, s2 = x.aflux * rl2p + x.adiag * rl2n;
    const double s5 = x.aflux * rl5p + x.adiag * rl5n;
    y[0] = y[0] * (1. + dt * s1);
    y[1] = y[1] * (1. + dt * s2);
    y[2] = y[2] * (1. + dt * s1);
    y[3] = y[3] * (1. + dt * s1);
    y[4] = y[4] * (1. + dt * s5);
    if (KE) {
        y[5] = y[5] * (1. + dturb * dt * (s1 + 0.));
        y[6] = y[6] * (1. + dturb * dt * (s1 + 0.));
        sym1ke(d, y, x.rk, x.c, x.ro, x.drdp, x.drdh, x.fx, x.fy, x.fz, a21, a22, a23, a31, a32, a33);
    } else {
        sym1i(d[0], d[1], d[2], d[3], d[4], y[0], y[1], y[2], y[3], y[4], x.c, x.ro, x.fx, x.fy, x.fz,
              a21, a22, a23, a31, a32, a33);
    }
}

// The recurrence of a line needs of each cell only values that do not depend on it (VOL*D,
// DT1*A, the face's basis, the scalars of SYI and SYM1I, the denominators, the eigenvalues):
// a record of them per cell, in LDS.  VD holds the quotients Y after the march.
template <bool KE>
struct DdRec {
    static constexpr int NV = KE ? 7 : 5, ND = KE ? 4 : 3;   // ND: denominators X1, X2, X5 (, K)
    static constexpr int VD = 0, M = NV, N = M + 1, T1 = N + 3, T2 = T1 + 3, ROC = T2 + 3, YP = ROC + 1,
                         PROC = YP + 1, SC = PROC + 1,       // KE: YDRP, DRH*RO, .667*RO; else RO
                         DEN = SC + (KE ? 3 : 1), REC = DEN + ND, X = REC + ND, NF = X + 3;
    static_assert(NF % 2 == 0, "the record is read in pairs");
};

// Lines and steps of a line per LDS buffer, and the waves that fill it
constexpr int DD_L = 32, DD_CH = 8, DD_PW = DD_L * DD_CH / 64;

// doubles of a step's records: pairs of fields, [pair][line][2], and 32 bytes so that the steps of
// one line (the I sweep's waves hold 8 of each line) fall in different banks
template <bool KE>
constexpr int dd_slot() { return DdRec<KE>::NF * DD_L + 4; }

typedef double dd2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ dd2 *dd_pair(double *rec, int q) { return (dd2 *)(rec + q * 2 * DD_L); }

// |x| in 2^-460 .. 2^460: the exponent's distance from the lower end (large for zero, infinity
// and NaN too)
__device__ __forceinline__ unsigned dd_mag(double x)
{
    return ((unsigned)((unsigned long long)__double_as_longlong(x) >> 32) << 1) - (563u << 21);
}
constexpr unsigned DD_MAG = 920u << 21;

// y/d, correctly rounded, from r = 1/d correctly rounded: two corrections of y*r with exact
// remainders (Markstein, IBM J. Res. Dev. 34, 1990).  Holds for d and the quotient in
// dd_mag's range, where no remainder underflows; the caller divides otherwise.  Five operations for
// a division's fifteen, on the march's chain.
__device__ __forceinline__ double dd_quot(double y, double d, double r)
{
    double q = y * r;
    q = fma(fma(-q, d, y), r, q);
    return fma(fma(-q, d, y), r, q);
}

// a denominator and its reciprocal, NaN where dd_quot does not hold
__device__ __forceinline__ double dd_recip(double d)
{
    return dd_mag(d) < DD_MAG ? 1. / d : __longlong_as_double(0x7ff8000000000000LL);
}

// SYM1I / SYM1KE with a record's values
template <bool KE>
__device__ __forceinline__ void dd_sym1(const double *f, const double *w, double *x)
{
    using R = DdRec<KE>;
    const double pc2 = .5 * f[R::YP];
    x[0] = w[0] + pc2 * (w[1] + w[4]);
    const double x2i = f[R::PROC] * (w[1] - w[4]);
    double x5 = .5 * (w[1] + w[4]);
    if (KE) {
        x5 = f[R::SC] * (x5 - f[R::SC + 1] * x[0] - f[R::SC + 2] * w[5]);
        x[5] = w[5];
        x[6] = w[6];
    }
    x[4] = x5;
#pragma unroll
    for (int q = 0; q < 3; q++) x[1 + q] = f[R::N + q] * x2i + f[R::T1 + q] * w[2] + f[R::T2 + q] * w[3];
}

// the record of a cell (m: its place on the line) to LDS
template <bool KE, bool FWD>
__device__ __forceinline__ void dd_record(const DdIn &x, int m, double *rec)
{
    using R = DdRec<KE>;
    const double cdiff = 2., dturb = 1., vrel = 1.E-21;
    double f[R::NF], d[7];
    if (FWD) {
        dd_diag<KE>(x, d);
    } else {
#pragma unroll
        for (int q = 0; q < R::NV; q++) d[q] = x.d[q];
    }
#pragma unroll
    for (int q = 0; q < R::NV; q++) f[R::VD + q] = x.vol * d[q];
    f[R::M] = x.dt1 * x.aflux;
    f[R::N] = x.fx; f[R::N + 1] = x.fy; f[R::N + 2] = x.fz;
    surfvects(x.fx, x.fy, x.fz, f[R::T1], f[R::T1 + 1], f[R::T1 + 2], f[R::T2], f[R::T2 + 1], f[R::T2 + 2]);
    const double ypro = 1. / x.ro, pc2 = .5 * ypro;
    f[R::ROC] = x.ro * x.c;
    f[R::YP] = ypro;
    f[R::PROC] = pc2 / x.c;
    const double rl1 = x.fx * x.u + x.fy * x.v + x.fz * x.w - 0.;
    const double rl2 = rl1 + x.c, rl5 = rl1 - x.c;
    const double ff = FWD ? .5 : (m == 1 ? .25 : .5);
    const double rnum = ff * (x.vol + x.voln) * (x.ro + x.ron);
    const double tt = cdiff * x.adiag / rnum * (x.vist + x.vis + x.vistn + x.visn);
    if (FWD) {
        f[R::X] = dmax(rl1, 0.) + tt; f[R::X + 1] = dmax(rl2, 0.) + tt; f[R::X + 2] = dmax(rl5, 0.) + tt;
    } else {
        f[R::X] = dmax(-rl1, 0.) + tt; f[R::X + 1] = dmax(-rl2, 0.) + tt; f[R::X + 2] = dmax(-rl5, 0.) + tt;
    }
    const double xa[3] = {fabs(rl1) + tt, fabs(rl2) + tt, fabs(rl5) + tt};
    if (KE) {
        const double drh = .667 * x.rk * (ypro * ypro) * x.drdh;
        f[R::SC] = 1. / (1. + .667 * x.rk * ypro * x.drdp);
        f[R::SC + 1] = drh * x.ro;
        f[R::SC + 2] = .667 * x.ro;
#pragma unroll
        for (int q = 0; q < 3; q++) f[R::DEN + q] = x.vol + vrel + x.dt1 * xa[q] * x.adiag;
        f[R::DEN + R::ND - 1] = x.vol + vrel + dturb * x.dt1 * (xa[0] * x.adiag + 0.);
    } else {
        f[R::SC] = x.ro;
#pragma unroll
        for (int q = 0; q < 3; q++) f[R::DEN + q] = x.vol + x.dt1 * xa[q] * x.adiag;
    }
#pragma unroll
    for (int q = 0; q < R::ND; q++) f[R::REC + q] = dd_recip(f[R::DEN + q]);
#pragma unroll
    for (int q = 0; q < R::NF / 2; q++) *dd_pair(rec, q) = dd2{f[2 * q], f[2 * q + 1]};
}

// PRED (FWD = false: backward along the line) or DIAG and CORR (FWD = true: forward) along
// every line of one direction; last: the end of IMPS on the interior cells as well, dh -> dT
// (DIVV12 imps3.f:483) and, with the k-omega model, D(rho k), D(rho omega) times RO (MULV12
// imps3.f:497-500).
//
// A line is a serial chain, and there are too few lines to fill the chip (96x72x50: 59 waves
// on the I sweep), so what counts is the time of one step.  Wave 0 of a workgroup marches 32
// lines from records in LDS: SYI, the quotients, the flux to the next cell, nothing else.
// The other four waves work a buffer of 8 steps ahead and one behind: they load the cells,
// form the records (two thirds of the arithmetic, with the square root and all divisions but
// the quotients') and, from the quotients the march left, the cells' increments.  On the I
// sweep a wave takes 8 steps of 8 lines, so that a load touches 8 runs of 64 bytes instead of
// 64 cache lines.  k-omega, 96x72x50: PRED 37 to 64 us, DIAG and CORR 37 to 64; with one thread
// per line doing all of it (and DIAG a pass of its own) the six sweeps took 910 us, 290 each on
// the I sweep, and the stage 1335 us against 538.
template <bool KE, bool FWD>
__global__ void __launch_bounds__((1 + DD_PW) * 64) k_ddadi_sweep(Prm p, Blk b, DdDir r, int dir, int nlines,
                                                                   int last)
{
    using R = DdRec<KE>;
    __shared__ __align__(16) double buf[2][DD_CH * dd_slot<KE>()];
    const int lane = threadIdx.x & 63, wv = threadIdx.x / 64;
    const int nch = (r.nm + DD_CH - 1) / DD_CH;
    if (wv == 0) {
        __builtin_amdgcn_s_setprio(3);
        int base, a0;
        const int t = blockIdx.x * DD_L + lane;
        const bool on = lane < DD_L && t < nlines && dd_line(r, dir, t, base, a0);
        double bd[7] = {0., 0., 0., 0., 0., 0., 0.};
        lds_step_barrier();
        for (int c = 0; c < nch; c++) {
            if (on) {
                double *const rec = buf[c & 1] + lane * 2;
                const int cnt = min(DD_CH, r.nm - c * DD_CH);
                double f[2][R::NF];
                auto read = [&](int s, double *g) {
#pragma unroll
                    for (int q = 0; q < R::NF / 2; q++) {
                        const dd2 v = *dd_pair(rec + s * dd_slot<KE>(), q);
                        g[2 * q] = v.x;
                        g[2 * q + 1] = v.y;
                    }
                };
                read(0, f[0]);
#pragma unroll
                for (int s = 0; s < DD_CH; s++) {
                    if (s >= cnt) break;
                    const double *g = f[s & 1];
                    // (past the last step of a line: a slot of the same buffer, not used)
                    if (s + 1 < DD_CH) read(s + 1, f[(s + 1) & 1]);
                    double x[7], y[7], z[7];
#pragma unroll
                    for (int q = 0; q < R::NV; q++) x[q] = g[R::M] * bd[q] + g[R::VD + q];
                    const double z2 = g[R::N] * x[1] + g[R::N + 1] * x[2] + g[R::N + 2] * x[3];
                    z[2] = g[R::T1] * x[1] + g[R::T1 + 1] * x[2] + g[R::T1 + 2] * x[3];
                    z[3] = g[R::T2] * x[1] + g[R::T2 + 1] * x[2] + g[R::T2 + 2] * x[3];
                    z[1] = g[R::ROC] * z2 + x[4];
                    z[4] = -g[R::ROC] * z2 + x[4];
                    if (KE) {
                        z[0] = x[0] - g[R::YP] * x[4];
                        z[5] = x[5];
                        z[6] = x[6];
                    } else {
                        double v = dd_quot(x[4], g[R::SC], g[R::YP]);
                        if (max(dd_mag(v), dd_mag(g[R::SC])) >= DD_MAG) v = x[4] / g[R::SC];
                        z[0] = x[0] - v;
                    }
                    constexpr int dn[7] = {0, 1, 0, 0, 2, R::ND - 1, R::ND - 1};
                    unsigned mag = 0;
#pragma unroll
                    for (int q = 0; q < R::NV; q++) {
                        y[q] = dd_quot(z[q], g[R::DEN + dn[q]], g[R::REC + dn[q]]);
                        mag = max(mag, dd_mag(y[q]));
                    }
                    if (mag >= DD_MAG) {
#pragma unroll
                        for (int q = 0; q < R::NV; q++) y[q] = z[q] / g[R::DEN + dn[q]];
                    }
                    double *const o = rec + s * dd_slot<KE>();
                    *dd_pair(o, 0) = dd2{y[0], y[1]};
                    *dd_pair(o, 1) = dd2{y[2], y[3]};
                    if (KE) {
                        *dd_pair(o, 2) = dd2{y[4], y[5]};
                        *(double *)dd_pair(o, 3) = y[6];
                    } else {
                        *(double *)dd_pair(o, 2) = y[4];
                    }
                    // the flux handed to the next cell of the line
                    constexpr int xs[7] = {0, 1, 0, 0, 2, 0, 0};
#pragma unroll
                    for (int q = 0; q < R::NV; q++) y[q] = g[R::X + xs[q]] * y[q];
                    dd_sym1<KE>(g, y, bd);
                }
            }
            lds_step_barrier();
        }
        return;
    }
    // this lane's line and its step within each buffer
    const int w = wv - 1;
    const int ln = dir == 1 ? w * (64 / DD_CH) + lane / DD_CH : lane % DD_L;
    const int st = dir == 1 ? lane % DD_CH : w * (64 / DD_L) + lane / DD_L;
    int base = 0, a0 = 0;
    const int t = blockIdx.x * DD_L + ln;
    const bool on = t < nlines && dd_line(r, dir, t, base, a0);
    double *const rec = buf[0] + st * dd_slot<KE>() + ln * 2;
    constexpr int BUF = DD_CH * dd_slot<KE>();
    double *D[7] = {FLD(b, FF_DRO), FLD(b, FF_DM), FLD(b, FF_DN), FLD(b, FF_DW), FLD(b, FF_DE),
                    FLD(b, FF_DRK), FLD(b, FF_DEPS)};
    auto cell = [&](int c, int &m) {
        const int s = c * DD_CH + st;
        m = FWD ? s + 1 : r.nm - s;
        return on && c < nch && s < r.nm;
    };
    DdIn in;
    int m;
    auto fetch = [&](int c) {
        if (cell(c, m)) dd_load<KE, FWD>(p, b, r, base + m * r.sm, in);
    };
    auto fill = [&](int c) {
        if (cell(c, m)) dd_record<KE, FWD>(in, m, rec + (c & 1) * BUF);
    };
    auto finish = [&](int c) {
        if (!cell(c, m)) return;
        const int n = base + m * r.sm;
        double f[R::NF], o[7];
#pragma unroll
        for (int q = 0; q < (R::DEN + 1) / 2; q++) {
            const dd2 v = *dd_pair(rec + (c & 1) * BUF, q);
            f[2 * q] = v.x;
            f[2 * q + 1] = v.y;
        }
        dd_sym1<KE>(f, f + R::VD, o);
        if (FWD && last && a0 >= FF_GHOST && a0 < FF_GHOST + r.na) {
            o[0] = o[0] / FLD(b, FF_CP)[n];
            if (KE) {
                o[5] = o[5] * FLD(b, FF_RO)[n];
                o[6] = o[6] * FLD(b, FF_RO)[n];
            }
        }
#pragma unroll
        for (int q = 0; q < R::NV; q++) D[q][n] = o[q];
    };
    fetch(0);
    fill(0);
    fetch(1);
    lds_step_barrier();
    for (int c = 0; c < nch; c++) {
        if (c > 0) finish(c - 1);
        fill(c + 1);
        fetch(c + 2);
        lds_step_barrier();
    }
    finish(nch - 1);
}

// the three DDADI directions in IMPS's order, K, I, J, each PRED, then DIAG and CORR; the
// last with the end of IMPS
static int ddadi_impl(ff_ctx *c, const Prm &kp, const Blk &b)
{
    const bool ke = c->prm.iturb == 6;
    auto pred = ke ? k_ddadi_sweep<true, false> : k_ddadi_sweep<false, false>;
    auto corr = ke ? k_ddadi_sweep<true, true> : k_ddadi_sweep<false, true>;
    for (int dir = 0; dir < 3; dir++) {
        const DdDir r = dd_dir(b, dir);
        const int nt = dd_threads(r, dir);
        const dim3 g((unsigned)((nt + DD_L - 1) / DD_L)), t((1 + DD_PW) * 64);
        int rc;
        if ((rc = launch(c, "k_ddadi", pred, g, t, kp, b, r, dir, nt, 0)) ||
            (rc = launch(c, "k_ddadi", corr, g, t, kp, b, r, dir, nt, dir == 2 ? 1 : 0)))
            return rc;
    }
    return FF_OK;
}
