// dcm_mpdata64.hip -- the FP64 MPDATA passes of mpdata_3d / mpdata_vec_3d
// (pamm/sfvt/advection_3d.F90:219-714, 1250-1753) as i-marching kernels: the
// first donor pass, the density-weighted antidiffusive velocities, the
// limiter factors and the limited donor pass.
//
// The arithmetic is that of the one-cell-per-thread kernels of
// dcm_advect.hip, expression by expression, so the results are the same bit
// for bit.  Those are bound by the issue of correctly rounded divisions (34 a
// cell in the antidiffusive pass, 6 to 8 in the others) and by one load per
// stencil neighbour (37 and 20 a cell).  Here
//   - a thread owns one (k,j) column and marches kPlanes planes: the values of
//     planes i-1, i, i+1 stay in registers (21 loads instead of 37), the next
//     plane's are in flight while a plane is computed;
//   - every denominator made of metrics is a constant of the thread (the
//     grid is uniform along x, a rule of the launch), so its quotients come
//     from its reciprocal, formed once per thread, by Markstein's theorem: 5
//     operations instead of 14.  The theorem's range is watched once per
//     cell: the exponents of the numerators are collected, and a cell with a
//     numerator below 2^-900 (zero apart) or a result that is not finite is
//     evaluated again with divisions.
// Measured at 256x256x128, per-cell kernel against marching: first donor pass
// 99 -> 84 us, antidiffusive velocities 304 -> 209, limiter factors 177 ->
// 141, limited pass 208 -> 159 (335, 470, 470 and 470 MB of compulsory
// traffic: 67, 94, 94 and 94 us at the card's copy rate).
#include <cmath>

#include "dcm_device.h"

namespace dcm {

namespace {

constexpr double kSmall = 1e-60;  // advection_3d.F90:19
constexpr int kMinExp = -900;

// a metric denominator and its reciprocal
struct Den {
    double b, y;
    __device__ __forceinline__ explicit Den(double v) : b(v), y(1.0 / v) {}
};
// quotients by metric denominators: IEEE divisions, or by the reciprocal with
// the smallest numerator exponent collected
struct Exact {
    __device__ __forceinline__ double operator()(double x, const Den &d) { return x / d.b; }
    __device__ __forceinline__ bool ok(double) const { return true; }
};
struct Fast {
    int e = 0;
    __device__ __forceinline__ double operator()(double x, const Den &d) {
        const int xe = __builtin_amdgcn_frexp_exp(x);  // 0 for 0, inf, NaN
        e = xe < e ? xe : e;
        const double q0 = x * d.y;
        const double q1 = __builtin_fma(__builtin_fma(-d.b, q0, x), d.y, q0);
        return __builtin_fma(__builtin_fma(-d.b, q1, x), d.y, q1);
    }
    // an infinite or NaN quotient makes every result below one
    __device__ __forceinline__ bool ok(double r) const { return e > kMinExp && isfinite(r); }
};

__device__ __forceinline__ double pos(double x) { return x > 0.0 ? x : 0.0; }
__device__ __forceinline__ double neg(double x) { return x < 0.0 ? x : 0.0; }
__device__ __forceinline__ double least3(double a, double b, double c) {
    double m = a;
    if (b < m) m = b;
    if (c < m) m = c;
    return m;
}

// element e of an array: a uniform base and a 32-bit byte offset
__device__ __forceinline__ double ld(const double *p, unsigned e) {
    return *(const double *)((const char *)p + e * 8u);
}
__device__ __forceinline__ void st(double *p, unsigned e, double v) {
    *(double *)((char *)p + e * 8u) = v;
}

// the thread's column and planes
struct Col {
    int k, j, i0, i1;
    unsigned c, SI, SJ;  // element of plane i0; strides
    bool act;
};
__device__ __forceinline__ Col column(const Geo &g, int planes) {
    Col q;
    q.k = blockIdx.x * blockDim.x + threadIdx.x + 1;
    q.j = blockIdx.y * blockDim.y + threadIdx.y + 1;
    q.i0 = blockIdx.z * planes + 1;
    q.i1 = min(q.i0 + planes - 1, g.ip);
    q.act = q.k <= g.kp && q.j <= g.jp;
    q.SI = (unsigned)g.si;
    q.SJ = (unsigned)g.sj;
    q.c = (unsigned)q.i0 * q.SI + (unsigned)q.j * q.SJ + (unsigned)q.k;
    return q;
}

// first_order_upstream_3d for one cell (:74-115)
struct DonorDen {
    Den x, y, z;  // 2 dxn, 2 dyn, (2 dzn) rhoan
    double ra, ram;
};
template <typename Q>
__device__ __forceinline__ double donor_cell(Q &q, const DonorDen &D, double dt, double uc,
                                             double ul, double vc, double vl, double wc,
                                             double wl, double pc, double pe, double pw,
                                             double pn, double ps, double pu, double pd, int k,
                                             int kp, int neumann) {
    const double fxr = q(((uc + fabs(uc)) * pc + (uc - fabs(uc)) * pe) * dt, D.x);
    const double fxl = q(((ul + fabs(ul)) * pw + (ul - fabs(ul)) * pc) * dt, D.x);
    const double fyr = q(((vc + fabs(vc)) * pc + (vc - fabs(vc)) * pn) * dt, D.y);
    const double fyl = q(((vl + fabs(vl)) * ps + (vl - fabs(vl)) * pc) * dt, D.y);
    double fzr = q((((wc + fabs(wc)) * D.ra) * pc + ((wc - fabs(wc)) * D.ra) * pu) * dt, D.z);
    double fzl = q((((wl + fabs(wl)) * D.ram) * pd + ((wl - fabs(wl)) * D.ram) * pc) * dt, D.z);
    if (neumann == 1) {  // :95-101
        if (k == 1) fzl = fzr;
        if (k == kp) fzr = fzl;
    } else if (neumann == 2) {  // :102-110
        if (k == 1) fzl = -fzr;
        if (k == kp) fzr = -fzl;
    }
    return ((pc - (fxr - fxl)) - (fyr - fyl)) - (fzr - fzl);
}

// The first donor pass on psi - m (k_upwind_first).  HBM: psi, u, v, w read,
// the result written (4.0 TB/s of those).
__global__ __launch_bounds__(256) void k64_donor1(const double *__restrict__ psi,
                                                  const double *__restrict__ mptr,
                                                  const double *__restrict__ u,
                                                  const double *__restrict__ v,
                                                  const double *__restrict__ w,
                                                  double *__restrict__ out, Geo g, Metrics M,
                                                  double dt, int neumann, int planes) {
    const Col q = column(g, planes);
    if (!q.act) return;
    const int k = q.k, j = q.j;
    const double m = *mptr;
    const DonorDen D{Den(2.0 * M.dxn[1]), Den(2.0 * M.dyn[j]), Den((2.0 * M.dzn[k]) * M.rhoan[k]),
                     M.rhoa[k], M.rhoa[k - 1]};
    unsigned c = q.c;
    struct Plane {
        double pc, pn, ps, pu, pd, uc, vc, vl, wc, wl;
    };
    auto load = [&](unsigned c) {
        return Plane{ld(psi, c),       ld(psi, c + q.SJ), ld(psi, c - q.SJ), ld(psi, c + 1),
                     ld(psi, c - 1),   ld(u, c),          ld(v, c),          ld(v, c - q.SJ),
                     ld(w, c),         ld(w, c - 1)};
    };
    double pw = ld(psi, c - q.SI) - m, ul = ld(u, c - q.SI);
    Plane P = load(c);
    for (int i = q.i0; i <= q.i1; ++i, c += q.SI) {
        const Plane N = load(c + q.SI);  // plane i+1 <= ip+1: inside the padded array
        const double pc = P.pc - m, pe = N.pc - m;
        auto cell = [&](auto Q) {
            const double r = donor_cell(Q, D, dt, P.uc, ul, P.vc, P.vl, P.wc, P.wl, pc, pe, pw,
                                        P.pn - m, P.ps - m, P.pu - m, P.pd - m, k, g.kp, neumann);
            st(out, c, r);
            return Q.ok(r);
        };
        if (__builtin_expect(!cell(Fast{}), 0)) cell(Exact{});
        pw = pc;
        ul = P.uc;
        P = N;
    }
}

// The antidiffusive velocities (k_antidiff<double, true>, :318-506).
// HBM: u, v, w and the field read, three velocities written; bound by FP64
// issue (25 quotients by reciprocals, 9 divisions by data a cell: about 140
// us of issue at full rate) at two waves a SIMD (240 VGPRs).
struct AntiDen {
    Den zg1, yg1, xg1, xg3, yg3, zg3;  // d{z,y,x}(-1) * g
    Den g1, g3, hx, hy, hz, dxn, dyn, dzn, xm, ym;
    double rn, rnp, ra, ram, rap, dx, dy, dz, rag3;
};
__global__ __launch_bounds__(256) void k64_antidiff(const double *__restrict__ ut,
                                                    const double *__restrict__ vt,
                                                    const double *__restrict__ wt,
                                                    const double *__restrict__ po,
                                                    double *__restrict__ us,
                                                    double *__restrict__ vs,
                                                    double *__restrict__ ws,
                                                    const int *__restrict__ flag, Geo g,
                                                    Metrics M, double dt, int planes) {
    if (*flag) return;
    const Col q = column(g, planes);
    if (!q.act) return;
    const int k = q.k, j = q.j;
    const unsigned SI = q.SI, SJ = q.SJ;
    const double rn = M.rhoan[k], rnp = M.rhoan[k + 1], g3 = 0.5 * (rn + rnp);
    const double dxm = M.dx[0], dym = M.dy[j - 1], dzm = M.dz[k - 1];
    const AntiDen D{Den(dzm * rn), Den(dym * rn), Den(dxm * rn), Den(dxm * g3), Den(dym * g3),
                    Den(dzm * g3), Den(rn), Den(g3), Den(0.5 * (M.dxn[0] + M.dxn[1])),
                    Den(0.5 * (M.dyn[j - 1] + M.dyn[j])), Den(0.5 * (M.dzn[k - 1] + M.dzn[k])),
                    Den(M.dxn[1]), Den(M.dyn[j]), Den(M.dzn[k]), Den(dxm), Den(dym),
                    rn, rnp, M.rhoa[k], M.rhoa[k - 1], M.rhoa[k + 1], M.dx[1], M.dy[j], M.dz[k],
                    M.rhoa[k] / g3};
    // values of one plane: suffixes n, s: j+1, j-1; u, d: k+1, k-1
    struct UP { double c, n, u; };
    struct VP { double c, s, n, u, us; };
    struct WP { double c, d, n, dn, u; };
    struct PP { double c, n, s, u, d, un, dn, us; };
    auto lu = [&](unsigned c) { return UP{ld(ut, c), ld(ut, c + SJ), ld(ut, c + 1)}; };
    auto lv = [&](unsigned c) {
        return VP{ld(vt, c), ld(vt, c - SJ), ld(vt, c + SJ), ld(vt, c + 1), ld(vt, c + 1 - SJ)};
    };
    auto lw = [&](unsigned c) {
        return WP{ld(wt, c), ld(wt, c - 1), ld(wt, c + SJ), ld(wt, c - 1 + SJ), ld(wt, c + 1)};
    };
    auto lp = [&](unsigned c) {
        return PP{ld(po, c),     ld(po, c + SJ),     ld(po, c - SJ),     ld(po, c + 1),
                  ld(po, c - 1), ld(po, c + 1 + SJ), ld(po, c - 1 + SJ), ld(po, c + 1 - SJ)};
    };
    unsigned c = q.c;
    UP Um = lu(c - SI), U = lu(c);
    VP V = lv(c);
    WP W = lw(c);
    PP P = lp(c);
    double Pw = ld(po, c - SI), Pwn = ld(po, c - SI + SJ), Pwu = ld(po, c - SI + 1);
    for (int i = q.i0; i <= q.i1; ++i, c += SI) {
        // plane i+1 <= ip+1: inside the padded arrays
        const UP Ue = lu(c + SI);
        const VP Ve = lv(c + SI);
        const WP We = lw(c + SI);
        const PP Pe = lp(c + SI);
        auto cell = [&](auto Q) {
            const double h = 0.5, qq = 0.25;
            const double d1 = Q(D.ra * (W.c + We.c) - D.ram * (W.d + We.d), D.zg1) +
                              Q(rn * (((V.c + Ve.c) - V.s) - Ve.s), D.yg1);
            const double d2 = Q(D.ra * (W.c + W.n) - D.ram * (W.d + W.dn), D.zg1) +
                              Q(rn * (((U.c + U.n) - Um.c) - Um.n), D.xg1);
            const double d3 = Q(rn * (U.c - Um.c) + rnp * (U.u - Um.u), D.xg3) +
                              Q(rn * (V.c - V.s) + rnp * (V.u - V.us), D.yg3);
            const double tz1 =
                Q((Q(qq * (((D.ra * We.c + D.ra * W.c) + D.ram * We.d) + D.ram * W.d), D.g1) *
                   (((Pe.u + P.u) - Pe.d) - P.d)) / ((((Pe.u + P.u) + Pe.d) + P.d) + kSmall), D.hz);
            const double ty1 =
                Q((Q(qq * (((rn * Ve.c + rn * V.c) + rn * Ve.s) + rn * V.s), D.g1) *
                   (((Pe.n + P.n) - Pe.s) - P.s)) / ((((Pe.n + P.n) + Pe.s) + P.s) + kSmall), D.hy);
            const double ujb1 = ((h * dt) * U.c) * (tz1 + ty1);
            const double tz2 =
                Q((Q(qq * (((D.ra * W.n + D.ra * W.c) + D.ram * W.dn) + D.ram * W.d), D.g1) *
                   (((P.un + P.u) - P.dn) - P.d)) / ((((P.un + P.u) + P.dn) + P.d) + kSmall), D.hz);
            const double tx2 =
                Q((Q(qq * (((rn * U.n + rn * U.c) + rn * Um.n) + rn * Um.c), D.g1) *
                   (((Pe.n + Pe.c) - Pwn) - Pw)) / ((((Pe.n + Pe.c) + Pwn) + Pw) + kSmall), D.hx);
            const double ujb2 = ((h * dt) * V.c) * (tz2 + tx2);
            const double ty3 =
                Q((Q(qq * (((rnp * V.u + rn * V.c) + rnp * V.us) + rn * V.s), D.g3) *
                   (((P.un + P.n) - P.us) - P.s)) / ((((P.un + P.n) + P.us) + P.s) + kSmall), D.hy);
            const double tx3 =
                Q((Q(qq * (((rnp * U.u + rn * U.c) + rnp * Um.u) + rn * Um.c), D.g3) *
                   (((Pe.u + Pe.c) - Pwu) - Pw)) / ((((Pe.u + Pe.c) + Pwu) + Pw) + kSmall), D.hx);
            const double ujb3 = ((h * dt) * W.c) * (ty3 + tx3);
            const double uc = U.c, vc = V.c, wc = W.c;
            double a = Q((((fabs(uc) * D.dx) - ((dt * uc) * uc)) * (Pe.c - P.c)) /
                             ((Pe.c + P.c) + kSmall), D.dxn) - ujb1;
            double b = Q((((fabs(vc) * D.dy) - ((dt * vc) * vc)) * (P.n - P.c)) /
                             ((P.n + P.c) + kSmall), D.dyn) - ujb2;
            double d = Q((((fabs(wc) * D.dz) - (((dt * D.rag3) * wc) * wc)) * (P.u - P.c)) /
                             ((P.u + P.c) + kSmall), D.dzn) - ujb3;
            a = a - ((qq * dt) * uc) * (Q(Ue.c - Um.c, D.xm) + d1);
            b = b - ((qq * dt) * vc) * (Q(V.n - V.s, D.ym) + d2);
            d = d - ((qq * dt) * wc) * (Q(D.rap * W.u - D.ram * W.d, D.zg3) + d3);
            st(us, c, a);
            st(vs, c, b);
            st(ws, c, d);
            return Q.ok((a + b) + d) && Q.ok(a) && Q.ok(b);
        };
        if (__builtin_expect(!cell(Fast{}), 0)) cell(Exact{});
        Pw = P.c;
        Pwn = P.n;
        Pwu = P.u;
        Um = U;
        U = Ue;
        V = Ve;
        W = We;
        P = Pe;
    }
}

// The limiter factors (k_beta<double, false>, :549-616).  HBM: psi, the
// field and three velocities read, two factors written.
__global__ __launch_bounds__(256) void k64_beta(const double *__restrict__ psi,
                                                const double *__restrict__ mptr,
                                                const double *__restrict__ po,
                                                const double *__restrict__ ut,
                                                const double *__restrict__ vt,
                                                const double *__restrict__ wt,
                                                double *__restrict__ bup,
                                                double *__restrict__ bdn,
                                                const int *__restrict__ flag, Geo g, Metrics M,
                                                double dt, int planes) {
    if (*flag) return;
    const Col q = column(g, planes);
    if (!q.act) return;
    const int k = q.k, j = q.j;
    const unsigned SI = q.SI, SJ = q.SJ;
    const double m = *mptr;
    const Den dx(M.dxn[1]), dy(M.dyn[j]), dz(M.dzn[k]);
    const double rn = M.rhoan[k], ra = M.rhoa[k], ram = M.rhoa[k - 1];
    struct Plane {
        double s, ss, sn, sd, su;  // psi at (k,j), j-1, j+1, k-1, k+1
        double p, ps, pn, pd, pu;  // the field
        double u, v, vl, w, wl;
    };
    auto load = [&](unsigned c) {
        return Plane{ld(psi, c),     ld(psi, c - SJ), ld(psi, c + SJ), ld(psi, c - 1),
                     ld(psi, c + 1), ld(po, c),       ld(po, c - SJ),  ld(po, c + SJ),
                     ld(po, c - 1),  ld(po, c + 1),   ld(ut, c),       ld(vt, c),
                     ld(vt, c - SJ), ld(wt, c),       ld(wt, c - 1)};
    };
    unsigned c = q.c;
    double sw = ld(psi, c - SI) - m, pw = ld(po, c - SI), ul = ld(ut, c - SI);
    Plane A = load(c);
    for (int i = q.i0; i <= q.i1; ++i, c += SI) {
        const Plane N = load(c + SI);
        const double sc = A.s - m, se = N.s - m, pc = A.p, pe = N.p;
        const double vals[14] = {sc, sw, se, A.ss - m, A.sn - m, A.sd - m, A.su - m,
                                 pc, pw, pe, A.ps,     A.pn,     A.pd,     A.pu};
        double mx = vals[0], mn = vals[0];
#pragma unroll
        for (int e = 1; e < 14; ++e) {
            if (vals[e] > mx) mx = vals[e];
            if (vals[e] < mn) mn = vals[e];
        }
        auto cell = [&](auto Q) {
            const double d1 =
                (dt * ((Q((pos(ul) * rn) * pw - (neg(A.u) * rn) * pe, dx) +
                        Q((pos(A.vl) * rn) * A.ps - (neg(A.v) * rn) * A.pn, dy)) +
                       Q((pos(A.wl) * ram) * A.pd - (neg(A.w) * ra) * A.pu, dz))) + kSmall;
            const double d2 = dt * (((Q((pos(A.u) * rn) * pc - (neg(ul) * rn) * pc, dx) +
                                      Q((pos(A.v) * rn) * pc - (neg(A.vl) * rn) * pc, dy)) +
                                     Q((pos(A.w) * ra) * pc - (neg(A.wl) * ram) * pc, dz)) +
                                    kSmall);
            st(bup, c, (rn * (mx - pc)) / d1);
            st(bdn, c, (rn * (pc - mn)) / d2);
            return Q.ok(d1) && Q.ok(d2);
        };
        if (__builtin_expect(!cell(Fast{}), 0)) cell(Exact{});
        sw = sc;
        pw = pc;
        ul = A.u;
        A = N;
    }
}

// limited velocity of eq 18 at a face: this side's factors, the other's
__device__ __forceinline__ double limit(double x, double up, double dn, double up2, double dn2) {
    return least3(1.0, dn, up2) * pos(x) + least3(1.0, up, dn2) * neg(x);
}

// The last donor pass with the limited velocities (k_upwind_limited<double,
// true>).  HBM: the field, three velocities and two factors read, psi
// written.
__global__ __launch_bounds__(256) void k64_limited(const double *__restrict__ src,
                                                   const double *__restrict__ us,
                                                   const double *__restrict__ vs,
                                                   const double *__restrict__ ws,
                                                   const double *__restrict__ bup,
                                                   const double *__restrict__ bdn,
                                                   double *__restrict__ psi_out,
                                                   const double *__restrict__ mptr,
                                                   const int *__restrict__ flag, Geo g,
                                                   Metrics M, double dt, int neumann,
                                                   int planes) {
    if (*flag) return;
    const Col q = column(g, planes);
    if (!q.act) return;
    const int k = q.k, j = q.j;
    const unsigned SI = q.SI, SJ = q.SJ;
    const double m = *mptr;
    const DonorDen D{Den(2.0 * M.dxn[1]), Den(2.0 * M.dyn[j]), Den((2.0 * M.dzn[k]) * M.rhoan[k]),
                     M.rhoa[k], M.rhoa[k - 1]};
    // the face below j: of cell j-1, or of its periodic image jp (the factors
    // of the face's other side are the cell's own)
    const unsigned js = j == 1 ? (unsigned)(g.jp - 1) * SJ : 0u - SJ;
    // (the image's upper neighbour is the halo row jp+1)
    const unsigned jn = js + SJ;
    struct Plane {
        double p, pn, ps, pu, pd, u, v, vl, w, wl;
        double bu, bd, bun, bdn, bus, bds, buu, bdu, bud, bdd, bui, bdi;
    };
    auto load = [&](unsigned c) {
        return Plane{ld(src, c),      ld(src, c + SJ), ld(src, c - SJ), ld(src, c + 1),
                     ld(src, c - 1),  ld(us, c),       ld(vs, c),       ld(vs, c + js),
                     ld(ws, c),       ld(ws, c - 1),   ld(bup, c),      ld(bdn, c),
                     ld(bup, c + SJ), ld(bdn, c + SJ), ld(bup, c + js), ld(bdn, c + js),
                     ld(bup, c + 1),  ld(bdn, c + 1),  ld(bup, c - 1),  ld(bdn, c - 1),
                     ld(bup, c + jn), ld(bdn, c + jn)};
    };
    unsigned c = q.c;
    // the face west of plane i0: of plane i0-1, or of its periodic image ip
    const unsigned cw = q.i0 == 1 ? c + (unsigned)(g.ip - 1) * SI : c - SI;
    double ul = limit(ld(us, cw), ld(bup, cw), ld(bdn, cw), ld(bup, cw + SI), ld(bdn, cw + SI));
    double pw = ld(src, c - SI);
    Plane A = load(c);
    for (int i = q.i0; i <= q.i1; ++i, c += SI) {
        const Plane N = load(c + SI);
        const double uc = limit(A.u, A.bu, A.bd, N.bu, N.bd);
        const double vc = limit(A.v, A.bu, A.bd, A.bun, A.bdn);
        const double vl = limit(A.vl, A.bus, A.bds, A.bui, A.bdi);
        const double wc = limit(A.w, A.bu, A.bd, A.buu, A.bdu);
        const double wl = k == 1 ? 0.0 : limit(A.wl, A.bud, A.bdd, A.bu, A.bd);
        auto cell = [&](auto Q) {
            const double r = donor_cell(Q, D, dt, uc, ul, vc, vl, wc, wl, A.p, N.p, pw, A.pn, A.ps,
                                        A.pu, A.pd, k, g.kp, neumann);
            st(psi_out, c, r + m);
            return Q.ok(r);
        };
        if (__builtin_expect(!cell(Fast{}), 0)) cell(Exact{});
        ul = uc;
        pw = A.p;
        A = N;
    }
}

}  // namespace

// Planes a thread marches (each march loads two planes beside its own): 16,
// fewer where that leaves less than about four blocks a CU
static Interior march_launch(const Geo &g, int *planes) {
    Interior L = interior_launch(g);
    int p = 16;
    while (p > 2 && (long long)L.grid.x * L.grid.y * ((g.ip + p - 1) / p) < 1024) p /= 2;
    *planes = p;
    L.grid.z = (unsigned)((g.ip + p - 1) / p);
    return L;
}

bool mpdata64_fast(const dcm_ctx *c) {
    return c->uniform_x && c->metrics_moderate && c->geo.ntot < (1LL << 29);
}

int mpdata64_donor1(dcm_ctx *c, double dt, const double *psi, const double *m, const double *u,
                    const double *v, const double *w, double *out, int neumann) {
    int planes;
    const Interior L = march_launch(c->geo, &planes);
    const int tok = prof_begin(c, "upwind_first");
    hipLaunchKernelGGL(k64_donor1, L.grid, L.block, 0, c->stream, psi, m, u, v, w, out, c->geo,
                       c->met, dt, neumann, planes);
    DCM_LAUNCH_CHECK();
    prof_end(c, tok);
    return DCM_OK;
}

int mpdata64_antidiff(dcm_ctx *c, double dt, const double *u, const double *v, const double *w,
                      const double *po, double *us, double *vs, double *ws, const int *flag) {
    int planes;
    const Interior L = march_launch(c->geo, &planes);
    const int tok = prof_begin(c, "antidiff");
    hipLaunchKernelGGL(k64_antidiff, L.grid, L.block, 0, c->stream, u, v, w, po, us, vs, ws, flag,
                       c->geo, c->met, dt, planes);
    DCM_LAUNCH_CHECK();
    prof_end(c, tok);
    return DCM_OK;
}

int mpdata64_beta(dcm_ctx *c, double dt, const double *psi, const double *m, const double *po,
                  const double *us, const double *vs, const double *ws, double *bup, double *bdn,
                  const int *flag) {
    int planes;
    const Interior L = march_launch(c->geo, &planes);
    const int tok = prof_begin(c, "beta");
    hipLaunchKernelGGL(k64_beta, L.grid, L.block, 0, c->stream, psi, m, po, us, vs, ws, bup, bdn,
                       flag, c->geo, c->met, dt, planes);
    DCM_LAUNCH_CHECK();
    prof_end(c, tok);
    return DCM_OK;
}

int mpdata64_limited(dcm_ctx *c, double dt, const double *src, const double *us, const double *vs,
                     const double *ws, const double *bup, const double *bdn, double *psi,
                     const double *m, const int *flag, int neumann) {
    int planes;
    const Interior L = march_launch(c->geo, &planes);
    const int tok = prof_begin(c, "upwind_limited");
    hipLaunchKernelGGL(k64_limited, L.grid, L.block, 0, c->stream, src, us, vs, ws, bup, bdn, psi,
                       m, flag, c->geo, c->met, dt, neumann, planes);
    DCM_LAUNCH_CHECK();
    prof_end(c, tok);
    return DCM_OK;
}

}  // namespace dcm
