// gasadj.hpp -- reverse-mode derivatives of the point fluxes of gas.hpp: given the adjoint Fb of a
// flux, the adjoints of its states, means and gradients in one pass.
//
// Each function restates the forward chain (the same branches) and walks it backwards.  One reverse
// pass costs a few times the flux whatever the number of inputs; evaluated on dual numbers the
// inviscid flux takes 20 passes and the viscous one 40.  Entropy fixes other than Harten-Yee, functions of
// seven scalars, are differentiated on dual numbers.
#pragma once
#include "dual.hpp"
#include "gas.hpp"

namespace dndsr
{
// Adjoints of the Roe average's fields and of the mean states' own quantities, summed over a face's points
struct RoeBar
{
    real v[3] = {0, 0, 0}, H = 0, a = 0, vsqr = 0, rho = 0, g1a2 = 0, inv2a = 0;
    real vL[3] = {0, 0, 0}, vR[3] = {0, 0, 0}, aL = 0, aR = 0, pL = 0, pR = 0;
};

// U -> (v, p, a, H) backwards: adds to Ub
__host__ __device__ inline void thermoBar(const real *U, real gamma, const real *v, real p, real a, real H,
                                          const real *vb_, real pb, real ab, real Hb, real *Ub)
{
    const real ri = rcpN(U[0]);
    real vb[3] = {vb_[0], vb_[1], vb_[2]};
    const real v2 = dot3(v, v);
    real rb = 0;
    if (ab != 0)
    {
        const real a2b = ab * 0.5 * rcpN(a);
        pb += gamma * ri * a2b;
        rb -= a * a * ri * a2b;
    }
    Ub[4] += Hb * ri;
    pb += Hb * ri;
    rb -= H * Hb * ri;
    Ub[4] += (gamma - 1) * pb;
    rb -= (gamma - 1) * 0.5 * v2 * pb;
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        vb[d] -= (gamma - 1) * U[1 + d] * pb;
        Ub[1 + d] += vb[d] * ri;
        rb -= v[d] * vb[d] * ri;
    }
    Ub[0] += rb;
}

// sideFlux backwards (pb, ab: further adjoints of the point's pressure and sound speed)
__host__ __device__ inline void sideFluxBar(const real *U, const real *n, real gamma, real p, real a, const real *Fb,
                                            real pb, real ab, real *Ub)
{
    const real ri = rcpN(U[0]);
    const real v[3] = {U[1] * ri, U[2] * ri, U[3] * ri};
    const real vn = dot3(v, n);
    real vnb = Fb[4] * p;
#pragma unroll
    for (int i = 0; i < 5; i++)
    {
        vnb += Fb[i] * U[i];
        Ub[i] += Fb[i] * vn;
    }
    pb += Fb[1] * n[0] + Fb[2] * n[1] + Fb[3] * n[2] + Fb[4] * vn;
    const real vb[3] = {vnb * n[0], vnb * n[1], vnb * n[2]};
    thermoBar(U, gamma, v, p, a, 0.0, vb, pb, ab, 0.0, Ub);
}

// roeAverage backwards
__host__ __device__ inline void roeAverageBar(const real *UL, const real *UR, real gamma, const RoeAve &r,
                                              const RoeBar &b, real *ULb, real *URb)
{
    const real riL = rcpN(UL[0]), riR = rcpN(UR[0]);
    const real HL = (UL[4] + r.pLm) * riL, HR = (UR[4] + r.pRm) * riR;
    const real sL = sqrt(UL[0]), sR = sqrt(UR[0]), sInv = rcpN(sL + sR);
    const real wL = sL * sInv, wR = sR * sInv;
    // a = sqrt(a2), g1a2 = (gamma - 1) / a2, inv2a = 1 / (2 a)
    const real ia = 2 * r.inv2a;
    const real a2b = (b.a - r.inv2a * ia * b.inv2a) * r.inv2a - r.g1a2 * ia * ia * b.g1a2;
    const real Hb = b.H + (gamma - 1) * a2b, v2b = b.vsqr - 0.5 * (gamma - 1) * a2b;
    real vb[3], vLb[3], vRb[3];
    real wLb = Hb * HL, wRb = Hb * HR;
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        vb[d] = b.v[d] + 2 * r.veloRoe[d] * v2b;
        wLb += vb[d] * r.veloLm[d], wRb += vb[d] * r.veloRm[d];
        vLb[d] = b.vL[d] + wL * vb[d], vRb[d] = b.vR[d] + wR * vb[d];
    }
    const real D = (wLb - wRb) * sInv * sInv;
    ULb[0] += (D * sR + b.rho * sR) * 0.5 * rcpN(sL);
    URb[0] += (b.rho * sL - D * sL) * 0.5 * rcpN(sR);
    thermoBar(UL, gamma, r.veloLm, r.pLm, r.aLm, HL, vLb, b.pL, b.aL, wL * Hb, ULb);
    thermoBar(UR, gamma, r.veloRm, r.pRm, r.aRm, HR, vRb, b.pR, b.aR, wR * Hb, URb);
}

// adjoints of the normal velocities and eigenvalues a flux form reads, besides RoeBar
struct WaveBar
{
    real vRN = 0, vLm0 = 0, vRm0 = 0, l0 = 0, l123 = 0, l4 = 0;
};

// roeDissipation backwards: f the adjoint of incF; dUb is set
__host__ __device__ inline void roeDissipationBar(const real *dU, const real *n, const RoeAve &r, real vRN, real lam0,
                                                  real lam123, real lam4, const real *f, real *dUb, RoeBar &b,
                                                  WaveBar &w)
{
    const real dUn = dU[1] * n[0] + dU[2] * n[1] + dU[3] * n[2], a = r.aRoe, H = r.HRoe;
    const real *v = r.veloRoe;
    real t[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
        t[d] = dU[1 + d] - dU[0] * v[d];
    const real tn = dot3(t, n);
#pragma unroll
    for (int d = 0; d < 3; d++)
        t[d] -= n[d] * tn;
    const real X = dU[0] * (H - vRN * vRN) + vRN * dUn - (dU[4] - dot3(t, v));
    const real al1 = r.g1a2 * X;
    const real Y = dU[0] * (vRN + a) - dUn - a * al1;
    const real al0 = Y * r.inv2a, al4 = dU[0] - (al0 + al1);
    const real A0 = al0 * lam0, A1 = al1 * lam123, A4 = al4 * lam4;
    const real fv = f[1] * v[0] + f[2] * v[1] + f[3] * v[2], fn = f[1] * n[0] + f[2] * n[1] + f[3] * n[2];
    const real A0b = f[0] + f[4] * (H - vRN * a) + fv - a * fn;
    const real A4b = f[0] + f[4] * (H + vRN * a) + fv + a * fn;
    const real A1b = f[0] + 0.5 * r.vsqrRoe * f[4] + fv;
    const real dA = A4 - A0, sA = A0 + A4;
    real Hb = f[4] * sA, vRNb = f[4] * a * dA, ab = (f[4] * vRN + fn) * dA;
    b.vsqr += 0.5 * f[4] * A1;
    real l1b = A1b * al1, tb[3], vb[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        const real Bb = f[4] * v[d] + f[1 + d];
        vb[d] = f[4] * t[d] * lam123 + f[1 + d] * (sA + A1);
        l1b += Bb * t[d];
        tb[d] = Bb * lam123;
    }
    w.l0 += A0b * al0, w.l123 += l1b, w.l4 += A4b * al4;
    const real al4b = A4b * lam4;
    real rb = al4b;
    const real al0b = A0b * lam0 - al4b;
    real al1b = A1b * lam123 - al4b;
    const real Yb = al0b * r.inv2a;
    b.inv2a += al0b * Y;
    rb += Yb * (vRN + a), vRNb += Yb * dU[0], ab += Yb * (dU[0] - al1);
    real dUnb = -Yb;
    al1b -= a * Yb;
    const real Xb = al1b * r.g1a2;
    b.g1a2 += al1b * X;
    rb += Xb * (H - vRN * vRN), Hb += Xb * dU[0], vRNb += Xb * (dUn - 2 * vRN * dU[0]), dUnb += Xb * vRN;
    // dU4b = dE - t . v enters X with -1
    dUb[4] = -Xb;
    real tbn = 0;
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        tb[d] += v[d] * Xb, vb[d] += t[d] * Xb;
        tbn += tb[d] * n[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        const real q = tb[d] - n[d] * tbn;
        dUb[1 + d] = q + n[d] * dUnb;
        rb -= q * v[d];
        vb[d] -= dU[0] * q;
        b.v[d] += vb[d];
    }
    dUb[0] = rb;
    b.H += Hb, b.a += ab, w.vRN += vRNb;
}

// Harten-Yee fix of one eigenvalue backwards: l = Flim(v, lam, lamL, lamR)
__host__ __device__ inline void hartenYeeBar(real v, real lam, real lamL, real lamR, real sHY, real lb, real &vb,
                                             real &lamb, real &lamLb, real &lamRb)
{
    const real d1 = lam - lamL, d2 = lamR - lam;
    const real mx = max3(0., d1, d2), th = mx * sHY;
    if (v < th)
    {
        const real q = v * rcpN(th);
        vb += lb * q;
        const real tb = lb * 0.5 * (1 - q * q) * sHY;
        if (d1 >= d2)
            lamb += tb, lamLb -= tb;
        else
            lamRb += tb, lamb -= tb;
    }
    else
        vb += lb;
}

// the eigenvalue fix (roeFix) of a Roe scheme backwards; vn quantities on the normal nv
template <int EIG>
__host__ __device__ inline void roeFixBar(const RoeAve &r, real vLm0, real vRm0, real vRN, real dLambda,
                                          const GasParams &gp, RoeBar &b, WaveBar &w)
{
    const real a = r.aRoe;
    if constexpr (EIG == 0)
    {
        const real sHY = 0.05 * gp.fixScale;
        const real s0 = vRN - a, s4 = vRN + a;
        real v0b = 0, v1b = 0, v4b = 0, m0 = 0, m0L = 0, m0R = 0, m1 = 0, m1L = 0, m1R = 0, m4 = 0, m4L = 0, m4R = 0;
        hartenYeeBar(fabs(s0), s0, vLm0 - r.aLm, vRm0 - r.aRm, sHY, w.l0, v0b, m0, m0L, m0R);
        hartenYeeBar(fabs(vRN) * gp.incFScale, vRN, vLm0, vRm0, sHY, w.l123, v1b, m1, m1L, m1R);
        hartenYeeBar(fabs(s4), s4, vLm0 + r.aLm, vRm0 + r.aRm, sHY, w.l4, v4b, m4, m4L, m4R);
        const real s0b = (s0 < 0 ? -v0b : v0b) + m0, s4b = (s4 < 0 ? -v4b : v4b) + m4;
        w.vRN += s0b + s4b + (vRN < 0 ? -v1b : v1b) * gp.incFScale + m1;
        b.a += s4b - s0b;
        w.vLm0 += m0L + m1L + m4L, w.vRm0 += m0R + m1R + m4R;
        b.aL += m4L - m0L, b.aR += m4R - m0R;
    }
    else
    {
        const real VA = sqrt(r.vsqrRoe);
        const real x[7] = {r.aLm, r.aRm, a, vLm0, vRm0, vRN, VA};
        real xb[7];
        constexpr int nDir = EIG == 7 || EIG == 8 ? 7 : 6;
        for (int d = 0; d < nDir; d++)
        {
            Dual q[7];
            for (int k = 0; k < 7; k++)
                q[k] = Dual(x[k], k == d ? 1.0 : 0.0);
            Dual l0 = fabs(q[5] - q[2]), l1 = fabs(q[5]), l4 = fabs(q[5] + q[2]);
            roeFix<EIG>(q[0], q[1], q[2], q[3], q[4], q[5], q[6], dLambda, gp.fixScale, gp.incFScale, l0, l1, l4);
            xb[d] = w.l0 * l0.d + w.l123 * l1.d + w.l4 * l4.d;
        }
        b.aL += xb[0], b.aR += xb[1], b.a += xb[2];
        w.vLm0 += xb[3], w.vRm0 += xb[4], w.vRN += xb[5];
        if (nDir == 7 && VA > 0)
            b.vsqr += xb[6] * 0.5 / VA;
    }
}

// bcGhost backwards: adds (d ghost / d UL)^T URb to ULb.  The linear ghosts (mirror, reversal, copy, given
// state) are their own transposes; the others go through dual numbers, one column of the Jacobian per pass.
__host__ __device__ inline void bcGhostBar(int type, const real *UL, const real *n, const real *far, real gamma,
                                           const real *URb, real *ULb)
{
    if (type == BC_IN)
        return;
    if (type == BC_WALL_INVIS || type == BC_SYM || type == BC_WALL || type == BC_OUT)
    {
        const real mn = URb[1] * n[0] + URb[2] * n[1] + URb[3] * n[2];
        ULb[0] += URb[0];
#pragma unroll
        for (int d = 0; d < 3; d++)
            ULb[1 + d] += type == BC_OUT ? URb[1 + d] : (type == BC_WALL ? -URb[1 + d] : URb[1 + d] - 2 * mn * n[d]);
        ULb[4] += URb[4];
        return;
    }
#pragma unroll 1
    for (int c = 0; c < 5; c++)
    {
        Dual D[5], DR[5];
#pragma unroll
        for (int v = 0; v < 5; v++)
            D[v] = Dual(UL[v], v == c ? 1.0 : 0.0);
        bcGhost(type, D, n, far, gamma, DR);
        real a = 0;
#pragma unroll
        for (int v = 0; v < 5; v++)
            a += URb[v] * DR[v].d;
#pragma unroll
        for (int v = 0; v < 5; v++)
            ULb[v] += v == c ? a : 0.0;
    }
}

// Riemann flux (riemannFluxR, or with BATCH roeBatchPoint on roeBatchSetup) backwards: adds to ULb, URb and
// b.  n the point normal, nm the mean normal (BATCH).
template <int RS, bool BATCH>
__host__ __device__ inline void riemannFluxBar(const real *UL, const real *UR, const RoeAve &r, const real *n,
                                               const real *nm, const GasParams &gp, real dLambda, const real *Fb,
                                               real *ULb, real *URb, RoeBar &b)
{
    const real gamma = gp.gamma;
    const real *nv = BATCH ? nm : n;
    real FL[5], FR[5], pL, pR, aL, aR, dU[5];
    sideFlux(UL, n, gamma, FL, pL, aL);
    sideFlux(UR, n, gamma, FR, pR, aR);
#pragma unroll
    for (int i = 0; i < 5; i++)
        dU[i] = UR[i] - UL[i];
    const real vRN = dot3(r.veloRoe, nv), vLm0 = dot3(r.veloLm, nv), vRm0 = dot3(r.veloRm, nv);
    WaveBar w;
    real FLb[5], FRb[5], dUb[5] = {0, 0, 0, 0, 0}, pLb = 0, pRb = 0, aLb = 0, aRb = 0;
    if constexpr (RS == RS_Roe_M2) // Lax-Friedrichs on the means
    {
        const real lL = fabs(vLm0) + r.aLm, lR = fabs(vRm0) + r.aRm, l = fmax(lL, lR);
        real lb = 0;
#pragma unroll
        for (int i = 0; i < 5; i++)
        {
            FLb[i] = FRb[i] = 0.5 * Fb[i];
            dUb[i] = -0.5 * l * Fb[i];
            lb -= 0.5 * Fb[i] * dU[i];
        }
        if (lL >= lR)
            b.aL += lb, w.vLm0 += vLm0 < 0 ? -lb : lb;
        else
            b.aR += lb, w.vRm0 += vRm0 < 0 ? -lb : lb;
    }
    else if constexpr (RS == RS_Roe || (RS >= RS_Roe_M1 && RS <= RS_Roe_M8) || RS == RS_HLLEP_V1)
    {
        real l0 = fabs(vRN - r.aRoe), l1 = fabs(vRN), l4 = fabs(vRN + r.aRoe), f[5];
#pragma unroll
        for (int i = 0; i < 5; i++)
            FLb[i] = FRb[i] = 0.5 * Fb[i], f[i] = -0.5 * Fb[i];
        if constexpr (RS == RS_HLLEP_V1)
        {
            // the eigenvalues from (vRN, a, vL, vR, aL, aR) on dual numbers
            const real x[6] = {vRN, r.aRoe, vLm0, vRm0, aL, aR};
            auto lams = [&](const Dual *q, Dual &d0, Dual &d1, Dual &d4) {
                const Dual SL = fmin(q[0] - q[1], q[2] - q[4]), SR = fmax(q[0] + q[1], q[3] + q[5]);
                const Dual dfix = q[1] * rcpN(q[1] + fmax(fabs(q[0]), Dual(dLambda * gp.fixScale)));
                const Dual SP = fmax(SR, Dual(0.0)), SM = fmin(SL, Dual(0.0));
                const Dual dinv = rcpN(SP - SM);
                d1 = fabs(((SP + SM) * q[0] - 2.0 * (1.0 - dfix) * (SP * SM)) * dinv);
                d4 = fabs(((SP + SM) * (q[0] + q[1]) - 2.0 * (SP * SM)) * dinv);
                d0 = fabs(((SP + SM) * (q[0] - q[1]) - 2.0 * (SP * SM)) * dinv);
            };
            Dual q[6], d0, d1, d4;
            for (int k = 0; k < 6; k++)
                q[k] = Dual(x[k], 0.0);
            lams(q, d0, d1, d4);
            roeDissipationBar(dU, n, r, vRN, d0.v, d1.v, d4.v, f, dUb, b, w);
            real xb[6];
            for (int d = 0; d < 6; d++)
            {
                for (int k = 0; k < 6; k++)
                    q[k] = Dual(x[k], k == d ? 1.0 : 0.0);
                lams(q, d0, d1, d4);
                xb[d] = w.l0 * d0.d + w.l123 * d1.d + w.l4 * d4.d;
            }
            w.vRN += xb[0], b.a += xb[1], w.vLm0 += xb[2], w.vRm0 += xb[3];
            aLb = xb[4], aRb = xb[5];
        }
        else
        {
            constexpr int EIG = RS == RS_Roe ? 0 : RS - 10;
            roeFix<EIG>(r.aLm, r.aRm, r.aRoe, vLm0, vRm0, vRN, sqrt(r.vsqrRoe), dLambda, gp.fixScale, gp.incFScale,
                        l0, l1, l4);
            roeDissipationBar(dU, n, r, vRN, l0, l1, l4, f, dUb, b, w);
            roeFixBar<EIG>(r, vLm0, vRm0, vRN, dLambda, gp, b, w);
        }
    }
    else if constexpr (RS == RS_HLLEP)
    {
        const real a = r.aRoe, *v = r.veloRoe;
        const real dUn = dU[1] * n[0] + dU[2] * n[1] + dU[3] * n[2];
        real t[3];
#pragma unroll
        for (int d = 0; d < 3; d++)
            t[d] = dU[1 + d] - dU[0] * v[d];
        const real tn = dot3(t, n);
#pragma unroll
        for (int d = 0; d < 3; d++)
            t[d] -= n[d] * tn;
        const real X = dU[0] * (r.HRoe - vRN * vRN) + vRN * dUn - (dU[4] - dot3(t, v));
        const real al1 = r.g1a2 * X;
        const real SLa = vRN - a, SLb = vLm0 - aL, SRa = vRN + a, SRb = vRm0 + aR;
        const real SL = fmin(SLa, SLb), SR = fmax(SRa, SRb);
        const real c = dLambda * gp.fixScale, mx = fmax(fabs(vRN), c), q = rcpN(a + mx), dfix = a * q;
        const real SP = fmax(SR, 0.0), SM = fmin(SL, 0.0);
        real div = SP - SM;
        div += signP(div) * kVerySmall;
        const real dinv = rcpN(div), spsm = SP * SM * dinv, dal = dfix * al1;
        const real rev[5] = {1, v[0], v[1], v[2], 0.5 * r.vsqrRoe};
        real SPb = 0, SMb = 0, dinvb = 0, spsmb = 0, dalb = 0;
#pragma unroll
        for (int i = 0; i < 5; i++)
        {
            FLb[i] = SP * dinv * Fb[i], FRb[i] = -SM * dinv * Fb[i];
            SPb += dinv * Fb[i] * FL[i], SMb -= dinv * Fb[i] * FR[i];
            dinvb += Fb[i] * (SP * FL[i] - SM * FR[i]);
            spsmb += Fb[i] * (dU[i] - rev[i] * dal);
            const real Wb = spsm * Fb[i];
            dUb[i] = Wb;
            dalb -= Wb * rev[i];
        }
#pragma unroll
        for (int d = 0; d < 3; d++)
            b.v[d] -= dal * dUb[1 + d];
        b.vsqr -= 0.5 * dal * dUb[4];
        SPb += spsmb * SM * dinv, SMb += spsmb * SP * dinv, dinvb += spsmb * SP * SM;
        const real divb = -dinv * dinv * dinvb;
        SPb += divb, SMb -= divb;
        const real dfixb = dalb * al1, Xb = dalb * dfix * r.g1a2;
        b.g1a2 += dalb * dfix * X;
        // X backwards
        real rb = Xb * (r.HRoe - vRN * vRN), tb[3], tbn = 0;
        b.H += Xb * dU[0];
        w.vRN += Xb * (dUn - 2 * vRN * dU[0]);
        dUb[4] -= Xb;
#pragma unroll
        for (int d = 0; d < 3; d++)
        {
            tb[d] = v[d] * Xb;
            b.v[d] += t[d] * Xb;
            tbn += tb[d] * n[d];
        }
#pragma unroll
        for (int d = 0; d < 3; d++)
        {
            const real s = tb[d] - n[d] * tbn;
            dUb[1 + d] += s + n[d] * Xb * vRN;
            rb -= s * v[d];
            b.v[d] -= dU[0] * s;
        }
        dUb[0] += rb;
        // wave speeds
        if (SR >= 0)
        {
            if (SRa >= SRb)
                w.vRN += SPb, b.a += SPb;
            else
                w.vRm0 += SPb, aRb += SPb;
        }
        if (SL <= 0)
        {
            if (SLa <= SLb)
                w.vRN += SMb, b.a -= SMb;
            else
                w.vLm0 += SMb, aLb -= SMb;
        }
        b.a += dfixb * mx * q * q;
        if (fabs(vRN) >= c)
            w.vRN -= (vRN < 0 ? -1.0 : 1.0) * dfixb * a * q * q;
    }
    else // HLLC
    {
        const real k = (gamma + 1) / (2 * gamma);
        const real pSr = 0.5 * (r.pLm + r.pRm) - 0.5 * (vLm0 - vRm0) * r.rhoRoe * r.aRoe, pS = fmax(0.0, pSr);
        const bool sl = pS > r.pLm, sr = pS > r.pRm;
        const real qL = sl ? sqrt(1 + k * (pS / r.pLm - 1)) : 1.0, qR = sr ? sqrt(1 + k * (pS / r.pRm - 1)) : 1.0;
        const real SL = vLm0 - r.aLm * qL, SR = vRm0 + r.aRm * qR;
        real SLb = 0, SRb = 0;
#pragma unroll
        for (int i = 0; i < 5; i++)
            FLb[i] = FRb[i] = 0;
        if (0 <= SL)
#pragma unroll
            for (int i = 0; i < 5; i++)
                FLb[i] = Fb[i];
        else if (SR <= 0)
#pragma unroll
            for (int i = 0; i < 5; i++)
                FRb[i] = Fb[i];
        else
        {
            const real cL = SL - vLm0, cR = SR - vRm0;
            const real mLn = UL[1] * n[0] + UL[2] * n[1] + UL[3] * n[2], mRn = UR[1] * n[0] + UR[2] * n[1] + UR[3] * n[2];
            const real div = UL[0] * cL - UR[0] * cR;
            const bool ok = fabs(div) > kVerySmall;
            const real SS = ok ? (pR - pL + mLn * cL - mRn * cR) / div : 0.0;
            const bool left = SS >= 0;
            const real S = left ? SL : SR, v0 = left ? vLm0 : vRm0, p = left ? pL : pR, dv = S - SS;
            real U[5], Fs[5], Fsb[5], Ub[5], SSb = 0, Sb = 0, v0b = 0, pb = 0;
#pragma unroll
            for (int i = 0; i < 5; i++)
                U[i] = left ? UL[i] : UR[i], Fs[i] = left ? FL[i] : FR[i], Ub[i] = 0;
            if (fabs(dv) < kVerySmall)
#pragma unroll
                for (int i = 0; i < 5; i++)
                    Fsb[i] = Fb[i];
            else
            {
                const real idv = 1.0 / dv, P = p + U[0] * (S - v0) * (SS - v0), Q = P * S;
                const real D[5] = {0, n[0], n[1], n[2], SS};
                real Qb = 0, dvb = 0;
#pragma unroll
                for (int i = 0; i < 5; i++)
                {
                    const real Nb = Fb[i] * idv, z = U[i] * S - Fs[i];
                    dvb -= Nb * (z * SS + D[i] * Q) * idv;
                    Ub[i] = Nb * S * SS;
                    Sb += Nb * U[i] * SS;
                    Fsb[i] = -Nb * SS;
                    SSb += Nb * z;
                    Qb += Nb * D[i];
                    if (i == 4)
                        SSb += Nb * Q;
                }
                Sb += dvb, SSb -= dvb;
                const real Pb = Qb * S;
                Sb += Qb * P;
                pb = Pb;
                Ub[0] += Pb * (S - v0) * (SS - v0);
                Sb += Pb * U[0] * (SS - v0), SSb += Pb * U[0] * (S - v0);
                v0b = -Pb * U[0] * ((SS - v0) + (S - v0));
            }
#pragma unroll
            for (int i = 0; i < 5; i++)
            {
                FLb[i] = left ? Fsb[i] : 0.0, FRb[i] = left ? 0.0 : Fsb[i];
                ULb[i] += left ? Ub[i] : 0.0, URb[i] += left ? 0.0 : Ub[i];
            }
            (left ? pLb : pRb) += pb;
            (left ? SLb : SRb) += Sb;
            (left ? w.vLm0 : w.vRm0) += v0b;
            if (ok)
            {
                const real nb = SSb / div, db = -SSb * SS / div;
                pRb += nb, pLb -= nb;
#pragma unroll
                for (int d = 0; d < 3; d++)
                    ULb[1 + d] += nb * cL * n[d], URb[1 + d] -= nb * cR * n[d];
                ULb[0] += db * cL, URb[0] -= db * cR;
                const real cLb = nb * mLn + db * UL[0], cRb = -nb * mRn - db * UR[0];
                SLb += cLb, w.vLm0 -= cLb, SRb += cRb, w.vRm0 -= cRb;
            }
        }
        if (0 <= SL || SR <= 0)
            SLb = SRb = 0;
        w.vLm0 += SLb, w.vRm0 += SRb;
        b.aL -= qL * SLb, b.aR += qR * SRb;
        real pSb = 0;
        if (sl)
        {
            const real rb = -r.aLm * SLb * k * 0.5 / qL;
            pSb += rb / r.pLm, b.pL -= rb * pS / (r.pLm * r.pLm);
        }
        if (sr)
        {
            const real rb = r.aRm * SRb * k * 0.5 / qR;
            pSb += rb / r.pRm, b.pR -= rb * pS / (r.pRm * r.pRm);
        }
        if (pSr > 0)
        {
            b.pL += 0.5 * pSb, b.pR += 0.5 * pSb;
            const real z = 0.5 * r.rhoRoe * r.aRoe * pSb, dv = 0.5 * (vLm0 - vRm0) * pSb;
            w.vLm0 -= z, w.vRm0 += z;
            b.rho -= dv * r.aRoe, b.a -= dv * r.rhoRoe;
        }
    }
#pragma unroll
    for (int i = 0; i < 5; i++)
        URb[i] += dUb[i], ULb[i] -= dUb[i];
    sideFluxBar(UL, n, gamma, pL, aL, FLb, pLb, aLb, ULb);
    sideFluxBar(UR, n, gamma, pR, aR, FRb, pRb, aRb, URb);
#pragma unroll
    for (int d = 0; d < 3; d++)
        b.v[d] += w.vRN * nv[d], b.vL[d] += w.vLm0 * nv[d], b.vR[d] += w.vRm0 * nv[d];
}

// viscousPointFlux backwards: adds to ULb, URb and sets Gb, the adjoint of the mean gradient GM (each side's
// gradient gets half).  Ga = (GL + GR) / 2, idist = 1 / distGRP; an adiabatic wall carries no heat.
__host__ __device__ inline void viscousPointBar(const GasParams &gp, const real *UL, const real *UR,
                                                const real (*Ga)[5], const real *n, real idist, bool adiabatic,
                                                const real *Fb, real *ULb, real *URb, real (*Gb)[5])
{
    const real g1 = gp.gamma - 1, Cp = cpGas(gp), lambda = -2. / 3.;
    real U[5], G[3][5];
#pragma unroll
    for (int v = 0; v < 5; v++)
    {
        U[v] = 0.5 * (UL[v] + UR[v]);
        const real j = (UR[v] - UL[v]) * idist;
#pragma unroll
        for (int d = 0; d < 3; d++)
            G[d][v] = Ga[d][v] + n[d] * j;
    }
    const real ri = rcpN(U[0]);
    const real v[3] = {U[1] * ri, U[2] * ri, U[3] * ri};
    const real v2 = dot3(v, v), p = g1 * (U[4] - 0.5 * U[0] * v2);
    const real c = gp.gamma * ri * ri / (g1 * Cp);
    real gv[3][3], dp[3], gT[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        real vm = 0;
#pragma unroll
        for (int j = 0; j < 3; j++)
            gv[d][j] = (G[d][1 + j] - v[j] * G[d][0]) * ri, vm += v[j] * G[d][1 + j];
        dp[d] = g1 * (G[d][4] - vm + 0.5 * v2 * G[d][0]);
        gT[d] = c * (U[0] * dp[d] - p * G[d][0]);
    }
    const real T = gasTemperature(gp, p, U[0]);
    const real mu = muEff(gp, U, T), kp = Cp / gp.prGas, k = kp * mu;
    const real tr = gv[0][0] + gv[1][1] + gv[2][2];
    real s[3], fb[3], fbn = 0, mub = 0, vb[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
    {
        s[i] = lambda * tr * n[i];
#pragma unroll
        for (int j = 0; j < 3; j++)
            s[i] += (gv[i][j] + gv[j][i]) * n[j];
        fb[i] = Fb[1 + i] + Fb[4] * v[i];
        fbn += fb[i] * n[i];
        mub += fb[i] * s[i];
        vb[i] = Fb[4] * mu * s[i];
    }
    const real hk = adiabatic ? 0.0 : Fb[4];
    mub += hk * kp * dot3(gT, n);
    real rb = 0, pb = 0, cb = 0;
#pragma unroll
    for (int d = 0; d < 3; d++)
    {
        const real gTb = hk * k * n[d];
        cb += gTb * (U[0] * dp[d] - p * G[d][0]);
        rb += c * gTb * dp[d];
        pb -= c * gTb * G[d][0];
        const real dpb = c * U[0] * gTb * g1;
        real g0 = -c * p * gTb + 0.5 * v2 * dpb;
        Gb[d][4] = dpb;
#pragma unroll
        for (int j = 0; j < 3; j++)
        {
            real q = mu * (fb[d] * n[j] + fb[j] * n[d]);
            if (d == j)
                q += lambda * mu * fbn;
            Gb[d][1 + j] = q * ri - v[j] * dpb;
            vb[j] += -G[d][1 + j] * dpb + v[j] * G[d][0] * dpb - q * G[d][0] * ri;
            g0 -= q * v[j] * ri;
            rb -= q * gv[d][j] * ri;
        }
        Gb[d][0] = g0;
    }
    rb -= 2 * c * ri * cb;
    if (gp.muModel == 1)
    {
        const real Tb = mub * mu * (1.5 / T - 1.0 / (T + gp.CSutherland));
        const real q = Tb * T * ri;
        rb -= q;
        pb += q * U[0] / p;
    }
    else if (gp.muModel == 2)
        rb += mub * gp.muGas;
    real Ub[5] = {rb, 0, 0, 0, 0};
    thermoBar(U, gp.gamma, v, p, 1.0, 0.0, vb, pb, 0.0, 0.0, Ub);
#pragma unroll
    for (int q = 0; q < 5; q++)
    {
        const real jb = idist * (n[0] * Gb[0][q] + n[1] * Gb[1][q] + n[2] * Gb[2][q]);
        ULb[q] += 0.5 * Ub[q] - jb;
        URb[q] += 0.5 * Ub[q] + jb;
    }
}
} // namespace dndsr
