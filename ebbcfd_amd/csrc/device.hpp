// Device code shared by the stage kernels: fluxes, ghost states, gradients and limiters,
// reconstruction, the cell update and the RMS leaf sums.  Included by every kernel file, so
// each of them runs the same arithmetic.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "dev.hpp"

namespace ebb {

#define DEV __device__ __forceinline__
constexpr double G_ = 1.4;
constexpr int BLK = 256;
static_assert(uint32_t(BLK) == FACE_TILE_LANES, "face tile padding assumes one lane per workgroup thread");

enum { BT_FULL = 0, BT_CONSTP, BT_INVWALL, BT_VISCWALL, BT_SYM, BT_TPIN, BT_DIRICHLET };

// workgroup b runs on XCD b % 8; hand each XCD a contiguous slice of the cells
DEV uint32_t xcdBlock(uint32_t b, uint32_t nb)
{
    const uint32_t nx = 8, per = nb / nx, rem = nb % nx, x = b % nx, k = b / nx;
    return x * per + (x < rem ? x : rem) + k;
}

// The same slices, each walked last to first (the k-th workgroup of XCD x takes the k-th
// item from its slice's end; k < the slice's length for every b < nb)
DEV uint32_t xcdBlockBack(uint32_t b, uint32_t nb)
{
    const uint32_t nx = 8, per = nb / nx, rem = nb % nx, x = b % nx, k = b / nx;
    const uint32_t len = per + (x < rem ? 1u : 0u);
    return x * per + (x < rem ? x : rem) + (len - 1 - k);
}

// The face, reconstruction and limiter arithmetic below is written once for the
// real type R it computes in: double on the FP64 path, float on the mixed path
// (extensions.precision = "mixed").  Every literal is converted to R, so the double
// instantiation performs exactly the operations of the FP64 path and the float one
// never promotes to double.
template <typename R>
DEV R pressure(const R q[4])
{
    const R a = q[1] / q[0], b = q[2] / q[0];
    return R(G_ - 1) * (q[3] - R(0.5) * q[0] * (a * a + b * b));
}

template <typename R>
DEV R dmax(R a, R b) { return a < b ? b : a; }

// Division by one denominator, several times.  FAST 0: IEEE division.  FAST 1: one refined
// reciprocal per denominator, in FP64, which a quotient is formed from in 3 instructions instead of 11.
// FP64 quotients take one Markstein correction (P. Markstein, IBM J. Res. Dev. 34, 1990): correctly
// rounded, so the same bits, for normal denominators and for numerators whose correction does not
// underflow (1e-290 and more, or zero; below that the last place may differ).  Denominators and sound
// speeds near the type's lower end are turned away by FastRange.  FP32 quotients are the product with
// the FP64 reciprocal, rounded: it is within 2^-51 and a quotient of two FP32 numbers is no nearer than
// 2^-49 to the middle of two others, so they are the same bits for every denominator but zero and
// infinity (of subnormal quotients those that are such a middle may differ).  Those two, and an
// infinite FP64 numerator, give NaN, which the flux carries to its caller (faceTileBody: fluxInRange),
// who then takes the IEEE form (exactFace).  FP32 reciprocals with FP32 corrections, which lose them
// from numerators of 2e-31 down, took as long: 100 RK2 steps of 1M cells 18.13 and 18.18 ms.
template <int FAST, typename R>
struct Div {
    R b;
    double r;
    DEV Div() {}
    DEV explicit Div(R d) : b(d), r(0)
    {
        if constexpr (FAST) {
            const double bd = double(b);
            const double r0 = __builtin_amdgcn_rcp(bd);
            const double r1 = __builtin_fma(__builtin_fma(-bd, r0, 1.0), r0, r0);
            r = __builtin_fma(__builtin_fma(-bd, r1, 1.0), r1, r1);
        }
    }
    DEV R operator()(R a) const
    {
        if constexpr (FAST && sizeof(R) == 8) {
            const R q = a * r;
            return __builtin_fma(__builtin_fma(-b, q, a), r, q);
        } else if constexpr (FAST) {
            return R(double(a) * r);
        } else {
            return a / b;
        }
    }
};

// sqrt, with FAST 1 (FP64) by Goldschmidt's iteration from the hardware's reciprocal root without
// the scaling that small arguments need: the correctly rounded root, the same bits, from 1e-290 on;
// NaN for zero and infinity, which takes the flux to its IEEE form like Div's.
template <int FAST, typename R>
DEV R root(R x)
{
    if constexpr (FAST && sizeof(R) == 8) {
        const R y = __builtin_amdgcn_rsq(x);
        R g = x * y, h = R(0.5) * y;
        const R e = __builtin_fma(-h, g, R(0.5));
        g = __builtin_fma(g, e, g);
        h = __builtin_fma(h, e, h);
        g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
        return __builtin_fma(__builtin_fma(-g, g, x), h, g);
    } else {
        return sqrt(x);
    }
}

// A state's velocity and pressure, by the operations of pressure(), with the divider by its
// density for the flux's further quotients.
template <int FAST, typename R>
struct Prim {
    Div<FAST, R> rho;
    R u, v, p;
    DEV Prim() {}
    DEV explicit Prim(const R q[4]) : rho(q[0])
    {
        u = rho(q[1]);
        v = rho(q[2]);
        p = R(G_ - 1) * (q[3] - R(0.5) * q[0] * (u * u + v * v));
    }
};

template <typename R>
DEV R harten(R lam, R eps)
{
    if (lam < eps) lam = (eps * eps + lam * lam) / (R(2.0) * eps);
    return lam;
}

// flux.d:19-24
template <typename R>
DEV void convective(R p, R u, R v, R rho, R e, R n0, R n1, R out[4])
{
    out[0] = (rho * u) * n0 + (rho * v) * n1;
    out[1] = (p + rho * (u * u)) * n0 + (rho * u * v) * n1;
    out[2] = (rho * u * v) * n0 + (p + rho * (v * v)) * n1;
    out[3] = (u * (p + e)) * n0 + (v * (p + e)) * n1;
}

// Least sound speed and density for which the FAST fluxes stand, with a flux in range (fluxInRange).
// In FP64 they keep the denominators, the arguments of the roots and the pressures clear of Div's and
// root's lower ends.  For the Rusanov flux they also keep finite what it leaves out: a flux in range
// bounds the pressure p, p bounds the energy E (a nonzero p is at least E's last place) and E the
// momenta, so that h <= E / rhoMin and G1 / a^2 <= 10 E / aMin^2: 1e216 and 1e218 in FP64, 4e37 and
// 4e36 in FP32.
template <typename R>
struct FastRange {
    static constexpr R aMin = sizeof(R) == 8 ? R(1e-50) : R(1e-5);
    static constexpr R rhoMin = sizeof(R) == 8 ? R(1e-100) : R(1e-12);
    static DEV bool holds(R a, R rhoL, R rhoR) { return a > aMin && fmin(rhoL, rhoR) > rhoMin; }
};

// flux.d:224-303
template <int FAST, typename R>
DEV void roeFlux(const R qL[4], const Prim<FAST, R>& wL, const R qR[4], const Prim<FAST, R>& wR, R n0, R n1, R out[4],
                 R& sMax)
{
    const R gm1 = R(G_ - 1), half = R(0.5);
    const R rhoL = qL[0], uL = wL.u, vL = wL.v, pL = wL.p;
    const R rvL0 = rhoL * uL, rvL1 = rhoL * vL;
    const R hL = wL.rho(qL[3] + pL);
    const R rhoR = qR[0], uR = wR.u, vR = wR.v, pR = wR.p;
    const R rvR0 = rhoR * uR, rvR1 = rhoR * vR;
    const R hR = wR.rho(qR[3] + pR);
    const R di = root<FAST, R>(wL.rho(rhoR));
    const R d1 = Div<FAST, R>(R(1.0) + di)(R(1.0));
    const R vel0 = (di * uR + uL) * d1, vel1 = (di * vR + vL) * d1;
    const R u = vel0 * n0 + vel1 * n1;
    const R h = (di * hR + hL) * d1;
    R a = root<FAST, R>(R(G_ - 1.0) * (h - half * (vel0 * vel0 + vel1 * vel1)));
    if constexpr (FAST && sizeof(R) == 8) a = FastRange<R>::holds(a, rhoL, rhoR) ? a : R(NAN);
    const R dRhoV0 = rvR0 - rvL0, dRhoV1 = rvR1 - rvL1;
    const R dRho = rhoR - rhoL, dRhoE = qR[3] - qL[3];
    const R eps = R(0.01) * a;
    const R lam1 = harten<R>(fabs(u + a), eps);
    const R lam2 = harten<R>(fabs(u - a), eps);
    const R lam3 = harten<R>(fabs(u), eps);
    const R lam4 = harten<R>(fabs(u), eps);
    sMax = dmax<R>(dmax<R>(dmax<R>(fabs(lam1), fabs(lam2)), fabs(lam3)), fabs(lam4));
    const R s1 = half * (lam1 + lam2), s2 = half * (lam1 - lam2);
    const R qq = sqrt(vel0 * vel0 + vel1 * vel1);
    const R G1 = gm1 * (((qq * qq) / R(2.0)) * dRho - (vel0 * dRhoV0 + vel1 * dRhoV1) + dRhoE);
    const R G2 = -u * dRho + (dRhoV0 * n0 + dRhoV1 * n1);
    const Div<FAST, R> byA(a), byA2(a * a);
    const R C1 = byA2(G1) * (s1 - lam3) + byA(G2) * s2;
    const R C2 = byA(G1) * s2 + (s1 - lam3) * G2;
    R fL[4], fR[4];
    convective<R>(pL, uL, vL, rhoL, qL[3], n0, n1, fL);
    convective<R>(pR, uR, vR, rhoR, qR[3], n0, n1, fR);
    const R d[4] = {lam3 * dRho + C1, lam3 * dRhoV0 + C1 * vel0 + C2 * n0,
                    lam3 * dRhoV1 + C1 * vel1 + C2 * n1, lam3 * dRhoE + C1 * h + C2 * u};
#pragma unroll
    for (int k = 0; k < 4; k++) out[k] = half * (fL[k] + fR[k]) - half * d[k];
}

// flux.d:66-141 (Roe-type averages, C1 = C2 = 0: central flux + sMax jump)
// FAST 1 leaves out what the form with C1 = C2 = 0 multiplies by zero (s1 - sm and s2, with G1,
// G2, h and the speed): the same bits as long as those factors are finite, which FastRange says.
template <int FAST, typename R>
DEV void rusanovFlux(const R qL[4], const Prim<FAST, R>& wL, const R qR[4], const Prim<FAST, R>& wR, R n0, R n1,
                     R out[4], R& sMax)
{
    const R half = R(0.5);
    const R rhoL = qL[0], uL = wL.u, vL = wL.v, pL = wL.p;
    const R rvL0 = rhoL * uL, rvL1 = rhoL * vL;
    const R rhoR = qR[0], uR = wR.u, vR = wR.v, pR = wR.p;
    const R rvR0 = rhoR * uR, rvR1 = rhoR * vR;
    const R rho = root<FAST, R>(rhoL * rhoR);
    const R sL = root<FAST, R>(rhoL), sR = root<FAST, R>(rhoR);
    const Div<FAST, R> mean(sL + sR);
    const R vel0 = mean(sL * uL + sR * uR);
    const R vel1 = mean(sL * vL + sR * vR);
    const R u = vel0 * n0 + vel1 * n1;
    const R p = mean(sL * pL + sR * pR);
    const R a = root<FAST, R>(R(G_) * Div<FAST, R>(rho)(p));
    const R dRhoV0 = rvR0 - rvL0, dRhoV1 = rvR1 - rvL1;
    const R dRho = rhoR - rhoL, dRhoE = qR[3] - qL[3];
    const R eps = R(0.01) * a;
    const R lam1 = harten<R>(fabs(u + a), eps);
    const R lam2 = harten<R>(fabs(u - a), eps);
    const R lam3 = harten<R>(fabs(u), eps);
    const R lam4 = harten<R>(fabs(u), eps);
    const R sm = dmax<R>(dmax<R>(dmax<R>(fabs(lam1), fabs(lam2)), fabs(lam3)), fabs(lam4));
    sMax = sm;
    R fL[4], fR[4];
    convective<R>(pL, uL, vL, rhoL, qL[3], n0, n1, fL);
    convective<R>(pR, uR, vR, rhoR, qR[3], n0, n1, fR);
    R d[4];
    if constexpr (FAST) {
        const R z = FastRange<R>::holds(a, rhoL, rhoR) ? sm : R(NAN);
        d[0] = z * dRho; d[1] = z * dRhoV0; d[2] = z * dRhoV1; d[3] = z * dRhoE;
    } else {
        const R hL = wL.rho(qL[3] + pL), hR = wR.rho(qR[3] + pR);
        const R h = (sL * hL + sR * hR) / (sL + sR);
        const R s1 = half * (sm + sm), s2 = half * (sm - sm);
        const R qq = sqrt(vel0 * vel0 + vel1 * vel1);
        const R G1 = R(G_ - 1) * ((qq * qq / R(2)) * dRho - (vel0 * dRhoV0 + vel1 * dRhoV1) + dRhoE);
        const R G2 = -u * dRho + (dRhoV0 * n0 + dRhoV1 * n1);
        const R C1 = (G1 / (a * a)) * (s1 - sm) + G2 / a * s2;
        const R C2 = (G1 / a) * s2 + (s1 - sm) * G2;
        d[0] = sm * dRho + C1;
        d[1] = sm * (dRhoV0) + C1 * vel0 + C2 * n0;
        d[2] = sm * (dRhoV1) + C1 * vel1 + C2 * n1;
        d[3] = sm * dRhoE + C1 * h + C2 * u;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) out[k] = half * (fL[k] + fR[k]) - half * d[k];
}

template <int FLUX, int FAST, typename R>
DEV void numFlux(const R qL[4], const Prim<FAST, R>& wL, const R qR[4], const Prim<FAST, R>& wR, R n0, R n1, R out[4],
                 R& sMax)
{
    if (FLUX == 1) roeFlux<FAST, R>(qL, wL, qR, wR, n0, n1, out, sMax);
    else rusanovFlux<FAST, R>(qL, wL, qR, wR, n0, n1, out, sMax);
}
template <int FLUX, typename R>
DEV void numFlux(const R qL[4], const R qR[4], R n0, R n1, R out[4], R& sMax)
{
    numFlux<FLUX, 0, R>(qL, Prim<0, R>(qL), qR, Prim<0, R>(qR), n0, n1, out, sMax);
}

// flux.d:28-64.  The four 4x4 matrices are applied entry by entry in column
// order; their structural zeros only ever add a signed zero, so they are skipped.
// Pr and mu are physical parameters (FP64), converted to R.
template <typename R, int FAST = 0>
DEV void viscousFlux(double Prd, double mud, const R q[4], const R dq[8], R n0, R n1, R out[4])
{
    const Div<FAST, R> rho(q[0]);
    const R u = rho(q[1]), v = rho(q[2]), E = rho(q[3]);
    const R gp = R(G_) / R(Prd);
    const R s = rho(R(mud));
    const R one = R(1.0);
    const R c43 = R(4.0 / 3.0), c23 = R(2.0 / 3.0), cm43 = R(-4.0 / 3.0), cm23 = R(-2.0 / 3.0), c231 = R(2.0 / 3.0 - 1.0);
    const R t0 = (cm43 + gp) * (u * u) + (-one + gp) * (v * v) - gp * E;
    const R t1 = (-one + gp) * (u * u) + (cm43 + gp) * (v * v) - gp * E;
    const R x0 = dq[0], x1 = dq[2], x2 = dq[4], x3 = dq[6];
    const R y0 = dq[1], y1 = dq[3], y2 = dq[5], y3 = dq[7];
    const R uv = c231 * u * v;
    const R G01 = ((s * (cm43 * u)) * x0 + (s * c43) * x1) + ((s * (c23 * v)) * y0 + (s * cm23) * y2);
    const R G02 = ((s * -v) * x0 + (s * one) * x2) + ((s * -u) * y0 + (s * one) * y1);
    const R G03 = ((s * t0) * x0 + (s * ((c43 - gp) * u)) * x1 + (s * ((one - gp) * v)) * x2 + (s * gp) * x3)
                + ((s * uv) * y0 + (s * v) * y1 + (s * (cm23 * u)) * y2);
    const R G11 = ((s * -v) * x0 + (s * one) * x2) + ((s * -u) * y0 + (s * one) * y1);
    const R G12 = ((s * (c23 * u)) * x0 + (s * cm23) * x2) + ((s * (cm43 * v)) * y0 + (s * c43) * y2);
    const R G13 = ((s * uv) * x0 + (s * (cm23 * v)) * x1 + (s * u) * x2)
                + ((s * t1) * y0 + (s * ((one - gp) * u)) * y1 + (s * ((c43 - gp) * v)) * y2 + (s * gp) * y3);
    out[0] = R(0.0);
    out[1] = G01 * n0 + G11 * n1;
    out[2] = G02 * n0 + G12 * n1;
    out[3] = G03 * n0 + G13 * n1;
}

DEV void ld4(const double4* p, uint32_t i, double o[4])
{
    const double4 t = p[i];
    o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
}
DEV void st4(double4* p, uint32_t i, const double o[4]) { p[i] = make_double4(o[0], o[1], o[2], o[3]); }
// gradients and limiters are read once, by the next kernel: stored non-temporally so
// they do not displace the neighbour data that kernel's gathers reuse from L2
typedef double ntd2 __attribute__((ext_vector_type(2)));
typedef float ntf4 __attribute__((ext_vector_type(4)));

// the FP32 shadow of a state row (mixed path): the stage's gathers read it in place of the FP64 row
DEV void ld4(const float4* p, uint32_t i, float o[4])
{
    const float4 t = p[i];
    o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
}
DEV void st4(float4* p, uint32_t i, const float o[4]) { p[i] = make_float4(o[0], o[1], o[2], o[3]); }

// ghost state from the owner state (solve.d:520-689); the owner is the only writer
// false where the reference would stop: a total-conditions inflow with no non-negative Mach
// root (solve.d:661-670)
template <typename R>
DEV bool ghostState(const BFace& b, const R qo[4], R qg[4], const R qgOld[4])
{
    const R g = R(G_), gm1 = R(G_ - 1), half = R(0.5), two = R(2.0);
    switch (b.type) {
    case BT_DIRICHLET:
        qg[0] = R(b.gq[0]); qg[1] = R(b.gq[1]); qg[2] = R(b.gq[2]); qg[3] = R(b.gq[3]);
        break;
    case BT_INVWALL:
    case BT_SYM: {
        const R v0 = qo[1] / qo[0], v1 = qo[2] / qo[0];
        R w0, w1;
        if (!b.vertical) {
            w0 = R(0.0) + R(b.R[0]) * v0 + R(b.R[1]) * v1;
            w1 = R(0.0) + R(b.R[2]) * v0 + R(b.R[3]) * v1;
        } else {
            w0 = -v0;
            w1 = v1;
        }
        qg[0] = qo[0]; qg[1] = qo[0] * w0; qg[2] = qo[0] * w1; qg[3] = qo[3];
        break;
    }
    case BT_VISCWALL:
        qg[0] = qo[0]; qg[1] = -qo[1]; qg[2] = -qo[2]; qg[3] = qo[3];
        break;
    case BT_CONSTP: {
        const R rhop = qo[0], up = qo[1] / qo[0], vp = qo[2] / qo[0];
        const R pp = pressure<R>(qo);
        const R ap = sqrt(g * (pp / rhop));
        const R Jp = up + (two * ap) / gm1;
        const R Sp = pp / pow(rhop, g);
        const R pb = R(b.data[0]);
        const R rhob = pow(pb / Sp, R(1.0) / g);
        const R ab = sqrt(g * (pb / rhob));
        const R ub = Jp - (two * ab) / gm1;
        const R vb = vp;
        const R mag = sqrt(ub * ub + vb * vb);
        const R rEb = pb / gm1 + half * rhob * (mag * mag);
        const R n0 = R(b.nrm[0]), n1 = R(b.nrm[1]);
        const R vpn = up * n0 + vp * n1, vbn = ub * n0 + vb * n1;
        qg[0] = rhob;
        qg[1] = rhob * (up - vpn * n0 + vbn * n0);
        qg[2] = rhob * (vp - vpn * n1 + vbn * n1);
        qg[3] = rEb;
        break;
    }
    case BT_TPIN: {
        // solve.d:625-683, including its four writes to component 0
        const R Tt = R(b.data[0]), Pt = R(b.data[1]), ni0 = R(b.data[2]), ni1 = R(b.data[3]);
        const R rhop = qo[0], up = qo[1] / qo[0];
        const R pp = pressure<R>(qo);
        const R ap = sqrt(g * (pp / rhop));
        const R Jp = up + (two * ap) / gm1;
        const R d = ni0 * R(b.nrm[0]) + ni1 * R(b.nrm[1]);
        const R Rg = R(b.Rgas);
        const R A = g * Rg * Tt * (d * d) - half * gm1 * (Jp * Jp);
        const R B = (R(4.0) * g * Rg * Tt * d) / gm1;
        const R Cc = (R(4.0) * g * Rg * Tt) / (gm1 * gm1) - Jp * Jp;
        const R M1 = (-B + sqrt(B * B - R(4) * A * Cc)) / (two * A);
        const R M2 = (-B - sqrt(B * B - R(4) * A * Cc)) / (two * A);
        R Mb = R(NAN);
        bool rootFound = true;
        if (M1 >= 0 && M2 >= 0) Mb = fmin(M1, M2);
        else if (M1 >= 0 && M2 < 0) Mb = M1;
        else if (M1 < 0 && M2 >= 0) Mb = M2;
        else rootFound = false;   // the reference stops here (enforce)
        const R Tb = Tt / (R(1) + half * gm1 * (Mb * Mb));
        const R pb = Pt * pow(Tb / Tt, g / gm1);
        const R rhob = pb / (Rg * Tb);
        const R ab = sqrt(g * (pb / rhob));
        const R vb0 = Mb * ab * ni0, vb1 = Mb * ab * ni1;
        const R mag = sqrt(vb0 * vb0 + vb1 * vb1);
        qg[0] = pb / gm1 + half * rhob * (mag * mag);
        qg[1] = qgOld[1]; qg[2] = qgOld[2]; qg[3] = qgOld[3];
        return rootFound;
    }
    default:  // FullState
        qg[0] = qo[0]; qg[1] = qo[1]; qg[2] = qo[2]; qg[3] = qo[3];
        break;
    }
    return true;
}

// solve.d:27-173 LP vector limiter: the all-inequality simplex of one variable's problem (at
// most 16 pivots), rows in the reference's order: x >= 0, y >= 0, -x >= -1, -y >= -1, then per
// real neighbour j  (ex_j, ey_j).(x, y) >= lo  and  (-ex_j, -ey_j).(x, y) >= hi.
// Held in registers: the rows come in pairs of opposite sign, so a pivot direction decreases at
// most one row of a pair and each pair costs one product sum and one quotient ((-a)p + (-b)q is
// -(ap + bq) exactly).  The first row of the smallest ratio is kept while the pairs go by, with
// its coefficients, instead of being looked up in arrays of rows, ratios and candidates (which
// lived in scratch memory).  The gradient launch of 10,414 triangles: 88 -> 29 us, and 10 with a lane
// per variable (gradientSplitBody).
template <int S>
DEV void lpSolve(const double ex[S], const double ey[S], const bool real[S], double lo, double hi, double c0, double c1,
                 double& x, double& y)
{
    int W0 = 0, W1 = 1;
    double a00 = 1, a01 = 0, a10 = 0, a11 = 1;   // the two working rows
    for (int k = 0; k <= 15; k++) {
        const double det = a00 * a11 - a01 * a10;
        const double s = 1.0 / det;
        const double i0 = a11 * s, i1 = -a01 * s, i2 = -a10 * s, i3 = a00 * s;
        const double lam0 = 0.0 + i0 * c0 + i2 * c1;
        const double lam1 = 0.0 + i1 * c0 + i3 * c1;
        if ((lam0 >= -10e-9) && (lam1 >= -10e-9)) break;
        const int q = (lam0 < lam1) ? W0 : W1;
        const double e0 = (lam0 < lam1) ? 1.0 : 0.0, e1 = (lam0 < lam1) ? 0.0 : 1.0;
        const double p0 = 0.0 + i0 * e0 + i1 * e1;
        const double p1 = 0.0 + i2 * e0 + i3 * e1;
        double alpha = INFINITY, t0 = 1, t1 = 0;
        int t = 0;
        bool found = false;
        // rows r (a, b, right side bp) and rm (na, nb = -a, -b, right side bm)
        auto pair = [&](int r, int rm, double a, double b, double na, double nb, double bp, double bm) {
            const double v = a * p0 + b * p1;
            const bool dn = v < -1e-11 && r != W0 && r != W1;
            const bool up = -v < -1e-11 && rm != W0 && rm != W1;
            if (!dn && !up) return;
            const double u = a * x + b * y;
            const double g = (dn ? u - bp : -u - bm) / (dn ? -v : v);
            const int i = dn ? r : rm;
            if (g < alpha || (g == alpha && (!found || i < t))) {
                alpha = g;
                t = i;
                t0 = dn ? a : na;
                t1 = dn ? b : nb;
                found = true;
            }
        };
        pair(0, 2, 1.0, 0.0, -1.0, 0.0, 0.0, -1.0);
        pair(1, 3, 0.0, 1.0, 0.0, -1.0, 0.0, -1.0);
#pragma unroll
        for (int j = 0; j < S; j++)
            if (real[j]) pair(4 + 2 * j, 5 + 2 * j, ex[j], ey[j], -ex[j], -ey[j], lo, hi);
        if (q == W0) { W0 = t; a00 = t0; a01 = t1; }
        else if (q == W1) { W1 = t; a10 = t0; a11 = t1; }
        x = x + alpha * p0;
        y = y + alpha * p1;
    }
}

// ---------------------------------------------------------------- gradient + limiter
// solve.d:324-497 for one interior cell, given its own state, its S neighbour
// states (ghosts already filled), LSQ weights, centroids and which slots are real
// neighbours (padding slots repeat the cell).  MODE 1: unlimited; 2: scalar
// limiter; 3: scalar limiter then the LP vector limiter.
// Least-squares weights (A^T A)^-1 A^T with A_j = centroid_j - centroid_i, in the
// operation order of the mesh set-up (source/mesh.d; mesh.cpp), so they equal the
// stored ones bit for bit; the padding slots (A_j = 0) add exact zeros, as the
// set-up's zero rows do.
template <int S>
DEV void lsqWeights(double2 ci, const double2 cn[S], double w[2][S])
{
    double ax[S], ay[S];
#pragma unroll
    for (int j = 0; j < S; j++) { ax[j] = cn[j].x - ci.x; ay[j] = cn[j].y - ci.y; }
    double b00 = 0.0, b01 = 0.0, b10 = 0.0, b11 = 0.0;
#pragma unroll
    for (int j = 0; j < S; j++) {
        b00 += ax[j] * ax[j];
        b01 += ax[j] * ay[j];
        b10 += ay[j] * ax[j];
        b11 += ay[j] * ay[j];
    }
    const double det = b00 * b11 - b01 * b10;
    const double id = 1.0 / det;
    const double i00 = b11 * id, i01 = -b01 * id, i10 = -b10 * id, i11 = b00 * id;
#pragma unroll
    for (int j = 0; j < S; j++) {
        w[0][j] = i00 * ax[j] + i01 * ay[j];
        w[1][j] = i10 * ax[j] + i11 * ay[j];
    }
}

// gm: stored weights ((dir, nbr)-major, stride gstride between entries), or null
// to compute them from the centroids.  Weights and centroid offsets are geometry,
// computed in FP64 and converted to R; the gradient, bounds and limiter are R.
// MODE 4: the Venkatakrishnan limiter at the same test points (neighbour centroids): for
// the unlimited increment t = grad . (x_j - x_i) and the bound difference d = max - q_i (t > 0)
// or min - q_i (t < 0), phi_j = [(d^2 + eps2) t + 2 t^2 d] / (t [d^2 + 2 t^2 + d t + eps2]),
// phi = min(1, min_j phi_j); eps2 = (K d_cell)^3 (FP64, passed in).
// V: the variables of this lane (all four, or one of them: each is independent of the others).
template <int S, int MODE, typename R, int V = 4>
DEV void gradLimit(const R qi[V], const R qn[S][V], const double* gm, uint32_t gstride, double2 ci,
                   const double2 cn[S], const bool real[S], int limit, double lpThresh, R g[V][2], R lx[V],
                   R ly[V], double eps2d = 0.0)
{
    static_assert(MODE != 3 || sizeof(R) == 8, "the LP vector limiter runs in FP64 only");
    R w[2][S];
    {
        double wd[2][S];
        if (gm) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int j = 0; j < S; j++) wd[r][j] = gm[(r * S + j) * gstride];
        } else {
            lsqWeights<S>(ci, cn, wd);
        }
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int j = 0; j < S; j++) w[r][j] = R(wd[r][j]);
    }
    R mn[V], mx[V], du[V][S];
#pragma unroll
    for (int k = 0; k < V; k++) { mn[k] = qi[k]; mx[k] = qi[k]; }
#pragma unroll
    for (int j = 0; j < S; j++)
#pragma unroll
        for (int k = 0; k < V; k++) {
            mn[k] = fmin(mn[k], qn[j][k]);
            mx[k] = fmax(mx[k], qn[j][k]);
            du[k][j] = qn[j][k] - qi[k];
        }
#pragma unroll
    for (int k = 0; k < V; k++)
#pragma unroll
        for (int r = 0; r < 2; r++) {
            R s = R(0.0);
#pragma unroll
            for (int j = 0; j < S; j++) s += w[r][j] * du[k][j];
            g[k][r] = s;
        }
#pragma unroll
    for (int k = 0; k < V; k++) { lx[k] = R(1.0); ly[k] = R(1.0); }
    if (MODE == 4 && limit) {
        const R eps2 = R(eps2d), two = R(2.0);
#pragma unroll
        for (int j = 0; j < S; j++) {
            const R dx = R(cn[j].x - ci.x), dy = R(cn[j].y - ci.y);
#pragma unroll
            for (int k = 0; k < V; k++) {
                const R t = g[k][0] * dx + g[k][1] * dy;
                R s = R(1.0);
                if (t != R(0.0)) {
                    const R d = t > R(0.0) ? mx[k] - qi[k] : mn[k] - qi[k];
                    s = ((d * d + eps2) * t + two * (t * t) * d) / (t * (d * d + two * (t * t) + d * t + eps2));
                }
                lx[k] = fmin(lx[k], s);
                ly[k] = lx[k];
            }
        }
        return;
    }
    if (MODE >= 2 && MODE <= 3 && limit) {
        R dxs[S], dys[S];
#pragma unroll
        for (int j = 0; j < S; j++) {
            const R dx = R(cn[j].x - ci.x), dy = R(cn[j].y - ci.y);
            dxs[j] = dx; dys[j] = dy;
#pragma unroll
            for (int k = 0; k < V; k++) {
                R s = R(1.0);
                const R t = g[k][0] * dx + g[k][1] * dy;
                const R qE = qi[k] + t;
                const bool under = qE < mn[k];
                if (under || qE > mx[k]) s = ((under ? mn[k] : mx[k]) - qi[k]) / t;
                lx[k] = fmin(lx[k], s);
                ly[k] = lx[k];
            }
        }
        if constexpr (MODE == 3) {
            if (lpThresh > 0) {
                int nn = 0;
#pragma unroll
                for (int j = 0; j < S; j++) nn += real[j] ? 1 : 0;
                // one copy of the simplex's code for the four variables, whose values are
                // selected instead of indexed (an indexed array would live in scratch)
                auto sel = [](int k, const double v[V]) {
                    if constexpr (V == 4) return k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
                    else return v[0];
                };
                double g0s[V], g1s[V];
#pragma unroll
                for (int k = 0; k < V; k++) { g0s[k] = g[k][0]; g1s[k] = g[k][1]; }
#pragma unroll 1
                for (int k = 0; k < V; k++) {
                    if (!(sel(k, lx) < lpThresh && (nn == 3 || nn == 4))) continue;
                    const double g0 = sel(k, g0s);
                    const double g1 = sel(k, g1s);
                    const double q = sel(k, qi);
                    double ex[S], ey[S];
#pragma unroll
                    for (int j = 0; j < S; j++) { ex[j] = dxs[j] * g0; ey[j] = dys[j] * g1; }
                    double x = 0.0, y = 0.0;
                    lpSolve<S>(ex, ey, real, sel(k, mn) - q, q - sel(k, mx),
                               -fabs(g0), -fabs(g1), x, y);
#pragma unroll
                    for (int c = 0; c < V; c++) {
                        lx[c] = c == k ? x : lx[c];
                        ly[c] = c == k ? y : ly[c];
                    }
                }
            }
        }
    }
}

// the owner's ghost state for boundary record b, with TempPresInflow's untouched components
DEV bool ghostFromOwner(const BFace& bf, const double qo[4], const double4* qbuf, uint32_t gIdx, double qg[4])
{
    double old[4] = {0, 0, 0, 0};
    if (bf.type == BT_TPIN) ld4(qbuf, gIdx, old);
    return ghostState(bf, qo, qg, old);
}

// MODE 0: ghost states only (order 1); 1: unlimited gradient (no limiter stored);
// 2: scalar limiter; 3: scalar limiter followed by the LP vector limiter (lim
// stored as x,y pairs).
// MIX 0: FP64 throughout.  MIX 1 (mixed precision): states are read from the FP32
// shadows, ghosts, gradients and limiters computed in FP32 (least-squares weights and
// centroid offsets in FP64, converted); gradients and limiters are stored as FP32
// rows (32 + 16 bytes per cell); each ghost is written to the shadow and, widened, to
// the FP64 row.
// LDS of one gradient workgroup: staging of the gradient rows and of the limiter rows
template <int MODE>
struct GradLds {
    static constexpr int LWS = (MODE == 2 || MODE == 4) ? 4 : 0;
    double sg[BLK][9];
    double sl[BLK][LWS + 1];
};

template <int MIX>
using RealOf = typename std::conditional<MIX == 1, float, double>::type;

// a stage-input row: the FP32 shadow on the mixed path
template <int MIX>
DEV void ldStage(const StageArgs& a, uint32_t c, RealOf<MIX> o[4])
{
    if constexpr (MIX == 1) ld4(a.qin32, c, o);
    else ld4(a.qin, c, o);
}
// a ghost row of the stage input; the mixed path also widens it into the FP64 row
template <int MIX>
DEV void stGhostRow(const StageArgs& a, uint32_t c, const RealOf<MIX> o[4])
{
    if constexpr (MIX == 1) {
        st4(a.qin32, c, o);
        a.qin[c] = make_double4(o[0], o[1], o[2], o[3]);
    } else {
        st4(a.qin, c, o);
    }
}

// Gradient and limiter of interior cell i (MODE 1-4) from the stage input, with the ghost
// states of its boundary faces, which are stored to the stage buffer where storeGhosts;
// nbrRow: its S neighbour ids (the mesh's row, or a tile's copy of it).
// Every neighbour row is loaded before any ghost is written, so the loads of all
// neighbours are in flight together.  A ghost slot belongs to this cell alone (the owner of
// its boundary face), so its row still holds the stage buffer's previous ghost state, which
// TempPresInflow keeps in the components it does not write.
template <int S, int MODE, int MIX>
DEV void cellGradient(const DevMesh& m, const PhysParams& p, const StageArgs& a, uint32_t i, const uint32_t* nbrRow,
                      bool storeGhosts, RealOf<MIX> g[4][2], RealOf<MIX> lx[4], RealOf<MIX> ly[4])
{
    using R = RealOf<MIX>;
    R qi[4];
    ldStage<MIX>(a, i, qi);
    uint32_t nb[S];
#pragma unroll
    for (int j = 0; j < S; j++) nb[j] = nbrRow[j];
    R qn[S][4];
    double2 cn[S];
#pragma unroll
    for (int j = 0; j < S; j++) { ldStage<MIX>(a, nb[j], qn[j]); cn[j] = m.cen[nb[j]]; }
    const double2 ci = m.cen[i];
#pragma unroll
    for (int j = 0; j < S; j++)
        if (nb[j] >= m.N) {
            const BFace& bf = m.bface[nb[j] - m.N];
            if (storeGhosts && a.ghostSave)
                a.ghostSave[nb[j] - m.N] = make_double4(qn[j][0], qn[j][1], qn[j][2], qn[j][3]);
            R old[4] = {0, 0, 0, 0};
            if (bf.type == BT_TPIN) {
#pragma unroll
                for (int k = 0; k < 4; k++) old[k] = qn[j][k];
            }
            if (!ghostState<R>(bf, qi, qn[j], old) && a.recordErrors)
                atomicMin(&a.sc->errBC, (uint64_t(a.stageId) << 32) | (nb[j] - m.N));
            if (storeGhosts) stGhostRow<MIX>(a, nb[j], qn[j]);
        }
    bool real[S];
#pragma unroll
    for (int j = 0; j < S; j++) real[j] = nb[j] != i;
    double eps2 = 0.0;
    if constexpr (MODE == 4) {
        const double kd = p.venkatK * m.cd[i];
        eps2 = kd * kd * kd;
    }
    gradLimit<S, MODE, R>(qi, qn, nullptr, 0, ci, cn, real, a.limit, p.lpThresh, g, lx, ly, eps2);
}

// whether a stage's gradient kernel runs
DEV bool stageRuns(const StageArgs& a)
{
    return !a.checkActive || (a.spec ? a.sc->specActive : a.sc->active);
}

// What one thread of a stage's gradient kernel sets before the stage's other kernels.  Rmax is per step
// (the time loop's epilogue takes it from the stages' partials instead).  A launch of its own in front
// of a residual or step call took 5 us.
DEV void stageBegin(const StageArgs& a)
{
    if (a.first && !a.checkActive) a.sc->rmaxBits = 0;
    if (a.callBegin) {
        a.sc->rmaxBits = a.callRmax;
        if (a.callSetDt) {
            a.sc->loopDt = a.sc->dt;
            a.sc->dt = a.callDt;
        }
    }
}

// whether the tile or face kernel of a stage runs; one thread of a step's first one passes a loop
// that has ended on to the next step's gradient kernel
DEV bool fluxRuns(const StageArgs& a, bool first)
{
    if (!a.checkActive || a.sc->active) return true;
    if (first && a.spec) a.sc->specActive = 0;
    return false;
}

// One workgroup of the gradient kernel on cell block `bid` of its mesh (the solo and the
// batched kernels run this same code).  Not MODE 3: the LP limiter runs in gradientSplitBody.
template <int S, int MODE, int MIX>
DEV void gradientBody(const DevMesh& m, const PhysParams& p, const StageArgs& a, uint32_t bid, GradLds<MODE>& L)
{
    using R = RealOf<MIX>;
    constexpr int LWS = GradLds<MODE>::LWS;
    auto& sg = L.sg;
    auto& sl = L.sl;
    if (!stageRuns(a)) return;
    if (bid == 0 && threadIdx.x == 0) stageBegin(a);
    const uint32_t i = bid * BLK + threadIdx.x;
    if (MODE == 0 && i >= m.N) return;
    const bool have = i < m.N;   // no early return below: the staged stores need every thread
    R g[4][2], lx[4], ly[4];
    if (have) {
        if constexpr (MODE == 0) {
            // order 1: the ghost states are the kernel's only output
            R qi[4];
            ldStage<MIX>(a, i, qi);
#pragma unroll
            for (int j = 0; j < S; j++) {
                const uint32_t nb = m.nbr[i * S + j];
                if (nb >= m.N) {
                    const BFace& bf = m.bface[nb - m.N];
                    R qg[4], old[4] = {0, 0, 0, 0};
                    if (bf.type == BT_TPIN || a.ghostSave) ldStage<MIX>(a, nb, old);
                    if (a.ghostSave) a.ghostSave[nb - m.N] = make_double4(old[0], old[1], old[2], old[3]);
                    if (!ghostState<R>(bf, qi, qg, old) && a.recordErrors)
                        atomicMin(&a.sc->errBC, (uint64_t(a.stageId) << 32) | (nb - m.N));
                    stGhostRow<MIX>(a, nb, qg);
                }
            }
            return;
        } else {
            cellGradient<S, MODE, MIX>(m, p, a, i, m.nbr + size_t(i) * S, true, g, lx, ly);
        }
    }
    if (MODE == 0) return;
    // stage the rows in LDS and store the workgroup's contiguous run of cells with
    // lane-consecutive 16-byte stores
    const uint32_t tid = threadIdx.x;
    const uint32_t base = bid * BLK, n = (m.N - base) < BLK ? (m.N - base) : BLK;
    if constexpr (MIX == 1) {
        float* fg = reinterpret_cast<float*>(&sg[0][0]);   // 8 floats per row
        float* fl = reinterpret_cast<float*>(&sl[0][0]);   // 4 floats per row
        if (have) {
#pragma unroll
            for (int c = 0; c < 4; c++) { fg[8 * tid + 2 * c] = g[c][0]; fg[8 * tid + 2 * c + 1] = g[c][1]; }
            if (MODE == 2 || MODE == 4) {
#pragma unroll
                for (int c = 0; c < 4; c++) fl[4 * tid + c] = lx[c];
            }
        }
        __syncthreads();
        float4* gd = reinterpret_cast<float4*>(a.grad32 + size_t(base) * 8);
        for (uint32_t c = tid; c < 2 * n; c += BLK)
            __builtin_nontemporal_store(*reinterpret_cast<const ntf4*>(fg + 4 * c), reinterpret_cast<ntf4*>(gd) + c);
        if (MODE == 2 || MODE == 4) {
            float4* ld = reinterpret_cast<float4*>(a.lim32 + size_t(base) * 4);
            for (uint32_t c = tid; c < n; c += BLK)
                __builtin_nontemporal_store(*reinterpret_cast<const ntf4*>(fl + 4 * c), reinterpret_cast<ntf4*>(ld) + c);
        }
        return;
    } else {
        if (have) {
#pragma unroll
            for (int c = 0; c < 4; c++) { sg[tid][2 * c] = g[c][0]; sg[tid][2 * c + 1] = g[c][1]; }
            if (MODE == 2 || MODE == 4) {
#pragma unroll
                for (int c = 0; c < 4; c++) sl[tid][c] = lx[c];
            }
        }
        __syncthreads();
        double2* gd = reinterpret_cast<double2*>(a.grad + size_t(base) * 8);
        for (uint32_t c = tid; c < 4 * n; c += BLK) __builtin_nontemporal_store((ntd2){sg[c / 4][2 * (c % 4)], sg[c / 4][2 * (c % 4) + 1]}, reinterpret_cast<ntd2*>(gd) + c);
        if constexpr (LWS > 0) {
            double2* ld = reinterpret_cast<double2*>(a.lim + size_t(base) * LWS);
            constexpr uint32_t PR = LWS / 2;
            for (uint32_t c = tid; c < PR * n; c += BLK) __builtin_nontemporal_store((ntd2){sl[c / PR][2 * (c % PR)], sl[c / PR][2 * (c % PR) + 1]}, reinterpret_cast<ntd2*>(ld) + c);
        }
    }
    // MODE 1 (unlimited stage): every limiter is 1; the face kernels take LP = 2 and read none
}

// One workgroup of the gradient kernel with LANES lanes per cell (4: a variable each, 2: two each) on
// block `bid` of BLK / LANES cells: the variables' gradients, bounds and limiters do not depend on each
// other (a boundary cell's lanes each form the whole ghost state), and a cell's row of four is still one
// access.  More workgroups with a shorter chain and fewer registers each, for meshes that do not fill
// the chip many times over.
template <int S, int MODE, int MIX, int LANES>
DEV void gradientSplitBody(const DevMesh& m, const PhysParams& p, const StageArgs& a, uint32_t bid)
{
    using R = RealOf<MIX>;
    constexpr int V = 4 / LANES;
    typedef R rowV __attribute__((ext_vector_type(V == 1 ? 2 : V)));
    if (!stageRuns(a)) return;
    if (bid == 0 && threadIdx.x == 0) stageBegin(a);
    const uint32_t i = bid * (BLK / LANES) + threadIdx.x / LANES, v = threadIdx.x % LANES * V;
    if (i >= m.N) return;
    const R* rows;
    if constexpr (MIX == 1) rows = reinterpret_cast<const R*>(a.qin32);
    else rows = reinterpret_cast<const R*>(a.qin);
    uint32_t nb[S];
#pragma unroll
    for (int j = 0; j < S; j++) nb[j] = m.nbr[size_t(i) * S + j];
    auto ldRow = [&](uint32_t c, R o[V]) {
        if constexpr (V == 2) {
            const rowV x = *reinterpret_cast<const rowV*>(rows + size_t(c) * 4 + v);
            o[0] = x[0];
            o[1] = x[1];
        } else {
            o[0] = rows[size_t(c) * 4 + v];
        }
    };
    R qi[V], qn[S][V];
    ldRow(i, qi);
    double2 cn[S];
#pragma unroll
    for (int j = 0; j < S; j++) { ldRow(nb[j], qn[j]); cn[j] = m.cen[nb[j]]; }
    const double2 ci = m.cen[i];
#pragma unroll
    for (int j = 0; j < S; j++)
        if (nb[j] >= m.N) {   // as in cellGradient; the first lane stores
            const uint32_t b = nb[j] - m.N;
            const BFace& bf = m.bface[b];
            R qo[4], qg[4], was[4], old[4] = {0, 0, 0, 0};
            ldStage<MIX>(a, i, qo);
            ldStage<MIX>(a, nb[j], was);
            if (bf.type == BT_TPIN) {
#pragma unroll
                for (int k = 0; k < 4; k++) old[k] = was[k];
            }
            const bool ok = ghostState<R>(bf, qo, qg, old);
            if (v == 0) {
                if (a.ghostSave) a.ghostSave[b] = make_double4(was[0], was[1], was[2], was[3]);
                if (!ok && a.recordErrors) atomicMin(&a.sc->errBC, (uint64_t(a.stageId) << 32) | b);
                stGhostRow<MIX>(a, nb[j], qg);
            }
            if constexpr (V == 2) {
                qn[j][0] = v ? qg[2] : qg[0];
                qn[j][1] = v ? qg[3] : qg[1];
            } else {
                qn[j][0] = v == 0 ? qg[0] : v == 1 ? qg[1] : v == 2 ? qg[2] : qg[3];
            }
        }
    bool real[S];
#pragma unroll
    for (int j = 0; j < S; j++) real[j] = nb[j] != i;
    double eps2 = 0.0;
    if constexpr (MODE == 4) {
        const double kd = p.venkatK * m.cd[i];
        eps2 = kd * kd * kd;
    }
    R g[V][2], lx[V], ly[V];
    gradLimit<S, MODE, R, V>(qi, qn, nullptr, 0, ci, cn, real, a.limit, p.lpThresh, g, lx, ly, eps2);
    const size_t o = size_t(i) * 4 + v;
    if constexpr (MIX == 1 && V == 2) {
        __builtin_nontemporal_store((ntf4){g[0][0], g[0][1], g[1][0], g[1][1]}, reinterpret_cast<ntf4*>(a.grad32 + 2 * o));
        if (MODE == 2 || MODE == 4) *reinterpret_cast<float2*>(a.lim32 + o) = make_float2(lx[0], lx[1]);
    } else if constexpr (V == 2) {
        ntd2* gd = reinterpret_cast<ntd2*>(a.grad) + o;
        __builtin_nontemporal_store((ntd2){g[0][0], g[0][1]}, gd);
        __builtin_nontemporal_store((ntd2){g[1][0], g[1][1]}, gd + 1);
        if (MODE == 2 || MODE == 4) __builtin_nontemporal_store((ntd2){lx[0], lx[1]}, reinterpret_cast<ntd2*>(a.lim + o));
    } else if constexpr (MIX == 1) {
        reinterpret_cast<float2*>(a.grad32)[o] = make_float2(g[0][0], g[0][1]);
        if (MODE == 2 || MODE == 4) a.lim32[o] = lx[0];
    } else {
        reinterpret_cast<double2*>(a.grad)[o] = make_double2(g[0][0], g[0][1]);
        if (MODE == 3) reinterpret_cast<double2*>(a.lim)[o] = make_double2(lx[0], ly[0]);
        else if (MODE == 2 || MODE == 4) a.lim[o] = lx[0];
    }
}

// ---------------------------------------------------------------- faces
// LP 0: scalar limiter (4 per cell); 1: LP vector limiter (x,y pairs); 2: an
// unlimited stage, every limiter 1 (1*g is exactly g, so the products round as with
// stored ones)
template <int LP>
DEV void loadLim(const double* lim, uint32_t c, double lx[4], double ly[4])
{
    if (LP == 2) {
#pragma unroll
        for (int k = 0; k < 4; k++) { lx[k] = 1.0; ly[k] = 1.0; }
    } else if (LP) {
        const double4 a = *reinterpret_cast<const double4*>(lim + size_t(c) * 8);
        const double4 b = *reinterpret_cast<const double4*>(lim + size_t(c) * 8 + 4);
        lx[0] = a.x; ly[0] = a.y; lx[1] = a.z; ly[1] = a.w; lx[2] = b.x; ly[2] = b.y; lx[3] = b.z; ly[3] = b.w;
    } else {
        const double4 a = *reinterpret_cast<const double4*>(lim + size_t(c) * 4);
        lx[0] = ly[0] = a.x; lx[1] = ly[1] = a.y; lx[2] = ly[2] = a.z; lx[3] = ly[3] = a.w;
    }
}
// FP32 rows of the mixed path (no LP vector limiter there)
template <int LP>
DEV void loadLim(const float* lim, uint32_t c, float lx[4], float ly[4])
{
    static_assert(LP != 1, "the LP vector limiter runs in FP64 only");
    if (LP == 2) {
#pragma unroll
        for (int k = 0; k < 4; k++) { lx[k] = 1.0f; ly[k] = 1.0f; }
    } else {
        const float4 a = *reinterpret_cast<const float4*>(lim + size_t(c) * 4);
        lx[0] = ly[0] = a.x; lx[1] = ly[1] = a.y; lx[2] = ly[2] = a.z; lx[3] = ly[3] = a.w;
    }
}

DEV void loadGrad(const double* grad, uint32_t c, double g[8])
{
    const double4 a = *reinterpret_cast<const double4*>(grad + size_t(c) * 8);
    const double4 b = *reinterpret_cast<const double4*>(grad + size_t(c) * 8 + 4);
    g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w; g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
}
DEV void loadGrad(const float* grad, uint32_t c, float g[8])
{
    const float4 a = *reinterpret_cast<const float4*>(grad + size_t(c) * 8);
    const float4 b = *reinterpret_cast<const float4*>(grad + size_t(c) * 8 + 4);
    g[0] = a.x; g[1] = a.y; g[2] = a.z; g[3] = a.w; g[4] = b.x; g[5] = b.y; g[6] = b.z; g[7] = b.w;
}

// solve.d:980-1010 (interior) reconstruction with the p<0 fallback; w: velocity and pressure of
// the state that it arrives at
template <int LP, int FAST, typename R>
DEV void reconstruct(const R qm[4], const R g[8], const R lx[4], const R ly[4], R dx, R dy, R out[4],
                     Prim<FAST, R>& w)
{
#pragma unroll
    for (int j = 0; j < 4; j++) out[j] = qm[j] + lx[j] * g[2 * j] * dx + ly[j] * g[2 * j + 1] * dy;
    w = Prim<FAST, R>(out);
    if (w.p < 0) {
        R l0 = R(1.0), l1 = R(1.0);
#pragma unroll
        for (int j = 0; j < 4; j++) { l0 = fmin(l0, lx[j]); l1 = fmin(l1, ly[j]); }
#pragma unroll
        for (int j = 0; j < 4; j++) out[j] = qm[j] + l0 * g[2 * j] * dx + l1 * g[2 * j + 1] * dy;
        w = Prim<FAST, R>(out);
    }
}

// solve.d:970-1033: one interior face from both cells' raw data.  Centroids, midpoint
// and normal are FP64 geometry; the offsets and the normal enter the R arithmetic.
template <int FLUX, int VISC, int ORDER, int LP, typename R, int FAST = 0>
DEV void interiorFace(const R qa[4], const R ga[8], const R lxa[4], const R lya[4], double2 ca,
                      const R qb[4], const R gb[8], const R lxb[4], const R lyb[4], double2 cb,
                      double2 n, double2 mid, const PhysParams& p, R qL[4], R qR[4], R F[4], R& sMax)
{
    Prim<FAST, R> wL, wR;
    if (ORDER > 1) {
        reconstruct<LP, FAST, R>(qa, ga, lxa, lya, R(mid.x - ca.x), R(mid.y - ca.y), qL, wL);
        reconstruct<LP, FAST, R>(qb, gb, lxb, lyb, R(mid.x - cb.x), R(mid.y - cb.y), qR, wR);
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) { qL[k] = qa[k]; qR[k] = qb[k]; }
        wL = Prim<FAST, R>(qL);
        wR = Prim<FAST, R>(qR);
    }
    // the face gradient is formed before the convective flux, so the two cell gradients
    // are not live across it
    R dq[8];
    if (VISC) {
#pragma unroll
        for (int k = 0; k < 8; k++) dq[k] = R(0.5) * (ga[k] + gb[k]);
    }
    numFlux<FLUX, FAST, R>(qL, wL, qR, wR, R(n.x), R(n.y), F, sMax);
    if (VISC) {
        R qa2[4], Fv[4];
#pragma unroll
        for (int k = 0; k < 4; k++) qa2[k] = R(0.5) * (qL[k] + qR[k]);
        viscousFlux<R, FAST>(p.Pr, p.mu, qa2, dq, R(n.x), R(n.y), Fv);
#pragma unroll
        for (int k = 0; k < 4; k++) F[k] = F[k] - Fv[k];
    }
}

// solve.d:283-319 + 769-968: one boundary face from its owner's data and ghost state
template <int FLUX, int VISC, int ORDER, int LP, typename R>
DEV void boundaryFace(const R qo[4], const R gO[8], const R lx[4], const R ly[4], double2 co,
                      const R qg[4], const BFace& bf, double2 nd, double2 mid, const PhysParams& p,
                      R qL[4], R qR[4], R F[4], R& sMax)
{
    const R g = R(G_), gm1 = R(G_ - 1), half = R(0.5);
    const R nx = R(nd.x), ny = R(nd.y);
    // updateBoundaryEdge: the fallback uses lim[0] for both directions
    if (ORDER > 1) {
        const R dx = R(mid.x - co.x), dy = R(mid.y - co.y);
#pragma unroll
        for (int j = 0; j < 4; j++) qL[j] = qo[j] + lx[j] * gO[2 * j] * dx + ly[j] * gO[2 * j + 1] * dy;
        if (pressure<R>(qL) < 0) {
            R l0 = R(1.0);
#pragma unroll
            for (int j = 0; j < 4; j++) l0 = fmin(l0, lx[j]);
#pragma unroll
            for (int j = 0; j < 4; j++) qL[j] = qo[j] + l0 * gO[2 * j] * dx + l0 * gO[2 * j + 1] * dy;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) qL[j] = qo[j];
    }
    const int type = bf.type;
    if (type == BT_FULL || type == BT_DIRICHLET) {
#pragma unroll
        for (int k = 0; k < 4; k++) qR[k] = R(bf.far[k]);
        numFlux<FLUX, R>(qL, qR, nx, ny, F, sMax);
        if (VISC) {
            R qa[4], dq[8], Fv[4];
#pragma unroll
            for (int k = 0; k < 4; k++) qa[k] = half * (qL[k] + qR[k]);
            if (type == BT_DIRICHLET) {
#pragma unroll
                for (int k = 0; k < 8; k++) dq[k] = half * (gO[k] + R(bf.gg[k]));
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) dq[k] = half * (gO[k] + R(0.0));
            }
            viscousFlux<R>(p.Pr, p.mu, qa, dq, nx, ny, Fv);
#pragma unroll
            for (int k = 0; k < 4; k++) F[k] = F[k] - Fv[k];
        }
    } else if (type == BT_INVWALL) {
        const R inv = R(1) / qL[0];
        const R v0 = inv * qL[1], v1 = inv * qL[2];
        const R vn = v0 * nx + v1 * ny;
        const R t0 = v0 - vn * nx, t1 = v1 - vn * ny;
        const R vel = sqrt(t0 * t0 + t1 * t1);
        R pw = gm1 * (qL[3] - half * qL[0] * (vel * vel));
        const R aw = sqrt(g * (pw / qL[0]));
        if (pw < 0) pw = R(1.0e-12);
        F[0] = R(0); F[1] = pw * nx; F[2] = pw * ny; F[3] = R(0);
        sMax = fabs(aw);
        for (int k = 0; k < 4; k++) qR[k] = qg[k];
    } else if (type == BT_VISCWALL) {
        const R vel = R(0.0);
        R pw = gm1 * (qL[3] - half * qL[0] * (vel * vel));
        const R aw = sqrt(g * (pw / qL[0]));
        if (pw < 0) pw = R(1.0e-12);
        qR[0] = qL[0]; qR[1] = qL[1] * R(-1); qR[2] = qL[2] * R(-1); qR[3] = qL[3];
        R qa[4], dq[8], Fv[4];
#pragma unroll
        for (int k = 0; k < 4; k++) qa[k] = half * (qL[k] + qR[k]);
        qa[1] = R(0.0); qa[2] = R(0.0);
#pragma unroll
        for (int k = 0; k < 8; k++) dq[k] = gO[k];
        dq[6] = (qa[3] / qa[0]) * dq[0];
        dq[7] = (qa[3] / qa[0]) * dq[1];
        viscousFlux<R>(p.Pr, p.mu, qa, dq, nx, ny, Fv);
        F[0] = R(0) - Fv[0]; F[1] = pw * nx - Fv[1]; F[2] = pw * ny - Fv[2]; F[3] = R(0) - Fv[3];
        sMax = fabs(aw);
    } else if (type == BT_CONSTP) {
        for (int k = 0; k < 4; k++) qR[k] = qg[k];
        const R pg = pressure<R>(qR);
        const R ug = qR[1] / qR[0], vg = qR[2] / qR[0];
        const R ag = sqrt(g * (pg / qR[0]));
        convective<R>(pg, ug, vg, qR[0], qR[3], nx, ny, F);
        sMax = fabs(ag);
    } else if (type == BT_SYM) {
        const R v0 = qL[1] / qL[0], v1 = qL[2] / qL[0];
        R w0, w1;
        if (!bf.vertical) {
            w0 = R(0.0) + R(bf.R[0]) * v0 + R(bf.R[1]) * v1;
            w1 = R(0.0) + R(bf.R[2]) * v0 + R(bf.R[3]) * v1;
        } else {
            w0 = -v0;
            w1 = v1;
        }
        qR[0] = qL[0]; qR[1] = qL[0] * w0; qR[2] = qL[0] * w1; qR[3] = qL[3];
        numFlux<FLUX, R>(qL, qR, nx, ny, F, sMax);
        if (VISC) {
            const R one = R(1), zero = R(0), two = R(2);
            R qa[4], bg[8], Fv[4];
#pragma unroll
            for (int k = 0; k < 4; k++) qa[k] = half * (qL[k] + qR[k]);
            const R o00 = nx * nx, o01 = nx * ny, o10 = ny * nx, o11 = ny * ny;
            const R V00 = one - o00, V01 = zero - o01, V10 = zero - o10, V11 = one - o11;
            const R T00 = one - two * o00, T01 = zero - two * o01, T10 = zero - two * o10, T11 = one - two * o11;
            // tmp1 = A*gradp with A = identity except the momentum block V (4x4 * 4x2, all columns)
            R t1[8];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                t1[0 + c] = zero + one * gO[0 + c] + zero * gO[2 + c] + zero * gO[4 + c] + zero * gO[6 + c];
                t1[2 + c] = zero + zero * gO[0 + c] + V00 * gO[2 + c] + V01 * gO[4 + c] + zero * gO[6 + c];
                t1[4 + c] = zero + zero * gO[0 + c] + V10 * gO[2 + c] + V11 * gO[4 + c] + zero * gO[6 + c];
                t1[6 + c] = zero + zero * gO[0 + c] + zero * gO[2 + c] + zero * gO[4 + c] + one * gO[6 + c];
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const R s30 = zero + t1[2 * r] * T00 + t1[2 * r + 1] * T10;
                const R s31 = zero + t1[2 * r] * T01 + t1[2 * r + 1] * T11;
                const R s10 = zero + gO[2 * r] * o00 + gO[2 * r + 1] * o10;
                const R s11 = zero + gO[2 * r] * o01 + gO[2 * r + 1] * o11;
                bg[2 * r] = s10 + s30;
                bg[2 * r + 1] = s11 + s31;
            }
            viscousFlux<R>(p.Pr, p.mu, qa, bg, nx, ny, Fv);
#pragma unroll
            for (int k = 0; k < 4; k++) F[k] = F[k] - Fv[k];
        }
    } else {  // TempPresInflow
        for (int k = 0; k < 4; k++) qR[k] = qg[k];
        numFlux<FLUX, R>(qL, qR, nx, ny, F, sMax);
        if (VISC) {
            R qa[4], Fv[4];
#pragma unroll
            for (int k = 0; k < 4; k++) qa[k] = half * (qL[k] + qR[k]);
            viscousFlux<R>(p.Pr, p.mu, qa, gO, nx, ny, Fv);
#pragma unroll
            for (int k = 0; k < 4; k++) F[k] = F[k] - Fv[k];
        }
    }
}

// Cell data a face reads: the FP64 rows, or on the mixed path (MIX 1) the FP32
// shadow of the state and the FP32 gradient and limiter rows.
template <int MIX>
struct FaceSrc {
    using R = typename std::conditional<MIX == 1, float, double>::type;
    const StageArgs& a;
    DEV void q(uint32_t c, R o[4]) const
    {
        if constexpr (MIX == 1) ld4(a.qin32, c, o);
        else ld4(a.qin, c, o);
    }
    DEV void grad(uint32_t c, R o[8]) const
    {
        if constexpr (MIX == 1) loadGrad(a.grad32, c, o);
        else loadGrad(a.grad, c, o);
    }
    template <int LP>
    DEV void lim(uint32_t c, R lx[4], R ly[4]) const
    {
        if constexpr (MIX == 1) loadLim<LP>(a.lim32, c, lx, ly);
        else loadLim<LP>(a.lim, c, lx, ly);
    }
};

// ---------------------------------------------------------------- residual + update
// Exchange between lanes of a row of 16 by DPP moves instead of __shfl_xor, whose two LDS permutes per
// double kept the LDS pipe busy for a third of a last stage's cell phase.  ROW_X1 and ROW_X2 swap with
// lane ^ 1 and lane ^ 2; the mirrors reach the other quad of an octet and the other octet of the row,
// whose lanes all hold the same value by then, so they stand for lane ^ 4 and lane ^ 8 of a butterfly.
// Every lane of the wave must be active.
enum { ROW_X1 = 0xB1, ROW_X2 = 0x4E, ROW_X4 = 0x141, ROW_X8 = 0x140 };
template <int CTRL>
DEV double rowSwap(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
DEV double laneValue(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
DEV double warpMin(double v)
{
    v = fmin(v, rowSwap<ROW_X1>(v));
    v = fmin(v, rowSwap<ROW_X2>(v));
    v = fmin(v, rowSwap<ROW_X4>(v));
    v = fmin(v, rowSwap<ROW_X8>(v));
    return fmin(fmin(laneValue(v, 0), laneValue(v, 16)), fmin(laneValue(v, 32), laneValue(v, 48)));
}
DEV double warpMax(double v)
{
    v = fmax(v, rowSwap<ROW_X1>(v));
    v = fmax(v, rowSwap<ROW_X2>(v));
    v = fmax(v, rowSwap<ROW_X4>(v));
    v = fmax(v, rowSwap<ROW_X8>(v));
    return fmax(fmax(laneValue(v, 0), laneValue(v, 16)), fmax(laneValue(v, 32), laneValue(v, 48)));
}

// solve.d:1092-1117 + the integrator's stage update for interior cell i, from
// its summed face fluxes r and sum of len*sMax
// met: (perimeter, d, -1/area) of the cell, or null to read them from the mesh
// qNew/qOld (optional): the new state and q^n when this stage completes a step
// qnI, accI (optional): the cell's q^n and RK accumulator rows already loaded
// the stage output row, and on the mixed path its FP32 shadow for the next stage's gathers
DEV void storeOut(const StageArgs& a, uint32_t i, const double o[4])
{
    st4(a.qout, i, o);
    if (a.qout32) a.qout32[i] = make_float4(float(o[0]), float(o[1]), float(o[2]), float(o[3]));
}

// Whether a stage's CFL time step is used: the last stage's is the step's (every stage overwrites
// it in the reference), a residual call returns its own, and local time steps keep theirs.
DEV bool stageWantsDt(const PhysParams& p, const StageArgs& a)
{
    return a.last || a.kind == SK_RESIDUAL || (p.localTimestep && a.dtUpdate);
}

// wantDt 0: sAve and the first two entries of met are not there
template <int KIND>
DEV void cellStage(const DevMesh& m, const PhysParams& p, const StageArgs& a, uint32_t i, const double r[4],
                   double sAve, const double* qinI, const double* met, double& dtCand, double& rCand,
                   double* qNew = nullptr, double* qOld = nullptr, const double* qnI = nullptr,
                   const double* accI = nullptr, bool wantDt = true)
{
    auto loadAcc = [&](double v[4]) {
        if (accI) { v[0] = accI[0]; v[1] = accI[1]; v[2] = accI[2]; v[3] = accI[3]; }
        else ld4(a.acc, i, v);
    };
    const double nia = met ? met[2] : m.nia[i];
    double dtc = 0.0;
    if (wantDt) {
        const double cper = met ? met[0] : m.cper[i], cd = met ? met[1] : m.cd[i];
        sAve /= cper;
        dtc = (a.sc->CFL * cd) / sAve;
        if (!isnan(dtc)) dtCand = fmin(dtCand, dtc);
    }
    double hc = 0.0;
    if (p.localTimestep) {
        if (a.dtUpdate) {
            hc = isnan(dtc) ? 0.0 : dtc;
            a.celldt[i] = hc;
        } else {
            hc = a.celldt[i];
        }
    }
#pragma unroll
    for (int k = 0; k < 4; k++) if (fabs(r[k]) > rCand) rCand = fabs(r[k]);
    const double s = nia;
    double R[4];
#pragma unroll
    for (int k = 0; k < 4; k++) R[k] = r[k] * s;
    if (m.src) {
        const double4 sv = m.src[i];
        R[0] = R[0] + sv.x; R[1] = R[1] + sv.y; R[2] = R[2] + sv.z; R[3] = R[3] + sv.w;
    }
    const double dt = a.sc->dt;
    const double h = p.localTimestep ? hc : dt;
    double qn[4], o[4];
    if (KIND != SK_RESIDUAL) {
        if (qnI) { qn[0] = qnI[0]; qn[1] = qnI[1]; qn[2] = qnI[2]; qn[3] = qnI[3]; }
        else ld4(a.qn, i, qn);
    }
    if (KIND == SK_RESIDUAL) {
        st4(a.R, m.refId[i], R);   // R is the caller's: reference numbering
    } else if (KIND == SK_EULER) {
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + h * R[k];
        storeOut(a, i, o);
    } else if (KIND == SK_RK2_1) {
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + (dt * R[k]);
        st4(a.acc, i, R);
        storeOut(a, i, o);
    } else if (KIND == SK_RK2_2) {
        double k1[4];
        loadAcc(k1);
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + (h / 2.0) * (k1[k] + R[k]);
        storeOut(a, i, o);
    } else if (KIND == SK_TVD_1) {
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + h * R[k];
        storeOut(a, i, o);
    } else if (KIND == SK_TVD_2) {
        double fe[4];
        if (qinI) { fe[0] = qinI[0]; fe[1] = qinI[1]; fe[2] = qinI[2]; fe[3] = qinI[3]; }
        else ld4(a.qin, i, fe);
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = 0.5 * (qn[k] + fe[k] + h * R[k]);
        storeOut(a, i, o);
    } else if (KIND == SK_RK4_1) {
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + ((dt / 2.0) * R[k]);
        st4(a.acc, i, R);
        storeOut(a, i, o);
    } else if (KIND == SK_RK4_2 || KIND == SK_RK4_3) {
        double ac[4];
        loadAcc(ac);
#pragma unroll
        for (int k = 0; k < 4; k++) ac[k] = ac[k] + 2.0 * R[k];
        const double c = (KIND == SK_RK4_2) ? (dt / 2.0) : dt;
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + (c * R[k]);
        st4(a.acc, i, ac);
        storeOut(a, i, o);
    } else if (KIND == SK_RK4_4) {
        double ac[4];
        loadAcc(ac);
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = qn[k] + (h / 6.0) * (ac[k] + R[k]);
        storeOut(a, i, o);
    }
    if (KIND != SK_RESIDUAL && a.last && a.recordErrors &&
        (isnan(o[0]) || isnan(o[1]) || isnan(o[2]) || isnan(o[3])))
        atomicMin(&a.sc->errCell, (uint64_t(a.stepId) << 32) | m.refId[i]);
    if ((KIND == SK_EULER || KIND == SK_RK2_2 || KIND == SK_TVD_2 || KIND == SK_RK4_4) && qNew) {
#pragma unroll
        for (int k = 0; k < 4; k++) { qNew[k] = o[k]; qOld[k] = qn[k]; }
    }
}

// Leaf sums of the RMS residual's pairwise sum (app/solver.d:153-168), fused into
// the stage that completes a step.  Each group of 16 lanes holds one aligned block
// of 16 consecutive reference cells, lane j its element j (absent cells add
// zeros); the xor butterfly adds exactly like the fixed 16-element tree, and lane
// 0 of the group stores the block's 8 sums: (new - old)^2 and new per variable.
// Every lane of the wave must call this.
DEV void rmsBlockLeaf(bool have, const double qNew[4], const double qOld[4], uint32_t refCell, double* rmsBlocks)
{
    double o[8];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const double x = have ? qNew[v] - qOld[v] : 0.0;
        o[v] = have ? x * x : 0.0;
        o[4 + v] = have ? qNew[v] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = o[q] + rowSwap<ROW_X1>(o[q]);
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = o[q] + rowSwap<ROW_X2>(o[q]);
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = o[q] + rowSwap<ROW_X4>(o[q]);
#pragma unroll
    for (int q = 0; q < 8; q++) o[q] = o[q] + rowSwap<ROW_X8>(o[q]);
    if (have && (threadIdx.x & 15u) == 0) {
        double* dst = rmsBlocks + size_t(refCell / 16) * 8;
        *reinterpret_cast<double4*>(dst) = make_double4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<double4*>(dst + 4) = make_double4(o[4], o[5], o[6], o[7]);
    }
}

// per-workgroup min dt / max |R| partial, combined later by k_reduce_stage (device-scope
// atomics from every workgroup on one address serialise across the XCDs)
DEV void blockPartial(double dtCand, double rCand, double* partial, uint32_t slot)
{
    __shared__ double sMin[BLK / 64], sMax_[BLK / 64];
    dtCand = warpMin(dtCand);
    rCand = warpMax(rCand);
    const int w = threadIdx.x / 64, l = threadIdx.x % 64;
    if (l == 0) { sMin[w] = dtCand; sMax_[w] = rCand; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a0 = sMin[0], b0 = sMax_[0];
#pragma unroll
        for (int k = 1; k < BLK / 64; k++) { a0 = fmin(a0, sMin[k]); b0 = fmax(b0, sMax_[k]); }
        partial[2 * slot] = a0;
        partial[2 * slot + 1] = b0;
    }
}
// Workgroup barrier for data shared through LDS: waits for this wave's LDS
// operations only.  __syncthreads() (and an LDS-scope fence, which covers the
// direct global-to-LDS copies) also waits for every outstanding global access,
// which would stall on the next tile's prefetch.  The "memory" clobber keeps the
// compiler from moving memory accesses across it.
DEV void ldsBarrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// newDt = min over the stage's workgroup partials; Rmax = max with the step's running value
void launchReduceStage(const double* partial, uint32_t n, DevScalars* sc, int checkActive, hipStream_t st);

}  // namespace ebb
