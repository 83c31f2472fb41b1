// dmx_math.h -- per-cell / per-face / per-edge arithmetic of the MHD step.
//
// Device functions templated on the bulk real type T (double or float).  In
// double they evaluate every expression in the reference's order (Fortran
// left-to-right association; MAX(a,b) = a > b ? a : b, MIN(a,b) = a < b ? a : b,
// SIGN(1,x) = copysign(1,x)) so that the float64 build, compiled with
// -ffp-contract=off, reproduces the reference bit for bit.  Each function
// names the reference routine it computes (paths relative to
// marcjoos-cea/dumses-hybrid/src).
#pragma once

#include <hip/hip_runtime.h>

namespace dmx {

template <typename T> struct K {
    static constexpr T zero = T(0), one = T(1), two = T(2), half = T(0.5), forth = T(0.25);
};
// smallr = smallc = 1e-10 (src/modules/commons.f90:50-51)
__device__ __forceinline__ double smallr_d() { return 1e-10; }

template <typename T> __device__ __forceinline__ T fmx(T a, T b) { return a > b ? a : b; }
template <typename T> __device__ __forceinline__ T fmn(T a, T b) { return a < b ? a : b; }
// float bulk (no bit-exactness to keep): one v_max_f32 / v_min_f32; differs
// from the comparison form only for NaN and the sign of a zero result
template <> __device__ __forceinline__ float fmx<float>(float a, float b) { return __builtin_fmaxf(a, b); }
template <> __device__ __forceinline__ float fmn<float>(float a, float b) { return __builtin_fminf(a, b); }
template <typename T> __device__ __forceinline__ T sgn1(T x) { return copysign(T(1), x); }
template <typename T> __device__ __forceinline__ T fab(T x) { return fabs(x); }

// TVD slope (minmod st=1, MC st=2), scheme.f90:452-477
template <typename T>
__device__ __forceinline__ T tvd_slope(T qm1, T q0, T qp1, int st)
{
    // st is 1 or 2: the division by st is an exact multiplication, where a
    // division by a run-time value would take 11 instructions in float64
    const T s = T(st), rs = st == 1 ? K<T>::one : K<T>::half;
    T dlft = s * (q0 - qm1);
    T drgt = s * (qp1 - q0);
    T dcen = K<T>::half * (dlft + drgt) * rs;
    T dsgn = sgn1(dcen);
    T slop = fmn(fab(dlft), fab(drgt));
    T dlim = slop;
    if ((dlft * drgt) <= K<T>::zero) dlim = K<T>::zero;
    return dsgn * fmn(dlim, fab(dcen));
}

// float64, 16 instructions instead of 20: st half / st is one factor (an exact
// scaling, st being 1 or 2), the lesser one-sided difference a hardware
// minimum, and the sign is copied (a NaN still comes through dcen).  The fused
// kernel takes 5.94 ms with it at 256^3 and 147 us at 64^3, 6.12 and 152 with
// the form above; the separate trace is within 1%.
template <>
__device__ __forceinline__ double tvd_slope<double>(double qm1, double q0, double qp1, int st)
{
    const double s = double(st), c = st == 1 ? 0.5 : 0.25;
    double dlft = s * (q0 - qm1);
    double drgt = s * (qp1 - q0);
    double dcen = c * (dlft + drgt);
    double dlim = __builtin_fmin(fab(dlft), fab(drgt));
    if ((dlft * drgt) <= 0.0) dlim = 0.0;
    return copysign(fmn(dlim, fab(dcen)), dcen);
}

// fast magnetosonic speed, the expression shared by comp_speed
// (physics.f90:148-164) and the Riemann solvers (solver.f90:675-683):
// b2 is passed already summed in the caller's order
template <typename T>
__device__ __forceinline__ T cfast_b2(T gamma, T ploc, T r, T bn, T b2)
{
    T c2 = gamma * ploc / r;
    T d2 = K<T>::half * (c2 + b2 / r);
    return sqrt(d2 + sqrt(d2 * d2 - c2 * bn * bn / r));
}

// ---------------------------------------------------------------------------
// 1D Riemann solvers, solver.f90:393-935.
// q = [r, p, u_n, B_n, u_t1, B_t1, u_t2, B_t2]; fg[8]; pstar = total pressure
// of the sampled state (HLLD only; 0 for the others, as pgstar is zeroed);
// entho = 1 / (gamma - 1).
//
// The energy chain -- total energies and pressures, v.B, the star-state
// energies, the energy flux, and the total-pressure differences that set
// the contact speed -- is evaluated in float64 (type D) in both precisions.
// At low beta the magnetic energy dominates each of these terms and their
// differences carry the thermal energy flux, which float32 would resolve
// only to about eps_32 / beta.  In the float64 build D is T and every
// expression keeps the reference's order, so the bits are unchanged.
// ---------------------------------------------------------------------------
typedef double D;

template <typename T>
__device__ __forceinline__ void phys_flux(T r, T ploc, T u, T v, T w, T a, T b, T c, D entho,
                                          T* f, T* cons, D& fE, D& cE)
{
    const T half = K<T>::half;
    T emag = half * ((a * a + b * b) + c * c);
    T ptot = ploc + emag;
    // energy chain in float64
    D ecinD = 0.5 * ((D(u) * u + D(v) * v) + D(w) * w) * r;
    D emagD = 0.5 * ((D(a) * a + D(b) * b) + D(c) * c);
    D etotD = (D(ploc) * entho + ecinD) + emagD;
    D ptotD = D(ploc) + emagD;
    fE = (etotD + ptotD) * u - D(a) * ((D(u) * a + D(v) * b) + D(w) * c);
    cE = etotD;
    f[0] = r * u;
    f[1] = T(fE);
    f[2] = (r * u * u + ptot) - a * a;
    f[3] = K<T>::zero;
    f[4] = r * u * v - a * b;
    f[5] = b * u - a * v;
    f[6] = r * u * w - a * c;
    f[7] = c * u - a * w;
    cons[0] = r; cons[1] = T(etotD); cons[2] = r * u; cons[3] = a;
    cons[4] = r * v; cons[5] = b; cons[6] = r * w; cons[7] = c;
}

// hlld, solver.f90:618-836
template <typename T>
__device__ __forceinline__ void hlld1d(const T* ql, const T* qr, T gamma, D entho, T ploc, T proc,
                                       T* fg, T& pstar)
{
    const T zero = K<T>::zero, half = K<T>::half;
    T rl = ql[0], ul = ql[2], al = ql[3], vl = ql[4], bl = ql[5], wl = ql[6], cl = ql[7];
    T rr = qr[0], ur = qr[2], ar = qr[3], vr = qr[4], br = qr[5], wr = qr[6], cr = qr[7];
    T a = half * (al + ar);
    T sgnm = sgn1(a);
    D ecinl = 0.5 * ((D(ul) * ul + D(vl) * vl) + D(wl) * wl) * rl;
    D emagl = 0.5 * ((D(a) * a + D(bl) * bl) + D(cl) * cl);
    D etotl = (D(ploc) * entho + ecinl) + emagl;
    D ptotl = D(ploc) + emagl;
    D vdotbl = (D(ul) * a + D(vl) * bl) + D(wl) * cl;
    D ecinr = 0.5 * ((D(ur) * ur + D(vr) * vr) + D(wr) * wr) * rr;
    D emagr = 0.5 * ((D(a) * a + D(br) * br) + D(cr) * cr);
    D etotr = (D(proc) * entho + ecinr) + emagr;
    D ptotr = D(proc) + emagr;
    D vdotbr = (D(ur) * a + D(vr) * br) + D(wr) * cr;
    T cfastl = cfast_b2(gamma, ploc, rl, a, (a * a + bl * bl) + cl * cl);
    T cfastr = cfast_b2(gamma, proc, rr, a, (a * a + br * br) + cr * cr);
    T sl = fmn(ul, ur) - fmx(cfastl, cfastr);
    T sr = fmx(ul, ur) + fmx(cfastl, cfastr);
    T rcl = rl * (ul - sl);
    T rcr = rr * (sr - ur);
    const D ustarD = ((D(rcr) * ur + D(rcl) * ul) + (ptotl - ptotr)) / (D(rcr) + rcl);
    const T ustar = T(ustarD);
    const D ptotstar = ((D(rcr) * ptotl + D(rcl) * ptotr) + D(rcl) * rcr * (D(ul) - ur)) / (D(rcr) + rcl);
    T vstarl, bstarl, wstarl, cstarl, vstarr, bstarr, wstarr, cstarr;
    T rstarl = rl * (sl - ul) / (sl - ustar);
    T estar = rl * (sl - ul) * (sl - ustar) - a * a;
    T el = rl * (sl - ul) * (sl - ul) - a * a;
    if (estar == zero) {
        vstarl = vl; bstarl = bl; wstarl = wl; cstarl = cl;
    } else {
        vstarl = vl - a * bl * (ustar - ul) / estar;
        bstarl = bl * el / estar;
        wstarl = wl - a * cl * (ustar - ul) / estar;
        cstarl = cl * el / estar;
    }
    D vdotbstarl = (ustarD * a + D(vstarl) * bstarl) + D(wstarl) * cstarl;
    D etotstarl = ((((D(sl) - ul) * etotl - ptotl * ul) + ptotstar * ustarD) + D(a) * (vdotbl - vdotbstarl))
                  / (D(sl) - ustarD);
    T sqrrstarl = sqrt(rstarl);
    T calfvenl = fab(a) / sqrrstarl;
    T sal = ustar - calfvenl;
    T rstarr = rr * (sr - ur) / (sr - ustar);
    estar = rr * (sr - ur) * (sr - ustar) - a * a;
    T er = rr * (sr - ur) * (sr - ur) - a * a;
    if (estar == zero) {
        vstarr = vr; bstarr = br; wstarr = wr; cstarr = cr;
    } else {
        vstarr = vr - a * br * (ustar - ur) / estar;
        bstarr = br * er / estar;
        wstarr = wr - a * cr * (ustar - ur) / estar;
        cstarr = cr * er / estar;
    }
    D vdotbstarr = (ustarD * a + D(vstarr) * bstarr) + D(wstarr) * cstarr;
    D etotstarr = ((((D(sr) - ur) * etotr - ptotr * ur) + ptotstar * ustarD) + D(a) * (vdotbr - vdotbstarr))
                  / (D(sr) - ustarD);
    T sqrrstarr = sqrt(rstarr);
    T calfvenr = fab(a) / sqrrstarr;
    T sar = ustar + calfvenr;
    T den = sqrrstarl + sqrrstarr;
    T vss = ((sqrrstarl * vstarl + sqrrstarr * vstarr) + sgnm * (bstarr - bstarl)) / den;
    T wss = ((sqrrstarl * wstarl + sqrrstarr * wstarr) + sgnm * (cstarr - cstarl)) / den;
    T bss = ((sqrrstarl * bstarr + sqrrstarr * bstarl) + sgnm * sqrrstarl * sqrrstarr * (vstarr - vstarl)) / den;
    T css = ((sqrrstarl * cstarr + sqrrstarr * cstarl) + sgnm * sqrrstarl * sqrrstarr * (wstarr - wstarl)) / den;
    D vdotbss = (ustarD * a + D(vss) * bss) + D(wss) * css;
    D etotssl = etotstarl - D(sgnm) * sqrrstarl * (vdotbstarl - vdotbss);
    D etotssr = etotstarr + D(sgnm) * sqrrstarr * (vdotbstarr - vdotbss);
    T ro, uo, vo, wo, bo, co;
    D uoD, ptoto, etoto, vdotbo;
    if (sl > zero) {
        ro = rl; uo = ul; vo = vl; wo = wl; bo = bl; co = cl; uoD = ul; ptoto = ptotl; etoto = etotl; vdotbo = vdotbl;
    } else if (sal > zero) {
        ro = rstarl; uo = ustar; vo = vstarl; wo = wstarl; bo = bstarl; co = cstarl; uoD = ustarD; ptoto = ptotstar;
        etoto = etotstarl; vdotbo = vdotbstarl;
    } else if (ustar > zero) {
        ro = rstarl; uo = ustar; vo = vss; wo = wss; bo = bss; co = css; uoD = ustarD; ptoto = ptotstar;
        etoto = etotssl; vdotbo = vdotbss;
    } else if (sar > zero) {
        ro = rstarr; uo = ustar; vo = vss; wo = wss; bo = bss; co = css; uoD = ustarD; ptoto = ptotstar;
        etoto = etotssr; vdotbo = vdotbss;
    } else if (sr > zero) {
        ro = rstarr; uo = ustar; vo = vstarr; wo = wstarr; bo = bstarr; co = cstarr; uoD = ustarD; ptoto = ptotstar;
        etoto = etotstarr; vdotbo = vdotbstarr;
    } else {
        ro = rr; uo = ur; vo = vr; wo = wr; bo = br; co = cr; uoD = ur; ptoto = ptotr; etoto = etotr; vdotbo = vdotbr;
    }
    fg[0] = ro * uo;
    fg[1] = T((etoto + ptoto) * uoD - D(a) * vdotbo);
    fg[2] = ro * uo * uo - a * a;
    fg[3] = zero;
    fg[4] = ro * uo * vo - a * bo;
    fg[5] = bo * uo - a * vo;
    fg[6] = ro * uo * wo - a * co;
    fg[7] = co * uo - a * wo;
    pstar = T(ptoto);
}

// llf (solver.f90:393-498), hll (:504-612), upwind (:842-935)
template <typename T, int SOLVER>
__device__ __forceinline__ void simple1d(const T* ql, const T* qr, T gamma, D entho, T ploc, T proc, T* fg)
{
    const T zero = K<T>::zero, half = K<T>::half;
    T rl = ql[0], ul = ql[2], al = ql[3], vl = ql[4], bl = ql[5], wl = ql[6], cl = ql[7];
    T rr = qr[0], ur = qr[2], ar = qr[3], vr = qr[4], br = qr[5], wr = qr[6], cr = qr[7];
    T a = half * (al + ar);
    T fl[8], cL[8], fr[8], cR[8];
    D flE, cLE, frE, cRE;
    phys_flux(rl, ploc, ul, vl, wl, a, bl, cl, entho, fl, cL, flE, cLE);
    phys_flux(rr, proc, ur, vr, wr, a, br, cr, entho, fr, cR, frE, cRE);
    if (SOLVER == 3) { // hll
        T vleft = cfast_b2(gamma, ploc, rl, a, (a * a + bl * bl) + cl * cl);
        T vright = cfast_b2(gamma, proc, rr, a, (a * a + br * br) + cr * cr);
        T sl = fmn(fmn(ul, ur) - fmx(vleft, vright), zero);
        T sr = fmx(fmx(ul, ur) + fmx(vleft, vright), zero);
#pragma unroll
        for (int n = 0; n < 8; n++) fg[n] = ((sr * fl[n] - sl * fr[n]) + sr * sl * (cR[n] - cL[n])) / (sr - sl);
        fg[1] = T(((D(sr) * flE - D(sl) * frE) + D(sr) * sl * (cRE - cLE)) / (D(sr) - sl));
    } else {
        T vel;
        if (SOLVER == 2) { // llf
            T vleft = cfast_b2(gamma, ploc, rl, a, (a * a + bl * bl) + cl * cl) + fab(ul);
            T vright = cfast_b2(gamma, proc, rr, a, (a * a + br * br) + cr * cr) + fab(ur);
            vel = fmx(vleft, vright);
        } else { // upwind
            vel = fab(half * (ul + ur));
        }
#pragma unroll
        for (int n = 0; n < 8; n++) fg[n] = half * (fl[n] + fr[n]) - vel * half * (cR[n] - cL[n]);
        fg[1] = T(0.5 * (flE + frE) - D(vel) * 0.5 * (cRE - cLE));
    }
}

template <typename T, int SOLVER>
__device__ __forceinline__ void riemann1d(const T* ql, const T* qr, T gamma, D entho, T c2iso, bool iso,
                                          T* fg, T& pstar)
{
    T ploc = iso ? ql[0] * c2iso : ql[1];
    T proc = iso ? qr[0] * c2iso : qr[1];
    if (SOLVER == 4) {
        hlld1d(ql, qr, gamma, entho, ploc, proc, fg, pstar);
    } else {
        simple1d<T, SOLVER>(ql, qr, gamma, entho, ploc, proc, fg);
        pstar = K<T>::zero;
    }
}

// ---------------------------------------------------------------------------
// 2D (edge) Riemann solvers, solver_magnetic.f90:241-727.
// corner q = [r, p, u, v, A, B, C, E]; returns emf*dt
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T cf2x(T gamma, const T* q)
{
    return cfast_b2(gamma, q[1], q[0], q[4], (q[4] * q[4] + q[5] * q[5]) + q[6] * q[6]);
}
template <typename T>
__device__ __forceinline__ T cf2y(T gamma, const T* q)
{
    return cfast_b2(gamma, q[1], q[0], q[5], (q[5] * q[5] + q[4] * q[4]) + q[6] * q[6]);
}

// hlld, solver_magnetic.f90:362-548
template <typename T>
__device__ __forceinline__ T hlld2d(const T* LL, const T* RL, const T* LR, const T* RR, T dt, T gamma)
{
    const T zero = K<T>::zero, one = K<T>::one, half = K<T>::half;
    const T smallc = T(1e-10);
    T rLL = LL[0], pLL = LL[1], uLL = LL[2], vLL = LL[3], ALL = LL[4], BLL = LL[5], CLL = LL[6], ELL = LL[7];
    T rRL = RL[0], pRL = RL[1], uRL = RL[2], vRL = RL[3], ARL = RL[4], BRL = RL[5], CRL = RL[6], ERL = RL[7];
    T rLR = LR[0], pLR = LR[1], uLR = LR[2], vLR = LR[3], ALR = LR[4], BLR = LR[5], CLR = LR[6], ELR = LR[7];
    T rRR = RR[0], pRR = RR[1], uRR = RR[2], vRR = RR[3], ARR = RR[4], BRR = RR[5], CRR = RR[6], ERR = RR[7];
    T cLLx = cf2x(gamma, LL), cLRx = cf2x(gamma, LR), cRLx = cf2x(gamma, RL), cRRx = cf2x(gamma, RR);
    T cLLy = cf2y(gamma, LL), cLRy = cf2y(gamma, LR), cRLy = cf2y(gamma, RL), cRRy = cf2y(gamma, RR);
    T SL = fmn(fmn(fmn(uLL, uLR), uRL), uRR) - fmx(fmx(fmx(cLLx, cLRx), cRLx), cRRx);
    T SR = fmx(fmx(fmx(uLL, uLR), uRL), uRR) + fmx(fmx(fmx(cLLx, cLRx), cRLx), cRRx);
    T SB = fmn(fmn(fmn(vLL, vLR), vRL), vRR) - fmx(fmx(fmx(cLLy, cLRy), cRLy), cRRy);
    T ST = fmx(fmx(fmx(vLL, vLR), vRL), vRR) + fmx(fmx(fmx(cLLy, cLRy), cRLy), cRRy);
    // total pressures in float64 (D): their differences set the contact
    // speeds, and at low beta the magnetic pressure dominates each of them
    D PtotLL = D(pLL) + 0.5 * ((D(ALL) * ALL + D(BLL) * BLL) + D(CLL) * CLL);
    D PtotLR = D(pLR) + 0.5 * ((D(ALR) * ALR + D(BLR) * BLR) + D(CLR) * CLR);
    D PtotRL = D(pRL) + 0.5 * ((D(ARL) * ARL + D(BRL) * BRL) + D(CRL) * CRL);
    D PtotRR = D(pRR) + 0.5 * ((D(ARR) * ARR + D(BRR) * BRR) + D(CRR) * CRR);
    T rcLLx = rLL * (uLL - SL), rcRLx = rRL * (SR - uRL);
    T rcLRx = rLR * (uLR - SL), rcRRx = rRR * (SR - uRR);
    T rcLLy = rLL * (vLL - SB), rcLRy = rLR * (ST - vLR);
    T rcRLy = rRL * (vRL - SB), rcRRy = rRR * (ST - vRR);
    T ustar = T(((((D(rcLLx) * uLL + D(rcLRx) * uLR) + D(rcRLx) * uRL) + D(rcRRx) * uRR)
                 + (((PtotLL - PtotRL) + PtotLR) - PtotRR)) / (((D(rcLLx) + rcLRx) + rcRLx) + rcRRx));
    T vstar = T(((((D(rcLLy) * vLL + D(rcLRy) * vLR) + D(rcRLy) * vRL) + D(rcRRy) * vRR)
                 + (((PtotLL - PtotLR) + PtotRL) - PtotRR)) / (((D(rcLLy) + rcLRy) + rcRLy) + rcRRy));
    T SLustar = one / (SL - ustar), SRustar = one / (SR - ustar);
    T SBvstar = one / (SB - vstar), STvstar = one / (ST - vstar);

    T rstarLLx = rLL * (SL - uLL) * SLustar, BstarLL = BLL * (SL - uLL) * SLustar;
    T rstarLLy = rLL * (SB - vLL) * SBvstar, AstarLL = ALL * (SB - vLL) * SBvstar;
    T rstarLL = rLL * (SL - uLL) * SLustar * (SB - vLL) * SBvstar;
    T EstarLLx = ustar * BstarLL - vLL * ALL, EstarLLy = uLL * BLL - vstar * AstarLL;
    T EstarLL = ustar * BstarLL - vstar * AstarLL;

    T rstarLRx = rLR * (SL - uLR) * SLustar, BstarLR = BLR * (SL - uLR) * SLustar;
    T rstarLRy = rLR * (ST - vLR) * STvstar, AstarLR = ALR * (ST - vLR) * STvstar;
    T rstarLR = rLR * (SL - uLR) * SLustar * (ST - vLR) * STvstar;
    T EstarLRx = ustar * BstarLR - vLR * ALR, EstarLRy = uLR * BLR - vstar * AstarLR;
    T EstarLR = ustar * BstarLR - vstar * AstarLR;

    T rstarRLx = rRL * (SR - uRL) * SRustar, BstarRL = BRL * (SR - uRL) * SRustar;
    T rstarRLy = rRL * (SB - vRL) * SBvstar, AstarRL = ARL * (SB - vRL) * SBvstar;
    T rstarRL = rRL * (SR - uRL) * SRustar * (SB - vRL) * SBvstar;
    T EstarRLx = ustar * BstarRL - vRL * ARL, EstarRLy = uRL * BRL - vstar * AstarRL;
    T EstarRL = ustar * BstarRL - vstar * AstarRL;

    T rstarRRx = rRR * (SR - uRR) * SRustar, BstarRR = BRR * (SR - uRR) * SRustar;
    T rstarRRy = rRR * (ST - vRR) * STvstar, AstarRR = ARR * (ST - vRR) * STvstar;
    T rstarRR = rRR * (SR - uRR) * SRustar * (ST - vRR) * STvstar;
    T EstarRRx = ustar * BstarRR - vRR * ARR, EstarRRy = uRR * BRR - vstar * AstarRR;
    T EstarRR = ustar * BstarRR - vstar * AstarRR;

    T sqLR = one / sqrt(rstarLR), sqRL = one / sqrt(rstarRL);
    T sqRR = one / sqrt(rstarRR), sqLL = one / sqrt(rstarLL);

    T calfvenL = fmx(fmx(fmx(fmx(fab(ALR) / sqrt(rstarLRx), fab(AstarLR) * sqLR),
                             fab(ALL) / sqrt(rstarLLx)), fab(AstarLL) * sqLL), smallc);
    T calfvenR = fmx(fmx(fmx(fmx(fab(ARR) / sqrt(rstarRRx), fab(AstarRR) * sqRR),
                             fab(ARL) / sqrt(rstarRLx)), fab(AstarRL) * sqRL), smallc);
    T calfvenB = fmx(fmx(fmx(fmx(fab(BLL) / sqrt(rstarLLy), fab(BstarLL) * sqLL),
                             fab(BRL) / sqrt(rstarRLy)), fab(BstarRL) * sqRL), smallc);
    T calfvenT = fmx(fmx(fmx(fmx(fab(BLR) / sqrt(rstarLRy), fab(BstarLR) * sqLR),
                             fab(BRR) / sqrt(rstarRRy)), fab(BstarRR) * sqRR), smallc);
    T SAL = fmn(ustar - calfvenL, zero), SAR = fmx(ustar + calfvenR, zero);
    T SAB = fmn(vstar - calfvenB, zero), SAT = fmx(vstar + calfvenT, zero);
    T SARSAL = one / (SAR - SAL);
    T SATSAB = one / (SAT - SAB);
    T AstarT = (SAR * AstarRR - SAL * AstarLR) * SARSAL;
    T AstarB = (SAR * AstarRL - SAL * AstarLL) * SARSAL;
    T BstarR = (SAT * BstarRR - SAB * BstarRL) * SATSAB;
    T BstarL = (SAT * BstarLR - SAB * BstarLL) * SATSAB;
    T E;
    if (SB > zero) {
        if (SL > zero) E = ELL;
        else if (SR < zero) E = ERL;
        else E = ((SAR * EstarLLx - SAL * EstarRLx) + SAR * SAL * (BRL - BLL)) * SARSAL;
    } else if (ST < zero) {
        if (SL > zero) E = ELR;
        else if (SR < zero) E = ERR;
        else E = ((SAR * EstarLRx - SAL * EstarRRx) + SAR * SAL * (BRR - BLR)) * SARSAL;
    } else if (SL > zero) {
        E = ((SAT * EstarLLy - SAB * EstarLRy) - SAT * SAB * (ALR - ALL)) * SATSAB;
    } else if (SR < zero) {
        E = ((SAT * EstarRLy - SAB * EstarRRy) - SAT * SAB * (ARR - ARL)) * SATSAB;
    } else {
        E = (((((SAL * SAB * EstarRR - SAL * SAT * EstarRL) - SAR * SAB * EstarLR) + SAR * SAT * EstarLL) * SARSAL) * SATSAB
             - SAT * SAB * SATSAB * (AstarT - AstarB))
            + SAR * SAL * SARSAL * (BstarR - BstarL);
    }
    return E * dt;
}

template <typename T>
__device__ __forceinline__ T llf2d_dir(T gamma, T rl, T pl, T ul, T al, T bl, T cl, T rr, T pr, T ur,
                                       T ar, T br, T cr, bool iso, T c2iso)
{
    // one direction of llf, solver_magnetic.f90:267-297
    const T half = K<T>::half;
    if (iso) {
        pl = rl * c2iso;
        pr = rr * c2iso;
    }
    al = half * (al + ar);
    ar = al;
    T vleft = cfast_b2(gamma, pl, rl, al, (al * al + bl * bl) + cl * cl) + fab(ul);
    T vright = cfast_b2(gamma, pr, rr, ar, (ar * ar + br * br) + cr * cr) + fab(ur);
    T vel = fmx(vleft, vright);
    return -vel * half * (br - bl);
}

template <typename T, int SOLVER>
__device__ __forceinline__ T riemann2d(const T* LL, const T* RL, const T* LR, const T* RR, T dt,
                                       T gamma, bool iso, T c2iso)
{
    const T zero = K<T>::zero, half = K<T>::half, forth = K<T>::forth;
    if (SOLVER == 4) return hlld2d(LL, RL, LR, RR, dt, gamma);
    if (SOLVER == 2) { // llf, solver_magnetic.f90:241-356
        T E = forth * (((LL[7] + RL[7]) + LR[7]) + RR[7]);
        T fx = llf2d_dir(gamma, half * (LL[0] + LR[0]), half * (LL[1] + LR[1]), half * (LL[2] + LR[2]),
                         half * (LL[4] + LR[4]), half * (LL[5] + LR[5]), half * (LL[6] + LR[6]),
                         half * (RR[0] + RL[0]), half * (RR[1] + RL[1]), half * (RR[2] + RL[2]),
                         half * (RR[4] + RL[4]), half * (RR[5] + RL[5]), half * (RR[6] + RL[6]), iso, c2iso);
        T fy = llf2d_dir(gamma, half * (LL[0] + RL[0]), half * (LL[1] + RL[1]), half * (LL[3] + RL[3]),
                         half * (LL[5] + RL[5]), half * (LL[4] + RL[4]), half * (LL[6] + RL[6]),
                         half * (RR[0] + LR[0]), half * (RR[1] + LR[1]), half * (RR[3] + LR[3]),
                         half * (RR[5] + LR[5]), half * (RR[4] + LR[4]), half * (RR[6] + LR[6]), iso, c2iso);
        T e = E + (fx - fy);
        return e * dt;
    }
    if (SOLVER == 5) { // upwind, solver_magnetic.f90:554-600
        T E = forth * (((LL[7] + RL[7]) + LR[7]) + RR[7]);
        T ul = half * (LL[2] + LR[2]), bl = half * (LL[5] + LR[5]);
        T ur = half * (RR[2] + RL[2]), br = half * (RR[5] + RL[5]);
        T vel = half * (ul + ur);
        T fx = -fab(vel) * half * (br - bl);
        ul = half * (LL[3] + RL[3]); bl = half * (LL[4] + RL[4]);
        ur = half * (RR[3] + LR[3]); br = half * (RR[4] + LR[4]);
        vel = half * (ul + ur);
        T fy = -fab(vel) * half * (br - bl);
        T e = E + (fx - fy);
        return e * dt;
    }
    // hlla, solver_magnetic.f90:688-727
    const T smallc = T(1e-10);
    T cLLx = sqrt(LL[4] * LL[4] / LL[0]), cLRx = sqrt(LR[4] * LR[4] / LR[0]);
    T cRLx = sqrt(RL[4] * RL[4] / RL[0]), cRRx = sqrt(RR[4] * RR[4] / RR[0]);
    T cLLy = sqrt(LL[5] * LL[5] / LL[0]), cLRy = sqrt(LR[5] * LR[5] / LR[0]);
    T cRLy = sqrt(RL[5] * RL[5] / RL[0]), cRRy = sqrt(RR[5] * RR[5] / RR[0]);
    T SL = fmn(fmn(fmn(fmn(LL[2], LR[2]), RL[2]), RR[2]) - fmx(fmx(fmx(fmx(cLLx, cLRx), cRLx), cRRx), smallc), zero);
    T SR = fmx(fmx(fmx(fmx(LL[2], LR[2]), RL[2]), RR[2]) + fmx(fmx(fmx(fmx(cLLx, cLRx), cRLx), cRRx), smallc), zero);
    T SB = fmn(fmn(fmn(fmn(LL[3], LR[3]), RL[3]), RR[3]) - fmx(fmx(fmx(fmx(cLLy, cLRy), cRLy), cRRy), smallc), zero);
    T ST = fmx(fmx(fmx(fmx(LL[3], LR[3]), RL[3]), RR[3]) + fmx(fmx(fmx(fmx(cLLy, cLRy), cRLy), cRRy), smallc), zero);
    T e = ((((SL * SB * RR[7] - SL * ST * RL[7]) - SR * SB * LR[7]) + SR * ST * LL[7]) / (SR - SL) / (ST - SB)
           - ST * SB / (ST - SB) * (RR[4] - LL[4]))
          + SR * SL / (SR - SL) * (RR[5] - LL[5]);
    return e * dt;
}

// ---------------------------------------------------------------------------
// float64 HLLD with shared reciprocals.
//
// An IEEE division of doubles is about 11 instructions here and a square root
// about 18, most of them scaling for operands near the ends of the exponent
// range, and the divisions by one denominator cannot share its reciprocal
// because the scaling depends on both operands.  With operands known to lie
// well inside the range the scaling is not needed: Newton's reciprocal (two
// steps from v_rcp_f64), then one residual correction per quotient
// (Markstein, IBM J. Res. Dev. 34, 1990), and Goldschmidt's square root with
// two residual corrections (Markstein, RNC-6, 2004) round correctly, so the
// bits are those of a / b and sqrt(x): 5 + 3 instructions per quotient,
// 5 + 3 n for n quotients over one denominator, and 10 per square root.
//
// hlld1d_fast and hlld2d_fast evaluate hlld1d and hlld2d with them, in the
// same order of operations, and return whether the operands were in range:
// no NaN or infinity, no speed or root that vanishes, no numerator that is
// tiny but not zero where its last bits could reach the result.  Otherwise
// the caller evaluates hlld1d or hlld2d.  A maximum of square roots is the
// root of the maximum (rounding is monotone), which removes the outer root
// of all fast speeds but one per direction.  The face/edge kernel at 256^3
// issues 4700 vector instructions a wave and plane instead of 6800 and takes
// 4.88 ms instead of 5.50: it is left bound by its reads of the trace summary
// (29 GB at 6.5 TB/s), 51% of its cycles issue vector instructions, 61%
// before.  At 32 x 64 x 32 it takes 0.047 ms instead of 0.055.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double rcp_nr(double b)
{
    double y = __builtin_amdgcn_rcp(b);
    double e = __builtin_fma(-b, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-b, y, 1.0);
    return __builtin_fma(y, e, y);
}
// a / b with y = rcp_nr(b); the sign of a zero quotient is lost when a is -0
__device__ __forceinline__ double div_nr(double a, double b, double y)
{
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
// the same with the sign of a zero quotient
__device__ __forceinline__ double div_nr0(double a, double b, double y)
{
    return __builtin_amdgcn_div_fixup(div_nr(a, b, y), b, a);
}
// 1 / b
__device__ __forceinline__ double inv_nr(double b)
{
    const double y = rcp_nr(b);
    return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
}
// sqrt(x), x > 0
__device__ __forceinline__ double sqrt_nr(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
// x is not zero but smaller than lim
__device__ __forceinline__ bool tiny(double x, double lim) { return __builtin_fabs(x) < lim && x != 0.0; }

// limits of the operand range: sums of densities, energies, pressures and
// speeds below 2^100; distances of the outer waves from the contact above
// 2^-100; discriminants of the fast speeds above 2^-500; numerators zero or
// above 2^-700, except where the quotient is lost in the sum it enters.
// Densities are at least 1e-10 (smallr).  With these every denominator lies
// in 2^+-400, every root's argument in 2^+-700, and every residual is exact.
constexpr double kHuge = 0x1p100, kGap = 0x1p-100, kDisc = 0x1p-500, kNum = 0x1p-700;

__device__ __forceinline__ bool hlld1d_fast(const double* ql, const double* qr, double gamma, double entho, double ploc,
                                            double proc, double* fg, double& pstar)
{
    const double zero = 0.0, half = 0.5;
    double rl = ql[0], ul = ql[2], al = ql[3], vl = ql[4], bl = ql[5], wl = ql[6], cl = ql[7];
    double rr = qr[0], ur = qr[2], ar = qr[3], vr = qr[4], br = qr[5], wr = qr[6], cr = qr[7];
    double a = half * (al + ar);
    double sgnm = sgn1(a);
    double ecinl = 0.5 * ((ul * ul + vl * vl) + wl * wl) * rl;
    double emagl = 0.5 * ((a * a + bl * bl) + cl * cl);
    double etotl = (ploc * entho + ecinl) + emagl;
    double ptotl = ploc + emagl;
    double vdotbl = (ul * a + vl * bl) + wl * cl;
    double ecinr = 0.5 * ((ur * ur + vr * vr) + wr * wr) * rr;
    double emagr = 0.5 * ((a * a + br * br) + cr * cr);
    double etotr = (proc * entho + ecinr) + emagr;
    double ptotr = proc + emagr;
    double vdotbr = (ur * a + vr * br) + wr * cr;
    // discriminant and half sum of the fast speed (cfast_b2)
    auto speed = [&](double p, double r, double b2, double& d2) {
        const double y = rcp_nr(r);
        const double c2 = div_nr(gamma * p, r, y);
        d2 = half * (c2 + div_nr(b2, r, y));
        return d2 * d2 - div_nr(c2 * a * a, r, y);
    };
    double d2l, d2r;
    const double discl = speed(ploc, rl, (a * a + bl * bl) + cl * cl, d2l);
    const double discr = speed(proc, rr, (a * a + br * br) + cr * cr, d2r);
    const double cf = sqrt_nr(__builtin_fmax(d2l + sqrt_nr(discl), d2r + sqrt_nr(discr)));
    const double umin = __builtin_fmin(ul, ur), umax = __builtin_fmax(ul, ur);
    const double sl = umin - cf, sr = umax + cf;
    double rcl = rl * (ul - sl);
    double rcr = rr * (sr - ur);
    const double den = rcr + rcl, yden = rcp_nr(den);
    const double nus = (rcr * ur + rcl * ul) + (ptotl - ptotr);
    const double ustar = div_nr(nus, den, yden);
    const double ptotstar = div_nr((rcr * ptotl + rcl * ptotr) + rcl * rcr * (ul - ur), den, yden);
    const double dl = sl - ustar, dr = sr - ustar;
    bool ok = __builtin_fmin(discl, discr) > kDisc && sl < umin && sr > umax && dl < -kGap && dr > kGap
              && ((etotl + etotr) + (rl + rr)) + ((sr - sl) + den) < kHuge && !tiny(nus, kNum);
    // n / d with y = rcp_nr(d), and v - n / d, where v may absorb a tiny quotient
    auto quot = [&](double n, double d, double y) {
        ok = ok && !tiny(n, kNum);
        return div_nr0(n, d, y);
    };
    auto less_quot = [&](double v, double n, double d, double y) {
        const double q = div_nr0(n, d, y);
        ok = ok && !(tiny(n, kNum) && !(fab(q) < 0x1p-60 * fab(v)));
        return v - q;
    };
    auto star = [&](double r, double u, double v, double w, double b, double c, double s, double ds, double etot,
                    double ptot, double vdotb, double& rstar, double& vstar, double& bstar, double& wstar,
                    double& cstar, double& vdotbstar, double& etotstar) {
        const double yd = rcp_nr(ds);
        rstar = div_nr(r * (s - u), ds, yd);
        const double estar = r * (s - u) * ds - a * a;
        const double e = r * (s - u) * (s - u) - a * a;
        ok = ok && estar != zero;
        const double ye = rcp_nr(estar);
        vstar = less_quot(v, a * b * (ustar - u), estar, ye);
        bstar = quot(b * e, estar, ye);
        wstar = less_quot(w, a * c * (ustar - u), estar, ye);
        cstar = quot(c * e, estar, ye);
        vdotbstar = (ustar * a + vstar * bstar) + wstar * cstar;
        etotstar = div_nr((((s - u) * etot - ptot * u) + ptotstar * ustar) + a * (vdotb - vdotbstar), ds, yd);
    };
    double rstarl, vstarl, bstarl, wstarl, cstarl, vdotbstarl, etotstarl;
    double rstarr, vstarr, bstarr, wstarr, cstarr, vdotbstarr, etotstarr;
    star(rl, ul, vl, wl, bl, cl, sl, dl, etotl, ptotl, vdotbl, rstarl, vstarl, bstarl, wstarl, cstarl, vdotbstarl,
         etotstarl);
    star(rr, ur, vr, wr, br, cr, sr, dr, etotr, ptotr, vdotbr, rstarr, vstarr, bstarr, wstarr, cstarr, vdotbstarr,
         etotstarr);
    const double sqrrstarl = sqrt_nr(rstarl), sqrrstarr = sqrt_nr(rstarr);
    const double sal = ustar - div_nr(fab(a), sqrrstarl, rcp_nr(sqrrstarl));
    const double sar = ustar + div_nr(fab(a), sqrrstarr, rcp_nr(sqrrstarr));
    const double dens = sqrrstarl + sqrrstarr, ys = rcp_nr(dens);
    const double vss = quot((sqrrstarl * vstarl + sqrrstarr * vstarr) + sgnm * (bstarr - bstarl), dens, ys);
    const double wss = quot((sqrrstarl * wstarl + sqrrstarr * wstarr) + sgnm * (cstarr - cstarl), dens, ys);
    const double bss = quot((sqrrstarl * bstarr + sqrrstarr * bstarl) + sgnm * sqrrstarl * sqrrstarr * (vstarr - vstarl),
                            dens, ys);
    const double css = quot((sqrrstarl * cstarr + sqrrstarr * cstarl) + sgnm * sqrrstarl * sqrrstarr * (wstarr - wstarl),
                            dens, ys);
    const double vdotbss = (ustar * a + vss * bss) + wss * css;
    const double etotssl = etotstarl - sgnm * sqrrstarl * (vdotbstarl - vdotbss);
    const double etotssr = etotstarr + sgnm * sqrrstarr * (vdotbstarr - vdotbss);
    // the sampled state: outer (0), star (1) or double star (2), left or right
    double ro, uo, vo, wo, bo, co, ptoto, etoto, vdotbo;
    if (sl > zero) {
        ro = rl; uo = ul; vo = vl; wo = wl; bo = bl; co = cl; ptoto = ptotl; etoto = etotl; vdotbo = vdotbl;
    } else if (sal > zero) {
        ro = rstarl; uo = ustar; vo = vstarl; wo = wstarl; bo = bstarl; co = cstarl; ptoto = ptotstar;
        etoto = etotstarl; vdotbo = vdotbstarl;
    } else if (ustar > zero) {
        ro = rstarl; uo = ustar; vo = vss; wo = wss; bo = bss; co = css; ptoto = ptotstar;
        etoto = etotssl; vdotbo = vdotbss;
    } else if (sar > zero) {
        ro = rstarr; uo = ustar; vo = vss; wo = wss; bo = bss; co = css; ptoto = ptotstar;
        etoto = etotssr; vdotbo = vdotbss;
    } else if (sr > zero) {
        ro = rstarr; uo = ustar; vo = vstarr; wo = wstarr; bo = bstarr; co = cstarr; ptoto = ptotstar;
        etoto = etotstarr; vdotbo = vdotbstarr;
    } else {
        ro = rr; uo = ur; vo = vr; wo = wr; bo = br; co = cr; ptoto = ptotr; etoto = etotr; vdotbo = vdotbr;
    }
    fg[0] = ro * uo;
    fg[1] = (etoto + ptoto) * uo - a * vdotbo;
    fg[2] = ro * uo * uo - a * a;
    fg[3] = zero;
    fg[4] = ro * uo * vo - a * bo;
    fg[5] = bo * uo - a * vo;
    fg[6] = ro * uo * wo - a * co;
    fg[7] = co * uo - a * wo;
    pstar = ptoto;
    return ok;
}

__device__ __forceinline__ bool hlld2d_fast(const double* LL, const double* RL, const double* LR, const double* RR,
                                            double dt, double gamma, double& emf)
{
    const double zero = 0.0, half = 0.5, smallc = 1e-10;
    double rLL = LL[0], pLL = LL[1], uLL = LL[2], vLL = LL[3], ALL = LL[4], BLL = LL[5], CLL = LL[6], ELL = LL[7];
    double rRL = RL[0], pRL = RL[1], uRL = RL[2], vRL = RL[3], ARL = RL[4], BRL = RL[5], CRL = RL[6], ERL = RL[7];
    double rLR = LR[0], pLR = LR[1], uLR = LR[2], vLR = LR[3], ALR = LR[4], BLR = LR[5], CLR = LR[6], ELR = LR[7];
    double rRR = RR[0], pRR = RR[1], uRR = RR[2], vRR = RR[3], ARR = RR[4], BRR = RR[5], CRR = RR[6], ERR = RR[7];
#define MX4(a, b, c, d) __builtin_fmax(__builtin_fmax(__builtin_fmax(a, b), c), d)
#define MN4(a, b, c, d) __builtin_fmin(__builtin_fmin(__builtin_fmin(a, b), c), d)
    // squared fast speeds along both directions, the least discriminant
    double cx2 = zero, cy2 = zero, disc = kHuge;
    auto speeds = [&](const double* q) {
        const double y = rcp_nr(q[0]);
        const double c2 = div_nr(gamma * q[1], q[0], y);
        const double d2 = half * (c2 + div_nr((q[4] * q[4] + q[5] * q[5]) + q[6] * q[6], q[0], y));
        const double x = d2 * d2 - div_nr(c2 * q[4] * q[4], q[0], y);
        const double z = d2 * d2 - div_nr(c2 * q[5] * q[5], q[0], y);
        disc = __builtin_fmin(disc, __builtin_fmin(x, z));
        cx2 = __builtin_fmax(cx2, d2 + sqrt_nr(x));
        cy2 = __builtin_fmax(cy2, d2 + sqrt_nr(z));
    };
    speeds(LL);
    speeds(LR);
    speeds(RL);
    speeds(RR);
    const double cx = sqrt_nr(cx2), cy = sqrt_nr(cy2);
    const double umin = MN4(uLL, uLR, uRL, uRR), umax = MX4(uLL, uLR, uRL, uRR);
    const double vmin = MN4(vLL, vLR, vRL, vRR), vmax = MX4(vLL, vLR, vRL, vRR);
    double SL = umin - cx, SR = umax + cx, SB = vmin - cy, ST = vmax + cy;
    double PtotLL = pLL + 0.5 * ((ALL * ALL + BLL * BLL) + CLL * CLL);
    double PtotLR = pLR + 0.5 * ((ALR * ALR + BLR * BLR) + CLR * CLR);
    double PtotRL = pRL + 0.5 * ((ARL * ARL + BRL * BRL) + CRL * CRL);
    double PtotRR = pRR + 0.5 * ((ARR * ARR + BRR * BRR) + CRR * CRR);
    double rcLLx = rLL * (uLL - SL), rcRLx = rRL * (SR - uRL);
    double rcLRx = rLR * (uLR - SL), rcRRx = rRR * (SR - uRR);
    double rcLLy = rLL * (vLL - SB), rcLRy = rLR * (ST - vLR);
    double rcRLy = rRL * (vRL - SB), rcRRy = rRR * (ST - vRR);
    const double nus = (((rcLLx * uLL + rcLRx * uLR) + rcRLx * uRL) + rcRRx * uRR)
                       + (((PtotLL - PtotRL) + PtotLR) - PtotRR);
    const double nvs = (((rcLLy * vLL + rcLRy * vLR) + rcRLy * vRL) + rcRRy * vRR)
                       + (((PtotLL - PtotLR) + PtotRL) - PtotRR);
    const double dus = ((rcLLx + rcLRx) + rcRLx) + rcRRx, dvs = ((rcLLy + rcLRy) + rcRLy) + rcRRy;
    const double ustar = div_nr(nus, dus, rcp_nr(dus)), vstar = div_nr(nvs, dvs, rcp_nr(dvs));
    const double dSL = SL - ustar, dSR = SR - ustar, dSB = SB - vstar, dST = ST - vstar;
    const bool ok = disc > kDisc && SL < umin && SR > umax && SB < vmin && ST > vmax && dSL < -kGap && dSR > kGap
                    && dSB < -kGap && dST > kGap && !tiny(nus, kNum) && !tiny(nvs, kNum)
                    && (((PtotLL + PtotLR) + (PtotRL + PtotRR)) + ((rLL + rLR) + (rRL + rRR)))
                               + (((SR - SL) + (ST - SB)) + (dus + dvs))
                           < kHuge;
    double SLustar = inv_nr(dSL), SRustar = inv_nr(dSR);
    double SBvstar = inv_nr(dSB), STvstar = inv_nr(dST);

    double rstarLLx = rLL * (SL - uLL) * SLustar, BstarLL = BLL * (SL - uLL) * SLustar;
    double rstarLLy = rLL * (SB - vLL) * SBvstar, AstarLL = ALL * (SB - vLL) * SBvstar;
    double rstarLL = rLL * (SL - uLL) * SLustar * (SB - vLL) * SBvstar;
    double EstarLLx = ustar * BstarLL - vLL * ALL, EstarLLy = uLL * BLL - vstar * AstarLL;
    double EstarLL = ustar * BstarLL - vstar * AstarLL;

    double rstarLRx = rLR * (SL - uLR) * SLustar, BstarLR = BLR * (SL - uLR) * SLustar;
    double rstarLRy = rLR * (ST - vLR) * STvstar, AstarLR = ALR * (ST - vLR) * STvstar;
    double rstarLR = rLR * (SL - uLR) * SLustar * (ST - vLR) * STvstar;
    double EstarLRx = ustar * BstarLR - vLR * ALR, EstarLRy = uLR * BLR - vstar * AstarLR;
    double EstarLR = ustar * BstarLR - vstar * AstarLR;

    double rstarRLx = rRL * (SR - uRL) * SRustar, BstarRL = BRL * (SR - uRL) * SRustar;
    double rstarRLy = rRL * (SB - vRL) * SBvstar, AstarRL = ARL * (SB - vRL) * SBvstar;
    double rstarRL = rRL * (SR - uRL) * SRustar * (SB - vRL) * SBvstar;
    double EstarRLx = ustar * BstarRL - vRL * ARL, EstarRLy = uRL * BRL - vstar * AstarRL;
    double EstarRL = ustar * BstarRL - vstar * AstarRL;

    double rstarRRx = rRR * (SR - uRR) * SRustar, BstarRR = BRR * (SR - uRR) * SRustar;
    double rstarRRy = rRR * (ST - vRR) * STvstar, AstarRR = ARR * (ST - vRR) * STvstar;
    double rstarRR = rRR * (SR - uRR) * SRustar * (ST - vRR) * STvstar;
    double EstarRRx = ustar * BstarRR - vRR * ARR, EstarRRy = uRR * BRR - vstar * AstarRR;
    double EstarRR = ustar * BstarRR - vstar * AstarRR;

    // Alfven speeds |field| / sqrt(density)
    auto alf = [](double b, double r) {
        const double s = sqrt_nr(r);
        return div_nr(fab(b), s, rcp_nr(s));
    };
    const double sqLR = inv_nr(sqrt_nr(rstarLR)), sqRL = inv_nr(sqrt_nr(rstarRL));
    const double sqRR = inv_nr(sqrt_nr(rstarRR)), sqLL = inv_nr(sqrt_nr(rstarLL));
    const double calfvenL = __builtin_fmax(
        MX4(alf(ALR, rstarLRx), fab(AstarLR) * sqLR, alf(ALL, rstarLLx), fab(AstarLL) * sqLL), smallc);
    const double calfvenR = __builtin_fmax(
        MX4(alf(ARR, rstarRRx), fab(AstarRR) * sqRR, alf(ARL, rstarRLx), fab(AstarRL) * sqRL), smallc);
    const double calfvenB = __builtin_fmax(
        MX4(alf(BLL, rstarLLy), fab(BstarLL) * sqLL, alf(BRL, rstarRLy), fab(BstarRL) * sqRL), smallc);
    const double calfvenT = __builtin_fmax(
        MX4(alf(BLR, rstarLRy), fab(BstarLR) * sqLR, alf(BRR, rstarRRy), fab(BstarRR) * sqRR), smallc);
#undef MX4
#undef MN4
    const double SAL = __builtin_fmin(ustar - calfvenL, zero), SAR = __builtin_fmax(ustar + calfvenR, zero);
    const double SAB = __builtin_fmin(vstar - calfvenB, zero), SAT = __builtin_fmax(vstar + calfvenT, zero);
    const double SARSAL = inv_nr(SAR - SAL);
    const double SATSAB = inv_nr(SAT - SAB);
    double AstarT = (SAR * AstarRR - SAL * AstarLR) * SARSAL;
    double AstarB = (SAR * AstarRL - SAL * AstarLL) * SARSAL;
    double BstarR = (SAT * BstarRR - SAB * BstarRL) * SATSAB;
    double BstarL = (SAT * BstarLR - SAB * BstarLL) * SATSAB;
    double E;
    if (SB > zero) {
        if (SL > zero) E = ELL;
        else if (SR < zero) E = ERL;
        else E = ((SAR * EstarLLx - SAL * EstarRLx) + SAR * SAL * (BRL - BLL)) * SARSAL;
    } else if (ST < zero) {
        if (SL > zero) E = ELR;
        else if (SR < zero) E = ERR;
        else E = ((SAR * EstarLRx - SAL * EstarRRx) + SAR * SAL * (BRR - BLR)) * SARSAL;
    } else if (SL > zero) {
        E = ((SAT * EstarLLy - SAB * EstarLRy) - SAT * SAB * (ALR - ALL)) * SATSAB;
    } else if (SR < zero) {
        E = ((SAT * EstarRLy - SAB * EstarRRy) - SAT * SAB * (ARR - ARL)) * SATSAB;
    } else {
        E = (((((SAL * SAB * EstarRR - SAL * SAT * EstarRL) - SAR * SAB * EstarLR) + SAR * SAT * EstarLL) * SARSAL) * SATSAB
             - SAT * SAB * SATSAB * (AstarT - AstarB))
            + SAR * SAL * SARSAL * (BstarR - BstarL);
    }
    emf = E * dt;
    return ok;
}

// float bulk takes the hardware's approximate division and root already
__device__ __forceinline__ bool hlld1d_fast(const float*, const float*, float, double, float, float, float*, float&)
{
    return false;
}
__device__ __forceinline__ bool hlld2d_fast(const float*, const float*, const float*, const float*, float, float, float&)
{
    return false;
}

} // namespace dmx
