// lt_terms64.h -- FP64 per-(halo, pixel) terms, map epilogues and launch geometry shared by the
// FP64 kernels (lt_kernels64.hip) and the FP32-compensated kernels (lt_kernels32.hip), which fall
// back to these terms near halo cores.
//
// Formulas (restated from the mathematics; reference equivalents cited):
//   SIS gradient  src/gradient.cpp:260-299      PIEMD gradient  src/gradient.hpp:64-76,
//   dPIE gradient src/gradient.cpp:744-809      PIEMD Hessian   src/gradient2.cpp:54-82, 92-205
//   potential     src/potential_GPU.cu:47-116   epilogues       src/grid_map_*_GPU.cu
#pragma once

#include <hip/hip_runtime.h>

#include "lenstool_hip/lt_status.h"
#include "lt_device.h"
#include "lt_kernels.h"
#include "lt_math.h"

// Contraction is off from here to the end of every file that includes this: only the written FMAs are fused, so that
// each instantiation (pixels per thread, parts, tiles) evaluates the same operations on the same inputs.
#pragma clang fp contract(off)

namespace lt {

// ------------------------------------------------------------------------------------------------
// per-halo Hessian contributions, accumulated in the lab frame as
//   T = a + c (trace, rotation invariant), D = a - c, B = b.
// Halo frame -> lab frame: D' = cos2t D - 2 sin2t B, B' = sin2t D / 2 + cos2t B; the halo amplitude is
// folded into hc2 = amph cos2t and hs2 = amph sin2t.
// ------------------------------------------------------------------------------------------------

// Every term comes in two forms: at a pixel (px, py), and `_at` a lab-frame offset (tx, ty) from the
// halo centre. FULL: reciprocals and inverse square roots with the third-order correction
// (lt_math.h), for the expansion nodes of lt_far.hip, whose values many pixels share.
template <bool FULL>
__device__ __forceinline__ double rsq_c(double q)
{
    return FULL ? rsq64(q) : rsq64_n2(q);
}

template <bool FULL>
__device__ __forceinline__ double rcp_c(double x)
{
    return FULL ? rcp64(x) : rcp64_n2(x);
}

struct PixelFrame {
    double x, y, x2, y2;
};

__device__ __forceinline__ PixelFrame halo_frame_at(const HaloRec& h, double tx, double ty)
{
    PixelFrame f;
    f.x = __builtin_fma(tx, h.cs, ty * h.sn);
    f.y = __builtin_fma(ty, h.cs, -(tx * h.sn));
    f.x2 = f.x * f.x;
    f.y2 = f.y * f.y;
    return f;
}

__device__ __forceinline__ PixelFrame halo_frame(const HaloRec& h, double px, double py)
{
    return halo_frame_at(h, px - h.xh, py - h.yh);
}

// One I_{0.5} term of the PIEMD Hessian in the halo frame (Kassiola & Kovner 1993) in the
// division-free form: with s = sqrt(e), a = 1/(1+e), b = 1/(1-e), cx1 = a/b and
// w = sqrt(r^2 + a^2 x^2 + b^2 y^2), the reference's N / D (src/gradient2.cpp:54-82) equals Q / S with
// Q = r + cx1 w + 2 i s a^2 x and S = w + r cx1 + 2 s a b y, and with U = b^2 y / w + 2 s a b,
// t = 2 s w - y / cx1 the second derivatives are, up to the factor 2 s a^2 ci:
//   phi_xx ~ (Re Q - cx1 a^2 x^2 / w) / |Q|^2,  phi_xy ~ x (2 s a^2 - cx1 U) / |Q|^2,
//   phi_yy ~ (Re Q + U t) / |Q|^2.
// Re Q >= r > 0: unlike the closed form, whose two pieces are both singular at halo-frame
// (0, 2 r s) and cancel there, nothing cancels anywhere. The trace needs no quotient: (xx + yy) / |Q|^2
// = 1 / W exactly (the term's convergence, elliptical in w; with the scaled W below), so only xx - yy
// and xy are divided by |Q|^2. Returned: the numerators of xx - yy and xy, |Q|^2 and 1 / W (the
// caller forms the reciprocals of |Q|^2: one for both radii of a dPIE).
struct PiemdQ {
    double dd, xy, q2, iW;
};

// Evaluated in scaled halo-frame coordinates X = cx1 a x, Y = cx1 b y (the scales are folded into
// the rotation constants csx .. sny) with W = cx1 w: then W^2 = cx1^2 r^2 + X^2 + Y^2,
// Re Q = W + r, and with U' = U / b = Y / W + 2 s a,
//   xx = Re Q - X^2 / W,  xy = k1 X - k2 X U',  yy = Re Q + U' (k3 W - k4 Y),  Im Q = k1 X,
// k1 = 2 s a / cx1, k2 = b / a, k3 = 2 s b / cx1, k4 = 1 / cx1^2, k5 = 2 s a: every pixel-dependent
// quantity is one operation from X, Y and W. xx - yy = -(X^2 / W + U' (k3 W - k4 Y)): Re Q drops out.
struct PiemdShared {
    double wq0, Qi2, A, Y, Qi, kx2, ky4;
};

__device__ __forceinline__ PiemdShared piemd_shared(const HaloRec& h, double tx, double ty)
{
    const double X = __builtin_fma(tx, h.csx, ty * h.snx);
    PiemdShared s;
    s.Y = __builtin_fma(ty, h.csy, -(tx * h.sny));
    s.A = X * X;
    s.wq0 = __builtin_fma(s.Y, s.Y, s.A);
    s.Qi = h.k1 * X;
    s.Qi2 = s.Qi * s.Qi;
    s.kx2 = h.k2 * X;
    s.ky4 = h.k4 * s.Y;
    return s;
}

// one core radius r (r2c = cx1^2 r^2)
template <bool FULL>
__device__ __forceinline__ PiemdQ piemd_q_term(const HaloRec& h, const PiemdShared& s, double r, double r2c)
{
    const double W2 = s.wq0 + r2c;
    const double iW = rsq_c<FULL>(W2);
    const double W = W2 * iW;
    const double Qr = __builtin_fma(W2, iW, r);
    const double U = __builtin_fma(s.Y, iW, h.k5);
    PiemdQ o;
    o.dd = -__builtin_fma(s.A, iW, U * __builtin_fma(h.k3, W, -s.ky4));
    o.xy = __builtin_fma(-s.kx2, U, s.Qi);
    o.q2 = __builtin_fma(Qr, Qr, s.Qi2);
    o.iW = iW;
    return o;
}

template <bool CUT, bool FULL>
__device__ __forceinline__ void hess_piemd_at(const HaloRec& h, double tx, double ty, double& aT, double& aD,
                                              double& aB)
{
    const PiemdShared s = piemd_shared(h, tx, ty);
    const PiemdQ a = piemd_q_term<FULL>(h, s, h.rc, h.ra2c);
    double dT, dD, dB;
    if (CUT) {
        const PiemdQ b = piemd_q_term<FULL>(h, s, h.rcut, h.rb2c);
        // one reciprocal for both radii: 1/|Qa|^2 = |Qb|^2 / (|Qa|^2 |Qb|^2), and the same for b
        const double ip = rcp_c<FULL>(a.q2 * b.q2);
        const double ia = b.q2 * ip, ib = a.q2 * ip;
        dT = a.iW - b.iW;
        dD = __builtin_fma(a.dd, ia, -(b.dd * ib));
        dB = __builtin_fma(a.xy, ia, -(b.xy * ib));
    } else {
        const double ia = rcp_c<FULL>(a.q2);
        dT = a.iW;
        dD = a.dd * ia;
        dB = a.xy * ia;
    }
    // dT, dD, dB: xx + yy, xx - yy and xy of the unscaled halo-frame derivatives (the scaling cancels)
    aT = __builtin_fma(h.qT, dT, aT);
    aD = __builtin_fma(h.qc2, dD, __builtin_fma(h.qs2m2, dB, aD));
    aB = __builtin_fma(h.qs2h, dD, __builtin_fma(h.qc2, dB, aB));
}

template <bool CUT>
__device__ __forceinline__ void hess_piemd(const HaloRec& h, double px, double py, double& aT, double& aD,
                                           double& aB)
{
    hess_piemd_at<CUT, false>(h, px - h.xh, py - h.yh, aT, aD, aB);
}

// SIS / SIE: phi = b0 R, R^2 = (1-e) x^2 + (1+e) y^2; halo-frame Hessian
// amph/R^3 (y^2, -xy, x^2) with amph = b0 (1-e)(1+e).
template <bool FULL>
__device__ __forceinline__ void hess_sis_at(const HaloRec& h, double tx, double ty, double& aT, double& aD,
                                            double& aB)
{
    PixelFrame f = halo_frame_at(h, tx, ty);
    double R2 = __builtin_fma(h.sa, f.x2, h.sb * f.y2);
    double iR = rsq_c<FULL>(R2);
    double g = iR * iR * iR;
    double dyx = __builtin_fma(-f.x, f.x, f.y2);
    double xy = f.x * f.y;
    aT = __builtin_fma(g * h.amph, __builtin_fma(f.x, f.x, f.y2), aT);
    aD = __builtin_fma(g, __builtin_fma(h.hc2, dyx, 2.0 * h.hs2 * xy), aD);
    aB = __builtin_fma(g, __builtin_fma(0.5 * h.hs2, dyx, -(h.hc2 * xy)), aB);
}

__device__ __forceinline__ void hess_sis(const HaloRec& h, double px, double py, double& aT, double& aD,
                                         double& aB)
{
    hess_sis_at<false>(h, px - h.xh, py - h.yh, aT, aD, aB);
}

// Circular SIS (e = 0): the Hessian b0/r^3 (y^2, -xy, x^2) holds in any frame, so it is formed from
// the lab-frame offsets, with no rotation to the halo frame and back (T = b0 / r). The square that is formed is that of the
// offset which a lane's pixels share: the row's ty here, the column's tx in `_at` (lt_far.hip).
template <bool FULL>
__device__ __forceinline__ void hess_sis_circ_at(const HaloRec& h, double tx, double ty, double& aT, double& aD,
                                                 double& aB)
{
    const double x2 = tx * tx;
    const double iR = rsq_c<FULL>(__builtin_fma(ty, ty, x2));
    const double ga = h.amph * (iR * iR * iR);
    aT = __builtin_fma(h.amph, iR, aT);
    aD = __builtin_fma(ga, __builtin_fma(ty, ty, -x2), aD);
    aB = __builtin_fma(-ga, tx * ty, aB);
}

__device__ __forceinline__ void hess_sis_circ(const HaloRec& h, double px, double py, double& aT, double& aD,
                                              double& aB)
{
    const double tx = px - h.xh, ty = py - h.yh, y2 = ty * ty;
    const double iR = rsq64_n2(__builtin_fma(tx, tx, y2));
    const double ga = h.amph * (iR * iR * iR);
    aT = __builtin_fma(h.amph, iR, aT);
    aD = __builtin_fma(ga, __builtin_fma(-tx, tx, y2), aD);
    aB = __builtin_fma(-ga, tx * ty, aB);
}

// ------------------------------------------------------------------------------------------------
// gradient terms, accumulated in the lab frame
// ------------------------------------------------------------------------------------------------

// N conj(D) of the I_{0.5} ratio Z = N/D (N = cx1 x + i t, D = x + i n2); its real part is
// non-negative everywhere, so arg Z lies in [-pi/2, pi/2].
// Z = N / D of the reference's I_{0.5} ratio (src/gradient.hpp:64-76), N = cx1 x + i (2 s w - y / cx1),
// D = x + i (2 r s - y) with s = sqrt(e), w = sqrt(r^2 + a^2 x^2 + b^2 y^2), a = 1/(1+e), b = 1/(1-e),
// taken in the form of the Hessian's division-free derivation (lt_kernels32.hip):
//   N / D = Q / S,   Q = r + cx1 w + i 2 s a^2 x,   S = w + r cx1 + 2 s a b y > 0,
// so arg Z = arg Q (Re Q >= r > 0) and ln|Z| = ln(|Q|^2 / S^2) / 2. N and D both vanish at the
// halo-frame point (0, 2 r s) and are differences of nearly equal numbers next to it, where the closed
// form loses up to 1e-7 relative; Q and S have no such cancellation.
struct QS64 {
    double R, Q2, S;  // Re Q, |Q|^2, S
};

template <bool FULL>
__device__ __forceinline__ QS64 qs64(const HaloRec& h, double rem2, double I2, double y, double r, double r2,
                                     double rcx)
{
    const double q = r2 + rem2;
    const double iw = rsq_c<FULL>(q);
    QS64 o;
    o.R = __builtin_fma(h.cx1, q * iw, r);
    o.Q2 = __builtin_fma(o.R, o.R, I2);
    o.S = __builtin_fma(h.gkv, y, __builtin_fma(q, iw, rcx));
    return o;
}

// PIEMD (CUT = false) or dPIE (CUT = true): (ampg arg, -ampg ln|.|) of Z(rc) or Z(rc) / Z(rcut). For
// the dPIE the two logarithms and the two arguments are merged into one of each, with I = Im Q the same
// for both radii: arg(Za / Zb) = atan2(I (Rb - Ra), Ra Rb + I^2) (Ra Rb + I^2 > 0: no unwrapping) and
// ln|Za / Zb| = ln(|Qa|^2 Sb^2 / (|Qb|^2 Sa^2)) / 2.
template <bool CUT, bool FULL>
__device__ __forceinline__ void grad_piemd_at(const HaloRec& h, double tx, double ty, double& gx, double& gy)
{
    PixelFrame f = halo_frame_at(h, tx, ty);
    const double rem2 = __builtin_fma(f.x2, h.kx, f.y2 * h.ky);
    const double I = h.gki * f.x;
    const double I2 = I * I;
    const QS64 a = qs64<FULL>(h, rem2, I2, f.y, h.rc, h.ra2, h.rca);
    double arg, ratio;
    if (CUT) {
        const QS64 b = qs64<FULL>(h, rem2, I2, f.y, h.rcut, h.rb2, h.rcb);
        arg = atan2p_lt(I * (b.R - a.R), __builtin_fma(a.R, b.R, I2));
        ratio = (a.Q2 * (b.S * b.S)) * rcp_c<FULL>(b.Q2 * (a.S * a.S));
    } else {
        arg = atan2p_lt(I, a.R);
        ratio = a.Q2 * rcp_c<FULL>(a.S * a.S);
    }
    const double lnr = 0.5 * log_lt(ratio);
    const double re = h.ampg * arg;
    const double im = -h.ampg * lnr;
    gx += __builtin_fma(re, h.cs, -(im * h.sn));
    gy += __builtin_fma(im, h.cs, re * h.sn);
}

template <bool CUT>
__device__ __forceinline__ void grad_piemd(const HaloRec& h, double px, double py, double& gx, double& gy)
{
    grad_piemd_at<CUT, false>(h, px - h.xh, py - h.yh, gx, gy);
}

__device__ __forceinline__ void grad_sis_at(const HaloRec& h, double tx, double ty, double& gx, double& gy)
{
    PixelFrame f = halo_frame_at(h, tx, ty);
    double R2 = __builtin_fma(h.sa, f.x2, h.sb * f.y2);
    double s = h.ampg * rsq64(R2);
    double rx = h.sa * f.x * s;
    double ry = h.sb * f.y * s;
    gx += __builtin_fma(rx, h.cs, -(ry * h.sn));
    gy += __builtin_fma(ry, h.cs, rx * h.sn);
}

__device__ __forceinline__ void grad_sis(const HaloRec& h, double px, double py, double& gx, double& gy)
{
    grad_sis_at(h, px - h.xh, py - h.yh, gx, gy);
}

// Circular SIS: b0 (x, y) / r in any frame, formed from the lab-frame offsets.
__device__ __forceinline__ void grad_sis_circ_at(const HaloRec& h, double tx, double ty, double& gx, double& gy)
{
    const double s = h.ampg * rsq64(__builtin_fma(ty, ty, tx * tx));
    gx = __builtin_fma(s, tx, gx);
    gy = __builtin_fma(s, ty, gy);
}

__device__ __forceinline__ void grad_sis_circ(const HaloRec& h, double px, double py, double& gx, double& gy)
{
    const double tx = px - h.xh, ty = py - h.yh;
    const double s = h.ampg * rsq64(__builtin_fma(tx, tx, ty * ty));
    gx = __builtin_fma(s, tx, gx);
    gy = __builtin_fma(s, ty, gy);
}

// ------------------------------------------------------------------------------------------------
// potential (the I_{0.5} potential of Kassiola & Kovner, src/potential_GPU.cu:47-72)
// ------------------------------------------------------------------------------------------------
// The reference evaluates the potential of a core radius r with complex cosh / sinh / log of
// eta = -asinh(e1 y / z) / 2 + i asin(e2 x / z) / 2 and zeta = ln((rem + sqrt(r^2 + rem^2)) / r) / 2
// (two complex logarithms and their arguments per radius). The same function is
//   phi_r = x alpha_x + y alpha_y - 2 sqrt(e) r ln((1 + e) |Q| / (2 r))            (halo frame)
// with (alpha_x, alpha_y) = (arg Q, ln(S / |Q|)) the I_{0.5} deflection of the gradient (grad_piemd,
// without its amplitude), Q = r + cx1 w + i 2 s a^2 x, S = w + r cx1 + 2 s a b y, s = sqrt(e),
// a = 1/(1+e), b = 1/(1-e), w = sqrt(r^2 + a^2 x^2 + b^2 y^2). It is the cored isothermal-ellipsoid
// potential (x . grad phi minus the logarithmic term that makes its Laplacian 2 kappa): both forms have
// the same gradient, and both vanish in the limit at the centre, where Q = c r with c = 1 + cx1 =
// 2 / (1 + e), so they are one function (they agree to a few 1e-15 relative, checked at 40 digits
// against the extended-precision reference form by tests/test_potential_form.py). With
// d = w - r = rem^2 / (w + r), Re Q = c r + cx1 d and S = c r + d + v (v = 2 s a b y), the logarithms
//   lq = ln(|Q|^2 / (c r)^2) = log1p((cx1 d (2 c r + cx1 d) + (Im Q)^2) / (c r)^2),
//   ls = ln(S / (c r))       = log1p((d + v) / (c r))
// have arguments formed without cancellation, and phi_r = x arg Q + y (ls - lq / 2) - s r lq (PIEMD).
// For the dPIE (core radius a minus cut radius b) the deflection parts are merged, with no difference
// of nearly equal numbers near the centre or far outside the cut radius:
//   * Rb - Ra = D (c - cx1 sigma), D = rcut - rcore, sigma = (da + db) / (wa + wb) in [0, 1)
//     (db - da = -D sigma), so arg(Qa / Qb) = atan2(I (Rb - Ra), Ra Rb + I^2);
//   * alpha_y,a - alpha_y,b = ln(Sa^2 |Qb|^2 / (Sb^2 |Qa|^2)) / 2 = log1p(N / (Sb^2 |Qa|^2)) / 2 with
//     N = Pa (|Qb|^2 - |Qa|^2) + |Qa|^2 (Pa - Pb), P = S^2 - |Q|^2 = g (S + Re Q) - I^2,
//     g = S - Re Q = (1 - cx1) d + v, |Qb|^2 - |Qa|^2 = (Rb - Ra)(Rb + Ra) and
//     Pa - Pb = -ga c D (2 - sigma) + (Sb + Rb)(1 - cx1) D sigma;
// leaving per dPIE halo x pixel one arctangent and three logarithms, against three of each in the
// reference's form. Measured in a float64 emulation against 30-digit values, over halos of
// e <= 0.63 (mass ellipticity up to 0.9) at distances 1e-3 to 1e3 cut radii: within 2.1e-14 of the
// potential (5e-13 at e = 0.85, where S = w + v + cx1 r is itself a difference next to the -y axis;
// the PIEMD form within 2.6e-14 there).
// At the halo centre itself the reference's potential is 0/0 (NaN); this form gives its limit 0 there,
// so the kernels track the smallest rem^2 of a pixel over its PIEMD halos and return NaN when it is 0.
struct PotRad {
    double q, iw, d, R, lq;  // w^2, 1 / w, w - r, Re Q, ln(|Q|^2 / (c r)^2)
};

template <bool FULL>
__device__ __forceinline__ PotRad pot_rad(const HaloRec& h, double rem2, double I2, double r, double r2, double cr,
                                          double icr2)
{
    PotRad o;
    o.q = r2 + rem2;
    o.iw = rsq_c<FULL>(o.q);
    o.d = rem2 * rcp_c<FULL>(__builtin_fma(o.q, o.iw, r));
    const double cd = h.cx1 * o.d;
    o.R = __builtin_fma(h.cx1, o.d, cr);
    o.lq = log1p_mul_lt(__builtin_fma(cd, __builtin_fma(2., cr, cd), I2), icr2);
    return o;
}

// pi05 of a PIEMD (type 8) or dPIE (type 81) halo without its amplitude; mn = min(mn, rem^2).
template <bool CUT, bool FULL = false>
__device__ __forceinline__ double pot_piemd(const HaloRec& h, const PixelFrame& f, double& mn)
{
    const double rem2 = __builtin_fma(f.x2, h.kx, f.y2 * h.ky);
    mn = min64(mn, rem2);
    const double I = h.gki * f.x;
    const double I2 = I * I;
    const PotRad a = pot_rad<FULL>(h, rem2, I2, h.rc, h.ra2, h.pcra, h.picra2);
    if (!CUT) {
        const double ls = log1p_mul_lt(__builtin_fma(h.gkv, f.y, a.d), h.picra);
        const double arg = atan2p_lt(I, a.R);
        const double ay = __builtin_fma(-0.5, a.lq, ls);
        return __builtin_fma(f.x, arg, __builtin_fma(f.y, ay, -(h.psra * a.lq)));
    }
    const PotRad b = pot_rad<FULL>(h, rem2, I2, h.rcut, h.rb2, h.pcrb, h.picrb2);
    const double sig = (a.d + b.d) * rcp_c<FULL>(__builtin_fma(a.q, a.iw, b.q * b.iw));
    const double dR = h.pdr * __builtin_fma(-h.cx1, sig, h.pc);
    const double arg = atan2p_lt(I * dR, __builtin_fma(a.R, b.R, I2));
    const double Q2a = __builtin_fma(a.R, a.R, I2);
    const double v = h.gkv * f.y;
    const double Sa = __builtin_fma(h.gkv, f.y, h.pcra + a.d), Sb = __builtin_fma(h.gkv, f.y, h.pcrb + b.d);
    const double ga = __builtin_fma(h.pomc, a.d, v);
    const double Pa = __builtin_fma(ga, Sa + a.R, -I2);
    const double dP = __builtin_fma(Sb + b.R, h.pomcdr * sig, -(ga * (h.pcdr * (2. - sig))));
    const double N = __builtin_fma(Pa, dR * (a.R + b.R), Q2a * dP);
    const double ay = 0.5 * log1p_mul_lt(N, rcp_c<FULL>((Sb * Sb) * Q2a));
    const double L = __builtin_fma(h.psra, a.lq, -(h.psrb * b.lq));
    return __builtin_fma(f.x, arg, __builtin_fma(f.y, ay, -L));
}

// One halo's potential at an offset from its centre added to acc (SIS: b0 R, R^2 = (1-e) x^2 + (1+e) y^2).
template <bool FULL>
__device__ __forceinline__ void add_pot_halo(const HaloRec& h, int type, double tx, double ty, double& acc, double& mn)
{
    const PixelFrame f = halo_frame_at(h, tx, ty);
    const double v = type == TYPE_SIS     ? sqrt(__builtin_fma(h.sa, f.x2, h.sb * f.y2))
                     : type == TYPE_PIEMD ? pot_piemd<false, FULL>(h, f, mn)
                                          : pot_piemd<true, FULL>(h, f, mn);
    acc = __builtin_fma(h.ampg, v, acc);
}

// ------------------------------------------------------------------------------------------------
// epilogues (src/grid_map_ampli_GPU.cu:329-572, grid_map_shear_GPU.cu:208-342,
// grid_map_mass_GPU.cu:307-322); T, D, B are the Hessian sums a+c, a-c, b.
// The map kind is a template parameter, and within a kind the mode picks the value by a scalar branch
// ahead of the store, so each kernel has a single store per output plane with a fixed base pointer.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ void eigen(double A, double B, double C, double& lam, double& mu)
{
    double e = sqrt(__builtin_fma(A - C, A - C, 4. * B * B));
    lam = .5 * (A + C + e);
    mu = .5 * (A + C - e);
}

// -2.5 log10(x), x >= 0: the library's log10 for zero, infinity, NaN and the largest and smallest numbers
__device__ __forceinline__ double magnitudes(double x)
{
    // 2^-1000 <= x < 2^1000 by the upper word
    if ((uint32_t)__double2hiint(x) - 0x01700000u < 0x7d000000u) return magnitudes_lt(x);
    return -2.5 * log10(x);
}

template <int KIND>
__device__ __forceinline__ void hess_epilogue(const OutDesc& o, int64_t idx, double T, double D, double B)
{
    const double a = 0.5 * (T + D), c = 0.5 * (T - D), b = B;
    const double r = o.r;
    if constexpr (KIND == LT_MAP_HESSIAN) {
        if (o.p0) o.p0[idx] = a;
        if (o.p1) o.p1[idx] = b;
        if (o.p2) o.p2[idx] = c;
        if (o.p3) o.p3[idx] = b;
    } else if constexpr (KIND == LT_MAP_FIELDS) {
        double kappa = 0.5 * T * r, g1 = 0.5 * D * r, g2 = B * r;
        double omk = 1. - kappa;
        double det = __builtin_fma(omk, omk, -__builtin_fma(g1, g1, g2 * g2));
        if (o.p0) o.p0[idx] = kappa;
        if (o.p1) o.p1[idx] = g1;
        if (o.p2) o.p2[idx] = g2;
        if (o.p3) o.p3[idx] = det;
        if (o.p4) o.p4[idx] = 1. / det;
    } else if constexpr (KIND == LT_MAP_AMPLI) {
        // the mode is the same for the whole launch: a scalar branch, and one store after it (with every mode's
        // value formed and one selected, 256 maps of 2048^2 and 11 halos took 13.2 ms in mode 3, 9.7 so; in mode
        // 1, 64 maps, 2.69 and 2.31; shear modes 2.48 and 2.23; mass maps, which now need T alone, 1.99 and 1.30)
        double v;
        if (o.mode <= 3) {
            // det A, the product of the eigenvalues of 1 - r H, without their square root
            const double omk = 1. - 0.5 * T * r, g1 = 0.5 * D * r, g2 = B * r;
            const double det = __builtin_fma(omk, omk, -__builtin_fma(g1, g1, g2 * g2));
            if (o.mode == 1) v = 1. / det;
            else if (o.mode == 2) v = 1. / fabs(det);
            else v = magnitudes(fabs(det));
        } else if (o.mode == 4) {
            const double kappa = (a + c) * r / 2., ga1 = (a - c) * r / 2., ga2 = b * r;
            const double gp = sqrt(__builtin_fma(ga1, ga1, ga2 * ga2)) / (1 - kappa);
            v = (1 - kappa) * __builtin_fma(gp, gp, 1.) / __builtin_fma(-gp, gp, 1.);
        } else if (o.mode == 5) {
            v = (a + c) / 2.;                                                   // kappa, no dlsds
        } else {
            const double h1 = (a - c) / 2.;
            v = sqrt(__builtin_fma(h1, h1, b * b));                             // 6: gamma, no dlsds
        }
        o.p0[idx] = v;
    } else if constexpr (KIND == LT_MAP_SHEAR) {
        double v;
        if (o.mode <= 2) {
            double lam, mu;
            eigen(__builtin_fma(-a, r, 1.), -b * r, __builtin_fma(-c, r, 1.), lam, mu);
            const double q = lam / mu;
            v = o.mode == 1 ? (lam - mu) / 2. : fabs(__builtin_fma(q, q, -1.) / __builtin_fma(q, q, 1.));
        } else {
            v = o.mode == 3 ? (a - c) * r / 2. : b * r;                         // gamma1, gamma2
        }
        o.p0[idx] = v;
    } else {  // LT_MAP_MASS: kappa from the trace alone
        o.p0[idx] = T * 0.5 * o.mult;
    }
}

// ------------------------------------------------------------------------------------------------
// kernels
// ------------------------------------------------------------------------------------------------
constexpr int WAVE = 64;
constexpr int ROWS = 4;

// orders a wavefront's own LDS accesses: what its lanes wrote before is what they read after
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sample s of a batch (blockIdx.z) uses its own halo records and output planes.
__device__ __forceinline__ const HaloRec* select_sample(const GridDesc& g, const HaloRec* halos, OutDesc& o)
{
    const int64_t s = blockIdx.z;
    const int64_t off = s * g.plane_stride;
    if (o.p0) o.p0 += off;
    if (o.p1) o.p1 += off;
    if (o.p2) o.p2 += off;
    if (o.p3) o.p3 += off;
    if (o.p4) o.p4 += off;
    return halos + s * g.halo_stride;
}

// How the halos of a pixel are summed: one after another by a wave; in kSplit parts (part p takes halos p, p + kSplit, ..
// of the model) by as many waves, whose sums are then added in the order of the parts; or the same parts one after
// another by one wave. The last two give the same bits: waves where a launch leaves the chip idle, one wave
// where it does not (a batch of small maps).
enum : int { SUM_PLAIN = 0, SUM_WAVES = 1, SUM_PARTS = 2 };

constexpr int parts_of(int form) { return form == SUM_PLAIN ? 1 : kSplit; }
constexpr int rows_of(int form) { return form == SUM_WAVES ? kSplit : ROWS; }  // waves of a work-group

// the halos of a run that belong to part `wave`: first, first + SPLIT, ..
template <int SPLIT>
__device__ __forceinline__ int first_halo(int start, int wave)
{
    return SPLIT == 1 ? start : start + ((wave - start) & (SPLIT - 1));
}

// sums of PX pixels over the SPLIT waves of a row segment: wave k gets those of its k-th pixel column, in v[0]; false
// for the waves that have none to store. Every wave of the work-group calls it.
template <int PX, int SPLIT, typename... V>
__device__ __forceinline__ bool split_sum(int wave, V&... v)
{
    __shared__ double part[SPLIT][sizeof...(V)][PX][WAVE];
    const int lane = threadIdx.x;
    int f = 0;
    auto put = [&](const double* x) {
#pragma unroll
        for (int k = 0; k < PX; ++k) part[wave][f][k][lane] = x[k];
        ++f;
    };
    (put(v), ...);
    __syncthreads();
    if (wave >= PX) return false;
    f = 0;
    auto get = [&](double* x) {
        double t = part[0][f][wave][lane];
#pragma unroll
        for (int p = 1; p < SPLIT; ++p) t += part[p][f][wave][lane];
        x[0] = t;
        ++f;
    };
    (get(v), ...);
    return true;
}

// the sums t of a part, of PX pixels, added to those of the parts before it, in the order of split_sum() (a part without
// halos is left out: it is +0 there)
template <int PX>
__device__ __forceinline__ void add_part(double* sum, const double* t)
{
#pragma unroll
    for (int k = 0; k < PX; ++k) sum[k] += t[k];
}

// Launch geometry: a 64 x 4 work-group, PX pixels per thread along a row, blockIdx.z = sample.
inline dim3 grid_for(const GridDesc& g, int px)
{
    return dim3((unsigned)((g.nx + WAVE * px - 1) / (WAVE * px)), (unsigned)((g.ny + ROWS - 1) / ROWS),
                (unsigned)(g.nsamples > 0 ? g.nsamples : 1));
}

// launch geometry: as grid_for(); for SUM_WAVES a work-group per row and 64 PX columns
template <int PX, int FORM>
inline void geometry(const GridDesc& g, dim3& grd, dim3& blk)
{
    grd = grid_for(g, PX);
    blk = dim3(WAVE, rows_of(FORM), 1);
    if (FORM == SUM_WAVES) grd.y = (unsigned)g.ny;
}

// pixels per thread of a SUM_PARTS launch: two, or one where the columns past the grid of two (whole segments of 128)
// cost more than the record loads that two pixels share (`share`: times of one pixel a thread to two, measured)
inline int parts_px(const GridDesc& g, double share)
{
    const auto cover = [&](int seg) { return (double)((g.nx + seg - 1) / seg * seg); };
    return cover(WAVE) * share < cover(2 * WAVE) ? 1 : 2;
}

}  // namespace lt
