// Point-wise end of the evaluation pipeline: the total potential and the
// energy sums of one grid point from rho and the inverse transforms of its
// spectra, and the analytic Hessian product's (kernels in eval.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

#include "../../include/ofdft_hip.h"
#include "fastmath.h"

namespace ofdft {

struct PostParams {
    int s_vw, s_wt, s_h;
    int s_wt2 = -1;  // alpha != beta: IFFT(K FFT(rho^alpha))
    const void *core = nullptr;  // NLCC: the XC term sees rho + core
    int b56;  // beta == 5/6
    unsigned terms;
    double x, y, alpha, beta;
    long long n;
    long long bs;  // work batch stride (reals)
    int want_v, want_e;
};

// PZ LDA constants (semilocal_xc.py:257-263)
constexpr double PZ_A = 0.0311, PZ_B = -0.048, PZ_C = 0.0020, PZ_D = -0.0116;
constexpr double PZ_G = -0.1423, PZ_B1 = 1.0529, PZ_B2 = 0.3334;
// 3/10 (3 pi^2)^(2/3), (3 / 4 pi)^(1/3), (3 / pi)^(1/3): literals, because the
// device library's pow and cbrt of constants are evaluated per thread
constexpr double kCtf = 2.871234000188191, kCbrt34Pi = 0.6203504908994001, kCbrt3Pi = 0.9847450218426965;

// Reciprocal and reciprocal square root: the hardware approximations (about
// 1 ulp) for the FP32-bulk pipeline; in FP64 the reciprocal by Newton steps
// (without the library division's scaling) and the library root.
template <typename CT> __device__ __forceinline__ CT rcp_p(CT x) { return fm::rcp(x); }
template <> __device__ __forceinline__ double rcp_p<double>(double x) { return fm::div_n(1.0, x); }
template <typename CT> __device__ __forceinline__ CT rsq_p(CT x) { return fm::rsq(x); }

// The powers of the density at a point that its terms use.  FP64 takes them
// all from one inverse sixth root (fastmath.h).
template <typename CT> struct RhoPowers {
    CT cr;     // cbrt(rho)
    CT isq;    // 1 / sqrt(rho > 0 ? rho : 1e-30)
    CT rb_rc;  // rho^(5/6) / rho of max(rho, 1e-30)
};
template <typename CT> __device__ __forceinline__ RhoPowers<CT> rho_powers(CT r) {
    RhoPowers<CT> w;
    const CT rc = r < (CT)1e-30 ? (CT)1e-30 : r;
    w.cr = fm::cbrt(r);
    w.isq = rsq_p<CT>((r > (CT)0 && r < (CT)1e-30) ? r : rc);
    w.rb_rc = (r < (CT)1e-30 ? (CT)1e-10 : w.cr) * rsq_p<CT>(rc);
    return w;
}
template <> __device__ __forceinline__ RhoPowers<double> rho_powers(double r) {
    RhoPowers<double> w;
    const double a = fabs(r);
    const fm::SixthRoot s(a);
    w.cr = (a > 0.0 && a < (double)INFINITY) ? copysign(s.cbrt(), r) : r;
    w.isq = r <= 0.0 ? 1e15 : (a < (double)INFINITY ? s.rsq() : (a == a ? 0.0 : a));
    w.rb_rc = r < 1e-30 ? 1e5 : s.inv_sixth();
    return w;
}

// PZ correlation at rs: energy per electron and potential
template <typename CT> __device__ __forceinline__ void pz_corr(CT rs, CT &ec, CT &vc) {
    if (rs < (CT)1) {
        const CT lr = fm::log(rs);
        ec = (CT)PZ_A * lr + (CT)PZ_B + (CT)PZ_C * rs * lr + (CT)PZ_D * rs;
        vc = lr * ((CT)PZ_A + (CT)(2.0 / 3.0 * PZ_C) * rs) + (CT)PZ_B - (CT)(1.0 / 3.0 * PZ_A) +
             (CT)(1.0 / 3.0 * (2 * PZ_D - PZ_C)) * rs;
    } else {
        const CT sr = fm::sqrt(rs);
        const CT iden = rcp_p<CT>((CT)1 + (CT)PZ_B1 * sr + (CT)PZ_B2 * rs);
        ec = (CT)PZ_G * iden;
        vc = ((CT)PZ_G + (CT)(7.0 / 6.0 * PZ_G * PZ_B1) * sr + (CT)(4.0 / 3.0 * PZ_G * PZ_B2) * rs) * (iden * iden);
    }
}

// One point: av, cv, c2v, hv the inverse transforms of the vW, WT, second WT
// and Hartree spectra, lv the local potential, corev the core density (each
// read only where its term is present).  acc: the seven sums of the energy
// terms (TF, vW, WT, XC, Hartree, PP, electrons).
template <typename CT>
__device__ __forceinline__ CT post_point(const PostParams &p, bool has_vloc, CT r, CT av, CT cv, CT c2v, CT hv, CT lv,
                                         CT corev, double (&acc)[7]) {
    const CT ctf = (CT)kCtf;
    const CT cbrt34pi = (CT)kCbrt34Pi;
    const CT cx_e = (CT)(-3.0 / 4.0 * kCbrt3Pi);
    const CT cx_v = (CT)(-kCbrt3Pi);
    CT v = (CT)0;
    const RhoPowers<CT> w = rho_powers<CT>(r);
    if (p.terms & OFDFT_TERM_TF) {
        const CT c2 = w.cr * w.cr;  // rho^(2/3)
        if (p.want_e) acc[0] += (double)(ctf * c2 * r);
        v += (CT)p.x * ((CT)(5.0 / 3.0) * ctf * c2);
    }
    if (p.s_vw >= 0) {
        const CT vw = (CT)p.y * (av * w.isq);
        if (p.want_e && r > (CT)0) acc[1] += (double)(r * vw);
        v += vw;
    }
    if (p.s_wt >= 0 && p.s_wt2 < 0) {
        const CT rc = r < (CT)1e-30 ? (CT)1e-30 : r;
        const CT rb_rc = p.b56 ? w.rb_rc : fm::pow(rc, (CT)p.beta) * rcp_p<CT>(rc);  // rho^beta / rho
        const CT vnl = (CT)(2.0 * p.alpha) * rb_rc * cv;
        if (p.want_e) acc[2] += (double)(vnl * r) * (0.5 / p.alpha);
        v += vnl;
    } else if (p.s_wt >= 0) {
        // alpha != beta (wt.py:23-25,44-56): cb = K * rho^beta, ca = K * rho^alpha
        const CT rc = r < (CT)1e-30 ? (CT)1e-30 : r;
        const CT cb = cv;
        const CT ca = c2v;
        const CT ra = fm::pow(rc, (CT)p.alpha), rb = fm::pow(rc, (CT)p.beta);
        const CT irc = rcp_p<CT>(rc);
        if (p.want_e) acc[2] += (double)(ra * cb);
        v += (CT)p.alpha * ra * irc * cb + (CT)p.beta * rb * irc * ca;
    }
    if (p.terms & OFDFT_TERM_XC) {
        // xc/__init__.py:59-74: with a core density the XC term is
        // evaluated at rho + core (energy sum_r eps(rho+core)(rho+core) dV)
        CT rx = r, rc3 = w.cr;
        if (p.core) {
            rx = r + corev;
            rc3 = fm::cbrt(rx);
        }
        if (rc3 < (CT)1e-30) rc3 = (CT)1e-30;
        CT ec, vc;
        pz_corr<CT>(cbrt34pi * rcp_p<CT>(rc3), ec, vc);
        if (p.want_e) acc[3] += (double)((cx_e * rc3 + ec) * rx);
        v += cx_v * rc3 + vc;
    }
    if (p.s_h >= 0) {
        if (p.want_e) acc[4] += 0.5 * (double)hv * (double)r;
        v += hv;
    }
    if (has_vloc) {
        if (p.want_e) acc[5] += (double)lv * (double)r;
        v += lv;
    }
    acc[6] += (double)r;
    return v;
}

// One point of the analytic Hessian product a = (V - mu) p + phi dV[2 phi p]:
// av, cv, hv the inverse transforms of the linear-response spectra, bav =
// 1/2 L(sqrt(rho)) and bcv = C(rho^beta) of the evaluation at rho.
template <typename T, typename CT>
__device__ __forceinline__ T hvp_point(const PostParams &pp, double m, T phi_i, T p_i, T rho_i, T pot_i, CT bav, CT avw,
                                       CT bcv, CT cwt, CT hv, double &acc) {
    const CT ctf = (CT)kCtf;
    const CT cbrt34pi = (CT)kCbrt34Pi;
    const CT cx3 = (CT)(-kCbrt3Pi / 3.0);
    const CT r = (CT)rho_i, dr = (CT)(T)(2.0 * (double)phi_i * (double)p_i);  // drho = 2 phi p
    const CT rp = r > (CT)1e-30 ? r : (CT)1e-30;
    const CT c_rp = fm::cbrt(rp);
    const CT ic = rcp_p<CT>(c_rp);  // rho^(-1/3)
    const CT irp = ic * ic * ic;    // 1 / rho
    CT dv = (CT)0;
    if (pp.terms & OFDFT_TERM_TF) dv += (CT)pp.x * (CT)(10.0 / 9.0) * ctf * ic * dr;  // tf.py:38-40
    if (pp.s_vw >= 0) {
        const CT isq = rsq_p<CT>((r > (CT)0 && r < (CT)1e-30) ? r : rp);  // 1 / sqrt(rho > 0 ? rho : 1e-30)
        const CT ds = (CT)0.5 * dr * isq;
        const CT vwb = (CT)pp.y * bav * isq;
        dv += ((CT)pp.y * avw - vwb * ds) * isq;
    }
    if (pp.s_wt >= 0) {
        const CT rb1 = pp.b56 ? c_rp * rsq_p<CT>(rp) : fm::pow(rp, (CT)pp.beta - (CT)1);  // rho^(beta-1)
        dv += (CT)(2.0 * pp.alpha) * (((CT)pp.beta - (CT)1) * rb1 * irp * dr * bcv + rb1 * cwt);
    }
    if (pp.terms & OFDFT_TERM_XC) {
        // semilocal_xc.py:291-303
        const CT rs = cbrt34pi * ic;
        CT fc;
        if (rs < (CT)1) {
            fc = -(CT)(PZ_A / 3.0) - ((CT)(PZ_C / 9.0) * (fm::log(rs) * (CT)2 + (CT)1) + (CT)(PZ_D * 2.0 / 9.0)) * rs;
        } else {
            const CT ta = (CT)PZ_B1 * fm::sqrt(rs), tb = (CT)PZ_B2 * rs;
            const CT ide = rcp_p<CT>((CT)1 + ta + tb);
            fc = (CT)(PZ_G / 36.0) *
                 ((CT)5 * ta + (CT)7 * ta * ta + (CT)8 * tb + (CT)16 * tb * tb + (CT)21 * ta * tb) * (ide * ide * ide);
        }
        dv += (cx3 * c_rp + fc) * irp * dr;
    }
    if (pp.s_h >= 0) dv += hv;
    const double a = ((double)pot_i - m) * (double)p_i + (double)phi_i * (double)dv;
    acc += (double)p_i * (double)(T)a;
    return (T)a;
}

}  // namespace ofdft
