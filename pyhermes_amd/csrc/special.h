// Device special functions and window transfer functions.
//
// *_f64: faithful FP64 restatements of the reference algorithms
//   spherical_jn_numba      special_functions.py:49-128
//   assoc_legendre_numba, spherical_harmonic_numba  special_functions.py:273-334 (without angles)
//   window transfer kernels window_functions.py:29-129, :426-438
// *_f32: the FP32 fast path used by the batched kernels (no acos/atan2: Y_lm is
//   evaluated from ((kx + i ky)/|k|)^m and the Legendre polynomial part, j_l from
//   an exact revolution count and upward recurrence / power series).
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/hermes_amd.h"

#define HERMES_PI 3.14159265358979323846

// ------------------------------------------------------------------ FP64 faithful
// Cylindrical Bessel J_NU(x), NU = 0 or 1, x = 2 pi t >= 0, to FP64 rounding (the reference's jn_numba,
// special_functions.py:131-270, uses 8-digit rational approximations instead):
//   x <= 4       the power series (x/2)^NU sum_k (-x^2/4)^k / (k! (k+NU)!) (largest term 4, so little
//                cancellation), by Horner's rule;
//   4 < x < 25   Miller's backward recurrence J_{n-1} = (2n/x) J_n - J_{n+1} from n = x + 10 sqrt(x) + 30,
//                normalised by J0 + 2 (J2 + J4 + ...) = 1 (values stay below 1e60 on the way down);
//   x >= 25      Hankel's asymptotic expansion sqrt(2/(pi x)) (P cos w - Q sin w), w = x - (2 NU + 1) pi/4, with
//                a_k = a_{k-1} (4 NU^2 - (2k-1)^2) / (8k), P = sum (-1)^k a_{2k} / x^{2k} and
//                Q = sum (-1)^k a_{2k+1} / x^{2k+1}, by Horner's rule up to k = 25 (below 1e-17 at x = 25);
//                sin and cos of x from the exact turn fraction t - floor(t).
template <int NU>
struct BesselCoef {
    static constexpr int NS = 18, NH = 13;
    double series[NS + 1];      // (-1)^k / (k! (k + NU)!)
    double hp[NH], hq[NH];      // (-1)^k a_{2k}, (-1)^k a_{2k+1}
    constexpr BesselCoef() : series{}, hp{}, hq{} {
        double t = 1.0;
        for (int k = 0; k <= NS; ++k) {
            series[k] = t;
            t /= -(double)((k + 1) * (k + 1 + NU));
        }
        double a = 1.0;
        for (int k = 0; k < 2 * NH; ++k) {
            const double sg = (k / 2) % 2 ? -1.0 : 1.0;
            if (k % 2) hq[k / 2] = sg * a;
            else hp[k / 2] = sg * a;
            a *= (4.0 * NU * NU - (2.0 * k + 1.0) * (2.0 * k + 1.0)) / (8.0 * (k + 1.0));
        }
    }
};

template <int NU>
__device__ inline double bessel_j_f64(double t) {
    constexpr BesselCoef<NU> B{};
    const double x = 2.0 * HERMES_PI * t;
    if (x <= 4.0) {
        const double h = 0.25 * x * x;
        double s = B.series[BesselCoef<NU>::NS];
#pragma unroll
        for (int k = BesselCoef<NU>::NS - 1; k >= 0; --k) s = fma(s, h, B.series[k]);
        return NU ? 0.5 * x * s : s;
    }
    if (x < 25.0) {
        const int n0 = 2 * (((int)(x + 10.0 * sqrt(x)) + 30) / 2);  // even start
        const double tox = 2.0 / x;
        // two steps at a time: jp = J_n (even n), jc = J_{n-1}; even_sum gathers J_2, J_4, ...
        double jp = 0.0, jc = 1e-30, even_sum = 0.0;
        for (int n = n0; n >= 2; n -= 2) {
            jp = fma((double)n * tox, jc, -jp);          // J_{n-1} from J_n (jc), J_{n+1} (jp)
            jc = fma((double)(n - 1) * tox, jp, -jc);    // J_{n-2}
            even_sum += jc;
        }
        const double norm = 2.0 * even_sum - jc;  // J0 + 2 (J2 + J4 + ...), jc = J0 counted twice in the sum
        return (NU ? jp : jc) / norm;
    }
    const double r = 1.0 / x, r2 = r * r;
    double P = B.hp[BesselCoef<NU>::NH - 1], Q = B.hq[BesselCoef<NU>::NH - 1];
#pragma unroll
    for (int k = BesselCoef<NU>::NH - 2; k >= 0; --k) {
        P = fma(P, r2, B.hp[k]);
        Q = fma(Q, r2, B.hq[k]);
    }
    Q *= r;
    // cos w and sin w from those of x: w = x - pi/4 (NU = 0) or x - 3 pi/4 (NU = 1); 1/sqrt(2) in the factor
    double s, c;
    sincospi(2.0 * (t - floor(t)), &s, &c);
    const double cw = NU ? s - c : c + s, sw = NU ? -(s + c) : s - c;
    return sqrt(r * (1.0 / HERMES_PI)) * (P * cw - Q * sw);
}

// Perpendicular factor of the line-of-sight windows at q = 2 pi t, t = k_perp R: J0 (ring, cylshell) or 2 J1(q)/q.
__device__ inline double los_perp_f64(bool ring, double t) {
    if (ring) return bessel_j_f64<0>(t);
    return t == 0.0 ? 1.0 : bessel_j_f64<1>(t) / (HERMES_PI * t);
}

// sum_k (-h/2)^k / (k! (2l+3)(2l+5)...(2l+2k+1)), h = x^2: j_l(x) (2l+1)!! / x^l.
template <int LO, int TERMS>
__device__ __forceinline__ double jl_series(double h) {
    double s = 1.0;
#pragma unroll
    for (int k = TERMS; k >= 1; --k) s = fma(s, h * (-1.0 / (2.0 * k * (2.0 * LO + 2.0 * k + 1.0))), 1.0);
    return s;
}

// sin and cos of 2 pi t from the exact turn fraction.
__device__ __forceinline__ void sincos_turns(double t, double* s, double* c) { sincospi(2.0 * (t - floor(t)), s, c); }

// j_l(2 pi t)
__device__ inline double jl_f64(int l, double t) {
    if (l < 0) return __builtin_nan("");
    if (t == 0.0) return l == 0 ? 1.0 : 0.0;
    const double x = 2.0 * HERMES_PI * t, ax = fabs(x);
    if (ax <= 5.0e-2) {  // the reference's truncated series
        double lead = 1.0;
        for (int n = 1; n <= l; ++n) lead *= x / (2.0 * n + 1.0);
        const double x2 = x * x;
        return lead * (1.0 - x2 / (2.0 * (2.0 * l + 3.0)) + x2 * x2 / (8.0 * (2.0 * l + 3.0) * (2.0 * l + 5.0)));
    }
    const double ix = 1.0 / x;
    double sx, cx;
    sincos_turns(t, &sx, &cx);
    const double j0 = sx * ix;
    if (l == 0) return j0;
    const double j1 = (j0 - cx) * ix;
    if (l == 1) return j1;
    if (ax < l + 1.0) {
        int n_stop = l + 40;
        double jp1 = 0.0, jcur = 1.0, jt = 0.0, jd0 = 0.0, jd1 = 0.0;
        for (int n = n_stop; n > 0; --n) {
            double jm1 = fma((2.0 * n + 1.0) * ix, jcur, -jp1);
            if (n - 1 == l) jt = jm1;
            if (n - 1 == 1) jd1 = jm1;
            if (n - 1 == 0) jd0 = jm1;
            jp1 = jcur;
            jcur = jm1;
            if (fabs(jcur) > 1.0e200) {
                jp1 *= 1.0e-200; jcur *= 1.0e-200; jt *= 1.0e-200; jd0 *= 1.0e-200; jd1 *= 1.0e-200;
            } else if (fabs(jcur) < 1.0e-200 && jcur != 0.0) {
                jp1 *= 1.0e200; jcur *= 1.0e200; jt *= 1.0e200; jd0 *= 1.0e200; jd1 *= 1.0e200;
            }
        }
        if (fabs(jd0) >= fabs(jd1) || jd1 == 0.0) return jt * (j0 / jd0);
        return jt * (j1 / jd1);
    }
    double jm1 = j0, jcur = j1;
    for (int ell = 1; ell < l; ++ell) {
        const double jn = fma((2.0 * ell + 1.0) * ix, jcur, -jm1);
        jm1 = jcur;
        jcur = jn;
    }
    return jcur;
}

// Y_l^m of a fixed (l, m) without angles: norm poly(mu) ((kx + i ky) / k)^|m| with poly the part of P_l^|m|
// free of (1 - mu^2)^(|m|/2), by its recurrence in l with coefficients tabulated on the host.
struct YlmTable {
    int l, m;
    double norm;           // N_l|m| (-1)^|m| (2|m| - 1)!!
    double a[41], b[41];   // poly_n = a[n] mu poly_{n-1} - b[n] poly_{n-2}, |m| + 2 <= n <= l
};

// ik = 1 / |k|, 0 for k = 0 (where Y_00 is its constant and every other order 0).
__device__ inline double2 ylm_f64(const YlmTable& Y, double kx, double ky, double kz, double ik) {
    const int am = Y.m < 0 ? -Y.m : Y.m;
    const double mu = kz * ik, ur = kx * ik, ui = ky * ik;
    double p = 1.0, q = (2.0 * am + 1.0) * mu;
    if (Y.l == am) q = 1.0;
    for (int n = am + 2; n <= Y.l; ++n) {
        const double r = fma(Y.a[n] * mu, q, -Y.b[n] * p);
        p = q;
        q = r;
    }
    double pr = Y.norm * q, pi = 0.0;
    for (int i = 0; i < am; ++i) {
        const double t = pr * ur - pi * ui;
        pi = pr * ui + pi * ur;
        pr = t;
    }
    if (ik == 0.0 && Y.l > 0) pr = pi = 0.0;
    if (Y.m < 0) {  // Y_{l,-m} = (-1)^m conj(Y_{l,m})
        const double sg = (am & 1) ? -1.0 : 1.0;
        return make_double2(sg * pr, -sg * pi);
    }
    return make_double2(pr, pi);
}

// N_l0 P_l(mu), the real spherical harmonic of m = 0 (0 at k = 0 unless l = 0: mu is then 0 and ik 0).
__device__ inline double yl0_f64(int l, double mu) {
    double p = 1.0, q = mu;
    if (l == 0) q = 1.0;
    for (int n = 2; n <= l; ++n) {
        const double r = ((2.0 * n - 1.0) * mu * q - (n - 1.0) * p) / n;
        p = q;
        q = r;
    }
    return sqrt((2.0 * l + 1.0) / (4.0 * HERMES_PI)) * q;
}

__device__ inline double win_sphere_f64(double k, double R) {
    // 3 j_1(q) / q; below q = 1 by its series (s - q c cancels)
    const double q = 2 * HERMES_PI * (k * R), q2 = q * q;
    if (q2 < 1.0) return jl_series<1, 9>(q2);
    double s, c;
    sincos_turns(k * R, &s, &c);
    return 3 * (s - q * c) / (q2 * q);
}

// The same as a call, for kernels that take any window: inlined, the three Bessel ranges double their registers (the
// general pair reduction: 290 and one wave per SIMD; 150 and three with the call).
__device__ __attribute__((noinline)) double los_perp_call(bool ring, double t) { return los_perp_f64(ring, t); }

// Line-of-sight windows (window_functions.py:164-319).  Along a coordinate axis they are even in every
// component of k, so the octant folds apply to them as to the isotropic ones; along any other direction
// they are only even under k -> -k (the half-spectrum sums still apply, the octant sharing does not).
// axis 3: the unit vector n (k_par = k . n, k_perp from |k|^2 - k_par^2, window_functions.py:164-319).
__device__ inline double los_window_f64(int type, double ki, double kj, double kk, double R, double H, int axis,
                                        const double* n = nullptr) {
    double kpar, kperp2;
    if (n != nullptr && axis == 3) {
        kpar = ki * n[0] + kj * n[1] + kk * n[2];
        kperp2 = fmax(ki * ki + kj * kj + kk * kk - kpar * kpar, 0.0);
    } else {
        kpar = axis == 0 ? ki : (axis == 1 ? kj : kk);
        const double u = axis == 0 ? kj : ki, v = axis == 2 ? kj : kk;  // the two perpendicular components
        kperp2 = u * u + v * v;
    }
    const double qpar = 2.0 * HERMES_PI * kpar * H;
    const double perp = los_perp_call(type == HERMES_WIN_RING || type == HERMES_WIN_CYLSHELL, sqrt(kperp2) * R);
    const double par = (type == HERMES_WIN_RING || type == HERMES_WIN_DISK)
                           ? cos(qpar)
                           : (qpar == 0.0 ? 1.0 : sin(qpar) / qpar);
    return perp * par;
}

// Transfer function of one isotropic window at |k| = k cycles per grid cell.
__device__ inline double isotropic_f64(int type, double k, double a0, double a1) {
    switch (type) {
    case HERMES_WIN_SPHERE: return win_sphere_f64(k, a0);
    case HERMES_WIN_GAUSSIAN: {
        double q = 2 * HERMES_PI * k * a0;
        return exp(-(q * q) / 2);
    }
    case HERMES_WIN_SHELL: {
        const double q = 2 * HERMES_PI * (k * a0);
        if (q == 0.0) return 1.0;
        return sinpi(2.0 * (k * a0 - floor(k * a0))) / q;
    }
    case HERMES_WIN_THICK_SHELL: {
        double ri = a0 - 0.5 * a1;
        if (ri < 0.0) ri = 0.0;
        double ro = a0 + 0.5 * a1;
        double den = ro * ro * ro - ri * ri * ri;
        if (den == 0.0) return 1.0;
        return (ro * ro * ro * win_sphere_f64(k, ro) - ri * ri * ri * win_sphere_f64(k, ri)) / den;
    }
    case HERMES_WIN_GAUSSIAN_SHELL: {
        if (k == 0) return 1.0;
        double qs = 2 * HERMES_PI * (k * a0);
        double qm = 2 * HERMES_PI * k * a1;
        double den = a0 * a0 + a1 * a1;
        if (den == 0.0) return 1.0;
        double sn, cs;
        sincos_turns(k * a0, &sn, &cs);
        double sinc = (qs == 0.0) ? 1.0 : sn / qs;
        return (a1 * a1 * cs + a0 * a0 * sinc) / den * exp(-(qm * qm) / 2);
    }
    case HERMES_WIN_INVERSE_LAPLACIAN:
        if (k == 0.0) return 0.0;
        return -1.0 / (((2.0 * HERMES_PI) * (2.0 * HERMES_PI)) * (k * k));
    }
    return __builtin_nan("");
}

// The same for any real, even window at k: the isotropic ones and, unless LOS is false, the line-of-sight ones.
template <bool LOS = true>
__device__ inline double iso_window_f64(int type, double ki, double kj, double kk, double a0, double a1,
                                        int axis = 2, const double* los = nullptr) {
    if (LOS && type >= HERMES_WIN_RING && type <= HERMES_WIN_CYLINDER)
        return los_window_f64(type, ki, kj, kk, a0, a1, axis, los);
    return isotropic_f64(type, sqrt(ki * ki + kj * kj + kk * kk), a0, a1);
}

// U_l(k) of a radial profile at k cycles per grid cell (hermes_radial_profile; FP64).
__device__ inline double radial_table_f64(const double* __restrict__ tab, int n, double x) {
    // x = k * k_scale, the fractional table index; radial_multipole_windows.py:186-210 lookup
    if (x <= 0.0) return tab[0];
    if (x >= (double)(n - 1)) return tab[n - 1];
    const int i = (int)x;
    const double t = x - i;
    if (i == 0 || i >= n - 2) return tab[i] * (1.0 - t) + tab[i + 1] * t;
    const double p0 = tab[i - 1], p1 = tab[i], p2 = tab[i + 1], p3 = tab[i + 2];
    return p1 + 0.5 * t * ((p2 - p0) + t * ((2.0 * p0 - 5.0 * p1 + 4.0 * p2 - p3) + t * (3.0 * (p1 - p2) + p3 - p0)));
}

__device__ inline double radial_profile_f64(const hermes_radial_profile& p, int l, double k) {
    switch (p.kind) {
    case HERMES_RADIAL_SHELL: return jl_f64(l, k * p.a0);
    case HERMES_RADIAL_TABLE: return radial_table_f64(p.table, p.n_table, k * p.k_scale);
    case HERMES_RADIAL_SPHERE: return isotropic_f64(HERMES_WIN_SPHERE, k, p.a0, p.a1);
    case HERMES_RADIAL_GAUSSIAN: return isotropic_f64(HERMES_WIN_GAUSSIAN, k, p.a0, p.a1);
    case HERMES_RADIAL_THICK_SHELL: return isotropic_f64(HERMES_WIN_THICK_SHELL, k, p.a0, p.a1);
    case HERMES_RADIAL_GAUSSIAN_SHELL: return isotropic_f64(HERMES_WIN_GAUSSIAN_SHELL, k, p.a0, p.a1);
    }
    return __builtin_nan("");
}

// Transfer function of a real window at signed k: the isotropic and line-of-sight ones and the m = 0 multipoles.
// general = false compiles out the non-axis line-of-sight branch (for callers that never see axis-3 descriptors).
template <bool LOS = true>
__device__ inline double real_window_f64(const hermes_window_desc& d, double ki, double kj, double kk,
                                         bool general = true) {
    if (d.type == HERMES_WIN_SHELL_MULTIPOLE) {
        const double k = sqrt(ki * ki + kj * kj + kk * kk);
        if (k == 0.0) return d.l == 0 ? sqrt(0.25 / HERMES_PI) : 0.0;
        return jl_f64(d.l, k * d.a0) * yl0_f64(d.l, kk / k);
    }
    return iso_window_f64<LOS>(d.type, ki, kj, kk, d.a0, d.a1, d.axis, general ? d.los : nullptr);
}

// ------------------------------------------------------------------ FP32 fast path
// j_l(2 pi t), FP32 fast path, from the exact revolution count t (FP64):
// l = 0 closed form; q >= l + 1 upward recurrence from j0, j1 (stable there,
// the same split as the reference); otherwise the power series
// j_l(q) = q^l/(2l+1)!! sum_k (-q^2/2)^k / (k! prod_{i=1..k}(2l+2i+1)).
__device__ inline float jl_f32(int l, double t) {
    if (t == 0.0) return l == 0 ? 1.0f : 0.0f;
    float q = (float)(2.0 * HERMES_PI * t);
    if (l == 0 || q >= (float)l + 1.0f) {
        // the argument is t turns: reduce in FP64, then the hardware sin/cos, which take turns
        // (sin(2 pi x); measured max abs error 1.1e-7 over a turn)
        const float fr = (float)(t - floor(t));
        const float s = __builtin_amdgcn_sinf(fr), c = __builtin_amdgcn_cosf(fr);
        const float iq = __builtin_amdgcn_rcpf(q);
        float j0 = s * iq;
        if (l == 0) return j0;
        float j1 = (j0 - c) * iq;
        float jm = j0, jc = j1;
        for (int n = 1; n < l; ++n) {
            float jn = (float)(2 * n + 1) * iq * jc - jm;
            jm = jc;
            jc = jn;
        }
        return jc;
    }
    float h = -0.5f * q * q;
    float ql = 1.0f, dfact = 1.0f;
    for (int n = 1; n <= l; ++n) {
        ql *= q;
        dfact *= (float)(2 * n + 1);
    }
    float term = 1.0f, sum = 1.0f;
    for (int k = 1; k < 80; ++k) {
        term *= h * __builtin_amdgcn_rcpf((float)(k * (2 * l + 2 * k + 1)));
        sum += term;
        if (fabsf(term) < 1e-9f * fabsf(sum)) break;
    }
    return ql / dfact * sum;
}

// j_l and j_{l+1} of 2 pi t together: the upward recurrence of jl_f32 run one step further where
// it serves both (q >= l + 2), otherwise each from jl_f32; the same values as two jl_f32 calls.
__device__ inline void jl_pair_f32(int l, double t, float& jl, float& jl1) {
    const float q = (float)(2.0 * HERMES_PI * t);
    if (t != 0.0 && q >= (float)l + 2.0f) {
        const float fr = (float)(t - floor(t));
        const float s = __builtin_amdgcn_sinf(fr), c = __builtin_amdgcn_cosf(fr);
        const float iq = __builtin_amdgcn_rcpf(q);
        float jm = s * iq;
        float jc = (jm - c) * iq;
        if (l == 0) {
            jl = jm;
            jl1 = jc;
            return;
        }
        for (int n = 1; n < l; ++n) {
            float jn = (float)(2 * n + 1) * iq * jc - jm;
            jm = jc;
            jc = jn;
        }
        jl = jc;
        jl1 = (float)(2 * l + 1) * iq * jc - jm;
        return;
    }
    jl = jl_f32(l, t);
    jl1 = jl_f32(l + 1, t);
}

// Y_l^m(a-hat) for integer lattice vector a (as floats), m >= 0; cnorm = N_lm (-1)^m (2m-1)!!.
__device__ inline float2 ylm_f32(int l, int m, float ax, float ay, float az, float cnorm) {
    float r2 = ax * ax + ay * ay + az * az;
    if (r2 == 0.0f) return make_float2((l == 0 && m == 0) ? 0.28209479177387814f : 0.0f, 0.0f);
    float ir = rsqrtf(r2);
    float x = az * ir;
    float ur = ax * ir, ui = ay * ir;  // sin(theta) e^{i phi}
    float pr = 1.0f, pi = 0.0f;
    for (int i = 0; i < m; ++i) {
        float t = pr * ur - pi * ui;
        pi = pr * ui + pi * ur;
        pr = t;
    }
    // polynomial part of P_l^m(x) / ((-1)^m (2m-1)!! (1-x^2)^{m/2})
    float pmm = 1.0f, poly;
    if (l == m) {
        poly = pmm;
    } else {
        float a = pmm, b = x * (float)(2 * m + 1);
        for (int ell = m + 2; ell <= l; ++ell) {
            float c = ((float)(2 * ell - 1) * x * b - (float)(ell + m - 1) * a) / (float)(ell - m);
            a = b;
            b = c;
        }
        poly = b;
    }
    float s = cnorm * poly;
    return make_float2(s * pr, s * pi);
}
