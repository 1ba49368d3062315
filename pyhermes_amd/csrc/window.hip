// Window stage: kernel builders, spectral multiply, fused pair reduction and the
// fused multipole window apply of the batched SH-3PCF path.
// P (|phi_hat|^2 samples, L+1 doubles) is a DEVICE pointer; window descriptors
// and shell radii are HOST arrays copied to the context workspace.
#include "../../include/hermes_amd.h"
#include "fft_lds.h"
#include "hermes_common.h"
#include "pair_los.h"
#include "pair_radial.h"
#include "reduce.h"
#include "special.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>

namespace {

constexpr int RED_THREADS = 256;

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ---------------------------------------------------------------- kernel builders
// Every built-in window has a definite symmetry under the reversal of a k component, and the alias sum of an
// octant position (x, y, z) in [0, L/2]^3 keeps it: the kernel at a mirrored position (L - x for x, ...) is
//   x: (-1)^m conj K,   y: conj K,   z: (-1)^(l+m) K      (real windows: l = m = 0),
// so one evaluation serves up to 8 positions.  (A zero component is its own mirror; its aliases are 0 and -L.)
// Only a line of sight off the axes lacks the symmetry: k_build_rfft_general and k_build_full_general.
// Window sums are FP64 VALU work: for a thin-shell multipole about 8 (sin, cos, recurrences) per position, the
// store of 8 positions otherwise.  One evaluation per position and Y_lm through acos, atan2, cos and sin took
// 7.50 ms (l <= 2, FP64, L = 256) before the product with the spectrum (0.14 ms); this takes 0.12 ms with it.

// Aliases of an octant position in the fold's order, (0,0,0) (1,0,0) (0,1,0) (0,0,1) (1,1,0) (1,0,1) (0,1,1)
// (1,1,1) of convolution.py:263-281; bit 2: x, bit 1: y, bit 0: z.
__device__ constexpr int FOLD_ORDER[8] = {0, 4, 2, 1, 6, 5, 3, 7};

// convolution.py:14-38 + :263-281: K[x,y,z] = sum over the 8 mirrors {x, L-x} x ... of
// P[i]P[j]P[k] W(i/L, j/L, k/L), for windows even in every component.
// LOS false compiles the line-of-sight windows out: their Bessel series double the registers.
template <typename T, bool LOS>
__global__ __launch_bounds__(256, 2) void k_build_rfft(int L, const double* __restrict__ P, hermes_window_desc d,
                                                    T* __restrict__ out) {
    const int Lh = L / 2 + 1;
    const int64_t n = (int64_t)Lh * Lh * Lh;
    const double inv_L = 1.0 / L;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(i % Lh), y = (int)((i / Lh) % Lh), x = (int)(i / ((int64_t)Lh * Lh));
        double t = 0.0;
        for (int a = 0; a < 8; ++a) {
            const int o = FOLD_ORDER[a];
            const int ii = (o & 4) ? L - x : x, jj = (o & 2) ? L - y : y, kk = (o & 1) ? L - z : z;
            t += P[ii] * P[jj] * P[kk] *
                 iso_window_f64<LOS>(d.type, ii * inv_L, jj * inv_L, kk * inv_L, d.a0, d.a1, d.axis, nullptr);
        }
        if (d.type == HERMES_WIN_INVERSE_LAPLACIAN && i == 0) t = 0.0;
        const int xm = (L - x) & (L - 1), ym = (L - y) & (L - 1);
        out[((int64_t)x * L + y) * Lh + z] = (T)t;
        if (xm != x) out[((int64_t)xm * L + y) * Lh + z] = (T)t;
        if (ym != y) out[((int64_t)x * L + ym) * Lh + z] = (T)t;
        if (xm != x && ym != y) out[((int64_t)xm * L + ym) * Lh + z] = (T)t;
    }
}

// The same for a line of sight off the axes (descriptor axis 3), even only under k -> -k: every position sums its
// signed aliases (the mirror alias L - x sits at k = -(L - x) / L).
template <typename T>
__global__ __launch_bounds__(256, 2) void k_build_rfft_general(int L, const double* __restrict__ P,
                                                               hermes_window_desc d, T* __restrict__ out) {
    const int Lh = L / 2 + 1;
    const int64_t n = (int64_t)L * L * Lh;
    const double inv_L = 1.0 / L;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(i % Lh), y = (int)((i / Lh) % L), x = (int)(i / ((int64_t)Lh * L));
        double t = 0.0;
        for (int a = 0; a < 8; ++a) {
            const int o = FOLD_ORDER[a];
            const int ii = (o & 4) ? x - L : x, jj = (o & 2) ? y - L : y, kk = (o & 1) ? z - L : z;
            t += P[ii < 0 ? -ii : ii] * P[jj < 0 ? -jj : jj] * P[kk < 0 ? -kk : kk] *
                 iso_window_f64(d.type, ii * inv_L, jj * inv_L, kk * inv_L, d.a0, d.a1, d.axis, d.los);
        }
        out[i] = (T)t;
    }
}

// Full-grid complex kernels in the alias order of radial_multipole_windows.py:147-183 ((x-L | x) per axis, "0"
// first), one octant position per thread.  KIND 0: a real window of desc (isotropic, line of sight along an
// axis); 1: j_l(2 pi |k| R) Y_lm with R = prof.a0; 2: U_l(|k|) Y_lm of a radial profile
// (radial_multipole_windows.py:186-264).  APPLY: writes spec * K * scale instead of K (FP64; the product of
// convolution.py:291-295 without storing K).
template <typename T, int KIND, bool APPLY>
__global__ __launch_bounds__(256, 2) void k_build_full(int L, const double* __restrict__ P, hermes_window_desc d,
                                                    hermes_radial_profile prof, YlmTable Y, double scale,
                                                    const double2* __restrict__ spec, T* __restrict__ out) {
    const int Lh = L / 2 + 1;
    const int64_t n = (int64_t)Lh * Lh * Lh;
    const double inv_L = 1.0 / L;
    const int am = Y.m < 0 ? -Y.m : Y.m;
    const double sx = KIND && (am & 1) ? -1.0 : 1.0, sz = KIND && ((Y.l + am) & 1) ? -1.0 : 1.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(i % Lh), y = (int)((i / Lh) % Lh), x = (int)(i / ((int64_t)Lh * Lh));
        double re = 0.0, im = 0.0;
        for (int a = 0; a < 8; ++a) {
            const int ax = (a & 4) ? x : x - L, ay = (a & 2) ? y : y - L, az = (a & 1) ? z : z - L;
            const double p = P[ax < 0 ? -ax : ax] * P[ay < 0 ? -ay : ay] * P[az < 0 ? -az : az];
            const double kx = ax * inv_L, ky = ay * inv_L, kz = az * inv_L;
            if (KIND == 0) {
                re += p * iso_window_f64(d.type, kx, ky, kz, d.a0, d.a1, d.axis, nullptr);
            } else {
                const double k = sqrt(kx * kx + ky * ky + kz * kz);
                const double rad = p * (KIND == 1 ? jl_f64(Y.l, k * prof.a0) : radial_profile_f64(prof, Y.l, k));
                const double2 yv = ylm_f64(Y, kx, ky, kz, k == 0.0 ? 0.0 : 1.0 / k);
                re += rad * yv.x;
                im += rad * yv.y;
            }
        }
        if (KIND == 0 && d.type == HERMES_WIN_INVERSE_LAPLACIAN && i == 0) re = 0.0;
        if (APPLY) {
            re *= scale;
            im *= scale;
        }
#pragma unroll
        for (int mode = 0; mode < 8; ++mode) {
            const bool fx = mode & 4, fy = mode & 2, fz = mode & 1;
            const int xx = fx ? (L - x) & (L - 1) : x, yy = fy ? (L - y) & (L - 1) : y,
                      zz = fz ? (L - z) & (L - 1) : z;
            if ((fx && xx == x) || (fy && yy == y) || (fz && zz == z)) continue;
            const double sg = (fx ? sx : 1.0) * (fz ? sz : 1.0);
            double kr = sg * re, ki = (fx != fy) ? -sg * im : sg * im;
            const int64_t o = ((int64_t)xx * L + yy) * L + zz;
            if (APPLY) {
                const double2 f = spec[o];
                const double t = f.x * kr - f.y * ki;
                ki = f.x * ki + f.y * kr;
                kr = t;
            }
            if constexpr (sizeof(T) == 8) *(double2*)(out + 2 * o) = make_double2(kr, ki);
            else *(float2*)(out + 2 * o) = make_float2((float)kr, (float)ki);
        }
    }
}

// A real window along a line of sight off the axes (descriptor axis 3), position by position.
template <typename T>
__global__ __launch_bounds__(256, 2) void k_build_full_general(int L, const double* __restrict__ P,
                                                               hermes_window_desc d, T* __restrict__ out) {
    const int64_t n = (int64_t)L * L * L;
    const double inv_L = 1.0 / L;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(i % L), y = (int)((i / L) % L), x = (int)(i / ((int64_t)L * L));
        double re = 0.0;
        for (int a = 0; a < 8; ++a) {
            const int ax = (a & 4) ? x : x - L, ay = (a & 2) ? y : y - L, az = (a & 1) ? z : z - L;
            re += P[ax < 0 ? -ax : ax] * P[ay < 0 ? -ay : ay] * P[az < 0 ? -az : az] *
                  iso_window_f64(d.type, ax * inv_L, ay * inv_L, az * inv_L, d.a0, d.a1, d.axis, d.los);
        }
        out[2 * i] = (T)re;
        out[2 * i + 1] = (T)0;
    }
}

template <typename T>
__global__ void k_spec_mul(int64_t n, T* __restrict__ spec, const T* __restrict__ ker, int kc, T scale) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        T a = spec[2 * i], b = spec[2 * i + 1];
        if (kc) {
            T c = ker[2 * i] * scale, e = ker[2 * i + 1] * scale;
            spec[2 * i] = a * c - b * e;
            spec[2 * i + 1] = a * e + b * c;
        } else {
            T c = ker[i] * scale;
            spec[2 * i] = a * c;
            spec[2 * i + 1] = b * c;
        }
    }
}

// ---------------------------------------------------------------- pair reduction
// Window value at signed lattice alias (ax, ay, az), FP32 fast path for shells and
// shell multipoles; other window types use the FP64 formula.
template <bool LOS>
__device__ __forceinline__ float window_value_f32(const hermes_window_desc& d, int ax, int ay, int az, int L,
                                                  float cnorm) {
    double n2 = (double)ax * ax + (double)ay * ay + (double)az * az;
    if (d.type == HERMES_WIN_SHELL) {
        double t = sqrt(n2) * d.a0 / L;
        return jl_f32(0, t);
    }
    if (d.type == HERMES_WIN_SHELL_MULTIPOLE) {
        double t = sqrt(n2) * d.a0 / L;
        float j = jl_f32(d.l, t);
        float2 y = ylm_f32(d.l, d.m, (float)ax, (float)ay, (float)az, cnorm);
        return j * y.x;  // m = 0 windows are real
    }
    double inv_L = 1.0 / L;
    // reached only by passes without non-axis line-of-sight windows
    return (float)iso_window_f64<LOS>(d.type, ax * inv_L, ay * inv_L, az * inv_L, d.a0, d.a1, d.axis, nullptr);
}

// One thread per octant representative (x, y, z) in [0, L/2]^3; its kernel value is
// shared by the (up to) 4 modes (x|L-x, y|L-y, z) of the half spectrum.  GEN: the pass holds a
// line-of-sight window along a non-axis direction (descriptor axis 3), whose value differs between the 4
// modes.  LOS: it holds a line-of-sight window at all.  Both are separate instantiations, so that the other passes
// keep their register budget (124 registers and four waves per SIMD without, 150 to 162 and three with them; FP32
// spectra, 20 shells and a sphere at L = 512: 7.1 ms, 16.4 with the Bessel series inlined and 290 registers; 20 shells
// and a disk: 8.5, 17.3).
template <typename C, bool FP64, bool GEN, bool LOS>
__global__ __launch_bounds__(RED_THREADS) void k_pair_reduce(int L, const C* __restrict__ F1,
                                                             const C* __restrict__ F2, const double* __restrict__ P,
                                                             const hermes_window_desc* __restrict__ descs,
                                                             const float* __restrict__ cnorms, int nd,
                                                             double* __restrict__ partial) {
    extern __shared__ double wacc[];  // [waves][nd]
    const int Lh = L / 2 + 1;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int nwaves = blockDim.x / 64;
    for (int i = threadIdx.x; i < nwaves * nd; i += blockDim.x) wacc[i] = 0.0;
    __syncthreads();
    const int64_t nrep = (int64_t)Lh * Lh * Lh;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t base = blockIdx.x * (int64_t)blockDim.x; base < nrep; base += stride) {
        int64_t r = base + threadIdx.x;
        bool active = r < nrep;
        double power = 0.0;
        double pw00 = 0.0, pw01 = 0.0, pw10 = 0.0, pw11 = 0.0;  // per mirror mode (x | L-x, y | L-y)
        int x = 0, y = 0, z = 0;
        if (active) {
            z = (int)(r % Lh);
            y = (int)((r / Lh) % Lh);
            x = (int)(r / ((int64_t)Lh * Lh));
            const int xm = (L - x) % L, ym = (L - y) % L;
            const int nxm = (xm != x) ? 2 : 1, nym = (ym != y) ? 2 : 1;
            const double wz = (z == 0 || z == L / 2) ? 1.0 : 2.0;
            for (int a = 0; a < nxm; ++a)
                for (int b = 0; b < nym; ++b) {
                    int xx = a ? xm : x, yy = b ? ym : y;
                    int64_t idx = ((int64_t)xx * L + yy) * Lh + z;
                    C f1 = F1[idx], f2 = F2[idx];
                    const double pab = wz * ((double)f1.x * (double)f2.x + (double)f1.y * (double)f2.y);
                    if (a == 0 && b == 0) pw00 = pab;
                    else if (a == 0) pw01 = pab;
                    else if (b == 0) pw10 = pab;
                    else pw11 = pab;
                    power += pab;
                }
        }
        for (int b = 0; b < nd; ++b) {
            double kb = 0.0;
            if (active) {
                const hermes_window_desc d = descs[b];
                // a window along a non-axis line of sight differs between the mirror modes: the aliases of
                // (L - x, y, z) are those of (x, y, z) with k_x negated, so each mode takes its own sum
                if (GEN && d.type >= HERMES_WIN_RING && d.axis == 3) {
                    const double inv_L = 1.0 / L;
                    for (int m = 0; m < 4; ++m) {
                        const double sx = (m & 2) ? -1.0 : 1.0, sy = (m & 1) ? -1.0 : 1.0;
                        const double pm = m == 0 ? pw00 : (m == 1 ? pw01 : (m == 2 ? pw10 : pw11));
                        if (pm == 0.0) continue;  // a mode that is its own mirror, or a zero product
                        double km = 0.0;
                        for (int a = 0; a < 8; ++a) {
                            int ax = (a & 4) ? x - L : x, ay = (a & 2) ? y - L : y, az = (a & 1) ? z - L : z;
                            int ix = ax < 0 ? -ax : ax, iy = ay < 0 ? -ay : ay, iz = az < 0 ? -az : az;
                            double p = P[ix] * P[iy] * P[iz];
                            const double w = real_window_f64<LOS>(d, sx * ax * inv_L, sy * ay * inv_L, az * inv_L);
                            km += FP64 ? p * w : (double)((float)p * (float)w);
                        }
                        kb += pm * km;
                    }
                } else {
                    for (int a = 0; a < 8; ++a) {
                        int ax = (a & 4) ? x - L : x, ay = (a & 2) ? y - L : y, az = (a & 1) ? z - L : z;
                        int ix = ax < 0 ? -ax : ax, iy = ay < 0 ? -ay : ay, iz = az < 0 ? -az : az;
                        double p = P[ix] * P[iy] * P[iz];
                        if (FP64) {
                            double inv_L = 1.0 / L;
                            kb += p * real_window_f64<LOS>(d, ax * inv_L, ay * inv_L, az * inv_L, GEN);
                        } else {
                            kb += (double)((float)p * window_value_f32<LOS>(d, ax, ay, az, L, cnorms[b]));
                        }
                    }
                    kb *= power;
                }
                if (d.type == HERMES_WIN_INVERSE_LAPLACIAN && x == 0 && y == 0 && z == 0) kb = 0.0;
            }
            double v = wave_sum(kb);
            if (lane == 0) wacc[wave * nd + b] += v;
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nd; b += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < nwaves; ++w) s += wacc[w * nd + b];
        partial[(int64_t)blockIdx.x * nd + b] = s;
    }
}

// out[d] = factor[d] * sums[ch_of[d]].
__global__ void k_plan_out(const double* __restrict__ sums, const int* __restrict__ ch_of,
                           const double* __restrict__ factor, int n_desc, double* __restrict__ out) {
    for (int d = blockIdx.x * blockDim.x + threadIdx.x; d < n_desc; d += gridDim.x * blockDim.x)
        out[d] = factor[d] * sums[ch_of[d]];
}

// ---------------------------------------------------------------- multipole apply (FP32)
constexpr int MAX_SHELLS = 64;
constexpr int SHELL_CHUNK = 16;

struct ApplyArgs {
    int L, l, m, n_shell;
    int group;  // shells per workgroup of the fused window kernel
    float cnorm, scale;
    float sx, sy, sz;  // sign factors for x-, y- (1) and z-mirrors: (-1)^m, (-1)^(l+m)
    double radii_over_L[MAX_SHELLS];
};

// Several orders m of one l (the fused window + z-FFT kernel shares the radial factors among them).
constexpr int MAX_MP = 2;
struct MultiM {
    int n;                  // 1..MAX_MP
    int l[MAX_MP];          // degree of each order (one l, or l and l + 1 for the packed m = 0 pair)
    int m[MAX_MP];
    float cnorm[MAX_MP];    // N_l|m| (-1)^|m| (2|m|-1)!!
    float sx[MAX_MP], sz[MAX_MP];
};

__device__ __forceinline__ float2 cmulf(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ float2 conjf2(float2 a) { return make_float2(a.x, -a.y); }

__global__ __launch_bounds__(256) void k_multipole_apply(const float2* __restrict__ H, const double* __restrict__ P,
                                                         ApplyArgs A, float2* __restrict__ out) {
    const int L = A.L, Lh = L / 2 + 1;
    const int64_t nrep = (int64_t)Lh * Lh * Lh;
    const int64_t N = (int64_t)L * L * L;
    for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < nrep; r += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(r % Lh), y = (int)((r / Lh) % Lh), x = (int)(r / ((int64_t)Lh * Lh));
        const int xm = (L - x) % L, ym = (L - y) % L, zm = (L - z) % L;
        // spectrum values at the 8 mirror modes from 4 half-spectrum reads
        const float2 h00 = H[((int64_t)x * L + y) * Lh + z], h10 = H[((int64_t)xm * L + y) * Lh + z];
        const float2 h01 = H[((int64_t)x * L + ym) * Lh + z], h11 = H[((int64_t)xm * L + ym) * Lh + z];
        // alias geometry
        float pw[8];
        float2 yv[8];
        double nrm[8];
#pragma unroll
        for (int a = 0; a < 8; ++a) {
            int ax = (a & 4) ? x - L : x, ay = (a & 2) ? y - L : y, az = (a & 1) ? z - L : z;
            pw[a] = (float)P[ax < 0 ? -ax : ax] * (float)P[ay < 0 ? -ay : ay] * (float)P[az < 0 ? -az : az];
            nrm[a] = sqrt((double)ax * ax + (double)ay * ay + (double)az * az);
            float2 yy = ylm_f32(A.l, A.m < 0 ? -A.m : A.m, (float)ax, (float)ay, (float)az, A.cnorm);
            if (A.m < 0) {  // Y_{l,-m} = (-1)^m conj(Y_{l,m})
                float sg = ((-A.m) & 1) ? -1.0f : 1.0f;
                yy = make_float2(sg * yy.x, -sg * yy.y);
            }
            yv[a] = yy;
        }
        for (int s0 = 0; s0 < A.n_shell; s0 += SHELL_CHUNK) {
            float2 K[SHELL_CHUNK];
#pragma unroll
            for (int s = 0; s < SHELL_CHUNK; ++s) K[s] = make_float2(0.0f, 0.0f);
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                if (pw[a] == 0.0f) continue;
#pragma unroll
                for (int s = 0; s < SHELL_CHUNK; ++s) {
                    if (s0 + s < A.n_shell) {
                        float j = jl_f32(A.l, nrm[a] * A.radii_over_L[s0 + s]) * pw[a];
                        K[s].x += j * yv[a].x;
                        K[s].y += j * yv[a].y;
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < SHELL_CHUNK; ++s) {
                if (s0 + s >= A.n_shell) break;
                float2* o = out + (int64_t)(s0 + s) * N;
                const float2 k = make_float2(K[s].x * A.scale, K[s].y * A.scale);
                const float2 kc = conjf2(k);
                // x-mirror: (-1)^m conj K; y-mirror: conj K; z-mirror: (-1)^(l+m) K
                o[((int64_t)x * L + y) * L + z] = cmulf(h00, k);
                if (xm != x) o[((int64_t)xm * L + y) * L + z] = cmulf(h10, make_float2(A.sx * kc.x, A.sx * kc.y));
                if (ym != y) o[((int64_t)x * L + ym) * L + z] = cmulf(h01, kc);
                if (xm != x && ym != y) o[((int64_t)xm * L + ym) * L + z] = cmulf(h11, make_float2(A.sx * k.x, A.sx * k.y));
                if (zm != z) {
                    const float szf = A.sz;
                    o[((int64_t)x * L + y) * L + zm] = cmulf(conjf2(h11), make_float2(szf * k.x, szf * k.y));
                    if (xm != x)
                        o[((int64_t)xm * L + y) * L + zm] =
                            cmulf(conjf2(h01), make_float2(szf * A.sx * kc.x, szf * A.sx * kc.y));
                    if (ym != y) o[((int64_t)x * L + ym) * L + zm] = cmulf(conjf2(h10), make_float2(szf * kc.x, szf * kc.y));
                    if (xm != x && ym != y)
                        o[((int64_t)xm * L + ym) * L + zm] =
                            cmulf(conjf2(h00), make_float2(szf * A.sx * k.x, szf * A.sx * k.y));
                }
            }
        }
    }
}

// Fused multipole window and inverse z-FFT (FP32).  Workgroup (x, y), 0 <= x, y <= L/2, evaluates
// K_{R_s,l,m} at its octant representatives (x, y, z <= L/2) exactly as k_multipole_apply does, forms
// the four mirror lines (x, y), (xm, y), (x, ym), (xm, ym) of H_full * K * scale in LDS with the same
// mirror rules, transforms them along z and writes each distinct line once.  Loops over the shells of its group:
// blockIdx.y splits them on small grids, where one workgroup per (x, y) leaves the SIMDs with a wave or less
// (mpwin_groups; each group evaluates the alias weights again).

// MP orders m of one l per launch: the radial factors j_l(2 pi |a| R_s) of the 8 aliases are
// evaluated once per (representative, shell) and shared by the MP windows; the weights
// P(a) Y_lm(a-hat) are kept per order (premultiplied).  The LDS z-FFT runs over 4 MP lines
// (line mi * 4 + row) and order mi's shell s lands at out + (mi * n_shell + s) * L^3.
template <int LOG2L>
constexpr int mpwin_threads() {
    // one z representative 0 .. L/2 - 1 per thread (at least a wave); for L >= 128 the Nyquist
    // plane z = L/2 is left over and its eight alias terms are computed by eight helper lanes
    return 64 * (((1 << LOG2L) / 2 + 63) / 64);
}

// PACK (MP = 2): the orders are (l, 0) and (l + 1, 0), whose windows are real with opposite parity
// under k -> -k, so the field of the even degree is real and that of the odd one imaginary: their
// windows are summed into one set of four lines (one field per shell, half the transforms), and the
// real and imaginary products of the Gram separate them again.
// PROF: the radial factor of shell s comes from the radial profile prof[s] (thin shell, table or closed-form
// monopole) instead of j_l(2 pi |a| R_s / L); prof is unused otherwise.
template <int LOG2L, int MP, bool PACK = false, bool PROF = false>
__global__ __launch_bounds__(mpwin_threads<LOG2L>()) void k_mpwin_zfft_multi(
    const float2* __restrict__ H, const double* __restrict__ P, ApplyArgs A, MultiM M,
    const float2* __restrict__ twg, float2* __restrict__ out, const hermes_radial_profile* __restrict__ prof) {
    static_assert(!PACK || MP == 2, "packing needs two orders");
    static_assert(!(PACK && PROF), "packed pairs take thin shells only");
    constexpr int L = 1 << LOG2L, Lh = L / 2 + 1;
    constexpr int NT = mpwin_threads<LOG2L>();
    constexpr bool NYQ = Lh > NT;  // z = L/2 by helper lanes 0..7
    constexpr int NLINE = PACK ? 4 : 4 * MP;  // lines transformed per shell
    using F = hermes_fft::LdsFft<LOG2L, NLINE, NT, 1, false>;
    __shared__ float2 lds[F::ELEMS];
    __shared__ float2 tw[L];
    __shared__ float2 nyq[8][MP];
    const int tid = threadIdx.x;
    const int x = blockIdx.x / Lh, y = blockIdx.x % Lh;
    const int xm = (L - x) & (L - 1), ym = (L - y) & (L - 1);
    const int64_t N = (int64_t)L * L * L;
    hermes_fft::load_twiddles<LOG2L>(tw, twg, tid, NT);
    // weights P(a) Y_lm(a-hat) of the 8 aliases per order (premultiplied) for this thread's z and, on the
    // helper lanes, alias tid of the Nyquist plane
    auto weights = [&](int z, int a, float2* w, double& nrm, bool& live) {
        const int ax = (a & 4) ? x - L : x, ay = (a & 2) ? y - L : y, az = (a & 1) ? z - L : z;
        const float pw = (float)P[ax < 0 ? -ax : ax] * (float)P[ay < 0 ? -ay : ay] * (float)P[az < 0 ? -az : az];
        live = pw != 0.0f;
        nrm = sqrt((double)ax * ax + (double)ay * ay + (double)az * az);
#pragma unroll
        for (int mi = 0; mi < MP; ++mi) {
            const int m = M.m[mi], am = m < 0 ? -m : m;
            float2 yy = ylm_f32(M.l[mi], am, (float)ax, (float)ay, (float)az, M.cnorm[mi]);
            if (m < 0) {  // Y_{l,-m} = (-1)^m conj(Y_{l,m})
                const float sg = (am & 1) ? -1.0f : 1.0f;
                yy = make_float2(sg * yy.x, -sg * yy.y);
            }
            w[mi] = make_float2(pw * yy.x, pw * yy.y);
        }
    };
    const int z = tid;
    const bool zact = z < Lh;
    float2 wy[8][MP];
    double nrm[8];
    float2 h[4];
    unsigned live = 0;
    if (zact) {
        h[0] = H[((int64_t)x * L + y) * Lh + z];
        h[1] = H[((int64_t)xm * L + y) * Lh + z];
        h[2] = H[((int64_t)x * L + ym) * Lh + z];
        h[3] = H[((int64_t)xm * L + ym) * Lh + z];
#pragma unroll
        for (int a = 0; a < 8; ++a) {
            bool lv;
            weights(z, a, wy[a], nrm[a], lv);
            if (lv) live |= 1u << a;
        }
    }
    float2 wn[MP], hn[4];
    double nrm_n = 0.0;
    bool live_n = false;
    if (NYQ && tid < 8) weights(L / 2, tid, wn, nrm_n, live_n);
    if (NYQ && tid < MP) {
        hn[0] = H[((int64_t)x * L + y) * Lh + L / 2];
        hn[1] = H[((int64_t)xm * L + y) * Lh + L / 2];
        hn[2] = H[((int64_t)x * L + ym) * Lh + L / 2];
        hn[3] = H[((int64_t)xm * L + ym) * Lh + L / 2];
    }
    // the four mirror rows of representative z (and, for z != -z, the rows of -z) for order mi
    auto put = [&](int mi, int zz, const float2 hh[4], float2 Km) {
        const float2 k = make_float2(Km.x * A.scale, Km.y * A.scale);
        const float2 kc = conjf2(k);
        const float sx = M.sx[mi], sz = M.sz[mi];
        const int r0 = 4 * mi;
        lds[F::addr(r0 + 0, zz)] = cmulf(hh[0], k);
        lds[F::addr(r0 + 1, zz)] = cmulf(hh[1], make_float2(sx * kc.x, sx * kc.y));
        lds[F::addr(r0 + 2, zz)] = cmulf(hh[2], kc);
        lds[F::addr(r0 + 3, zz)] = cmulf(hh[3], make_float2(sx * k.x, sx * k.y));
        const int zm = (L - zz) & (L - 1);
        if (zm != zz) {
            lds[F::addr(r0 + 0, zm)] = cmulf(conjf2(hh[3]), make_float2(sz * k.x, sz * k.y));
            lds[F::addr(r0 + 1, zm)] = cmulf(conjf2(hh[2]), make_float2(sz * sx * kc.x, sz * sx * kc.y));
            lds[F::addr(r0 + 2, zm)] = cmulf(conjf2(hh[1]), make_float2(sz * kc.x, sz * kc.y));
            lds[F::addr(r0 + 3, zm)] = cmulf(conjf2(hh[0]), make_float2(sz * sx * k.x, sz * sx * k.y));
        }
    };
    // packed pair: the sum of the two orders' mirrored window values on each of the four lines (the
    // products with H distribute over the sum)
    auto put_pack = [&](int zz, const float2 hh[4], float2 K0, float2 K1) {
        const float2 k0 = make_float2(K0.x * A.scale, K0.y * A.scale), kc0 = conjf2(k0);
        const float2 k1 = make_float2(K1.x * A.scale, K1.y * A.scale), kc1 = conjf2(k1);
        const float sx0 = M.sx[0], sz0 = M.sz[0], sx1 = M.sx[1], sz1 = M.sz[1];
        auto mix = [](float a0, float2 u0, float a1, float2 u1) {
            return make_float2(a0 * u0.x + a1 * u1.x, a0 * u0.y + a1 * u1.y);
        };
        lds[F::addr(0, zz)] = cmulf(hh[0], mix(1.0f, k0, 1.0f, k1));
        lds[F::addr(1, zz)] = cmulf(hh[1], mix(sx0, kc0, sx1, kc1));
        lds[F::addr(2, zz)] = cmulf(hh[2], mix(1.0f, kc0, 1.0f, kc1));
        lds[F::addr(3, zz)] = cmulf(hh[3], mix(sx0, k0, sx1, k1));
        const int zm = (L - zz) & (L - 1);
        if (zm != zz) {
            lds[F::addr(0, zm)] = cmulf(conjf2(hh[3]), mix(sz0, k0, sz1, k1));
            lds[F::addr(1, zm)] = cmulf(conjf2(hh[2]), mix(sz0 * sx0, kc0, sz1 * sx1, kc1));
            lds[F::addr(2, zm)] = cmulf(conjf2(hh[1]), mix(sz0, kc0, sz1, kc1));
            lds[F::addr(3, zm)] = cmulf(conjf2(hh[0]), mix(sz0 * sx0, k0, sz1 * sx1, k1));
        }
    };
    // radial factor of an alias of norm nrm (grid points) for each order (one l, or l and l + 1 when packed)
    hermes_radial_profile pr{};
    auto radial = [&](double nrm_a, double rs, float* j) {
        if (PACK) {
            jl_pair_f32(M.l[0], nrm_a * rs, j[0], j[MP - 1]);
        } else {
            float jj;
            if (PROF)
                jj = pr.kind == HERMES_RADIAL_SHELL ? jl_f32(M.l[0], nrm_a * (pr.a0 / L))
                                                    : (float)radial_profile_f64(pr, M.l[0], nrm_a / L);
            else
                jj = jl_f32(M.l[0], nrm_a * rs);
#pragma unroll
            for (int mi = 0; mi < MP; ++mi) j[mi] = jj;
        }
    };
    const int sb = blockIdx.y * A.group, se = min(A.n_shell, sb + A.group);
    for (int s = sb; s < se; ++s) {
        const double rs = A.radii_over_L[s];
        if (PROF) pr = prof[s];
        if (zact) {
            float2 K[MP];
#pragma unroll
            for (int mi = 0; mi < MP; ++mi) K[mi] = make_float2(0.0f, 0.0f);
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                if (!((live >> a) & 1u)) continue;
                float j[MP];
                radial(nrm[a], rs, j);
#pragma unroll
                for (int mi = 0; mi < MP; ++mi) {
                    K[mi].x += j[mi] * wy[a][mi].x;
                    K[mi].y += j[mi] * wy[a][mi].y;
                }
            }
            if (PACK) {
                put_pack(z, h, K[0], K[MP - 1]);
            } else {
#pragma unroll
                for (int mi = 0; mi < MP; ++mi) put(mi, z, h, K[mi]);
            }
        }
        if (NYQ) {
            if (tid < 8) {
                float j[MP];
                if (live_n) {
                    radial(nrm_n, rs, j);
                } else {
#pragma unroll
                    for (int mi = 0; mi < MP; ++mi) j[mi] = 0.0f;
                }
#pragma unroll
                for (int mi = 0; mi < MP; ++mi) nyq[tid][mi] = make_float2(j[mi] * wn[mi].x, j[mi] * wn[mi].y);
            }
            hermes_fft::lds_barrier();
            if (tid < (PACK ? 1 : MP)) {
                float2 K[MP];
#pragma unroll
                for (int mi = 0; mi < MP; ++mi) K[mi] = make_float2(0.0f, 0.0f);
                for (int a = 0; a < 8; ++a) {
#pragma unroll
                    for (int mi = 0; mi < MP; ++mi) {
                        if (!PACK && mi != tid) continue;
                        K[mi].x += nyq[a][mi].x;
                        K[mi].y += nyq[a][mi].y;
                    }
                }
                if (PACK) {
                    put_pack(L / 2, hn, K[0], K[MP - 1]);
                } else {
#pragma unroll
                    for (int mi = 0; mi < MP; ++mi)
                        if (mi == tid) put(mi, L / 2, hn, K[mi]);
                }
            }
        }
        hermes_fft::lds_barrier();
        F::run(lds, tw, tid);
        // lines known at compile time: the skip of a mirror line that coincides with line 0 / 2 and the
        // line's base address are uniform, and a line's LDS reads are all issued before its stores
        constexpr int EPT = (L + NT - 1) / NT;  // elements per thread and line
#pragma unroll
        for (int line = 0; line < NLINE; ++line) {
            const int mi = line >> 2, row = line & 3;
            const bool dx = row & 1, dy = row & 2;
            if ((dx && xm == x) || (dy && ym == y)) continue;
            const int rx = dx ? xm : x, ry = dy ? ym : y;
            float2* __restrict__ o = out + (int64_t)(mi * A.n_shell + s) * N + ((int64_t)rx * L + ry) * L;
            float2 v[EPT];
#pragma unroll
            for (int q = 0; q < EPT; ++q)
                if (L % NT == 0 || tid + q * NT < L) v[q] = lds[F::addr(line, tid + q * NT)];
#pragma unroll
            for (int q = 0; q < EPT; ++q)
                if (L % NT == 0 || tid + q * NT < L) {
                    if (LOG2L >= 8)  // the fields are written once and read by the next pass from HBM
                        hermes_fft::stream_store(o + tid + q * NT, v[q]);
                    else
                        o[tid + q * NT] = v[q];
                }
        }
        hermes_fft::lds_barrier();
    }
}

// ---------------------------------------------------------------- FP64 sums
template <typename T>
__global__ __launch_bounds__(RED_THREADS) void k_reduce_sum(const T* __restrict__ x, int64_t n, int ncomp,
                                                            double* __restrict__ partial) {
    __shared__ double sh[2][RED_THREADS / 64];
    double s0 = 0.0, s1 = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        if (ncomp == 1) {
            s0 += (double)x[i];
        } else {
            s0 += (double)x[2 * i];
            s1 += (double)x[2 * i + 1];
        }
    }
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    if (threadIdx.x % 64 == 0) {
        sh[0][threadIdx.x / 64] = s0;
        sh[1][threadIdx.x / 64] = s1;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double t = 0.0;
        for (int w = 0; w < RED_THREADS / 64; ++w) t += sh[threadIdx.x][w];
        partial[2 * blockIdx.x + threadIdx.x] = t;
    }
}

int check_desc(const hermes_window_desc& d) {
    if (d.type < 0 || d.type > HERMES_WIN_CYLINDER) {
        hermes_set_error("unknown window type %d", d.type);
        return 2;
    }
    if (d.type >= HERMES_WIN_RING && (d.axis < 0 || d.axis > 3)) {
        hermes_set_error("line-of-sight window: axis %d is not 0, 1, 2 or 3", d.axis);
        return 2;
    }
    if (d.type >= HERMES_WIN_RING && d.axis == 3) {
        const double n2 = d.los[0] * d.los[0] + d.los[1] * d.los[1] + d.los[2] * d.los[2];
        if (!(std::fabs(n2 - 1.0) < 1e-12)) {
            hermes_set_error("line-of-sight window: los is not a unit vector (|los|^2 = %g)", n2);
            return 2;
        }
    }
    if (d.type == HERMES_WIN_SHELL_MULTIPOLE && (d.l < 0 || d.l > 40 || d.m > d.l || d.m < -d.l)) {
        hermes_set_error("invalid multipole (l=%d, m=%d)", d.l, d.m);
        return 2;
    }
    return 0;
}

double factorial_d(int n) {
    double o = 1.0;
    for (int i = 2; i <= n; ++i) o *= i;
    return o;
}

}  // namespace

// N_lm (-1)^m (2m-1)!! for the FP32 spherical harmonics (m >= 0).
double hermes_ylm_cnorm(int l, int m) {
    double n = sqrt((2.0 * l + 1.0) / (4.0 * HERMES_PI) * factorial_d(l - m) / factorial_d(l + m));
    double df = 1.0;
    for (int i = 1; i <= m; ++i) df *= (2.0 * i - 1.0);
    return ((m & 1) ? -1.0 : 1.0) * df * n;
}

extern "C" {

int hermes_window_build_rfft(hermes_ctx* ctx, int J, const double* P, const hermes_window_desc* desc, int dbl,
                             void* out) {
    HERMES_REQUIRE(ctx && desc && P && out, "hermes_window_build_rfft: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(desc->type != HERMES_WIN_SHELL_MULTIPOLE, "multipole windows need the full complex layout");
    if (int rc = check_desc(*desc)) return rc;
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int L = 1 << J, Lh = L / 2 + 1;
    if (desc->type >= HERMES_WIN_RING && desc->axis == 3) {
        const unsigned nb = hermes_blocks((int64_t)L * L * Lh, 256, 65536);
        if (dbl) k_build_rfft_general<double><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (double*)out);
        else k_build_rfft_general<float><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (float*)out);
    } else {
        const unsigned nb = hermes_blocks((int64_t)Lh * Lh * Lh, 256, 65536);
        const bool los = desc->type >= HERMES_WIN_RING;
        if (dbl && los) k_build_rfft<double, true><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (double*)out);
        else if (dbl) k_build_rfft<double, false><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (double*)out);
        else if (los) k_build_rfft<float, true><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (float*)out);
        else k_build_rfft<float, false><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (float*)out);
    }
    HERMES_LAUNCH_CHECK();
    return 0;
}

static YlmTable ylm_table(int l, int m) {
    YlmTable Y{};
    const int am = m < 0 ? -m : m;
    Y.l = l;
    Y.m = m;
    Y.norm = hermes_ylm_cnorm(l, am);
    for (int n = am + 2; n <= l; ++n) {
        Y.a[n] = (2.0 * n - 1.0) / (n - am);
        Y.b[n] = (n + am - 1.0) / (n - am);
    }
    return Y;
}

// One launch of k_build_full: kind as its KIND; spec != nullptr applies it (FP64).
static hipError_t launch_build_full(hermes_ctx* ctx, int J, int kind, const double* P, const hermes_window_desc& d,
                                    const hermes_radial_profile& prof, int l, int m, int dbl, double scale,
                                    const double2* spec, void* out) {
    const int L = 1 << J, Lh = L / 2 + 1;
    const unsigned nb = hermes_blocks((int64_t)Lh * Lh * Lh, 256, 65536);
    const YlmTable Y = ylm_table(l, m);
#define HERMES_BUILD(T, KIND, APPLY) \
    k_build_full<T, KIND, APPLY><<<nb, 256, 0, ctx->stream>>>(L, P, d, prof, Y, scale, spec, (T*)out)
    if (spec && kind == 1) HERMES_BUILD(double, 1, true);
    else if (spec) HERMES_BUILD(double, 2, true);
    else if (dbl && kind == 0) HERMES_BUILD(double, 0, false);
    else if (dbl && kind == 1) HERMES_BUILD(double, 1, false);
    else if (dbl) HERMES_BUILD(double, 2, false);
    else if (kind == 0) HERMES_BUILD(float, 0, false);
    else if (kind == 1) HERMES_BUILD(float, 1, false);
    else HERMES_BUILD(float, 2, false);
#undef HERMES_BUILD
    return hipGetLastError();
}

int hermes_window_build_full(hermes_ctx* ctx, int J, const double* P, const hermes_window_desc* desc, int dbl,
                             void* out) {
    HERMES_REQUIRE(ctx && desc && P && out, "hermes_window_build_full: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    if (int rc = check_desc(*desc)) return rc;
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    hermes_radial_profile prof{};
    if (desc->type == HERMES_WIN_SHELL_MULTIPOLE) {
        prof.a0 = desc->a0;
        HERMES_CHECK_HIP(launch_build_full(ctx, J, 1, P, *desc, prof, desc->l, desc->m, dbl, 1.0, nullptr, out));
    } else if (desc->type >= HERMES_WIN_RING && desc->axis == 3) {
        const int L = 1 << J;
        const unsigned nb = hermes_blocks((int64_t)L * L * L, 256, 65536);
        if (dbl) k_build_full_general<double><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (double*)out);
        else k_build_full_general<float><<<nb, 256, 0, ctx->stream>>>(L, P, *desc, (float*)out);
        HERMES_LAUNCH_CHECK();
    } else {
        HERMES_CHECK_HIP(launch_build_full(ctx, J, 0, P, *desc, prof, 0, 0, dbl, 1.0, nullptr, out));
    }
    return 0;
}

static int check_profile(const hermes_radial_profile& p, int l, const char* who) {
    HERMES_REQUIRE(p.kind >= HERMES_RADIAL_SHELL && p.kind <= HERMES_RADIAL_GAUSSIAN_SHELL, "%s: unknown radial kind %d",
                   who, p.kind);
    HERMES_REQUIRE(std::isfinite(p.a0) && std::isfinite(p.a1) && p.a0 >= 0.0, "%s: invalid profile lengths", who);
    HERMES_REQUIRE(p.kind <= HERMES_RADIAL_TABLE || l == 0,
                   "%s: closed-form profile kinds are monopoles (l = 0), got l = %d", who, l);
    if (p.kind == HERMES_RADIAL_TABLE)
        HERMES_REQUIRE(p.table && p.n_table >= 4 && std::isfinite(p.k_scale) && p.k_scale > 0.0,
                       "%s: a table profile needs a device table of >= 4 values and k_scale > 0", who);
    return 0;
}

int hermes_window_build_full_profile(hermes_ctx* ctx, int J, const double* P, const hermes_radial_profile* prof, int l,
                                     int m, int dbl, void* out) {
    HERMES_REQUIRE(ctx && P && prof && out, "hermes_window_build_full_profile: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(l >= 0 && l <= 40 && m >= -l && m <= l, "invalid multipole (l=%d, m=%d)", l, m);
    if (int rc = check_profile(*prof, l, "hermes_window_build_full_profile")) return rc;
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    HERMES_CHECK_HIP(launch_build_full(ctx, J, prof->kind == HERMES_RADIAL_SHELL ? 1 : 2, P, hermes_window_desc{}, *prof,
                                       l, m, dbl, 1.0, nullptr, out));
    return 0;
}

int hermes_window_apply_full_f64(hermes_ctx* ctx, int J, const double* P, const hermes_radial_profile* prof, int l,
                                 int m, double scale, const void* spec, void* out) {
    HERMES_REQUIRE(ctx && P && prof && spec && out && spec != out, "hermes_window_apply_full_f64: invalid argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(l >= 0 && l <= 40 && m >= -l && m <= l, "invalid multipole (l=%d, m=%d)", l, m);
    if (int rc = check_profile(*prof, l, "hermes_window_apply_full_f64")) return rc;
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    HERMES_CHECK_HIP(launch_build_full(ctx, J, prof->kind == HERMES_RADIAL_SHELL ? 1 : 2, P, hermes_window_desc{}, *prof,
                                       l, m, 1, scale, (const double2*)spec, out));
    return 0;
}

int hermes_spectrum_mul(hermes_ctx* ctx, int J, int half, int dbl, void* spec, const void* kernel, int kernel_complex,
                        double scale) {
    HERMES_REQUIRE(ctx && spec && kernel, "hermes_spectrum_mul: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    int L = 1 << J;
    int64_t n = (int64_t)L * L * (half ? (L / 2 + 1) : L);
    if (dbl)
        k_spec_mul<double><<<hermes_blocks(n, 256, 65536), 256, 0, ctx->stream>>>(n, (double*)spec, (const double*)kernel,
                                                                                 kernel_complex, scale);
    else
        k_spec_mul<float><<<hermes_blocks(n, 256, 65536), 256, 0, ctx->stream>>>(n, (float*)spec, (const float*)kernel,
                                                                                kernel_complex, (float)scale);
    HERMES_LAUNCH_CHECK();
    return 0;
}

// Radius-grouped channels of a descriptor list: unique (radius, order) pairs, each descriptor a
// channel times a constant.  False when some descriptor is not a thin shell or an m = 0 multipole
// of even order <= 10 (FP32) or <= 4 (FP64), or the channels do not fit the kernel's LDS.
struct RadialChannels {
    int LM = 0, nu = 0, nch = 0;
    int rot = 0;                 // >= 3 equally spaced radii R0 + u dR: rotated phases
    double R0 = 0.0, dR = 0.0;
    std::vector<double> radii;   // |R| / L per radius (the windows are even in R)
    std::vector<int> chan;       // nu x (LM + 1): channel or -1
    std::vector<int> ch_of;      // per descriptor
    std::vector<double> factor;  // per descriptor
};

static bool radial_channels(int J, int dbl, const hermes_window_desc* descs, int n_desc, RadialChannels& rc) {
    int lmax = 0;
    for (int b = 0; b < n_desc; ++b) {
        const hermes_window_desc& d = descs[b];
        if (d.type == HERMES_WIN_SHELL) continue;
        if (d.type != HERMES_WIN_SHELL_MULTIPOLE || d.m != 0 || d.l > (dbl ? 4 : 10)) return false;
        lmax = d.l > lmax ? d.l : lmax;
    }
    rc.LM = lmax == 0 ? 0 : (lmax <= 4 ? 4 : 10);
    const int L = 1 << J;
    rc.ch_of.resize(n_desc);
    rc.factor.resize(n_desc);
    for (int b = 0; b < n_desc; ++b) {
        const hermes_window_desc& d = descs[b];
        const double R = std::fabs(d.a0) / L;
        size_t u = 0;
        while (u < rc.radii.size() && rc.radii[u] != R) ++u;
        if (u == rc.radii.size()) {
            rc.radii.push_back(R);
            rc.chan.insert(rc.chan.end(), rc.LM + 1, -1);
        }
        const int l = d.type == HERMES_WIN_SHELL ? 0 : d.l;
        int& c = rc.chan[u * (rc.LM + 1) + l];
        if (c < 0) c = rc.nch++;
        rc.ch_of[b] = c;
        rc.factor[b] = d.type == HERMES_WIN_SHELL ? 1.0 : hermes_ylm_cnorm(d.l, 0);
    }
    rc.nu = (int)rc.radii.size();
    if (rc.nu >= 3) {
        const double r0 = rc.radii[0], d = (rc.radii[rc.nu - 1] - r0) / (rc.nu - 1);
        double rmax = 0.0;
        for (double r : rc.radii) rmax = std::max(rmax, r);
        bool uniform = d != 0.0;
        // a linear binning is met to a few ulps; a phase error grows with 2 pi |a| R / L, up to a few thousand
        for (int u = 0; u < rc.nu && uniform; ++u) uniform = std::fabs(rc.radii[u] - (r0 + u * d)) <= 1e-14 * rmax;
        if (uniform) {
            rc.rot = 1;
            rc.R0 = r0;
            rc.dR = d;
        }
    }
    return sizeof(double) * (RED_THREADS / 64) * rc.nch <= 64 * 1024;
}

// Device table of the radii: R / L, then L / R.
static std::vector<double> radius_table(const RadialChannels& ch) {
    std::vector<double> t(2 * (size_t)ch.nu);
    for (int u = 0; u < ch.nu; ++u) {
        t[u] = ch.radii[u];
        t[ch.nu + u] = 1.0 / ch.radii[u];
    }
    return t;
}

static int radial_block_side(int J) { return J >= 8 ? 8 : 4; }

// Rows of partial sums (workgroups) of the radial kernel: a block triple each while there are no more than 2048.
static int radial_rows(int J) {
    const int nb = ((1 << J) / 2 + 1 + radial_block_side(J) - 1) / radial_block_side(J);
    return std::min(2048, hermes_pair::tetra(nb));
}

// Groups of radii, `per` in each.  Without rotated phases every radius costs a sin/cos per alias, a serial chain that
// one wave per block of positions does not hide on small grids: there the radii are split (their channels are disjoint,
// so a row of partial sums serves all groups) until a wave per SIMD is there; from L = 128 on the blocks fill the chip.
// 30 log-spaced shells, FP32 spectra, whole calls: L = 64 106 us with all radii in one group, 53 now.
static int radial_groups(int rows, int waves, int rot, int nu, int step, int* per) {
    const int steps = (nu + step - 1) / step;
    const int groups = rot ? 1 : std::max(1, std::min(steps, 1024 / (rows * waves)));
    *per = (steps + groups - 1) / groups * step;
    return (nu + *per - 1) / *per;
}

static hipError_t launch_radial(hipStream_t st, int J, int dbl, int LM, int rows, const void* F1, const void* F2,
                                const double* P, const double* d_radii, int nu, int rot, double R0, double dR,
                                const int* d_chan, int nch, double* partial) {
    using namespace hermes_pair;
    const int L = 1 << J, bt = radial_block_side(J), nb = (L / 2 + 1 + bt - 1) / bt, nblk = tetra(nb);
    hipError_t e = hipSuccess;
    int per = nu;
    const int groups = radial_groups(rows, bt == 8 ? 4 : 1, rot, nu, radial_step(LM), &per);
    auto go = [&](auto kernel, int threads, auto* f1, auto* f2) {
        const size_t shmem = sizeof(double) * (threads / 64) * nch;
        if (shmem > 32 * 1024)  // beside up to 25 KB of powers
            e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e == hipSuccess)
            kernel<<<dim3(rows, groups), threads, shmem, st>>>(L, f1, f2, P, d_radii, nu, R0, dR, d_chan, nch, nblk,
                                                               per, partial);
    };
#define HERMES_RADIAL(LMV, ROT)                                                                                      \
    do {                                                                                                             \
        if (dbl && bt == 8) go(k_pair_radial<LMV, ROT, 8, double2>, 256, (const double2*)F1, (const double2*)F2);    \
        else if (dbl) go(k_pair_radial<LMV, ROT, 4, double2>, 64, (const double2*)F1, (const double2*)F2);           \
        else if (bt == 8) go(k_pair_radial<LMV, ROT, 8, float2>, 256, (const float2*)F1, (const float2*)F2);         \
        else go(k_pair_radial<LMV, ROT, 4, float2>, 64, (const float2*)F1, (const float2*)F2);                       \
    } while (0)
    if (LM == 0 && rot) HERMES_RADIAL(0, true);
    else if (LM == 0) HERMES_RADIAL(0, false);
    else if (LM == 4 && rot) HERMES_RADIAL(4, true);
    else if (LM == 4) HERMES_RADIAL(4, false);
    else if (rot) HERMES_RADIAL(10, true);
    else HERMES_RADIAL(10, false);
#undef HERMES_RADIAL
    return e != hipSuccess ? e : hipGetLastError();
}

// Pair reductions have at most 2048 rows of partial sums: one launch, no scratch.
static hipError_t sum_columns(hipStream_t st, const double* partial, int rows, int n, double* out) {
    return hermes_reduce::sum_columns(st, partial, n, rows, n, nullptr, out);
}

// Scratch of the pair reduction: the context's grow-only slot, or, for the allocation-free entry point, a
// fixed buffer of fixed_cap bytes (a request beyond it fails with status 2 and a message).
static char* pair_workspace(hermes_ctx* ctx, char* fixed_ws, size_t fixed_cap, size_t need) {
    if (!fixed_ws) return (char*)hermes_workspace(ctx, WS_REDUCE, need);
    if (need > fixed_cap) {
        hermes_set_error("hermes_pair_reduce_noalloc: this reduction needs %zu bytes of scratch, more than the "
                         "fixed %zu (split the windows over several calls)", need, fixed_cap);
        return nullptr;
    }
    return fixed_ws;
}

// Scratch bytes of `rows` rows of n partial sums, their group sums of 64 rows and the result row.  (The group
// sums are not formed; their room is kept so that the fixed scratch accepts and refuses the same requests.)
static size_t pair_partial_bytes(int rows, int n) {
    return sizeof(double) * ((size_t)rows * n + (size_t)((rows + 63) / 64) * n + n);
}

// The radial path of hermes_pair_reduce.  Returns false (rc untouched) when it does not apply;
// true with rc = the status otherwise.
static bool pair_reduce_radial(hermes_ctx* ctx, int J, int dbl, const void* F1, const void* F2, const double* P,
                               const hermes_window_desc* descs, int n_desc, int nblocks, double* out_host,
                               char* fixed_ws, size_t fixed_cap, int& rc) {
    RadialChannels ch;
    if (!radial_channels(J, dbl, descs, n_desc, ch)) return false;
    rc = 0;
    const int nu = ch.nu, nch = ch.nch;
    const size_t off_chan = sizeof(double) * 2 * nu;
    const size_t off_part = (off_chan + sizeof(int) * ch.chan.size() + 7) / 8 * 8;
    const int rows = radial_rows(J);
    // asked for: one double per radius, the channels and the partial sums with their group sums, whose room the second
    // double of a radius takes (nch >= nu); more only on the small grids, far from the fixed scratch's size
    const size_t asked = (sizeof(double) * nu + sizeof(int) * ch.chan.size() + 255) / 256 * 256 +
                         pair_partial_bytes(nblocks, nch);
    const size_t need = std::max(asked, off_part + sizeof(double) * ((size_t)rows + 1) * nch);
    char* ws = pair_workspace(ctx, fixed_ws, fixed_cap, need);
    if (!ws) {
        rc = fixed_ws ? 2 : 1;
        return true;
    }
    double* d_radii = (double*)ws;
    int* d_chan = (int*)(ws + off_chan);
    double* d_out = (double*)(ws + off_part);
    double* partial = d_out + nch;
    auto fail = [&](hipError_t e) {
        hermes_set_error("pair reduction: %s", hipGetErrorString(e));
        rc = 1;
        return true;
    };
    std::vector<char> tables(off_part);  // radii and channels in one copy
    const std::vector<double> rt = radius_table(ch);
    memcpy(tables.data(), rt.data(), off_chan);
    memcpy(tables.data() + off_chan, ch.chan.data(), sizeof(int) * ch.chan.size());
    hipError_t e = hipMemcpyAsync(ws, tables.data(), off_part, hipMemcpyHostToDevice, ctx->stream);
    if (e != hipSuccess) return fail(e);
    if ((e = launch_radial(ctx->stream, J, dbl, ch.LM, rows, F1, F2, P, d_radii, nu, ch.rot, ch.R0, ch.dR, d_chan,
                           nch, partial)) != hipSuccess)
        return fail(e);
    if ((e = sum_columns(ctx->stream, partial, rows, nch, d_out)) != hipSuccess) return fail(e);
    std::vector<double> chs(nch);
    e = hipMemcpyAsync(chs.data(), d_out, sizeof(double) * nch, hipMemcpyDeviceToHost, ctx->stream);
    if (e != hipSuccess) return fail(e);
    if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return fail(e);
    for (int b = 0; b < n_desc; ++b) out_host[b] = ch.factor[b] * chs[ch.ch_of[b]];
    return true;
}

// The separable path of hermes_pair_reduce for line-of-sight windows that share one coordinate axis; false
// (rc untouched) when some window is of another kind or axis.
static bool pair_reduce_los(hermes_ctx* ctx, int J, int dbl, const void* F1, const void* F2, const double* P,
                            const hermes_window_desc* descs, int n_desc, int nblocks, double* out_host, char* fixed_ws,
                            size_t fixed_cap, int& rc) {
    using namespace hermes_pair;
    for (int b = 0; b < n_desc; ++b)
        if (descs[b].type < HERMES_WIN_RING || descs[b].axis > 2 || descs[b].axis != descs[0].axis) return false;
    rc = 0;
    auto fail = [&](hipError_t e) {
        hermes_set_error("pair reduction: %s", hipGetErrorString(e));
        rc = 1;
        return true;
    };
    const int L = 1 << J, Lh = L / 2 + 1, nptile = (Lh * Lh + LOS_ROWS - 1) / LOS_ROWS, ntile = (n_desc + 15) / 16;
    const int ncol = ntile * 16, rows = std::min(nptile, 1024);
    // window tiles split over workgroups (multiples of the 4 waves) until about 1024 of them share the chip; each
    // group forms the powers of its positions again
    int groups = (1024 + rows - 1) / rows;
    groups = std::max(1, std::min(groups, (ntile + 3) / 4));
    const int tpb = ((ntile + groups - 1) / groups + 3) / 4 * 4;
    groups = (ntile + tpb - 1) / tpb;
    const size_t off_tab = (sizeof(hermes_window_desc) * n_desc + 255) / 256 * 256;
    const size_t off_out = off_tab + sizeof(double) * (size_t)los_par_pad(L) * ncol;
    const size_t need = std::max(off_out + sizeof(double) * ((size_t)rows + 1) * n_desc,
                                 sizeof(hermes_window_desc) * n_desc + sizeof(float) * n_desc + 64 +
                                     pair_partial_bytes(nblocks, n_desc));
    char* ws = pair_workspace(ctx, fixed_ws, fixed_cap, need);
    if (!ws) {
        rc = fixed_ws ? 2 : 1;
        return true;
    }
    hermes_window_desc* d_desc = (hermes_window_desc*)ws;
    double* tab = (double*)(ws + off_tab);
    double* d_out = (double*)(ws + off_out);
    double* partial = d_out + n_desc;
    hipError_t e = hipMemcpyAsync(d_desc, descs, sizeof(hermes_window_desc) * n_desc, hipMemcpyHostToDevice, ctx->stream);
    if (e != hipSuccess) return fail(e);
    const unsigned tab_blocks = hermes_blocks((int64_t)los_par_pad(L) * ncol, 256, 4096);
    k_los_par_table<<<tab_blocks, 256, 0, ctx->stream>>>(L, P, d_desc, n_desc, ncol, tab);
    if ((e = hipGetLastError()) != hipSuccess) return fail(e);
    const size_t shmem = sizeof(double) * ((size_t)los_par_pad(L) * LOS_PITCH + (size_t)tpb * 16);
    auto go = [&](auto kernel, auto* f1, auto* f2) {
        if (shmem > 48 * 1024)
            e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return;
        kernel<<<dim3(rows, groups), LOS_THREADS, shmem, ctx->stream>>>(L, descs[0].axis, f1, f2, P, d_desc, n_desc, tab,
                                                                        ncol, tpb, nptile, partial);
        e = hipGetLastError();
    };
    if (dbl) go(k_pair_los<double2>, (const double2*)F1, (const double2*)F2);
    else go(k_pair_los<float2>, (const float2*)F1, (const float2*)F2);
    if (e != hipSuccess) return fail(e);
    if ((e = sum_columns(ctx->stream, partial, rows, n_desc, d_out)) != hipSuccess) return fail(e);
    if ((e = hipMemcpyAsync(out_host, d_out, sizeof(double) * n_desc, hipMemcpyDeviceToHost, ctx->stream)) != hipSuccess)
        return fail(e);
    if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return fail(e);
    return true;
}

struct hermes_pair_plan {
    int J = 0, dbl = 0, LM = 0, nu = 0, nch = 0, n_desc = 0, nblocks = 0;
    int rot = 0;
    double R0 = 0.0, dR = 0.0;
    char* mem = nullptr;  // radii | chan | ch_of | factor | partial | channel sums
    double* radii = nullptr;
    int* chan = nullptr;
    int* ch_of = nullptr;
    double* factor = nullptr;
    double* partial = nullptr;
    double* sums = nullptr;
};

int hermes_pair_plan_destroy(hermes_pair_plan* plan) {
    if (!plan) return 0;
    if (plan->mem) (void)hipFree(plan->mem);
    delete plan;
    return 0;
}

int hermes_pair_plan_create(hermes_ctx* ctx, int J, int dbl, const hermes_window_desc* descs, int n_desc,
                            hermes_pair_plan** out) {
    HERMES_REQUIRE(ctx && descs && out, "hermes_pair_plan_create: null argument");
    HERMES_REQUIRE(!ctx->capturing, "hermes_pair_plan_create: the stream is being captured");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(n_desc >= 1 && n_desc <= 4096, "hermes_pair_plan_create: n_desc=%d out of range", n_desc);
    *out = nullptr;
    for (int b = 0; b < n_desc; ++b) {
        if (int rc = check_desc(descs[b])) return rc;
        HERMES_REQUIRE(descs[b].type != HERMES_WIN_SHELL_MULTIPOLE || (descs[b].m == 0 && descs[b].l % 2 == 0),
                       "pair reduction supports only m = 0, even-l multipole windows");
    }
    RadialChannels ch;
    HERMES_REQUIRE(radial_channels(J, dbl, descs, n_desc, ch),
                   "hermes_pair_plan_create: plans take thin shells and even-l m = 0 shell multipoles "
                   "(l <= 10 in FP32, l <= 4 in FP64)");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    hermes_pair_plan* p = new hermes_pair_plan();
    p->J = J;
    p->dbl = dbl;
    p->LM = ch.LM;
    p->nu = ch.nu;
    p->nch = ch.nch;
    p->rot = ch.rot;
    p->R0 = ch.R0;
    p->dR = ch.dR;
    p->n_desc = n_desc;
    p->nblocks = radial_rows(J);
    auto al = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t o_chan = al(sizeof(double) * 2 * ch.nu), o_chof = o_chan + al(sizeof(int) * ch.chan.size()),
                 o_fac = o_chof + al(sizeof(int) * n_desc), o_part = o_fac + al(sizeof(double) * n_desc),
                 o_sums = o_part + al(sizeof(double) * (size_t)p->nblocks * ch.nch),
                 total = o_sums + sizeof(double) * (size_t)ch.nch;
    if (hipMalloc(&p->mem, total) != hipSuccess) {
        delete p;
        hermes_set_error("hermes_pair_plan_create: hipMalloc of %zu bytes failed", total);
        return 1;
    }
    p->radii = (double*)p->mem;
    p->chan = (int*)(p->mem + o_chan);
    p->ch_of = (int*)(p->mem + o_chof);
    p->factor = (double*)(p->mem + o_fac);
    p->partial = (double*)(p->mem + o_part);
    p->sums = (double*)(p->mem + o_sums);
    const std::vector<double> rt = radius_table(ch);
    hipError_t e = hipMemcpy(p->radii, rt.data(), sizeof(double) * rt.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->chan, ch.chan.data(), sizeof(int) * ch.chan.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->ch_of, ch.ch_of.data(), sizeof(int) * n_desc, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->factor, ch.factor.data(), sizeof(double) * n_desc, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        hermes_pair_plan_destroy(p);
        hermes_set_error("hermes_pair_plan_create: upload failed: %s", hipGetErrorString(e));
        return 1;
    }
    *out = p;
    return 0;
}

int hermes_pair_reduce_planned(hermes_ctx* ctx, const hermes_pair_plan* plan, const void* F1, const void* F2,
                               const double* P, double* out_dev) {
    HERMES_REQUIRE(ctx && plan && F1 && F2 && P && out_dev, "hermes_pair_reduce_planned: null argument");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    HERMES_CHECK_HIP(launch_radial(ctx->stream, plan->J, plan->dbl, plan->LM, plan->nblocks, F1, F2, P, plan->radii,
                                   plan->nu, plan->rot, plan->R0, plan->dR, plan->chan, plan->nch, plan->partial));
    HERMES_CHECK_HIP(sum_columns(ctx->stream, plan->partial, plan->nblocks, plan->nch, plan->sums));
    k_plan_out<<<hermes_blocks(plan->n_desc, 64), 64, 0, ctx->stream>>>(plan->sums, plan->ch_of, plan->factor,
                                                                       plan->n_desc, out_dev);
    HERMES_LAUNCH_CHECK();
    return 0;
}

static int pair_reduce_impl(hermes_ctx* ctx, int J, int dbl, const void* F1, const void* F2, const double* P,
                            const hermes_window_desc* descs, int n_desc, double* out_host, char* fixed_ws,
                            size_t fixed_cap) {
    HERMES_REQUIRE(ctx && F1 && F2 && P && descs && out_host, "hermes_pair_reduce: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(n_desc >= 1 && n_desc <= 4096, "hermes_pair_reduce: n_desc=%d out of range", n_desc);
    for (int b = 0; b < n_desc; ++b) {
        if (int rc = check_desc(descs[b])) return rc;
        HERMES_REQUIRE(descs[b].type != HERMES_WIN_SHELL_MULTIPOLE || descs[b].m == 0,
                       "pair reduction supports only m = 0 multipole windows");
        // the half-spectrum sum assumes W(-k) = W(k); an odd-l window is odd in k and its
        // pair product of real fields vanishes identically
        HERMES_REQUIRE(descs[b].type != HERMES_WIN_SHELL_MULTIPOLE || descs[b].l % 2 == 0,
                       "pair reduction supports only even-l multipole windows (odd l gives 0 for real fields)");
    }
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int L = 1 << J;
    const int Lh = L / 2 + 1;
    const int64_t nrep = (int64_t)Lh * Lh * Lh;
    const int nblocks = (int)hermes_blocks(nrep, RED_THREADS, 2048);
    {
        int rc = -1;
        if (pair_reduce_radial(ctx, J, dbl, F1, F2, P, descs, n_desc, nblocks, out_host, fixed_ws, fixed_cap, rc))
            return rc;
        HERMES_REQUIRE(sizeof(double) * (RED_THREADS / 64) * n_desc <= 64 * 1024, "too many windows for one fused pass");
        if (pair_reduce_los(ctx, J, dbl, F1, F2, P, descs, n_desc, nblocks, out_host, fixed_ws, fixed_cap, rc))
            return rc;
    }
    size_t need = sizeof(hermes_window_desc) * n_desc + sizeof(float) * n_desc + 64 + pair_partial_bytes(nblocks, n_desc);
    char* ws = pair_workspace(ctx, fixed_ws, fixed_cap, need);
    if (!ws) return fixed_ws ? 2 : 1;
    hermes_window_desc* d_desc = (hermes_window_desc*)ws;
    float* d_cn = (float*)(ws + sizeof(hermes_window_desc) * n_desc);
    double* partial = (double*)(ws + ((sizeof(hermes_window_desc) * n_desc + sizeof(float) * n_desc + 63) / 64) * 64);
    double* d_out = partial + (size_t)nblocks * n_desc;
    std::vector<float> cn(n_desc);
    for (int b = 0; b < n_desc; ++b)
        cn[b] = descs[b].type == HERMES_WIN_SHELL_MULTIPOLE ? (float)hermes_ylm_cnorm(descs[b].l, 0) : 0.0f;
    HERMES_CHECK_HIP(hipMemcpyAsync(d_desc, descs, sizeof(hermes_window_desc) * n_desc, hipMemcpyHostToDevice, ctx->stream));
    HERMES_CHECK_HIP(hipMemcpyAsync(d_cn, cn.data(), sizeof(float) * n_desc, hipMemcpyHostToDevice, ctx->stream));
    size_t shmem = sizeof(double) * (RED_THREADS / 64) * n_desc;
    bool gen = false, los = false;
    for (int b = 0; b < n_desc; ++b) {
        los = los || descs[b].type >= HERMES_WIN_RING;
        gen = gen || (descs[b].type >= HERMES_WIN_RING && descs[b].axis == 3);
    }
    auto go = [&](auto kernel, auto* f1, auto* f2) {
        kernel<<<nblocks, RED_THREADS, shmem, ctx->stream>>>(L, f1, f2, P, d_desc, d_cn, n_desc, partial);
    };
    if (dbl) {
        auto f1 = (const double2*)F1, f2 = (const double2*)F2;
        if (gen) go(k_pair_reduce<double2, true, true, true>, f1, f2);
        else if (los) go(k_pair_reduce<double2, true, false, true>, f1, f2);
        else go(k_pair_reduce<double2, true, false, false>, f1, f2);
    } else {
        auto f1 = (const float2*)F1, f2 = (const float2*)F2;
        if (gen) go(k_pair_reduce<float2, false, true, true>, f1, f2);
        else if (los) go(k_pair_reduce<float2, false, false, true>, f1, f2);
        else go(k_pair_reduce<float2, false, false, false>, f1, f2);
    }
    HERMES_LAUNCH_CHECK();
    HERMES_CHECK_HIP(sum_columns(ctx->stream, partial, nblocks, n_desc, d_out));
    HERMES_CHECK_HIP(hipMemcpyAsync(out_host, d_out, sizeof(double) * n_desc, hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return 0;
}

int hermes_pair_reduce(hermes_ctx* ctx, int J, int dbl, const void* F1, const void* F2, const double* P,
                       const hermes_window_desc* descs, int n_desc, double* out_host) {
    return pair_reduce_impl(ctx, J, dbl, F1, F2, P, descs, n_desc, out_host, nullptr, 0);
}

// Grid of the fused window kernel: octant positions (x, y) by groups of shells.  At L = 64 a single group is 1089
// waves, about one per SIMD; groups are added up to 8 waves per SIMD (8 shells, l <= 6, two orders: 44 us with one
// group, 34 us with eight; 73 against 84 us at L = 128; from L = 256 one group always fills the chip).
static dim3 mpwin_groups(int J, int threads, ApplyArgs* A) {
    const int nblk = ((1 << J) / 2 + 1) * ((1 << J) / 2 + 1), waves = nblk * (threads / 64);
    int groups = std::max(1, std::min(A->n_shell, (8192 + waves / 2) / waves));
    A->group = (A->n_shell + groups - 1) / groups;
    return dim3(nblk, (A->n_shell + A->group - 1) / A->group);
}

static int make_apply_args(hermes_ctx* ctx, int J, const double* radii, int n_shell, int l, int m, double scale,
                           ApplyArgs* A) {
    HERMES_REQUIRE(n_shell >= 1 && n_shell <= MAX_SHELLS, "n_shell=%d outside 1..%d", n_shell, MAX_SHELLS);
    HERMES_REQUIRE(l >= 0 && l <= 40 && m >= -l && m <= l, "invalid multipole (l=%d, m=%d)", l, m);
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int L = 1 << J;
    A->L = L;
    A->l = l;
    A->m = m;
    A->n_shell = n_shell;
    const int am = m < 0 ? -m : m;
    A->cnorm = (float)hermes_ylm_cnorm(l, am);
    A->scale = (float)scale;
    A->sx = (am & 1) ? -1.0f : 1.0f;
    A->sy = 1.0f;
    A->sz = ((l + am) & 1) ? -1.0f : 1.0f;
    A->group = n_shell;
    for (int s = 0; s < MAX_SHELLS; ++s) A->radii_over_L[s] = s < n_shell ? radii[s] / L : 0.0;
    return 0;
}

int hermes_multipole_apply_f32(hermes_ctx* ctx, int J, const void* H, const double* P, const double* radii,
                               int n_shell, int l, int m, double scale, void* out) {
    HERMES_REQUIRE(ctx && H && P && radii && out, "hermes_multipole_apply_f32: null argument");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    ApplyArgs A;
    int rc = make_apply_args(ctx, J, radii, n_shell, l, m, scale, &A);
    if (rc) return rc;
    const int L = 1 << J;
    const int64_t nrep = (int64_t)(L / 2 + 1) * (L / 2 + 1) * (L / 2 + 1);
    k_multipole_apply<<<hermes_blocks(nrep, 256, 1 << 20), 256, 0, ctx->stream>>>((const float2*)H, P, A,
                                                                                   (float2*)out);
    HERMES_LAUNCH_CHECK();
    return 0;
}

int hermes_multipole_window_ifft_f32(hermes_ctx* ctx, int J, const void* H, const double* P, const double* radii,
                                     int n_shell, int l, int m, double scale, void* out) {
    return hermes_multipole_window_ifft_multi_f32(ctx, J, H, P, radii, n_shell, l, &m, 1, scale, out);
}

// The window + z-pass launch of n_m orders of one l: thin shells at radii (prof_dev = nullptr), or per shell
// the device radial profiles prof_dev (radii unused).
static int mpwin_zpass(hermes_ctx* ctx, int J, const void* H, const double* P, const double* radii,
                       const hermes_radial_profile* prof_dev, int n_shell, int l, const int* ms_host, int n_m,
                       double scale, void* out);

int hermes_multipole_window_zpass_multi_f32(hermes_ctx* ctx, int J, const void* H, const double* P,
                                            const double* radii, int n_shell, int l, const int* ms_host, int n_m,
                                            double scale, void* out) {
    HERMES_REQUIRE(radii, "hermes_multipole_window_zpass_multi_f32: null argument");
    return mpwin_zpass(ctx, J, H, P, radii, nullptr, n_shell, l, ms_host, n_m, scale, out);
}

int hermes_multipole_window_ifft_profiles_f32(hermes_ctx* ctx, int J, const void* H, const double* P,
                                              const hermes_radial_profile* profs_host, int n_shell, int l,
                                              const int* ms_host, int n_m, double scale, void* out) {
    HERMES_REQUIRE(ctx && profs_host, "hermes_multipole_window_ifft_profiles_f32: null argument");
    HERMES_REQUIRE(!ctx->capturing, "hermes_multipole_window_ifft_profiles_f32: not capturable");
    HERMES_REQUIRE(n_shell >= 1 && n_shell <= MAX_SHELLS, "n_shell=%d outside 1..%d", n_shell, MAX_SHELLS);
    for (int s = 0; s < n_shell; ++s)
        if (int rc = check_profile(profs_host[s], l, "hermes_multipole_window_ifft_profiles_f32")) return rc;
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    auto* dev = (hermes_radial_profile*)hermes_workspace(ctx, WS_PROFILE, sizeof(hermes_radial_profile) * n_shell);
    HERMES_REQUIRE(dev, "%s", hermes_last_error());
    HERMES_CHECK_HIP(hipMemcpyAsync(dev, profs_host, sizeof(hermes_radial_profile) * n_shell, hipMemcpyHostToDevice,
                                    ctx->stream));
    const int rc = mpwin_zpass(ctx, J, H, P, nullptr, dev, n_shell, l, ms_host, n_m, scale, out);
    if (rc) return rc;
    // the pageable source of the copy must outlive it: wait before returning to the caller
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return hermes_fft3_inverse_yx(ctx, J, n_m * n_shell, (float2*)out);
}

static int mpwin_zpass(hermes_ctx* ctx, int J, const void* H, const double* P, const double* radii,
                       const hermes_radial_profile* prof_dev, int n_shell, int l, const int* ms_host, int n_m,
                       double scale, void* out) {
    HERMES_REQUIRE(ctx && H && P && ms_host && out, "hermes_multipole_window_zpass_multi_f32: null argument");
    HERMES_REQUIRE(J >= 3 && J <= 10, "hermes_multipole_window_zpass_multi_f32: J=%d outside 3..10", J);
    HERMES_REQUIRE(n_m >= 1 && n_m <= MAX_MP, "hermes_multipole_window_zpass_multi_f32: n_m=%d outside 1..%d", n_m,
                   MAX_MP);
    ApplyArgs A;
    const double zeros[MAX_SHELLS] = {0.0};
    int rc = make_apply_args(ctx, J, radii ? radii : zeros, n_shell, l, ms_host[0], scale, &A);
    if (rc) return rc;
    MultiM M{};
    M.n = n_m;
    for (int i = 0; i < n_m; ++i) {
        const int m = ms_host[i], am = m < 0 ? -m : m;
        HERMES_REQUIRE(m >= -l && m <= l, "invalid multipole (l=%d, m=%d)", l, m);
        M.l[i] = l;
        M.m[i] = m;
        M.cnorm[i] = (float)hermes_ylm_cnorm(l, am);
        M.sx[i] = (am & 1) ? -1.0f : 1.0f;
        M.sz[i] = ((l + am) & 1) ? -1.0f : 1.0f;
    }
    const float2* twg = hermes_twiddles(ctx, J, 1);
    HERMES_REQUIRE(twg, "%s", hermes_last_error());
    const dim3 nblk = mpwin_groups(J, J <= 7 ? 64 : 64 << (J - 7), &A);
    const float2* h = (const float2*)H;
    float2* o = (float2*)out;
#define HERMES_MPW(LG)                                                                                         \
    if (prof_dev && n_m == 1)                                                                                  \
        k_mpwin_zfft_multi<LG, 1, false, true><<<nblk, mpwin_threads<LG>(), 0, ctx->stream>>>(h, P, A, M, twg, o, \
                                                                                              prof_dev);       \
    else if (prof_dev)                                                                                         \
        k_mpwin_zfft_multi<LG, 2, false, true><<<nblk, mpwin_threads<LG>(), 0, ctx->stream>>>(h, P, A, M, twg, o, \
                                                                                              prof_dev);       \
    else if (n_m == 1)                                                                                         \
        k_mpwin_zfft_multi<LG, 1><<<nblk, mpwin_threads<LG>(), 0, ctx->stream>>>(h, P, A, M, twg, o, nullptr);   \
    else                                                                                                       \
        k_mpwin_zfft_multi<LG, 2><<<nblk, mpwin_threads<LG>(), 0, ctx->stream>>>(h, P, A, M, twg, o, nullptr);
    switch (J) {
        case 3: HERMES_MPW(3) break;
        case 4: HERMES_MPW(4) break;
        case 5: HERMES_MPW(5) break;
        case 6: HERMES_MPW(6) break;
        case 7: HERMES_MPW(7) break;
        case 8: HERMES_MPW(8) break;
        case 9: HERMES_MPW(9) break;
        default:
            // L = 1024: two orders per launch would not fit the registers; one launch per order
            for (int i = 0; i < n_m; ++i) {
                MultiM Mi{};
                Mi.n = 1;
                Mi.l[0] = M.l[i];
                Mi.m[0] = M.m[i];
                Mi.cnorm[0] = M.cnorm[i];
                Mi.sx[0] = M.sx[i];
                Mi.sz[0] = M.sz[i];
                if (prof_dev)
                    k_mpwin_zfft_multi<10, 1, false, true><<<nblk, mpwin_threads<10>(), 0, ctx->stream>>>(
                        h, P, A, Mi, twg, o + (size_t)i * n_shell * ((size_t)1 << 30), prof_dev);
                else
                    k_mpwin_zfft_multi<10, 1><<<nblk, mpwin_threads<10>(), 0, ctx->stream>>>(
                        h, P, A, Mi, twg, o + (size_t)i * n_shell * ((size_t)1 << 30), nullptr);
                HERMES_LAUNCH_CHECK();
            }
            break;
    }
#undef HERMES_MPW
    HERMES_LAUNCH_CHECK();
    return 0;
}

int hermes_multipole_window_zpass_pack0_f32(hermes_ctx* ctx, int J, const void* H, const double* P,
                                            const double* radii, int n_shell, int l, double scale, void* out) {
    HERMES_REQUIRE(ctx && H && P && radii && out, "hermes_multipole_window_zpass_pack0_f32: null argument");
    HERMES_REQUIRE(J >= 3 && J <= 9, "hermes_multipole_window_zpass_pack0_f32: J=%d outside 3..9", J);
    HERMES_REQUIRE(l >= 0 && l < 40, "hermes_multipole_window_zpass_pack0_f32: l=%d", l);
    ApplyArgs A;
    int rc = make_apply_args(ctx, J, radii, n_shell, l, 0, scale, &A);
    if (rc) return rc;
    MultiM M{};
    M.n = 2;
    for (int i = 0; i < 2; ++i) {
        M.l[i] = l + i;
        M.m[i] = 0;
        M.cnorm[i] = (float)hermes_ylm_cnorm(l + i, 0);
        M.sx[i] = 1.0f;
        M.sz[i] = ((l + i) & 1) ? -1.0f : 1.0f;
    }
    const float2* twg = hermes_twiddles(ctx, J, 1);
    HERMES_REQUIRE(twg, "%s", hermes_last_error());
    const dim3 nblk = mpwin_groups(J, J <= 7 ? 64 : 64 << (J - 7), &A);
    const float2* h = (const float2*)H;
    float2* o = (float2*)out;
#define HERMES_MPWP(LG) \
    k_mpwin_zfft_multi<LG, 2, true><<<nblk, mpwin_threads<LG>(), 0, ctx->stream>>>(h, P, A, M, twg, o, nullptr);
    switch (J) {
        case 3: HERMES_MPWP(3) break;
        case 4: HERMES_MPWP(4) break;
        case 5: HERMES_MPWP(5) break;
        case 6: HERMES_MPWP(6) break;
        case 7: HERMES_MPWP(7) break;
        case 8: HERMES_MPWP(8) break;
        default: HERMES_MPWP(9) break;
    }
#undef HERMES_MPWP
    HERMES_LAUNCH_CHECK();
    return 0;
}

int hermes_multipole_window_ifft_pack0_f32(hermes_ctx* ctx, int J, const void* H, const double* P,
                                           const double* radii, int n_shell, int l, double scale, void* out) {
    const int rc = hermes_multipole_window_zpass_pack0_f32(ctx, J, H, P, radii, n_shell, l, scale, out);
    if (rc) return rc;
    return hermes_fft3_inverse_yx(ctx, J, n_shell, (float2*)out);
}

int hermes_multipole_window_ifft_multi_f32(hermes_ctx* ctx, int J, const void* H, const double* P,
                                           const double* radii, int n_shell, int l, const int* ms_host, int n_m,
                                           double scale, void* out) {
    const int rc = hermes_multipole_window_zpass_multi_f32(ctx, J, H, P, radii, n_shell, l, ms_host, n_m, scale, out);
    if (rc) return rc;
    return hermes_fft3_inverse_yx(ctx, J, n_m * n_shell, (float2*)out);
}

int hermes_reduce_sum(hermes_ctx* ctx, const void* x, int64_t n, int ncomp, int dbl, double* out_host) {
    HERMES_REQUIRE(ctx && x && out_host, "hermes_reduce_sum: null argument");
    HERMES_REQUIRE(ncomp == 1 || ncomp == 2, "ncomp must be 1 or 2");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int nb = (int)hermes_blocks(n, RED_THREADS, 1024);
    double* ws = (double*)hermes_workspace(ctx, WS_MISC, sizeof(double) * (2 * nb + 2));
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    if (dbl) k_reduce_sum<double><<<nb, RED_THREADS, 0, ctx->stream>>>((const double*)x, n, ncomp, ws);
    else k_reduce_sum<float><<<nb, RED_THREADS, 0, ctx->stream>>>((const float*)x, n, ncomp, ws);
    HERMES_LAUNCH_CHECK();
    HERMES_CHECK_HIP(hermes_reduce::sum_columns(ctx->stream, ws, 2, nb, 2, nullptr, ws + 2 * nb));
    double h[2];
    HERMES_CHECK_HIP(hipMemcpyAsync(h, ws + 2 * nb, sizeof(double) * 2, hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    out_host[0] = h[0];
    if (ncomp == 2) out_host[1] = h[1];
    return 0;
}

}  // extern "C"

// ---------------------------------------------------------------- allocation-free pair reduction
// hermes_pair_reduce_noalloc runs the kernels of hermes_pair_reduce with their scratch (window tables,
// per-block partial sums, group sums, the result row) in this fixed device array instead of the context's
// grow-only workspace, so it never allocates device memory.  Each device holds its own copy until the
// process ends; its address on a device comes from hipGetSymbolAddress, called once per device when the
// first context on it is created (hermes_ctx_create).  Host code must use that address, never the array's
// name.  Every call on a device shares the array, so calls that overlap on one device race; the kernels
// write every scratch word they read, so nothing needs clearing between calls.
constexpr size_t PAIR_SCRATCH_BYTES = size_t(8) << 20;
static __device__ __align__(256) char scratch[PAIR_SCRATCH_BYTES];

constexpr int SCRATCH_MAX_DEVICES = 64;
static char* g_scratch_ptr[SCRATCH_MAX_DEVICES] = {nullptr};
static std::mutex g_scratch_mu;

int hermes_scratch_setup(int device) {
    HERMES_REQUIRE(device >= 0 && device < SCRATCH_MAX_DEVICES, "device %d beyond the scratch table", device);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return 0;
    void* ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        hermes_set_error("hipGetSymbolAddress(scratch) on device %d failed: %s", device, hipGetErrorString(e));
        return 1;
    }
    g_scratch_ptr[device] = (char*)ptr;
    return 0;
}

int hermes_pair_reduce_noalloc(hermes_ctx* ctx, int J, int dbl, const void* F1, const void* F2, const double* P,
                               const hermes_window_desc* descs, int n_desc, double* out_host) {
    HERMES_REQUIRE(ctx, "hermes_pair_reduce_noalloc: null context");
    HERMES_REQUIRE(ctx->device >= 0 && ctx->device < SCRATCH_MAX_DEVICES && g_scratch_ptr[ctx->device],
                   "hermes_pair_reduce_noalloc: no scratch address for device %d", ctx->device);
    return pair_reduce_impl(ctx, J, dbl, F1, F2, P, descs, n_desc, out_host, g_scratch_ptr[ctx->device],
                            PAIR_SCRATCH_BYTES);
}
