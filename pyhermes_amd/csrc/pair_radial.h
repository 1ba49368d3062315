// Pair reduction of thin shells and even-l, m = 0 shell multipoles, all channels in one pass.
//
// For an octant position (x, y, z) in [0, L/2]^3 and its 8 aliases a the window of radius R and order l is
// sum_a P(a) j_l(2 pi |a| R / L) P_l(a_z / |a|).  The radial factor depends on |a| only, so it is shared by
// the (up to six) positions whose coordinates are permutations of one sorted triple i >= j >= k: their powers
// are gathered per coordinate that takes the z role,
//   w[a][l] = P(a) sum_c power_c P_l(a_c / |a|),   out[R, l] = sum_triples sum_a j_l(2 pi |a| R / L) w[a][l],
// which leaves a sixth of the radial evaluations.  All arithmetic is FP64 (spectra FP32 or FP64): without
// packed instructions an FP32 multiply-add issues at the FP64 rate here, so FP32 windows would save nothing.
//
// ROT (equally spaced radii R0 + u dR): sin and cos of x = 2 pi |a| R_u / L by rotating those at R0 through
// the angle 2 pi |a| dR / L (both reduced from exact turn fractions once per alias), four FMAs per radius; each
// rotation adds about two ulps to |sin|, |cos| <= 1.  1 / x comes from 1 / (2 pi |a|) times 1 / R.  The orders
// follow by the upward recurrence for x >= XMIN (where the second solution, which amplifies rounding, is of
// order one) and otherwise by the power series of the two top orders and the downward recurrence.
//
// Bound by FP64 VALU issue (about 0.6 ms of instructions at L = 512) with the gather of the powers, 0.3 ms, partly
// beside it: 250 registers leave two waves per SIMD.  Thin shells and l = 0, 2, 4 at 30 radii: 5.70 ms per pass at
// L = 512 (FP32 spectra) and 5.36 ms at L = 256 (FP64) with one thread per position, an FP32 sin/cos or an FP64
// sincos and divisions per (alias, radius), and a wave reduction per channel and position; 1.23 ms and 0.20 ms with
// this sharing; 0.93 and 0.18 with unconditional loads, one series test per radius and everything a step needs
// fetched a step ahead.  Four aliases at a time and three waves per SIMD: 1.04 and 0.23 (twice the reductions).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "special.h"

namespace hermes_pair {

__device__ __forceinline__ double make_f64(unsigned lo, unsigned hi) {
    return __hiloint2double((int)hi, (int)lo);
}

// a summed over the two half-waves in lanes 0..31, b in lanes 32..63.
__device__ __forceinline__ double merge32(double a, double b) {
    const unsigned al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
    const auto lo = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return make_f64(lo[0], hi[0]) + make_f64(lo[1], hi[1]);
}

// Rows of 16 lanes: a summed over row pairs (0, 1) and (2, 3) in rows 0 and 2, b in rows 1 and 3.
__device__ __forceinline__ double merge16(double a, double b) {
    const unsigned al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b), bh = __double2hiint(b);
    const auto lo = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return make_f64(lo[0], hi[0]) + make_f64(lo[1], hi[1]);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// Sum over the 16 lanes of a row, in every lane (row rotations by 8, 4, 2, 1).
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_f64<0x128>(v);
    v += dpp_f64<0x124>(v);
    v += dpp_f64<0x122>(v);
    v += dpp_f64<0x121>(v);
    return v;
}

// Four wave sums at once: row r of 16 lanes ends with the sum of v[QUAD_OF_ROW(r)].
__device__ __forceinline__ double quad_sum(double v0, double v1, double v2, double v3) {
    return row_sum(merge16(merge32(v0, v1), merge32(v2, v3)));
}
__device__ __forceinline__ int quad_of_row(int row) { return ((row & 1) << 1) | (row >> 1); }

// sum over the mirror modes (x | L-x, y | L-y, z | L-z) of Re F1 conj F2 from the half spectra (SAME: F2 is F1).  The
// four loads are unconditional, a mirror that is the mode itself is left out afterwards: a load under a condition is
// waited for before the next one is issued.
template <bool SAME, typename C>
__device__ __forceinline__ double octant_power(const C* __restrict__ F1, const C* __restrict__ F2, int L, int x, int y,
                                               int z) {
    const int Lh = L / 2 + 1;
    const int xm = (L - x) & (L - 1), ym = (L - y) & (L - 1);
    const double wz = (z == 0 || z == L / 2) ? 1.0 : 2.0;
    C f[4], g[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int64_t i = ((int64_t)(a >> 1 ? xm : x) * L + ((a & 1) ? ym : y)) * Lh + z;
        f[a] = F1[i];
        g[a] = SAME ? f[a] : F2[i];
    }
    double p = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const double t = (double)f[a].x * (double)g[a].x + (double)f[a].y * (double)g[a].y;
        p += ((a >> 1 && xm == x) || ((a & 1) && ym == y)) ? 0.0 : wz * t;
    }
    return p;
}

template <int N>
__device__ __forceinline__ double ipow(double x) {
    if constexpr (N == 0) return 1.0;
    else if constexpr (N % 2) return x * ipow<N - 1>(x);
    else {
        const double h = ipow<N / 2>(x);
        return h * h;
    }
}

constexpr double odd_factorial(int l) {  // (2l + 1)!!
    double f = 1.0;
    for (int n = 1; n <= l; ++n) f *= 2.0 * n + 1.0;
    return f;
}

// below XMIN the series (TERMS terms: the last is under 1e-18 of the first at x = XMIN)
constexpr double radial_xmin(int lmax) { return lmax == 0 ? 1.0 : (lmax == 4 ? 3.0 : 7.0); }
constexpr int radial_terms(int lmax) { return lmax == 0 ? 9 : (lmax == 4 ? 13 : 20); }

// j_0 .. j_LMAX at x = h^(1/2) >= 0 below XMIN; ix = 1 / x (not used at x = 0).
template <int LMAX>
__device__ __forceinline__ void radial_small(double x, double ix, double* j) {
    constexpr int T = radial_terms(LMAX);
    const double h = x * x;
    if constexpr (LMAX == 0) {
        j[0] = jl_series<0, T>(h);
    } else {
        j[LMAX] = jl_series<LMAX, T>(h) * (ipow<LMAX>(x) * (1.0 / odd_factorial(LMAX)));
        j[LMAX - 1] = jl_series<LMAX - 1, T>(h) * (ipow<LMAX - 1>(x) * (1.0 / odd_factorial(LMAX - 1)));
#pragma unroll
        for (int n = LMAX - 1; n >= 1; --n) j[n - 1] = (2.0 * n + 1.0) * ix * j[n] - j[n + 1];
        if (x < 1e-8) {  // the recurrence's 1 / x; below, every order is its leading term
            j[0] = 1.0;
#pragma unroll
            for (int l = 1; l <= LMAX; ++l) j[l] = ipow<1>(x) * (l == 1 ? 1.0 / 3.0 : 0.0);
        }
    }
}

// Blocks of BT^3 positions: the six arrangements of a sorted triple of blocks are read along z (runs of BT
// values: 64 bytes or more) into LDS, and the sorted triples inside, listed without gaps, go to the threads.
// BT = 8 with 4 waves for L >= 256; BT = 4 with one wave below, where 8^3 blocks would leave CUs idle.
template <int BT>
constexpr int radial_threads() {
    return BT == 8 ? 256 : 64;
}

__host__ __device__ inline int tetra(int n) { return n * (n + 1) * (n + 2) / 6; }

// Radii whose sums are reduced together.
constexpr int radial_step(int lmax) { return lmax == 0 ? 4 : 1; }

// Aliases whose state (6 + LMAX / 2 doubles each) a thread holds at a time: all eight in 256 registers up to l = 4;
// beyond, eight leave 160 registers in scratch, four 60.
constexpr int radial_aliases(int lmax) { return lmax <= 4 ? 8 : 4; }

// Workgroup (row, group): blocks row, row + gridDim.x, ... and the `per` radii from group * per on (all of them unless
// the rows alone leave SIMDs idle, see radial_groups).
template <int LMAX, bool ROT, int BT, typename C>
__global__ __launch_bounds__(radial_threads<BT>(), 2) void k_pair_radial(int L, const C* __restrict__ F1,
                                                                      const C* __restrict__ F2,
                                                                      const double* __restrict__ P,
                                                                      const double* __restrict__ radii, int nu,
                                                                      double R0, double dR,
                                                                      const int* __restrict__ chan, int nch, int nblk,
                                                                      int per, double* __restrict__ partial) {
    constexpr int NT = radial_threads<BT>(), NW = NT / 64, B3 = BT * BT * BT, PER = B3 / NT;
    constexpr int NE = LMAX / 2 + 1;         // even orders
    constexpr int UC = radial_step(LMAX);    // radii per reduction
    constexpr int NA = radial_aliases(LMAX);
    constexpr int NQ = (UC * NE + 3) / 4;    // groups of four wave sums
    constexpr double XMIN = radial_xmin(LMAX);
    extern __shared__ double wacc[];  // [waves][nch]
    __shared__ double pw[6 * B3];     // powers of the arrangements ijk, jik, ikj, kij, jki, kji
    __shared__ unsigned short list[B3];
    __shared__ int cnt[PER * NW];
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int half = L / 2;
    const int ub = ROT ? 0 : blockIdx.y * per, ue = ROT ? nu : min(nu, ub + per);
    for (int i = tid; i < NW * nch; i += NT) wacc[i] = 0.0;
    for (int blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        int bi = (int)cbrtf(6.0f * (float)blk);
        while (tetra(bi) > blk) --bi;
        while (tetra(bi + 1) <= blk) ++bi;
        const int rem = blk - tetra(bi);
        int bj = (int)sqrtf(2.0f * (float)rem);
        while (bj * (bj + 1) / 2 > rem) --bj;
        while ((bj + 1) * (bj + 2) / 2 <= rem) ++bj;
        const int bk = rem - bj * (bj + 1) / 2;
        __syncthreads();  // the previous block's powers and list are consumed
        auto gather = [&](auto same) {
#pragma unroll
            for (int o = 0; o < 6; ++o) {
                const int X = (o == 0 || o == 2) ? bi : ((o == 1 || o == 4) ? bj : bk);
                const int Y = (o == 1 || o == 3) ? bi : ((o == 0 || o == 5) ? bj : bk);
                const int Z = (o >= 4) ? bi : (o >= 2 ? bj : bk);
#pragma unroll
                for (int q = 0; q < PER; ++q) {
                    const int r = tid + q * NT;
                    const int x = X * BT + r / (BT * BT), y = Y * BT + (r / BT) % BT, z = Z * BT + r % BT;
                    const double p = octant_power<decltype(same)::value>(F1, F2, L, min(x, half), min(y, half),
                                                                         min(z, half));
                    pw[o * B3 + r] = (x <= half && y <= half && z <= half) ? p : 0.0;
                }
            }
        };
        if (F1 == F2) gather(std::true_type());
        else gather(std::false_type());
        // the sorted triples of the block, in order
        bool val[PER];
        int rank[PER];
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int r = tid + q * NT;
            const int i = bi * BT + r / (BT * BT), j = bj * BT + (r / BT) % BT, k = bk * BT + r % BT;
            val[q] = i <= half && i >= j && j >= k;
            const unsigned long long m = __ballot(val[q]);
            rank[q] = __popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) cnt[q * NW + wave] = __popcll(m);
        }
        __syncthreads();
        int nact = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q)
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                if (w == wave && val[q]) list[nact + rank[q]] = (unsigned short)(tid + q * NT);
                nact += cnt[q * NW + w];
            }
        __syncthreads();
        for (int base = wave * 64; base < nact; base += NT) {
            const bool active = base + lane < nact;
            const int r = list[active ? base + lane : 0];
            const int a0 = r / (BT * BT), b0 = (r / BT) % BT, c0 = r % BT;
            const int i = bi * BT + a0, j = bj * BT + b0, k = bk * BT + c0;
            auto at = [&](int o, int a, int b, int c) { return pw[o * B3 + (a * BT + b) * BT + c]; };
            // power of the arrangements with k, j, i in the z role, each position once
            double pk = at(0, a0, b0, c0), pj = 0.0, pi = 0.0;
            if (i != j) pk += at(1, b0, a0, c0);
            if (i != j && j != k) pj = at(2, a0, c0, b0) + at(3, c0, a0, b0);
            if (i != k) {
                pi = at(4, b0, c0, a0);
                if (j != k) pi += at(5, c0, b0, a0);
            }
            if (!active) pk = pj = pi = 0.0;
#pragma unroll 1
            for (int h = 0; h < 8; h += NA) {
                double w[NA][NE], iq[NA];
                double sn[NA], cs[NA], sd[NA], cd[NA], ra[NA];
#pragma unroll
                for (int a = 0; a < NA; ++a) {
                    const int ax = (a + h & 4) ? i - L : i, ay = (a + h & 2) ? j - L : j, az = (a + h & 1) ? k - L : k;
                    const double p = P[ax < 0 ? -ax : ax] * P[ay < 0 ? -ay : ay] * P[az < 0 ? -az : az];
                    const int n2 = ax * ax + ay * ay + az * az;
                    const double rn = sqrt((double)n2), inv = n2 ? 1.0 / rn : 0.0;
                    ra[a] = rn;
                    iq[a] = n2 ? inv * (0.5 / HERMES_PI) : __builtin_inf();
                    w[a][0] = p * (pi + pj + pk);
                    if constexpr (NE > 1) {
                        const double mus[3] = {ax * inv, ay * inv, az * inv}, ps[3] = {pi, pj, pk};
#pragma unroll
                        for (int e = 1; e < NE; ++e) w[a][e] = 0.0;
#pragma unroll
                        for (int c = 0; c < 3; ++c) {
                            const double v = n2 ? p * ps[c] : 0.0;
                            double pm = 1.0, pc = mus[c];
#pragma unroll
                            for (int n = 1; n < LMAX; ++n) {
                                const double pn = ((2.0 * n + 1.0) * mus[c] * pc - n * pm) * (1.0 / (n + 1.0));
                                pm = pc;
                                pc = pn;
                                if (n % 2) w[a][(n + 1) / 2] += v * pn;
                            }
                        }
                    }
                    if constexpr (ROT) {
                        const double t0 = rn * R0, td = rn * dR;
                        sincospi(2.0 * (t0 - floor(t0)), &sn[a], &cs[a]);
                        sincospi(2.0 * (td - floor(td)), &sd[a], &cd[a]);
                    }
                }
                // radii and channels of the next step are fetched a step ahead, and the channels' sums are read before
                // the step's arithmetic: two waves per SIMD do not cover their latencies
                double Rn[UC], iRn[UC];
                int chn[NQ];
                auto fetch = [&](int u0) {
#pragma unroll
                    for (int q = 0; q < UC; ++q) {
                        const int u = u0 + q < nu ? u0 + q : nu - 1;
                        Rn[q] = radii[u];
                        iRn[q] = radii[nu + u];
                    }
#pragma unroll
                    for (int g = 0; g < NQ; ++g) {
                        const int n = 4 * g + quad_of_row(lane / 16), u = u0 + n / NE;
                        chn[g] = (lane % 16 == 0 && n < UC * NE && u < nu) ? chan[u * (LMAX + 1) + 2 * (n % NE)] : -1;
                    }
                };
                fetch(ub);
                for (int u0 = ub; u0 < ue; u0 += UC) {
                    double kb[NQ * 4], Ru[UC], iRu[UC], sum[NQ];
                    int ch[NQ];
#pragma unroll
                    for (int q = 0; q < UC; ++q) Ru[q] = Rn[q], iRu[q] = iRn[q];
#pragma unroll
                    for (int g = 0; g < NQ; ++g) {
                        ch[g] = chn[g];
                        sum[g] = ch[g] >= 0 ? wacc[wave * nch + ch[g]] : 0.0;
                    }
                    fetch(u0 + UC);
#pragma unroll
                    for (int v = 0; v < NQ * 4; ++v) kb[v] = 0.0;
#pragma unroll
                    for (int q = 0; q < UC; ++q) {
                        const int u = u0 + q;
                        if (u < nu) {
                            const double R = Ru[q], iR = iRu[q];
                            // One test for all of them (the first is the nearest to the origin): without a branch per
                            // alias the eight serial chains of the recurrence overlap.
                            auto add = [&](auto recurrence_only) {
#pragma unroll
                                for (int a = 0; a < NA; ++a) {
                                    double s = 0.0, c = 0.0;
                                    if constexpr (ROT) {
                                        s = sn[a];
                                        c = cs[a];
                                        sn[a] = fma(s, cd[a], c * sd[a]);  // for the next radius
                                        cs[a] = fma(c, cd[a], -(s * sd[a]));
                                    } else {
                                        const double t = ra[a] * R;
                                        sincospi(2.0 * (t - floor(t)), &s, &c);
                                    }
                                    double jv[LMAX + 1];
                                    const double ix = iq[a] * iR;
                                    if (decltype(recurrence_only)::value || R >= XMIN * iq[a]) {
                                        jv[0] = s * ix;
                                        if constexpr (LMAX >= 1) {
                                            jv[1] = (jv[0] - c) * ix;
#pragma unroll
                                            for (int n = 1; n < LMAX; ++n)
                                                jv[n + 1] = (2.0 * n + 1.0) * ix * jv[n] - jv[n - 1];
                                        }
                                    } else {
                                        radial_small<LMAX>(ROT ? 1.0 / ix : 2.0 * HERMES_PI * (ra[a] * R), ix, jv);
                                    }
#pragma unroll
                                    for (int e = 0; e < NE; ++e) kb[q * NE + e] = fma(jv[2 * e], w[a][e], kb[q * NE + e]);
                                }
                            };
                            if (__all(R >= XMIN * iq[0])) add(std::true_type());
                            else add(std::false_type());
                        }
                    }
#pragma unroll
                    for (int g = 0; g < NQ; ++g) {
                        const double v = quad_sum(kb[4 * g], kb[4 * g + 1], kb[4 * g + 2], kb[4 * g + 3]);
                        if (ch[g] >= 0) wacc[wave * nch + ch[g]] = sum[g] + v;
                    }
                }
            }
        }
    }
    __syncthreads();
    auto finish = [&](int b) {
        double s = 0.0;
        for (int w = 0; w < NW; ++w) s += wacc[w * nch + b];
        partial[(int64_t)blockIdx.x * nch + b] = s;
    };
    if constexpr (ROT) {
        for (int b = tid; b < nch; b += NT) finish(b);
    } else {  // the channels of these radii
        for (int i = ub * (LMAX + 1) + tid; i < ue * (LMAX + 1); i += NT)
            if (chan[i] >= 0) finish(chan[i]);
    }
}

}  // namespace hermes_pair
