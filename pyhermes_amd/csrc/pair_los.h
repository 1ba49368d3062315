// Pair reduction of line-of-sight windows along one coordinate axis (ring, disk, cylshell, cylinder).
//
// Such a window is a product W = p(k_perp) q(k_par), and so is the alias weight P P P, so the sum over the 8
// aliases of an octant position separates: K(perp position, par position) = A(perp) B(par) with A a sum over
// 4 aliases and B over 2.  Then, with S the powers of the octant positions,
//   out[b] = sum_perp A_b(perp) sum_par S(perp, par) B_b(par):
// a matrix product S B on the FP64 matrix cores (rows perp, columns windows) whose result meets A_b in the
// lane that holds it.  The Bessel function of A is evaluated once per (perp alias, window) instead of once per
// (alias, window, position): L / 2 + 1 times 2 fewer.  200 ring windows at L = 128: 30.17 ms that way, 0.13 ms
// now.
// Bound by the Bessel functions (FP64 VALU): 4 (L/2 + 1)^2 of them per window.
#pragma once
#include <hip/hip_runtime.h>

#include "pair_radial.h"
#include "special.h"

namespace hermes_pair {

typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr int LOS_THREADS = 256, LOS_ROWS = 16, LOS_PITCH = 17;  // perp positions per tile; LDS pitch of S

__host__ __device__ inline int los_par_pad(int L) { return (L / 2 + 1 + 3) / 4 * 4; }

// B table: tab[q * ncol + b] = sum over the 2 aliases of par position q; zero beyond the positions and windows.
__global__ void k_los_par_table(int L, const double* __restrict__ P, const hermes_window_desc* __restrict__ descs,
                                int nd, int ncol, double* __restrict__ tab) {
    const int n = los_par_pad(L) * ncol;
    const double inv_L = 1.0 / L;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int q = i / ncol, b = i % ncol;
        double t = 0.0;
        if (q <= L / 2 && b < nd) {
            const double H = descs[b].a1;
            const bool cosine = descs[b].type == HERMES_WIN_RING || descs[b].type == HERMES_WIN_DISK;
            for (int a = 0; a < 2; ++a) {
                const int k = a ? L - q : q;
                const double f = 2.0 * HERMES_PI * (k * inv_L) * H;
                t += P[k] * (cosine ? cos(f) : (f == 0.0 ? 1.0 : sin(f) / f));
            }
        }
        tab[i] = t;
    }
}

// Workgroup (row, group): perp tiles row, row + gridDim.x, ... of 16 positions, and window tiles
// [group * tpb, ...) of 16 windows, one wave each in turn.  axis: 0, 1, 2 = x, y, z; the perp position index
// runs over the other two coordinates, the later one fastest.
template <typename C>
__global__ __launch_bounds__(LOS_THREADS, 2) void k_pair_los(int L, int axis, const C* __restrict__ F1,
                                                          const C* __restrict__ F2, const double* __restrict__ P,
                                                          const hermes_window_desc* __restrict__ descs, int nd,
                                                          const double* __restrict__ tab, int ncol, int tpb,
                                                          int nptile, double* __restrict__ partial) {
    extern __shared__ double smem[];  // S [par][LOS_PITCH] | window sums [tpb * 16]
    const int Lh = L / 2 + 1, LhP = los_par_pad(L), half = L / 2;
    double* S = smem;
    double* wacc = smem + LhP * LOS_PITCH;
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int nperp = Lh * Lh;
    const double inv_L = 1.0 / L;
    const int t0 = blockIdx.y * tpb, nt = min(tpb, ncol / 16 - t0);
    for (int i = tid; i < tpb * 16; i += LOS_THREADS) wacc[i] = 0.0;
    for (int pt = blockIdx.x; pt < nptile; pt += gridDim.x) {
        __syncthreads();
        // along z (axis 2) consecutive threads take consecutive par positions, otherwise perp positions: both z
        for (int e = tid; e < LhP * LOS_ROWS; e += LOS_THREADS) {
            const int r = axis == 2 ? e / LhP : e % LOS_ROWS, q = axis == 2 ? e % LhP : e / LOS_ROWS;
            const int p = pt * LOS_ROWS + r, u = p / Lh, v = p % Lh;
            double s = 0.0;
            if (p < nperp && q <= half) {
                const int x = axis == 0 ? q : u, y = axis == 0 ? u : (axis == 1 ? q : v), z = axis == 2 ? q : v;
                s = F1 == F2 ? octant_power<true>(F1, F2, L, x, y, z) : octant_power<false>(F1, F2, L, x, y, z);
            }
            S[q * LOS_PITCH + r] = s;
        }
        __syncthreads();
        for (int t = wave; t < nt; t += LOS_THREADS / 64) {
            const int b = (t0 + t) * 16 + lane % 16;
            const double* tb = tab + (lane / 16) * ncol + b;
            const double* sa = S + (lane / 16) * LOS_PITCH + lane % 16;
            double4_t acc = {0.0, 0.0, 0.0, 0.0};
            for (int q = 0; q < LhP; q += 4)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sa[q * LOS_PITCH], tb[q * ncol], acc, 0, 0, 0);
            // acc[j]: row 4 j + lane / 16 (perp position of the tile), column lane % 16 (window)
            const hermes_window_desc* d = descs + (b < nd ? b : nd - 1);
            const double R = d->a0;
            const bool ring = d->type == HERMES_WIN_RING || d->type == HERMES_WIN_CYLSHELL;
            double sum = 0.0;
            for (int j = 0; j < 4; ++j) {
                const int p = min(pt * LOS_ROWS + 4 * j + lane / 16, nperp - 1), u = p / Lh, v = p % Lh;
                double A = 0.0;
                for (int a = 0; a < 4; ++a) {
                    const int iu = (a & 2) ? L - u : u, iv = (a & 1) ? L - v : v;
                    const double ku = iu * inv_L, kv = iv * inv_L;
                    A += P[iu] * P[iv] * los_perp_f64(ring, sqrt(ku * ku + kv * kv) * R);
                }
                sum = fma(acc[j], A, sum);
            }
            const double s4 = merge32(sum, sum);
            const double tot = merge16(s4, s4);
            if (lane < 16) wacc[t * 16 + lane] += tot;
        }
    }
    __syncthreads();
    for (int i = tid; i < nt * 16; i += LOS_THREADS) {
        const int b = t0 * 16 + i;
        if (b < nd) partial[(int64_t)blockIdx.x * nd + b] = wacc[i];
    }
}

}  // namespace hermes_pair
