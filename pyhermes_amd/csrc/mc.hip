// Monte-Carlo 3PCF kernels.
//
// * hermes_interpolate: n(x) = sum_27 eps[(c - s) & mask] phi phi phi at scaled
//   positions (+ offset), FP64 (wavelet_grid.py:143-186).
// * hermes_mc_triplet_box: the box-random-centre estimator of
//   corr3pcf_kernels.py:100-140 for one (R1, R2, mu): sum over rotations and
//   centres of n1 n2 n3 / (n_rot N), rotation uniforms supplied by the caller,
//   triangle geometry of corr3pcf_kernels.py:21-63, deterministic FP64 sums.
// * hermes_mc_binned: binned triangle sampler over (r1, r2, cos theta) bins with
//   an optional importance proposal (tables built by the host from the learned
//   proposal), Philox4x32-10 counter-based random numbers, per-bin sums of
//   w f, (w f)^2 and counts accumulated with deterministic int64 fixed-point
//   atomics.  Optionally records per-sample features for proposal training.
// * hermes_mc_bucketize: the proposal's density buckets on a sub-cell grid and
//   the stable per-bucket list of sub-cells the sampler draws from.
#include "../../include/hermes_amd.h"
#include "hermes_common.h"
#include "reduce.h"

#include <algorithm>
#include <cmath>

namespace {

constexpr double TWO_PI = 6.283185307179586476925286766559;

// Field layouts the interpolation reads (all FP64).
//   GRID_PLAIN    (L, L, L) z fastest, one point per lane, 8-byte loads (any alignment)
//   GRID_ALIGNED  the same on a 16-byte aligned grid: aligned pairs of z neighbours by one load
//   GRID_BRICK    2 x 2 x 4 cells (x, y, z) to a 128-byte line (k_brick), eight lanes to a point: a lane holds one
//                 16-byte pair of the line, so each of the 4 or 8 lines that a 3 x 3 x 3 neighbourhood meets (6 on
//                 average; 9 * 1.125 in the plain layout) is requested once, by one instruction
// Interpolation at random points is bound by the lines a CU can have outstanding, not by bytes or arithmetic: more
// waves per SIMD or fewer lines read by one lane at a time do not help (whole calls of 2e7 triangles at L = 256:
// 11.1 ms with one wave per SIMD, 11.8 with four, 13.9 with bricks read by one lane), fewer line requests do (7.6).
enum GridLayout { GRID_PLAIN = 0, GRID_ALIGNED = 1, GRID_BRICK = 2 };

template <int LAYOUT>
__device__ __forceinline__ int off_x(int x, int lg) {
    return LAYOUT == GRID_BRICK ? ((x >> 1) << (2 * lg + 1)) + ((x & 1) << 3) : x << (2 * lg);
}
template <int LAYOUT>
__device__ __forceinline__ int off_y(int y, int lg) {
    return LAYOUT == GRID_BRICK ? ((y >> 1) << (lg + 2)) + ((y & 1) << 2) : y << lg;
}
template <int LAYOUT>
__device__ __forceinline__ int off_z(int z) {
    return LAYOUT == GRID_BRICK ? ((z >> 2) << 4) + (z & 3) : z;
}

// Cell of a scaled coordinate reduced to [0, L) (exact for |s| < 2^53) and its fraction index.
__device__ __forceinline__ void cell_of(double s, int L, int res, int& cell, int& frac) {
    const double c = floor(s);
    // s in (-2^-54, 0) rounds s - floor(s) to 1.0; keep the phi index inside the table
    frac = min((int)((s - c) * res), res - 1);
    cell = (int)(c - L * floor(c * (1.0 / L)));
}

// n(s) = sum over the 27 cells c - (a, b, e) of g phi phi phi.  SPHI: phi holds the table interleaved,
// phi[3 f + a] = phi(a + f / res) (LDS copies); otherwise phi[f + a res].  The three z taps are one aligned pair
// and one single: two loads a row, with the weights put in their order.
template <int LAYOUT, bool SPHI>
__device__ __forceinline__ double interp_at(const double* __restrict__ g, const double* phi, int lg, int res,
                                            double sx, double sy, double sz) {
    const int L = 1 << lg, m = L - 1;
    int cx, cy, cz, fx, fy, fz;
    cell_of(sx, L, res, cx, fx);
    cell_of(sy, L, res, cy, fy);
    cell_of(sz, L, res, cz, fz);
    auto tap = [&](int f, int a) { return SPHI ? phi[3 * f + a] : phi[f + a * res]; };
    const int z0 = (cz - 2) & m;  // first cell of the row; taps 2, 1, 0 in ascending z
    const bool odd = z0 & 1;
    const int zp = odd ? (z0 + 1) & m : z0, zs = odd ? z0 : (z0 + 2) & m;
    const double t0 = tap(fz, 0), t1 = tap(fz, 1), t2 = tap(fz, 2);
    const double wa = odd ? t1 : t2, wb = odd ? t0 : t1, ws = odd ? t2 : t0;
    const int op = off_z<LAYOUT>(zp), os = off_z<LAYOUT>(zs);
    double acc = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int ox = off_x<LAYOUT>((cx - a) & m, lg);
        const double px = tap(fx, a);
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const double* row = g + (int64_t)(ox + off_y<LAYOUT>((cy - b) & m, lg));
            const double s1 = row[os];
            double va, vb;
            if (LAYOUT == GRID_PLAIN) {
                va = row[op];
                vb = row[op + 1];
            } else {
                const double2 v = *(const double2*)(row + op);
                va = v.x;
                vb = v.y;
            }
            acc = fma(px * tap(fy, b), fma(va, wa, fma(vb, wb, s1 * ws)), acc);
        }
    }
    return acc;
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// interp_at on a bricked grid for the 64 points of a wave (all lanes must call; lane l gets the value of its own
// point): in round r the lanes 8 k .. 8 k + 7 take the point of lane 8 r + k, one pair of cells of a line each.
// Cells outside the neighbourhood are neither read nor added.
__device__ __forceinline__ double interp_bricks(const double* __restrict__ g, const double* sphi, int lg, int res,
                                                double sx, double sy, double sz) {
    const int L = 1 << lg, m = L - 1, lane = threadIdx.x & 63;
    int cx, cy, cz, fx, fy, fz;
    cell_of(sx, L, res, cx, fx);
    cell_of(sy, L, res, cy, fy);
    cell_of(sz, L, res, cz, fz);
    const int cells = ((cx - 2) & m) | ((cy - 2) & m) << 10 | ((cz - 2) & m) << 20;  // the neighbourhood's first cell
    const int fracs = fx | fy << 10 | fz << 20;
    const int ix = (lane >> 2) & 1, iy = (lane >> 1) & 1, iz = lane & 1;  // this lane's pair of a line
    double mine = 0.0;
#pragma unroll 2
    for (int r = 0; r < 8; ++r) {
        const int src = 8 * r + (lane >> 3);
        const int c = __shfl(cells, src, 64), f = __shfl(fracs, src, 64);
        const int x0 = c & 1023, y0 = (c >> 10) & 1023, z0 = (c >> 20) & 1023;
        const double* tx = sphi + 3 * (f & 1023);
        const double* ty = sphi + 3 * ((f >> 10) & 1023);
        const double* tz = sphi + 3 * ((f >> 20) & 1023);
        // cell o = 0, 1, 2 of the window has tap 2 - o
        int ox[2], oy[2];
        double wx[2], wy[2];
        bool vx[2], vy[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int a = 2 * q + ix - (x0 & 1), b = 2 * q + iy - (y0 & 1);
            vx[q] = a >= 0 && a <= 2;
            vy[q] = b >= 0 && b <= 2;
            wx[q] = tx[vx[q] ? 2 - a : 0];
            wy[q] = ty[vy[q] ? 2 - b : 0];
            ox[q] = off_x<GRID_BRICK>((x0 + a) & m, lg);
            oy[q] = off_y<GRID_BRICK>((y0 + b) & m, lg);
        }
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int e0 = 4 * q + 2 * iz - (z0 & 3), e1 = e0 + 1;
            const bool v0 = e0 >= 0 && e0 <= 2, v1 = e1 >= 0 && e1 <= 2;
            const double w0 = tz[v0 ? 2 - e0 : 0], w1 = tz[v1 ? 2 - e1 : 0];
            const int oz = off_z<GRID_BRICK>((z0 + e0) & m);  // even: z0 + e0 = 4 k + 2 iz
            const bool vz = v0 || v1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (vz && vx[i >> 1] && vy[i & 1]) {
                    const double2 v = *(const double2*)(g + (int64_t)(ox[i >> 1] + oy[i & 1] + oz));
                    const double t = (v0 ? v.x * w0 : 0.0) + (v1 ? v.y * w1 : 0.0);
                    acc = fma(wx[i >> 1] * wy[i & 1], t, acc);
                }
            }
        }
        acc += dpp_f64<0xB1>(acc);   // quad_perm 1 0 3 2
        acc += dpp_f64<0x4E>(acc);   // quad_perm 2 3 0 1
        acc += dpp_f64<0x141>(acc);  // row_half_mirror: the other four lanes of the eight
        const double v = __shfl(acc, (lane & 7) * 8, 64);
        if ((lane >> 3) == r) mine = v;
    }
    return mine;
}

template <int LAYOUT>
__device__ __forceinline__ double interp(const double* __restrict__ g, const double* sphi, int lg, int res, double sx,
                                         double sy, double sz) {
    if constexpr (LAYOUT == GRID_BRICK) return interp_bricks(g, sphi, lg, res, sx, sy, sz);
    else return interp_at<LAYOUT, true>(g, sphi, lg, res, sx, sy, sz);
}

// Bricked copy of a grid (GRID_BRICK), L >= 4.
__global__ __launch_bounds__(256) void k_brick(const double* __restrict__ g, int lg, double* __restrict__ out) {
    const int64_t n = (int64_t)1 << (3 * lg);
    const int m = (1 << lg) - 1;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int z = (int)(i & m), y = (int)(i >> lg) & m, x = (int)(i >> (2 * lg));
        out[off_x<GRID_BRICK>(x, lg) + off_y<GRID_BRICK>(y, lg) + off_z<GRID_BRICK>(z)] = g[i];
    }
}

// The scaling function in LDS, tap-interleaved; res = 1024.  All loads are in flight before the first store (a call of
// 60,000 triangles is one workgroup to a CU and waits for them twice).
template <int NT>
__device__ __forceinline__ void load_phi(double* sphi, const double* __restrict__ phi, int tid) {
    static_assert(3 * 1024 % NT == 0, "table staging");
    double v[3 * 1024 / NT];
#pragma unroll
    for (int j = 0; j < 3 * 1024 / NT; ++j) v[j] = phi[tid + j * NT];
#pragma unroll
    for (int j = 0; j < 3 * 1024 / NT; ++j) {
        const int i = tid + j * NT;
        sphi[3 * (i & 1023) + (i >> 10)] = v[j];
    }
}

__global__ void k_interpolate(const double* __restrict__ g, const double* __restrict__ spos, int64_t n,
                              const double* __restrict__ phi, int lg, int res, double dx, double dy, double dz,
                              double* __restrict__ out) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x)
        out[p] = interp_at<GRID_PLAIN, false>(g, phi, lg, res, spos[3 * p] + dx, spos[3 * p + 1] + dy,
                                              spos[3 * p + 2] + dz);
}

// corr3pcf_kernels.py:21-63
__device__ __forceinline__ void triangle_offsets(double R1, double R2, double mu, double ph, double ct1, double al,
                                                 double o[6]) {
    const double st1 = sqrt(1.0 - ct1 * ct1);
    double sp, cp;
    sincos(ph, &sp, &cp);
    const double dx1 = st1 * cp, dy1 = st1 * sp, dz1 = ct1;
    o[0] = R1 * dx1;
    o[1] = R1 * dy1;
    o[2] = R1 * dz1;
    double ox1, oy1, oz1;
    if (fabs(dx1) > 1e-10 || fabs(dy1) > 1e-10) {
        ox1 = -dy1; oy1 = dx1; oz1 = 0.0;
    } else {
        ox1 = 0.0; oy1 = -dz1; oz1 = dy1;
    }
    const double nrm = sqrt(ox1 * ox1 + oy1 * oy1 + oz1 * oz1);
    ox1 /= nrm; oy1 /= nrm; oz1 /= nrm;
    const double ox2 = dy1 * oz1 - dz1 * oy1, oy2 = dz1 * ox1 - dx1 * oz1, oz2 = dx1 * oy1 - dy1 * ox1;
    double sa, ca;
    sincos(al, &sa, &ca);
    double st2 = 1.0 - mu * mu;
    if (st2 < 0.0) st2 = 0.0;
    const double st = sqrt(st2);
    o[3] = R2 * (mu * dx1 + st * (ca * ox1 + sa * ox2));
    o[4] = R2 * (mu * dy1 + st * (ca * oy1 + sa * oy2));
    o[5] = R2 * (mu * dz1 + st * (ca * oz1 + sa * oz2));
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

constexpr int MC_THREADS = 256;

// The two edge vectors of every rotation (they depend on nothing else).
__global__ void k_triplet_offsets(double R1, double R2, double mu, const double* __restrict__ abc, int n_rot,
                                  double* __restrict__ off) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n_rot) return;
    double o[6];
    triangle_offsets(R1, R2, mu, TWO_PI * abc[3 * r], 2.0 * abc[3 * r + 1] - 1.0, TWO_PI * abc[3 * r + 2], o);
    for (int i = 0; i < 6; ++i) off[6 * r + i] = o[i];
}

// blockIdx.y: rotation (strided); blockIdx.x: centres (strided); per-block partial sums.  Bound by random lines of
// the grids and the latency of their loads.  SPHI: the scaling function in LDS, for its usual 1024 samples to a cell;
// tables of another resolution are read where they are (plain layout only).
template <int LAYOUT, bool SPHI = true>
__global__ __launch_bounds__(MC_THREADS, 4) void k_triplet_box(const double* __restrict__ spos,
                                                               const double* __restrict__ n1, int64_t n, int n_rot,
                                                               const double* __restrict__ off,
                                                               const double* __restrict__ g2,
                                                               const double* __restrict__ g3,
                                                               const double* __restrict__ phi, int lg, int res,
                                                               double* __restrict__ partial) {
    static_assert(SPHI || LAYOUT == GRID_PLAIN, "a table in global memory goes with the plain layout");
    __shared__ double sphi[SPHI ? 3 * 1024 : 1];
    __shared__ double sh[MC_THREADS / 64];
    if constexpr (SPHI) {
        load_phi<MC_THREADS>(sphi, phi, threadIdx.x);
        __syncthreads();
    }
    auto value = [&](const double* g, double x, double y, double z) {
        if constexpr (SPHI) return interp<LAYOUT>(g, sphi, lg, res, x, y, z);
        else return interp_at<GRID_PLAIN, false>(g, phi, lg, res, x, y, z);
    };
    double s = 0.0;
    for (int r = blockIdx.y; r < n_rot; r += gridDim.y) {
        const double* o = off + 6 * r;
        // whole waves (the lanes of a bricked interpolation work together): lanes past the end repeat the last centre
        for (int64_t q = blockIdx.x * (int64_t)MC_THREADS + (threadIdx.x & ~63); q < n;
             q += (int64_t)gridDim.x * MC_THREADS) {
            const int64_t mine = q + (threadIdx.x & 63), p = mine < n ? mine : n - 1;
            const double x = spos[3 * p], y = spos[3 * p + 1], z = spos[3 * p + 2];
            const double v2 = value(g2, x + o[0], y + o[1], z + o[2]);
            const double v3 = value(g3, x + o[3], y + o[4], z + o[5]);
            if (mine < n) s += n1[p] * v2 * v3;
        }
    }
    s = wave_sum(s);
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < MC_THREADS / 64; ++w) t += sh[w];
        partial[blockIdx.y * gridDim.x + blockIdx.x] = t;
    }
}

// ---------------------------------------------------------------- Philox4x32-10
struct u4 {
    uint32_t x, y, z, w;
};

__device__ __forceinline__ u4 philox(uint64_t counter, uint64_t key) {
    uint32_t c0 = (uint32_t)counter, c1 = (uint32_t)(counter >> 32), c2 = 0x9E3779B9u, c3 = 0x85EBCA6Bu;
    uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t h0 = (uint32_t)(p0 >> 32), l0 = (uint32_t)p0, h1 = (uint32_t)(p1 >> 32), l1 = (uint32_t)p1;
        const uint32_t n0 = h1 ^ c1 ^ k0, n2 = h0 ^ c3 ^ k1;
        c0 = n0; c1 = l1; c2 = n2; c3 = l0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return {c0, c1, c2, c3};
}

__device__ __forceinline__ double u53(uint32_t a, uint32_t b) {
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

struct BinnedArgs {
    int L, lg, res, nr1, nr2, nmu;
    double rmin1, rmax1, rmin2, rmax2;  // grid units, uniform (linear) bins
    double cap;                          // |w f| above cap goes to the overflow list (main pass)
    double scale_wf, scale_wf2;          // fixed-point scales for sum(w f) and sum((w f)^2)
    int64_t n;                           // samples (pilot, main) or overflow entries (fix-up)
    uint64_t seed;
    int importance;
    double alpha;                        // defensive mixture weight of the uniform proposal
    int nbucket;
    int sub;                             // proposal sub-cells per cell and axis (1, 2, 4, 8)
    int anchors;                         // 1: the drawn point is the apex; 3: any vertex, balance-heuristic weight
    int record;                          // write per-sample features for the first n_record samples
    int64_t n_record;
    int64_t over_cap;                    // capacity of the overflow list
};

struct ProposalTables {
    const unsigned char* cell_bucket;
    const int* bucket_cells;
    const int64_t* bucket_off;
    const float* bucket_cdf;
    const double* bucket_density;
    const float* bin_cdf;
    const float* bin_pdf;
};

__device__ __forceinline__ int upper_bound_f(const float* __restrict__ cdf, int n, float u) {
    int lo = 0, hi = n;  // first index with cdf[i] > u
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (cdf[mid] > u) hi = mid;
        else lo = mid + 1;
    }
    return lo < n ? lo : n - 1;
}

// Two uniforms in [0, 1) from stream `stream` of sample i.
__device__ __forceinline__ void uniforms2(uint64_t i, uint64_t seed, uint64_t stream, double& a, double& b) {
    const u4 r = philox(i, seed ^ (0x9E3779B97F4A7C15ULL * (stream + 1)));
    a = u53(r.x, r.y);
    b = u53(r.z, r.w);
}

// Sub-cell of a point (cell units) on the periodic grid of side Ls = L * sub.
__device__ __forceinline__ int subcell_of(double x, double y, double z, int Ls, double sub) {
    const int m = Ls - 1;
    return ((((int)floor(x * sub)) & m) * Ls + (((int)floor(y * sub)) & m)) * Ls + (((int)floor(z * sub)) & m);
}

struct Sample {
    int bin;
    int k[3];  // proposal bucket of each vertex's sub-cell (-1 without tables)
    double wf, r1, r2, mu, f;
};

// Sample i: apex c, bin (r1, r2, mu), orientation; vertices c, c + o1, c + o2;
// f = n1 n2 n3.  Plain: apex uniform in the box, bin uniform.  Importance
// (defensive mixture): with probability alpha as plain, otherwise bucket
// k ~ bucket_cdf, a uniform sub-cell of that bucket, a uniform point p in it,
// bin ~ bin_cdf[k] and, with anchors = 3, a uniformly chosen vertex a placed at
// p (c = p - o_a); with anchors = 1 the apex is p.  Each anchor proposes
// q_a = p_uniform * R(k(v_a), b) with R(k, b) = bucket_density[k] * bin_pdf[k][b],
// so the weight is w = 1 / (alpha + (1 - alpha) * mean_a R(k(v_a), b)) over the
// vertices v_a of the drawn triangle (one anchor: the apex only).  The same i
// always gives the same sample, whichever pass evaluates it.
template <int LAYOUT>
__device__ __forceinline__ void draw_sample(const BinnedArgs& A, const double* __restrict__ g1,
                                            const double* __restrict__ g2, const double* __restrict__ g3,
                                            const double* sphi, const ProposalTables& T, int64_t i, Sample& S) {
    const int L = A.L;
    const int B = A.nr1 * A.nr2 * A.nmu;
    const int Ls = L * A.sub;
    const double sub = (double)A.sub;
    const double dr1 = (A.rmax1 - A.rmin1) / A.nr1, dr2 = (A.rmax2 - A.rmin2) / A.nr2, dmu = 2.0 / A.nmu;
    double ux, uy, uz, ubin, upick = 0.0, umix = 0.0, ubin2, w1, w2, w3, oph, oct, oal, uanc;
    uniforms2((uint64_t)i, A.seed, 0, ux, uy);
    uniforms2((uint64_t)i, A.seed, 1, uz, ubin);
    if (A.importance) uniforms2((uint64_t)i, A.seed, 2, upick, umix);
    uniforms2((uint64_t)i, A.seed, 3, ubin2, w1);
    uniforms2((uint64_t)i, A.seed, 4, w2, w3);
    uniforms2((uint64_t)i, A.seed, 5, oph, oct);
    uniforms2((uint64_t)i, A.seed, 6, oal, uanc);
    double px, py, pz;
    int bin, anchor = 0;
    if (!A.importance || umix < A.alpha) {
        px = ux * L;
        py = uy * L;
        pz = uz * L;
        bin = (int)(ubin * B);
        if (bin >= B) bin = B - 1;
    } else {
        const int k = upper_bound_f(T.bucket_cdf, A.nbucket, (float)ubin);
        const int64_t c0 = T.bucket_off[k], c1 = T.bucket_off[k + 1];
        int64_t pick = c0 + (int64_t)(upick * (double)(c1 - c0));
        if (pick >= c1) pick = c1 - 1;
        // well-formed tables never select an empty bucket; keep malformed ones in bounds
        const int64_t ncell = (int64_t)Ls * Ls * Ls;
        pick = pick < 0 ? 0 : (pick >= ncell ? ncell - 1 : pick);
        int64_t sc = T.bucket_cells[pick];
        sc = sc < 0 ? 0 : (sc >= ncell ? ncell - 1 : sc);
        const int zs = (int)(sc % Ls), ys = (int)((sc / Ls) % Ls), xs = (int)(sc / ((int64_t)Ls * Ls));
        px = (xs + ux) / sub;
        py = (ys + uy) / sub;
        pz = (zs + uz) / sub;
        bin = upper_bound_f(T.bin_cdf + (int64_t)k * B, B, (float)ubin2);
        if (A.anchors == 3) anchor = min((int)(uanc * 3.0), 2);
    }
    const int imu = bin % A.nmu, ir2 = (bin / A.nmu) % A.nr2, ir1 = bin / (A.nmu * A.nr2);
    const double r1 = A.rmin1 + (ir1 + w1) * dr1, r2 = A.rmin2 + (ir2 + w2) * dr2;
    const double mu = -1.0 + (imu + w3) * dmu;
    double o[6];
    triangle_offsets(r1, r2, mu, TWO_PI * oph, 2.0 * oct - 1.0, TWO_PI * oal, o);
    double cx = px, cy = py, cz = pz;
    if (anchor == 1) {
        cx = px - o[0];
        cy = py - o[1];
        cz = pz - o[2];
    } else if (anchor == 2) {
        cx = px - o[3];
        cy = py - o[4];
        cz = pz - o[5];
    }
    // one vertex at a time, so that the registers allow several waves per SIMD
    double f = 1.0;
#pragma unroll 1
    for (int v = 0; v < 3; ++v) {
        const double* g = v == 0 ? g1 : (v == 1 ? g2 : g3);
        const double x = v == 0 ? cx : (v == 1 ? cx + o[0] : cx + o[3]);
        const double y = v == 0 ? cy : (v == 1 ? cy + o[1] : cy + o[4]);
        const double z = v == 0 ? cz : (v == 1 ? cz + o[2] : cz + o[5]);
        f *= interp<LAYOUT>(g, sphi, A.lg, A.res, x, y, z);
    }
    double w = 1.0;
    S.k[0] = S.k[1] = S.k[2] = -1;
    if (T.cell_bucket) {
        S.k[0] = min((int)T.cell_bucket[subcell_of(cx, cy, cz, Ls, sub)], A.nbucket - 1);
        S.k[1] = min((int)T.cell_bucket[subcell_of(cx + o[0], cy + o[1], cz + o[2], Ls, sub)], A.nbucket - 1);
        S.k[2] = min((int)T.cell_bucket[subcell_of(cx + o[3], cy + o[4], cz + o[5], Ls, sub)], A.nbucket - 1);
        if (A.importance) {
            double rel = T.bucket_density[S.k[0]] * (double)T.bin_pdf[(int64_t)S.k[0] * B + bin];
            if (A.anchors == 3) {
                rel += T.bucket_density[S.k[1]] * (double)T.bin_pdf[(int64_t)S.k[1] * B + bin];
                rel += T.bucket_density[S.k[2]] * (double)T.bin_pdf[(int64_t)S.k[2] * B + bin];
                rel *= (1.0 / 3.0);
            }
            w = 1.0 / (A.alpha + (1.0 - A.alpha) * rel);
        }
    }
    S.bin = bin;
    S.wf = w * f;
    S.r1 = r1;
    S.r2 = r2;
    S.mu = mu;
    S.f = f;
}

enum McPass { MC_PILOT = 0, MC_MAIN = 1, MC_FIXUP = 2 };

// PASS = MC_PILOT: only max |w f| over samples [0, A.n).
// PASS = MC_MAIN: samples [0, A.n): counts; w f and (w f)^2 into acc at scale
//   (cap) when |w f| <= cap, else the sample index goes to the overflow list.
// PASS = MC_FIXUP: the A.n listed samples into acc_hi at scale (max |w f|).
// Every pass folds max |w f| (inf for a non-finite value) into stats[0] as the
// bit pattern of a non-negative double, whose integer order is the numeric order;
// stats[1] counts overflow samples.  Fixed-point sums make the result
// independent of the order of the atomics.
// Bound by the random lines of the grids (see GridLayout).  2e7 uniform triangles at L = 256, the main pass alone:
// 10.4 ms with one lane per triangle and 27 loads per vertex, 7.0 ms with bricks.
template <int PASS, int LAYOUT>
__global__ __launch_bounds__(MC_THREADS, 4) void k_mc_binned(
    const double* __restrict__ g1, const double* __restrict__ g2, const double* __restrict__ g3,
    const double* __restrict__ phi, BinnedArgs A, ProposalTables T, const int64_t* __restrict__ fix_list,
    unsigned long long* __restrict__ acc, unsigned long long* __restrict__ acc_hi,
    unsigned long long* __restrict__ stats, int64_t* __restrict__ over_list, float* __restrict__ rec) {
    __shared__ double red[MC_THREADS / 64];
    __shared__ double sphi[3 * 1024];
    load_phi<MC_THREADS>(sphi, phi, threadIdx.x);
    __syncthreads();
    const int B = A.nr1 * A.nr2 * A.nmu;
    double mx = 0.0;
    // whole waves (the lanes of a bricked interpolation work together): lanes past the end repeat the last sample
    for (int64_t q = blockIdx.x * (int64_t)MC_THREADS + (threadIdx.x & ~63); q < A.n;
         q += (int64_t)gridDim.x * MC_THREADS) {
        const bool mine = q + (threadIdx.x & 63) < A.n;
        const int64_t t = mine ? q + (threadIdx.x & 63) : A.n - 1;
        const int64_t i = PASS == MC_FIXUP ? fix_list[t] : t;
        Sample S;
        draw_sample<LAYOUT>(A, g1, g2, g3, sphi, T, i, S);
        if (!mine) continue;
        const double a = fabs(S.wf);
        mx = (a == a) ? fmax(mx, a) : INFINITY;
        if (PASS == MC_FIXUP) {
            atomicAdd(&acc_hi[S.bin], (unsigned long long)__double2ll_rn(S.wf * A.scale_wf));
            atomicAdd(&acc_hi[B + S.bin], (unsigned long long)__double2ll_rn(S.wf * S.wf * A.scale_wf2));
        } else if (PASS == MC_MAIN) {
            atomicAdd(&acc[2 * B + S.bin], 1ull);
            if (a <= A.cap) {
                atomicAdd(&acc[S.bin], (unsigned long long)__double2ll_rn(S.wf * A.scale_wf));
                atomicAdd(&acc[B + S.bin], (unsigned long long)__double2ll_rn(S.wf * S.wf * A.scale_wf2));
            } else {
                const unsigned long long slot = atomicAdd(&stats[1], 1ull);
                if ((int64_t)slot < A.over_cap) over_list[slot] = i;
            }
            if (A.record && i < A.n_record) {
                float* rr = rec + 8 * i;
                rr[0] = (float)S.r1;
                rr[1] = (float)S.r2;
                rr[2] = (float)S.mu;
                rr[3] = (float)S.f;
                rr[4] = (float)S.bin;
                rr[5] = (float)S.k[0];
                rr[6] = (float)S.k[1];
                rr[7] = (float)S.k[2];
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int w = 1; w < MC_THREADS / 64; ++w) m = fmax(m, red[w]);
        if (m > 0.0) atomicMax(&stats[0], (unsigned long long)__double_as_longlong(m));
    }
}

// ---------------------------------------------------------------- proposal buckets
// The proposal's sub-cell grid (side Ls = L * sub): each sub-cell's bucket is
// the number of edges <= the interpolated field at its centre; bucket_cells
// lists the sub-cells bucket by bucket, ascending within a bucket (a stable,
// deterministic counting sort).  A block owns BK_CHUNK consecutive sub-cells.
constexpr int BK_THREADS = 256;
constexpr int BK_PER_THREAD = 64;
constexpr int BK_CHUNK = BK_THREADS * BK_PER_THREAD;

__global__ __launch_bounds__(BK_THREADS) void k_bucket_assign(const double* __restrict__ g,
                                                              const double* __restrict__ phi, int lg, int res,
                                                              int sub, const double* __restrict__ edges,
                                                              int nbucket, int64_t ncell,
                                                              unsigned char* __restrict__ cell_bucket,
                                                              int* __restrict__ hist) {
    __shared__ int h[256];
    for (int k = threadIdx.x; k < 256; k += BK_THREADS) h[k] = 0;
    __syncthreads();
    const int64_t Ls = (int64_t)sub << lg;
    const double inv = 1.0 / sub;
    const int64_t base = (int64_t)blockIdx.x * BK_CHUNK;
    for (int j = 0; j < BK_PER_THREAD; ++j) {
        const int64_t i = base + (int64_t)j * BK_THREADS + threadIdx.x;
        if (i < ncell) {
            const int64_t zs = i % Ls, ys = (i / Ls) % Ls, xs = i / (Ls * Ls);
            const double v = interp_at<GRID_PLAIN, false>(g, phi, lg, res, (xs + 0.5) * inv, (ys + 0.5) * inv,
                                                          (zs + 0.5) * inv);
            int lo = 0, hi = nbucket - 1;  // first edge > v
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (edges[mid] > v) hi = mid;
                else lo = mid + 1;
            }
            cell_bucket[i] = (unsigned char)lo;
            atomicAdd(&h[lo], 1);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < nbucket; k += BK_THREADS) hist[(int64_t)k * gridDim.x + blockIdx.x] = h[k];
}

// One block per bucket: exclusive prefix over blocks of hist[k][*] in place; total -> tot[k].
__global__ __launch_bounds__(1024) void k_bucket_scan(int* __restrict__ hist, int nblocks,
                                                      int64_t* __restrict__ tot) {
    __shared__ int64_t wsum[16];
    int* row = hist + (int64_t)blockIdx.x * nblocks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int64_t carry = 0;
    for (int base = 0; base < nblocks; base += 1024) {
        const int i = base + threadIdx.x;
        const int64_t v = i < nblocks ? row[i] : 0;
        int64_t x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[wave] = x;
        __syncthreads();
        int64_t pre = 0, all = 0;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) pre += wsum[w];
            all += wsum[w];
        }
        if (i < nblocks) row[i] = (int)(carry + pre + x - v);
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

// Thread t of block b owns sub-cells [b*CHUNK + 64 t, +64).  For each bucket in
// turn the block ranks its matches (per-thread popcount, block exclusive scan)
// and writes their indices in ascending order.  ncell is a multiple of 64.
__global__ __launch_bounds__(BK_THREADS) void k_bucket_scatter(const unsigned char* __restrict__ cell_bucket,
                                                               int64_t ncell, int nbucket,
                                                               const int* __restrict__ offs,
                                                               const int64_t* __restrict__ bucket_off,
                                                               int* __restrict__ bucket_cells) {
    __shared__ int wtot[BK_THREADS / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t base = (int64_t)blockIdx.x * BK_CHUNK + (int64_t)threadIdx.x * BK_PER_THREAD;
    const bool valid = base < ncell;
    uint32_t wv[16];
    if (valid) {
        const uint4* p = (const uint4*)(cell_bucket + base);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint4 t = p[q];
            wv[4 * q] = t.x;
            wv[4 * q + 1] = t.y;
            wv[4 * q + 2] = t.z;
            wv[4 * q + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 16; ++q) wv[q] = 0;
    }
    for (int k = 0; k < nbucket; ++k) {
        const uint32_t kk = 0x01010101u * (uint32_t)k;
        uint32_t m[16];
        int cnt = 0;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const uint32_t x = wv[q] ^ kk;  // zero byte <=> match
            uint32_t t = (x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu;
            t = ~(t | x | 0x7F7F7F7Fu);    // bit 7 of each zero byte
            m[q] = valid ? t : 0u;
            cnt += __popc(m[q]);
        }
        int x = cnt;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) wtot[wave] = x;
        __syncthreads();
        int pre = x - cnt;
        for (int w = 0; w < wave; ++w) pre += wtot[w];
        __syncthreads();
        if (cnt) {
            int64_t dst = bucket_off[k] + offs[(int64_t)k * gridDim.x + blockIdx.x] + pre;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                uint32_t t = m[q];
                while (t) {
                    const int byte = (__ffs(t) - 1) >> 3;
                    bucket_cells[dst++] = (int)(base + 4 * q + byte);
                    t &= t - 1;
                }
            }
        }
    }
}

}  // namespace

// Whether `items` lanes' work fills the rounds of waves that `waves` per SIMD give, the last one to a share of
// `least`.  A wave on bricks walks eight rounds of lines a vertex, and a round of waves that is nearly empty costs as
// much as a full one; a point per lane loses less there.
static bool rounds_filled(hermes_ctx* ctx, double items, int waves, double least) {
    const double rounds = items / (256.0 * waves * ctx->n_cu);
    return rounds >= 3.0 || rounds >= least * std::ceil(rounds);
}

// Layout for `points` interpolations on the n_grid grids g (replaced by their bricked copies where they are made).
// filled: by rounds_filled (2e5, 3e5 and 1e6 triangles at L = 128: 318, 369 and 974 us by a point per lane, 301, 441
// and 832 with bricks).  A copy reads and writes the grid once, which pays from about one point per 14 cells on while
// source and copy stay near the last-level cache (L = 256, 2.5e5 and 4e5 triangles: 407 and 603 us plain, 378 and 547
// bricked), one per 8 up to 512 MiB of copies and one per 5 beyond (L = 512, 6e6: 4.8 ms plain, 5.1 bricked; 1e7: 7.4
// and 7.2).  Below L = 128 the grid stays in the L2 caches and a point per lane is the faster way (whole calls of 2e7
// uniform triangles: L = 64 3.8 ms, with bricks 4.4; L = 128 8.8 and 7.2; L = 256 11.8 and 7.6).  The copies are kept
// within 4 GiB.  Grids not aligned to 16 bytes are bricked under the same rule or read by 8 bytes.
static int grid_layout(hermes_ctx* ctx, int J, double points, bool filled, const double** g, int n_grid) {
    const size_t n = (size_t)1 << (3 * J);
    bool aligned = true;
    for (int i = 0; i < n_grid; ++i) aligned = aligned && ((uintptr_t)g[i] & 15) == 0;
    const int plain = aligned ? GRID_ALIGNED : GRID_PLAIN;
    int copies = 0, of[3];
    const double* distinct[3];
    for (int i = 0; i < n_grid; ++i) {
        int k = 0;
        while (k < copies && distinct[k] != g[i]) ++k;
        if (k == copies) distinct[copies++] = g[i];
        of[i] = k;
    }
    const double cells = (double)n * copies;
    const double per = cells <= 0x1p24 ? 14.0 : (cells <= 0x1p26 ? 8.0 : 5.0);
    if (J < 7 || !filled || points * per < cells || cells * sizeof(double) > 0x1p32) return plain;
    double* ws = (double*)hermes_workspace(ctx, WS_SPEC, copies * n * sizeof(double));
    if (!ws) return plain;
    for (int k = 0; k < copies; ++k)
        k_brick<<<hermes_blocks((int64_t)n, 256, 16384), 256, 0, ctx->stream>>>(distinct[k], J, ws + k * n);
    for (int i = 0; i < n_grid; ++i) g[i] = ws + of[i] * n;
    return GRID_BRICK;
}

extern "C" {

int hermes_interpolate(hermes_ctx* ctx, int J, const double* grid, const double* spos, int64_t n, const double* phi,
                       int phi_res, double dx, double dy, double dz, double* out) {
    HERMES_REQUIRE(ctx && grid && phi && (n == 0 || (spos && out)), "hermes_interpolate: null argument");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(phi_res == 1024, "phi_res must be 1024");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    if (n == 0) return 0;
    k_interpolate<<<hermes_blocks(n, 256, 65536), 256, 0, ctx->stream>>>(grid, spos, n, phi, J, phi_res, dx, dy,
                                                                         dz, out);
    HERMES_LAUNCH_CHECK();
    return 0;
}

int hermes_mc_triplet_box(hermes_ctx* ctx, int J, double R1, double R2, double mu, const double* spos,
                          const double* n1, int64_t n, int n_rot, const double* abc_host, const double* g2,
                          const double* g3, const double* phi, int phi_res, double* out_host) {
    HERMES_REQUIRE(ctx && spos && n1 && abc_host && g2 && g3 && phi && out_host, "hermes_mc_triplet_box: null arg");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(n > 0 && n_rot > 0, "need centres and rotations");
    HERMES_REQUIRE(phi_res >= 1, "phi_res must be positive");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    // about 2048 workgroups: the centres by the rotations
    const int nbx = (int)hermes_blocks(n, MC_THREADS, 2048);
    const int nby = (int)std::min<int64_t>(n_rot, std::max(1, 2048 / nbx));
    const int nb = nbx * nby;
    double* ws = (double*)hermes_workspace(ctx, WS_MC, sizeof(double) * ((size_t)nb + 8 + 9 * (size_t)n_rot));
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    double *d_abc = ws + nb + 8, *d_off = d_abc + 3 * (size_t)n_rot;
    HERMES_CHECK_HIP(hipMemcpyAsync(d_abc, abc_host, sizeof(double) * 3 * n_rot, hipMemcpyHostToDevice, ctx->stream));
    k_triplet_offsets<<<hermes_blocks(n_rot, 64), 64, 0, ctx->stream>>>(R1, R2, mu, d_abc, n_rot, d_off);
    HERMES_LAUNCH_CHECK();
    const double* g[2] = {g2, g3};
    const double items = (double)n * n_rot;
    // the LDS table and the packed fractions of the faster layouts hold 1024 samples to a cell
    const bool filled = rounds_filled(ctx, items, 6, 0.55);
    const int layout = phi_res == 1024 ? grid_layout(ctx, J, 2.0 * items, filled, g, 2) : -1;
    auto go = [&](auto kernel) {
        kernel<<<dim3(nbx, nby), MC_THREADS, 0, ctx->stream>>>(spos, n1, n, n_rot, d_off, g[0], g[1], phi, J, phi_res,
                                                               ws);
    };
    if (layout == GRID_BRICK) go(k_triplet_box<GRID_BRICK>);
    else if (layout == GRID_ALIGNED) go(k_triplet_box<GRID_ALIGNED>);
    else if (layout == GRID_PLAIN) go(k_triplet_box<GRID_PLAIN>);
    else go(k_triplet_box<GRID_PLAIN, false>);
    HERMES_LAUNCH_CHECK();
    HERMES_CHECK_HIP(hermes_reduce::sum_columns(ctx->stream, ws, 1, nb, 1, nullptr, ws + nb));
    double s = 0.0;
    HERMES_CHECK_HIP(hipMemcpyAsync(&s, ws + nb, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    *out_host = s / ((double)n_rot * (double)n);
    return 0;
}

int hermes_mc_binned(hermes_ctx* ctx, int J, const double* g1, const double* g2, const double* g3, const double* phi,
                     int phi_res, int nr1, int nr2, int nmu, double rmin1, double rmax1, double rmin2, double rmax2,
                     int64_t n_samples, uint64_t seed, double wf_cap, const hermes_mc_proposal* prop, float* record,
                     int64_t n_record, double* sum_wf_host, double* sum_wf2_host, int64_t* count_host) {
    HERMES_REQUIRE(ctx && g1 && g2 && g3 && phi && sum_wf_host && sum_wf2_host && count_host,
                   "hermes_mc_binned: null argument");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(phi_res == 1024, "phi_res must be 1024");
    HERMES_REQUIRE(nr1 >= 1 && nr2 >= 1 && nmu >= 1 && (int64_t)nr1 * nr2 * nmu <= (1 << 20), "invalid binning");
    HERMES_REQUIRE(rmax1 > rmin1 && rmax2 > rmin2 && rmin1 >= 0.0 && rmin2 >= 0.0, "invalid radial ranges");
    HERMES_REQUIRE(n_samples >= 1 && wf_cap >= 0.0, "n_samples must be positive and wf_cap non-negative");
    HERMES_REQUIRE(record == nullptr || n_record >= 0, "invalid record count");
    if (prop) {
        HERMES_REQUIRE(prop->cell_bucket && prop->bucket_cells && prop->bucket_off && prop->bucket_cdf &&
                           prop->bucket_density && prop->bin_cdf && prop->bin_pdf,
                       "hermes_mc_binned: incomplete proposal tables");
        HERMES_REQUIRE(prop->nbucket >= 1 && prop->nbucket <= 256, "nbucket must be in 1..256");
        HERMES_REQUIRE(prop->alpha > 0.0 && prop->alpha <= 1.0, "alpha must be in (0, 1]");
        HERMES_REQUIRE(prop->sub == 1 || prop->sub == 2 || prop->sub == 4 || prop->sub == 8,
                       "sub must be 1, 2, 4 or 8");
        HERMES_REQUIRE((1 << J) * prop->sub <= 1024, "L * sub must not exceed 1024");
        HERMES_REQUIRE(prop->anchors == 1 || prop->anchors == 3, "anchors must be 1 or 3");
    }
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int B = nr1 * nr2 * nmu;
    constexpr int64_t OVER_CAP = 1 << 20;
    constexpr int64_t PILOT = 1 << 20;
    BinnedArgs A;
    A.L = 1 << J;
    A.lg = J;
    A.res = phi_res;
    A.nr1 = nr1;
    A.nr2 = nr2;
    A.nmu = nmu;
    A.rmin1 = rmin1;
    A.rmax1 = rmax1;
    A.rmin2 = rmin2;
    A.rmax2 = rmax2;
    A.seed = seed;
    A.importance = prop != nullptr;
    A.alpha = prop ? prop->alpha : 1.0;
    A.nbucket = prop ? prop->nbucket : 0;
    A.sub = prop ? prop->sub : 1;
    A.anchors = prop ? prop->anchors : 1;
    A.record = record != nullptr;
    A.n_record = record ? n_record : 0;
    A.over_cap = OVER_CAP;
    ProposalTables T{};
    if (prop)
        T = {prop->cell_bucket, prop->bucket_cells, prop->bucket_off, prop->bucket_cdf, prop->bucket_density,
             prop->bin_cdf, prop->bin_pdf};
    // workspace: acc (3B: sum wf, sum wf^2, count) | acc_hi (2B) | stats (2) | overflow list
    const size_t n_acc = 5 * (size_t)B + 2;
    char* ws = (char*)hermes_workspace(ctx, WS_MC, sizeof(unsigned long long) * n_acc + sizeof(int64_t) * OVER_CAP);
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    unsigned long long* acc = (unsigned long long*)ws;
    unsigned long long* acc_hi = acc + 3 * (size_t)B;
    unsigned long long* stats = acc_hi + 2 * (size_t)B;
    int64_t* over_list = (int64_t*)(ws + sizeof(unsigned long long) * n_acc);
    const double* g[3] = {g1, g2, g3};
    const double all = (double)n_samples, pilot = wf_cap > 0.0 ? 0.0 : (double)std::min(n_samples, PILOT);
    const int layout = grid_layout(ctx, J, 3.0 * (all + pilot), rounds_filled(ctx, all, 4, 0.67), g, 3);
    // workgroups load the scaling function once and loop over samples
    auto launch = [&](auto brick, auto aligned, auto plain, const BinnedArgs& args, const int64_t* list, float* out) {
        auto kernel = layout == GRID_BRICK ? brick : (layout == GRID_ALIGNED ? aligned : plain);
        kernel<<<hermes_blocks(args.n, MC_THREADS, 2048), MC_THREADS, 0, ctx->stream>>>(
            g[0], g[1], g[2], phi, args, T, list, acc, acc_hi, stats, over_list, out);
    };
    unsigned long long st[2];
    auto read_stats = [&]() -> int {
        HERMES_CHECK_HIP(hipMemcpyAsync(st, stats, sizeof(st), hipMemcpyDeviceToHost, ctx->stream));
        HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
        return 0;
    };
    auto max_of = [&]() { return __builtin_bit_cast(double, st[0]); };

    // The fixed-point scale comes from a cap on |w f|: given by the caller, or the
    // maximum over the first PILOT samples (the main pass draws the same ones).
    double cap = wf_cap;
    if (!(cap > 0.0)) {
        HERMES_CHECK_HIP(hipMemsetAsync(stats, 0, 2 * sizeof(unsigned long long), ctx->stream));
        A.n = n_samples < PILOT ? n_samples : PILOT;
        launch(k_mc_binned<MC_PILOT, GRID_BRICK>, k_mc_binned<MC_PILOT, GRID_ALIGNED>,
               k_mc_binned<MC_PILOT, GRID_PLAIN>, A, nullptr, nullptr);
        HERMES_LAUNCH_CHECK();
        if (read_stats()) return 1;
        cap = max_of();
        HERMES_REQUIRE(std::isfinite(cap), "hermes_mc_binned: non-finite triangle weight");
        if (!(cap > 0.0)) cap = 1.0;
    }
    for (int attempt = 0;; ++attempt) {
        HERMES_CHECK_HIP(hipMemsetAsync(acc, 0, sizeof(unsigned long long) * n_acc, ctx->stream));
        A.n = n_samples;
        A.cap = cap;
        // |w f| <= cap for every accumulated sample: each bin sum stays below 2^62
        A.scale_wf = ldexp(1.0, 62) / ((double)n_samples * cap);
        A.scale_wf2 = ldexp(1.0, 62) / ((double)n_samples * cap * cap);
        launch(k_mc_binned<MC_MAIN, GRID_BRICK>, k_mc_binned<MC_MAIN, GRID_ALIGNED>,
               k_mc_binned<MC_MAIN, GRID_PLAIN>, A, nullptr, record);
        HERMES_LAUNCH_CHECK();
        if (read_stats()) return 1;
        if (st[1] == 0) break;
        HERMES_REQUIRE(std::isfinite(max_of()), "hermes_mc_binned: non-finite triangle weight");
        if ((int64_t)st[1] <= OVER_CAP) break;
        // too many samples above the cap for the list: redo with the exact maximum
        HERMES_REQUIRE(attempt == 0, "hermes_mc_binned: overflow list exceeded twice");
        cap = max_of();
    }
    const int64_t n_over = (int64_t)st[1];
    double scale_hi = 0.0, scale_hi2 = 0.0;
    if (n_over > 0) {
        const double mx = max_of();
        BinnedArgs F = A;
        F.n = n_over;
        F.record = 0;
        F.scale_wf = scale_hi = ldexp(1.0, 62) / ((double)n_over * mx);
        F.scale_wf2 = scale_hi2 = ldexp(1.0, 62) / ((double)n_over * mx * mx);
        launch(k_mc_binned<MC_FIXUP, GRID_BRICK>, k_mc_binned<MC_FIXUP, GRID_ALIGNED>,
               k_mc_binned<MC_FIXUP, GRID_PLAIN>, F, over_list, nullptr);
        HERMES_LAUNCH_CHECK();
    }
    std::vector<long long> h(5 * (size_t)B);
    HERMES_CHECK_HIP(hipMemcpyAsync(h.data(), acc, sizeof(long long) * 5 * (size_t)B, hipMemcpyDeviceToHost,
                                    ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    for (int b = 0; b < B; ++b) {
        sum_wf_host[b] = (double)h[b] / A.scale_wf;
        sum_wf2_host[b] = (double)h[B + b] / A.scale_wf2;
        if (n_over > 0) {
            sum_wf_host[b] += (double)h[3 * (size_t)B + b] / scale_hi;
            sum_wf2_host[b] += (double)h[4 * (size_t)B + b] / scale_hi2;
        }
        count_host[b] = h[2 * B + b];
    }
    return 0;
}

int hermes_mc_bucketize(hermes_ctx* ctx, int J, const double* grid, const double* phi, int phi_res, int sub,
                        const double* edges_host, int nbucket, uint8_t* cell_bucket, int32_t* bucket_cells,
                        int64_t* bucket_off, int64_t* counts_host) {
    HERMES_REQUIRE(ctx && grid && phi && cell_bucket && bucket_cells && bucket_off && counts_host,
                   "hermes_mc_bucketize: null argument");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    HERMES_REQUIRE(phi_res == 1024, "phi_res must be 1024");
    HERMES_REQUIRE(sub == 1 || sub == 2 || sub == 4 || sub == 8, "sub must be 1, 2, 4 or 8");
    HERMES_REQUIRE((1 << J) * sub <= 1024, "L * sub must not exceed 1024");
    HERMES_REQUIRE(nbucket >= 1 && nbucket <= 256, "nbucket must be in 1..256");
    HERMES_REQUIRE(nbucket == 1 || edges_host, "hermes_mc_bucketize: edges missing");
    for (int k = 1; k + 1 < nbucket; ++k)
        HERMES_REQUIRE(edges_host[k] >= edges_host[k - 1], "edges must be ascending");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int64_t Ls = (int64_t)(1 << J) * sub;
    const int64_t ncell = Ls * Ls * Ls;  // a multiple of 64 since Ls >= 4
    const int nblocks = (int)((ncell + BK_CHUNK - 1) / BK_CHUNK);
    const size_t hist_bytes = sizeof(int) * (size_t)nbucket * nblocks;
    char* ws = (char*)hermes_workspace(ctx, WS_MC, hist_bytes + sizeof(int64_t) * 256 + sizeof(double) * 256);
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    int* hist = (int*)ws;
    int64_t* tot = (int64_t*)(ws + hist_bytes);
    double* edges = (double*)(ws + hist_bytes + sizeof(int64_t) * 256);
    if (nbucket > 1)
        HERMES_CHECK_HIP(hipMemcpyAsync(edges, edges_host, sizeof(double) * (nbucket - 1), hipMemcpyHostToDevice,
                                        ctx->stream));
    k_bucket_assign<<<nblocks, BK_THREADS, 0, ctx->stream>>>(grid, phi, J, phi_res, sub, edges, nbucket, ncell,
                                                             cell_bucket, hist);
    HERMES_LAUNCH_CHECK();
    k_bucket_scan<<<nbucket, 1024, 0, ctx->stream>>>(hist, nblocks, tot);
    HERMES_LAUNCH_CHECK();
    std::vector<int64_t> t(nbucket), off(nbucket + 1);
    HERMES_CHECK_HIP(hipMemcpyAsync(t.data(), tot, sizeof(int64_t) * nbucket, hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    off[0] = 0;
    for (int k = 0; k < nbucket; ++k) {
        off[k + 1] = off[k] + t[k];
        counts_host[k] = t[k];
    }
    HERMES_REQUIRE(off[nbucket] == ncell, "hermes_mc_bucketize: bucket counts do not add up");
    HERMES_CHECK_HIP(hipMemcpyAsync(bucket_off, off.data(), sizeof(int64_t) * (nbucket + 1), hipMemcpyHostToDevice,
                                    ctx->stream));
    k_bucket_scatter<<<nblocks, BK_THREADS, 0, ctx->stream>>>(cell_bucket, ncell, nbucket, hist, bucket_off,
                                                              bucket_cells);
    HERMES_LAUNCH_CHECK();
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return 0;
}

}  // extern "C"
