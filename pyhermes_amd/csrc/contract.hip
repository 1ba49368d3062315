// Spherical-harmonic 3PCF triple-product contraction.
//
// Plain FP64 path (faithful to compute_3d_result_gpu + reduce_complex_sum_kernel,
// corr3pcf_multipoles.py:33-58, :99-131):
//   S = sum_x d1[x] sum_{l1} F1[x-l1] sum_{l2} G3(l1,l2) F2[x-l2]   (complex128)
// fused with a deterministic FP64 reduction.
//
// Batched FP32 path (MFMA): for up to 16 x 16 shells at once
//   G[s1][s2] = sum_x d1[x] sum_{l1,l2} G3(l1,l2) Re(U_s1[x-l1] W_s2[x-l2])
// as a 16 x 16 Gram matrix accumulated with v_mfma_f32_16x16x4f32 (lane = shell x cell); with
// Gamma = Q diag(lam) Q^T the y stencil is an eigen-filter on the fields, the x and z stencils sit on d1 (see
// k_gram_auto, k_gram_cross).  FP32 sums go to FP64 every few planes; per-workgroup FP64 partials are summed in
// fixed order.
#include "../../include/hermes_amd.h"
#include "hermes_common.h"
#include "reduce.h"

namespace {

__device__ __forceinline__ double wave_sum_d(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ---------------------------------------------------------------- plain FP64
// One thread owns a (y, z) column of an x segment and walks along x.  Per plane it forms once
//   V[ly][lz] = sum_{l2} G[ly][l2y] G[lz][l2z] F2(x, y - l2y, z - l2z)     (9 complex values)
// and keeps V of the last two planes.  With U[ly][lz] = F1(x, y - ly, z - lz), U.V the sum over the 9 taps and the
// x stencil moved onto d1 (c_t = sum_j d(x + j) G[j][j + t], e_t = sum_j d(x + j) G[j + t][j]) the plane x adds
//   U(x) . (c_0 V(x) + c_1 V(x-1) + c_2 V(x-2)) + (e_1 U(x-1) + e_2 U(x-2)) . V(x),
// about 340 FP64 multiply-adds per cell where the direct sum takes over 2000 and 729 loads.  A workgroup of 64 z by
// 4 y columns stages the planes of both fields with their halo in LDS, one plane ahead (four planes of F1, two of
// F2: 38 KB).  Bound by FP64 VALU with LDS reads of the same order.  L = 256: 7.61 ms for the direct sum, 0.69 ms
// with the taps loaded through L1, 0.46 ms now.
constexpr int SUM_THREADS = 256;
constexpr int SUM_TILE = 6 * 66;  // largest haloed tile (64 x 4 columns; smaller grids: 32 x 8, 16 x 16, ...)

struct Gamma3 {
    double g[9];  // row major
};

// In place: v[ly][lz] <- sum_{a, b} G[ly][a] G[lz][b] v[a][b].
__device__ __forceinline__ void summand_filter(const Gamma3& G, double2 v[9]) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const double2 a = v[3 * r], b = v[3 * r + 1], c = v[3 * r + 2];
#pragma unroll
        for (int l = 0; l < 3; ++l)
            v[3 * r + l] = make_double2(G.g[3 * l] * a.x + G.g[3 * l + 1] * b.x + G.g[3 * l + 2] * c.x,
                                        G.g[3 * l] * a.y + G.g[3 * l + 1] * b.y + G.g[3 * l + 2] * c.y);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const double2 a = v[q], b = v[3 + q], c = v[6 + q];
#pragma unroll
        for (int l = 0; l < 3; ++l)
            v[3 * l + q] = make_double2(G.g[3 * l] * a.x + G.g[3 * l + 1] * b.x + G.g[3 * l + 2] * c.x,
                                        G.g[3 * l] * a.y + G.g[3 * l + 1] * b.y + G.g[3 * l + 2] * c.y);
    }
}

__global__ __launch_bounds__(SUM_THREADS, 2) void k_summand_f64(int L, int tz, int ty, int xseg,
                                                                const double* __restrict__ d1,
                                                                const double2* __restrict__ F1,
                                                                const double2* __restrict__ F2, Gamma3 G,
                                                                double* __restrict__ partial) {
    __shared__ double2 uring[4][SUM_TILE], vring[2][SUM_TILE];
    __shared__ double sh[2][SUM_THREADS / 64];
    const int m = L - 1, tid = threadIdx.x;
    const int64_t LL = (int64_t)L * L;
    const int nzb = L / tz;
    const int z0 = (blockIdx.x % nzb) * tz, y0 = (blockIdx.x / nzb) * ty;
    const int x0 = blockIdx.y * xseg, xend = x0 + xseg;
    const int W = tz + 2, ntile = W * (ty + 2);
    const int lz = tid % tz, ly = tid / tz;
    const bool act = ly < ty;
    // this thread's staged elements (tile row r holds y0 - 2 + r, column c holds z0 - 2 + c)
    const bool st1 = tid + SUM_THREADS < ntile;
    int off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = tid + i * SUM_THREADS, r = e / W, c = e % W;
        off[i] = ((y0 - 2 + r) & m) * L + ((z0 - 2 + c) & m);
    }
    const bool st0 = tid < ntile;
    double2 pu[2], pv[2];
    auto load = [&](int x) {
        const int64_t o = (int64_t)(x & m) * LL;
        if (st0) {
            pu[0] = F1[o + off[0]];
            pv[0] = F2[o + off[0]];
        }
        if (st1) {
            pu[1] = F1[o + off[1]];
            pv[1] = F2[o + off[1]];
        }
    };
    auto store = [&](int x) {
        if (st0) {
            uring[x & 3][tid] = pu[0];
            vring[x & 1][tid] = pv[0];
        }
        if (st1) {
            uring[x & 3][tid + SUM_THREADS] = pu[1];
            vring[x & 1][tid + SUM_THREADS] = pv[1];
        }
    };
    const int t0 = (ly + 2) * W + lz + 2;  // tap (l, k) at t0 - l W - k
    const double* g = G.g;
    auto vplane = [&](int x, double2 v[9]) {
        if (!act) return;
#pragma unroll
        for (int t = 0; t < 9; ++t) v[t] = vring[x & 1][t0 - (t / 3) * W - t % 3];
        summand_filter(G, v);
    };
    double2 V0[9], V1[9], V2[9];
    double tr = 0.0, ti = 0.0;
    // x from x0 - 2 (ring slots of negative x: & works on two's complement)
    load(x0 - 2);
    store(x0 - 2);
    load(x0 - 1);
    __syncthreads();
    vplane(x0 - 2, V1);
    store(x0 - 1);
    load(x0);
    __syncthreads();
    vplane(x0 - 1, V2);
    store(x0);
    const int64_t yz = (int64_t)(y0 + ly) * L + z0 + lz;
    auto dat = [&](int x) { return act ? d1[(int64_t)(x & m) * LL + yz] : 0.0; };
    double d0 = dat(x0), da = dat(x0 + 1);
    // plane x into VC; V1x, V2x hold planes x - 1, x - 2
    auto step = [&](int x, double2 VC[9], double2 V1x[9], double2 V2x[9]) {
        __syncthreads();  // plane x is staged; the slots of plane x + 1 are no longer read
        load(x + 1);
        const double db = dat(x + 2);
        vplane(x, VC);
        if (act) {
            const double c0 = g[0] * d0 + g[4] * da + g[8] * db;
            const double c1 = g[1] * d0 + g[5] * da, c2 = g[2] * d0;  // U(x) with V(x - 1), V(x - 2)
            const double e1 = g[3] * d0 + g[7] * da, e2 = g[6] * d0;  // V(x) with U(x - 1), U(x - 2)
            const double2 *f0 = uring[x & 3], *f1 = uring[(x - 1) & 3], *f2 = uring[(x - 2) & 3];
#pragma unroll
            for (int t = 0; t < 9; ++t) {
                const int o = t0 - (t / 3) * W - t % 3;
                const double2 u0 = f0[o], u1 = f1[o], u2 = f2[o];
                const double wr = c0 * VC[t].x + c1 * V1x[t].x + c2 * V2x[t].x,
                             wi = c0 * VC[t].y + c1 * V1x[t].y + c2 * V2x[t].y;
                const double ur = e1 * u1.x + e2 * u2.x, ui = e1 * u1.y + e2 * u2.y;
                tr += u0.x * wr - u0.y * wi + (ur * VC[t].x - ui * VC[t].y);
                ti += u0.x * wi + u0.y * wr + (ur * VC[t].y + ui * VC[t].x);
            }
        }
        d0 = da;
        da = db;
        store(x + 1);
    };
    for (int x = x0; x < xend;) {
        step(x, V0, V2, V1);
        if (++x >= xend) break;
        step(x, V1, V0, V2);
        if (++x >= xend) break;
        step(x, V2, V1, V0);
        ++x;
    }
    tr = wave_sum_d(tr);
    ti = wave_sum_d(ti);
    if (threadIdx.x % 64 == 0) {
        sh[0][threadIdx.x / 64] = tr;
        sh[1][threadIdx.x / 64] = ti;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double t = 0.0;
        for (int w = 0; w < SUM_THREADS / 64; ++w) t += sh[threadIdx.x][w];
        partial[2 * (blockIdx.y * gridDim.x + blockIdx.x) + threadIdx.x] = t;
    }
}

// ---------------------------------------------------------------- batched FP32 MFMA Gram
struct GramArgs {
    int L, S1, S2, cross, xseg;
    int xs, ys;       // element strides of x and y in the fields U, V (x-major: L^2, L; y-major: L, L^2)
    float vsign;      // sign applied to V's imaginary part in the cross case (-1: Re(U V))
    float gx[9];      // Gamma[l1 * 3 + l2] = sum_a Q[l1][a] lam_a Q[l2][a]
    float Qs[9];      // Q[tap][col] sqrt|lam_col|, columns sorted by ascending lam
};

typedef float float4_t __attribute__((ext_vector_type(4)));

// Auto Gram with the z-direction Gamma stencil also moved onto d1 (the y stencil stays on the fields as
// the eigen-filter T_b(y) = sum_ly Qs[ly][b] F(y - ly), column b scaled by sqrt|lam_b|, sign s_b).  For the
// cells (p, r) of a column plane and delta = (dx, dz),
//   sum_{x, z} d(x, z) sum_{l1, l2} G[l1x][l2x] G[l1z][l2z] T^a(x - l1) T^b*(x - l2) = A[a][b] + A[b][a],
//   A = sum_{p, r} T^a(p, r) B^b(p, r),  B(p, r) = sum_{delta in H} w_delta C_delta(p, r) T*(p + dx, r + dz),
//   C_delta(p, r) = sum_{l1x} G[l1x][l1x - dx] E_dz(p + l1x, r),  E_dz(x', r) = sum_{l1z} G[l1z][l1z - dz] d(x', r + l1z),
// each sum over the taps that keep l1 - delta in 0 .. 2; H = {(0, 0) with weight 1/2, (0, 1), (0, 2),
// (1, -2 .. 2), (2, -2 .. 2)} (the pair delta, -delta gives the transposed term).  Per channel b one right
// operand B of 13 terms and one MFMA pair: 6 MFMAs per plane instead of 18, and no z filter.
//
// Each y-filtered plane q is read from LDS once (at z - 2 .. z + 2 of the lane's cell, step q - 2) and
// scattered into the right operands of the three planes it serves: B(q - 2) (dx = 2), B(q - 1) (dx = 1) and
// B(q) (dx = 0); B(q - 2) is then complete and meets its left operand T(q - 2, z), kept since it was read.
// C and E depend on the cell only; E of a plane is computed once and kept for three steps.
//
// LDS: y-filtered planes in 2 buffers (step p reads plane p+2 while plane p+3 is written), raw halo'd
// tiles in 2; the z halo is 2 on both sides.  Step p, after its one barrier: plane p+2 into the operands
// (and the MFMAs of plane p), y taps of plane p+3 from raw buffer (p+3)&1, store of staged plane p+4 into
// raw buffer (p+4)&1, load of plane p+5 into registers.  A workgroup of 8 waves owns 2 (y) x 16 (z) cells
// and 50 KB of LDS.
// Tile geometry with TY rows of TZ cells: a wave takes 4 cells along z.  The raw
// tile keeps 16 shells per (row, z) position, the shell slot XOR-swizzled by z & 15 so that both the
// z-fastest staging stores and the shell-fastest y-tap reads spread over the banks.
template <int TY, int TZ_>
struct D2Geom {
    static constexpr int NROW = TY, TZ = TZ_, WAVES = TY * TZ / 4;
    static constexpr int RY = TY + 2, RZ = TZ + 4;   // raw rows y0-2 .. y0+TY-1, z z0-2 .. z0+TZ+1
    static constexpr int RP = 16;
    static constexpr int TILE = RY * RZ * RP;        // float2 per raw buffer
    static constexpr int TB = TY * RZ * 16;          // float2 per channel of a T buffer
    static constexpr int TBUF = 3 * TB;              // float2 per T buffer: [b][row][z][shell]
    static constexpr int STAGE = RY * RZ * 16;       // elements staged per plane
    static constexpr int SPT = (STAGE + 64 * WAVES - 1) / (64 * WAVES);
    static constexpr int TPT = (TB + 64 * WAVES - 1) / (64 * WAVES);
    static_assert((2 * TILE + 2 * TBUF) * 8 >= WAVES * 256 * 8, "reduction reuses the tile buffers");
    // tiles, and the split variant's per-wave imaginary sums, in at most 80 KB: two workgroups per CU
    static_assert((2 * TILE + 2 * TBUF) * 8 + WAVES * 256 * 8 <= 80 * 1024, "LDS of two workgroups per CU");
};
// 2 rows per workgroup: 8 waves and at most 66 KB of LDS, so two workgroups and four waves per SIMD
using D2 = D2Geom<2, 16>;
// the cross kernel: 4 waves and 39 KB; its 160 registers allow three waves per SIMD, so three workgroups per CU
// (with 8 waves two per SIMD and one barrier for all: 540 us instead of 388 for 11 x 15 shells at L = 128; held to
// 128 registers it spills 32: 874 us)
using D2X = D2Geom<2, 8>;

template <int NNEG, bool SPLIT = false>
__global__ __launch_bounds__(64 * D2::WAVES, 4) void k_gram_auto(const float* __restrict__ d1,
                                                           const float2* __restrict__ U, GramArgs g,
                                                           double* __restrict__ partial) {
    using GM = D2;
    __shared__ __align__(16) float2 smem[2 * GM::TILE + 2 * GM::TBUF];
    __shared__ double redi[SPLIT ? GM::WAVES * 256 : 1];  // imaginary sums per wave (SPLIT: registers are full)
    auto raw = [&](int q) -> float2* { return smem + (q & 1) * GM::TILE; };
    auto tb = [&](int q) -> float2* { return smem + 2 * GM::TILE + (q & 1) * GM::TBUF; };
    const int L = g.L, m = L - 1;
    const int tid = threadIdx.x;
    const int lane = tid % 64, wave = tid / 64;
    const int s = lane % 16, k = lane / 16;
    const int zw = wave % 4, yw = wave / 4;
    // Workgroups are dealt to the 8 XCDs round-robin; the remap gives each XCD a contiguous range of
    // logical blocks (x segment slowest, then columns 8 tiles wide walked along y), so co-resident
    // workgroups share halo rows in the XCD's L2 (columns 1, 2, 4, 16, 32 tiles wide measured 14%, 8%, 1%,
    // 1% and 4% slower).
    const int nzb = L / GM::TZ, nyb = L / GM::NROW;
    const int nb = nzb * nyb * (L / g.xseg);
    const int q = (nb % 8 == 0) ? (int)(blockIdx.x % 8) * (nb / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int xs = q / (nzb * nyb);
    const int rr = q % (nzb * nyb);
    const int PZ = nzb < 8 ? nzb : 8;
    const int zb = (rr / (PZ * nyb)) * PZ + (rr % (PZ * nyb)) % PZ;
    const int yb = (rr % (PZ * nyb)) / PZ;
    const int z0 = zb * GM::TZ, y0 = yb * GM::NROW;
    const int x0 = xs * g.xseg, xend = x0 + g.xseg;
    const int64_t N = (int64_t)L * L * L;
    const int64_t LL = (int64_t)L * L;

    float Q[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) Q[i] = g.Qs[i];
    const float G00 = g.gx[0], G11 = g.gx[4], G22 = g.gx[8], G10 = g.gx[3], G21 = g.gx[7], G20 = g.gx[6];
    const float H00 = 0.5f * G00, H11 = 0.5f * G11, H22 = 0.5f * G22;  // the weight 1/2 of delta = (0, 0)
    // this lane's cell (y0 + yw, z0 + cz); d1 offsets of z, z + 1, z + 2 within a plane
    const int cz = 4 * zw + k;
    const int yrow = (y0 + yw) * L, zc = z0 + cz;

    constexpr int SPT = GM::SPT;
    const float2* src[SPT];
    int dst[SPT];
    bool act[SPT];
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        const int e = tid + i * 64 * GM::WAVES;
        act[i] = e < GM::STAGE;
        const int ee = act[i] ? e : 0;
        const int sh = ee / (GM::RY * GM::RZ), ry = (ee / GM::RZ) % GM::RY, rz = ee % GM::RZ;
        src[i] = U + (int64_t)(sh < g.S1 ? sh : 0) * N + (int64_t)((y0 - 2 + ry) & m) * g.ys + ((z0 - 2 + rz) & m);
        dst[i] = (ry * GM::RZ + rz) * GM::RP + (sh ^ (rz & 15));
    }
    float2 stg[SPT];
    auto stage_load = [&](int plane) {
#pragma unroll
        for (int i = 0; i < SPT; ++i)
            if (act[i]) stg[i] = src[i][(int64_t)(plane & m) * g.xs];
    };
    auto stage_store = [&](int plane) {
#pragma unroll
        for (int i = 0; i < SPT; ++i)
            if (act[i]) raw(plane)[dst[i]] = stg[i];
    };
    // y taps: position u = (row * GM::RZ + z') * 16 + sh reads raw rows row + 2 - ly (tile row r holds
    // y0 - 2 + r) and writes T[b][row][z'][sh]
    int traw[GM::TPT];
    bool tact[GM::TPT];
#pragma unroll
    for (int i = 0; i < GM::TPT; ++i) {
        const int u = tid + i * 64 * GM::WAVES;
        tact[i] = u < GM::TB;
        const int uu = tact[i] ? u : 0;
        const int sh = uu % 16, zp = (uu / 16) % GM::RZ, row = uu / (16 * GM::RZ);
        traw[i] = ((row + 2) * GM::RZ + zp) * GM::RP + (sh ^ (zp & 15));
    }
    auto tphase = [&](int plane) {
        const float2* rw = raw(plane);
        float2* t = tb(plane);
#pragma unroll
        for (int i = 0; i < GM::TPT; ++i) {
            if (!tact[i]) continue;
            const float2 r0 = rw[traw[i]];
            const float2 r1 = rw[traw[i] - GM::RZ * GM::RP];
            const float2 r2 = rw[traw[i] - 2 * GM::RZ * GM::RP];
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const float q0 = Q[0 * 3 + b], q1 = Q[1 * 3 + b], q2 = Q[2 * 3 + b];
                t[b * GM::TB + tid + i * 64 * GM::WAVES] =
                    make_float2(q0 * r0.x + q1 * r1.x + q2 * r2.x, q0 * r0.y + q1 * r1.y + q2 * r2.y);
            }
        }
    };
    // E_dz of a plane from its d1 values at z, z + 1, z + 2 (index dz + 2); G symmetric
    auto efun = [&](const float dd[3], float E[5]) {
        E[0] = G20 * dd[0];
        E[1] = G10 * dd[0] + G21 * dd[1];
        E[2] = G00 * dd[0] + G11 * dd[1] + G22 * dd[2];
        E[3] = G10 * dd[1] + G21 * dd[2];
        E[4] = G20 * dd[2];
    };
    auto dload = [&](int plane, float dd[3]) {
        const float* dp = d1 + (int64_t)(plane & m) * LL;
        dd[0] = dp[yrow + (zc & m)];
        dd[1] = dp[yrow + ((zc + 1) & m)];
        dd[2] = dp[yrow + ((zc + 2) & m)];
    };
    const int tme = (yw * GM::RZ + cz + 2) * 16 + s;  // this lane's T index at dz = 0 (channel 0)

    double acc_slot[4] = {0.0, 0.0, 0.0, 0.0};  // this lane's G entries 4 (lane / 16) + j, column lane % 16
    double* islot = redi + (SPLIT ? wave * 256 + (4 * (lane / 16)) * 16 + (lane % 16) : 0);
    if (SPLIT) {
#pragma unroll
        for (int j = 0; j < 4; ++j) islot[j * 16] = 0.0;
    }

    // warm-up: T of plane x0, raw plane x0+1, staged plane x0+2; E of planes x0, x0+1; d of plane x0+2.  The
    // loop starts at p = x0 - 2, whose first two steps only fill the operands of planes x0 and x0+1.
    float E0[5], E1[5], E2[5], dn[3];
    float2 B0[3], B1[3], B2[3], A0[3], A1[3], A2[3];
    stage_load(x0);
    stage_store(x0);
    stage_load(x0 + 1);
    dload(x0, dn);
    efun(dn, E0);
    dload(x0 + 1, dn);
    efun(dn, E1);
    dload(x0 + 2, dn);
    __syncthreads();
    tphase(x0);
    stage_store(x0 + 1);
    stage_load(x0 + 2);

    float4_t accr = {0.f, 0.f, 0.f, 0.f}, acci = {0.f, 0.f, 0.f, 0.f};
    // step p: slots C* hold plane p (complete now), N* plane p+1, F* plane p+2 (started now); EA = E(p+2),
    // EB = E(p+3), EF = E(p+4) (computed now)
#define D2_STEP(FIN, MID, BC, BN, BF, AC, AN, AF, EA, EB, EF)                                         \
    if (p < xend) {                                                                                 \
        __syncthreads();                                                                            \
        efun(dn, EF);                                                                               \
        dload(p + 5, dn);                                                                           \
        float c2[5], c1[5];                                                                         \
        _Pragma("unroll") for (int j = 0; j < 5; ++j) {                                             \
            c2[j] = G20 * EA[j];                                                                    \
            c1[j] = G10 * EA[j] + G21 * EB[j];                                                      \
        }                                                                                           \
        const float c00 = H00 * EA[2] + H11 * EB[2] + H22 * EF[2];                                  \
        const float c01 = G00 * EA[3] + G11 * EB[3] + G22 * EF[3];                                  \
        const float c02 = G00 * EA[4] + G11 * EB[4] + G22 * EF[4];                                  \
        if (lead) {                                                                                 \
            tphase(p + 3);                                                                          \
            stage_store(p + 4);                                                                     \
            stage_load(p + 5);                                                                      \
        }                                                                                           \
        const float2* t = tb(p + 2) + tme;                                                          \
        _Pragma("unroll") for (int b = 0; b < 3; ++b) {                                             \
            const float sg = b < NNEG ? -1.0f : 1.0f;                                               \
            float2 u[5];                                                                            \
            _Pragma("unroll") for (int j = 0; j < 5; ++j) u[j] = t[b * GM::TB + (j - 2) * 16];       \
            /* plane p + 2 as dx = 2 of plane p: its right operand is complete */                   \
            if (FIN) {                                                                              \
                float bx = BC[b].x, by = BC[b].y;                                                   \
                _Pragma("unroll") for (int j = 0; j < 5; ++j) {                                     \
                    bx = (sg * c2[j]) * u[j].x + bx;                                                \
                    by = (sg * c2[j]) * u[j].y + by;                                                \
                }                                                                                   \
                accr = __builtin_amdgcn_mfma_f32_16x16x4f32(AC[b].x, bx, accr, 0, 0, 0);            \
                if (SPLIT)                                                                          \
                    acci = __builtin_amdgcn_mfma_f32_16x16x4f32(AC[b].y, by, acci, 0, 0, 0);        \
                else                                                                                \
                    accr = __builtin_amdgcn_mfma_f32_16x16x4f32(AC[b].y, by, accr, 0, 0, 0);        \
            }                                                                                       \
            /* dx = 1 of plane p + 1 */                                                             \
            if (MID) {                                                                              \
                _Pragma("unroll") for (int j = 0; j < 5; ++j) {                                     \
                    BN[b].x = (sg * c1[j]) * u[j].x + BN[b].x;                                      \
                    BN[b].y = (sg * c1[j]) * u[j].y + BN[b].y;                                      \
                }                                                                                   \
            }                                                                                       \
            /* dx = 0 of plane p + 2 (its first terms) and its left operand */                      \
            BF[b].x = (sg * c00) * u[2].x;                                                          \
            BF[b].y = (sg * c00) * u[2].y;                                                          \
            BF[b].x = (sg * c01) * u[3].x + BF[b].x;                                                \
            BF[b].y = (sg * c01) * u[3].y + BF[b].y;                                                \
            BF[b].x = (sg * c02) * u[4].x + BF[b].x;                                                \
            BF[b].y = (sg * c02) * u[4].y + BF[b].y;                                                \
            AF[b] = u[2];                                                                           \
        }                                                                                           \
        if (SPLIT && FIN) { /* the imaginary sums go to LDS every step (no registers to keep them) */ \
            _Pragma("unroll") for (int j = 0; j < 4; ++j) {                                         \
                islot[j * 16] += (double)acci[j];                                                   \
                acci[j] = 0.f;                                                                      \
            }                                                                                       \
        }                                                                                           \
        if (!lead) {                                                                                \
            tphase(p + 3);                                                                          \
            stage_store(p + 4);                                                                     \
            stage_load(p + 5);                                                                      \
        }                                                                                           \
        ++p;                                                                                        \
    }
    // Half of the waves (two per SIMD whichever way waves are dealt to SIMDs) do the y taps and staging of
    // a step before its operand work, the others after, so that every SIMD has LDS and arithmetic work from
    // different phases within a barrier interval (the y taps write a buffer that no wave reads this step).
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const bool lead = ((wv >> 2) ^ wv) & 1;
    int p = x0 - 2;
    // steps x0 - 2 and x0 - 1 only start the operands of planes x0 and x0 + 1
    D2_STEP(false, false, B0, B1, B2, A0, A1, A2, E0, E1, E2)
    D2_STEP(false, true, B1, B2, B0, A1, A2, A0, E1, E2, E0)
    while (p < xend) {
        D2_STEP(true, true, B2, B0, B1, A2, A0, A1, E2, E0, E1)
        D2_STEP(true, true, B0, B1, B2, A0, A1, A2, E0, E1, E2)
        D2_STEP(true, true, B1, B2, B0, A1, A2, A0, E1, E2, E0)
        // FP32 sums of at most six planes (144 products per entry) move into the FP64 slots
        if ((p - x0) % 6 == 0 || p >= xend) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc_slot[j] += (double)accr[j];
                accr[j] = 0.f;
            }
        }
    }
#undef D2_STEP
    // per-wave G blocks through LDS (the tile buffers are free after this barrier), summed in a fixed order
    constexpr int ROW = SPLIT ? 512 : 256;
    double* red = (double*)smem;  // [GM::WAVES][256]
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave * 256 + (4 * (lane / 16) + j) * 16 + (lane % 16)] = acc_slot[j];
    __syncthreads();
    for (int i = tid; i < 256; i += 64 * GM::WAVES) {
        double tsum = 0.0;
#pragma unroll
        for (int w = 0; w < GM::WAVES; ++w) tsum += red[w * 256 + i];
        partial[(int64_t)blockIdx.x * ROW + i] = tsum;
        if (SPLIT) {
            double usum = 0.0;
#pragma unroll
            for (int w = 0; w < GM::WAVES; ++w) usum += redi[w * 256 + i];
            partial[(int64_t)blockIdx.x * ROW + 256 + i] = usum;
        }
    }
}

// Cross Gram (U and V different fields, or different blocks of 16 shells of one field): the same form without the
// symmetry, so the right operand of a cell has all 25 offsets delta = (dx, dz), |dx|, |dz| <= 2,
//   G[a][b] = sum_{p, r} T^a(p, r) B^b(p, r),  B(p, r) = sum_delta C_delta(p, r) T_V(p + dx, r + dz),
// and a y-filtered plane q of V serves the operands of five planes, q - 2 (dx = 2, then complete) .. q + 2.  The
// left operand T^a needs the cell's own z only: each lane filters it from the raw U tile (no halo in z) when its
// plane is complete.  250 VALU instructions and 6 matrix instructions per wave and plane, where the eigen form in
// all three directions took 54 matrix instructions, about 600 VALU instructions and uncoalesced loads (each lane
// read its shell's taps from memory).  Bound by VALU and LDS.  11 x 15 shells at L = 128: 1417 us before, 388 us now.
// FP32 sums go to FP64 after at most four planes, 96 products (the eigen form's chains: 108).  Against FP64 on the same
// fields the largest error is 0.5 to 1.2e-7 of the largest entry at L = 32 to 128, the eigen form's 1.3 to 1.4e-7.
// Step p (W = V): planes of V: p+2 into the operands, y taps of p+3, staged store of p+4, load of p+5; planes of U:
// p finished, staged store of p+1, load of p+2.
template <int NNEG>
__global__ __launch_bounds__(64 * D2X::WAVES, 3) void k_gram_cross(const float* __restrict__ d1,
                                                                  const float2* __restrict__ U,
                                                                  const float2* __restrict__ V, GramArgs g,
                                                                  double* __restrict__ partial) {
    using GM = D2X;
    constexpr int UT = GM::RY * GM::TZ * 16;  // raw U values per plane
    __shared__ __align__(16) float2 smem[2 * GM::TILE + 2 * GM::TBUF];
    __shared__ __align__(16) float2 useg[2][UT];
    auto raw = [&](int q) -> float2* { return smem + (q & 1) * GM::TILE; };
    auto tb = [&](int q) -> float2* { return smem + 2 * GM::TILE + (q & 1) * GM::TBUF; };
    const int L = g.L, m = L - 1;
    const int tid = threadIdx.x;
    const int lane = tid % 64, wave = tid / 64;
    const int s = lane % 16, k = lane / 16;
    const int zw = wave % (GM::TZ / 4), yw = wave / (GM::TZ / 4);
    const int nzb = L / GM::TZ, nyb = L / GM::NROW;
    const int nb = nzb * nyb * (L / g.xseg);
    const int q = (nb % 8 == 0) ? (int)(blockIdx.x % 8) * (nb / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
    const int xs = q / (nzb * nyb);
    const int rr = q % (nzb * nyb);
    const int PZ = nzb < 16 ? nzb : 16;
    const int zb = (rr / (PZ * nyb)) * PZ + (rr % (PZ * nyb)) % PZ;
    const int yb = (rr % (PZ * nyb)) / PZ;
    const int z0 = zb * GM::TZ, y0 = yb * GM::NROW;
    const int x0 = xs * g.xseg, xend = x0 + g.xseg;
    const int64_t N = (int64_t)L * L * L;
    const int64_t LL = (int64_t)L * L;
    const float* Q = g.Qs;
    const float G00 = g.gx[0], G11 = g.gx[4], G22 = g.gx[8], G10 = g.gx[3], G21 = g.gx[7], G20 = g.gx[6];
    const int cz = 4 * zw + k;
    const int yrow = (y0 + yw) * L, zc = z0 + cz;

    // staging: SHT threads per shell, positions z fastest
    constexpr int SHT = 4 * GM::WAVES;
    constexpr int VP = GM::RY * GM::RZ, UP = GM::RY * GM::TZ;  // positions per shell
    constexpr int VPT = (VP + SHT - 1) / SHT, UPT = UP / SHT;
    const int sh = tid / SHT, sj = tid % SHT;
    const float2* vbase = V + (int64_t)(sh < g.S2 ? sh : 0) * N;
    const float2* ubase = U + (int64_t)(sh < g.S1 ? sh : 0) * N;
    int voff[VPT], uoff[UPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int e = sj + SHT * i < VP ? sj + SHT * i : 0, ry = e / GM::RZ, rz = e % GM::RZ;
        voff[i] = ((y0 - 2 + ry) & m) * g.ys + ((z0 - 2 + rz) & m);
    }
#pragma unroll
    for (int i = 0; i < UPT; ++i) {
        const int e = sj + SHT * i;
        uoff[i] = ((y0 - 2 + e / GM::TZ) & m) * g.ys + ((z0 + e % GM::TZ) & m);
    }
    float2 vst[VPT], ust[UPT];
    auto vload = [&](int plane) {
        const float2* p = vbase + (int64_t)(plane & m) * g.xs;
#pragma unroll
        for (int i = 0; i < VPT; ++i)
            if (sj + SHT * i < VP) vst[i] = p[voff[i]];
    };
    auto vstore = [&](int plane) {
        float2* t = raw(plane);
#pragma unroll
        for (int i = 0; i < VPT; ++i) {
            const int e = sj + SHT * i, rz = e % GM::RZ;
            if (e < VP) t[e * GM::RP + (sh ^ (rz & 15))] = vst[i];
        }
    };
    auto uload = [&](int plane) {
        const float2* p = ubase + (int64_t)(plane & m) * g.xs;
#pragma unroll
        for (int i = 0; i < UPT; ++i) ust[i] = p[uoff[i]];
    };
    auto ustore = [&](int plane) {
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int e = sj + SHT * i;
            useg[plane & 1][e * 16 + (sh ^ (e % GM::TZ))] = ust[i];
        }
    };
    int traw[GM::TPT];
    bool tact[GM::TPT];
#pragma unroll
    for (int i = 0; i < GM::TPT; ++i) {
        const int u = tid + i * 64 * GM::WAVES;
        tact[i] = u < GM::TB;
        const int uu = tact[i] ? u : 0;
        const int ts = uu % 16, zp = (uu / 16) % GM::RZ, row = uu / (16 * GM::RZ);
        traw[i] = ((row + 2) * GM::RZ + zp) * GM::RP + (ts ^ (zp & 15));
    }
    auto tphase = [&](int plane) {
        const float2* rw = raw(plane);
        float2* t = tb(plane);
#pragma unroll
        for (int i = 0; i < GM::TPT; ++i) {
            if (!tact[i]) continue;
            const float2 r0 = rw[traw[i]];
            const float2 r1 = rw[traw[i] - GM::RZ * GM::RP];
            const float2 r2 = rw[traw[i] - 2 * GM::RZ * GM::RP];
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const float q0 = Q[0 * 3 + b], q1 = Q[1 * 3 + b], q2 = Q[2 * 3 + b];
                t[b * GM::TB + tid + i * 64 * GM::WAVES] =
                    make_float2(q0 * r0.x + q1 * r1.x + q2 * r2.x, q0 * r0.y + q1 * r1.y + q2 * r2.y);
            }
        }
    };
    auto efun = [&](const float dd[3], float E[5]) {
        E[0] = G20 * dd[0];
        E[1] = G10 * dd[0] + G21 * dd[1];
        E[2] = G00 * dd[0] + G11 * dd[1] + G22 * dd[2];
        E[3] = G10 * dd[1] + G21 * dd[2];
        E[4] = G20 * dd[2];
    };
    auto dload = [&](int plane, float dd[3]) {
        const float* dp = d1 + (int64_t)(plane & m) * LL;
        dd[0] = dp[yrow + (zc & m)];
        dd[1] = dp[yrow + ((zc + 1) & m)];
        dd[2] = dp[yrow + ((zc + 2) & m)];
    };
    const int tme = (yw * GM::RZ + cz + 2) * 16 + s;  // this lane's T index at dz = 0 (channel 0)
    const int ume = ((yw + 2) * GM::TZ + cz) * 16 + (s ^ cz);

    double acc_slot[4] = {0.0, 0.0, 0.0, 0.0};
    // warm-up: T of plane x0 - 2, raw plane x0 - 1, staged plane x0 of V (the loop starts at p = x0 - 4; its first
    // four steps only fill operands); E of planes x0 - 2, x0 - 1, d of plane x0
    float E0[5], E1[5], E2[5], dn[3];
    float2 B0[3], B1[3], B2[3], B3[3], B4[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) B0[b] = B1[b] = B2[b] = B3[b] = B4[b] = make_float2(0.f, 0.f);
    vload(x0 - 2);
    vstore(x0 - 2);
    vload(x0 - 1);
    dload(x0 - 2, dn);
    efun(dn, E0);
    dload(x0 - 1, dn);
    efun(dn, E1);
    dload(x0, dn);
    __syncthreads();
    tphase(x0 - 2);
    vstore(x0 - 1);
    vload(x0);
    uload(x0 - 3);
    float4_t accr = {0.f, 0.f, 0.f, 0.f};
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    const bool lead = ((wv >> 2) ^ wv) & 1;
    // step p: slots S0 .. S4 hold planes p .. p+4; EA = E(p+2), EB = E(p+3), EF = E(p+4) (computed now)
#define CROSS_STEP(S0, S1, S2, S3, S4, EA, EB, EF)                                                  \
    if (p < xend) {                                                                                 \
        __syncthreads();                                                                            \
        efun(dn, EF);                                                                               \
        dload(p + 5, dn);                                                                           \
        if (lead) {                                                                                 \
            tphase(p + 3);                                                                          \
            vstore(p + 4);                                                                          \
            vload(p + 5);                                                                           \
            ustore(p + 1);                                                                          \
            uload(p + 2);                                                                           \
        }                                                                                           \
        const float2* t = tb(p + 2) + tme;                                                          \
        _Pragma("unroll") for (int j = 0; j < 5; ++j) {                                             \
            const float c2 = G20 * EA[j], c1 = G10 * EA[j] + G21 * EB[j];                           \
            const float c0 = G00 * EA[j] + G11 * EB[j] + G22 * EF[j];                               \
            const float m1 = G10 * EB[j] + G21 * EF[j], m2 = G20 * EF[j];                           \
            _Pragma("unroll") for (int b = 0; b < 3; ++b) {                                         \
                const float2 w = t[b * GM::TB + (j - 2) * 16];                                      \
                const float sg = b < NNEG ? -1.0f : 1.0f;                                           \
                S0[b].x = (sg * c2) * w.x + S0[b].x;                                          \
                S0[b].y = (sg * c2) * w.y + S0[b].y;                                          \
                S1[b].x = (sg * c1) * w.x + S1[b].x;                                          \
                S1[b].y = (sg * c1) * w.y + S1[b].y;                                          \
                S2[b].x = (sg * c0) * w.x + S2[b].x;                                          \
                S2[b].y = (sg * c0) * w.y + S2[b].y;                                          \
                S3[b].x = (sg * m1) * w.x + S3[b].x;                                          \
                S3[b].y = (sg * m1) * w.y + S3[b].y;                                          \
                S4[b].x = j ? (sg * m2) * w.x + S4[b].x : (sg * m2) * w.x;              \
                S4[b].y = j ? (sg * m2) * w.y + S4[b].y : (sg * m2) * w.y;              \
            }                                                                                       \
        }                                                                                           \
        if (p >= x0) {                                                                              \
            const float2 r0 = useg[p & 1][ume], r1 = useg[p & 1][ume - GM::TZ * 16];                \
            const float2 r2 = useg[p & 1][ume - 2 * GM::TZ * 16];                                   \
            _Pragma("unroll") for (int b = 0; b < 3; ++b) {                                         \
                const float q0 = Q[0 * 3 + b], q1 = Q[1 * 3 + b], q2 = Q[2 * 3 + b];                \
                const float ax = q0 * r0.x + q1 * r1.x + q2 * r2.x;                                 \
                const float ay = g.vsign * (q0 * r0.y + q1 * r1.y + q2 * r2.y);                     \
                accr = __builtin_amdgcn_mfma_f32_16x16x4f32(ax, S0[b].x, accr, 0, 0, 0);            \
                accr = __builtin_amdgcn_mfma_f32_16x16x4f32(ay, S0[b].y, accr, 0, 0, 0);            \
            }                                                                                       \
        }                                                                                           \
        if (!lead) {                                                                                \
            tphase(p + 3);                                                                          \
            vstore(p + 4);                                                                          \
            vload(p + 5);                                                                           \
            ustore(p + 1);                                                                          \
            uload(p + 2);                                                                           \
        }                                                                                           \
        if ((p - x0) % 4 == 3 || p + 1 >= xend) { /* at most four planes in FP32 */                 \
            _Pragma("unroll") for (int j = 0; j < 4; ++j) {                                         \
                acc_slot[j] += (double)accr[j];                                                     \
                accr[j] = 0.f;                                                                      \
            }                                                                                       \
        }                                                                                           \
        ++p;                                                                                        \
    }
    int p = x0 - 4;
    while (p < xend) {  // 15 steps: the operand slots turn by five, the E planes by three
        CROSS_STEP(B0, B1, B2, B3, B4, E0, E1, E2)
        CROSS_STEP(B1, B2, B3, B4, B0, E1, E2, E0)
        CROSS_STEP(B2, B3, B4, B0, B1, E2, E0, E1)
        CROSS_STEP(B3, B4, B0, B1, B2, E0, E1, E2)
        CROSS_STEP(B4, B0, B1, B2, B3, E1, E2, E0)
        CROSS_STEP(B0, B1, B2, B3, B4, E2, E0, E1)
        CROSS_STEP(B1, B2, B3, B4, B0, E0, E1, E2)
        CROSS_STEP(B2, B3, B4, B0, B1, E1, E2, E0)
        CROSS_STEP(B3, B4, B0, B1, B2, E2, E0, E1)
        CROSS_STEP(B4, B0, B1, B2, B3, E0, E1, E2)
        CROSS_STEP(B0, B1, B2, B3, B4, E1, E2, E0)
        CROSS_STEP(B1, B2, B3, B4, B0, E2, E0, E1)
        CROSS_STEP(B2, B3, B4, B0, B1, E0, E1, E2)
        CROSS_STEP(B3, B4, B0, B1, B2, E1, E2, E0)
        CROSS_STEP(B4, B0, B1, B2, B3, E2, E0, E1)
    }
#undef CROSS_STEP
    double* red = (double*)smem;  // [GM::WAVES][256]
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave * 256 + (4 * (lane / 16) + j) * 16 + (lane % 16)] = acc_slot[j];
    __syncthreads();
    for (int i = tid; i < 256; i += 64 * GM::WAVES) {
        double tsum = 0.0;
#pragma unroll
        for (int w = 0; w < GM::WAVES; ++w) tsum += red[w * 256 + i];
        partial[(int64_t)blockIdx.x * 256 + i] = tsum;
    }
}

// Lane-layout self check of the 16x16x4 FP32 MFMA: C = A B for A[m][k] = m + 16 k,
// B[k][n] = (k + 1) * (n - 7).
__global__ void k_mfma_selftest(float* out) {
    const int lane = threadIdx.x;
    const int m = lane % 16, kk = lane / 16;
    float a = (float)(m + 16 * kk), b = (float)((kk + 1) * (lane % 16 - 7));
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
    for (int j = 0; j < 4; ++j) out[(4 * (lane / 16) + j) * 16 + (lane % 16)] = acc[j];
}

}  // namespace

extern "C" {

int hermes_multipole_summand_f64(hermes_ctx* ctx, int J, const double* d1, const void* F1, const void* F2,
                                 const double* gamma3x3_host, double* out_host) {
    HERMES_REQUIRE(ctx && d1 && F1 && F2 && gamma3x3_host && out_host, "hermes_multipole_summand_f64: null argument");
    HERMES_REQUIRE(J >= 2 && J <= 10, "J=%d unsupported", J);
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int L = 1 << J;
    // x segments: two planes are read ahead of each, so long ones, but at least 1024 workgroups while they last
    const int tz = L < 64 ? L : 64, ty = SUM_THREADS / tz < L ? SUM_THREADS / tz : L, nyz = (L / tz) * (L / ty);
    int xseg = L < 64 ? L : 64;
    while (xseg > 4 && nyz * (L / xseg) < 1024) xseg /= 2;
    const int nb = nyz * (L / xseg);
    const size_t scratch = 2 * (size_t)hermes_reduce::sum_scratch_rows(nb);
    double* ws = (double*)hermes_workspace(ctx, WS_CONTRACT, sizeof(double) * (2 * (size_t)nb + 2 + scratch));
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    Gamma3 G;
    for (int i = 0; i < 9; ++i) G.g[i] = gamma3x3_host[i];
    k_summand_f64<<<dim3(nyz, L / xseg), SUM_THREADS, 0, ctx->stream>>>(L, tz, ty, xseg, d1, (const double2*)F1,
                                                                       (const double2*)F2, G, ws);
    HERMES_LAUNCH_CHECK();
    HERMES_CHECK_HIP(hermes_reduce::sum_columns(ctx->stream, ws, 2, nb, 2, ws + 2 * nb + 2, ws + 2 * nb));
    HERMES_CHECK_HIP(hipMemcpyAsync(out_host, ws + 2 * nb, sizeof(double) * 2, hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return 0;
}

// Waits for the recorded (start, end) event pairs of timed Gram launches and adds their
// durations to the totals (launches may sit on any stream).
static int gram_flush(hermes_ctx* ctx) {
    for (size_t i = 0; i < ctx->gram_pending; ++i) {
        float ms = 0.0f;
        HERMES_CHECK_HIP(hipEventSynchronize(ctx->gram_ev[2 * i + 1]));
        HERMES_CHECK_HIP(hipEventElapsedTime(&ms, ctx->gram_ev[2 * i], ctx->gram_ev[2 * i + 1]));
        ctx->gram_ms += ms;
        ctx->gram_calls += 1;
    }
    ctx->gram_pending = 0;
    return 0;
}

// Launches the Gram kernel and the fixed-order row reduction; the 16 x 16 raw sums land in
// out_dev (256 doubles; row i, column j at i * 16 + j).  No host synchronisation.
static int gram_launch(hermes_ctx* ctx, int J, const float* d1, const void* U, int n_u, const void* V, int n_v,
                       int v_conj, const double* Q3x3_host, const double* lam3_host, double* out_dev, GramArgs* gout,
                       bool split = false) {
    HERMES_REQUIRE(ctx && d1 && U && Q3x3_host && lam3_host && out_dev, "hermes_multipole_gram_f32: null argument");
    HERMES_REQUIRE(J >= 3 && J <= 10, "hermes_multipole_gram_f32: J=%d unsupported (needs L >= 8)", J);
    HERMES_REQUIRE(n_u >= 1 && n_u <= 16, "n_u=%d outside 1..16", n_u);
    HERMES_REQUIRE(V == nullptr || (n_v >= 1 && n_v <= 16), "n_v=%d outside 1..16", n_v);
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int L = 1 << J;
    GramArgs g;
    g.L = L;
    g.xs = ctx->field_layout ? L : L * L;  // x-major fields: (x L + y) L + z; y-major: (y L + x) L + z
    g.ys = ctx->field_layout ? L * L : L;
    g.S1 = n_u;
    g.cross = V != nullptr;
    g.S2 = g.cross ? n_v : n_u;
    g.vsign = v_conj ? 1.0f : -1.0f;  // Re(U V) needs -V.im, Re(U conj V) needs +V.im
    // planes per workgroup: each segment pays a warm-up of two (auto) or four (cross) planes and a final reduction,
    // so it takes 512 planes (8192 workgroups at L = 512, 16 per workgroup slot; 256- and 128-plane segments
    // measured 2% and 3% slower), and shorter ones, down to 8, where the columns alone do not give the 512
    // workgroups that fill the chip (L = 64: 65 us with whole columns, 128 workgroups; 34 us with 16 planes)
    const int ncol = g.cross ? (L / D2X::TZ) * (L / D2X::NROW) : (L / D2::TZ) * (L / D2::NROW);
    const int fill = g.cross ? 2 * 768 : 512;  // cross: 768 slots, at least two rounds of them
    g.xseg = L < 512 ? L : 512;
    while (g.xseg > 8 && ncol * (L / g.xseg) < fill) g.xseg /= 2;
    for (int l1 = 0; l1 < 3; ++l1)
        for (int l2 = 0; l2 < 3; ++l2) {
            double t = 0.0;
            for (int a = 0; a < 3; ++a) t += Q3x3_host[l1 * 3 + a] * lam3_host[a] * Q3x3_host[l2 * 3 + a];
            g.gx[l1 * 3 + l2] = (float)t;
        }
    int order[3] = {0, 1, 2}, nneg = 0;  // eigenvalues ascending (insertion sort of three)
    for (int i = 1; i < 3; ++i)
        for (int j = i; j > 0 && lam3_host[order[j]] < lam3_host[order[j - 1]]; --j) {
            const int t = order[j];
            order[j] = order[j - 1];
            order[j - 1] = t;
        }
    for (int c = 0; c < 3; ++c) {
        const double lc = lam3_host[order[c]];
        if (lc < 0.0) ++nneg;
        for (int tap = 0; tap < 3; ++tap) g.Qs[tap * 3 + c] = (float)(Q3x3_host[tap * 3 + order[c]] * sqrt(fabs(lc)));
    }
    HERMES_REQUIRE(g.cross || J >= 4, "hermes_multipole_gram_f32: J=%d, the auto Gram needs J >= 4", J);
    const int nblocks = ncol * (L / g.xseg);
    HERMES_REQUIRE(!split || !g.cross, "hermes_multipole_gram_f32: split sums are for the auto Gram");
    const int row = split ? 512 : 256;
    double* ws = (double*)hermes_workspace(
        ctx, WS_CONTRACT, sizeof(double) * row * ((size_t)nblocks + (size_t)hermes_reduce::sum_scratch_rows(nblocks)));
    HERMES_REQUIRE(ws, "%s", hermes_last_error());
    const bool timed = ctx->time_gram && !ctx->capturing;
    size_t slot = 0;
    if (timed) {
        if (ctx->gram_pending >= 4096 && gram_flush(ctx)) return 1;
        slot = 2 * ctx->gram_pending;
        while (ctx->gram_ev.size() < slot + 2) {
            hipEvent_t e = nullptr;
            HERMES_CHECK_HIP(hipEventCreate(&e));
            ctx->gram_ev.push_back(e);
        }
        HERMES_CHECK_HIP(hipEventRecord(ctx->gram_ev[slot], ctx->stream));
    }
    const float2 *u = (const float2*)U, *v = (const float2*)V;
    if (g.cross)
        switch (nneg) {
            case 0: k_gram_cross<0><<<nblocks, 64 * D2X::WAVES, 0, ctx->stream>>>(d1, u, v, g, ws); break;
            case 1: k_gram_cross<1><<<nblocks, 64 * D2X::WAVES, 0, ctx->stream>>>(d1, u, v, g, ws); break;
            case 2: k_gram_cross<2><<<nblocks, 64 * D2X::WAVES, 0, ctx->stream>>>(d1, u, v, g, ws); break;
            default: k_gram_cross<3><<<nblocks, 64 * D2X::WAVES, 0, ctx->stream>>>(d1, u, v, g, ws); break;
        }
    else
        switch (nneg + (split ? 4 : 0)) {
            case 0: k_gram_auto<0><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 1: k_gram_auto<1><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 2: k_gram_auto<2><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 3: k_gram_auto<3><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 4: k_gram_auto<0, true><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 5: k_gram_auto<1, true><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            case 6: k_gram_auto<2, true><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
            default: k_gram_auto<3, true><<<nblocks, 64 * D2::WAVES, 0, ctx->stream>>>(d1, (const float2*)U, g, ws); break;
        }
    HERMES_LAUNCH_CHECK();
    if (timed) {
        HERMES_CHECK_HIP(hipEventRecord(ctx->gram_ev[slot + 1], ctx->stream));
        ctx->gram_pending += 1;
    }
    HERMES_CHECK_HIP(hermes_reduce::sum_columns(ctx->stream, ws, row, nblocks, row, ws + (size_t)nblocks * row, out_dev));
    if (gout) *gout = g;
    return 0;
}

int hermes_multipole_gram_f32(hermes_ctx* ctx, int J, const float* d1, const void* U, int n_u, const void* V, int n_v,
                              int v_conj, const double* Q3x3_host, const double* lam3_host, double* out_host) {
    HERMES_REQUIRE(ctx && out_host, "hermes_multipole_gram_f32: null argument");
    HERMES_REQUIRE(!ctx->capturing, "hermes_multipole_gram_f32 returns host data; capture hermes_multipole_gram_f32_dev");
    double* dst = (double*)hermes_workspace(ctx, WS_MISC, sizeof(double) * 256);
    HERMES_REQUIRE(dst, "%s", hermes_last_error());
    GramArgs g;
    if (int rc = gram_launch(ctx, J, d1, U, n_u, V, n_v, v_conj, Q3x3_host, lam3_host, dst, &g)) return rc;
    double h[256];
    HERMES_CHECK_HIP(hipMemcpyAsync(h, dst, sizeof(double) * 256, hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < g.S1; ++i)
        for (int j = 0; j < g.S2; ++j)
            out_host[i * g.S2 + j] = g.cross ? h[i * 16 + j] : h[i * 16 + j] + h[j * 16 + i];
    return 0;
}

int hermes_multipole_gram_f32_dev(hermes_ctx* ctx, int J, const float* d1, const void* U, int n_u, const void* V,
                                  int n_v, int v_conj, const double* Q3x3_host, const double* lam3_host,
                                  double* out_dev) {
    return gram_launch(ctx, J, d1, U, n_u, V, n_v, v_conj, Q3x3_host, lam3_host, out_dev, nullptr);
}

int hermes_multipole_gram_f32_dev_ri(hermes_ctx* ctx, int J, const float* d1, const void* U, int n_u,
                                     const double* Q3x3_host, const double* lam3_host, double* out_dev) {
    return gram_launch(ctx, J, d1, U, n_u, nullptr, 0, 0, Q3x3_host, lam3_host, out_dev, nullptr, true);
}

int hermes_profile_gram(hermes_ctx* ctx, int enable, double* total_ms_out, int64_t* calls_out) {
    HERMES_REQUIRE(ctx, "hermes_profile_gram: null context");
    HERMES_REQUIRE(!ctx->capturing, "hermes_profile_gram: the stream is being captured");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    if (gram_flush(ctx)) return 1;
    if (total_ms_out) *total_ms_out = ctx->gram_ms;
    if (calls_out) *calls_out = ctx->gram_calls;
    if (enable) {
        ctx->gram_ms = 0.0;
        ctx->gram_calls = 0;
    }
    ctx->time_gram = enable != 0;
    return 0;
}

int hermes_mfma_selftest(hermes_ctx* ctx, double* max_abs_err) {
    HERMES_REQUIRE(ctx && max_abs_err, "null argument");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    float* d = (float*)hermes_workspace(ctx, WS_MISC, sizeof(float) * 256);
    HERMES_REQUIRE(d, "%s", hermes_last_error());
    k_mfma_selftest<<<1, 64, 0, ctx->stream>>>(d);
    HERMES_LAUNCH_CHECK();
    float h[256];
    HERMES_CHECK_HIP(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    HERMES_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    double err = 0.0;
    for (int m = 0; m < 16; ++m)
        for (int n = 0; n < 16; ++n) {
            double ref = 0.0;
            for (int k = 0; k < 4; ++k) ref += (double)(m + 16 * k) * (double)((k + 1) * (n - 7));
            double e = fabs(ref - h[m * 16 + n]);
            if (e > err) err = e;
        }
    *max_abs_err = err;
    return 0;
}

}  // extern "C"
