// 3-D FFTs over (L, L, L) grids; plans cached per context.
// Replaces scipy.fft rfftn/irfftn/fftn/ifftn in convolution.py:284-295.
// Grids of 128^3 and more: the contiguous z lines by a 1-D rocFFT plan (it runs at the rate of a copy), the strided y
// and x lines by k_fft_lines.  Smaller ones: a 3-D rocFFT plan.
// Transforms are unnormalised (the inverse is not divided by N); callers fold
// 1/N into the spectral multiply.
#include <rocfft/rocfft.h>

#include <map>
#include <mutex>
#include <tuple>

#include "../../include/hermes_amd.h"
#include "fft_lds.h"
#include "hermes_common.h"

namespace {
std::once_flag g_rocfft_once;

struct Plan {
    rocfft_plan plan = nullptr;
    rocfft_execution_info info = nullptr;
    size_t work_bytes = 0;
    void* work = nullptr;
};

// key: (L, kind, double, batch, inplace, dimensions)
using PlanKey = std::tuple<int, int, int, int64_t, int, int>;
}  // namespace

struct hermes_fft_cache {
    std::map<PlanKey, Plan> plans;
};

void hermes_fft_cache_destroy(hermes_fft_cache* c) {
    if (!c) return;
    for (auto& kv : c->plans) {
        if (kv.second.info) rocfft_execution_info_destroy(kv.second.info);
        if (kv.second.plan) rocfft_plan_destroy(kv.second.plan);
        if (kv.second.work) (void)hipFree(kv.second.work);
    }
    delete c;
}

namespace {
// kind: 0 = r2c forward, 1 = c2r inverse, 2 = c2c forward, 3 = c2c inverse
// dims = 3: batch grids; dims = 1: batch contiguous lines of L values.
int get_plan(hermes_ctx* ctx, int L, int kind, int dbl, int64_t batch, int inplace, int dims, Plan** out) {
    std::call_once(g_rocfft_once, []() { rocfft_setup(); });
    if (!ctx->fft) ctx->fft = new hermes_fft_cache();
    PlanKey key{L, kind, dbl, batch, inplace, dims};
    auto it = ctx->fft->plans.find(key);
    if (it != ctx->fft->plans.end()) {
        *out = &it->second;
        return 0;
    }
    Plan p;
    size_t lengths[3] = {(size_t)L, (size_t)L, (size_t)L};
    rocfft_transform_type tt = kind == 0   ? rocfft_transform_type_real_forward
                               : kind == 1 ? rocfft_transform_type_real_inverse
                               : kind == 2 ? rocfft_transform_type_complex_forward
                                           : rocfft_transform_type_complex_inverse;
    rocfft_precision prec = dbl ? rocfft_precision_double : rocfft_precision_single;
    rocfft_result_placement pl = inplace ? rocfft_placement_inplace : rocfft_placement_notinplace;
    rocfft_status s = rocfft_plan_create(&p.plan, pl, tt, prec, (size_t)dims, lengths, (size_t)batch, nullptr);
    if (s != rocfft_status_success) {
        hermes_set_error("rocfft_plan_create failed (status %d) L=%d kind=%d dbl=%d batch=%lld", (int)s, L, kind,
                         dbl, (long long)batch);
        return 3;
    }
    rocfft_plan_get_work_buffer_size(p.plan, &p.work_bytes);
    rocfft_execution_info_create(&p.info);
    if (p.work_bytes) {
        if (hipMalloc(&p.work, p.work_bytes) != hipSuccess) {
            hermes_set_error("hipMalloc of %zu bytes for the rocFFT work buffer failed", p.work_bytes);
            return 1;
        }
        rocfft_execution_info_set_work_buffer(p.info, p.work, p.work_bytes);
    }
    auto res = ctx->fft->plans.emplace(key, p);
    *out = &res.first->second;
    return 0;
}

int run_plan(hermes_ctx* ctx, int J, int kind, int dbl, int64_t batch, int dims, const void* in, void* out) {
    const int inplace = (in == out) ? 1 : 0;
    Plan* p = nullptr;
    int rc = get_plan(ctx, 1 << J, kind, dbl, batch, inplace, dims, &p);
    if (rc) return rc;
    rocfft_execution_info_set_stream(p->info, ctx->stream);
    void* ib[1] = {const_cast<void*>(in)};
    void* ob[1] = {out};
    rocfft_status s = rocfft_execute(p->plan, ib, inplace ? nullptr : ob, p->info);
    if (s != rocfft_status_success) {
        hermes_set_error("rocfft_execute failed (status %d)", (int)s);
        return 3;
    }
    return 0;
}

// Strided lines of L = 2^LOG2L values, in place: element e of column c < ncols of block o is at o * outer + c + e * es
// (y lines: a block is an x plane, its columns the z of a row; x lines: one block, its columns the positions of a
// plane).  A workgroup stages TW columns in LDS, so every access is a run of TW values and each value is read and
// written once; bound by HBM.  TW values are one 128-byte line (for half spectra the rows of y lines, L / 2 + 1 values
// apart, start anywhere in a line: neighbouring tiles, on one XCD, share it in its L2).  Plain loads and stores: with
// the streaming hint the shared lines and what the previous pass left in the last-level cache are lost (512^3 FP32,
// y lines: 218 us plain, 446 streaming; 256^3 FP64, x lines: 40 and 80).  The library's strided kernels took 598 us
// (512^3 FP32, half spectrum: 1.8 TB/s; now y 218, x 272) and 86 us (256^3 FP64: 3.1 TB/s; now 39 and 40).
// CONV (x lines of a convolution with a real kernel of the same layout, DIR = -1): the line is transformed, multiplied
// by kernel * scale and transformed back while it is in LDS, which leaves out one pass over the spectrum and the
// product's own (256^3 FP64: 40 + 51 + 40 us as three passes).
template <class C, int LOG2L, int TW, int NT, int DIR, bool CONV = false>
__global__ __launch_bounds__(NT) void k_fft_lines(C* data, const C* __restrict__ twg, int64_t es, int64_t outer,
                                                  int64_t ncols, int ntile,
                                                  const decltype(C::x)* __restrict__ kernel = nullptr,
                                                  decltype(C::x) scale = 0) {
    constexpr int L = 1 << LOG2L;
    static_assert(NT % TW == 0 && TW * L % NT == 0, "a thread keeps one column of the tile");
    using F = hermes_fft::LdsFft<LOG2L, TW, NT, DIR, true, C>;
    extern __shared__ __align__(16) char lines_lds[];
    C* tw = (C*)lines_lds;
    C* lds = tw + L;
    const int tid = threadIdx.x;
    // workgroups are dealt to the 8 XCDs round-robin: each XCD takes a contiguous range of tiles
    const int64_t nb = gridDim.x, xcd = blockIdx.x % 8, rem = nb % 8;
    const int64_t b = xcd * (nb / 8) + (xcd < rem ? xcd : rem) + blockIdx.x / 8;
    const int64_t col = (b % ntile) * TW + tid % TW;
    const bool inside = col < ncols;  // the last tile of a block may be partly empty
    const int64_t first = (b / ntile) * outer + (inside ? col : 0) + (int64_t)(tid / TW) * es;
    C* p = data + first;
    const int64_t step = (int64_t)(NT / TW) * es;
    hermes_fft::load_twiddles<LOG2L>(tw, twg, tid, NT);
    constexpr int PER = TW * L / NT;
    C v[PER];  // the whole tile is in flight before the first store to LDS
#pragma unroll
    for (int k = 0; k < PER; ++k) v[k] = p[k * step];
    decltype(C::x) w[CONV ? PER : 1];
    if constexpr (CONV) {
#pragma unroll
        for (int k = 0; k < PER; ++k) w[k] = kernel[first + k * step];
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) lds[tid + k * NT] = v[k];
    __syncthreads();
    F::run(lds, tw, tid);
    if constexpr (CONV) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const decltype(C::x) c = w[k] * scale;
            C& z = lds[tid + k * NT];
            z.x *= c;
            z.y *= c;
        }
        for (int k = tid; k < L; k += NT) tw[k].y = -tw[k].y;
        __syncthreads();
        hermes_fft::LdsFft<LOG2L, TW, NT, -DIR, true, C>::run(lds, tw, tid);
    }
    if (!inside) return;
#pragma unroll
    for (int k = 0; k < PER; ++k) p[k * step] = lds[tid + k * NT];
}

// Tile of the strided passes: 128 bytes wide; 128^3 takes 16 values in FP64 as well (21 us for 24 with 8).
template <class C, int LOG2L>
struct LineTile {
    static constexpr int L = 1 << LOG2L;
    static constexpr int TW = LOG2L == 7 ? 16 : 128 / (int)sizeof(C);
    static constexpr int NT = TW * L > 4096 ? 512 : 256;
    static constexpr size_t lds = sizeof(C) * (size_t)(L + TW * L);
    static_assert(lds <= 160 * 1024, "LDS of a CU");
};

// y and x lines of `batch` grids of (L, L, M) values, in place.
template <class C, int LOG2L, int DIR>
int run_lines(hermes_ctx* ctx, int64_t batch, int64_t M, C* data, const C* twg) {
    using Tile = LineTile<C, LOG2L>;
    constexpr int L = Tile::L, TW = Tile::TW, NT = Tile::NT;
    auto k = k_fft_lines<C, LOG2L, TW, NT, DIR>;
    HERMES_CHECK_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Tile::lds));
    const int64_t yt = (M + TW - 1) / TW, xt = (L * M + TW - 1) / TW;
    k<<<(unsigned)(batch * L * yt), NT, Tile::lds, ctx->stream>>>(data, twg, M, L * M, M, (int)yt, nullptr, 0);
    HERMES_LAUNCH_CHECK();
    k<<<(unsigned)(batch * xt), NT, Tile::lds, ctx->stream>>>(data, twg, L * M, L * L * M, L * M, (int)xt, nullptr, 0);
    HERMES_LAUNCH_CHECK();
    return 0;
}

// y lines forward, x lines forward times kernel * scale and back, y lines back, of one half spectrum, in place.
template <class C, int LOG2L>
int run_conv(hermes_ctx* ctx, C* data, const C* fwd, const C* inv, const decltype(C::x)* kernel, double scale) {
    using Tile = LineTile<C, LOG2L>;
    constexpr int L = Tile::L, TW = Tile::TW, NT = Tile::NT;
    constexpr int64_t M = L / 2 + 1, yt = (M + TW - 1) / TW, xt = (L * M + TW - 1) / TW;
    auto kf = k_fft_lines<C, LOG2L, TW, NT, -1>;
    auto kb = k_fft_lines<C, LOG2L, TW, NT, 1>;
    auto kx = k_fft_lines<C, LOG2L, TW, NT, -1, true>;
    for (const void* k : {(const void*)kf, (const void*)kb, (const void*)kx})
        HERMES_CHECK_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)Tile::lds));
    kf<<<(unsigned)(L * yt), NT, Tile::lds, ctx->stream>>>(data, fwd, M, L * M, M, (int)yt, nullptr, 0);
    HERMES_LAUNCH_CHECK();
    kx<<<(unsigned)xt, NT, Tile::lds, ctx->stream>>>(data, fwd, L * M, L * L * M, L * M, (int)xt, kernel,
                                                    (decltype(C::x))scale);
    HERMES_LAUNCH_CHECK();
    kb<<<(unsigned)(L * yt), NT, Tile::lds, ctx->stream>>>(data, inv, M, L * M, M, (int)yt, nullptr, 0);
    HERMES_LAUNCH_CHECK();
    return 0;
}

template <class C>
int conv_lines(hermes_ctx* ctx, int J, C* data, const C* fwd, const C* inv, const void* kernel, double scale) {
    HERMES_REQUIRE(fwd && inv, "%s", hermes_last_error());
    auto w = (const decltype(C::x)*)kernel;
    switch (J) {
        case 7: return run_conv<C, 7>(ctx, data, fwd, inv, w, scale);
        case 8: return run_conv<C, 8>(ctx, data, fwd, inv, w, scale);
        case 9: return run_conv<C, 9>(ctx, data, fwd, inv, w, scale);
        default: return run_conv<C, 10>(ctx, data, fwd, inv, w, scale);
    }
}

template <class C, int DIR>
int lines(hermes_ctx* ctx, int J, int64_t batch, int64_t M, C* data, const C* twg) {
    HERMES_REQUIRE(twg, "%s", hermes_last_error());
    switch (J) {
        case 7: return run_lines<C, 7, DIR>(ctx, batch, M, data, twg);
        case 8: return run_lines<C, 8, DIR>(ctx, batch, M, data, twg);
        case 9: return run_lines<C, 9, DIR>(ctx, batch, M, data, twg);
        default: return run_lines<C, 10, DIR>(ctx, batch, M, data, twg);
    }
}

int strided(hermes_ctx* ctx, int J, int dbl, int64_t batch, int64_t M, int dir, void* data) {
    if (dbl)
        return dir > 0 ? lines<double2, 1>(ctx, J, batch, M, (double2*)data, hermes_twiddles_f64(ctx, J, 1))
                       : lines<double2, -1>(ctx, J, batch, M, (double2*)data, hermes_twiddles_f64(ctx, J, -1));
    return dir > 0 ? lines<float2, 1>(ctx, J, batch, M, (float2*)data, hermes_twiddles(ctx, J, 1))
                   : lines<float2, -1>(ctx, J, batch, M, (float2*)data, hermes_twiddles(ctx, J, -1));
}

// Own strided passes from 128^3 on.  Below, the 3-D plan takes two launches (64^3: 13 us) and this way three.
constexpr int LINES_MIN_J = 7;

int run(hermes_ctx* ctx, int J, int kind, int dbl, int batch, const void* in, void* out) {
    HERMES_REQUIRE(ctx, "null context");
    HERMES_REQUIRE(J >= 1 && J <= 10, "FFT: J=%d unsupported", J);
    HERMES_REQUIRE(batch >= 1, "FFT: batch must be >= 1");
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    HERMES_REQUIRE(!(in == out && (kind == 0 || kind == 1)), "real<->complex FFTs must be out of place");
    if (J < LINES_MIN_J) return run_plan(ctx, J, kind, dbl, batch, 3, in, out);
    const int64_t L = (int64_t)1 << J, nlines = batch * L * L;
    if (kind == 1) {  // the real lines last
        const int rc = strided(ctx, J, dbl, batch, L / 2 + 1, 1, const_cast<void*>(in));
        return rc ? rc : run_plan(ctx, J, kind, dbl, nlines, 1, in, out);
    }
    const int rc = run_plan(ctx, J, kind, dbl, nlines, 1, in, out);
    return rc ? rc : strided(ctx, J, dbl, batch, kind == 0 ? L / 2 + 1 : L, kind == 3 ? 1 : -1, out);
}
}  // namespace

extern "C" {

int hermes_fft_r2c(hermes_ctx* ctx, int J, int batch, int dbl, const void* in_real, void* out_half) {
    return run(ctx, J, 0, dbl, batch, in_real, out_half);
}

int hermes_fft_c2r(hermes_ctx* ctx, int J, int batch, int dbl, void* in_half, void* out_real) {
    return run(ctx, J, 1, dbl, batch, in_half, out_real);
}

int hermes_fft_c2c(hermes_ctx* ctx, int J, int batch, int dbl, int inverse, const void* in, void* out) {
    return run(ctx, J, inverse ? 3 : 2, dbl, batch, in, out);
}

int hermes_convolve_real(hermes_ctx* ctx, int J, int dbl, const void* in_real, const void* kernel_half, double scale,
                         void* spec, void* out_real) {
    HERMES_REQUIRE(ctx && in_real && kernel_half && spec && out_real, "hermes_convolve_real: null argument");
    HERMES_REQUIRE(J >= 1 && J <= 10, "hermes_convolve_real: J=%d unsupported", J);
    if (J < LINES_MIN_J) {
        int rc = run(ctx, J, 0, dbl, 1, in_real, spec);
        if (rc == 0) rc = hermes_spectrum_mul(ctx, J, 1, dbl, spec, kernel_half, 0, scale);
        return rc ? rc : run(ctx, J, 1, dbl, 1, spec, out_real);
    }
    HERMES_CHECK_HIP(hipSetDevice(ctx->device));
    const int64_t nlines = (int64_t)1 << (2 * J);
    if (int rc = run_plan(ctx, J, 0, dbl, nlines, 1, in_real, spec)) return rc;
    const int rc = dbl ? conv_lines(ctx, J, (double2*)spec, hermes_twiddles_f64(ctx, J, -1),
                                    hermes_twiddles_f64(ctx, J, 1), kernel_half, scale)
                       : conv_lines(ctx, J, (float2*)spec, hermes_twiddles(ctx, J, -1), hermes_twiddles(ctx, J, 1),
                                    kernel_half, scale);
    return rc ? rc : run_plan(ctx, J, 1, dbl, nlines, 1, spec, out_real);
}

}  // extern "C"
