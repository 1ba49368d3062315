// Fixed-order column sums of FP64 partial sums (one row per workgroup of the kernel that wrote them).
//
// A workgroup takes COLS columns and 256 / COLS phases: phase p adds rows p, p + phases, ... of its row range, and
// the phases are added pairwise, so results do not depend on scheduling.  More than 64 rows per phase are summed in
// two launches over ranges of 512 rows.  (One thread per column over the rows, or a single workgroup in a second
// stage, is a serial chain of loads: 102 us for 1024 rows of 2, 115 us for 8192 rows of 256, 26 us for 1073 rows of
// 20; now 6, 13 and 5 us.)
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace hermes_reduce {

constexpr int THREADS = 256;

template <int COLS>
__global__ __launch_bounds__(THREADS) void k_sum_columns(const double* __restrict__ in, int64_t stride, int rows,
                                                         int rows_per, int n, double* __restrict__ out) {
    constexpr int PHASES = THREADS / COLS;
    __shared__ double sh[THREADS];
    const int c = blockIdx.x * COLS + threadIdx.x % COLS;
    const int r0 = blockIdx.y * rows_per, r1 = r0 + rows_per < rows ? r0 + rows_per : rows;
    double s = 0.0;
    if (c < n) {
#pragma unroll 8
        for (int r = r0 + threadIdx.x / COLS; r < r1; r += PHASES) s += in[(int64_t)r * stride + c];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
#pragma unroll
    for (int h = THREADS / 2; h >= COLS; h /= 2) {
        if (threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x < COLS && c < n) out[(int64_t)blockIdx.y * n + c] = sh[threadIdx.x];
}

// Rows of the scratch `tmp` (n doubles each) that sum_columns may use for this many rows.
inline int sum_scratch_rows(int rows) { return (rows + 511) / 512; }

// out[c] = sum of in[r * stride + c] over r < rows, c < n; tmp as sum_scratch_rows (unused up to 64 rows a phase).
inline hipError_t sum_columns(hipStream_t st, const double* in, int64_t stride, int rows, int n, double* tmp,
                              double* out) {
    auto launch = [&](auto kernel, int cols) {
        const int phases = THREADS / cols, nb = (n + cols - 1) / cols;
        if (rows <= 64 * phases) {
            kernel<<<nb, THREADS, 0, st>>>(in, stride, rows, rows, n, out);
            return;
        }
        const int groups = sum_scratch_rows(rows);
        kernel<<<dim3(nb, groups), THREADS, 0, st>>>(in, stride, rows, 512, n, tmp);
        kernel<<<nb, THREADS, 0, st>>>(tmp, n, groups, groups, n, out);
    };
    if (n == 1) launch(k_sum_columns<1>, 1);
    else if (n == 2) launch(k_sum_columns<2>, 2);
    else launch(k_sum_columns<8>, 8);
    return hipGetLastError();
}

}  // namespace hermes_reduce
