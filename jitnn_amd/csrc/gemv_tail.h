// The last k % 256 values of a row for a few activation rows: what gemv_rows_kernel and gemv_held_kernel, which work on whole columns of
// 256 values, leave of rows of 32-value blocks.
#pragma once
#include "common.h"
#include "dequant.h"

namespace jitnn {

constexpr int GT_ROWS = 16, GT_B = 4, GT_THREADS = 256;  // weight rows of a workgroup, activation rows of a thread (64 in all at most)
__host__ __device__ constexpr size_t gemv_tail_lds_bytes(int rows, int blocks) { return (size_t)(rows + GT_ROWS) * (8 * blocks + 1) * sizeof(float4); }

// y[b, row] += sum over the last `blocks` (1..7) blocks of W [n, k], in FP32: the dequantiser's values, one FMA each, in four sums.
// The tails of the workgroup's weight rows, dequantised once, and of the activations wait in LDS, rows an odd number of quads apart, so that
// the rows a wave reads at a time lie in different banks; a thread takes one weight row and GT_B activation rows.
// Bound by the narrow loads of the blocks: 9.8 us for 14336 weight rows, 7 blocks and 16 activation rows, 12 for 8000 rows of Q8_0 and 40; with
// every thread dequantising its own row from memory - sixteen of them the same one - the first took 20.
// grid ceil(n / GT_ROWS); gemv_tail_lds_bytes() of dynamic LDS; rows <= 64.
template <int FMT>
__global__ void __launch_bounds__(GT_THREADS) gemv_tail_kernel(const uint8_t *__restrict__ W, const float *__restrict__ x, float *__restrict__ y, int n, int k, int rows, int blocks) {
    extern __shared__ __align__(16) uint8_t gt_smem[];
    const int tid = threadIdx.x, quads = 8 * blocks, pitch = quads + 1, k0 = k - 32 * blocks, n0 = blockIdx.x * GT_ROWS;
    float4 *xs = reinterpret_cast<float4 *>(gt_smem), *ws = xs + rows * pitch;
    for (int i = tid; i < rows * quads; i += GT_THREADS) {
        const int b = i / quads, q = i - b * quads;
        xs[b * pitch + q] = *reinterpret_cast<const float4 *>(x + (size_t)b * k + k0 + 4 * q);
    }
    const size_t rowbytes = (size_t)(k / block_values(FMT)) * block_bytes(FMT);
    for (int i = tid; i < GT_ROWS * quads; i += GT_THREADS) {
        const int r = i / quads, q = i - r * quads;
        ws[r * pitch + q] = dequant4<FMT>(W + (size_t)min(n0 + r, n - 1) * rowbytes, (size_t)k0 + 4 * q);
    }
    __syncthreads();
    const int r = tid & (GT_ROWS - 1), b0 = GT_B * (tid / GT_ROWS);
    if (n0 + r >= n || b0 >= rows) return;
    const float4 *wp = ws + r * pitch, *xp[GT_B];
#pragma unroll
    for (int i = 0; i < GT_B; ++i) xp[i] = xs + min(b0 + i, rows - 1) * pitch;
    float4 acc[GT_B] = {};
    for (int q = 0; q < quads; ++q) {
        const float4 w = wp[q];
#pragma unroll
        for (int i = 0; i < GT_B; ++i) {
            const float4 v = xp[i][q];
            acc[i].x = __builtin_fmaf(w.x, v.x, acc[i].x);
            acc[i].y = __builtin_fmaf(w.y, v.y, acc[i].y);
            acc[i].z = __builtin_fmaf(w.z, v.z, acc[i].z);
            acc[i].w = __builtin_fmaf(w.w, v.w, acc[i].w);
        }
    }
#pragma unroll
    for (int i = 0; i < GT_B; ++i)
        if (b0 + i < rows) y[(size_t)(b0 + i) * n + n0 + r] += (acc[i].x + acc[i].y) + (acc[i].z + acc[i].w);
}

}  // namespace jitnn
