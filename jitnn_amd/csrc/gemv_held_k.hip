// gemv_held_kernel for the formats of 256-value blocks, and the join of its K slices.
#include "gemv_held_launch.h"

namespace jitnn {

// y[b, row] = sum over the K slices of part[slice][b, row], slices in order (+ bias[row]) (+ res[b, row]); count = rows * n.
// (y, bias and res are the caller's: no alignment beyond a float's; part may be y, one slice)
__global__ void __launch_bounds__(256) rows_join_kernel(const float *part, float *y, int count, int n, int slices,
                                                         const float *__restrict__ bias, const float *res) {
    for (int i = (int)blockIdx.x * 256 + (int)threadIdx.x; i < count; i += (int)gridDim.x * 256) {
        float sum = 0.f;
        for (int z0 = 0; z0 < slices; z0 += 8) {  // (eight slices' loads under way at once)
            float v[8];
#pragma unroll
            for (int z = 0; z < 8; ++z) v[z] = part[(size_t)min(z0 + z, slices - 1) * count + i];
#pragma unroll
            for (int z = 0; z < 8; ++z) sum = z0 + z < slices ? sum + v[z] : sum;
        }
        y[i] = sum + (bias ? bias[i % n] : 0.f) + (res ? res[i] : 0.f);
    }
}

KernelRef gemv_held_kernel_k(int fmt, int groups_held) {
    switch (fmt) {
    case F_Q4_K: return held_ref<F_Q4_K>(groups_held);
    case F_Q5_K: return held_ref<F_Q5_K>(groups_held);
    case F_Q6_K: return held_ref<F_Q6_K>(groups_held);
    case F_Q2_K: return held_ref<F_Q2_K>(groups_held);
    default: return {nullptr, 0};
    }
}

void rows_join_launch(hipStream_t s, const float *part, float *y, int rows, int n, int slices, const float *bias, const float *res, unsigned cus) {
    const int count = rows * n;
    const unsigned need = (unsigned)((count + 255) / 256), cap = cus * 8;  // (eight workgroups of four waves fill a CU)
    hipLaunchKernelGGL(rows_join_kernel, dim3(need < cap ? need : cap), dim3(256), 0, s, part, y, count, n, slices, bias, res);
}

}  // namespace jitnn
