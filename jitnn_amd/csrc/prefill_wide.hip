// prefill_wide_kernel and the pass that dequantises its weights.
#include "prefill_wide.h"

namespace jitnn {

template <bool DUAL, int RT>
static constexpr size_t wide_lds() { return (size_t)PW_STAGES * (RT + 8) * 2048; }

KernelRef prefill_wide_kernel_ref(bool dual, int rt) {
    if (dual) return rt == 8 ? KernelRef{(const void *)prefill_wide_kernel<true, 8>, wide_lds<true, 8>()} : KernelRef{nullptr, 0};
    switch (rt) {
    case 8: return {(const void *)prefill_wide_kernel<false, 8>, wide_lds<false, 8>()};
    case 6: return {(const void *)prefill_wide_kernel<false, 6>, wide_lds<false, 6>()};
    case 4: return {(const void *)prefill_wide_kernel<false, 4>, wide_lds<false, 4>()};
    default: return {nullptr, 0};
    }
}

void prefill_wide_launch(bool dual, int rt, hipStream_t s, const PwArgs &a) {
    const dim3 grid((unsigned)a.tiles_n * (unsigned)a.tiles_m), block(PW_THREADS);
    if (dual) hipLaunchKernelGGL((prefill_wide_kernel<true, 8>), grid, block, (wide_lds<true, 8>()), s, a);
    else if (rt == 8) hipLaunchKernelGGL((prefill_wide_kernel<false, 8>), grid, block, (wide_lds<false, 8>()), s, a);
    else if (rt == 6) hipLaunchKernelGGL((prefill_wide_kernel<false, 6>), grid, block, (wide_lds<false, 6>()), s, a);
    else hipLaunchKernelGGL((prefill_wide_kernel<false, 4>), grid, block, (wide_lds<false, 4>()), s, a);
}

void wide_dequant_launch(int fmt, hipStream_t s, const uint8_t *W, _Float16 *wo, int n, int k, int half) {
    const dim3 grid((n + 31) / 32, (k + 1023) / 1024), block(256);
    switch (fmt) {
    case F_Q4_0: hipLaunchKernelGGL(wide_dequant_kernel<F_Q4_0>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q4_1: hipLaunchKernelGGL(wide_dequant_kernel<F_Q4_1>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q8_0: hipLaunchKernelGGL(wide_dequant_kernel<F_Q8_0>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q5_1: hipLaunchKernelGGL(wide_dequant_kernel<F_Q5_1>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q4_K: hipLaunchKernelGGL(wide_dequant_kernel<F_Q4_K>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q5_K: hipLaunchKernelGGL(wide_dequant_kernel<F_Q5_K>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q6_K: hipLaunchKernelGGL(wide_dequant_kernel<F_Q6_K>, grid, block, 0, s, W, wo, n, k, half); break;
    case F_Q2_K: hipLaunchKernelGGL(wide_dequant_kernel<F_Q2_K>, grid, block, 0, s, W, wo, n, k, half); break;
    default: break;
    }
}

}  // namespace jitnn
