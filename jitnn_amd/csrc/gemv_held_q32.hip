// gemv_held_kernel for the formats of 32-value blocks.
#include "gemv_held_launch.h"

namespace jitnn {

KernelRef gemv_held_kernel_q32(int fmt, int groups_held) {
    switch (fmt) {
    case F_Q4_0: return held_ref<F_Q4_0>(groups_held);
    case F_Q4_1: return held_ref<F_Q4_1>(groups_held);
    case F_Q8_0: return held_ref<F_Q8_0>(groups_held);
    case F_Q5_1: return held_ref<F_Q5_1>(groups_held);
    default: return {nullptr, 0};
    }
}

}  // namespace jitnn
