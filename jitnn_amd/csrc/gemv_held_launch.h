// The variants of gemv_held_kernel of a format, by the groups of eight rows a wave holds.
#pragma once
#include "gemv_held.h"
#include "tu.h"

namespace jitnn {

template <int FMT>
static KernelRef held_ref(int groups_held) {
    switch (groups_held) {
    case 1: return {(const void *)gemv_held_kernel<FMT, 1>, gemv_held_lds_bytes<FMT>(1)};
    case 2: return {(const void *)gemv_held_kernel<FMT, 2>, gemv_held_lds_bytes<FMT>(2)};
    case 3: return {(const void *)gemv_held_kernel<FMT, 3>, gemv_held_lds_bytes<FMT>(3)};
    case 4: return {(const void *)gemv_held_kernel<FMT, 4>, gemv_held_lds_bytes<FMT>(4)};
    case 5: return {(const void *)gemv_held_kernel<FMT, 5>, gemv_held_lds_bytes<FMT>(5)};
    default: return {nullptr, 0};
    }
}

}  // namespace jitnn
