// gemv_rows_kernel: the formats it is built for, and which launches are gemv_held_kernel's instead.
#include <algorithm>

#include "gemv_held.h"
#include "tu.h"

namespace jitnn {

bool gemv_rows_supported(int fmt) { return gemv_rows_layout(fmt) >= 0; }

size_t gemv_rows_scratch_bytes(int rows, int k) {
    const int groups = (rows + 7) / 8;
    return gemv_rows_ops_bytes(groups, k) + gemv_rows_inv_bytes(groups, k);
}


// Two tiles per wave where that still gives every CU a workgroup - and, for many groups of activation rows, where it gives
// every other CU one: two tiles share the activation operands, which are what the launch waits for, and the idle half of the
// device takes a share of the groups (below).  4096 x 14336 at 40 rows, one tile against two: Q6_K 81.1 / 53.9 us, Q4_K 42.4 /
// 35.7, Q5_K 44.3 / 40.6, Q4_1 42.4 / 38.1; 4096 x 4096 Q4_K 18.9 / 17.3 - at 24 rows they are level or the single tile ahead
// (Q5_K 33.1 / 35.0), and Q4_0 and Q8_0 lose up to 40 rows (Q8_0 4096 x 4096 18.8 / 21.1) and gain little at 64: not for those.
// Without the sharing of groups only Q6_K, with its sixteen operands per tile, gains from two tiles on half the CUs (64.9;
// Q4_K 47.0, Q8_0 58.5 against 46.0).
static int tiles_per_wave(int fmt, int n, int k, int rows, unsigned max_blocks) {
    const unsigned pairs = (unsigned)(((n + 15) / 16 + 1) / 2);
    bool half = fmt == F_Q6_K && rows > 16 && k >= 8192;
    if (rows > 32 && k >= 4096 && (fmt == F_Q4_K || fmt == F_Q5_K || fmt == F_Q6_K || fmt == F_Q4_1)) half = true;
    return pairs >= max_blocks || (half && 2 * pairs >= max_blocks) ? 2 : 1;
}

struct RowsGeo {
    int tiles, batches, shares;  // tiles per wave, batches of them, workgroups that share out the groups of rows of one
};
static RowsGeo rows_geometry(int fmt, int n, int k, int rows, unsigned max_blocks) {
    const int T = tiles_per_wave(fmt, n, k, rows, max_blocks), nbatch = ((n + 15) / 16 + T - 1) / T, groups = (rows + 7) / 8;
    // Few tiles: the groups of activation rows are shared out over as many workgroups per tile as the device has room for -
    // each decodes the tile's weights again (the device would idle otherwise) and writes whole outputs of its own rows.
    // 1024 x 4096 at 40 rows: Q6_K 30.0 -> 19.4 us, Q4_K 17.5 -> 13.5; twice as many workgroups as CUs: 23.4, 13.9.
    int gy = 1;
    if ((unsigned)nbatch * 2 <= max_blocks) {
        const int cap = (int)(max_blocks / (unsigned)nbatch), gper = (groups + cap - 1) / cap;
        gy = (groups + gper - 1) / gper;
    }
    return {T, nbatch, gy};
}

template <int FMT>
static KernelRef kernel_ref(bool two) {
    return {two ? (const void *)gemv_rows_kernel<FMT, 2> : (const void *)gemv_rows_kernel<FMT, 1>,
            gemv_rows_lds_bytes(two ? 2 : 1) + gemv_rows_stage_bytes<FMT>(two ? 2 : 1)};
}

KernelRef gemv_rows_kernel_ref(int fmt, int n, int k, int rows, unsigned max_blocks) {
    const bool two = tiles_per_wave(fmt, n, k, rows, max_blocks) == 2;
    switch (fmt) {
    case F_Q4_K: return kernel_ref<F_Q4_K>(two);
    case F_Q5_K: return kernel_ref<F_Q5_K>(two);
    case F_Q6_K: return kernel_ref<F_Q6_K>(two);
    case F_Q4_0: return kernel_ref<F_Q4_0>(two);
    case F_Q4_1: return kernel_ref<F_Q4_1>(two);
    case F_Q8_0: return kernel_ref<F_Q8_0>(two);
    case F_Q5_1: return kernel_ref<F_Q5_1>(two);
    case F_Q2_K: return kernel_ref<F_Q2_K>(two);
    default: return {nullptr, 0};
    }
}

template <int FMT>
static constexpr int layout_of() {
    using R = RTile<FMT>;
    return R::SUMS == 16 ? GR_LAYOUT_SUMS16 : R::HALVES ? GR_LAYOUT_HALVES : GR_LAYOUT_PLAIN;
}

int gemv_rows_layout(int fmt) {
    switch (fmt) {
    case F_Q4_K: return layout_of<F_Q4_K>();
    case F_Q5_K: return layout_of<F_Q5_K>();
    case F_Q6_K: return layout_of<F_Q6_K>();
    case F_Q4_0: return layout_of<F_Q4_0>();
    case F_Q4_1: return layout_of<F_Q4_1>();
    case F_Q8_0: return layout_of<F_Q8_0>();
    case F_Q5_1: return layout_of<F_Q5_1>();
    case F_Q2_K: return layout_of<F_Q2_K>();
    default: return -1;
    }
}

static_assert(GR_LAYOUT_PLAIN == 0 && GR_LAYOUT_SUMS16 == 1 && GR_LAYOUT_HALVES == 2 && GR_LAYOUTS == 3, "RowsPrepareOut is indexed by layout");

void gemv_rows_prepare_launch(hipStream_t s, const float *x, const float *swiglu_up, void *const *scratch, int k, int rows, int slices) {
    const int groups = (rows + 7) / 8, ncol = k / 256;
    RowsPrepareOut o{};
    for (int l = 0; l < GR_LAYOUTS; ++l) {
        if (!scratch[l]) continue;
        o.ops[l] = reinterpret_cast<_Float16 *>(scratch[l]);
        o.inv[l] = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(scratch[l]) + gemv_rows_ops_bytes(groups, k));
    }
    const dim3 grid(ncol, groups);
    if (swiglu_up) hipLaunchKernelGGL(rows_prepare_kernel<true>, grid, dim3(64), 0, s, x, swiglu_up, rows, k, slices, o);
    else hipLaunchKernelGGL(rows_prepare_kernel<false>, grid, dim3(64), 0, s, x, swiglu_up, rows, k, slices, o);
}

template <int FMT>
static void launch(unsigned max_blocks, hipStream_t s, const uint8_t *W, const void *scratch, const float *bias, const float *res, float *y, int n, int k,
                   int rows) {
    const int groups = (rows + 7) / 8;
    const _Float16 *ops = reinterpret_cast<const _Float16 *>(scratch);
    const float *inv = reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(scratch) + gemv_rows_ops_bytes(groups, k));
    const RowsGeo geo = rows_geometry(FMT, n, k, rows, max_blocks);
    const int T = geo.tiles, gy = geo.shares;
    const unsigned blocks = (unsigned)geo.batches < max_blocks ? (unsigned)geo.batches : max_blocks;
    if (T == 2) hipLaunchKernelGGL((gemv_rows_kernel<FMT, 2>), dim3(blocks, gy), dim3(GR_THREADS), gemv_rows_lds_bytes(2) + gemv_rows_stage_bytes<FMT>(2), s, W, ops, inv, n, k, rows, groups, blocks | ((unsigned)gy << 16), bias, res, y);
    else hipLaunchKernelGGL((gemv_rows_kernel<FMT, 1>), dim3(blocks, gy), dim3(GR_THREADS), gemv_rows_lds_bytes(1) + gemv_rows_stage_bytes<FMT>(1), s, W, ops, inv, n, k, rows, groups, blocks | ((unsigned)gy << 16), bias, res, y);
}

void gemv_rows_main_launch(int fmt, unsigned max_blocks, hipStream_t s, const uint8_t *W, const void *scratch, const float *bias, const float *res, float *y,
                           int n, int k, int rows) {
    switch (fmt) {
    case F_Q4_K: launch<F_Q4_K>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q5_K: launch<F_Q5_K>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q6_K: launch<F_Q6_K>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q4_0: launch<F_Q4_0>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q4_1: launch<F_Q4_1>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q8_0: launch<F_Q8_0>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q5_1: launch<F_Q5_1>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    case F_Q2_K: launch<F_Q2_K>(max_blocks, s, W, scratch, bias, res, y, n, k, rows); break;
    default: break;
    }
}


KernelRef gemv_held_kernel_ref(int fmt, int groups_held) {
    return block_values(fmt) == 256 ? gemv_held_kernel_k(fmt, groups_held) : gemv_held_kernel_q32(fmt, groups_held);
}

// Which of the two kernels takes a launch.  An estimate of each, preparation and join included, in us, from the work of a wave - one
// decoded tile of 16 rows and a 256-value column, met by its groups of rows:
//   streaming:  base + long_row k / 4096 + mb (MB of weights) + units (decode T + meet g + meet_tile g T), units = rounds x columns per
//               wave, T tiles
//   held:       base + long_row k / 4096 + mb (MB of weights) + join (sliced) + sums (MB of slices / 4) + start G + steps (decode +
//               meet G + five (G = 5: operands in LDS))
// Fitted at 13228 launches of both kernels (eight formats, 270 shapes of 512 to 31488 rows of 1024 to 20480 values; 9 to 64 rows, and 3 to 8
// on long ones; profiles/linears_9_to_64_rows_both_kernels.txt) by what the choice costs: the time lost on the slower kernel, once and a
// half for launches the held kernel slows down, a fifth of the weight on each estimate's own error.  116 of the 13228 are slower than
// with the streaming kernel by more than 1.5 % and 27 by more than 4 (the worst by 14); the mean gain is 1.08 (Q5_1) to 1.30 (Q6_K), at
// most 0.003 below the better kernel each time.  At 1793 launches of 40 other shapes 65 are slower by more than 1.5 %, 19 by more than 4
// (9 at worst), mean gain 1.12.
// The held kernel wins where the streaming one has no whole round of workgroups (4096 x 14336, 14336 x 4096, rows of odd numbers
// of columns) or decodes much per tile (Q6_K): Q6_K 4096 x 14336 at 12 / 24 / 40 rows 45.2 / 43.1 / 48.8 -> 32.0 / 34.7 / 43.4, Q6_K
// 2000 x 6912 27.9 -> 18.3 (24 rows), Q4_K 14336 x 4096 25.4 -> 23.6, Q4_0 24000 x 2048 26.4 -> 23.5.  It loses where every CU has
// exactly one batch, by its second launch (Q4_K 4096 x 4096 15.6 against 16.2, 8192 x 4096 17.2 against 18.7), and with five groups in the
// formats of 32-value blocks and minima (4096 x 8192 at 40 rows Q4_1 23.7 against 25.2, 14336 x 4096 Q5_1 35.3 against 36.8).
struct RowsCost {
    float s_base, s_decode, s_meet_tile, s_meet, s_long, s_mb;
    float h_base, h_join, h_start, h_decode, h_meet, h_sums, h_long, h_five, h_mb;
};
static const RowsCost &rows_cost(int fmt) {
    static const RowsCost q40 = {8.81f, 1.33f, 0.21f, 0.36f, -0.66f, -0.04f, 7.63f, 3.16f, 0.58f, 1.47f, 0.18f, 4.09f, -0.02f, 0.30f, -0.09f};
    static const RowsCost q41 = {8.75f, 0.63f, 0.17f, 0.51f, -0.07f, 0.02f, 8.22f, 2.75f, 0.85f, 0.97f, 0.15f, 4.23f, -0.01f, 0.53f, -0.08f};
    static const RowsCost q51 = {9.06f, 0.84f, 0.20f, 0.39f, -0.29f, 0.05f, 8.51f, 3.76f, 0.82f, 1.31f, 0.16f, 4.42f, -0.31f, 0.38f, -0.05f};
    static const RowsCost q80 = {8.71f, 1.64f, 0.31f, 0.25f, -1.10f, -0.00f, 6.86f, 3.85f, 0.99f, 1.67f, 0.14f, 3.05f, -0.17f, 0.14f, -0.03f};
    static const RowsCost q2 = {9.70f, 0.46f, 0.00f, 0.76f, -0.11f, 0.02f, 7.96f, 3.42f, 0.69f, 0.94f, 0.13f, 2.17f, -0.17f, 0.24f, -0.09f};
    static const RowsCost q4 = {9.51f, 0.64f, -0.04f, 0.81f, -0.43f, 0.03f, 7.56f, 3.78f, 0.78f, 0.91f, 0.12f, 1.91f, -0.20f, 0.40f, -0.04f};
    static const RowsCost q5 = {9.72f, 0.62f, 0.04f, 0.67f, 0.09f, 0.03f, 8.68f, 3.34f, 0.34f, 1.24f, 0.11f, 3.73f, -0.11f, 0.48f, -0.05f};
    static const RowsCost q6 = {11.24f, 1.21f, -0.59f, 2.01f, -0.01f, 0.05f, 8.88f, 2.77f, 0.23f, 1.80f, 0.23f, 3.59f, 0.81f, 0.34f, -0.05f};
    switch (fmt) {
    case F_Q6_K: return q6;
    case F_Q5_K: return q5;
    case F_Q2_K: return q2;
    case F_Q8_0: return q80;
    case F_Q4_0: return q40;
    case F_Q4_1: return q41;
    case F_Q5_1: return q51;
    default: return q4;
    }
}

// The held kernel's launch, or groups_held = 0: the streaming kernel's.
HeldPlan gemv_held_plan(int fmt, int n, int k, int rows, int join, int cus, int weights) {
    HeldPlan best;
    const RowsCost &cost = rows_cost(fmt);
    const int ncol = k / 256, ntiles = (n + 15) / 16 * weights, groups = (rows + 7) / 8;
    HeldGeo geo;
    geo.slices = (ncol + GR_WAVES - 1) / GR_WAVES;
    geo.cols = (ncol + geo.slices - 1) / geo.slices;
    geo.slices = (ncol + geo.cols - 1) / geo.cols;
    geo.lanes = GR_WAVES / geo.cols;
    if (geo.slices > cus || geo.slices > 4095) return best;
    const int steps = (ntiles + geo.lanes - 1) / geo.lanes, part = geo.slices > 1 || join != HELD_JOIN_SLICES ? geo.slices : 0;
    const RowsGeo st = rows_geometry(fmt, n, k, rows, (unsigned)cus);
    const float units = (float)((st.batches + cus - 1) / cus * ((ncol + GR_WAVES - 1) / GR_WAVES)), gper = (float)((groups + st.shares - 1) / st.shares),
                tiles = (float)st.tiles;
    const float mb = (float)n * 1e-6f * (float)(k / block_values(fmt) * block_bytes(fmt));
    // (a reader's join has no launch: half the line's join.  432 prompts of 9 to 64 tokens through 24 models, against the streaming kernel
    // alone: the worst is 0.997 times as fast, the mean 1.20; with all of it, three quarters or a quarter 0.1 % less)
    const float launch = join == HELD_JOIN_READER ? 0.5f : 1.f;
    // (a pair of streaming launches is taken at twice one: the preparation they share is paid by their second round of CUs; the
    // estimates err by a few per cent: a launch changes kernels for three)
    float best_us = 0.97f * (float)weights * (cost.s_base + cost.s_long * k / 4096.f + cost.s_mb * mb + units * (cost.s_decode * tiles + cost.s_meet * gper + cost.s_meet_tile * gper * tiles));
    for (int shares = 1; shares <= groups; ++shares) {
        const int held = (groups + shares - 1) / shares;
        if (held > GH_G_MAX || (groups + held - 1) / held != shares || geo.slices * shares > cus) continue;
        const int per_slice = std::min({cus / (geo.slices * shares), steps, 4095}), walk = (steps + per_slice - 1) / per_slice;
        const float us = cost.h_base + cost.h_long * k / 4096.f + cost.h_mb * mb * weights + (part ? cost.h_join * launch + cost.h_sums * 1e-6f * part * rows * n * weights : 0.f) +
                         cost.h_start * held + walk * (cost.h_decode + cost.h_meet * held + (held == 5 ? cost.h_five : 0.f));
        if (us < best_us) {
            best_us = us;
            geo.per_slice = (steps + walk - 1) / walk;
            best.groups_held = held;
            best.shares = shares;
            best.slices = geo.slices;
            best.per_slice = geo.per_slice;
            best.part = part;
            best.where = geo.packed();
        }
    }
    return best;
}

static void held_launch(const HeldPlan &plan, int fmt, hipStream_t s, unsigned blocks, const uint8_t *W, const uint8_t *W2, const void *scratch, int first_column,
                        uint32_t where, float *y, int n, int k, int rows) {
    int groups = (rows + 7) / 8;
    const _Float16 *ops = reinterpret_cast<const _Float16 *>(scratch) + (size_t)first_column * GR_OP_HALVES;
    const float *inv = reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(scratch) + gemv_rows_ops_bytes(groups, k)) + (size_t)first_column * 8;
    const KernelRef kr = gemv_held_kernel_ref(fmt, plan.groups_held);
    W += (size_t)first_column * (256 / block_values(fmt)) * block_bytes(fmt);
    void *args[] = {&W, &W2, &ops, &inv, &n, &k, &rows, &groups, &where, &y};
    (void)hipLaunchKernel(kr.fn, dim3(blocks, (unsigned)plan.shares), dim3(GR_THREADS), args, kr.lds, s);
}

void gemv_held_slices_launch(const HeldPlan &plan, int fmt, hipStream_t s, const uint8_t *W, const uint8_t *W2, const void *scratch, float *part, int n, int k,
                             int rows) {
    held_launch(plan, fmt, s, (unsigned)(plan.slices * plan.per_slice), W, W2, scratch, 0, plan.where, part, n, k, rows);
}

void gemv_held_launch(const HeldPlan &plan, int fmt, int cus, hipStream_t s, const uint8_t *W, const void *scratch, const float *bias, const float *res,
                      float *y, float *part, int n, int k, int rows) {
    if (plan.part && !part) {  // slice after slice into y: the order, and so the bits, of the join
        HeldGeo geo = HeldGeo::unpacked(plan.where);
        const int cols = geo.cols;
        for (int z = 0; z < plan.slices; ++z) {
            geo.cols = std::min(cols, k / 256 - z * cols);
            geo.slices = z == 0;
            held_launch(plan, fmt, s, (unsigned)plan.per_slice, W, nullptr, scratch, z * cols, geo.packed(), y, n, k, rows);
        }
        rows_join_launch(s, y, y, rows, n, 1, bias, res, (unsigned)cus);
        return;
    }
    gemv_held_slices_launch(plan, fmt, s, W, nullptr, scratch, plan.part ? part : y, n, k, rows);
    if (plan.part) rows_join_launch(s, part, y, rows, n, plan.slices, bias, res, (unsigned)cus);
}

}  // namespace jitnn
