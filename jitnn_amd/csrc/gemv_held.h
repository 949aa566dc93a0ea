// 9..64 activation rows (3..64 of rows of 12288 values and more) against raw GGUF blocks with the ACTIVATION operands held in registers: the main kernel of
// gemv_rows.h (same operands from rows_prepare_kernel, same decoders RTile, same FP32-grade products) with the roles of what
// stays and what streams exchanged.
//
// gemv_rows_kernel holds two tiles of decoded weights and streams the activation operands past them, 9 KiB per group of eight
// rows, column and pair of tiles: at 40 rows of a 14336 x 4096 weight 330 MB through the L1s against 33 MB of weights, and that
// is its time.  Here wave w of a workgroup owns one 256-value column of K for the kernel's life and keeps that column's
// operands - hi and lo part of every row and the block sums, 36 registers per group of eight rows - while the workgroup walks
// tiles of 16 weight rows: it fetches and decodes its 16 x 256 piece, runs it against its G groups and leaves the sums in LDS,
// where the workgroup's waves are added up in wave order.  An operand is read once per workgroup instead of once per pair of
// tiles, and a wave's G chains of products are independent of one another.  Rows longer than the workgroup's columns are cut
// into slices of K, workgroups of their own; their sums meet in rows_join_kernel, or in the kernel that reads them next, in slice
// order (no atomics).
// What bounds it: the vector instructions of a step - decoding about 170 of them per 16 x 256 tile of Q4_K, folding 10 per group;
// 0.8 to 1.8 us by format and 0.2 to 0.4 us per group for the two waves of a SIMD - and per launch 0.6 to 0.9 us per group for the
// operands' way into the registers.  Q4_K 14336 x 4096 at 40 rows: 20 us, seven steps.  A second step's weights under way (9 to 17
// more registers) measured the same or, spilling, slower.
#pragma once
#include "gemv_rows.h"

namespace jitnn {

constexpr int GH_WAIT_VMCNT0 = 0x0f70;  // s_waitcnt vmcnt(0): no wait on the other counters (gfx9 encoding)
constexpr int GH_G_MAX = 5;  // groups of eight rows a wave holds at most: 36 registers each of the 256 a wave has at two per SIMD
// At five groups an operand or two wait in LDS instead - the block sums', one product in nine to seventeen, and for Q6_K, whose
// decoder holds twice the weight operands, the last sub-block's: 13 to 32 registers spilled otherwise.
__host__ __device__ constexpr int gh_ops_in_lds(int fmt, int groups_held) { return groups_held < 5 ? 0 : fmt == F_Q4_K || fmt == F_Q2_K ? 1 : 2; }

template <int FMT>
__host__ __device__ constexpr size_t gemv_held_lds_bytes(int groups_held) {
    return 2 * (size_t)GR_WAVES * groups_held * 64 * sizeof(float2) + gemv_rows_stage_bytes<FMT>(1) +
           (size_t)gh_ops_in_lds(FMT, groups_held) * GR_WAVES * groups_held * 1024;
}

// whether the request for the next weights is kept from being scheduled late (36 -> 35 us, Q4_K 14336 x 4096 at 64 rows); where
// registers are short that spills some
__host__ __device__ constexpr bool gh_pin_fetch(int fmt, int groups_held) { return groups_held < 5 && !(fmt == F_Q6_K && groups_held == 4); }

// Where the workgroups of a launch work; one dword to the kernel, with the arguments that are preloaded.
struct HeldGeo {
    int cols;       // columns of K per workgroup, one per wave: 1..8
    int lanes;      // tiles a workgroup works on side by side: its waves are `lanes` sets of cols (cols * lanes <= 8)
    int slices;     // slices of K: ceil(k / 256 / cols); 0: the one slice of this launch, added to y
    int per_slice;  // workgroups per slice: gridDim.x = slices * per_slice
    __host__ __device__ uint32_t packed() const { return (uint32_t)cols | (uint32_t)lanes << 4 | (uint32_t)slices << 8 | (uint32_t)per_slice << 20; }
    __host__ __device__ static HeldGeo unpacked(uint32_t v) { return {(int)(v & 15u), (int)(v >> 4 & 15u), (int)(v >> 8 & 4095u), (int)(v >> 20)}; }
};

// y[slice][b, row] = sum over the slice's k of W[row, k] x[b, k], for the rows b of this workgroup's G groups (blockIdx.y);
// k a multiple of 256 - or, blocks of 32 values, the whole columns of any row of those -, n >= 16, per_slice at most the number of steps.  A bias and a residual are rows_join_kernel's: loads here would be waited for with the weights.
template <int FMT, int G>
__global__ void __launch_bounds__(GR_THREADS) gemv_held_kernel(const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2, const _Float16 *__restrict__ ops, const float *__restrict__ inv,
                                                                int n, int k, int rows, int groups, const uint32_t where, float *__restrict__ y) {
    typedef RTile<FMT> R;
    constexpr int NOPS = R::NOPS;
    const HeldGeo geo = HeldGeo::unpacked(where);
    extern __shared__ __attribute__((aligned(16))) uint8_t gh_smem[];
    float2 *red = reinterpret_cast<float2 *>(gh_smem);  // [buffer][wave][group][lane]
    constexpr int BUF = GR_WAVES * G * 64;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *stage = gh_smem + 2 * (size_t)BUF * sizeof(float2) + (size_t)wave * R::STAGE_BYTES;
    constexpr int PARKED = gh_ops_in_lds(FMT, G), HELD = 9 - PARKED;  // operands of a group in LDS, in registers
    f16x8 *parked = reinterpret_cast<f16x8 *>(gh_smem + 2 * (size_t)BUF * sizeof(float2) + gemv_rows_stage_bytes<FMT>(1)) + wave * PARKED * G * 64 + lane;
    const int ncol = k >> 8, each = (n + 15) >> 4, ntiles = W2 ? 2 * each : each, nsteps = (ntiles + geo.lanes - 1) / geo.lanes;
    const size_t rowbytes = (size_t)(k / block_values(FMT)) * block_bytes(FMT);
    const int slice = (int)blockIdx.x / geo.per_slice, first = (int)blockIdx.x - slice * geo.per_slice;
    const int c0 = slice * geo.cols, cols = min(geo.cols, ncol - c0);  // (the last slice may be short)
    const int tl = wave / geo.cols, c = c0 + wave - tl * geo.cols;
    const bool works = tl < geo.lanes && c < ncol;  // wave-uniform
    const int g0 = (int)blockIdx.y * G;

    // the last tile of a ragged matrix is the last 16 rows: in bounds, its first rows computed twice, stored once
    typename R::Raw raw;
    auto fetch = [&](int step) {
        const int t = min(step * geo.lanes + tl, ntiles - 1), second = t >= each;
        R::load(raw, R::ptr(second ? W2 : W, min((second ? t - each : t) * 16, n - 16), rowbytes, lane), c);
    };
    f16x8 A[G][HELD];
    float2 iv[G];
    if (works) {
        fetch(first);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int gg = min(g0 + g, groups - 1);  // (groups past the last: computed, not stored)
            const _Float16 *op = ops + ((size_t)gg * ncol + c) * GR_OP_HALVES + lane * 8;
#pragma unroll
            for (int s = 0; s < 9; ++s) {
                if (s == 8 && !R::MINS) continue;
                const f16x8 v = *reinterpret_cast<const f16x8 *>(op + s * 512);
                if (s < HELD) A[g][s < HELD ? s : 0] = v;
                else parked[(g * PARKED + s - HELD) * 64] = v;  // (read by this lane alone)
            }
            iv[g] = *reinterpret_cast<const float2 *>(inv + ((size_t)gg * ncol + c) * 8 + 2 * kq);
        }
    }
    auto operand = [&](int g, int s) { return s < HELD ? A[g][s < HELD ? s : 0] : parked[(g * PARKED + s - HELD) * 64]; };
    float *ys = y + (size_t)slice * rows * n;
    const bool adds_up = geo.slices == 0;
    // the sums of a step, added up in wave order and stored: (tile, group) tg by wave tg % 8
    auto join = [&](int step, int buf) {
        for (int tg = wave; tg < geo.lanes * G; tg += GR_WAVES) {
            const int t = tg / G, g = tg - t * G, at = step * geo.lanes + t, second = at >= each, tile = second ? at - each : at;
            const float2 *p = red + buf * BUF + (t * geo.cols * G + g) * 64 + lane;
            float2 v[GR_WAVES];
#pragma unroll
            for (int w = 0; w < GR_WAVES; ++w) v[w] = p[min(w, cols - 1) * G * 64];
            float2 sum = v[0];
#pragma unroll
            for (int w = 1; w < GR_WAVES; ++w) {
                sum.x += w < cols ? v[w].x : 0.f;
                sum.y += w < cols ? v[w].y : 0.f;
            }
            const int row = min(tile * 16, n - 16) + (lane & 15), b = (g0 + g) * 8 + 2 * kq;
            if (at < ntiles && row >= tile * 16) {  // rows of a ragged last tile that an earlier tile already wrote are skipped
                float *to = ys + ((size_t)(second ? geo.slices : 0) * rows + b) * n + row;
                if (adds_up) {
                    if (b < rows) to[0] += sum.x;
                    if (b + 1 < rows) to[n] += sum.y;
                } else {
                    if (b < rows) to[0] = sum.x;
                    if (b + 1 < rows) to[n] = sum.y;
                }
            }
        }
    };
    int buf = 0;
    for (int step = first; step < nsteps; step += geo.per_slice, buf ^= 1) {
        if (works) {
            // The weights requested a step ago, and before the first step the operands, have arrived.  Said here, all at once: the
            // compiler's own waits - for the last operand at its first product, for a chunk that only some lanes use - stand
            // behind later requests, and one counter, in order, makes them waits for those too.
            __builtin_amdgcn_s_waitcnt(GH_WAIT_VMCNT0);
            f16x8 B[NOPS], Bm;
            float d = 0.f, dmin64 = 0.f;
            float dblk[8];
            const uint8_t *row = R::park(raw, stage, lane);
            const uint32_t tail = raw.tail;
            // the step before is joined here, in front of the request for the next weights: the wait for those is then not one
            // for its stores
            if (step != first) join(step - geo.per_slice, buf ^ 1);
            if (step + geo.per_slice < nsteps) fetch(step + geo.per_slice);
            // (not later, as the scheduler would have it - but where registers are short, which it then runs out of)
            if constexpr (gh_pin_fetch(FMT, G)) __builtin_amdgcn_sched_barrier(0);
            if constexpr (R::BLOCK_SCALES) {
                R::decode(row, tail, lane, B, Bm, dblk);
            } else {
                float dm;
                R::decode(row, tail, lane, B, Bm, d, dm);
                dmin64 = dm * 64.f;
            }
            float2 *mine = red + buf * BUF + wave * G * 64 + lane;
            if constexpr (R::BLOCK_SCALES) {
                float u0[G], u1[G];
#pragma unroll
                for (int g = 0; g < G; ++g) u0[g] = u1[g] = 0.f;
#pragma unroll
                for (int s = 0; s < 8; ++s) {
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const f32x4 cs = mfma16(operand(g, s), B[s]);
                        u0[g] = __builtin_fmaf(dblk[s], cs[0] + cs[1], u0[g]);
                        u1[g] = __builtin_fmaf(dblk[s], cs[2] + cs[3], u1[g]);
                    }
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if constexpr (R::MINS) {
                        const f32x4 cm = mfma16(operand(g, 8), Bm);
                        u0[g] = __builtin_fmaf(64.f, cm[0] + cm[1], u0[g]);
                        u1[g] = __builtin_fmaf(64.f, cm[2] + cm[3], u1[g]);
                    }
                    mine[g * 64] = make_float2(iv[g].x * u0[g], iv[g].y * u1[g]);
                }
            } else {
                f32x4 cs[G];
#pragma unroll
                for (int g = 0; g < G; ++g) cs[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < NOPS; ++s) {
#pragma unroll
                    for (int g = 0; g < G; ++g) cs[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(g, R::aidx(s)), B[s], cs[g], 0, 0, 0);
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const f32x4 cm = mfma16(operand(g, 8), Bm);
                    const float s0 = cs[g][0] + cs[g][1], s1 = cs[g][2] + cs[g][3], m0 = cm[0] + cm[1], m1 = cm[2] + cm[3];
                    const float u0 = __builtin_fmaf(d, s0, -dmin64 * m0), u1 = __builtin_fmaf(d, s1, -dmin64 * m1);
                    mine[g * 64] = make_float2(iv[g].x * u0, iv[g].y * u1);
                }
            }
        } else if (step != first) {
            join(step - geo.per_slice, buf ^ 1);
        }
        // one barrier per step: the sums of the next step go to the other buffer, and a wave writes this one again only behind
        // the next barrier, which every wave reaches after reading this one
        __syncthreads();
    }
    join(first + (nsteps - 1 - first) / geo.per_slice * geo.per_slice, buf ^ 1);
}

}  // namespace jitnn
