// Many-row linear for long calls (more than 512 rows): y[M, N] = x[M, K] W[N, K]^T in two passes.
//   1. wide_dequant_kernel writes the weights once per call as FP16 in matrix-core operand order (the decoders, and so the
//      values, are those of prefill.h), 2 bytes per value into the calling thread's scratch;
//   2. prefill_wide_kernel is then a plain FP16 product: both operands go from memory straight into LDS.
// prefill_mfma_kernel decodes a weight once per 256 tokens, in the instruction stream of its one wave per SIMD; here a
// weight is decoded once, and the product has no vector arithmetic left in its loop.  What the first pass costs (2.6 bytes
// moved per value: 37 us for a Q4_K 14336 x 4096 weight) is paid back where wide_pays estimates it to be: from 513 rows on for a
// single weight that fills the chip, from 1025 (down) to 1875 (attn_o) rows on in an 8B layer, for its gate / up in ranges above 2048.
#pragma once
#include "common.h"
#include "prefill.h"
#include "tu.h"

#include <type_traits>

namespace jitnn {

constexpr int PW_TM = 256, PW_STAGES = 4, PW_THREADS = 512;

// W [n, k] -> wo: 1 KiB pieces [32-row block][K step of 16][lane][8], lane l holding row 32 rb + l % 32, values
// 16 ks + 8 (l / 32) .. + 7 in the order 0, 2, 1, 3 of each group of four (as x_to_operand_kernel stores the activations).
// grid (32-row blocks, ceil(K / 1024)), a wave takes 32 rows x 256 values: the lanes of a store write 512 consecutive
// bytes, and the loads - 32 rows a stride apart - use up their cache lines within the wave.  Bound by memory, four
// fifths of it stores: 4.1 TB/s moved on Q4_K, 3.1 on Q6_K (14336 x 4096 values; a large copy: 5.2).  half >= 0: the row blocks of a gate (0) and an up (1) weight alternate in
// pairs, as the dual form of the product wants them.  Values past the end of a row repeat its last ones and meet zeros.
template <int FMT>
__global__ void __launch_bounds__(256) wide_dequant_kernel(const uint8_t *__restrict__ W, _Float16 *__restrict__ wo, int n, int k, int half) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, dhalf = lane >> 5;
    const int rb = blockIdx.x, nsteps = (k + PF_BK - 1) / PF_BK, s0 = (blockIdx.y * 4 + wave) * 4;
    const uint8_t *row = W + (size_t)min(32 * rb + r, n - 1) * ((size_t)(k / block_values(FMT)) * block_bytes(FMT));
    const int drb = half < 0 ? rb : (rb >> 2) * 8 + ((rb >> 1) & 1) * 4 + (rb & 1) + 2 * half;
    f16x8 *dst = reinterpret_cast<f16x8 *>(wo) + (size_t)drb * pf_ksteps(k) * 64 + r;
    PfRaw<FMT> raw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) pf_load<FMT>(raw[i], row, min(min(s0 + i, nsteps - 1) * PF_BK + 32 * dhalf, k - 32));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (s0 + i >= nsteps) break;
        const int kk = min((s0 + i) * PF_BK + 32 * dhalf, k - 32);
        f16x8 o[4];
        if constexpr (pf_packed(FMT)) {
            pf_decode_h<FMT>(raw[i], kk, o);
        } else {
            float v[32];
            pf_decode<FMT>(raw[i], kk, v);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) o[c][(e & ~3) | pf_perm4(e & 3)] = (_Float16)v[8 * c + e];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) dst[(size_t)((s0 + i) * 4 + 2 * dhalf + (c >> 1)) * 64 + 32 * (c & 1)] = o[c];
    }
}

// one 1 KiB operand piece from memory straight into LDS (16 bytes a lane, consecutive lanes consecutive in LDS)
__device__ __forceinline__ void pw_dma(const void *g, _Float16 *l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g, (__attribute__((address_space(3))) void *)l, 16, 0, 0);
}

// A workgroup of eight waves takes 32 RT weight rows x 256 tokens, wave w the rows [16 RT (w / 4), +16 RT) and the tokens
// [64 (w % 4), +64).  K goes by in steps of 32 through four LDS stages (up to 128 KiB), a step's pieces requested three and a
// half steps ahead; every piece of an operand is 1 KiB of consecutive bytes in memory and in LDS.
//   * one barrier per step, in its middle: it says that the next step has arrived and that this one has been read.  The
//     operands of the first half of a step's products are read under the second half of the step before, those of the second
//     half under the first - no product waits for a read just issued.
//   * v_mfma_f32_16x16x32_f16 and not 32x32x16: with operands that toggle the chip is held by its power, and the smaller tile
//     with the longer K moves half the accumulator bytes per multiply-add.  Products alone, normal operands: 1990 against 1740
//     TFLOP/s (zeros: 2440 and 2470).  This kernel on 4096 x 14336 x 4096 tokens: 1380, on zero activations 1840; the matrix
//     cores are busy 82 % of its cycles, at 1.6 GHz.
// RT = 8 where its tiles fill the device, 6 and 4 for launches whose last round would be half empty (wide_plan).  DUAL: as in
// prefill_mfma_body; a wave's first RT / 2 tiles of rows are gate rows, the others the same rows of the up weight.
template <bool DUAL, int RT>
__global__ void __launch_bounds__(PW_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) prefill_wide_kernel(const PwArgs a) {
    extern __shared__ __align__(16) uint8_t pf_smem[];
    _Float16 *sm = reinterpret_cast<_Float16 *>(pf_smem);  // [stage][RT row blocks, 8 token blocks][2][512]
    constexpr int TN = 32 * RT, PIECE = 512, SIDE = RT * 2 * PIECE, STAGE = SIDE + 8 * 2 * PIECE;
    constexpr int WC = 4, TT = 4, NA = RT == 4 ? 1 : 2, NB = 2;  // waves along the tokens, 16-token tiles per wave, pieces a wave copies per step
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / WC, wc = wave % WC;
    // ---- which tile: workgroup i runs on XCD i % 8; each XCD takes a run of consecutive tiles, eight row tiles by the token
    // tiles, so that the 32 tiles it works on at a time share operands in its L2 (8 x 4 against 4 x 8: 1 to 3 % faster)
    const int total = a.tiles_n * a.tiles_m, xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
    const int lin = xcd * q8 + min(xcd, r8) + (blockIdx.x >> 3);
    const int gsz = 8 * a.tiles_m, grp = lin / gsz, in = lin - grp * gsz, gh = min(8, a.tiles_n - 8 * grp);
    const int tm = in / gh, tn = 8 * grp + in - tm * gh;
    const int nst = a.ksteps >> 1;                // K steps of 32, an even number
    const size_t blk = (size_t)a.ksteps * PIECE;  // halves per 32-row block
    const int ra = RT == 4 ? wave >> 1 : min(wave, RT - 1);  // (RT = 6: two waves repeat the last block's copy, the same bytes to the same place)
    const int pa = RT == 4 ? (wave & 1) * PIECE : 0;
    const _Float16 *ga = a.wo + (size_t)(RT * tn + ra) * blk + pa + 8 * lane, *gb = a.xo + (size_t)(8 * tm + wave) * blk + 8 * lane;
    auto dma_a = [&](int s) {
        _Float16 *d = sm + (s & (PW_STAGES - 1)) * STAGE + ra * 2 * PIECE + pa;
        const size_t off = (size_t)min(s, nst - 1) * 2 * PIECE;
#pragma unroll
        for (int i = 0; i < NA; ++i) pw_dma(ga + off + i * PIECE, d + i * PIECE);
    };
    auto dma_b = [&](int s) {
        _Float16 *d = sm + (s & (PW_STAGES - 1)) * STAGE + SIDE + wave * 2 * PIECE;
        const size_t off = (size_t)min(s, nst - 1) * 2 * PIECE;
#pragma unroll
        for (int i = 0; i < NB; ++i) pw_dma(gb + off + i * PIECE, d + i * PIECE);
    };
    f32x4 acc[RT][TT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    f16x8 fa[2][RT / 2], fb[2][TT];
    // a 16 x 32 operand out of two 1 KiB pieces [k / 8][32 rows][8]: lane l takes row l % 16 (+ 16), values 8 (l / 16) .. + 7
    const int lo = (lane >> 4) * 256 + (lane & 15) * 8;
    auto read_a = [&](int h, int s) {
        const _Float16 *p = sm + (s & (PW_STAGES - 1)) * STAGE + wr * (RT / 2) * 2 * PIECE + lo;
#pragma unroll
        for (int i = h * (RT / 2); i < (h + 1) * (RT / 2); ++i) fa[h][i - h * (RT / 2)] = *reinterpret_cast<const f16x8 *>(p + (i >> 1) * 2 * PIECE + (i & 1) * 128);
    };
    auto read_b = [&](int set, int s) {
        const _Float16 *p = sm + (s & (PW_STAGES - 1)) * STAGE + SIDE + (TT / 2) * wc * 2 * PIECE + lo;
#pragma unroll
        for (int j = 0; j < TT; ++j) fb[set][j] = *reinterpret_cast<const f16x8 *>(p + (j >> 1) * 2 * PIECE + (j & 1) * 128);
    };
    auto mul = [&](int h, int set) {
#pragma unroll
        for (int i = 0; i < RT / 2; ++i)
#pragma unroll
            for (int j = 0; j < TT; ++j)
                acc[(RT / 2) * h + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[h][i], fb[set][j], acc[(RT / 2) * h + i][j], 0, 0, 0);
    };
    constexpr auto vm = [](int rest, int n) { return rest | (n & 15) | ((n >> 4) << 14); };
    auto interleave = [](auto nread, auto ndma) {
        constexpr int NR = decltype(nread)::value, ND = decltype(ndma)::value, NM = RT / 2 * TT;
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            if (i < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            else if (i < NR + ND) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
    };
    using std::integral_constant;
    auto step = [&](int s, int set) {
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_sched_barrier(0);
        read_a(1, s);
        dma_b(s + 3);
        mul(0, set);
        interleave(integral_constant<int, RT / 2>{}, integral_constant<int, NB>{});
        __builtin_amdgcn_sched_barrier(0);
        // step s + 1 has arrived and step s has been read, in every wave
        __builtin_amdgcn_s_waitcnt(vm(0x0070, 2 * (NA + NB)));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        read_b(set ^ 1, s + 1);
        read_a(0, s + 1);
        dma_a(s + 4);
        mul(1, set);
        interleave(integral_constant<int, RT / 2 + TT>{}, integral_constant<int, NA>{});
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        dma_a(s);
        dma_b(s);
    }
    dma_a(3);
    __builtin_amdgcn_s_waitcnt(vm(0x0f70, 2 * (NA + NB) + NA));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_b(0, 0);
    read_a(0, 0);
    for (int s = 0; s < nst; s += 2) {
        step(s, 0);
        step(s + 1, 1);
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // nothing may still be on its way into this workgroup's LDS
    // ---- epilogue
    int seg = 0, row0 = tn * TN;
    if constexpr (!DUAL) {
        if (tn >= a.tile0[1]) seg = tn >= a.tile0[2] ? 2 : 1;
        row0 = (tn - a.tile0[seg]) * TN;
    }
    const int n = a.n[seg], m = a.m, tok0 = tm * PW_TM + 16 * TT * wc + (lane & 15), r0 = 4 * (lane >> 4);
    float *y = a.y[seg];
    const float *bias = a.bias, *res = a.res;
    float isc[TT];
#pragma unroll
    for (int j = 0; j < TT; ++j) isc[j] = a.inv_scale[min(tok0 + 16 * j, m - 1)];
    auto finish = [&](auto whole) {
        constexpr bool WHOLE = decltype(whole)::value;
#pragma unroll
        for (int i = 0; i < (DUAL ? RT / 2 : RT); ++i) {
            const int row = DUAL ? tn * (TN / 2) + TN / 4 * wr + 16 * i + r0 : row0 + TN / 2 * wr + 16 * i + r0;
            f32x4 bv = {0.f, 0.f, 0.f, 0.f};
            if (!DUAL && bias) {
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[e] = bias[min(row + e, n - 1)];
            }
            f32x4 v[TT];
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                if constexpr (DUAL) {
                    auto sw = [](float g, float u) { return (g / (1.f + __expf(-g))) * u; };
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[j][e] = sw(acc[i][j][e] * isc[j], acc[i + RT / 2][j][e] * isc[j]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[j][e] = acc[i][j][e] * isc[j] + bv[e];
                }
            }
            if (!DUAL && res) {
                f32x4 rv[TT];
#pragma unroll
                for (int j = 0; j < TT; ++j) {
                    if constexpr (WHOLE) rv[j] = *reinterpret_cast<const f32x4 *>(res + (size_t)(tok0 + 16 * j) * n + row);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) rv[j][e] = res[(size_t)min(tok0 + 16 * j, m - 1) * n + min(row + e, n - 1)];
                    }
                }
#pragma unroll
                for (int j = 0; j < TT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[j][e] = v[j][e] + rv[j][e];
            }
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                float *yp = y + (size_t)(tok0 + 16 * j) * n + row;
                if constexpr (WHOLE) *reinterpret_cast<f32x4 *>(yp) = v[j];
                else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (row + e < n && tok0 + 16 * j < m) yp[e] = v[j][e];
                }
            }
        }
    };
    if (tm * PW_TM + PW_TM <= m && (n & 3) == 0 && (DUAL ? (tn + 1) * (TN / 2) : row0 + TN) <= n) finish(std::true_type{});
    else finish(std::false_type{});
}

}  // namespace jitnn
