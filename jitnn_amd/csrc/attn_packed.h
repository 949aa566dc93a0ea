// Causal attention of long prompts on keys and values packed as FP16 matrix-core operands beforehand, for heads of 64 or 128 values.
//
// attn_prefill_mfma_kernel (glue.h) converts and transposes 64 keys and values per chunk in every workgroup: at 4096 tokens each of
// them 128 times a layer.  Here attn_pack_kernel does it once per layer, for all positions the prompt sees, and
// attn_packed_kernel moves a chunk's 2 x 64 x D halves from memory straight into LDS.  What that frees - the registers of the requests under
// way, the conversions, the transposing stores - lets a wave take two tiles of 16 rows against ALL 64 keys of a chunk, not
// against half of them: the running maximum, and with it the rescaling of the output, is paid once per 64 keys.
#pragma once
#include <type_traits>

#include "common.h"

namespace jitnn {

constexpr int AP_CH = 64;                                // keys per chunk
constexpr int AP_WAVES = 4, AP_THREADS = 64 * AP_WAVES;  // a wave takes AP_RT tiles of 16 rows
constexpr int AP_RT = 2, AP_ROWS = 16 * AP_RT * AP_WAVES;
constexpr size_t ap_chunk_halves(int D) { return (size_t)2 * AP_CH * D; }  // keys, then values
constexpr size_t ap_lds_bytes(int D) { return 2 * ap_chunk_halves(D) * sizeof(_Float16); }
// the packed keys and values of `keys` positions
constexpr size_t ap_bytes(int D, int kv_heads, int keys) { return (size_t)kv_heads * ((keys + AP_CH - 1) / AP_CH) * ap_chunk_halves(D) * sizeof(_Float16); }

// Whether the packing pays, for `blocks` workgroups of 128 rows.  Whole prompts of six layers, us per layer, with it / with the form of
// attn_prefill_mfma_kernel that runs otherwise.  128 values, 32 heads over 8: 4096 tokens (1024 workgroups) 1066 / 1134, 3000 (752) 881 / 915,
// 2048 (512) 562 / 561, 1536 (384) 479 / 472, 1024 (256) 330 / 327, 900 (232) 318 / 327, 720 (184) 284 / 285; 16 over 4, 3000 (376) 389 / 397;
// 8 over 8, 3000 (192) 262 / 283; 8 over 4, 3000 (188) 231 / 245.  From 128 to 176 the other kernel's blocks, of 64 rows there, need a
// second place on some CUs, which costs where all blocks walk about the same number of keys: 600 tokens from position 900 (152) 299 / 321,
// 560 from 3000 (144) 341 / 402, 1200 from 900 (152, 16 over 4) 226 / 228, but 2200 from 900 (140, 8 over 4) 218 / 211, 2500 from 0 (160)
// 208 / 202, 640 from 0 (160) 278 / 275; 512 from 2000 (128) 276 / 275.
// From 256 to 511, where the other kernel has 128 rows too, the two are level (24 prompts: 2.2 % slower to 2.1 % faster, 0.2 % slower in the
// mean): packed, for its smaller error.
// 64 values: 1024 workgroups 458 / 481, 528 299 / 308, 376 213 / 220, 328 to 340 205 / 209, 192 / 203 and 195 / 197; 256 to 304 173 / 169, 193 / 191, 181 / 177.
constexpr bool attn_packed_pays(int D, int blocks, int pos0, int tokens, int cus) {
    return D == 64 ? 4 * blocks >= 5 * cus : 16 * blocks >= 11 * cus || (2 * blocks > cus && 4 * pos0 >= 3 * tokens);
}

// kcache, vcache [keys, kv_heads, D] -> packed[kv head][chunk]:
//   keys    [tile of 16 keys][32 values][lane][8]: lane n + 16 kq holds key n of the tile, values 8 kq .. + 7 of the 32;
//   values  [16 values of D][32 keys][lane][8]: lane n + 16 kq holds value n of the 16; its slot i < 4 is key 4 kq + i of the 32, slot
//           4 + i key 16 + 4 kq + i - the order in which a lane of attn_packed_kernel ends up with the probabilities of a row.
// Keys past the last repeat it (their scores are masked, their values cleared).  grid (chunks, kv_heads), AP_THREADS threads.
// Bound by memory: 12 bytes moved per key and value.
template <int D>
__global__ void __launch_bounds__(AP_THREADS) attn_pack_kernel(const float *__restrict__ kcache, const float *__restrict__ vcache, _Float16 *__restrict__ packed,
                                                               int kv_heads, int keys) {
    constexpr int PIECES = AP_CH * D / 8, DB = D / 32;
    __shared__ float vs[AP_CH][D + 4];  // the chunk's values, read along the rows and written along the columns
    const int c = blockIdx.x, g = blockIdx.y, j0 = c * AP_CH;
    f16x8 *out = reinterpret_cast<f16x8 *>(packed + ((size_t)g * gridDim.x + c) * ap_chunk_halves(D));
    // (a finite key beyond FP16 is the largest FP16 holds: as infinity it would meet a query's two parts, of either sign, as inf - inf)
    auto key = [](float x) { return (_Float16)(fabsf(x) < INFINITY ? fminf(fmaxf(x, -65504.f), 65504.f) : x); };
    auto row = [&](int j) { return ((size_t)min(j0 + j, keys - 1) * kv_heads + g) * D; };
    for (int i = threadIdx.x; i < AP_CH * D / 4; i += AP_THREADS) {
        const int j = i / (D / 4), e = 4 * (i % (D / 4));
        *reinterpret_cast<float4 *>(&vs[j][e]) = *reinterpret_cast<const float4 *>(vcache + row(j) + e);
    }
    for (int p = threadIdx.x; p < PIECES; p += AP_THREADS) {
        const int lane = p & 63, n = lane & 15, kq = lane >> 4, b = (p >> 6) % DB, t = (p >> 6) / DB;
        const float *k = kcache + row(16 * t + n) + 32 * b + 8 * kq;
        const float4 x = *reinterpret_cast<const float4 *>(k), y = *reinterpret_cast<const float4 *>(k + 4);
        out[p] = f16x8{key(x.x), key(x.y), key(x.z), key(x.w), key(y.x), key(y.y), key(y.z), key(y.w)};
    }
    __syncthreads();
    for (int p = threadIdx.x; p < PIECES; p += AP_THREADS) {
        const int lane = p & 63, n = lane & 15, kq = lane >> 4, ks = (p >> 6) & 1, d = 16 * (p >> 7) + n;
        f16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = (_Float16)vs[32 * ks + 16 * (i >> 2) + 4 * kq + (i & 3)][d];
        out[PIECES + p] = v;
    }
}

// The largest of a value and those of the lanes 16, 32 and 48 away (the lanes of one row of scores): the halves, then the odd and even
// sixteens of two copies trade places.  (In assembly: of the builtin's two results for equal operands the compiler uses one twice.)
__device__ __forceinline__ float ap_max4(float v) {
    float a = v, b = v;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    a = b = fmaxf(a, b);
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return fmaxf(a, b);
}

// A workgroup of four waves takes 128 (token, query head) rows of one key/value head: q [T, heads, D] at positions pos0 .., out
// [T, heads, D]; wave w the rows [32 w, +32) as two tiles of 16.  FP16 operands, FP32 sums and softmax (base 2).
//   * scores, transposed: S^T = K Q^T, so that a lane holds the scores of ONE row (lane % 16) against the keys 4 (lane / 16) + i of the
//     chunk's four 16-key tiles, and those registers, converted, are its slots of the P operand of O^T = V^T P^T - no
//     probability goes through LDS; the output is transposed too, so that the factor that rescales a row is the lane's own.
//   * a chunk is two runs of 1 KiB operands in memory and in LDS: every LDS read is 64 lanes x 16 consecutive bytes and feeds both tiles.
//     (Reads scheduled four to six ahead of their products by hand: level to 10 % slower - it keeps the compiler from laying the
//     exponentials of one tile under the other's products.)
//   * one barrier per chunk, behind a wait for both counters: it says that the chunk has arrived and that the buffer of the one before has been read, which the request for the
//     next chunk then fills - two workgroups a CU work under each other's barriers.
// The last keys a row does not see are masked in the chunks that reach past the block's first token, with their values cleared past its
// last token: what a later block's token holds (infinities, NaN) does not reach this one.
// Longest blocks first; the key/value head is the fast index, so that with eight of them each has an XCD and its L2 for itself.
// grid (kv_heads, blocks of 128 / group tokens), AP_THREADS threads, ap_lds_bytes(D) of dynamic LDS; group <= 16.
template <int D>
__global__ void __launch_bounds__(AP_THREADS, D == 64 ? 3 : 2) attn_packed_kernel(const float *__restrict__ q, const _Float16 *__restrict__ packed, float *__restrict__ out,
                                                                    int heads, int kv_heads, int pos0, int T, int chunks, float scale) {
    constexpr int CH = AP_CH, DB = D / 32, DT = D / 16, RT = AP_RT, KT = CH / 16, HALF = CH * D;  // HALF: halves of the keys, of the values
    constexpr int COPIES = 2 * HALF / 512 / AP_WAVES;  // 1 KiB pieces a wave copies per chunk
    extern __shared__ __align__(16) uint8_t ap_smem[];
    _Float16 *sm = reinterpret_cast<_Float16 *>(ap_smem);  // [2][keys, values]
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = heads / kv_heads, QT = AP_ROWS / group, rows = QT * group;
    const int g = blockIdx.x, t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * QT;
    const int jlast = pos0 + min(t0 + QT, T) - 1;  // last key any row of the block sees
    const int nchunks = jlast / CH + 1;
    // (buffer form: with the flat one in flight the compiler waits for all LDS reads where it needs one)
    const auto src = __builtin_amdgcn_make_buffer_rsrc((void *)(packed + (size_t)g * chunks * (2 * HALF)), 0, chunks * (2 * HALF) * (int)sizeof(_Float16), 0x00020000);
    auto request = [&](int c) {
        _Float16 *to = sm + (c & 1) * (2 * HALF) + wave * COPIES * 512;
#pragma unroll
        for (int i = 0; i < COPIES; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (__attribute__((address_space(3))) void *)(to + i * 512), 16, lane * 16, (c * (2 * HALF) + (wave * COPIES + i) * 512) * (int)sizeof(_Float16), 0, 0);
    };
    request(0);
    bool live[RT];
    int jmax[RT];  // the last key the row sees
    size_t at[RT];  // the row's place in q and out
    // q comes times 1 / sqrt(D) and log2(e): scores in base-2 units, whose largest less itself is 0 at any magnitude.  (Scaled behind the
    // product, by an FMA with the rounded maximum, it is the rounding of that: beyond 2^28 a weight past what FP16 holds.)
    // It comes in two parts, qb + ql, 22 bits.  Against FP64 (64 and 128 values, 600 to 2048 tokens, queries of width 1, 3 and 8) the output is
    // off by 0.86 to 0.90, 0.77 to 0.80 and 0.75 to 0.80 times what it is off by in attn_prefill_mfma_kernel; with one part 1.004 times in the
    // mean - that kernel's two running maxima per row make two weights of a row exact.  The products with ql take 22 of 203 us (4096 tokens, 32
    // heads over 8 of 128 values); heads of 64 values lose nothing by them but at the longest prompts (127 against 117 us there).
    const float scale2 = scale * 1.44269504088896341f;
    f16x8 qb[RT][DB], ql[RT][DB];
#pragma unroll
    for (int u = 0; u < RT; ++u) {
        const int r = 16 * (RT * wave + u) + n, tq = r / group, hq = r - tq * group;
        live[u] = r < rows && t0 + tq < T;
        jmax[u] = pos0 + t0 + tq;
        at[u] = ((size_t)(t0 + (live[u] ? tq : 0)) * heads + g * group + (live[u] ? hq : 0)) * D;
        const float f = live[u] ? scale2 : 0.f;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            const float *qp = q + at[u] + 32 * b + 8 * kq;
            const float4 x = *reinterpret_cast<const float4 *>(qp), y = *reinterpret_cast<const float4 *>(qp + 4);
            const float v[8] = {x.x * f, x.y * f, x.z * f, x.w * f, y.x * f, y.y * f, y.z * f, y.w * f};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                qb[u][b][i] = (_Float16)v[i];
                ql[u][b][i] = (_Float16)(v[i] - (float)qb[u][b][i]);
            }
        }
    }
    f32x4 o[RT][DT];
    float mrun[RT], lrun[RT];  // the row's maximum so far (base 2), this lane's share of its sum
#pragma unroll
    for (int u = 0; u < RT; ++u) {
        mrun[u] = -INFINITY;
        lrun[u] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) o[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // (uniform for the block: only the chunks from here on reach past some row's last key; rows that do not exist are zeros, and not stored)
    const int masked_from = (pos0 + t0 + 1) / CH;
    auto chunk = [&](int c, auto with_mask) {
        constexpr bool MASK = decltype(with_mask)::value;
        // vmcnt(0): this wave's share of chunk c has arrived; lgkmcnt(0): it has read what it needs of chunk c - 1, whose buffer the others
        // fill behind the barrier (the products have taken those reads by then: no time)
        __builtin_amdgcn_s_waitcnt(0x0070);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (c + 1 < nchunks) request(c + 1);
        const f16x8 *kp = reinterpret_cast<const f16x8 *>(sm + (c & 1) * (2 * HALF)) + lane, *vp = kp + HALF / 8;
        const int j0 = c * CH;
        f32x4 st[RT][KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
#pragma unroll
            for (int u = 0; u < RT; ++u) st[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const f16x8 a = kp[(t * DB + b) * 64];
#pragma unroll
                for (int u = 0; u < RT; ++u) st[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qb[u][b], st[u][t], 0, 0, 0);
#pragma unroll
                for (int u = 0; u < RT; ++u) st[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, ql[u][b], st[u][t], 0, 0, 0);
            }
        }
        f16x8 pa[RT][2];
#pragma unroll
        for (int u = 0; u < RT; ++u) {
            float mc = -INFINITY;
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if constexpr (MASK) st[u][t][i] = j0 + 16 * t + 4 * kq + i <= jmax[u] ? st[u][t][i] : -INFINITY;
                    mc = fmaxf(mc, st[u][t][i]);
                }
            const float mn = fmaxf(mrun[u], ap_max4(mc));
            const float alpha = mrun[u] > -INFINITY ? __builtin_amdgcn_exp2f(mrun[u] - mn) : 0.f;
            mrun[u] = mn;
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float p = __builtin_amdgcn_exp2f(st[u][t][i] - mn);
                    if constexpr (MASK) p = st[u][t][i] > -INFINITY ? p : 0.f;  // (a row without a visible key: -inf minus -inf)
                    st[u][t][i] = p;
                }
            // the row's sum, of the weights as they are multiplied: what their rounding adds to the output it adds to the sum as well
            float ls = 0.f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int i = 0; i < 8; ++i) pa[u][h][i] = (_Float16)st[u][2 * h + (i >> 2)][i & 3];
#pragma unroll
                for (int i = 0; i < 8; i += 2) ls = __builtin_amdgcn_fdot2(f16x2{pa[u][h][i], pa[u][h][i + 1]}, f16x2{(_Float16)1.f, (_Float16)1.f}, ls, false);
            }
            lrun[u] = __builtin_fmaf(lrun[u], alpha, ls);
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[u][t][i] *= alpha;
        }
        u32x4 keep[2];
        if constexpr (MASK) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 8; i += 2) {
                    const int j = j0 + 32 * h + 16 * (i >> 2) + 4 * kq + (i & 3);
                    keep[h][i >> 1] = (j <= jlast ? 0xffffu : 0u) | (j + 1 <= jlast ? 0xffff0000u : 0u);
                }
        }
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f16x8 v = vp[(t * 2 + h) * 64];
                if constexpr (MASK) v = __builtin_bit_cast(f16x8, __builtin_bit_cast(u32x4, v) & keep[h]);
#pragma unroll
                for (int u = 0; u < RT; ++u) o[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, pa[u][h], o[u][t], 0, 0, 0);
            }
    };
    int c = 0;
    for (; c < min(masked_from, nchunks); ++c) chunk(c, std::false_type{});
    for (; c < nchunks; ++c) chunk(c, std::true_type{});
    // ---- the lane holds values 16 t + 4 kq + i of row n
#pragma unroll
    for (int u = 0; u < RT; ++u) {
        float l = lrun[u];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        const float il = 1.f / l;
        if (live[u]) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
                *reinterpret_cast<float4 *>(out + at[u] + 16 * t + 4 * kq) = make_float4(o[u][t][0] * il, o[u][t][1] * il, o[u][t][2] * il, o[u][t][3] * il);
        }
    }
}

}  // namespace jitnn
