// One token's attention over a long cache, for heads of 64 or 128 values and up to four query heads per key/value head: what
// attn_decode_kernel (glue.h) does, with every wave on keys of its own.
#pragma once
#include "attn_packed.h"
#include "common.h"

namespace jitnn {

constexpr int AS_WAVES = 4, AS_GMAX = 4;                     // waves per workgroup, query heads per key/value head
constexpr int as_keys(int P) { return 8 * P * AS_WAVES; }  // keys of a workgroup

// The sum of a value over the lanes 16, 32 and 48 away (as ap_max4).
__device__ __forceinline__ float as_sum4(float v) {
    float a = v, b = v;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    a = b = a + b;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return a + b;
}
__device__ __forceinline__ float as_ror8(float v) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true)); }  // the lane 8 away of 16

// Arguments, caches, rotary forms and `part` [heads, chunks, D + 2] as attn_decode_kernel, with chunks of 32 P keys.
//   * eight lanes share a key: lane l holds the values 4 (l % 8) + 32 i .. + 3 of the keys l / 8 + 8 p of its wave, so that a load
//     instruction touches eight whole cache lines, the rotary partner of a value is the lane's own in both forms, and a score is
//     complete, in all eight lanes, after three lane exchanges - the weight is where the value row is multiplied.  No key or value goes through LDS.
//   * all keys and values of a wave are requested before the first is used: 128 KiB per workgroup (P = 4, 128 values).
//   * the eight partial sums of a value meet in registers, two at a time in swapped lane halves (each step halves the registers), the
//     four waves in LDS.
// Groups of up to four: a query head of 128 values takes 16 registers of a lane and its sums 16 more, so that eight heads alone would fill the
// 256 that two workgroups to a CU leave, with 64 or 128 for keys and values still to come.
// Keys past the new token repeat its row; their scores are masked, their values cleared.
// Bound by the cache's way from memory, one round trip for all of it: 4000 positions of 8 key/value heads of 128 values (32.8 MB), with its
// merge, 4.2 us per layer less than attn_decode_kernel (whose three workgroups per CU stage a chunk in LDS and wait for it in step), the
// decode step of 32 such layers 1787 -> 1655 us.  Error against FP64 0.4 to 1.0 times that kernel's.
// grid (chunks, kv_heads), 256 threads.
template <int D, int G, int P>
__global__ void __launch_bounds__(64 * AS_WAVES, 2) attn_split_kernel(const float *__restrict__ qkv, const float *__restrict__ cosv, const float *__restrict__ sinv,
                                                                    float *__restrict__ kcache, float *__restrict__ vcache, float *__restrict__ part,
                                                                    const uint32_t head_counts, const uint32_t pos_pairing) {
    constexpr int NI = D / 32, HALF = D / 2, NV = 4 * NI, KEYS = 8 * P;
    __shared__ float red[AS_WAVES][G][D], sm[AS_WAVES][G], sl[AS_WAVES][G];
    const int heads = (int)(head_counts & 0xffffu), kv_heads = (int)(head_counts >> 16), pos = (int)(pos_pairing & 0x7fffffffu);
    const bool interleaved = (pos_pairing >> 31) != 0;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), sub = lane >> 3, e0 = 4 * (lane & 7);
    const int g = blockIdx.y, c = blockIdx.x, chunks = gridDim.x, j0 = c * as_keys(P) + wave * KEYS;
    const float *q_raw = qkv + (size_t)g * G * D, *k_raw = qkv + (size_t)(heads + g) * D, *v_raw = k_raw + (size_t)kv_heads * D;

    auto load_row = [&](float4(&r)[NI], const float *row) {
#pragma unroll
        for (int i = 0; i < NI; ++i) r[i] = *reinterpret_cast<const float4 *>(row + 32 * i + e0);
    };
    float4 q[G][NI], k[P][NI], v[P][NI];
#pragma unroll
    for (int h = 0; h < G; ++h) load_row(q[h], q_raw + h * D);
    // the angles of this lane's values: rotate-half, those of the values 32 u + e0 .. + 3; interleaved, two each of the quads 2 u and 2 u + 1
    float2 cs[NI], sn[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const size_t at = (size_t)pos * HALF + (interleaved ? 16 * i + (e0 >> 1) : 32 * (i >> 1) + e0 + 2 * (i & 1));
        cs[i] = *reinterpret_cast<const float2 *>(cosv + at);
        sn[i] = *reinterpret_cast<const float2 *>(sinv + at);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int j = j0 + 8 * p + sub;
        load_row(k[p], j < pos ? kcache + ((size_t)j * kv_heads + g) * D : k_raw);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int j = j0 + 8 * p + sub;
        load_row(v[p], j < pos ? vcache + ((size_t)j * kv_heads + g) * D : v_raw);
    }
    __builtin_amdgcn_sched_barrier(0);  // (the compiler would move them to their uses)

    auto rotate = [&](float4(&r)[NI]) {
        if (interleaved) {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const float4 a = r[i];
                r[i] = make_float4(a.x * cs[i].x - a.y * sn[i].x, a.x * sn[i].x + a.y * cs[i].x, a.z * cs[i].y - a.w * sn[i].y, a.z * sn[i].y + a.w * cs[i].y);
            }
        } else {
#pragma unroll
            for (int u = 0; u < NI / 2; ++u) {
                const float4 a = r[u], b = r[u + NI / 2];
                const float2 c0 = cs[2 * u], c1 = cs[2 * u + 1], s0 = sn[2 * u], s1 = sn[2 * u + 1];
                r[u] = make_float4(a.x * c0.x - b.x * s0.x, a.y * c0.y - b.y * s0.y, a.z * c1.x - b.z * s1.x, a.w * c1.y - b.w * s1.y);
                r[u + NI / 2] = make_float4(a.x * s0.x + b.x * c0.x, a.y * s0.y + b.y * c0.y, a.z * s1.x + b.z * c1.x, a.w * s1.y + b.w * c1.y);
            }
        }
    };
#pragma unroll
    for (int h = 0; h < G; ++h) rotate(q[h]);
    if (pos >= j0 && pos < j0 + KEYS) {  // the new token's row: rotated, and appended to the cache
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (j0 + 8 * p + sub == pos) {
                rotate(k[p]);
                const size_t row = ((size_t)pos * kv_heads + g) * D;
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    *reinterpret_cast<float4 *>(kcache + row + 32 * i + e0) = k[p][i];
                    *reinterpret_cast<float4 *>(vcache + row + 32 * i + e0) = v[p][i];
                }
            }
        }
    }
    if (j0 + KEYS > pos + 1) {  // (no weight, and nothing for it to meet)
#pragma unroll
        for (int p = 0; p < P; ++p)
            if (j0 + 8 * p + sub > pos) {
#pragma unroll
                for (int i = 0; i < NI; ++i) v[p][i] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
    }
    // ---- scores, the wave's softmax statistics and weights
    const float scale = 1.0f / sqrtf((float)D);
    float w[P][G];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        float m = -INFINITY;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            float dot = 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                dot = __builtin_fmaf(q[h][i].x, k[p][i].x, dot);
                dot = __builtin_fmaf(q[h][i].y, k[p][i].y, dot);
                dot = __builtin_fmaf(q[h][i].z, k[p][i].z, dot);
                dot = __builtin_fmaf(q[h][i].w, k[p][i].w, dot);
            }
            dot = group_sum<8>(dot);
            w[p][h] = j0 + 8 * p + sub <= pos ? dot * scale : -INFINITY;
            m = fmaxf(m, w[p][h]);
        }
        m = ap_max4(fmaxf(m, as_ror8(m)));
        float l = 0.f;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            w[p][h] = w[p][h] > -INFINITY ? __expf(w[p][h] - m) : 0.f;
            l += w[p][h];
        }
        l = as_sum4(l + as_ror8(l));
        if (lane == 0) {
            sm[wave][h] = m;
            sl[wave][h] = l;
        }
    }
    // ---- weighted sums of the values: acc[NV h + 4 i + e], value 32 i + e0 + e over this lane's keys
    float acc[G * NV];
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int p = 0; p < P; ++p) {
                a.x = __builtin_fmaf(w[p][h], v[p][i].x, a.x);
                a.y = __builtin_fmaf(w[p][h], v[p][i].y, a.y);
                a.z = __builtin_fmaf(w[p][h], v[p][i].z, a.z);
                a.w = __builtin_fmaf(w[p][h], v[p][i].w, a.w);
            }
            acc[NV * h + 4 * i] = a.x;
            acc[NV * h + 4 * i + 1] = a.y;
            acc[NV * h + 4 * i + 2] = a.z;
            acc[NV * h + 4 * i + 3] = a.w;
        }
    // of a pair of sums the lanes 0 .. 31 keep the first, 32 .. 63 the second; then of a pair of those the even and the odd sixteens
#pragma unroll
    for (int r = 0; r < G * NI; ++r) {
        float t[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            float a = acc[4 * r + 2 * u], b = acc[4 * r + 2 * u + 1];
            asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
            t[u] = a + b;
        }
        asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(t[0]), "+v"(t[1]));
        float s = t[0] + t[1];
        s += as_ror8(s);
        if ((lane & 8) == 0) red[wave][r / NI][32 * (r % NI) + e0 + 2 * ((lane >> 4) & 1) + (lane >> 5)] = s;
    }
    __syncthreads();
    for (int i = tid; i < G * D; i += 64 * AS_WAVES) {
        const int h = i / D, d = i - h * D;
        float m = sm[0][h], l = 0.f, a = 0.f;  // (the first key of a workgroup is a token's)
#pragma unroll
        for (int u = 1; u < AS_WAVES; ++u) m = fmaxf(m, sm[u][h]);
#pragma unroll
        for (int u = 0; u < AS_WAVES; ++u) {
            const float f = sm[u][h] > -INFINITY ? __expf(sm[u][h] - m) : 0.f;  // (a workgroup whose scores are all -inf: -inf minus -inf)
            l += sl[u][h] * f;
            a += red[u][h][d] * f;
        }
        float *o = part + ((size_t)(g * G + h) * chunks + c) * (D + 2);
        o[d] = a;
        if (d == 0) {
            o[D] = m;
            o[D + 1] = l;
        }
    }
}

}  // namespace jitnn
