// Drives attn_prefill_mfma_kernel of jitnn_amd/csrc/glue.h by itself, on queries, keys and values chosen for it, against FP64.
// Prints the name of each check; exit status 0: all hold.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "glue.h"

using namespace jitnn;

#define HIP(e)                                                       \
    do {                                                             \
        const hipError_t rc = (e);                                   \
        if (rc != hipSuccess) {                                      \
            printf("%s: %s\n", #e, hipGetErrorString(rc));           \
            exit(1);                                                 \
        }                                                            \
    } while (0)

struct Case {
    int heads, kv, pos0, tokens;
    std::vector<float> q, k, v;  // [tokens, heads, D], [pos0 + tokens, kv, D] twice
};

template <int D, int RT>
static std::vector<float> attention(const Case &c) {
    const size_t nq = (size_t)c.tokens * c.heads * D, nk = (size_t)(c.pos0 + c.tokens) * c.kv * D;
    if (c.q.size() != nq || c.k.size() != nk || c.v.size() != nk || c.heads % c.kv || c.heads / c.kv > ATT_GMAX) exit(1);
    float *q, *k, *v, *o;
    HIP(hipMalloc(&q, nq * 4));
    HIP(hipMalloc(&o, nq * 4));
    HIP(hipMalloc(&k, nk * 4));
    HIP(hipMalloc(&v, nk * 4));
    HIP(hipMemcpy(q, c.q.data(), nq * 4, hipMemcpyHostToDevice));
    HIP(hipMemcpy(k, c.k.data(), nk * 4, hipMemcpyHostToDevice));
    HIP(hipMemcpy(v, c.v.data(), nk * 4, hipMemcpyHostToDevice));
    std::vector<float> out(nq, NAN);
    HIP(hipMemcpy(o, out.data(), nq * 4, hipMemcpyHostToDevice));
    constexpr size_t lds = attn_prefill_mfma_lds_bytes<D, RT>();
    HIP(hipFuncSetAttribute((const void *)attn_prefill_mfma_kernel<D, RT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int qt = RT * AM_ROWS / (c.heads / c.kv), blocks = (c.tokens + qt - 1) / qt;
    hipLaunchKernelGGL((attn_prefill_mfma_kernel<D, RT>), RT == 1 ? dim3(blocks, c.kv) : dim3(c.kv, blocks), dim3(AM_THREADS), lds, 0, q, k, v, o, c.heads, c.kv,
                       c.pos0, c.tokens, 1.f / sqrtf((float)D));
    HIP(hipGetLastError());
    HIP(hipDeviceSynchronize());
    HIP(hipMemcpy(out.data(), o, nq * 4, hipMemcpyDeviceToHost));
    for (float *p : {q, k, v, o}) HIP(hipFree(p));
    return out;
}

// log2 of the unnormalised weights of (token t, head h), and the largest sum of |q_e k_e| / sqrt(D) over its keys
template <int D>
static std::vector<double> scores(const Case &c, int t, int h, double *size) {
    std::vector<double> s(c.pos0 + t + 1);
    *size = 0;
    for (size_t j = 0; j < s.size(); ++j) {
        double a = 0, b = 0;
        for (int e = 0; e < D; ++e) {
            const double p = (double)c.q[((size_t)t * c.heads + h) * D + e] * c.k[(j * c.kv + h / (c.heads / c.kv)) * D + e];
            a += p;
            b += fabs(p);
        }
        s[j] = a / sqrt((double)D) * 1.4426950408889634;
        *size = std::max(*size, b / sqrt((double)D));
    }
    return s;
}

// One key takes nearly all of a row's weight, and the row meets it after a first chunk whose largest score is up to 2^8 times
// less.  All values are 1.5: what the output differs from it by is the rounding of the weights to FP16.  The largest weight is 1 by
// itself, without rounding, where it stands against the running maximum; the other one, w, rounds by at most 2^-11 of itself;
// 1e-6 for the FP32 sums and the exponentials.
template <int D, int RT>
static bool largest_weight_is_exact() {
    Case c{4, 2, 192, 70, {}, {}, {}};
    c.q.assign((size_t)c.tokens * c.heads * D, 0.f);
    c.k.assign((size_t)(c.pos0 + c.tokens) * c.kv * D, 0.f);
    c.v.assign(c.k.size(), 1.5f);
    const double unit = sqrt((double)D) / 1.4426950408889634;  // a key whose score against a query of 1 is 1 in base 2
    for (int i = 0; i < c.tokens * c.heads; ++i) c.q[(size_t)i * D] = (float)(0.75 + 0.25 * i / (c.tokens * c.heads));
    for (int j = 0; j < c.pos0 + c.tokens; ++j)
        for (int g = 0; g < c.kv; ++g) c.k[((size_t)j * c.kv + g) * D] = (float)(_Float16)(unit * (j == 0 ? 0.0 : j == 67 ? 7.9 : -200.0));
    const std::vector<float> out = attention<D, RT>(c);
    for (int t = 0; t < c.tokens; ++t)
        for (int h = 0; h < c.heads; ++h) {
            const double q = (float)(_Float16)c.q[((size_t)t * c.heads + h) * D], s = q * c.k[(size_t)67 * c.kv * D] / unit, w = 1 / (1 + exp2(s));
            for (int e = 0; e < D; ++e) {
                const double off = fabs(out[((size_t)t * c.heads + h) * D + e] / 1.5 - 1);
                if (!(off <= w * 0x1p-11 + 1e-6)) {
                    printf("token %d head %d value %d: off by %.3e, at most %.3e\n", t, h, e, off, w * 0x1p-11 + 1e-6);
                    return false;
                }
            }
        }
    return true;
}

// Keys that grow along the positions: in most chunks the maximum of some rows of a wave grows by far more than 1 and that of others
// not at all - in chunks that need the mask and in others -, so that the outputs so far are rescaled row by row.
// A score is off by at most d = (2^-10 + 2^-22) sum |q_e k_e| / sqrt(D) (two FP16 operands) and 2^-20 of itself (FP32), so the
// weights by factors within exp(+-d), after normalisation exp(+-2 d); a weight and a value round by 2^-11 each.  Against the
// sum of |weight value|.
template <int D, int RT>
static bool rows_rescale_one_by_one(int group) {
    Case c{2 * group, 2, 70, 170, {}, {}, {}};  // (the keys in front of the first block end inside a chunk, the last block is partly filled)
    std::mt19937 gen(D + RT);
    std::normal_distribution<float> normal;
    c.q.resize((size_t)c.tokens * c.heads * D);
    c.k.resize((size_t)(c.pos0 + c.tokens) * c.kv * D);
    c.v.resize(c.k.size());
    for (float &x : c.q) x = normal(gen);
    for (float &x : c.v) x = normal(gen);
    for (size_t i = 0; i < c.k.size(); ++i) c.k[i] = normal(gen) * exp2f((float)(i / ((size_t)c.kv * D)) / 64.f - 1.f);
    const std::vector<float> out = attention<D, RT>(c);
    const int qt = RT * AM_ROWS / group;
    int mixed[2] = {};  // (tile of 16 rows, half of a chunk) pairs with rows that rescale and rows that do not: unmasked, masked
    for (int g = 0; g < c.kv; ++g)
        for (int t0 = 0; t0 < c.tokens; t0 += qt)
            for (int tile = 0; tile < 4 * RT; ++tile) {
                std::vector<std::vector<double>> s;
                for (int r = 16 * tile; r < 16 * tile + 16; ++r) {
                    const int t = t0 + r / group, h = g * group + r % group;
                    if (r >= qt * group || t >= c.tokens) continue;
                    double size;
                    s.push_back(scores<D>(c, t, h, &size));
                    const std::vector<double> &row = s.back();
                    const double top = *std::max_element(row.begin(), row.end()), d = (0x1p-10 + 0x1p-22 + 0x1p-20) * size;
                    double sum = 0;
                    for (double x : row) sum += exp2(x - top);
                    for (int e = 0; e < D; ++e) {
                        double want = 0, mag = 0;
                        for (size_t j = 0; j < row.size(); ++j) {
                            const double p = exp2(row[j] - top) / sum * c.v[(j * c.kv + g) * D + e];
                            want += p;
                            mag += fabs(p);
                        }
                        const double got = out[((size_t)t * c.heads + h) * D + e], bar = mag * (exp(2 * d) - 1 + 0x1p-10 + 1e-5);
                        if (!(fabs(got - want) <= bar)) {
                            printf("token %d head %d value %d: %.6f, not %.6f (at most %.1e off)\n", t, h, e, got, want, bar);
                            return false;
                        }
                    }
                }
                for (int half = 0; half < 2; ++half) {
                    std::vector<double> top(s.size(), -INFINITY);
                    for (int j0 = 0; j0 < c.pos0 + c.tokens; j0 += AM_CH) {
                        int grown = 0, kept = 0;
                        for (size_t r = 0; r < s.size(); ++r) {
                            double m = -INFINITY;
                            for (size_t j = j0 + 32 * half; j < std::min((size_t)j0 + 32 * half + 32, s[r].size()); ++j) m = std::max(m, s[r][j]);
                            if (m == -INFINITY) continue;
                            grown += top[r] > -INFINITY && m > top[r] + 1;
                            kept += m <= top[r];
                            top[r] = std::max(top[r], m);
                        }
                        const bool masked = j0 + AM_CH - 1 > c.pos0 + t0 || t0 + qt > c.tokens || qt * group != RT * AM_ROWS;
                        mixed[masked] += grown && kept;
                    }
                }
            }
    if (mixed[1] < 10 || (RT * AM_ROWS % group == 0 && mixed[0] < 10)) {  // (groups that do not fill a block: every chunk is masked)
        printf("%d and %d waves with rows of both kinds\n", mixed[0], mixed[1]);
        return false;
    }
    return true;
}

template <int D, int RT>
static void check() {
    printf("largest weight is exact, %d values, %d tiles\n", D, RT);
    fflush(stdout);
    if (!largest_weight_is_exact<D, RT>()) exit(1);
    for (int group : {3, 4}) {
        printf("rows rescale one by one, %d values, %d tiles, groups of %d\n", D, RT, group);
        fflush(stdout);
        if (!rows_rescale_one_by_one<D, RT>(group)) exit(1);
    }
}

int main() {
    // what attn_two_tiles_from counts on: two workgroups of 128 rows on a CU where heads have 64 values, one where they have 128
    printf("workgroups on a CU\n");
    int fit64 = 0, fit128 = 0;
    HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit64, attn_prefill_mfma_kernel<64, 2>, AM_THREADS, attn_prefill_mfma_lds_bytes<64, 2>()));
    HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit128, attn_prefill_mfma_kernel<128, 2>, AM_THREADS, attn_prefill_mfma_lds_bytes<128, 2>()));
    if (fit64 != attn_two_tiles_from(64, 1) || fit128 != attn_two_tiles_from(128, 1)) {
        printf("%d and %d\n", fit64, fit128);
        return 1;
    }
    check<64, 1>();
    check<64, 2>();
    check<128, 1>();
    check<128, 2>();
    printf("all hold\n");
    return 0;
}
