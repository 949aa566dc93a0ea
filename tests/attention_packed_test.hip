// Drives attn_pack_kernel and attn_packed_kernel of jitnn_amd/csrc/attn_packed.h by themselves against FP64: blocks, chunks and groups of
// query heads that do not divide one another, positions in front of the prompt, and values that are not finite in a later block.
// Prints the name of each check; exit status 0: all hold.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "attn_packed.h"

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

template <int D>
static std::vector<float> attention(const Case &c) {
    const int keys = c.pos0 + c.tokens, group = c.heads / c.kv;
    const size_t nq = (size_t)c.tokens * c.heads * D, nk = (size_t)keys * c.kv * D;
    if (c.q.size() != nq || c.k.size() != nk || c.v.size() != nk || c.heads % c.kv || group > AP_ROWS) exit(1);
    float *q, *k, *v, *o;
    _Float16 *p;
    HIP(hipMalloc(&q, nq * 4));
    HIP(hipMalloc(&o, nq * 4));
    HIP(hipMalloc(&k, nk * 4));
    HIP(hipMalloc(&v, nk * 4));
    HIP(hipMalloc(&p, ap_bytes(D, c.kv, keys)));
    HIP(hipMemcpy(q, c.q.data(), nq * 4, hipMemcpyHostToDevice));
    HIP(hipMemcpy(k, c.k.data(), nk * 4, hipMemcpyHostToDevice));
    HIP(hipMemcpy(v, c.v.data(), nk * 4, hipMemcpyHostToDevice));
    std::vector<float> out(nq, NAN);
    HIP(hipMemcpy(o, out.data(), nq * 4, hipMemcpyHostToDevice));
    HIP(hipFuncSetAttribute((const void *)attn_packed_kernel<D>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ap_lds_bytes(D)));
    const int qt = AP_ROWS / group, chunks = (keys + AP_CH - 1) / AP_CH;
    hipLaunchKernelGGL(attn_pack_kernel<D>, dim3(chunks, c.kv), dim3(AP_THREADS), 0, 0, k, v, p, c.kv, keys);
    hipLaunchKernelGGL(attn_packed_kernel<D>, dim3(c.kv, (c.tokens + qt - 1) / qt), dim3(AP_THREADS), ap_lds_bytes(D), 0, q, p, o, c.heads, c.kv, c.pos0, c.tokens, chunks,
                       1.f / sqrtf((float)D));
    HIP(hipGetLastError());
    HIP(hipDeviceSynchronize());
    HIP(hipMemcpy(out.data(), o, nq * 4, hipMemcpyDeviceToHost));
    for (void *x : {(void *)q, (void *)k, (void *)v, (void *)o, (void *)p}) HIP(hipFree(x));
    return out;
}

// Row by row against FP64.  A score is off by at most d = `off` sum |q_e k_e| / sqrt(D) (2^-10 + 2^-22 + 2^-20: two FP16 operands, FP32 sums), so
// the weights, after normalisation, by factors within exp(+-2 d); a weight and a value round by 2^-11 each; 1e-5 for the FP32 sums
// and the exponentials.  Against the sum of |weight value|.
template <int D>
static bool rows_match(const Case &c, const std::vector<float> &out, int tokens, double off = 0x1p-10 + 0x1p-22 + 0x1p-20) {
    const int group = c.heads / c.kv;
    for (int t = 0; t < tokens; ++t)
        for (int h = 0; h < c.heads; ++h) {
            std::vector<double> s(c.pos0 + t + 1);
            double size = 0, sum = 0;
            for (size_t j = 0; j < s.size(); ++j) {
                double a = 0, b = 0;
                for (int e = 0; e < D; ++e) {
                    const double p = (double)c.q[((size_t)t * c.heads + h) * D + e] * c.k[(j * c.kv + h / group) * D + e];
                    a += p;
                    b += fabs(p);
                }
                s[j] = a / sqrt((double)D);
                size = std::max(size, b / sqrt((double)D));
            }
            const double top = *std::max_element(s.begin(), s.end()), d = off * size;
            for (double &x : s) sum += x = exp(x - top);
            for (int e = 0; e < D; ++e) {
                double want = 0, mag = 0;
                for (size_t j = 0; j < s.size(); ++j) {
                    const double p = s[j] / sum * c.v[(j * c.kv + h / group) * D + e];
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
    return true;
}

// grow: keys that grow along the positions, so that rows of one wave rescale in different chunks
template <int D>
static Case random_case(int heads, int kv, int pos0, int tokens, bool grow) {
    Case c{heads, kv, pos0, tokens, {}, {}, {}};
    std::mt19937 gen(D + heads + tokens);
    std::normal_distribution<float> normal;
    c.q.resize((size_t)tokens * heads * D);
    c.k.resize((size_t)(pos0 + tokens) * kv * D);
    c.v.resize(c.k.size());
    for (float &x : c.q) x = normal(gen);
    for (float &x : c.v) x = normal(gen);
    for (size_t i = 0; i < c.k.size(); ++i) c.k[i] = normal(gen) * (grow ? exp2f((float)(i / ((size_t)kv * D)) / 64.f - 1.f) : 1.f);
    return c;
}

template <int D>
static bool run(int heads, int kv, int pos0, int tokens, bool grow) {
    printf("%d values, %d heads over %d, %d tokens from position %d%s\n", D, heads, kv, tokens, pos0, grow ? ", growing keys" : "");
    fflush(stdout);
    const Case c = random_case<D>(heads, kv, pos0, tokens, grow);
    return rows_match<D>(c, attention<D>(c), tokens);
}

// The tokens of the second block hold infinities and NaN as values: the first block's outputs are what they are without them.
template <int D>
static bool later_blocks_do_not_reach_earlier_ones() {
    printf("%d values, a second block that is not finite\n", D);
    fflush(stdout);
    Case c = random_case<D>(4, 1, 5, 40, false);  // blocks of 32 tokens; the first ends at key 36 of the first chunk
    for (int j = c.pos0 + 32; j < c.pos0 + c.tokens; ++j)
        for (int e = 0; e < D; ++e) c.v[(size_t)j * D + e] = e % 3 == 0 ? INFINITY : e % 3 == 1 ? -INFINITY : NAN;
    return rows_match<D>(c, attention<D>(c), 32);
}

// Wide scores on keys that FP16 holds as they are: the queries' 22 bits are what is left to be off by, d = (2^-22 + 2^-20) sum |q_e k_e| /
// sqrt(D) - whichever place a key has in its chunk.
template <int D>
static bool queries_in_two_parts() {
    printf("%d values, queries of 22 bits\n", D);
    fflush(stdout);
    Case c = random_case<D>(4, 2, 3, 140, false);
    for (float &x : c.q) x *= 32.f;
    for (float &x : c.k) x = (float)(_Float16)x;
    return rows_match<D>(c, attention<D>(c), c.tokens, 0x1p-22 + 0x1p-20);
}

// Keys beyond what FP16 holds, against the queries' signs: no weight lies on them, whatever their size.
template <int D>
static bool keys_beyond_fp16() {
    printf("%d values, keys of -7e4\n", D);
    fflush(stdout);
    Case c = random_case<D>(4, 2, 70, 75, false);
    for (float &x : c.q) x = 0.1f + fabsf(x);
    std::vector<float> out[2];
    for (int i = 0; i < 2; ++i) {
        for (int j : {3, 40, 63, 64, 100, 130})
            for (int e = 0; e < c.kv * D; ++e) c.k[(size_t)j * c.kv * D + e] = i ? -7e4f : -6e4f;
        out[i] = attention<D>(c);
    }
    for (size_t i = 0; i < out[0].size(); ++i)
        if (!(out[0][i] == out[1][i])) {
            printf("output %zu: %.6f, not %.6f\n", i, out[1][i], out[0][i]);
            return false;
        }
    return true;
}

// Scores around 2^32 (positive queries and keys up to 3e4): a row's weight lies on its best key alone, and its output is that key's value as
// FP16 holds it.  A score is off by less than 2^-10 of itself (FP16 queries, FP32 sums): rows whose best two are closer than 2^-9 are left out.
template <int D>
static bool large_scores() {
    printf("%d values, scores around 2^32\n", D);
    fflush(stdout);
    Case c = random_case<D>(4, 2, 70, 75, false);
    std::mt19937 gen(D);
    std::uniform_real_distribution<float> spread(0.5f, 1.f), rank(0.25f, 1.f);
    for (float &x : c.q) x = 3e4f * spread(gen);
    for (size_t i = 0; i < c.k.size(); i += D) {
        const float r = rank(gen);
        for (int e = 0; e < D; ++e) c.k[i + e] = (float)(_Float16)(3e4f * r * spread(gen));
    }
    const std::vector<float> out = attention<D>(c);
    int clear = 0;
    for (int t = 0; t < c.tokens; ++t)
        for (int h = 0; h < c.heads; ++h) {
            int best = 0;
            double top = 0, second = 0;
            for (int j = 0; j <= c.pos0 + t; ++j) {
                double a = 0;
                for (int e = 0; e < D; ++e) a += (double)c.q[((size_t)t * c.heads + h) * D + e] * c.k[((size_t)j * c.kv + h / 2) * D + e];
                if (a > top) best = j;
                second = std::max(second, std::min(a, top));
                top = std::max(top, a);
            }
            if (top - second < 0x1p-9 * top) continue;
            ++clear;
            for (int e = 0; e < D; ++e) {
                const float got = out[((size_t)t * c.heads + h) * D + e], want = (float)(_Float16)c.v[((size_t)best * c.kv + h / 2) * D + e];
                if (!(fabsf(got - want) <= 1e-6f * fabsf(want))) {
                    printf("token %d head %d value %d: %.7f, not %.7f\n", t, h, e, got, want);
                    return false;
                }
            }
        }
    if (clear < c.tokens) printf("%d rows of %d with a clear best key\n", clear, c.tokens * c.heads);
    return clear >= c.tokens;
}

int main() {
    bool ok = true;
    for (int grow = 0; grow < 2; ++grow) {
        ok = ok && run<128>(4, 1, 0, 65, grow) && run<128>(6, 2, 63, 130, grow) && run<128>(2, 2, 1, 129, grow) && run<128>(7, 1, 70, 37, grow);
        ok = ok && run<64>(8, 2, 0, 64, grow) && run<64>(3, 1, 62, 91, grow) && run<64>(4, 4, 130, 130, grow) && run<64>(16, 1, 64, 9, grow);
    }
    ok = ok && later_blocks_do_not_reach_earlier_ones<128>() && later_blocks_do_not_reach_earlier_ones<64>();
    ok = ok && queries_in_two_parts<128>() && queries_in_two_parts<64>();
    ok = ok && keys_beyond_fp16<128>() && keys_beyond_fp16<64>();
    ok = ok && large_scores<128>() && large_scores<64>();
    printf(ok ? "all hold\n" : "FAILED\n");
    return ok ? 0 : 1;
}
