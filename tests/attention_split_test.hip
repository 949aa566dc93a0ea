// Drives attn_split_kernel of jitnn_amd/csrc/attn_split.h and attn_merge_kernel by themselves against FP64, both rotary forms: the new token
// at the edges of a wave's and a workgroup's keys, one chunk and many, cache rows behind the new token that are not finite.
// Prints the name of each check with its error and attn_decode_kernel's; exit status 0: all hold.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "attn_split.h"
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

constexpr int KV = 2, MAX_CTX = 2304;

template <class T>
static T *device(const std::vector<T> &v) {
    T *p;
    HIP(hipMalloc(&p, v.size() * sizeof(T)));
    HIP(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return p;
}

// the error of `out` against `want`, 2-norm
static double distance(const std::vector<float> &out, const std::vector<double> &want) {
    double d = 0, n = 0;
    for (size_t i = 0; i < want.size(); ++i) {
        d += (out[i] - want[i]) * (out[i] - want[i]);
        n += want[i] * want[i];
    }
    return sqrt(d / n);
}

template <int D, int G, int P>
static bool run(int pos, bool interleaved, float width) {
    const int heads = KV * G, split_chunks = pos / as_keys(P) + 1, chunks = pos / AttCfg<D>::CH + 1;
    if (pos >= MAX_CTX) exit(1);
    std::mt19937 gen(D + 8 * G + pos);
    std::normal_distribution<float> normal;
    std::vector<float> qkv((size_t)(heads + 2 * KV) * D), cosv((size_t)MAX_CTX * D / 2), sinv(cosv.size()), k((size_t)MAX_CTX * KV * D), v(k.size());
    for (float &x : qkv) x = normal(gen) * width;
    for (size_t i = 0; i < cosv.size(); ++i) {
        const double a = (double)(i / (D / 2)) * pow(1e4, -2.0 * (i % (D / 2)) / D);
        cosv[i] = (float)cos(a);
        sinv[i] = (float)sin(a);
    }
    for (size_t i = 0; i < k.size(); ++i) {
        const bool past = i >= (size_t)pos * KV * D;
        k[i] = past ? NAN : normal(gen);
        v[i] = past ? (i % 2 ? INFINITY : NAN) : normal(gen);
    }
    float *qd = device(qkv), *cd = device(cosv), *sd = device(sinv), *kd = device(k), *vd = device(v), *part, *out;
    HIP(hipMalloc(&part, (size_t)heads * std::max(split_chunks, chunks) * (D + 2) * 4));
    HIP(hipMalloc(&out, (size_t)heads * D * 4));
    std::vector<float> got[2], rows(2 * (size_t)KV * D);
    for (int which = 0; which < 2; ++which) {  // attn_decode_kernel first; attn_split_kernel appends the row again
        const int n = which ? split_chunks : chunks;
        HIP(hipMemcpy(kd, k.data(), k.size() * 4, hipMemcpyHostToDevice));
        HIP(hipMemcpy(vd, v.data(), v.size() * 4, hipMemcpyHostToDevice));
        if (which) hipLaunchKernelGGL((attn_split_kernel<D, G, P>), dim3(n, KV), dim3(256), 0, 0, qd, cd, sd, kd, vd, part, (uint32_t)heads | ((uint32_t)KV << 16), (uint32_t)pos | (interleaved ? 0x80000000u : 0u));
        else hipLaunchKernelGGL(attn_decode_kernel<D>, dim3(n, KV), dim3(256), 0, 0, qd, cd, sd, kd, vd, part, (uint32_t)heads | ((uint32_t)KV << 16), (uint32_t)pos | (interleaved ? 0x80000000u : 0u));
        hipLaunchKernelGGL((attn_merge_kernel<D, 2>), dim3(heads), dim3(2 * D), 0, 0, part, out, n);
        HIP(hipGetLastError());
        HIP(hipDeviceSynchronize());
        got[which].resize((size_t)heads * D);
        HIP(hipMemcpy(got[which].data(), out, got[which].size() * 4, hipMemcpyDeviceToHost));
    }
    HIP(hipMemcpy(rows.data(), kd + (size_t)pos * KV * D, (size_t)KV * D * 4, hipMemcpyDeviceToHost));
    HIP(hipMemcpy(rows.data() + (size_t)KV * D, vd + (size_t)pos * KV * D, (size_t)KV * D * 4, hipMemcpyDeviceToHost));
    std::vector<float> behind((size_t)KV * D, 0.f);
    const bool room = pos + 1 < MAX_CTX;
    if (room) HIP(hipMemcpy(behind.data(), kd + (size_t)(pos + 1) * KV * D, behind.size() * 4, hipMemcpyDeviceToHost));
    for (void *p : {(void *)qd, (void *)cd, (void *)sd, (void *)kd, (void *)vd, (void *)part, (void *)out}) HIP(hipFree(p));

    // rotated query and key heads, and the appended row: the same FP32 expression, bit for bit
    std::vector<float> rot(qkv.begin(), qkv.begin() + (size_t)(heads + KV) * D);
    for (int h = 0; h < heads + KV; ++h)
        for (int p = 0; p < D / 2; ++p) {
            const size_t i0 = (size_t)h * D + (interleaved ? 2 * p : p), i1 = (size_t)h * D + (interleaved ? 2 * p + 1 : p + D / 2);
            const float a = qkv[i0], b = qkv[i1], c = cosv[(size_t)pos * (D / 2) + p], s = sinv[(size_t)pos * (D / 2) + p];
            rot[i0] = a * c - b * s;
            rot[i1] = a * s + b * c;
        }
    bool ok = memcmp(rows.data(), &rot[(size_t)heads * D], (size_t)KV * D * 4) == 0 && memcmp(&rows[(size_t)KV * D], &qkv[(size_t)(heads + KV) * D], (size_t)KV * D * 4) == 0;
    for (size_t i = 0; room && i < behind.size(); ++i) ok = ok && std::isnan(behind[i]);  // the row behind it is as it was
    if (!ok) printf("the appended row differs\n");
    std::copy(rows.begin(), rows.begin() + (size_t)KV * D, k.begin() + (size_t)pos * KV * D);
    std::copy(rows.begin() + (size_t)KV * D, rows.end(), v.begin() + (size_t)pos * KV * D);

    // A score is a sum of D products in at most D / 8 + 4 FP32 roundings in a row: off by d = (D / 8 + 5) 2^-24 sum |q k| / sqrt(D) at
    // most, the weights by factors within exp(+-2 d) after normalisation; 1e-5 for the exponentials and the FP32 sums.
    std::vector<double> want((size_t)heads * D), s(pos + 1);
    for (int h = 0; h < heads; ++h) {
        double size = 0, sum = 0;
        for (int j = 0; j <= pos; ++j) {
            double a = 0, b = 0;
            for (int e = 0; e < D; ++e) {
                const double p = (double)rot[(size_t)h * D + e] * k[((size_t)j * KV + h / G) * D + e];
                a += p;
                b += fabs(p);
            }
            s[j] = a / sqrt((double)D);
            size = std::max(size, b / sqrt((double)D));
        }
        const double top = *std::max_element(s.begin(), s.end()), d = (D / 8 + 5) * 0x1p-24 * size;
        for (double &x : s) sum += x = exp(x - top);
        for (int e = 0; e < D; ++e) {
            double mag = 0, &w = want[(size_t)h * D + e];
            for (int j = 0; j <= pos; ++j) {
                const double p = s[j] / sum * v[((size_t)j * KV + h / G) * D + e];
                w += p;
                mag += fabs(p);
            }
            const double bar = mag * (exp(2 * d) - 1 + 1e-5);
            if (ok && !(fabs(got[1][(size_t)h * D + e] - w) <= bar)) {
                printf("head %d value %d: %.7f, not %.7f (at most %.1e off)\n", h, e, got[1][(size_t)h * D + e], w, bar);
                ok = false;
            }
        }
    }
    printf("%d values, %d heads over %d, %d keys per workgroup, position %d%s, width %.0f: error %.2e, attn_decode_kernel %.2e\n", D, heads, KV, as_keys(P), pos,
           interleaved ? ", interleaved" : "", width, distance(got[1], want), distance(got[0], want));
    fflush(stdout);
    return ok;
}

// All scores of one workgroup's keys are -inf (their FP32 dot products overflow): those keys have no weight, as in attn_decode_kernel, and
// the others the weights they have without them.  Unrotated (angle zero); 1e-5 of the sum of |weight value|, the scores are at most 30.
template <int D, int G, int P>
static bool keys_without_weight() {
    constexpr int heads = KV * G, first = 2 * as_keys(P), last = first + as_keys(P), pos = last + 40, chunks = pos / as_keys(P) + 1;
    printf("%d values, %d heads over %d, %d keys per workgroup, one of them without weight\n", D, heads, KV, as_keys(P));
    fflush(stdout);
    std::mt19937 gen(D + P);
    std::normal_distribution<float> normal;
    std::vector<float> qkv((size_t)(heads + 2 * KV) * D), cosv((size_t)MAX_CTX * D / 2, 1.f), sinv(cosv.size(), 0.f), k((size_t)MAX_CTX * KV * D), v(k.size());
    for (size_t i = 0; i < qkv.size(); ++i) qkv[i] = i < (size_t)heads * D ? 0.5f + 0.5f * fabsf(normal(gen)) : normal(gen);
    for (size_t i = 0; i < k.size(); ++i) {
        const int j = (int)(i / ((size_t)KV * D));
        k[i] = j >= first && j < last ? -3e38f : normal(gen);
        v[i] = normal(gen);
    }
    float *qd = device(qkv), *cd = device(cosv), *sd = device(sinv), *kd = device(k), *vd = device(v), *part, *out;
    HIP(hipMalloc(&part, (size_t)heads * chunks * (D + 2) * 4));
    HIP(hipMalloc(&out, (size_t)heads * D * 4));
    hipLaunchKernelGGL((attn_split_kernel<D, G, P>), dim3(chunks, KV), dim3(256), 0, 0, qd, cd, sd, kd, vd, part, (uint32_t)heads | ((uint32_t)KV << 16), (uint32_t)pos);
    hipLaunchKernelGGL((attn_merge_kernel<D, 2>), dim3(heads), dim3(2 * D), 0, 0, part, out, chunks);
    HIP(hipGetLastError());
    HIP(hipDeviceSynchronize());
    std::vector<float> got((size_t)heads * D);
    HIP(hipMemcpy(got.data(), out, got.size() * 4, hipMemcpyDeviceToHost));
    for (void *p : {(void *)qd, (void *)cd, (void *)sd, (void *)kd, (void *)vd, (void *)part, (void *)out}) HIP(hipFree(p));
    std::copy(qkv.begin() + (size_t)heads * D, qkv.begin() + (size_t)(heads + KV) * D, k.begin() + (size_t)pos * KV * D);
    std::copy(qkv.begin() + (size_t)(heads + KV) * D, qkv.end(), v.begin() + (size_t)pos * KV * D);
    for (int h = 0; h < heads; ++h) {
        std::vector<double> w(pos + 1), sum(D), mag(D);
        double all = 0;
        for (int j = 0; j <= pos; ++j) {
            double a = 0;
            for (int e = 0; e < D; ++e) a += (double)qkv[(size_t)h * D + e] * k[((size_t)j * KV + h / G) * D + e];
            all += w[j] = exp(a / sqrt((double)D));
        }
        for (int j = 0; j <= pos; ++j)
            for (int e = 0; e < D; ++e) {
                const double p = w[j] / all * v[((size_t)j * KV + h / G) * D + e];
                sum[e] += p;
                mag[e] += fabs(p);
            }
        for (int e = 0; e < D; ++e)
            if (!(fabs(got[(size_t)h * D + e] - sum[e]) <= 1e-5 * mag[e])) {
                printf("head %d value %d: %.7f, not %.7f\n", h, e, got[(size_t)h * D + e], sum[e]);
                return false;
            }
    }
    return true;
}

template <int D, int G>
static bool positions() {
    bool ok = true;
    for (int pos : {0, 7, 8, 31, 32, 63, 64, 127, 128, 129, 1000, 1023, 2303}) {
        ok = ok && run<D, G, 2>(pos, pos % 2 == 0, 1.f);
        ok = ok && run<D, G, 4>(pos, pos % 2 != 0, 1.f);
    }
    return ok && run<D, G, 4>(1500, false, 8.f) && run<D, G, 2>(1500, true, 8.f);
}

int main() {
    bool ok = positions<128, 1>() && positions<128, 2>() && positions<128, 3>() && positions<128, 4>() && positions<64, 1>() && positions<64, 2>() &&
                    positions<64, 3>() && positions<64, 4>();
    ok = ok && keys_without_weight<128, 4, 2>() && keys_without_weight<128, 2, 4>() && keys_without_weight<64, 3, 2>() && keys_without_weight<64, 1, 4>();
    printf(ok ? "all hold\n" : "FAILED\n");
    return ok ? 0 : 1;
}
