// The walk of one query over its pages in float32: what the generic attention kernel (attention_generic.hip, which says how the work is cut and in
// which order everything is added) and the kernel that runs a small model's whole step (small_step.hip) share, so that both give the same bits.
#pragma once
#include "common.h"

#define ATT_STRIPES 8
#define ATT_MAX_D 256

// four elements that lie together, at a multiple of four elements
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const bf16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u));
}

// lane j's value, j the same for the whole wave
__device__ __forceinline__ float lane_value(float v, int j) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), j)); }

// dot + the product of 4 N elements, in their order, N loads under way together
template <int N, typename T>
__device__ __forceinline__ float key_dot(const float* q, const T* k, float dot) {
    float4 kv[N];
#pragma unroll
    for (int u = 0; u < N; ++u) kv[u] = load4(k + 4 * u);
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const float4 qv = *reinterpret_cast<const float4*>(q + 4 * u);
        dot = fmaf(qv.x, kv[u].x, dot);
        dot = fmaf(qv.y, kv[u].y, dot);
        dot = fmaf(qv.z, kv[u].z, dot);
        dot = fmaf(qv.w, kv[u].w, dot);
    }
    return dot;
}

// sum + the weighted values of 4 N positions from j on (a multiple of four), in their order, N loads under way together
template <int N, typename T>
__device__ __forceinline__ float value_sum(const T* row, float p, int j, float sum) {
    float4 v[N];
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = load4(row + value_place(j + 4 * u));
#pragma unroll
    for (int u = 0; u < N; ++u) {
        sum = fmaf(lane_value(p, j + 4 * u), v[u].x, sum);
        sum = fmaf(lane_value(p, j + 4 * u + 1), v[u].y, sum);
        sum = fmaf(lane_value(p, j + 4 * u + 2), v[u].z, sum);
        sum = fmaf(lane_value(p, j + 4 * u + 3), v[u].w, sum);
    }
    return sum;
}

// What scores are taken from before their exponential: the maximum so far, or 0 while every score is -inf (a stripe may begin with such pages), so that
// those have weight 0 and what follows counts as if they were not there.
__device__ __forceinline__ float from_max(float m) { return m == -INFINITY ? 0.f : m; }

// A stripe's first page from `first` on.
__device__ __forceinline__ int page_of(int stripe, int first) { return first + (stripe - first % ATT_STRIPES + ATT_STRIPES) % ATT_STRIPES; }

// What a stripe leaves: maximum, sum, and this lane's output elements (one of each 64 of the head).
template <int NACC>
struct Stripe {
    float m, l, acc[NACC];
};

// The pages of one stripe for one query: its values in LDS (qf), keys lo .. pos.
// UNROLL: loads of four elements of a key under way together.  NACC: the head is no larger than 64 NACC.
template <typename T, int UNROLL, int NACC>
__device__ __forceinline__ Stripe<NACC> walk(int stripe, const float* qf, const T* keys, const T* values, const int32_t* pages, int pos, int lo, int kvh,
                                       int n_kv_heads, int head_dim, float scale, int wide_keys, int wide_values, int lane) {
    const size_t page_stride = (size_t)n_kv_heads * TQK_PAGE * head_dim;
    Stripe<NACC> r;
#pragma unroll
    for (int i = 0; i < NACC; ++i) r.acc[i] = 0.f;
    r.m = -INFINITY;
    r.l = 0.f;
    for (int pg = page_of(stripe, lo / TQK_PAGE); pg * TQK_PAGE <= pos; pg += ATT_STRIPES) {
        const int kb = pg * TQK_PAGE, page = pages[pg];
        const int j = kb + lane;
        const bool valid = j >= lo && j <= pos && page >= 0;
        const size_t base = (size_t)(page < 0 ? 0 : page) * page_stride + (size_t)kvh * TQK_PAGE * head_dim;
        float s = -INFINITY;
        if (valid) {
            const T* kr = keys + base + (size_t)lane * head_dim;
            float dot = 0.f;
            int i = 0;
            if (wide_keys) {
                // (fewer loads at a time for what is left of the head, or of a small one, and not one)
                if (UNROLL > 8) for (; i + 64 <= head_dim; i += 64) dot = key_dot<16>(qf + i, kr + i, dot);
                for (; i + 32 <= head_dim; i += 32) dot = key_dot<8>(qf + i, kr + i, dot);
                for (; i + 16 <= head_dim; i += 16) dot = key_dot<4>(qf + i, kr + i, dot);
                for (; i < head_dim; i += 4) dot = key_dot<1>(qf + i, kr + i, dot);
            }
            for (; i < head_dim; ++i) dot = fmaf(qf[i], to_float(kr[i]), dot);
            s = dot * scale;
        }
        const float m_new = fmaxf(r.m, wave_max(s)), m_at = from_max(m_new);
        const float p = valid ? expf(s - m_at) : 0.f;
        const float alpha = expf(r.m - m_at);           // exp(-inf) = 0 on the stripe's first page
        r.l = fmaf(r.l, alpha, wave_sum(p));
        r.m = m_new;
        const int n_keys = min(TQK_PAGE, pos - kb + 1);
        const int first_key = max(0, lo - kb);           // keys before the window are never read
        const T* vb = values + base;
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            const int c = lane + a * TQK_WAVE;
            float sum = r.acc[a] * alpha;
            if (a * TQK_WAVE < head_dim) {
                // (lanes past the head read its last row and drop the result)
                const T* row = vb + (size_t)min(c, head_dim - 1) * TQK_PAGE;
                auto one = [&](int jj) { sum = fmaf(lane_value(p, jj), to_float(row[value_place(jj)]), sum); };
                // four positions from a multiple of four lie together
                int jj = first_key;
                for (; jj < n_keys && jj % 4 != 0; ++jj) one(jj);
                if (wide_values) {
                    if (UNROLL > 8) for (; jj + 32 <= n_keys; jj += 32) sum = value_sum<8>(row, p, jj, sum);
                    for (; jj + 16 <= n_keys; jj += 16) sum = value_sum<4>(row, p, jj, sum);
                    for (; jj + 4 <= n_keys; jj += 4) sum = value_sum<1>(row, p, jj, sum);
                }
                for (; jj < n_keys; ++jj) one(jj);
            }
            r.acc[a] = sum;
        }
    }
    return r;
}

// The next stripe joins the ones before it: what the sums so far and the stripe's are multiplied by.
__device__ __forceinline__ void join(float& m, float& l, float stripe_m, float stripe_l, float& of_sum, float& of_stripe) {
    const float mn = fmaxf(m, stripe_m), at = from_max(mn);
    of_sum = expf(m - at);                              // exp(-inf) = 0 for the first one
    of_stripe = expf(stripe_m - at);
    l = fmaf(l, of_sum, stripe_l * of_stripe);
    m = mn;
}
