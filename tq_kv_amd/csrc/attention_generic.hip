// Softmax attention over the paged cache, one wave per (token, query head), float32
// arithmetic throughout.  It serves the float32 path for prompts and for decoding
// alike, and any head size; the bfloat16 path uses it where the MFMA kernels do
// not apply.
//
// Formulas: scores q.k / sqrt(d), mask, softmax (max-subtract, exp, normalise), p.v
// as src/models/turbo_generic.rs:1620-1631 and :56-62; query head h reads kv head
// h / (heads / kv_heads) (:195-204).  The reference's mask is only right for a
// prompt at position 0 (:1937-1956); here the query at absolute position i sees
// keys lo..i of its own sequence for any split into steps, lo being 0 or, with a
// window of W, max(0, i - W + 1).
//
// Work of one wave: keys are taken in blocks of 64 (one page); lane j computes the
// score of key j of the block, the softmax runs online over blocks, then lane c
// accumulates output element c (+64, +128, ...) over the block's keys.  Pages are dealt to
// eight stripes by their number, each walked on its own, and the stripes meet in their order: either
// one wave walks all of them (many queries), or a wave each (few queries, or in float32 the heads of a kv head together).  The order of
// operations for a query depends only on its position, never on the batch or on which of the two it is.
// Cache pages: keys [kv head][position][head_dim], values [kv head][head_dim][place of
// the position] (value_place in common.h).
#include "attention_walk.h"
#include "tq_kernels.h"

#include <type_traits>

#define ATT_WAVES 4

// Bound by latency, a page costs a wave 6 us: the float32 step of four tokens after 300 (28 heads of 128) takes 13.6 us with a wave per stripe and
// up to 16 loads under way, 37.0 with one wave for all and up to 8.  What is left of a head or a page after the last 16 loads goes by
// 8 and 4 before single ones: one after the other it was most of the time of small heads and short contexts (heads of 32, 20 positions 5.4 -> 4.5 us).
// SPLIT: a block of a wave per stripe for one query.
template <typename T, bool SPLIT>
__global__ __launch_bounds__((SPLIT ? ATT_STRIPES : ATT_WAVES) * TQK_WAVE)
void attention_generic_kernel(const T* __restrict__ q, const T* __restrict__ keys, const T* __restrict__ values,
                              const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ tok_pos,
                              const int32_t* __restrict__ page_table, int table_width, int window, float scale,
                              T* __restrict__ out, int n_tokens, int n_heads, int n_kv_heads, int head_dim, int wide_keys, int wide_values) {
    constexpr int NACC = ATT_MAX_D / TQK_WAVE;
    __shared__ __attribute__((aligned(16))) float q_lds[SPLIT ? ATT_STRIPES : ATT_WAVES][ATT_MAX_D];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TQK_WAVE), lane = threadIdx.x % TQK_WAVE;
    const int t = SPLIT ? blockIdx.x : blockIdx.x * ATT_WAVES + wave;
    const int head = blockIdx.y;
    if (t >= n_tokens) return;
    // (every wave keeps a copy of its query: nobody waits for anybody, and waves without a page are gone at once)
    float* qf = q_lds[wave];
    const T* qv = q + ((size_t)t * n_heads + head) * head_dim;
    for (int i = lane; i < head_dim; i += TQK_WAVE) qf[i] = to_float(qv[i]);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    const int pos = tok_pos[t];
    const int32_t* pages = page_table + (size_t)tok_seq[t] * table_width;
    const int kvh = head / (n_heads / n_kv_heads);
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    T* o = out + ((size_t)t * n_heads + head) * head_dim;
    float m = -INFINITY, l = 0.f, of_sum, of_stripe;

    if constexpr (SPLIT) {
        __shared__ float met[ATT_STRIPES][ATT_MAX_D], ml[ATT_STRIPES][2];
        const bool alone = lo / TQK_PAGE == pos / TQK_PAGE;             // one page: its stripe is the result
        if (alone && wave > 0) return;
        const Stripe<NACC> r = walk<T, 16, NACC>(alone ? lo / TQK_PAGE % ATT_STRIPES : wave, qf, keys, values, pages, pos, lo, kvh, n_kv_heads, head_dim, scale, wide_keys, wide_values, lane);
        if (alone) {
#pragma unroll
            for (int a = 0; a < NACC; ++a) {
                const int c = lane + a * TQK_WAVE;
                if (c < head_dim) o[c] = from_float<T>(r.acc[a] / r.l);
            }
            return;
        }
#pragma unroll
        for (int a = 0; a < NACC; ++a) met[wave][lane + a * TQK_WAVE] = r.acc[a];
        if (lane == 0) { ml[wave][0] = r.m; ml[wave][1] = r.l; }
        __syncthreads();
        float acc = 0.f;
        const int c = threadIdx.x;
        if (c >= head_dim) return;
        for (int s = 0; s < ATT_STRIPES; ++s) {
            if (page_of(s, lo / TQK_PAGE) * TQK_PAGE > pos) continue;
            join(m, l, ml[s][0], ml[s][1], of_sum, of_stripe);
            acc = fmaf(acc, of_sum, met[s][c] * of_stripe);
        }
        o[c] = from_float<T>(acc / l);
    } else {
        float acc[NACC];
#pragma unroll
        for (int a = 0; a < NACC; ++a) acc[a] = 0.f;
        for (int s = 0; s < ATT_STRIPES; ++s) {
            if (page_of(s, lo / TQK_PAGE) * TQK_PAGE > pos) continue;
            const Stripe<NACC> r = walk<T, 8, NACC>(s, qf, keys, values, pages, pos, lo, kvh, n_kv_heads, head_dim, scale, wide_keys, wide_values, lane);
            join(m, l, r.m, r.l, of_sum, of_stripe);
#pragma unroll
            for (int a = 0; a < NACC; ++a) acc[a] = fmaf(acc[a], of_sum, r.acc[a] * of_stripe);
        }
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            const int c = lane + a * TQK_WAVE;
            if (c < head_dim) o[c] = from_float<T>(acc[a] / l);
        }
    }
}

// The heads of one kv head together, for prompts in float32: HEADS of them (the last one again where there are fewer), a wave a stripe, head_dim <= 64 NACC.
// A wave's loads of keys and values touch a line a lane, and a unit takes a line a cycle: so they are what the general kernel waits for, and here they are
// made once for all heads, with the queries in scalar registers.  The same operations in the same order, so that the bits are the general kernel's.
// 28 heads over 4 of 128, us before and after: prompts of 64, 300, 1000, 2000 tokens 19.0, 192, 1652, 6338 and 11.4, 54, 335, 1137; 40 queries after 333
// positions 92 and 29.  Then bound by the loads' lines up to two blocks a unit, by the multiplies (a seventh of the vector units' rate) beyond.
template <int HEADS, int NACC>
__global__ __launch_bounds__(ATT_STRIPES * TQK_WAVE)
void attention_heads_kernel(const float* __restrict__ q, const float* __restrict__ keys, const float* __restrict__ values,
                            const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ page_table,
                            int table_width, int window, float scale, float* __restrict__ out, int n_heads, int n_kv_heads, int head_dim) {
    __shared__ float met[ATT_STRIPES][HEADS][NACC * TQK_WAVE], ml[ATT_STRIPES][HEADS][2];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TQK_WAVE), lane = threadIdx.x % TQK_WAVE;
    const int t = blockIdx.x, group = n_heads / n_kv_heads, parts = (group + HEADS - 1) / HEADS;
    const int kvh = blockIdx.y / parts, first = blockIdx.y % parts * HEADS, n = min(HEADS, group - first);
    const size_t row = (size_t)t * n_heads + (size_t)kvh * group + first;
    const float* qv = q + row * head_dim;
    float* o = out + row * head_dim;
    const int pos = tok_pos[t], lo = window > 0 ? max(0, pos - window + 1) : 0, first_page = lo / TQK_PAGE;
    const int32_t* pages = page_table + (size_t)tok_seq[t] * table_width;
    const size_t page_stride = (size_t)n_kv_heads * TQK_PAGE * head_dim;

    float m[HEADS], l[HEADS], acc[HEADS][NACC];
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int a = 0; a < NACC; ++a) acc[h][a] = 0.f;
    }
    for (int pg = page_of(wave, first_page); pg * TQK_PAGE <= pos; pg += ATT_STRIPES) {
        const int kb = pg * TQK_PAGE, page = pages[pg];
        const int j = kb + lane;
        const bool valid = j >= lo && j <= pos && page >= 0;
        const size_t base = (size_t)(page < 0 ? 0 : page) * page_stride + (size_t)kvh * TQK_PAGE * head_dim;
        float s[HEADS];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) s[h] = 0.f;
        if (valid) {
            const float* kr = keys + base + (size_t)lane * head_dim;
            auto some = [&](auto loads, int i) {
                constexpr int N = decltype(loads)::value;
                float4 kv[N];
#pragma unroll
                for (int u = 0; u < N; ++u) kv[u] = load4(kr + i + 4 * u);
#pragma unroll
                for (int h = 0; h < HEADS; ++h) {
                    const float* qh = qv + min(h, n - 1) * head_dim + i;
#pragma unroll
                    for (int u = 0; u < N; ++u) {
                        s[h] = fmaf(qh[4 * u], kv[u].x, s[h]);
                        s[h] = fmaf(qh[4 * u + 1], kv[u].y, s[h]);
                        s[h] = fmaf(qh[4 * u + 2], kv[u].z, s[h]);
                        s[h] = fmaf(qh[4 * u + 3], kv[u].w, s[h]);
                    }
                }
            };
            int i = 0;
            for (; i + 32 <= head_dim; i += 32) some(std::integral_constant<int, 8>(), i);
            if (i + 16 <= head_dim) { some(std::integral_constant<int, 4>(), i); i += 16; }
            for (; i < head_dim; i += 4) some(std::integral_constant<int, 1>(), i);
        }
        float p[HEADS];
#pragma unroll
        for (int h = 0; h < HEADS; ++h) {
            const float score = valid ? s[h] * scale : -INFINITY;
            const float m_new = fmaxf(m[h], wave_max(score)), m_at = from_max(m_new);
            p[h] = valid ? expf(score - m_at) : 0.f;
            const float alpha = expf(m[h] - m_at);
            l[h] = fmaf(l[h], alpha, wave_sum(p[h]));
            m[h] = m_new;
#pragma unroll
            for (int a = 0; a < NACC; ++a) acc[h][a] *= alpha;
        }
        const int n_keys = min(TQK_PAGE, pos - kb + 1), first_key = max(0, lo - kb);         // keys before the window are never read
        const float* rows[NACC];
#pragma unroll
        for (int a = 0; a < NACC; ++a) rows[a] = values + base + (size_t)min(lane + a * TQK_WAVE, head_dim - 1) * TQK_PAGE;
        auto add = [&](int jj, const float (&v)[NACC]) {
#pragma unroll
            for (int h = 0; h < HEADS; ++h) {
                const float w = lane_value(p[h], jj);
#pragma unroll
                for (int a = 0; a < NACC; ++a) acc[h][a] = fmaf(w, v[a], acc[h][a]);
            }
        };
        auto one = [&](int jj) {
            float v[NACC];
#pragma unroll
            for (int a = 0; a < NACC; ++a) v[a] = rows[a][value_place(jj)];
            add(jj, v);
        };
        auto fours = [&](auto loads, int jj) {
            constexpr int N = decltype(loads)::value;
            float4 v[N][NACC];
#pragma unroll
            for (int u = 0; u < N; ++u)
#pragma unroll
                for (int a = 0; a < NACC; ++a) v[u][a] = load4(rows[a] + value_place(jj + 4 * u));
#pragma unroll
            for (int u = 0; u < N; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float of[NACC];
#pragma unroll
                    for (int a = 0; a < NACC; ++a) of[a] = (&v[u][a].x)[e];
                    add(jj + 4 * u + e, of);
                }
        };
        int jj = first_key;
        for (; jj < n_keys && jj % 4 != 0; ++jj) one(jj);
        for (; jj + 16 <= n_keys; jj += 16) fours(std::integral_constant<int, 4>(), jj);
        for (; jj + 4 <= n_keys; jj += 4) fours(std::integral_constant<int, 1>(), jj);
        for (; jj < n_keys; ++jj) one(jj);
    }
#pragma unroll
    for (int h = 0; h < HEADS; ++h) {
#pragma unroll
        for (int a = 0; a < NACC; ++a) met[wave][h][lane + a * TQK_WAVE] = acc[h][a];
        if (lane == 0) { ml[wave][h][0] = m[h]; ml[wave][h][1] = l[h]; }
    }
    __syncthreads();
    for (int h = wave; h < n; h += ATT_STRIPES) {
        float mh = -INFINITY, lh = 0.f, sum[NACC], of_sum, of_stripe;
#pragma unroll
        for (int a = 0; a < NACC; ++a) sum[a] = 0.f;
        for (int st = 0; st < ATT_STRIPES; ++st) {
            if (page_of(st, first_page) * TQK_PAGE > pos) continue;
            join(mh, lh, ml[st][h][0], ml[st][h][1], of_sum, of_stripe);
#pragma unroll
            for (int a = 0; a < NACC; ++a) sum[a] = fmaf(sum[a], of_sum, met[st][h][lane + a * TQK_WAVE] * of_stripe);
        }
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
            const int c = lane + a * TQK_WAVE;
            if (c < head_dim) o[(size_t)h * head_dim + c] = sum[a] / lh;
        }
    }
}

extern "C" int tqk_attention_max_head_dim(void) { return ATT_MAX_D; }

// How many heads share a wave's loads (0: the general kernel).  Fewer heads a wave are more blocks and less work one after the other, more heads fewer loads:
// what counts is whether the blocks fill the chip and how many pages a query has.  us with 2, 4 and 8 heads together (general kernel in brackets):
// prompts of 40, 64, 150, 300 tokens, 28 heads over 4 of 128: 9.1, 9.9, 13.7 (12.6); 14.1, 11.3, 15.5 (19.0); 35, 25, 28 (58); 113, 64, 54 (192).  12 over 2:
// 64, 150, 300 tokens 8.8, 10.2, 14.9 (12.2); 18, 15, 17 (34); 52, 41, 38 (99).  40 over 8: 40, 64, 300 tokens 11.9, 10.5, 14.0 (12.9); 19, 18, 16 (26); 160, 114, 94 (255).
// With 1500 positions 100 queries of 28 heads over 4: 437, 259, 134 (525), and 8 heads win however few the blocks.
// Where the general kernel takes a wave a stripe it has as many waves as 2 heads together have from twice the queries: 28 heads, 12 queries after 20, 300, 1500
// positions 6.6, 14.8, 64 with 2 heads (7.7, 23.5, 104), 18 queries, more than a block a unit, 6.9, 30.8, 137 (6.6, 31.0, 129), 8 queries 6.7, 13.9, 57 (6.5, 14.6, 54).
static int heads_together(int n_tokens, int group, int n_kv_heads, int head_dim, int table_width, int window) {
    if (group == 1 || head_dim > 128) return 0;
    auto blocks = [&](int heads) { return (long long)n_tokens * n_kv_heads * ((group + heads - 1) / heads); };
    if (blocks(1) <= 512) return blocks(1) > 256 && blocks(2) <= 256 ? 2 : 0;
    const bool few_pages = table_width <= 4 || (window > 0 && window <= 2 * TQK_PAGE);
    if (few_pages && blocks(4) <= 400) return 2;
    return group <= 2 ? 2 : group <= 4 || few_pages ? 4 : 8;
}

extern "C" int tqk_attention(const void* q, const void* keys, const void* values, int act_dtype,
                             const int32_t* tok_seq, const int32_t* tok_pos, const int32_t* page_table,
                             int table_width, int n_seqs, int n_pages, int window, float scale, void* out,
                             int n_tokens, int n_heads, int n_kv_heads, int head_dim, void* stream) {
    TQK_REQUIRE(q && keys && values && tok_seq && tok_pos && page_table && out, "tqk_attention: null pointer");
    TQK_REQUIRE(n_tokens >= 0 && n_heads > 0 && n_kv_heads > 0 && head_dim > 0, "tqk_attention: bad sizes");
    TQK_REQUIRE(n_heads % n_kv_heads == 0, "tqk_attention: %d heads are not a multiple of %d kv heads", n_heads, n_kv_heads);
    TQK_REQUIRE(head_dim <= ATT_MAX_D, "tqk_attention: head_dim %d is more than %d", head_dim, ATT_MAX_D);
    TQK_REQUIRE(n_heads <= 65535, "tqk_attention: too many heads for the grid");
    TQK_REQUIRE(table_width > 0 && n_pages > 0 && n_seqs > 0, "tqk_attention: empty page table");
    TQK_REQUIRE(window >= 0, "tqk_attention: negative window");
    if (n_tokens == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    // Where heads are not taken together: a wave per stripe while no unit gets more than two blocks of them; the results are the same.  us with a wave per stripe and with one for all,
    // float32, 28 heads of 128: 504 waves of queries after 20, 128, 300 and 1500 positions 6.3, 12.1, 23.0, 97 and 7.3, 18.7, 37.5, 173; 616 of them 6.8, 19.5,
    // 39.4, 137 and 7.3, 18.8, 37.7, 173; 1008 of them 7.5, 21.2, 41.5, 187 and 7.3, 19.1, 37.6, 173.  Heads of 32: 512 4.5, 6.5, 9.2, 29 and 4.9, 8.9, 15.9, 61;
    // 616 4.9, 10.1, 14.9, 40 and 4.9, 9.0, 16.1, 60; 2048 7.4, 18.5, 28.1, 97 and 5.6, 11.9, 23.3, 96.  bfloat16 alike.
    const bool split = (long long)n_tokens * n_heads <= 512;
    const dim3 grid(split ? n_tokens : (n_tokens + ATT_WAVES - 1) / ATT_WAVES, n_heads);
    // four elements a load where keys and values begin at a multiple of four elements (a caller's memory need not) and rows of keys do, too
    const size_t four = act_dtype == TQK_F32 ? 16 : 8;
    const int wide_keys = head_dim % 4 == 0 && (uintptr_t)keys % four == 0, wide_values = (uintptr_t)values % four == 0;
#define LAUNCH(T, SPLIT) attention_generic_kernel<T, SPLIT><<<grid, (SPLIT ? ATT_STRIPES : ATT_WAVES) * TQK_WAVE, 0, s>>>( \
            (const T*)q, (const T*)keys, (const T*)values, tok_seq, tok_pos, page_table, table_width, \
            window, scale, (T*)out, n_tokens, n_heads, n_kv_heads, head_dim, wide_keys, wide_values)
    const int group = n_heads / n_kv_heads, heads = wide_keys && wide_values && act_dtype == TQK_F32 ? heads_together(n_tokens, group, n_kv_heads, head_dim, table_width, window) : 0;
    if (heads) {
        const dim3 blocks(n_tokens, n_kv_heads * ((group + heads - 1) / heads));
#define HEADS_LAUNCH(HEADS, NACC) attention_heads_kernel<HEADS, NACC><<<blocks, ATT_STRIPES * TQK_WAVE, 0, s>>>( \
            (const float*)q, (const float*)keys, (const float*)values, tok_seq, tok_pos, page_table, table_width, window, scale, (float*)out, n_heads, n_kv_heads, head_dim)
#define OF_HEADS(HEADS) do { if (head_dim <= 64) HEADS_LAUNCH(HEADS, 1); else HEADS_LAUNCH(HEADS, 2); } while (0)
        if (heads == 8) OF_HEADS(8); else if (heads == 4) OF_HEADS(4); else OF_HEADS(2);
#undef OF_HEADS
#undef HEADS_LAUNCH
        return tqk_check_launch("tqk_attention");
    }
    if (act_dtype == TQK_F32) {
        if (split) LAUNCH(float, true); else LAUNCH(float, false);
    } else if (act_dtype == TQK_BF16) {
        if (split) LAUNCH(bf16_t, true); else LAUNCH(bf16_t, false);
    } else
#undef LAUNCH
        return tqk_fail("tqk_attention: unknown dtype %d", act_dtype);
    return tqk_check_launch("tqk_attention");
}
