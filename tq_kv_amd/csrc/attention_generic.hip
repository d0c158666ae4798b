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
// one wave walks all of them (many queries), or a wave each (few queries).  The order of
// operations for a query depends only on its position, never on the batch or on which of the two it is.
// Cache pages: keys [kv head][position][head_dim], values [kv head][head_dim][place of
// the position] (value_place in common.h).
#include "attention_walk.h"
#include "tq_kernels.h"

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

extern "C" int tqk_attention_max_head_dim(void) { return ATT_MAX_D; }

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
    // A wave per stripe while no unit gets more than two blocks of them; the results are the same.  us with a wave per stripe and with one for all,
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
    if (act_dtype == TQK_F32) {
        if (split) LAUNCH(float, true); else LAUNCH(float, false);
    } else if (act_dtype == TQK_BF16) {
        if (split) LAUNCH(bf16_t, true); else LAUNCH(bf16_t, false);
    } else
#undef LAUNCH
        return tqk_fail("tqk_attention: unknown dtype %d", act_dtype);
    return tqk_check_launch("tqk_attention");
}
