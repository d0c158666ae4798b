// Attention for decoding: one new token per sequence attends over its sequence's pages
// of the cache.  bfloat16 in, MFMA, float32 softmax.  Bound by the bytes of keys and
// values, so the work is cut for memory: a block of 4 waves (2 in large grids, 1 where a block has one page) per (sequence, kv head,
// partition of the pages); the partitions take the live pages in turn (partition p the pages
// first + p, first + p + parts, ...: however long the sequence is, they get the same share)
// and so do the four waves inside a partition; all
// query heads that share the kv head ride in the same wave, so keys and values are
// read once for the whole group (the reference expands them per query head instead,
// src/models/turbo_generic.rs:195-204, 1620-1621).  The waves' results are merged
// through LDS; with one partition the block writes the result itself, with more a
// second kernel merges the partitions in their order.  (Merging in the last block to
// finish, behind a device-wide fence, was measured to cost more than the second launch.)
// Formulas as src/models/turbo_generic.rs:1622-1631, :56-62.
//
// Matrix-core mapping (v_mfma_f32_16x16x32_bf16, D[16x16] += A[16x32] B[32x16]):
//   scores^T[key][head] = K[key][:] . Q^T[:][head]
//       A = 16 keys x 32 elements of head_dim: lane l reads 16 contiguous bytes of key row
//           l%16 straight from the page; B = the heads' query rows, read the same way.
//       The lane then holds, for head l%16, the keys 4*(l/16)+r (r=0..3) of the 16.
//   out^T[element][head] = V^T[element][key] . P^T[key][head]
//       B needs for head l%16 eight keys per lane: the lane already holds them, the four
//       of one group of 16 keys and the four of the next (slot j<4: key 4g+j, j>=4: key
//       16+4g+j-4), so P never leaves its registers.  A must pair the same keys with the
//       slots: the cache keeps values transposed and in exactly this order inside a page
//       (value_place in common.h), 16 contiguous bytes per lane.
// Keys outside [lo, pos] get probability exactly 0 and their values are replaced by 0
// before the product, so nothing stored at such places can reach the result.
#include "common.h"
#include "tq_kernels.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef floatx4_t floatx4_any_t __attribute__((aligned(4)));         // at any float's address
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int wave_of_block() { return threadIdx.x / TQK_WAVE; }

union pack8 {
    bf16x8_t v;
    uint16_t u[8];
    uint4 q;
};

#define AD_WAVES 4            // the most; blocks of 2 where the grid alone is more than the memory can serve at once

// The step's q, k and v as the sums over pieces of K that their product left (mid_product.hip), with what makes them queries and cache
// entries: the work of tqk_rope_store_sums for one row.
struct DecodeSums {
    const float* sums;              // [n][rows][(heads + 2 kv heads) * head_dim]
    int n;
    size_t stride;
    const bf16_t* bias;             // or null
    const float *cos_table, *sin_table;         // [max_positions, head_dim / 2]
    int max_positions;
    bf16_t *keys, *values;          // the cache, to write
};

// A block's part of that work: the queries of its heads (n_live of them from head0 on) into LDS, rows of D + 8, and the row's new key and value
// behind them; where the block reads the row's own position (owner), also into the cache.  A job is twice four values, D / 2 apart, that
// rotate with each other.  The first job's loads are issued by `ask`, so that a page's loads can be on their way behind them while the sums
// are added up by `finish`: the block does not read what it writes to the cache, it takes the new key and value out of LDS.
template <int D>
struct RowFinish {
    static constexpr int PER = D / 8, BATCH = 8;
    const DecodeSums& in;
    const int seq, head0, n_live, kvh, n_heads, n_kv_heads;
    uint2 b_lo, b_hi;
    floatx4_t pa[BATCH], pb[BATCH];

    __device__ __forceinline__ size_t feature_of(int job) const {
        const int which = min(job / PER, n_live + 1), i = (job % PER) * 4;
        return (size_t)(which < n_live ? head0 + which : n_heads + (which - n_live) * n_kv_heads + kvh) * D + i;
    }
    // the bias and up to eight pieces, all under way together
    __device__ __forceinline__ void ask(int job, int s0) {
        const size_t feature = feature_of(job), at = (size_t)seq * (n_heads + 2 * n_kv_heads) * D + feature;
        if (s0 == 0) {
            b_lo = b_hi = make_uint2(0, 0);
            if (in.bias) {
                b_lo = *reinterpret_cast<const uint2*>(in.bias + feature);
                b_hi = *reinterpret_cast<const uint2*>(in.bias + feature + D / 2);
            }
        }
        auto half = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = u0; u < u0 + BATCH / 2; ++u) {
                const float* src = in.sums + (size_t)min(s0 + u, in.n - 1) * in.stride + at;
                pa[u] = *reinterpret_cast<const floatx4_t*>(src);
                pb[u] = *reinterpret_cast<const floatx4_t*>(src + D / 2);
            }
        };
        half(0);
        if (s0 + BATCH / 2 < in.n) half(BATCH / 2);
    }
    // the values at their rounding to bfloat16 and the bias added: the pieces in their order
    __device__ __forceinline__ void sum(int job, float (&lo)[4], float (&hi)[4]) {
        floatx4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
        auto add = [&](int s) {
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
                const bool there = s + u < in.n;
#pragma unroll
                for (int k = 0; k < 4; ++k) { a[k] = there ? a[k] + pa[u][k] : a[k]; b[k] = there ? b[k] + pb[u][k] : b[k]; }
            }
        };
        add(0);
        for (int s = BATCH; s < in.n; s += BATCH) {
            ask(job, s);
            add(s);
        }
        const float bias_lo[4] = {__uint_as_float(b_lo.x << 16), __uint_as_float(b_lo.x & 0xffff0000u), __uint_as_float(b_lo.y << 16), __uint_as_float(b_lo.y & 0xffff0000u)};
        const float bias_hi[4] = {__uint_as_float(b_hi.x << 16), __uint_as_float(b_hi.x & 0xffff0000u), __uint_as_float(b_hi.y << 16), __uint_as_float(b_hi.y & 0xffff0000u)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lo[k] = to_float(from_float<bf16_t>(a[k]));
            hi[k] = to_float(from_float<bf16_t>(b[k]));
            if (in.bias) { lo[k] += bias_lo[k]; hi[k] += bias_hi[k]; }
        }
    }
    // (c4, s4: the angles of the first job, asked for before)
    __device__ __forceinline__ void finish(int pos, int page, bool owner, float4 c4, float4 s4, bf16_t* q_lds, bf16_t* new_lds) {
        const int jobs = (n_live + (owner ? 2 : 0)) * PER;
        auto one = [&](int job) __attribute__((always_inline)) {
            const int which = job / PER, i = (job % PER) * 4;
            const int kind = which < n_live ? 0 : which - n_live + 1;
            float lo[4], hi[4];
            sum(job, lo, hi);
            if (kind != 2 && pos < in.max_positions) {
                const float c[4] = {c4.x, c4.y, c4.z, c4.w}, sn[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) rotate_pair(lo[k], hi[k], c[k], sn[k]);
            }
            uint32_t l[4], h[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) { l[k] = float_to_bf16_bits(lo[k]); h[k] = float_to_bf16_bits(hi[k]); }
            const uint2 l4 = make_uint2(l[0] | (l[1] << 16), l[2] | (l[3] << 16)), h4 = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
            bf16_t* dst = kind == 0 ? q_lds + which * (D + 8) : new_lds + (kind - 1) * D;
            *reinterpret_cast<uint2*>(dst + i) = l4;
            *reinterpret_cast<uint2*>(dst + i + D / 2) = h4;
            // (blocks that share a kv head and a page write the same values)
            if (kind == 1) {
                bf16_t* key = in.keys + (((size_t)page * n_kv_heads + kvh) * TQK_PAGE + pos % TQK_PAGE) * D;
                *reinterpret_cast<uint2*>(key + i) = l4;
                *reinterpret_cast<uint2*>(key + i + D / 2) = h4;
            } else if (kind == 2) {
                bf16_t* value = in.values + ((size_t)page * n_kv_heads + kvh) * TQK_PAGE * D + value_place(pos % TQK_PAGE);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    value[(size_t)(i + k) * TQK_PAGE].bits = (uint16_t)l[k];
                    value[(size_t)(i + D / 2 + k) * TQK_PAGE].bits = (uint16_t)h[k];
                }
            }
        };
        if ((int)threadIdx.x < jobs) one(threadIdx.x);          // (apart, so that its waits are counted and leave a page's loads under way)
        for (int job = threadIdx.x + blockDim.x; job < jobs; job += blockDim.x) {
            ask(job, 0);
            const size_t angle = (size_t)min(pos, in.max_positions - 1) * (D / 2) + (job % PER) * 4;
            c4 = *reinterpret_cast<const float4*>(in.cos_table + angle);
            s4 = *reinterpret_cast<const float4*>(in.sin_table + angle);
            one(job);
        }
        __syncthreads();
    }
};

// With a page or two a wave the kernel is bound by what a block does one thing after the other, not by bytes.  Stamps of one launch (32 rows of up to
// 1024 positions, 12 heads on 2, sums of 3 pieces, us from its start, the last block): position known 1.9, loads asked for 5.6, sums finished
// 6.5, page there 7.1, page done 8.7, written 9.8.  A page that is not whole took 4 us longer while each of its values was compared with the
// positions (bits to keep are found once for all elements now), the sums 1.3 in front of the page's loads instead of over them, and the
// waves' results 1.3 when one wave added up all of them.  ms a step, together: 7B, 1, 8 and 64 sequences 2.882 -> 2.832, 3.130 -> 3.058 and
// 3.921 -> 3.793; 1.5B, 32 sequences 1.766 -> 1.657; 32B with 8 layers, 16 sequences 1.843 -> 1.816.
// SUMS: q, k and v come as `in` and are finished here (keys and values are then written, too, so nothing promises that they are not); SUMS_EARLY: the
// first page is asked for while the sums are added up.
enum { NO_SUMS = 0, SUMS_FIRST = 1, SUMS_EARLY = 2 };
template <int D, bool NT, int W, int SUMS>
__global__ __launch_bounds__(AD_WAVES * TQK_WAVE)
void attention_decode_kernel(const DecodeSums in, const bf16_t* __restrict__ q, const bf16_t* keys,
                             const bf16_t* values, const int32_t* __restrict__ tok_pos,
                             const int32_t* __restrict__ page_table, int table_width, int window, float scale,
                             int n_parts, int n_heads, int n_kv_heads, int q_blocks,
                             float* __restrict__ part_out, float* __restrict__ part_ml,
                             bf16_t* __restrict__ out) {
    constexpr int KB = D / 32;          // k-blocks of the score product
    constexpr int DB = D / 16;          // 16-element blocks of the output
    // Head size 128: a page comes in with loads of 1 KB of contiguous memory each and goes through LDS into the matrix
    // cores' order, a region of 16 KB per wave (see below); the waves' results change hands through the same memory.
    // (Worth it where the step reads so much that the memory's rate counts, which is where the loads are marked as
    // read-once, NT: 64 sequences of 2100 positions 56.2 -> 49.7 us, 128 sequences 106 -> 89 us; 8 sequences 13.2 -> 14.2.)
    constexpr bool VIA_LDS = D == 128 && NT;
    constexpr bool EARLY = SUMS == SUMS_EARLY;
    constexpr int XCH_WAVE = DB * TQK_WAVE + TQK_WAVE / 2;      // pieces of 16 bytes a wave hands over: its out^T values, m, l
    constexpr int XCH = W > 1 ? W * XCH_WAVE : 1, TURN = VIA_LDS ? W * 1024 : 0;
    __shared__ u32x4_t lds_all[XCH > TURN ? XCH : TURN];
    floatx4_t* const xch = reinterpret_cast<floatx4_t*>(lds_all);
    u32x4_t* const turn = lds_all + wave_of_block() * 1024;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TQK_WAVE), lane = threadIdx.x % TQK_WAVE;
    const int col = lane % 16, g = lane / 16;
    const int part = blockIdx.x;
    const int kvh = blockIdx.y / q_blocks, qb = blockIdx.y % q_blocks;
    const int seq = blockIdx.z;
    const int n_rep = n_heads / n_kv_heads;
    // What a block waits for before its pages is a chain of loads that miss all caches, about a microsecond each, so nothing waits that need not:
    // without a window the name of the wave's first page is asked for first, then the sums, then the position, and none is looked at before.
    const int32_t* pages = page_table + (size_t)seq * table_width;
    int page = 0;
    if (window == 0) page = __builtin_amdgcn_readfirstlane(pages[min(part + wave * n_parts, table_width - 1)]);
    __shared__ __attribute__((aligned(16))) bf16_t q_lds[SUMS ? 16 * (D + 8) : 8], new_lds[SUMS ? 2 * D : 8];
    RowFinish<SUMS ? D : 32> finish = {in, seq, kvh * n_rep + qb * 16, min(16, n_rep - qb * 16), kvh, n_heads, n_kv_heads};
    if constexpr (EARLY) {
        finish.ask(threadIdx.x, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    const int pos = __builtin_amdgcn_readfirstlane(tok_pos[seq]);
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    // exponentials to base 2 (one instruction each): the scores carry log2(e), and so do the running
    // maxima m here, in part_ml and in the merge kernel
    const float scale2 = scale * 1.4426950408889634f;

    // the query head of this lane's column
    const int rep = qb * 16 + col;
    const bool head_live = rep < n_rep;
    const int head = kvh * n_rep + (head_live ? rep : 0);

    const int first_page = lo / TQK_PAGE, last_page = pos / TQK_PAGE;
    const int start_page = first_page + part + wave * n_parts;          // this wave's first page
    if (window > 0) page = __builtin_amdgcn_readfirstlane(pages[min(start_page, table_width - 1)]);

    float m = -INFINITY, l = 0.f;
    floatx4_t o[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) o[i] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // all of a page's loads together, so that they are in flight together
    bf16x8_t ka[4][KB], va[DB][2];
    u32x4_t kr[VIA_LDS ? 16 : 1], vr[VIA_LDS ? 16 : 1];
    auto load_page = [&](int page, int lane) __attribute__((always_inline)) {
        const int col = lane % 16, g = lane / 16;
        const size_t at = ((size_t)page * n_kv_heads + kvh) * TQK_PAGE * D;
        const bf16_t *kp = keys + at, *vp = values + at;
        if constexpr (VIA_LDS) {
            // A load of a wave takes 1 KB of contiguous memory (four key rows, eight value rows): the memory serves
            // such loads at 6.9 TB/s and loads of 64 bytes out of each of 16 rows, which is what the matrix cores'
            // order asks of a page as it lies in the cache, at 5.9.  The pieces of 16 bytes then go through the wave's
            // region of LDS to the lanes that need them, XOR-swizzled so that neither the writes nor the reads meet
            // a bank twice: the keys first, and the values through the same region once the scores are done.
            const u32x4_t* kg = reinterpret_cast<const u32x4_t*>(kp) + lane;
            const u32x4_t* vg = reinterpret_cast<const u32x4_t*>(vp) + lane;
#pragma unroll
            for (int j = 0; j < 16; ++j) kr[j] = __builtin_nontemporal_load(kg + j * 64);
#pragma unroll
            for (int j = 0; j < 16; ++j) vr[j] = __builtin_nontemporal_load(vg + j * 64);
        } else {
            auto load = [](const bf16_t* p) { return NT ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(p)) : *reinterpret_cast<const bf16x8_t*>(p); };
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) ka[t][kb] = load(kp + (size_t)(t * 16 + col) * D + kb * 32 + g * 8);
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int pr = 0; pr < 2; ++pr) va[db][pr] = load(vp + (size_t)(db * 16 + col) * TQK_PAGE + pr * 32 + g * 8);
        }
    };

    if constexpr (SUMS) {
        const int row_page = __builtin_amdgcn_readfirstlane(pages[last_page]);
        const size_t angle = (size_t)min(pos, in.max_positions - 1) * (D / 2) + (threadIdx.x % (D / 8)) * 4;
        const float4 c4 = *reinterpret_cast<const float4*>(in.cos_table + angle), s4 = *reinterpret_cast<const float4*>(in.sin_table + angle);
        __builtin_amdgcn_sched_barrier(0);
        if (!EARLY) finish.ask(threadIdx.x, 0);
        // (a wave without a page asks for a few lines of some page, so that the count of loads under way is the same)
        const bool live = start_page <= last_page && page >= 0;
        if (EARLY) load_page(live ? page : 0, live ? lane : 0);
        __builtin_amdgcn_sched_barrier(0);
        const bool owner = (last_page - first_page) % n_parts == part && row_page >= 0;
        finish.finish(pos, row_page, owner, c4, s4, q_lds, new_lds);
    }

    if (start_page <= last_page) {
        pack8 zero;
        zero.q = make_uint4(0, 0, 0, 0);
        // the heads' queries: B operand of the score product
        bf16x8_t bq[KB];
        const bf16_t* qrow = q + ((size_t)seq * n_heads + head) * D + g * 8;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            bq[kb] = head_live ? *reinterpret_cast<const bf16x8_t*>(SUMS ? q_lds + col * (D + 8) + g * 8 + kb * 32 : qrow + kb * 32) : zero.v;

        for (int pg = start_page; pg <= last_page; pg += W * n_parts) {
            const int next_pg = pg + W * n_parts;
            const int next = __builtin_amdgcn_readfirstlane(pages[min(next_pg, last_page)]);        // the same in all lanes: the page's address is then a scalar
            const int here = page;
            page = next;
            if (here < 0) continue;                     // the host never lets this happen
            if (!EARLY || pg != start_page) load_page(here, lane);
            const int key0 = pg * TQK_PAGE;
            const bool newest = SUMS && pg == last_page;            // its last key and value are those that the block has finished itself
            const bool edge = newest || key0 < lo || key0 + TQK_PAGE - 1 > pos;

            if constexpr (VIA_LDS) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int key = 4 * j + lane / 16, oct = lane % 16;
                    turn[key * 16 + (oct ^ (key & 15))] = kr[j];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) {
                        const int key = t * 16 + col, oct = kb * 4 + g;
                        const u32x4_t piece = turn[key * 16 + (oct ^ (key & 15))];
                        ka[t][kb] = __builtin_bit_cast(bf16x8_t, piece);
                    }
                __builtin_amdgcn_wave_barrier();
            }
            if (newest) {
                const int at = pos % TQK_PAGE;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) {
                    const bf16x8_t k = *reinterpret_cast<const bf16x8_t*>(new_lds + kb * 32 + g * 8);
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (at == t * 16 + col) ka[t][kb] = k;
                }
            }

            // scores^T for the page's four groups of 16 keys
            floatx4_t s[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                s[t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
                    s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[t][kb], bq[kb], s[t], 0, 0, 0);
            }
            // mask, scale, running maximum (the lane's head is its column; its keys are
            // key0 + 16 t + 4 g + r)
            float mx = m;
            if (edge) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = key0 + t * 16 + g * 4 + r;
                        const float v = (j >= lo && j <= pos) ? s[t][r] * scale2 : -INFINITY;
                        s[t][r] = v;
                        mx = fmaxf(mx, v);
                    }
            } else {                                    // a page wholly inside [lo, pos]: nothing to mask
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        s[t][r] *= scale2;
                        mx = fmaxf(mx, s[t][r]);
                    }
            }
            float2 both = with_lane_16(mx);
            mx = fmaxf(both.x, both.y);
            both = with_lane_32(mx);
            mx = fmaxf(both.x, both.y);
            // mx is finite: the page holds at least one key of [lo, pos]
            const float alpha = __builtin_amdgcn_exp2f(m - mx);     // 2^(-inf) = 0 on the wave's first page
            m = mx;
            float psum = 0.f;
            pack8 pb[2];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = __builtin_amdgcn_exp2f(s[t][r] - mx);          // a masked key: 2^(-inf) = 0
                    // the probability enters the product as bfloat16; the sum uses the same rounded value
                    const uint16_t pbits = float_to_bf16_bits(p);
                    psum += __uint_as_float(((uint32_t)pbits) << 16);
                    pb[t / 2].u[(t % 2) * 4 + r] = pbits;
                }
            l = l * alpha + psum;
            if constexpr (VIA_LDS) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int d = 8 * j + lane / 8, oct = lane % 8;
                    turn[d * 8 + (oct ^ ((d >> 1) & 7))] = vr[j];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int pr = 0; pr < 2; ++pr) {
                        const int d = db * 16 + col, oct = pr * 4 + g;
                        const u32x4_t piece = turn[d * 8 + (oct ^ ((d >> 1) & 7))];
                        va[db][pr] = __builtin_bit_cast(bf16x8_t, piece);
                    }
                __builtin_amdgcn_wave_barrier();
            }
            if (edge) {
                // Which of a lane's values count, and which one is the new one, is the same for all elements of the head, so it is found once, as
                // bits to keep and to put in pairs of values.
                uint32_t keep[2][4], put[2][4];
#pragma unroll
                for (int pr = 0; pr < 2; ++pr)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const int j = key0 + (2 * pr + w / 2) * 16 + g * 4 + 2 * (w % 2);
                        const int in0 = j >= lo && j <= pos, in1 = j + 1 >= lo && j + 1 <= pos;
                        put[pr][w] = !newest ? 0u : j == pos ? 0xffffu : j + 1 == pos ? 0xffff0000u : 0u;
                        keep[pr][w] = ((in0 ? 0xffffu : 0u) | (in1 ? 0xffff0000u : 0u)) & ~put[pr][w];
                    }
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    const uint32_t v = SUMS ? new_lds[D + db * 16 + col].bits * 0x10001u : 0u;
#pragma unroll
                    for (int pr = 0; pr < 2; ++pr) {
                        u32x4_t u = __builtin_bit_cast(u32x4_t, va[db][pr]);
#pragma unroll
                        for (int w = 0; w < 4; ++w) u[w] = (u[w] & keep[pr][w]) | (SUMS ? v & put[pr][w] : 0u);
                        va[db][pr] = __builtin_bit_cast(bf16x8_t, u);
                    }
                }
            }
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                o[db][0] *= alpha; o[db][1] *= alpha; o[db][2] *= alpha; o[db][3] *= alpha;
#pragma unroll
                for (int pr = 0; pr < 2; ++pr) o[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[db][pr], pb[pr].v, o[db], 0, 0, 0);
            }
        }
        float2 both = with_lane_16(l);
        l = both.x + both.y;
        both = with_lane_32(l);
        l = both.x + both.y;
    }

    // The waves' results meet in wave order, each wave taking its share of the elements.
    if constexpr (W > 1) {
        if (VIA_LDS) __syncthreads();               // (the memory they change hands through is the regions of the pages)
        floatx4_t* mine = xch + (size_t)wave * XCH_WAVE + lane;
#pragma unroll
        for (int db = 0; db < DB; ++db) mine[db * TQK_WAVE] = o[db];
        float* ml = reinterpret_cast<float*>(xch + (size_t)wave * XCH_WAVE + DB * TQK_WAVE);
        ml[lane] = m;
        ml[TQK_WAVE + lane] = l;
        __syncthreads();
    }
    const size_t row = ((size_t)seq * n_heads + head) * n_parts + part;
    bool some[W];                                   // whether a wave had a page
    float of_others[W], of_sum[W];                  // what the sum so far and the wave's are multiplied by
    if constexpr (W > 1) {
        const float* ml = reinterpret_cast<const float*>(xch + DB * TQK_WAVE) + lane;
        m = ml[0];
        l = ml[TQK_WAVE];
#pragma unroll
        for (int w = 1; w < W; ++w) {
            const float m2 = ml[(size_t)w * XCH_WAVE * 4], l2 = ml[(size_t)w * XCH_WAVE * 4 + TQK_WAVE];
            const float mn = fmaxf(m, m2);
            some[w] = m2 != -INFINITY;
            of_sum[w] = __builtin_amdgcn_exp2f(m - mn);
            of_others[w] = __builtin_amdgcn_exp2f(m2 - mn);
            if (!some[w]) continue;
            l = l * of_sum[w] + l2 * of_others[w];
            m = mn;
        }
    }
    if (!head_live) return;
#pragma unroll
    for (int d0 = 0; d0 < DB; d0 += W) {
        const int db = d0 + (W > 1 ? wave : 0);
        if (DB % W != 0 && db >= DB) break;
        floatx4_t v = o[d0];
        if constexpr (W > 1) {
            const floatx4_t* from = xch + (size_t)db * TQK_WAVE + lane;
            v = from[0];
#pragma unroll
            for (int w = 1; w < W; ++w) {
                const floatx4_t theirs = from[(size_t)w * XCH_WAVE];
                if (some[w]) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = v[r] * of_sum[w] + theirs[r] * of_others[w];
                }
            }
        }
        if (n_parts == 1) {
            // the only partition: this is the result, out[head, element db*16 + 4g + r]
            bf16_t* po = out + ((size_t)seq * n_heads + head) * D + db * 16 + g * 4;
            const float inv = 1.f / l;
#pragma unroll
            for (int r = 0; r < 4; ++r) po[r] = from_float<bf16_t>(v[r] * inv);
        } else {
            *reinterpret_cast<floatx4_any_t*>(part_out + row * D + db * 16 + g * 4) = v;
        }
    }
    if (n_parts > 1 && wave == 0 && g == 0) { part_ml[row * 2] = m; part_ml[row * 2 + 1] = l; }
}

// weight * value, rounded whatever is done with it (the compiler would fuse it with the sum it goes into): a decoding step's bits go by it.
__device__ __forceinline__ float rounded_product(float weight, float value) {
#pragma clang fp contract(off)
    return weight * value;
}

// out[seq, head, :] = sum_p exp(m_p - M) o_p / sum_p exp(m_p - M) l_p, partitions in order.
// Bound by the loads it waits for one after the other (each misses every cache), so those of up to 16 partitions are asked for
// together, and up to 16 partitions take one round for maxima, sums and outputs alike: with four partitions of 32 rows and 12 heads a step of the 1.5B
// shape takes 1.65 -> 1.605 ms against a loop that took eight at a time and a remainder one after the other.  More go by 16 and what is left by 8: in a
// second round of 16, 17 partitions took longer than in that loop (attention and merge of 3 rows, 8 heads of 32 6.7 us, 7.1, now 6.7; 4 heads of 96, which
// two waves share now, 8.7, 9.3, 7.2).  A partition without keys (m = -inf) has weight 0 and its (unwritten) output is not looked at.
template <int N> struct Count { static constexpr int n = N; };
template <int BATCH, bool ONE_ROUND>
__global__ void attention_merge_kernel(const float* __restrict__ part_out, const float* __restrict__ part_ml,
                                       int n_parts, int head_dim, bf16_t* __restrict__ out) {
    const size_t row = blockIdx.x;                     // seq * n_heads + head
    const float2* ml = reinterpret_cast<const float2*>(part_ml) + row * n_parts;
    float M = -INFINITY;
    if (!ONE_ROUND) {
        const int lane = threadIdx.x % TQK_WAVE;
        for (int p = lane; p < n_parts; p += TQK_WAVE) M = fmaxf(M, ml[p].x);
        M = wave_max(M);
    }
    for (int c = threadIdx.x; c < head_dim; c += blockDim.x) {
        float acc = 0.f, denom = 0.f;
        const float* po = part_out + row * n_parts * head_dim + c;
        // (written out for B partitions from p0 on: what is left after rounds of 16 goes by 8)
        auto round = [&](int p0, auto batch) __attribute__((always_inline)) {
            constexpr int B = decltype(batch)::n;
            float2 s[B];
            float v[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int p = min(p0 + u, n_parts - 1);
                s[u] = ml[p];
                v[u] = po[(size_t)p * head_dim];
            }
            __builtin_amdgcn_sched_barrier(0);
            if (ONE_ROUND) {
#pragma unroll
                for (int u = 0; u < B; ++u) M = fmaxf(M, s[u].x);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const bool live = s[u].x != -INFINITY && p0 + u < n_parts;
                const float wgt = live ? __builtin_amdgcn_exp2f(s[u].x - M) : 0.f;
                denom = fmaf(wgt, s[u].y, denom);
                acc += live ? rounded_product(wgt, v[u]) : 0.f;
            }
        };
        // (a loop where there is one round, too: without it maxima are looked at before outputs are asked for)
        int p0 = 0;
        for (; ONE_ROUND ? p0 < n_parts : p0 + BATCH <= n_parts; p0 += BATCH) round(p0, Count<BATCH>{});
        if (!ONE_ROUND) for (; p0 < n_parts; p0 += 8) round(p0, Count<8>{});
        out[row * head_dim + c] = from_float<bf16_t>(acc / denom);
    }
}

extern "C" int tqk_attention_decode_supported(int head_dim) {
    return head_dim == 64 || head_dim == 128 || head_dim == 256 || head_dim == 32 || head_dim == 96;
}

static int attention_decode(const DecodeSums& in, const void* q, const void* keys, const void* values, const int32_t* tok_pos,
                            const int32_t* page_table, int table_width, int n_seqs, int n_pages, int window,
                            float scale, int n_parts, void* part_out, void* part_ml,
                            void* out, int n_heads, int n_kv_heads, int head_dim, void* stream) {
    TQK_REQUIRE((q || in.sums) && keys && values && tok_pos && page_table && out, "tqk_attention_decode: null pointer");
    TQK_REQUIRE(n_parts == 1 || (part_out && part_ml), "tqk_attention_decode: more than one partition needs part_out and part_ml");
    TQK_REQUIRE(n_seqs >= 0 && n_heads > 0 && n_kv_heads > 0, "tqk_attention_decode: bad sizes");
    TQK_REQUIRE(n_heads % n_kv_heads == 0, "tqk_attention_decode: %d heads are not a multiple of %d kv heads", n_heads, n_kv_heads);
    TQK_REQUIRE(tqk_attention_decode_supported(head_dim), "tqk_attention_decode: head_dim %d is not one of 32, 64, 96, 128, 256", head_dim);
    TQK_REQUIRE(table_width > 0 && n_pages > 0, "tqk_attention_decode: empty page table");
    TQK_REQUIRE(n_parts > 0 && n_parts <= 65535, "tqk_attention_decode: %d partitions", n_parts);
    TQK_REQUIRE(window >= 0, "tqk_attention_decode: negative window");
    const int q_blocks = (n_heads / n_kv_heads + 15) / 16;
    TQK_REQUIRE(n_seqs <= 65535 && n_kv_heads * q_blocks <= 65535, "tqk_attention_decode: grid too large");
    if (n_seqs == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    dim3 grid(n_parts, n_kv_heads * q_blocks, n_seqs);
    // Keys and values are read once per step.  Saying so in the loads pays where the step reads more of them than the
    // caches hold (64 sequences of 2100 positions at the 7B sizes: 56.2 against 57.5 us) and costs where it reads little
    // (8 sequences: 14.4 against 13.6 us), so it goes by the most that the step's tables can name.
    const bool nt = (double)n_seqs * table_width * n_kv_heads * TQK_PAGE * head_dim * 4.0 > 128e6;
    // Four waves a block; two where there are 512 blocks or more without partitions: then the memory has more
    // pages asked of it at once than it serves well (128 sequences x 4 kv heads of 2100 positions: 106 against 114 us).
    const bool two = n_parts == 1 && (long long)n_seqs * n_kv_heads * q_blocks >= 512;
#define LAUNCH_S(DD, NT, W, SUMS) attention_decode_kernel<DD, NT, W, SUMS><<<grid, W * TQK_WAVE, 0, s>>>( \
        in, (const bf16_t*)q, (const bf16_t*)keys, (const bf16_t*)values, tok_pos, page_table, table_width, window, scale, \
        n_parts, n_heads, n_kv_heads, q_blocks, (float*)part_out, (float*)part_ml, (bf16_t*)out)
    // A partition per page of the table: a block then has one page to read, and one wave does it (4 sequences of 2100
    // positions: 8.8 against 10.7 us with four waves on four pages each; one sequence 5.8 against 9.0).
    const bool one = n_parts > 1 && n_parts >= table_width;
    // Sums are finished by blocks of four waves alone: fewer lanes take the heads' values in two or three rounds (20 rows of 200 positions at the
    // 7B sizes, blocks of one wave: 3.435 ms a step against 3.400 with the rotation's own kernel).
    // The first page beside the sums, where the registers hold both (heads up to 128) and a unit gets one block: with both there is room for one only.  us
    // beside and after the sums, 8 kv heads of 128: 64 rows of up to 24, 200 and 1000 positions 13.6, 18.9, 45.1 and 8.5, 14.5, 46.5, 100 rows
    // 25.7, 33.7, 73.3 and 14.3, 31.3, 73.9; 4 kv heads, 100 rows 13.2, 17.5, 40.7 and 8.1, 13.5, 40.9.  One block a unit: see the kernel.
    const bool early = in.sums && (long long)n_seqs * n_kv_heads * q_blocks * n_parts <= 256;
#define LAUNCH_W(DD, W, SUMS) { if (nt) LAUNCH_S(DD, true, W, SUMS); else LAUNCH_S(DD, false, W, SUMS); }
#define LAUNCH(DD) { if (early && DD <= 128) LAUNCH_W(DD, 4, (DD <= 128 ? SUMS_EARLY : SUMS_FIRST)) else if (in.sums) LAUNCH_W(DD, 4, SUMS_FIRST) \
        else if (one) LAUNCH_W(DD, 1, NO_SUMS) else if (two) LAUNCH_W(DD, 2, NO_SUMS) else LAUNCH_W(DD, 4, NO_SUMS) }
    switch (head_dim) {
        case 32: LAUNCH(32); break;
        case 64: LAUNCH(64); break;
        case 96: LAUNCH(96); break;
        case 128: LAUNCH(128); break;
        case 256: LAUNCH(256); break;
    }
#undef LAUNCH_W
#undef LAUNCH_S
#undef LAUNCH
    if (tqk_check_launch("tqk_attention_decode")) return -1;
    if (n_parts == 1) return 0;
    const int threads = head_dim > 64 ? 128 : 64;
#define MERGE(BATCH, ONE) attention_merge_kernel<BATCH, ONE><<<n_seqs * n_heads, threads, 0, s>>>((const float*)part_out, (const float*)part_ml, n_parts, head_dim, (bf16_t*)out)
    if (n_parts <= 4) MERGE(4, true);
    else if (n_parts <= 8) MERGE(8, true);
    else if (n_parts <= 16) MERGE(16, true);
    else MERGE(16, false);
#undef MERGE
    return tqk_check_launch("tqk_attention_decode merge");
}

extern "C" int tqk_attention_decode(const void* q, const void* keys, const void* values, const int32_t* tok_pos,
                                    const int32_t* page_table, int table_width, int n_seqs, int n_pages, int window,
                                    float scale, int n_parts, void* part_out, void* part_ml,
                                    void* out, int n_heads, int n_kv_heads, int head_dim, void* stream) {
    const DecodeSums none = {};
    TQK_REQUIRE(q, "tqk_attention_decode: null pointer");
    return attention_decode(none, q, keys, values, tok_pos, page_table, table_width, n_seqs, n_pages, window, scale, n_parts, part_out, part_ml, out,
                            n_heads, n_kv_heads, head_dim, stream);
}

/* The same with the step's q, k and v product given as its sums over n_sums pieces of K, float32 [n_sums][n_seqs][(heads + 2 kv heads) *
 * head_dim]: bias (bfloat16 or null), rotation in halves over the whole head and the cache write happen here, as tqk_rope_store_sums
 * does them (16-byte aligned operands), and keys and values are written at the rows' positions. */
extern "C" int tqk_attention_decode_sums(const float* sums, int n_sums, const void* bias, const float* cos_table, const float* sin_table, int max_positions,
                                         void* keys, void* values, const int32_t* tok_pos, const int32_t* page_table, int table_width, int n_seqs,
                                         int n_pages, int window, float scale, int n_parts, void* part_out, void* part_ml,
                                         void* out, int n_heads, int n_kv_heads, int head_dim, void* stream) {
    TQK_REQUIRE(sums && n_sums > 0, "tqk_attention_decode_sums: no sums given");
    TQK_REQUIRE(cos_table && sin_table && max_positions > 0, "tqk_attention_decode_sums: no angle tables");
    TQK_REQUIRE(((((uintptr_t)sums) | ((uintptr_t)bias) | ((uintptr_t)cos_table) | ((uintptr_t)sin_table) | ((uintptr_t)keys)) & 15) == 0,
                "tqk_attention_decode_sums: operands must be 16-byte aligned");
    const DecodeSums in = {sums, n_sums, (size_t)n_seqs * (n_heads + 2 * n_kv_heads) * head_dim, (const bf16_t*)bias, cos_table, sin_table, max_positions,
                           (bf16_t*)keys, (bf16_t*)values};
    return attention_decode(in, nullptr, keys, values, tok_pos, page_table, table_width, n_seqs, n_pages, window, scale, n_parts, part_out, part_ml, out,
                            n_heads, n_kv_heads, head_dim, stream);
}
