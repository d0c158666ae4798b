// A whole step of a small decoder in one launch: embedding, every layer, final norm and the head's logits, in one block.
//
// A model of a few hundred kilobytes a layer is bound by nothing but launches: its step is ten kernels a layer, each of which works for a
// microsecond and costs two to four in a replayed graph, and about as much again on the host.  One block on one compute unit runs
// the step with barriers in place of launches.  It pulls weights and does a row's work at a fraction of the chip's rate, so this is the better way only
// while that takes no longer than the launches it stands for: tqk_small_step_pays says where that is.  Two layers of 64 values, 3 sequences after
// 20 tokens, five steps asked for together: 27.1 us a step in bfloat16 and 30.7 in float32 for what a replayed graph of 21 kernels does in 75 and 87; three of 96: 35.5 and 64 for 79 and 115.
// What a phase between two barriers takes (three of 96, bfloat16, attention by vector instructions, as other heads than those of 32 and 64 have it, us): norm 0.6 to 0.8, q/k/v 0.6, rotation 0.7,
// attention 2.6, o 1.2, gate and up 1.5, down 1.3, none of it bytes or products but a wave's instructions one after the other, 4 and more cycles each.
//
// The step's rows stay in LDS: the stream h in float32, the operand of the next product (`a`: normed rows, then the attention's output),
// and that product's result (`b`: q, k and v, then the gated values).  A wave takes tiles of 16 output features and all rows; its
// weights come straight from memory, those of its first tile before the barrier in front of the product, so that they travel while the work
// before it is finished; in decoding steps of few rows out of LDS, where two waves bring them (SmallRing).
//
// Every sum has the order that the kernels of larger models give it, and every rounding its place, so a position's result has the same bits whichever way
// its step went.  In float32 that is gemm_generic.hip, elementwise.hip and attention_walk.h (within a page by the matrix cores where that is faster, attend_page).  In bfloat16 the order goes by the kind of step
// (SmallPlan): norms that are divided by behind their product in decoding steps of up to 16 rows (skinny_fused.hip), and the matrix cores' attention of
// attention_decode.hip and attention_prefill.hip for heads of 32 and 64.  Steps with more than a page of positions for such heads, and products whose K
// those kernels deal out to waves or cut into pieces, are left to them.
//
// (Eight or twelve waves in place of 16: more rows take 1.1 to 1.4 times as long.  The o product's first weights asked for before the attention: 3 us a step more, the
// registers spill.  All heads of a kv head, or two queries, side by side in a wave's attention, so that keys are read once or chains overlap: slower,
// 27 to 45 us for few rows, as lanes without a key then load, too.)
#include "attention_walk.h"
#include "tq_kernels.h"
#include <atomic>
#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

#define SS_WAVES 16
#define SS_THREADS (SS_WAVES * TQK_WAVE)
#define SS_BRING 2              // waves that bring weights into the ring, where there is one
#define SS_AHEAD 4              // units of 1 KB that each of them has under way besides one
#define SS_FEW 4                // rows that float32 steps with a ring have at most
#define SS_QUERIES 4            // queries whose weights a wave keeps at a time
#define SS_STEPS 4              // steps of k whose weights are under way together

// A lane's operands of a step of k, of weights and of x alike, are the 16 bytes at 16 (lane / 16) of 64 of row lane % 16: float32 16 k a step, bfloat16 32.
// The sums: row (of x) lane % 16, features 4 (lane / 16) .. + 3.  float32 sums go by chunks of 8 steps, each from zero, as gemm_generic.hip has them.
__device__ __forceinline__ void multiply(float, floatx4_t& acc, u32x4_t w, u32x4_t x) {
    const floatx4_t wf = __builtin_bit_cast(floatx4_t, w), xf = __builtin_bit_cast(floatx4_t, x);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i], xf[i], acc, 0, 0, 0);
}
__device__ __forceinline__ void multiply(bf16_t, floatx4_t& acc, u32x4_t w, u32x4_t x) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
}
__device__ __forceinline__ void put4(float* p, floatx4_t v) { *reinterpret_cast<floatx4_t*>(p) = v; }
__device__ __forceinline__ void put4(bf16_t* p, floatx4_t v) {
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)float_to_bf16_bits(v[0]) | (uint32_t)float_to_bf16_bits(v[1]) << 16,
                                              (uint32_t)float_to_bf16_bits(v[2]) | (uint32_t)float_to_bf16_bits(v[3]) << 16);
}
template <typename T> __device__ __forceinline__ floatx4_t rounded(floatx4_t v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = to_float(from_float<T>(v[i]));
    return v;
}

// A barrier for what lies in LDS: loads from memory may stay under way across it (__syncthreads waits for them, and a product's first
// weights are asked for in front of one).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What of a bfloat16 step's arithmetic goes by the kernels that it would run through otherwise.
struct SmallPlan {
    int behind, first_behind;               // norms are divided by behind their product: those in front of gate and up and of the head; those in front of q, k and v
    int attention, last_attention;          // (last: the last layer's, where it runs for the last rows alone)
};
static_assert(sizeof(TqkSmallStep) + sizeof(SmallPlan) <= 4096, "a kernel's arguments");
enum { SMALL_ROWS = 1, SMALL_TILES = 2 };          // attention_decode.hip, attention_prefill.hip (heads that they do not take: attention_walk.h)

// y[rows, N] = x[rows, K] w[N, K]^T of rows in LDS, for P weights at once (gate and up rows of the same features).  A wave takes tiles of 16
// features by 16 rows, the rows' tiles of some features one after the other.  `ask` loads the first steps of the wave's first tile; emit(row, first feature,
// four features' sums[P]) takes the results.  N: up to where rows of the weight are read (those behind it repeat the last); K whole steps.
template <typename T, int P>
struct SmallProduct {
    const char* w[P];
    int N, bytes, row_tiles, lane, wave;                // bytes: of a row of the weight
    u32x4_t first[P][SS_STEPS];

    __device__ __forceinline__ void load(int tile, int b0) {
        const uint32_t at = (uint32_t)(min(tile * 16 + lane % 16, N - 1) * bytes + b0 + lane / 16 * 16);
#pragma unroll
        for (int u = 0; u < SS_STEPS; ++u) {
            if (b0 + 64 * u >= bytes) break;
#pragma unroll
            for (int p = 0; p < P; ++p) first[p][u] = *reinterpret_cast<const u32x4_t*>(w[p] + (at + 64 * u));
        }
    }
    __device__ __forceinline__ int tile_of(int unit) const { return row_tiles == 1 ? unit : unit / row_tiles; }
    __device__ __forceinline__ void ask() { if (tile_of(wave) * 16 < N) load(tile_of(wave), 0); }

    template <typename F>
    __device__ __forceinline__ void run(const T* x, int ldx, int rows, F&& emit) {
#pragma unroll 1
        for (int unit = wave;; unit += SS_WAVES) {
            const int tile = tile_of(unit), r0 = (unit - tile * row_tiles) * 16;
            if (tile * 16 >= N) break;
            floatx4_t acc[P], total[P];
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p] = total[p] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            const char* xr = (const char*)(x + (r0 + lane % 16) * ldx) + lane / 16 * 16;
#pragma unroll 1
            for (int b0 = 0; b0 < bytes; b0 += 64 * SS_STEPS) {
                if (unit != wave || b0 != 0) load(tile, b0);
#pragma unroll
                for (int u = 0; u < SS_STEPS; ++u) {
                    if (b0 + 64 * u >= bytes) break;
                    const u32x4_t xv = *reinterpret_cast<const u32x4_t*>(xr + b0 + 64 * u);
#pragma unroll
                    for (int p = 0; p < P; ++p) multiply(T(), acc[p], first[p][u], xv);
                }
                if (sizeof(T) == 4 && (b0 % (128 * SS_STEPS) != 0 || b0 + 64 * SS_STEPS >= bytes))
#pragma unroll
                    for (int p = 0; p < P; ++p) { total[p] += acc[p]; acc[p] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
            }
            if (r0 + lane % 16 < rows) emit(r0 + lane % 16, tile * 16 + lane / 16 * 4, sizeof(T) == 4 ? total : acc);
        }
    }
};

// Decoding steps of few rows: the weights' way into LDS.  Two waves of the block do nothing but bring them in, by loads that end there, ahead of the products.  A compute unit is served 12 to
// 20 bytes a cycle by the second-level cache whoever asks, and where the computing waves asked, a product's barrier waited until the next one's loads had been taken.  The
// weights lie in a ring: a layer's q/k/v, o, gate and up, down, and in the end the head, each in units of 1 KB, the ring as large as the most that is in use and on its way together.
// Rows one after the other, their pieces of 16 bytes turned by the row (`turned`), so that the 16 rows of an operand meet different banks.
// Cycles of one layer's phases before and now (two of 64 values, 3 rows, float32, stamps of the clock; with RingFewProduct): first norm 2160 and 1390, o 3700 and 1630, gate and up 5640 and
// 3460, down 4370 and 3200; the step 31.2 -> 28.3 us, three layers of 96 in bfloat16, 4 rows, 34.7 -> 32.8.  Each of the two has few units under way (SS_AHEAD), since what the other waves ask for waits
// behind them (attention 9000 -> 8400 cycles), and a weight is brought in the phases that leave time for it (down's and the next q/k/v's in thirds: gate and up 3900 -> 3460, down 3670 -> 3200).
struct SmallRing {
    int qkv, o, gate_up, down, head, bytes;         // a weight's size in units' bytes, and the ring's
};
static __device__ __host__ inline SmallRing small_ring(const TqkSmallStep& p) {
    const int size = p.act_dtype == TQK_F32 ? 4 : 2, q = p.n_heads * p.head_dim, all = (p.n_heads + 2 * p.n_kv_heads) * p.head_dim;
    auto up = [&](long long n) { n = (n * size + 1023) / 1024 * 1024; return (int)(n < 1 << 20 ? n : 1 << 20); };
    SmallRing r;
    r.qkv = up((long long)all * p.hidden);
    r.o = up((long long)p.hidden * q);
    r.gate_up = up(2ll * p.inter * p.hidden);
    r.down = up((long long)p.hidden * p.inter);
    r.head = up((long long)p.vocab * p.hidden);
    const int together[5] = {r.qkv + r.o, r.o + r.gate_up, r.gate_up + r.down, r.down + r.qkv, p.n_want > 0 ? r.down + r.head : 0};
    r.bytes = 0;
    for (int n : together) r.bytes = n > r.bytes ? n : r.bytes;
    return r;
}
// by what a row's pieces of 16 bytes are turned (exclusive or): rows of an even number of 64 bytes by three bits
__device__ __forceinline__ int turned(int row, int row_bytes) { return row & (row_bytes % 128 == 0 ? 7 : 3); }

// a bringing wave's (number `which` of them): its units of a weight of `rows` rows into the ring, where the weight lies from `at` on; those of the thirds
// from .. to - 1 of it.  Returns the place behind the weight, once it is whole.
__device__ __forceinline__ int bring(const void* w, int rows, int row_bytes, char* ring, int ring_bytes, int at, int from, int to, int which, int lane) {
    const int pieces = row_bytes / 16, all = rows * row_bytes, third = all / (3 * SS_BRING * 1024) * SS_BRING * 1024;
    const float of_pieces = 1.f / (float)pieces;
    const __amdgpu_buffer_rsrc_t mem = __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, all, 0x00020000);
#pragma unroll 2
    for (int unit = from * third + which * 1024; unit < (to == 3 ? all : to * third); unit += SS_BRING * 1024) {
        const int piece = unit / 16 + lane, row = (int)(((float)piece + 0.5f) * of_pieces), source = piece ^ turned(row, row_bytes);       // (numbers this small: exact)
        const int place = at + unit;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(mem, (lds_ptr_t)(ring + (place >= ring_bytes ? place - ring_bytes : place)), 16, source * 16, 0, 0, 0);
        __builtin_amdgcn_s_waitcnt(0x0f70 | SS_AHEAD);          // (no more under way: what the others ask for waits behind them)
    }
    at += to == 3 ? (all + 1023) / 1024 * 1024 : 0;
    return at >= ring_bytes ? at - ring_bytes : at;
}
__device__ __forceinline__ void brought() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// SmallProduct with the weights in the ring from `at` on, by W waves; the second weight's rows N rows further on.
template <typename T, int P, int W>
struct RingProduct {
    const char* ring;
    int ring_bytes, at, N, bytes, row_tiles, lane, wave;

    template <typename F>
    __device__ __forceinline__ void run(const T* x, int ldx, int rows, F&& emit) const {
#pragma unroll 1
        for (int unit = wave;; unit += W) {
            const int tile = row_tiles == 1 ? unit : unit / row_tiles, r0 = (unit - tile * row_tiles) * 16;
            if (tile * 16 >= N) break;
            uint32_t even[P], odd[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int row = min(tile * 16 + lane % 16, N - 1) + p * N, turn = turned(row, bytes);
                const uint32_t start = at + row * bytes + ((lane / 16) ^ (turn & 3)) * 16;
                even[p] = start + (turn & 4) * 16;
                odd[p] = start - (turn & 4) * 16;
            }
            floatx4_t acc[P], total[P];
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p] = total[p] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            const char* xr = (const char*)(x + (r0 + lane % 16) * ldx) + lane / 16 * 16;
#pragma unroll 1
            for (int b0 = 0; b0 < bytes; b0 += 64 * SS_STEPS) {
                u32x4_t xv[SS_STEPS], wv[P][SS_STEPS];
#pragma unroll
                for (int u = 0; u < SS_STEPS; ++u) {
                    if (b0 + 64 * u >= bytes) break;
                    xv[u] = *reinterpret_cast<const u32x4_t*>(xr + b0 + 64 * u);
#pragma unroll
                    for (int p = 0; p < P; ++p) {
                        const uint32_t to = (u % 2 ? odd[p] : even[p]) + b0 + 64 * u;
                        wv[p][u] = *reinterpret_cast<const u32x4_t*>(ring + min(to, to - (uint32_t)ring_bytes));
                    }
                }
#pragma unroll
                for (int u = 0; u < SS_STEPS; ++u) {
                    if (b0 + 64 * u >= bytes) break;
#pragma unroll
                    for (int p = 0; p < P; ++p) multiply(T(), acc[p], wv[p][u], xv[u]);
                }
                if (sizeof(T) == 4 && (b0 % (128 * SS_STEPS) != 0 || b0 + 64 * SS_STEPS >= bytes))
#pragma unroll
                    for (int p = 0; p < P; ++p) { total[p] += acc[p]; acc[p] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
            }
            if (r0 + lane % 16 < rows) emit(r0 + lane % 16, tile * 16 + lane / 16 * 4, sizeof(T) == 4 ? total : acc);
        }
    }
};

// The same for up to four rows in float32, 64 features a wave: 4 x 4 x 1 instructions, whose 16 blocks are 64 features by four rows (8 cycles a k), where 16 x 16 x 4 take
// as long a k for 16 features.  That pays where the matrix cores are what a product waits for: gate and up (160 features of 64 k: 6100 -> 3500 cycles), the head, q/k/v; o and down have fewer tiles than
// SIMDs and wait for a chain of sums, 12 cycles a k here and 8 there.
// Each k enters its sum on its own, in the order that it has there: the same bits.  emit(feature, the four rows' sums[P]); x: rows that are not there may hold anything.
template <int P, int W>
struct RingFewProduct {
    const char* ring;
    int ring_bytes, at, N, bytes, lane, wave;

    template <typename F>
    __device__ __forceinline__ void run(const float* x, int ldx, F&& emit) const {
#pragma unroll 1
        for (int n0 = wave * 64; n0 < N; n0 += W * 64) {
            uint32_t start[P], turn[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int row = min(n0 + lane, N - 1) + p * N;
                start[p] = at + row * bytes;
                turn[p] = turned(row, bytes) * 16;
            }
            floatx4_t acc[P], total[P];
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p] = total[p] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            const float* xr = x + (lane % 4) * ldx + lane / 4;
#pragma unroll 2
            for (int b0 = 0; b0 < bytes; b0 += 64) {
                const float xv = xr[b0 / 4];
                floatx4_t wv[P][4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int p = 0; p < P; ++p) {
                        const uint32_t to = start[p] + ((b0 + 16 * u) ^ turn[p]);
                        wv[p][u] = *reinterpret_cast<const floatx4_t*>(ring + min(to, to - (uint32_t)ring_bytes));
                    }
#define FEW_K(k) _Pragma("unroll") for (int p = 0; p < P; ++p) acc[p] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv, wv[p][(k) / 4][(k) % 4], acc[p], 4, k, 0);
                FEW_K(0) FEW_K(4) FEW_K(8) FEW_K(12) FEW_K(1) FEW_K(5) FEW_K(9) FEW_K(13)
                FEW_K(2) FEW_K(6) FEW_K(10) FEW_K(14) FEW_K(3) FEW_K(7) FEW_K(11) FEW_K(15)
#undef FEW_K
                if (b0 % 512 == 448 || b0 + 64 >= bytes)
#pragma unroll
                    for (int p = 0; p < P; ++p) { total[p] += acc[p]; acc[p] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
            }
            if (n0 + lane < N) emit(n0 + lane, total);
        }
    }
};

// How a step's rows lie in LDS, in bytes: the step's arrays, the layers' arguments, the norms' weights and the biases of all layers, the rows' angles, the waves' probabilities, then
// the stream and the two buffers.  Rows begin 16 bytes past a multiple of the banks' width, so that the 16 rows of an operand meet different ones.
struct SmallLayout {
    int ld_h, ld_a, ld_b, layers, norms, biases, angles, probs, squares, a, b, h, bytes;       // ld_h in floats, ld_a in T, ld_b in bytes
};
// (waves: that compute, all 16, or 14 beside the ring, which gets the room that few queries leave)
static __device__ __host__ inline int queries_together(const TqkSmallStep& p, int waves) {
    const int width = p.head_dim <= 16 ? 16 : p.head_dim <= 32 ? 32 : 64, each = (p.n_rows * p.n_heads + waves - 1) / waves;
    return each < TQK_WAVE / width ? each : TQK_WAVE / width;
}
static __device__ __host__ inline SmallLayout small_layout(const TqkSmallStep& p, int waves) {
    const int size = p.act_dtype == TQK_F32 ? 4 : 2, q = p.n_heads * p.head_dim, all = (p.n_heads + 2 * p.n_kv_heads) * p.head_dim;
    const int rows = (p.n_rows + 15) / 16 * 16;
    SmallLayout l;
    auto up = [](int n) { return (n + 15) / 16 * 16; };
    l.ld_h = p.hidden + 4;
    l.ld_a = (p.hidden > q ? p.hidden : q) + 16 / size;
    l.ld_b = up(all * 4 > p.inter * size ? all * 4 : p.inter * size) + 16;
    l.layers = up(p.n_ints * 4);
    l.norms = l.layers + up(p.n_layers * (int)sizeof(TqkSmallLayer));
    l.biases = l.norms + up((2 * p.n_layers + 1) * p.hidden * size);
    l.angles = l.biases + up(p.n_layers * all * size);
    l.probs = l.angles + up(p.n_rows * p.head_dim * 4);
    l.squares = l.probs + waves * (waves == SS_WAVES ? SS_QUERIES : queries_together(p, waves)) * TQK_PAGE * 4;             // (one root mean square of a row, then the squares' sums of 16 columns each, up to 16 rows)
    l.h = l.squares + (size == 2 && p.decode && p.n_rows <= 16 ? 64 + p.hidden * 4 : 0);
    l.a = l.h + rows * l.ld_h * 4;
    l.b = l.a + up(rows * l.ld_a * size);
    l.bytes = l.b + rows * l.ld_b;
    return l;
}

// One query of the wave: row r's head, its values in LDS (q).
struct SmallQuery {
    const float* q;
    int pos, lo, kvh, page, row, head;           // page: of the cache, where pos and lo lie in one
    bool one_page;
};

// 16 bytes as floats: element i of them
__device__ __forceinline__ float element(float, u32x4_t v, int i) { return __uint_as_float(v[i]); }
__device__ __forceinline__ float element(bf16_t, u32x4_t v, int i) { return __uint_as_float(i & 1 ? v[i / 2] & 0xffff0000u : v[i / 2] << 16); }

// The weights of a query's keys, unnormalised and in LDS (weights[key of the page]), and their sum: attention_walk.h's for a single page.  A lane is a key,
// and takes its row by 16 bytes, four loads together (many queries are bound by the first-level cache's lines: every lane's are its own).
template <typename T>
__device__ __forceinline__ float small_scores(const SmallQuery& y, const T* keys, int n_kv_heads, int d, float scale, float* weights, int lane) {
    constexpr int PER = 16 / sizeof(T);
    const bool valid = lane >= y.lo % TQK_PAGE && lane <= y.pos % TQK_PAGE;
    float s = -INFINITY;
    if (valid) {                            // (none for places without a key)
        const T* kr = keys + ((size_t)y.page * n_kv_heads + y.kvh) * TQK_PAGE * d + lane * d;
        float dot = 0.f;
#pragma unroll 1
        for (int e0 = 0; e0 < d; e0 += 4 * PER) {
            u32x4_t k[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) if (e0 + u * PER < d) k[u] = *reinterpret_cast<const u32x4_t*>(kr + e0 + u * PER);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (e0 + u * PER >= d) break;
#pragma unroll
                for (int i = 0; i < PER; i += 4) {
                    const float4 q = *reinterpret_cast<const float4*>(y.q + e0 + u * PER + i);
                    dot = fmaf(q.x, element(T(), k[u], i), dot);
                    dot = fmaf(q.y, element(T(), k[u], i + 1), dot);
                    dot = fmaf(q.z, element(T(), k[u], i + 2), dot);
                    dot = fmaf(q.w, element(T(), k[u], i + 3), dot);
                }
            }
        }
        s = dot * scale;
    }
    const float at = from_max(wave_max(s)), w = valid ? expf(s - at) : 0.f;
    weights[lane] = w;
    return wave_sum(w);
}

// The weighted values of a page, in the order of the positions: this lane's element of its query (base: the element's row of the page).  Half of the row is
// asked for at once, since the positions lie in another order in it (value_place).  What lies outside of first .. last is not looked at (it may be anything).
template <typename T>
__device__ __forceinline__ float small_values(const T* base, const float* weights, int first, int last, int wave_first, int wave_last) {
    constexpr int LOADS = 32 * sizeof(T) / 16;
    float sum = 0.f;
#pragma unroll 1
    for (int b0 = wave_first & 32; b0 <= wave_last; b0 += 32) {
        u32x4_t v[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; ++u) v[u] = reinterpret_cast<const u32x4_t*>(base + b0)[u];
#pragma unroll
        for (int g = 0; g < 8; ++g) {                           // positions b0 + 4 g .. + 3 lie together, at place 8 (g % 4) + 4 (g / 4)
            const int j = b0 + 4 * g, at = 8 * (g % 4) + 4 * (g / 4);
            if (j > wave_last) break;
            if (j + 3 < wave_first) continue;
            const float4 w = *reinterpret_cast<const float4*>(weights + j);
            auto one = [&](int i, float weight) {
                const float value = element(T(), v[(at + i) * sizeof(T) / 16], (at + i) % (16 / (int)sizeof(T)));
                sum = fmaf(weight, j + i >= first && j + i <= last ? value : 0.f, sum);
            };
            one(0, w.x); one(1, w.y); one(2, w.z); one(3, w.w);
        }
    }
    return sum;
}

// eight values in bfloat16 already, as an operand of the matrix cores
__device__ __forceinline__ bf16x8_t operand8(const float* p) {
    u32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float2 two = *reinterpret_cast<const float2*>(p + 2 * i);
        v[i] = __float_as_uint(two.x) >> 16 | (__float_as_uint(two.y) & 0xffff0000u);
    }
    return __builtin_bit_cast(bf16x8_t, v);
}

// The heads of a kv head (no more than 16) for one row whose keys lie in one page, as attention_decode.hip takes them: q its heads' values, positions lo .. pos of the page.
// divided: what that kernel's partitions leave is divided by their sum, and not multiplied by its inverse.
template <int D>
__device__ __forceinline__ void attend_row(const float* q, int n_live, const bf16_t* keys, const bf16_t* values, int lo, int pos, float scale, bool divided,
                                           bf16_t* out, int lane) {
    constexpr int KB = D / 32, DB = D / 16;
    const int col = lane % 16, g = lane / 16;
    const bool live = col < n_live;
    const float scale2 = scale * 1.4426950408889634f;
    bf16x8_t bq[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
        const bf16x8_t none = {0, 0, 0, 0, 0, 0, 0, 0};
        bq[kb] = live ? operand8(q + col * D + kb * 32 + g * 8) : none;
    }
    floatx4_t s[4];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        s[t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(keys + (t * 16 + col) * D + kb * 32 + g * 8), bq[kb], s[t], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = t * 16 + g * 4 + r;
            s[t][r] = j >= lo && j <= pos ? s[t][r] * scale2 : -INFINITY;
            mx = fmaxf(mx, s[t][r]);
        }
    }
    float2 both = with_lane_16(mx);
    mx = fmaxf(both.x, both.y);
    both = with_lane_32(mx);
    mx = fmaxf(both.x, both.y);
    float l = 0.f;
    u32x4_t pb[2];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            const uint32_t a = float_to_bf16_bits(__builtin_amdgcn_exp2f(s[t][r] - mx)), b = float_to_bf16_bits(__builtin_amdgcn_exp2f(s[t][r + 1] - mx));
            l += __uint_as_float(a << 16);
            l += __uint_as_float(b << 16);
            pb[t / 2][(t % 2) * 2 + r / 2] = a | b << 16;
        }
    both = with_lane_16(l);
    l = both.x + both.y;
    both = with_lane_32(l);
    l = both.x + both.y;
    uint32_t keep[2][4];                    // (whatever lies at places without a key must not count, not even with probability 0)
#pragma unroll
    for (int pr = 0; pr < 2; ++pr)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = (2 * pr + i / 2) * 16 + g * 4 + 2 * (i % 2);
            keep[pr][i] = (j >= lo && j <= pos ? 0xffffu : 0u) | (j + 1 >= lo && j + 1 <= pos ? 0xffff0000u : 0u);
        }
    const float inv = 1.f / l;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        floatx4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
            u32x4_t v = *reinterpret_cast<const u32x4_t*>(values + (db * 16 + col) * TQK_PAGE + pr * 32 + g * 8);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] &= keep[pr][i];
            o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, v), __builtin_bit_cast(bf16x8_t, pb[pr]), o, 0, 0, 0);
        }
        if (!live) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = divided ? (0.f + o[r]) / l : o[r] * inv;
        put4(out + col * D + db * 16 + g * 4, o);
    }
}

// 32 columns (a query and a head each) of one sequence and kv head whose keys lie in one page, as attention_prefill.hip takes them: q and out the lane's query and head;
// positions lo .. pos of the page (none: pos < 0), the sequence's end after the step, and how far any of the columns sees.
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16_t;
template <int D>
__device__ __forceinline__ void attend_columns(const float* q, const bf16_t* keys, const bf16_t* values, int lo, int pos, int end, int furthest, float scale, bf16_t* out, int lane) {
    constexpr int KS = D / 16, DT = D / 32;
    const int c32 = lane % 32, h = lane / 32;
    const bool live = pos >= 0;
    const float c2 = scale * 1.44269504088896340736f;
    bf16x8_t bq[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const bf16x8_t none = {0, 0, 0, 0, 0, 0, 0, 0};
        bq[ks] = live ? operand8(q + ks * 16 + h * 8) : none;
    }
    float m = 0.f, pass = -INFINITY, l = 0.f;
    floatx16_t o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    const int key = 4 * (2 * (c32 >> 4) + (c32 >> 2 & 1)) + 16 * (c32 >> 3 & 1) + (c32 & 3);      // that row c32 of a tile holds
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
        if (32 * t > furthest) break;
        floatx16_t s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(keys + (32 * t + key) * D + ks * 16 + h * 8), bq[ks], s, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int a = i >> 2, j = 32 * t + 4 * (2 * (a >> 1) + h) + 16 * (a & 1) + (i & 3);
            if (j < lo || j > pos) s[i] = -INFINITY;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], c2, -m);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
        const float2 both = with_lane_32(mx);
        mx = fmaxf(both.x, both.y);
        const bool raise = mx > pass;
        if (__any(raise)) {
            const float up = raise ? mx : 0.f, alpha = __builtin_amdgcn_exp2f(-fmaxf(up, 0.f));
            m += up;
            if (raise) pass = 8.f;
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] -= up;
        }
        bf16x8_t pb[2];
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float pr = __builtin_amdgcn_exp2f(s[i]);
            psum += pr;
            pb[i >> 3][i & 7] = (__bf16)pr;
        }
        l += psum;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const int place = (4 * t + 2 * st + h) * 8;
            uint32_t keep[4];                       // (values beyond the sequence are zeros)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                keep[i] = (value_position(place + 2 * i) < end ? 0xffffu : 0u) | (value_position(place + 2 * i + 1) < end ? 0xffff0000u : 0u);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                u32x4_t v = *reinterpret_cast<const u32x4_t*>(values + (32 * dt + c32) * TQK_PAGE + place);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] &= keep[i];
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, v), pb[st], o[dt], 0, 0, 0);
            }
        }
    }
    const float2 both = with_lane_32(l);
    l = both.x + both.y;
    if (!live) return;
    const float inv = 1.f / l;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            put4(out + 32 * dt + 8 * a + 4 * h, floatx4_t{o[dt][4 * a] * inv, o[dt][4 * a + 1] * inv, o[dt][4 * a + 2] * inv, o[dt][4 * a + 3] * inv});
}

// float32, up to 16 columns (a query and a head each) of one sequence and kv head whose keys lie in one page, by the matrix cores: the sums of attention_walk.h in their order, element after
// element in the scores and position after position in the output, which is what the instruction does with its four k (an instruction's sums are those of four fmaf).  Row i of a tile of 16 keys
// is key 4 (i % 4) + i / 4, so that what a lane holds of the weights is its operand of the output's product.  q and out: the lane's column; lo .. pos its positions of the page; first:
// the first position that any column sees; end: the sequence's after the step.  M: heads of up to 16 M.
// A value that is not finite would reach columns that do not see it, by 0 times it; where there is one, the columns' outputs are worked out one by one.
// Bound by a wave's instructions one after the other: a few hundred cycles each to look the unit up, ask for keys, multiply, weigh, sum, multiply and divide.  Cycles of the phase where every query's keys and
// values went by vector instructions, and now (two layers of 64, 4 heads on 2 of 16): 12 queries of up to 25 positions 7900 and 6900, a prompt's 132 of up to 17 39500 and 9400; us a step with
// queries by vector instructions and now, prompts of 8, 33 and 64 tokens 41, 93, 150 and 35, 69, 93; three layers of 96, one head of keys of 64: 94, 286 and 79, 189.
__device__ __forceinline__ void turn_4x4(floatx4_t& v) {       // register m of lanes 16 g .. + 15 <-> register g of lanes 16 m .. + 15
    auto swap32 = [&](int a, int b) { const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[a]), __float_as_uint(v[b]), false, false); v[a] = __uint_as_float(r[0]); v[b] = __uint_as_float(r[1]); };
    auto swap16 = [&](int a, int b) { const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[a]), __float_as_uint(v[b]), false, false); v[a] = __uint_as_float(r[0]); v[b] = __uint_as_float(r[1]); };
    swap32(0, 2); swap32(1, 3); swap16(0, 1); swap16(2, 3);
}
template <int M>
__device__ __forceinline__ void attend_page(const float* q, const float* keys, const float* values, int d, int lo, int pos, int first, int end, float scale, float* out, bool live, int lane) {
    const int i = lane % 16, g = lane / 16, furthest = end - 1;
    constexpr bool AHEAD = M == 1;          // (all loads together, where the registers hold them)
    floatx4_t k[AHEAD ? 4 : 1][M], v[4];
    auto ask_values = [&](int row) {
#pragma unroll
        for (int t = 0; t < 4; ++t)             // positions 16 t + 4 g .. + 3 (value_place)
            if (16 * t <= furthest) v[t] = *reinterpret_cast<const floatx4_t*>(values + row * TQK_PAGE + t / 2 * 32 + 8 * g + t % 2 * 4);
    };
    auto ask_keys = [&](int t) {
#pragma unroll
        for (int m = 0; m < M; ++m) k[AHEAD ? t : 0][m] = *reinterpret_cast<const floatx4_t*>(keys + (16 * t + 4 * (i % 4) + i / 4) * d + min(16 * m + 4 * g, d - 4));
    };
    if (AHEAD) {
#pragma unroll
        for (int t = 0; t < 4; ++t) if (16 * t <= furthest) ask_keys(t);
        ask_values(min(i, d - 1));
    }
    float qv[4 * M];
#pragma unroll
    for (int m = 0; m < 4 * M; ++m) qv[m] = q[min(4 * m + g, d - 1)];
    floatx4_t s[4];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        s[t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        if (16 * t <= furthest) {
            if (!AHEAD) ask_keys(t);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (16 * m >= d) break;
                floatx4_t& of = k[AHEAD ? t : 0][m];
                turn_4x4(of);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (16 * m + 4 * e < d) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(of[e], qv[4 * m + e], s[t], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (16 * t > furthest) break;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 16 * t + 4 * r + g;
            s[t][r] = j >= lo && j <= pos ? s[t][r] * scale : -INFINITY;
            mx = fmaxf(mx, s[t][r]);
        }
    }
    float2 both = with_lane_32(mx);
    mx = fmaxf(both.x, both.y);
    both = with_lane_16(mx);
    mx = fmaxf(both.x, both.y);
    const float from = from_max(mx);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (16 * t > furthest) break;               // (nothing there: they are 0)
#pragma unroll
        for (int r = 0; r < 4; ++r) s[t][r] = expf(s[t][r] - from);         // (a position that is not seen: exp(-inf) = 0)
    }
    // their sum as wave_sum has it: positions 32 apart first, then 16, 8, 4, 2 and 1
    const floatx4_t sums = (s[0] + s[2]) + (s[1] + s[3]);
    float sum = (sums[0] + sums[2]) + (sums[1] + sums[3]);
    both = with_lane_32(sum);
    sum = both.x + both.y;
    both = with_lane_16(sum);
    sum = both.x + both.y;
#pragma unroll 1
    for (int e0 = 0; e0 < d; e0 += 16) {
        if (!AHEAD || e0 > 0) ask_values(min(e0 + i, d - 1));
        // (one: the column whose output is worked out alone; -1, all of them)
#pragma unroll 1
        for (int one = -1; one < 16; ++one) {
            const int from_j = one < 0 ? first : __builtin_amdgcn_readlane(lo, one), to_j = one < 0 ? end : __builtin_amdgcn_readlane(pos, one) + 1;
            floatx4_t o = {0.f, 0.f, 0.f, 0.f};
            uint32_t largest = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (16 * t > furthest) break;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int j = 16 * t + 4 * g + e;
                    v[t][e] = j >= from_j && j < to_j ? v[t][e] : 0.f;
                    largest = max(largest, __float_as_uint(v[t][e]) & 0x7fffffffu);
                }
                turn_4x4(v[t]);
#pragma unroll
                for (int r = 0; r < 4; ++r) o = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][r], s[t][r], o, 0, 0, 0);
            }
            const bool again = one < 0 && __any(largest >= 0x7f800000u);
            if (live && !again && (one < 0 || one == i) && e0 + 4 * g < d) put4(out + e0 + 4 * g, floatx4_t{o[0] / sum, o[1] / sum, o[2] / sum, o[3] / sum});
            if (one < 0 && !again) break;
            ask_values(min(e0 + i, d - 1));
        }
    }
}

// The weights' way into the second-level cache of the die that runs the step: block 0 alone would wait for memory at every product.  Blocks are dealt to
// the eight dies in turn, so those whose number is a multiple of 8 read a layer's weights each (where they run elsewhere, nothing is lost but
// the time saved).
template <typename T>
__device__ __forceinline__ void warm(const T* w, size_t n) {
    const u32x4_t* p = reinterpret_cast<const u32x4_t*>(w);
    const int count = (int)(n * sizeof(T) / 16);
#pragma unroll 4
    for (int i = threadIdx.x; i < count; i += SS_THREADS) {
        const u32x4_t v = p[i];
        asm volatile("" :: "v"(v));
    }
}

// D: the heads' size where the matrix cores take them (bfloat16: 32 or 64; float32, where tqk_small_step_pages has it so: up to 16, 32 or 64), or 0.  RING: two waves bring the
// weights into LDS (tqk_small_step_rings: decoding steps of up to 4 rows in float32, 12 in bfloat16).
template <typename T, int D, bool RING>
__global__ __launch_bounds__(SS_THREADS)
void small_step_kernel(const TqkSmallStep p, const SmallPlan plan) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid % TQK_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / TQK_WAVE);
    const int rows = p.n_rows, hidden = p.hidden, d = p.head_dim, half = d / 2, nh = p.n_heads, nkv = p.n_kv_heads, inter = p.inter;
    const int qd = nh * d, qkv = (nh + 2 * nkv) * d, row_tiles = (rows + 15) / 16;
    if (blockIdx.x > 0) {
        if (blockIdx.x % 8) return;
        const int which = blockIdx.x / 8 - 1;
        if (which < p.n_layers) {
            const TqkSmallLayer& l = p.layers[which];
            warm((const T*)l.qkv, (size_t)qkv * hidden);
            warm((const T*)l.o, (size_t)hidden * qd);
            warm((const T*)l.gate_up, (size_t)2 * inter * hidden);
            warm((const T*)l.down, (size_t)hidden * inter);
        } else warm((const T*)p.head, (size_t)p.vocab * hidden);
        return;
    }
    constexpr int W = RING ? SS_WAVES - SS_BRING : SS_WAVES;           // waves that compute
    const SmallLayout at = small_layout(p, W);
    const SmallRing sizes = RING ? small_ring(p) : SmallRing{};
    char* const ring = lds + at.bytes;
    if (RING && wave >= W) {
        // (the barriers are the others'.  A weight's place is free once what lay there is done with, and its units are dealt to the phases so that no barrier waits for loads to be asked for.)
        int to = 0;
        auto next = [&](const void* w, int n, int k, int from_third, int to_third) { to = bring(w, n, k * (int)sizeof(T), ring, sizes.bytes, to, from_third, to_third, wave - W, lane); };
        next(p.layers[0].qkv, qkv, hidden, 0, 3);
        lds_barrier();
        lds_barrier();
#pragma unroll 1
        for (int layer = 0; layer < p.n_layers; ++layer) {
            const TqkSmallLayer& l = p.layers[layer];
            if (layer > 0) next(l.qkv, qkv, hidden, 2, 3);
            brought();
            lds_barrier();                                      // q, k and v
            next(l.o, hidden, qd, 0, 3);
            lds_barrier();                                      // rotation
            brought();
            lds_barrier();                                      // attention
            next(l.gate_up, 2 * inter, hidden, 0, 3);
            lds_barrier();                                      // o
            lds_barrier();                                      // norm
            next(l.down, hidden, inter, 0, 1);
            brought();
            lds_barrier();                                      // gate and up
            next(l.down, hidden, inter, 1, 3);
            brought();
            lds_barrier();                                      // down
            if (layer + 1 < p.n_layers) next(p.layers[layer + 1].qkv, qkv, hidden, 0, 2);
            else if (p.n_want > 0) next(p.head, p.vocab, hidden, 0, 2);
            lds_barrier();
        }
        if (p.n_want == 0) return;
        next(p.head, p.vocab, hidden, 2, 3);
        brought();
        lds_barrier();
        return;
    }
    int32_t* ints = reinterpret_cast<int32_t*>(lds);
    const TqkSmallLayer* layers = reinterpret_cast<const TqkSmallLayer*>(lds + at.layers);      // (the arguments lie far away)
    T *norms = reinterpret_cast<T*>(lds + at.norms), *biases = reinterpret_cast<T*>(lds + at.biases);
    float *angles = reinterpret_cast<float*>(lds + at.angles), *probs = reinterpret_cast<float*>(lds + at.probs) + wave * (RING ? queries_together(p, W) : SS_QUERIES) * TQK_PAGE;
    float* h = reinterpret_cast<float*>(lds + at.h);
    T* a = reinterpret_cast<T*>(lds + at.a);
    char* b = lds + at.b;
    auto round = [](float v) { return to_float(from_float<T>(v)); };

    // (bfloat16, norms divided by behind their product: the rows' inverse root mean squares and the sums of the squares of 16 columns each, [columns / 16][row])
    constexpr bool BF16 = sizeof(T) == 2;
    constexpr bool FEW = RING && !BF16;             // (float32 has a ring for up to SS_FEW rows alone)
    const bool behind = BF16 && plan.behind;
    float *inverse = reinterpret_cast<float*>(lds + at.squares), *square_sums = inverse + 16;

    // a product, its weights in the ring from `in_ring` on (which goes on behind them by `size`), or on their way to the wave from here on
    int in_ring = 0;
    auto product = [&](const void* w, int n, int k, int tiles, int size) {
        if constexpr (RING) {
            const RingProduct<T, 1, W> one = {ring, sizes.bytes, in_ring, n, k * (int)sizeof(T), tiles, lane, wave};
            in_ring += size;
            in_ring -= in_ring >= sizes.bytes ? sizes.bytes : 0;
            return one;
        } else {
            SmallProduct<T, 1> one = {{(const char*)w}, n, k * (int)sizeof(T), tiles, lane, wave};
            one.ask();
            return one;
        }
    };
    for (int i = tid; i < p.n_ints; i += W * TQK_WAVE) ints[i] = p.ints[i];
    for (int i = tid * 4; i < p.n_layers * (int)sizeof(TqkSmallLayer); i += W * TQK_WAVE * 4)
        __builtin_memcpy(__builtin_assume_aligned(lds + at.layers + i, 4), reinterpret_cast<const char*>(p.layers) + i, 4);
    for (int layer = wave; layer < p.n_layers; layer += W) {
        const TqkSmallLayer& l = p.layers[layer];
        for (int i = lane; i < hidden; i += TQK_WAVE) {
            norms[2 * layer * hidden + i] = ((const T*)l.norm1)[i];
            norms[(2 * layer + 1) * hidden + i] = ((const T*)l.norm2)[i];
        }
        if (l.qkv_bias) for (int i = lane; i < qkv; i += TQK_WAVE) biases[layer * qkv + i] = ((const T*)l.qkv_bias)[i];
    }
    for (int i = tid; i < hidden; i += W * TQK_WAVE) norms[2 * p.n_layers * hidden + i] = ((const T*)p.final_norm)[i];
    lds_barrier();
    const int32_t *tokens = p.device_tokens ? p.device_tokens : ints + p.tokens, *tok_seq = ints + p.tok_seq, *tok_pos = ints + p.tok_pos;
    for (int r = wave; r < rows; r += W) {
        const int id = tokens[r], pos = min(tok_pos[r], p.max_positions - 1);
        const bool ok = id >= 0 && id < p.vocab;
        const T* row = (const T*)p.embedding + (size_t)(ok ? id : 0) * hidden;
        for (int i = lane; i < hidden; i += TQK_WAVE) h[r * at.ld_h + i] = ok ? to_float(row[i]) : 0.f;
        if (BF16 && plan.first_behind) {                // the first norm's squares: eight neighbouring values a lane
            float sum = 0.f;
            for (int i0 = 0; i0 < hidden / 8; i0 += TQK_WAVE) {
                const int i = i0 + lane;
                float ss = 0.f;
                if (i < hidden / 8 && ok)
#pragma unroll
                    for (int j = 0; j < 8; ++j) { const float v = to_float(row[8 * i + j]); ss = fmaf(v, v, ss); }
                sum += wave_sum(ss);
            }
            if (lane == 0) square_sums[r] = sum;
        }
        for (int i = lane; i < d; i += TQK_WAVE) angles[r * d + i] = i < half ? p.cos_table[(size_t)pos * half + i] : p.sin_table[(size_t)pos * half + i - half];
    }
    lds_barrier();

    // row `from` of the stream normed into row `to` of a: a wave's lanes hold four neighbouring values each, up to four times
    auto norm_row = [&](int from, int to, const T* weight, float eps) {
        const float* hr = h + from * at.ld_h;
        floatx4_t v[4];
        float total = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j * 256 >= hidden) break;
            const int i = j * 256 + lane * 4;
            v[j] = i < hidden ? *reinterpret_cast<const floatx4_t*>(hr + i) : floatx4_t{0.f, 0.f, 0.f, 0.f};
            total += wave_sum(squares(make_float4(v[j][0], v[j][1], v[j][2], v[j][3])));
        }
        const float rms = sqrtf(total / (float)hidden + eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j * 256 >= hidden) break;
            const int i = j * 256 + lane * 4;
            if (i >= hidden) break;
            const float4 w = load4(weight + i);
            put4(a + to * at.ld_a + i, floatx4_t{(v[j][0] / rms) * w.x, (v[j][1] / rms) * w.y, (v[j][2] / rms) * w.z, (v[j][3] / rms) * w.w});
        }
    };
    // A norm that is divided by behind its product: row `from` of the stream times the weight into row `to` of a, and the inverse of its root mean square.
    // The sums of squares (of `sums` times 16 columns) are added as the product's kernel adds them.
    auto norm_behind = [&](int from, int to, const T* weight, float eps, int sums) {
        for (int i = lane * 4; i < hidden; i += 4 * TQK_WAVE) {
            const floatx4_t v = *reinterpret_cast<const floatx4_t*>(h + from * at.ld_h + i);
            const float4 w = load4(weight + i);
            put4(a + to * at.ld_a + i, floatx4_t{v[0] * w.x, v[1] * w.y, v[2] * w.z, v[3] * w.w});
        }
        float ss = lane / 4 < sums ? square_sums[lane / 4 * 16 + from] : 0.f;
        for (int s = 16 + lane / 4; s < sums; s += 16) ss += square_sums[s * 16 + from];
        ss += lane_xor_4(ss);
        ss += lane_xor_8(ss);
        float2 both = with_lane_16(ss);
        ss = both.x + both.y;
        both = with_lane_32(ss);
        ss = both.x + both.y;
        if (lane == 0) inverse[to] = 1.f / sqrtf(ss / (float)hidden + eps);
    };
    auto divided = [&](floatx4_t v, int row, bool by) {
        if (!BF16 || !by) return v;
        const float f = inverse[row];
        return floatx4_t{v[0] * f, v[1] * f, v[2] * f, v[3] * f};
    };
    auto add_to_stream = [&](int row, int n, const floatx4_t* v) {
        floatx4_t* to = reinterpret_cast<floatx4_t*>(h + row * at.ld_h + n);
        const floatx4_t sum = *to + rounded<T>(v[0]);
        *to = sum;
        if (behind) {
            // the squares of the tile's 16 columns: the four lanes of the row, in lane order
            const float sq = fmaf(sum[3], sum[3], fmaf(sum[2], sum[2], fmaf(sum[1], sum[1], sum[0] * sum[0])));
            const float s1 = with_lane_16(sq).y, s2 = with_lane_32(sq).y, s3 = with_lane_32(s1).y;
            if (lane < 16) square_sums[n + row] = ((sq + s1) + s2) + s3;
        }
    };
    // queries a wave takes together: their elements side by side in its lanes
    const int width = d <= 16 ? 16 : d <= 32 ? 32 : 64, n_queries = rows * nh;
    const int together = queries_together(p, W);
    const float of_rows = 1.f / (float)rows, of_group = 1.f / (float)(nh / nkv);
    auto quotient = [&](int n) { return __builtin_amdgcn_readfirstlane((int)(((float)n + 0.5f) * of_rows)); };         // n / rows (numbers this small: exact)

    // float32, steps that go by units: up to 16 columns of a sequence and kv head, a wave each; a lane knows a sequence's first row, rows, first position and the units up to its end
    int my_r0 = 0, my_n = 0, my_start = 0, units_to = 0, n_units = 0;
    if constexpr (!BF16 && D > 0) {
        if (lane < p.n_seqs) {
            my_r0 = ints[p.seq_first + lane];
            my_n = ints[p.seq_first + lane + 1] - my_r0;
            my_start = tok_pos[my_r0];
            units_to = (my_n * (nh / nkv) + 15) / 16 * nkv;
        }
        auto add = [&](auto ctrl, auto rows_of) { units_to += __builtin_amdgcn_update_dpp(0, units_to, decltype(ctrl)::value, decltype(rows_of)::value, 0xf, true); };
        add(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});          // 1, 2, 4 and 8 lanes before, then the last lanes of 16 and of 32
        add(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
        add(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
        add(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
        add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
        add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
        n_units = __builtin_amdgcn_readlane(units_to, 63);
    }

#pragma unroll 1
    for (int layer = 0; layer < p.n_layers; ++layer) {
        // this layer's arguments, the same for all lanes
        struct Words { int32_t w[sizeof(TqkSmallLayer) / 4]; } words;
        __builtin_memcpy(&words, layers + layer, sizeof(words));
#pragma unroll
        for (int i = 0; i < (int)(sizeof(words) / 4); ++i) words.w[i] = __builtin_amdgcn_readfirstlane(words.w[i]);
        const TqkSmallLayer l = __builtin_bit_cast(TqkSmallLayer, words);
        const int32_t* table = ints + l.table;
        const bool last = layer == p.n_layers - 1 && p.n_last >= 0;         // (what follows the cache's rows counts for the last rows alone)
        const RingFewProduct<1, W> few_qkv = {ring, sizes.bytes, in_ring, qkv, hidden * 4, lane, wave};
        auto w_qkv = product(l.qkv, qkv, hidden, row_tiles, sizes.qkv);
        for (int r = wave; r < rows; r += W) {
            if (BF16 && plan.first_behind) norm_behind(r, r, norms + 2 * layer * hidden, l.eps1, layer == 0 ? 1 : hidden / 16);
            else norm_row(r, r, norms + 2 * layer * hidden, l.eps1);
        }
        lds_barrier();
        float* bf = reinterpret_cast<float*>(b);
        const int ld_b = at.ld_b / 4;
        if constexpr (FEW)
            few_qkv.run((const float*)a, at.ld_a, [&](int n, const floatx4_t* v) {
#pragma unroll
                for (int r = 0; r < 4; ++r) if (r < rows) bf[r * ld_b + n] = v[0][r];
            });
        else w_qkv.run(a, at.ld_a, rows, [&](int row, int n, const floatx4_t* v) { put4(bf + row * ld_b + n, rounded<T>(divided(v[0], row, plan.first_behind))); });
        lds_barrier();
        // biases, rotation of q and k, keys and values into the row's page: a wave a row's heads in turn, a lane a pair that rotates together
        const int per = half <= 16 ? 4 : half <= 32 ? 2 : 1, sub = TQK_WAVE / per;      // heads a wave takes at once
#pragma unroll 1
        for (int e = wave; e < rows * ((nh + 2 * nkv + per - 1) / per); e += W) {
            const int heads0 = quotient(e), r = e - heads0 * rows, head = heads0 * per + lane / sub, i = lane % sub;
            if (i >= half || head >= nh + 2 * nkv) continue;
            const int pos = tok_pos[r];
            float* src = bf + r * ld_b + head * d;
            float lo = src[i], hi = src[i + half];
            if (l.qkv_bias) {
                lo += to_float(biases[layer * qkv + head * d + i]);
                hi += to_float(biases[layer * qkv + head * d + i + half]);
            }
            if (head < nh + nkv && pos < p.max_positions) {
                const float co = angles[r * d + i], si = angles[r * d + i + half], x0 = lo, x1 = hi;
                if (BF16) rotate_pair(lo, hi, co, si);
                else {                                      // (which product is rounded is the kernels' of the type)
                    lo = fmaf(x0, co, -(x1 * si));
                    hi = fmaf(x1, co, x0 * si);
                }
            }
            if (head < nh) {
                src[i] = round(lo);
                src[i + half] = round(hi);
                continue;
            }
            const bool key = head < nh + nkv;
            const int kvh = key ? head - nh : head - nh - nkv, page = table[tok_seq[r] * l.width + pos / TQK_PAGE];
            if (page < 0) continue;                            // the host never lets this happen
            const size_t base = ((size_t)page * nkv + kvh) * TQK_PAGE * d;
            T* dst = key ? (T*)l.keys + base + (size_t)(pos % TQK_PAGE) * d : (T*)l.values + base + value_place(pos % TQK_PAGE);
            const int stride = key ? 1 : TQK_PAGE;
            dst[(size_t)i * stride] = from_float<T>(lo);
            dst[(size_t)(i + half) * stride] = from_float<T>(hi);
        }
        __syncthreads();                                    // (keys and values are read back out of memory)
        if constexpr (D > 0 && BF16) {
            const int group = nh / nkv;
            const size_t page_size = (size_t)TQK_PAGE * D;
            if (RING || (last ? plan.last_attention : plan.attention) == SMALL_ROWS) {          // (decoding steps: rows)
                const int n = last ? p.n_last : rows;
#pragma unroll 1
                for (int e = wave; e < n * nkv; e += W) {
                    const int kvh = __builtin_amdgcn_readfirstlane(e / n), which = __builtin_amdgcn_readfirstlane(e - kvh * n), head0 = kvh * group;
                    const int r = __builtin_amdgcn_readfirstlane(last ? ints[p.last_rows + which] : which), pos = __builtin_amdgcn_readfirstlane(tok_pos[r]);
                    const int page = __builtin_amdgcn_readfirstlane(table[tok_seq[r] * l.width]);
                    if (page < 0) continue;                 // the host never lets this happen
                    const size_t base = ((size_t)page * nkv + kvh) * page_size;
                    const int lo = l.window > 0 ? max(0, pos - l.window + 1) : 0;
                    attend_row<D>(bf + r * ld_b + head0 * D, group, (const bf16_t*)l.keys + base, (const bf16_t*)l.values + base, lo, pos, l.scale, l.divided != 0,
                                  a + r * at.ld_a + head0 * D, lane);
                }
            } else {
                int before = 0;                             // units of the sequences before
#pragma unroll 1
                for (int seq = 0; seq < p.n_seqs; ++seq) {
                    const int r0 = __builtin_amdgcn_readfirstlane(ints[p.seq_first + seq]), n = __builtin_amdgcn_readfirstlane(ints[p.seq_first + seq + 1]) - r0;
                    const int tiles = (n * group + 31) / 32, units = tiles * nkv;
                    const int page = __builtin_amdgcn_readfirstlane(table[seq * l.width]), end = __builtin_amdgcn_readfirstlane(tok_pos[r0]) + n;
#pragma unroll 1
                    for (int e = (wave - before) & (SS_WAVES - 1); e < units; e += W) {
                        if (page < 0) continue;             // the host never lets this happen
                        const int kvh = __builtin_amdgcn_readfirstlane(e % nkv), col = e / nkv * 32 + lane % 32;
                        const bool live = col < n * group;
                        const int of_group_ = live ? col / n : 0, r = r0 + (live ? col - of_group_ * n : 0), head = kvh * group + of_group_;
                        const int pos = live ? tok_pos[r] : -1, lo = l.window > 0 ? max(0, pos - l.window + 1) : 0;
                        const size_t base = ((size_t)page * nkv + kvh) * page_size;
                        attend_columns<D>(bf + r * ld_b + head * D, (const bf16_t*)l.keys + base, (const bf16_t*)l.values + base, lo, pos, end, end - 1, l.scale,
                                          a + r * at.ld_a + head * D, lane);
                    }
                    before += units;
                }
            }
        } else if constexpr (D > 0) {
            int at_lane = lane;
            asm volatile("" : "+v"(at_lane));               // (what follows from it is not held in registers across the layers)
            const int group = nh / nkv;
#pragma unroll 1
            for (int e = wave; e < n_units; e += W) {
                const int seq = __builtin_popcountll(__ballot(units_to <= e)), before = seq > 0 ? __builtin_amdgcn_readlane(units_to, seq - 1) : 0;
                const int r0 = __builtin_amdgcn_readlane(my_r0, seq), n = __builtin_amdgcn_readlane(my_n, seq), tiles = (n * group + 15) / 16;
                const int kvh = __builtin_amdgcn_readfirstlane((int)(((float)(e - before) + 0.5f) / (float)tiles)), c = (e - before - kvh * tiles) * 16 + at_lane % 16, col = min(c, n * group - 1);
                const int of_group_ = (int)(((float)col + 0.5f) / (float)n), r = r0 + col - of_group_ * n, head = kvh * group + of_group_;
                const int page = __builtin_amdgcn_readfirstlane(table[seq * l.width]), start = __builtin_amdgcn_readlane(my_start, seq);
                if (page < 0) continue;                     // the host never lets this happen
                const int pos = start + r - r0, lo = l.window > 0 ? max(0, pos - l.window + 1) : 0, first = l.window > 0 ? max(0, start - l.window + 1) : 0;
                const size_t base = ((size_t)page * nkv + kvh) * TQK_PAGE * d;
                attend_page<D / 16>(bf + r * ld_b + head * d, (const float*)l.keys + base, (const float*)l.values + base, d, lo, pos, first, start + n, l.scale, (float*)a + r * at.ld_a + head * d,
                                    c < n * group, at_lane);
            }
        } else
#pragma unroll 1
        for (int e0 = wave * together; e0 < n_queries; e0 += W * together) {
            SmallQuery mine;                                // the query whose elements this lane's are
            float my_sum = 1.f;
            bool done = false;
            int wave_first = TQK_PAGE, wave_last = -1;
            auto query = [&](int e) {
                SmallQuery y;
                y.head = quotient(e);
                y.row = e - y.head * rows;
                y.pos = __builtin_amdgcn_readfirstlane(tok_pos[y.row]);
                y.lo = l.window > 0 ? max(0, y.pos - l.window + 1) : 0;
                y.kvh = __builtin_amdgcn_readfirstlane((int)(((float)y.head + 0.5f) * of_group));
                y.q = bf + y.row * ld_b + y.head * d;
                y.page = __builtin_amdgcn_readfirstlane(table[tok_seq[y.row] * l.width + y.pos / TQK_PAGE]);
                y.one_page = y.lo / TQK_PAGE == y.pos / TQK_PAGE && y.page >= 0;
                return y;
            };
            auto several_pages = [&](const SmallQuery& y, int k) {
                const int32_t* pages = table + __builtin_amdgcn_readfirstlane(tok_seq[y.row]) * l.width;
                float m = -INFINITY, sum = 0.f, acc = 0.f, of_sum, of_stripe;
#pragma unroll 1
                for (int st = 0; st < ATT_STRIPES; ++st) {
                    if (page_of(st, y.lo / TQK_PAGE) * TQK_PAGE > y.pos) continue;
                    const Stripe<1> one = walk<T, 8, 1>(st, y.q, (const T*)l.keys, (const T*)l.values, pages, y.pos, y.lo, y.kvh, nkv, d, l.scale, 1, 1, lane);
                    join(m, sum, one.m, one.l, of_sum, of_stripe);
                    acc = fmaf(acc, of_sum, one.acc[0] * of_stripe);
                }
                if (lane < d) a[y.row * at.ld_a + y.head * d + lane] = from_float<T>(acc / sum);
                if (lane / width == k) done = true;
            };
            const int last_query = min(e0 + together, n_queries) - 1;
#pragma unroll 1
            for (int k = 0; e0 + k <= last_query; ++k) {
                const SmallQuery y = query(e0 + k);
                if (!y.one_page) {
                    several_pages(y, k);
                    continue;
                }
                const float sum = small_scores(y, (const T*)l.keys, nkv, d, l.scale, probs + k * TQK_PAGE, lane);
                wave_first = min(wave_first, y.lo % TQK_PAGE);
                wave_last = max(wave_last, y.pos % TQK_PAGE);
                if (lane / width == k) { mine = y; my_sum = sum; }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int c = lane % width;
            if (!done && e0 + lane / width <= last_query && c < d) {
                const T* base = (const T*)l.values + ((size_t)mine.page * nkv + mine.kvh) * TQK_PAGE * d + c * TQK_PAGE;
                const float v = small_values(base, probs + lane / width * TQK_PAGE, mine.lo % TQK_PAGE, mine.pos % TQK_PAGE, wave_first, wave_last);
                a[mine.row * at.ld_a + mine.head * d + c] = from_float<T>(v / my_sum);
            }
            __builtin_amdgcn_wave_barrier();
        }
        auto w_o = product(l.o, hidden, qd, row_tiles, sizes.o);
        const RingFewProduct<2, W> few_gate_up = {ring, sizes.bytes, in_ring, inter, hidden * 4, lane, wave};
        auto w_gate_up = [&]() {
            if constexpr (RING) {
                const RingProduct<T, 2, W> two = {ring, sizes.bytes, in_ring, inter, hidden * (int)sizeof(T), row_tiles, lane, wave};
                in_ring += sizes.gate_up;
                in_ring -= in_ring >= sizes.bytes ? sizes.bytes : 0;
                return two;
            } else return SmallProduct<T, 2>{{(const char*)l.gate_up, (const char*)((const T*)l.gate_up + (size_t)inter * hidden)}, inter, hidden * (int)sizeof(T), row_tiles, lane, wave};
        }();
        lds_barrier();
        w_o.run(a, at.ld_a, rows, add_to_stream);
        if constexpr (!RING) w_gate_up.ask();
        lds_barrier();
        for (int r = wave; r < rows; r += W) {
            if (behind) norm_behind(r, r, norms + (2 * layer + 1) * hidden, l.eps2, hidden / 16);
            else norm_row(r, r, norms + (2 * layer + 1) * hidden, l.eps2);
        }
        lds_barrier();
        T* act = reinterpret_cast<T*>(b);
        const int ld_act = at.ld_b / (int)sizeof(T);
        if constexpr (FEW)
            few_gate_up.run((const float*)a, at.ld_a, [&](int n, const floatx4_t* v) {
#pragma unroll
                for (int r = 0; r < 4; ++r) if (r < rows) act[r * ld_act + n] = from_float<T>(gate_value(TQK_GATE_SILU, 0.f, 1.f, v[0][r], v[1][r]));
            });
        else w_gate_up.run(a, at.ld_a, rows, [&](int row, int n, const floatx4_t* v) {
            const floatx4_t g = rounded<T>(divided(v[0], row, behind)), u = rounded<T>(divided(v[1], row, behind));
            floatx4_t y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = gate_value(TQK_GATE_SILU, 0.f, 1.f, g[i], u[i]);
            put4(act + row * ld_act + n, y);
        });
        auto w_down = product(l.down, hidden, inter, row_tiles, sizes.down);
        lds_barrier();
        w_down.run(act, ld_act, rows, add_to_stream);
        lds_barrier();
    }

    if (p.n_want == 0) return;
    const RingFewProduct<1, W> few_head = {ring, sizes.bytes, in_ring, p.vocab, hidden * 4, lane, wave};
    auto w_head = product(p.head, p.vocab, hidden, (p.n_want + 15) / 16, sizes.head);
    const int32_t* want = ints + p.want;
    for (int r = wave; r < p.n_want; r += W) {
        if (behind) norm_behind(want[r], r, norms + 2 * p.n_layers * hidden, p.final_eps, hidden / 16);
        else norm_row(want[r], r, norms + 2 * p.n_layers * hidden, p.final_eps);
    }
    lds_barrier();
    if constexpr (FEW)
        few_head.run((const float*)a, at.ld_a, [&](int n, const floatx4_t* v) {
#pragma unroll
            for (int r = 0; r < 4; ++r) if (r < p.n_want) p.logits[(size_t)r * p.vocab + n] = v[0][r];
        });
    else w_head.run(a, at.ld_a, p.n_want, [&](int row, int n, const floatx4_t* v) {
        const floatx4_t y = divided(v[0], row, behind);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < p.vocab) p.logits[(size_t)row * p.vocab + n + i] = y[i];
    });
}

// Whether the kernels that a bfloat16 step would run through add up its products by increasing k, as this one does.
static bool in_order(const TqkSmallStep& p, int n_rows, int last, int n_want, bool decode) {
    const int few = tqk_skinny_max_rows(), q = p.n_heads * p.head_dim, all = q + 2 * p.n_kv_heads * p.head_dim;
    auto whole = [&](int rows, int n, int k, bool pairs, bool gated) { return (rows <= few ? tqk_fused_waves(n, k, pairs) : tqk_mid_splits(n, k, gated)) == 1; };
    auto rest = [&](int rows) { return whole(rows, p.hidden, q, false, false) && whole(rows, 2 * p.inter, p.hidden, true, true) && whole(rows, p.hidden, p.inter, false, false); };
    return whole(n_rows, all, p.hidden, decode && p.head_dim % 32 == 0, false) && rest(n_rows) && rest(last) && whole(n_want, p.vocab, p.hidden, false, false);
}
// Whether the matrix cores' attention of one page does for a bfloat16 step's heads.
static bool heads_fit(const TqkSmallStep& p, int positions) {
    return !tqk_attention_decode_supported(p.head_dim) || (positions <= TQK_PAGE && p.n_heads / p.n_kv_heads <= 16);
}

/* Whether the kernel takes a step: what of `step` describes the model and the step's size is filled in, pointers need not be. */
extern "C" int tqk_small_step_takes(const TqkSmallStep* step) {
    const TqkSmallStep& p = *step;
    const int size = p.act_dtype == TQK_F32 ? 4 : 2;
    if (p.act_dtype != TQK_F32 && p.act_dtype != TQK_BF16) return 0;
    if (p.n_layers < 1 || p.n_layers > TQK_SMALL_LAYERS || p.n_ints < 0 || p.n_ints > TQK_SMALL_INTS) return 0;
    if (p.n_rows < 1 || p.n_rows > 64 || p.n_want < 0 || p.n_want > p.n_rows) return 0;
    if (p.hidden < 4 || p.hidden > 1024 || p.inter < 1 || p.inter > 1024 || p.head_dim < 2 || p.head_dim > TQK_WAVE || p.head_dim * size % 16) return 0;
    if (p.n_heads < 1 || p.n_kv_heads < 1 || p.n_heads % p.n_kv_heads || p.n_heads * p.head_dim > 1024 || p.vocab < 1) return 0;
    // whole steps of k, and whole tiles
    const int q = p.n_heads * p.head_dim, whole = 64 / size;
    if (p.hidden % whole || p.inter % whole || q % whole || (p.n_kv_heads * p.head_dim * 2) % 16) return 0;
    if ((long long)p.vocab * p.hidden * size > 0x7fffffff) return 0;          // (a weight's bytes are counted in 32 bits)
    if (small_layout(p, SS_WAVES).bytes > 160 * 1024) return 0;
    if (p.act_dtype == TQK_BF16 && !(heads_fit(p, p.max_end) && in_order(p, p.n_rows, p.n_last >= 0 ? p.n_last : p.n_rows, p.n_want, p.decode != 0))) return 0;
    // (larger products have another order of summation there)
    if (p.act_dtype == TQK_F32 && (tqk_gemm_takes_apart(p.vocab, p.hidden) || tqk_gemm_takes_apart(2 * p.inter, p.hidden) || tqk_gemm_takes_apart(q + 2 * p.n_kv_heads * p.head_dim, p.hidden))) return 0;
    return 1;
}

// Units of a float32 step's attention: up to 16 columns (a query and a head each) of a sequence and kv head.
static int units_of(const TqkSmallStep& p, int rows) { return (rows * (p.n_heads / p.n_kv_heads) + 15) / 16 * p.n_kv_heads; }
static int attention_units(const TqkSmallStep& p) {
    int units = 0;
    for (const int32_t *first = p.ints + p.seq_first, *end = first + p.n_seqs; first < end; ++first) units += units_of(p, first[1] - first[0]);
    return units;
}
/* Whether a float32 step within a page has its attention by the matrix cores, a wave a unit (attend_page), and not a query a wave: where units are few beside the queries.  Heads of up to 16:
 * a unit costs four queries for every 16 positions, and what a step saves beside them pays for ten.  Larger heads: a query of d elements costs d, a wave's turn of units, whose loads take 16 elements of a row at a
 * time, 9 d, and each unit 50 for what it is served.  us a step by queries and by units, two layers: 3, 16 and 40 sequences, four heads of 16 on two 32.3 and 30.9 (units), 54 and 56, 109 and 117
 * (queries), on four 32.7 and 32.9, 56 and 76, 112 and 168 (queries), on one 32.2 and 29.1, 54 and 46, 107 and 89 (units); 16 sequences, eight heads of 4 57 and 102
 * (queries); one, four and 16 sequences, four heads of 32 on two 32.5 and 33.3, 39.4 and 38.0, 71 and 69 (queries), eight on two 40.0 and 40.7 (queries), 51.6 and 44.3, 102 and 70 (units), one head of
 * 64 30.4 and 35.7, 34.4 and 38.2, 52 and 60 (queries), four on two 58 and 64 (queries), 71.5 and 69.7, 122 and 109 (units); prompts of 16 and 63 tokens, four heads of 16 on two 48
 * and 37, 149 and 92, one head of 64 45 and 39, 150 and 92 (units).  925 steps of 40 shapes with heads of 4 to 64: 1.004 of the faster way's time (at most 1.14), and at most 1.045 of that by queries. */
static bool by_units(const TqkSmallStep& p, int units, int n_rows, int positions) {
    const int queries = n_rows * p.n_heads;
    if (p.act_dtype != TQK_F32 || positions > TQK_PAGE) return false;
    if (p.head_dim <= 16) return (4 * units - queries) * ((positions + 15) / 16) < 40;
    return queries * p.head_dim >= 50 * units + 9 * ((units + SS_WAVES - 1) / SS_WAVES) * p.head_dim;
}
extern "C" int tqk_small_step_pages(const TqkSmallStep* step) {
    const TqkSmallStep& p = *step;
    return p.seq_first >= 0 && p.n_seqs > 0 && p.seq_first + p.n_seqs + 1 <= TQK_SMALL_INTS && by_units(p, attention_units(p), p.n_rows, p.max_end);
}

/* Whether that is the faster way, by an estimate in microseconds (n_rows: of the step; decode: one token a sequence, which the other kernels run as a replayed graph; positions: the
 * furthest one).  One block: 5 a layer for its barriers and chains of short operations, its weights at 33 KB (27 in float32) a microsecond, and for every row what
 * its products, its other work and its heads' pages take; the head's weights at 39 KB.  The other kernels, ten launches a layer: 20 a layer in a graph (33 in float32) and 32 (45) one by one.
 * Measured, one block and the other kernels, two layers of 64 values with 160 in the feed-forward, bfloat16: 1, 16 and 40 sequences 31 and 72, 65 and 79, 92 and 88, prompts of 8, 33
 * and 64 tokens 31 and 96, 61 and 96, 109 and 97; three of 96 with 224 and heads of 32: 47 and 73, 75 and 82, 108 and 97, then 35 and 132, 70 and 134, 95 and 135; with heads of 64: 66 and 78, 87
 * and 83, 156 and 106, then 43 and 132, 87 and 137, 133 and 137; four of 128 with 224: 69 and 83, 94 and 88, 207 and 122, then 55 and 175, 126 and 179, 175 and 179.  float32, two of 64: 1, 4, 16
 * and 40 sequences 29 and 82, 31 and 85, 52 and 87, 106 and 115, prompts of 8, 33 and 64 tokens 33 and 100, 67 and 102, 91 and 105; three of 96 62 and 111, 69 and 111, 85 and 116, 194 and 156, then 64 and 128,
 * 147 and 145, 198 and 153; with heads of 64 74 and 109, 84 and 113, 109 and 117, 256 and 166, then 77 and 130, 188 and 154; four of 128 with 512: 152 and 145, 163 and 149, 219 and 155, then 153 and 159. */
extern "C" int tqk_small_step_pays(const TqkSmallStep* step, int n_rows, int decode, int positions) {
    const TqkSmallStep& p = *step;
    const bool f32 = p.act_dtype == TQK_F32;
    if (!f32 && !(heads_fit(p, positions) && in_order(p, n_rows, n_rows, n_rows, decode != 0))) return 0;         // (what the kernel does not take)
    const double size = f32 ? 4 : 2, q = (double)p.n_heads * p.head_dim;
    const double thousands = 1e-3 * p.hidden * (2 * q + 2. * p.n_kv_heads * p.head_dim + 3. * p.inter);            // weights of a layer
    const double heads = 0.08 * p.n_heads * ((positions + TQK_PAGE - 1) / TQK_PAGE);
    // (float32 by units: columns of a sequence and kv head share an instruction.  A prompt is taken for one sequence's; eight chunks of three tokens, three layers of 96, six heads of 16 on as many:
    // 155 us here, 144 there; 20 sequences after 38 tokens, four layers of 64, four heads of 48 on as many, which go by queries: 329 and 194)
    const bool units = by_units(p, decode ? n_rows * units_of(p, 1) : units_of(p, n_rows), n_rows, positions);
    const double a_row = units ? 0.15 + 0.0085 * thousands + (decode ? heads : 0.03 * p.n_kv_heads) : 0.15 + (f32 ? 0.0115 : 0.0043) * thousands + heads;
    const double here = 8 + p.n_layers * (5 + thousands * size / (f32 ? 27 : 33) + n_rows * a_row) + 1e-3 * p.vocab * p.hidden * size / 39;
    const double there = decode ? 15 + p.n_layers * (f32 ? 33 : 20) : 15 + p.n_layers * (f32 ? 45 : 32);
    return here < there;
}

// Which kernels a step in bfloat16 would run through: decoding steps of up to 16 rows with their norms behind the products (heads by 32: the
// first ones too), and the attention of heads that the matrix cores take, the last layer for the last rows alone.
static SmallPlan small_plan(const TqkSmallStep& p) {
    SmallPlan plan = {};
    if (p.act_dtype != TQK_BF16) return plan;
    plan.behind = p.decode && p.n_rows <= tqk_skinny_max_rows();
    plan.first_behind = plan.behind && p.head_dim % 32 == 0;
    if (tqk_attention_decode_supported(p.head_dim)) {
        plan.attention = p.decode ? SMALL_ROWS : SMALL_TILES;
        plan.last_attention = p.decode || (p.n_last >= 0 && p.n_last <= TQK_SMALL_LAST_ROWS) ? SMALL_ROWS : SMALL_TILES;
    }
    return plan;
}

template <typename T, int D, bool RING>
static int launch_small(const TqkSmallStep& p, int lds, hipStream_t s) {
    // (a limit of each device's own: raised once for it, or a few times by threads that meet here)
    static std::atomic<uint64_t> grown{0};
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    const uint64_t bit = device < 64 ? 1ull << device : 0;
    if (e == hipSuccess && !(grown.load(std::memory_order_acquire) & bit)) {
        e = hipFuncSetAttribute((const void*)small_step_kernel<T, D, RING>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e == hipSuccess) grown.fetch_or(bit, std::memory_order_release);
    }
    if (e != hipSuccess) return tqk_fail("tqk_small_step: %s", hipGetErrorString(e));
    small_step_kernel<T, D, RING><<<1 + 8 * (p.n_layers + 1), SS_THREADS, lds, s>>>(p, small_plan(p));
    return tqk_check_launch("tqk_small_step");
}

/* Whether a step's weights come into LDS by waves of their own: decoding steps of few rows, where the ring fits beside the rows and two waves fewer take no more turns for the attention's
 * queries or units.  us a step without and with it, steps asked for one by one: float32, two layers of 64, 1, 3, 4, 5 and 16 rows 36.5, 37.8, 37.5, 39.4, 54.0 and 33.3, 34.1, 35.8, 40.1, 57.3;
 * bfloat16, heads of 32, three layers of 96, 1, 5, 8, 12 and 16 rows 38.2, 40.9, 42.0, 46.3, 81.5 and 36.0, 38.5, 41.3, 45.4, 81.8.  bfloat16 with other heads, whose attention every wave has a part
 * in, loses: two layers of 64, 1, 4, 8 and 16 rows 28.1, 29.5, 33.0, 42.1 and 28.3, 29.8, 34.0, 48.1.  A turn more (six asked for together): float32, four heads of 16, 4 sequences after 240
 * tokens 62.3 and 68.6, eight of 4, 2 after 90 and 240 34.1 and 38.8, 49.7 and 61.2; bfloat16, four heads of 32 on two, 8 sequences 30.2 and 32.0. */
extern "C" int tqk_small_step_rings(const TqkSmallStep* step) {
    const TqkSmallStep& p = *step;
    const bool f32 = p.act_dtype == TQK_F32, few = f32 ? p.n_rows <= SS_FEW : p.n_rows <= 12 && (p.head_dim == 32 || p.head_dim == 64);
    if (!p.decode || !few || small_layout(p, SS_WAVES - SS_BRING).bytes + small_ring(p).bytes > 160 * 1024) return 0;
    const int work = !f32 ? p.n_rows * p.n_kv_heads : tqk_small_step_pages(&p) ? attention_units(p) : p.n_rows * p.n_heads;
    return (work + SS_WAVES - SS_BRING - 1) / (SS_WAVES - SS_BRING) == (work + SS_WAVES - 1) / SS_WAVES;
}

template <typename T, int D>
static int launch_small(const TqkSmallStep& p, hipStream_t s) {
    if constexpr (D > 0 || sizeof(T) == 4) {
        if (tqk_small_step_rings(&p)) return launch_small<T, D, true>(p, small_layout(p, SS_WAVES - SS_BRING).bytes + small_ring(p).bytes, s);
    }
    return launch_small<T, D, false>(p, small_layout(p, SS_WAVES).bytes, s);
}

extern "C" int tqk_small_step(const TqkSmallStep* step, void* stream) {
    TQK_REQUIRE(step && tqk_small_step_takes(step), "tqk_small_step: this step is not for the one-block kernel");
    const TqkSmallStep& p = *step;
    TQK_REQUIRE(p.embedding && p.final_norm && p.head && p.cos_table && p.sin_table && (p.logits || p.n_want == 0) && p.max_positions > 0, "tqk_small_step: null pointer");
    for (int i = 0; i < p.n_layers; ++i) {
        const TqkSmallLayer& l = p.layers[i];
        TQK_REQUIRE(l.norm1 && l.qkv && l.o && l.norm2 && l.gate_up && l.down && l.keys && l.values, "tqk_small_step: null pointer in layer %d", i);
        TQK_REQUIRE((((uintptr_t)l.qkv | (uintptr_t)l.o | (uintptr_t)l.gate_up | (uintptr_t)l.down | (uintptr_t)l.keys | (uintptr_t)l.values) & 15) == 0,
                    "tqk_small_step: layer %d: weights and cache must be 16-byte aligned", i);
        TQK_REQUIRE(l.width > 0 && l.window >= 0 && l.table >= 0 && l.table + l.width <= p.n_ints, "tqk_small_step: layer %d: no page table", i);
    }
    TQK_REQUIRE((((uintptr_t)p.head) & 15) == 0, "tqk_small_step: the head must be 16-byte aligned");
    TQK_REQUIRE(p.tok_seq >= 0 && p.tok_pos >= 0 && p.want >= 0 && p.tok_seq + p.n_rows <= p.n_ints && p.tok_pos + p.n_rows <= p.n_ints && p.want + p.n_want <= p.n_ints && p.seq_first >= 0 && p.n_seqs > 0 &&
                    p.seq_first + p.n_seqs + 1 <= p.n_ints && (p.n_last < 0 || (p.last_rows >= 0 && p.last_rows + p.n_last <= p.n_ints)) &&
                    (p.device_tokens || (p.tokens >= 0 && p.tokens + p.n_rows <= p.n_ints)), "tqk_small_step: the step's arrays do not lie in what was given");
    hipStream_t s = (hipStream_t)stream;
    if (p.act_dtype == TQK_F32) {
        if (!tqk_small_step_pages(&p)) return launch_small<float, 0>(p, s);
        return p.head_dim <= 16 ? launch_small<float, 16>(p, s) : p.head_dim <= 32 ? launch_small<float, 32>(p, s) : launch_small<float, 64>(p, s);
    }
    return p.head_dim == 32 ? launch_small<bf16_t, 32>(p, s) : p.head_dim == 64 ? launch_small<bf16_t, 64>(p, s) : launch_small<bf16_t, 0>(p, s);
}
