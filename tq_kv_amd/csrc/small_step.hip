// A whole step of a small decoder in one launch: embedding, every layer, final norm and the head's logits, in one block.
//
// A model of a few hundred kilobytes a layer is bound by nothing but launches: its step is ten kernels a layer, each of which works for a
// microsecond and costs two to four in a replayed graph, and about as much again on the host.  One block on one compute unit runs
// the step with barriers in place of launches.  It pulls weights and does a row's work at a fraction of the chip's rate, so this is the better way only
// while that takes no longer than the launches it stands for: tqk_small_step_pays says where that is.  Two layers of 64 values, 3 sequences after
// 20 tokens: 22.2 us in bfloat16 and 30.2 in float32 for what a replayed graph of 21 kernels does in 65 and 81; three of 96: 34.3 and 62.5 for 76 and 110.
// What a phase between two barriers takes (three of 96, bfloat16, us): norm 0.6 to 0.8, q/k/v 0.6, rotation 0.7, attention 2.6, o 1.2,
// gate and up 1.5, down 1.3, none of it bytes or products but a wave's instructions one after the other, 4 and more cycles each.
//
// The step's rows stay in LDS: the stream h in float32, the operand of the next product (`a`: normed rows, then the attention's output),
// and that product's result (`b`: q, k and v, then the gated values).  A wave takes tiles of 16 output features and all rows; its
// weights come straight from memory, those of its first tile before the barrier in front of the product, so that they travel while the work
// before it is finished.
//
// Every sum has the order that the kernels of larger models give it (gemm_generic.hip, elementwise.hip, attention_walk.h), and every rounding its
// place, so in float32 a position's result has the same bits whichever way its step went.  In bfloat16 the products' sums go by
// increasing k and the probabilities stay in float32.
//
// (Eight or twelve waves in place of 16: more rows take 1.1 to 1.4 times as long.  The o product's first weights asked for before the attention: 3 us a step more, the
// registers spill.  All heads of a kv head, or two queries, side by side in a wave's attention, so that keys are read once or chains overlap: slower,
// 27 to 45 us for few rows, as lanes without a key then load, too.)
#include "attention_walk.h"
#include "tq_kernels.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

static_assert(sizeof(TqkSmallStep) <= 4000, "a kernel's arguments");

#define SS_WAVES 16
#define SS_THREADS (SS_WAVES * TQK_WAVE)
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

// How a step's rows lie in LDS, in bytes: the step's arrays, the layers' arguments, the norms' weights and the biases of all layers, the rows' angles, the waves' probabilities, then
// the stream and the two buffers.  Rows begin 16 bytes past a multiple of the banks' width, so that the 16 rows of an operand meet different ones.
struct SmallLayout {
    int ld_h, ld_a, ld_b, layers, norms, biases, angles, probs, a, b, h, bytes;       // ld_h in floats, ld_a in T, ld_b in bytes
};
static __device__ __host__ inline SmallLayout small_layout(const TqkSmallStep& p) {
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
    l.h = l.probs + SS_WAVES * SS_QUERIES * TQK_PAGE * 4;
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

template <typename T>
__global__ __launch_bounds__(SS_THREADS)
void small_step_kernel(const TqkSmallStep p) {
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
    const SmallLayout at = small_layout(p);
    int32_t* ints = reinterpret_cast<int32_t*>(lds);
    const TqkSmallLayer* layers = reinterpret_cast<const TqkSmallLayer*>(lds + at.layers);      // (the arguments lie far away)
    T *norms = reinterpret_cast<T*>(lds + at.norms), *biases = reinterpret_cast<T*>(lds + at.biases);
    float *angles = reinterpret_cast<float*>(lds + at.angles), *probs = reinterpret_cast<float*>(lds + at.probs) + wave * SS_QUERIES * TQK_PAGE;
    float* h = reinterpret_cast<float*>(lds + at.h);
    T* a = reinterpret_cast<T*>(lds + at.a);
    char* b = lds + at.b;
    auto round = [](float v) { return to_float(from_float<T>(v)); };

    auto product = [&](const void* w, int n, int k, int tiles) {
        SmallProduct<T, 1> one = {{(const char*)w}, n, k * (int)sizeof(T), tiles, lane, wave};
        one.ask();
        return one;
    };
    for (int i = tid; i < p.n_ints; i += SS_THREADS) ints[i] = p.ints[i];
    for (int i = tid; i < p.n_layers * (int)(sizeof(TqkSmallLayer) / 4); i += SS_THREADS)
        reinterpret_cast<int32_t*>(lds + at.layers)[i] = reinterpret_cast<const int32_t*>(p.layers)[i];
    for (int layer = wave; layer < p.n_layers; layer += SS_WAVES) {
        const TqkSmallLayer& l = p.layers[layer];
        for (int i = lane; i < hidden; i += TQK_WAVE) {
            norms[2 * layer * hidden + i] = ((const T*)l.norm1)[i];
            norms[(2 * layer + 1) * hidden + i] = ((const T*)l.norm2)[i];
        }
        if (l.qkv_bias) for (int i = lane; i < qkv; i += TQK_WAVE) biases[layer * qkv + i] = ((const T*)l.qkv_bias)[i];
    }
    for (int i = tid; i < hidden; i += SS_THREADS) norms[2 * p.n_layers * hidden + i] = ((const T*)p.final_norm)[i];
    lds_barrier();
    const int32_t *tokens = p.device_tokens ? p.device_tokens : ints + p.tokens, *tok_seq = ints + p.tok_seq, *tok_pos = ints + p.tok_pos;
    for (int r = wave; r < rows; r += SS_WAVES) {
        const int id = tokens[r], pos = min(tok_pos[r], p.max_positions - 1);
        const bool ok = id >= 0 && id < p.vocab;
        const T* row = (const T*)p.embedding + (size_t)(ok ? id : 0) * hidden;
        for (int i = lane; i < hidden; i += TQK_WAVE) h[r * at.ld_h + i] = ok ? to_float(row[i]) : 0.f;
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
    auto add_to_stream = [&](int row, int n, const floatx4_t* v) {
        floatx4_t* to = reinterpret_cast<floatx4_t*>(h + row * at.ld_h + n);
        *to = *to + rounded<T>(v[0]);
    };
    // queries a wave takes together: their elements side by side in its lanes
    const int width = d <= 16 ? 16 : d <= 32 ? 32 : 64, n_queries = rows * nh;
    const int together = min(TQK_WAVE / width, (n_queries + SS_WAVES - 1) / SS_WAVES);
    const float of_rows = 1.f / (float)rows, of_group = 1.f / (float)(nh / nkv);
    auto quotient = [&](int n) { return __builtin_amdgcn_readfirstlane((int)(((float)n + 0.5f) * of_rows)); };         // n / rows (numbers this small: exact)

#pragma unroll 1
    for (int layer = 0; layer < p.n_layers; ++layer) {
        TqkSmallLayer l;                                    // this layer's arguments, the same for all lanes
#pragma unroll
        for (int i = 0; i < (int)(sizeof(l) / 4); ++i)
            reinterpret_cast<int32_t*>(&l)[i] = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int32_t*>(layers + layer)[i]);
        const int32_t* table = ints + l.table;
        SmallProduct<T, 1> w_qkv = product(l.qkv, qkv, hidden, row_tiles);
        for (int r = wave; r < rows; r += SS_WAVES) norm_row(r, r, norms + 2 * layer * hidden, l.eps1);
        lds_barrier();
        float* bf = reinterpret_cast<float*>(b);
        const int ld_b = at.ld_b / 4;
        w_qkv.run(a, at.ld_a, rows, [&](int row, int n, const floatx4_t* v) { put4(bf + row * ld_b + n, rounded<T>(v[0])); });
        lds_barrier();
        // biases, rotation of q and k, keys and values into the row's page: a wave a row's heads in turn, a lane a pair that rotates together
        const int per = half <= 16 ? 4 : half <= 32 ? 2 : 1, sub = TQK_WAVE / per;      // heads a wave takes at once
#pragma unroll 1
        for (int e = wave; e < rows * ((nh + 2 * nkv + per - 1) / per); e += SS_WAVES) {
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
                lo = fmaf(x0, co, -(x1 * si));
                hi = fmaf(x1, co, x0 * si);
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
#pragma unroll 1
        for (int e0 = wave * together; e0 < n_queries; e0 += SS_WAVES * together) {
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
        SmallProduct<T, 1> w_o = product(l.o, hidden, qd, row_tiles);
        SmallProduct<T, 2> w_gate_up = {{(const char*)l.gate_up, (const char*)((const T*)l.gate_up + (size_t)inter * hidden)}, inter, hidden * (int)sizeof(T), row_tiles, lane, wave};
        lds_barrier();
        w_o.run(a, at.ld_a, rows, add_to_stream);
        w_gate_up.ask();
        lds_barrier();
        for (int r = wave; r < rows; r += SS_WAVES) norm_row(r, r, norms + (2 * layer + 1) * hidden, l.eps2);
        lds_barrier();
        T* act = reinterpret_cast<T*>(b);
        const int ld_act = at.ld_b / (int)sizeof(T);
        w_gate_up.run(a, at.ld_a, rows, [&](int row, int n, const floatx4_t* v) {
            const floatx4_t g = rounded<T>(v[0]), u = rounded<T>(v[1]);
            floatx4_t y;
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = gate_value(TQK_GATE_SILU, 0.f, 1.f, g[i], u[i]);
            put4(act + row * ld_act + n, y);
        });
        SmallProduct<T, 1> w_down = product(l.down, hidden, inter, row_tiles);
        lds_barrier();
        w_down.run(act, ld_act, rows, add_to_stream);
        lds_barrier();
    }

    if (p.n_want == 0) return;
    SmallProduct<T, 1> w_head = product(p.head, p.vocab, hidden, (p.n_want + 15) / 16);
    const int32_t* want = ints + p.want;
    for (int r = wave; r < p.n_want; r += SS_WAVES) norm_row(want[r], r, norms + 2 * p.n_layers * hidden, p.final_eps);
    lds_barrier();
    w_head.run(a, at.ld_a, p.n_want, [&](int row, int n, const floatx4_t* v) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < p.vocab) p.logits[(size_t)row * p.vocab + n + i] = v[0][i];
    });
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
    if (small_layout(p).bytes > 160 * 1024) return 0;
    // (larger products have another order of summation there)
    if (p.act_dtype == TQK_F32 && (tqk_gemm_takes_apart(p.vocab, p.hidden) || tqk_gemm_takes_apart(2 * p.inter, p.hidden) || tqk_gemm_takes_apart(q + 2 * p.n_kv_heads * p.head_dim, p.hidden))) return 0;
    return 1;
}

/* Whether that is the faster way, by an estimate in microseconds (decode: a step of one token a sequence, which the other kernels run as a replayed graph; positions: the
 * furthest one of the step).  One block: 5 a layer for its barriers and chains of short operations, its weights at 33 KB (27 in float32) a microsecond, and for every row what
 * its products, its other work and its heads' pages take; the head's weights at 39 KB.  The other kernels, ten launches a layer: 20 a layer in a graph (33 in float32) and 32 (45) one by one.
 * Measured, one block and the other kernels, two layers of 64 values with 160 in the feed-forward, bfloat16: 1 and 16 sequences 35 and 72, 63 and 68, 40 sequences 90 and 73, prompts of 8, 33
 * and 64 tokens 31 and 88, 61 and 88, 109 and 90; three of 96 with 224: 37 and 74, 77 and 77, 135 and 97, 40 and 120, 99 and 117, 165 and 118; four of 128 with 512: 88 and 83, 193 and 89, then 94
 * and 138, 263 and 141; four of 256 with 512: 171 and 98, 374 and 102, then 184 and 138.  float32: 36 and 81, 76 and 85, 38 and 91, 90 and 93, 149 and 99; three of 96: 64 and 108, 116 and 113, 71 and 117, 196 and 136. */
extern "C" int tqk_small_step_pays(const TqkSmallStep* step, int decode, int positions) {
    const TqkSmallStep& p = *step;
    const bool f32 = p.act_dtype == TQK_F32;
    const double size = f32 ? 4 : 2, q = (double)p.n_heads * p.head_dim;
    const double thousands = 1e-3 * p.hidden * (2 * q + 2. * p.n_kv_heads * p.head_dim + 3. * p.inter);            // weights of a layer
    const double a_row = 0.15 + (f32 ? 0.0115 : 0.0043) * thousands + 0.08 * p.n_heads * ((positions + TQK_PAGE - 1) / TQK_PAGE);
    const double here = 8 + p.n_layers * (5 + thousands * size / (f32 ? 27 : 33) + p.n_rows * a_row) + 1e-3 * p.vocab * p.hidden * size / 39;
    const double there = decode ? 15 + p.n_layers * (f32 ? 33 : 20) : 15 + p.n_layers * (f32 ? 45 : 32);
    return here < there;
}

template <typename T>
static int launch_small(const TqkSmallStep& p, hipStream_t s) {
    static const hipError_t grown = hipFuncSetAttribute((const void*)small_step_kernel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (grown != hipSuccess) return tqk_fail("tqk_small_step: %s", hipGetErrorString(grown));
    small_step_kernel<T><<<1 + 8 * (p.n_layers + 1), SS_THREADS, small_layout(p).bytes, s>>>(p);
    return tqk_check_launch("tqk_small_step");
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
    TQK_REQUIRE(p.tok_seq >= 0 && p.tok_pos >= 0 && p.want >= 0 && p.tok_seq + p.n_rows <= p.n_ints && p.tok_pos + p.n_rows <= p.n_ints && p.want + p.n_want <= p.n_ints &&
                    (p.device_tokens || (p.tokens >= 0 && p.tokens + p.n_rows <= p.n_ints)), "tqk_small_step: the step's arrays do not lie in what was given");
    hipStream_t s = (hipStream_t)stream;
    return p.act_dtype == TQK_F32 ? launch_small<float>(p, s) : launch_small<bf16_t>(p, s);
}
