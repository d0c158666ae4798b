// y[M,N] = x[M,K] w[N,K]^T (+ bias): the plain product of the float32 path, and of
// any dtype mix the fast kernels do not take.  The reference's linear layers are
// candle matmuls (src/models/turbo_generic.rs:68-91, 779-781).
//
// float32 throughout, K a multiple of 4 and operands at 16 bytes (every product of the float32 path of a usual model):
// v_mfma_f32_16x16x4_f32, whose products and sums are float32 ones, and for large weights v_mfma_f32_16x16x32_bf16 on numbers taken apart
// without loss.  Everything else: LDS-tiled, 64x64 outputs per block, 4x4 per thread, float32 FMA.
//
// The order of summation is fixed and the same for all numbers of rows, so that a result does
// not depend on M or on where a row stands in the batch: k is
// cut into chunks of 128 and groups of 8 chunks; a chunk is summed from zero, a group is the sum of its chunks in order,
// the result the sum of the groups in order (and then the bias).  Within a chunk the FMA kernel goes by increasing k; the
// matrix-core kernels take 16 k at a time, four instructions of which number i adds the k with k % 4 == i to what the ones
// before it left (a lane then reads its operands of all four as 16 contiguous bytes), with the same operands in the same
// registers in both, so those two give the same bits.  Products with large weights (tqk_gemm_takes_apart) go by three bfloat16 numbers for a float32 one, 32 k at a time, again
// in one order in all their kernels.  Which of the three orders a product gets is a matter of types, N, K and addresses alone.
//
// For up to 16 rows of x (decoding in the 32-bit path) the weights are the whole cost: a wave takes 16 output features and one
// group of k and streams their weights through LDS, 12 KB of them under way; groups beyond the first meet in a second
// kernel.  More rows: a block of four waves takes 64 rows by 64 features (up to 128, for large weights) through LDS; where that gives
// few blocks they are also dealt out along the groups.  Measured at the 7B layers' sizes: see the kernels.
#include "common.h"
#include "tq_kernels.h"

#include <type_traits>
#include <utility>

#define GT 64      // tile edge
#define GK 16      // k per stage
#define G_CHUNK 128                 // k per chunk
#define G_GROUP (8 * G_CHUNK)       // k per group

template <typename TX, typename TW, typename TB, typename TY>
__global__ __launch_bounds__(256)
void gemm_generic_kernel(const TX* __restrict__ x, const TW* __restrict__ w, const TB* __restrict__ bias,
                         TY* __restrict__ y, int M, int N, int K) {
    __shared__ float xs[GK][GT + 4];
    __shared__ float ws[GK][GT + 4];
    const int tid = threadIdx.x;
    const int tm = tid / 16, tn = tid % 16;            // thread's 4x4 patch: rows tm*4.., cols tn*4..
    const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
    float acc[4][4], group[4][4], total[4][4];      // the chunk, the group and the result so far
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = group[i][j] = total[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += GK) {
        // 64 rows x 16 k = 1024 elements per operand, 4 per thread
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int idx = tid + e * 256;
            const int r = idx / GK, kk = idx % GK;
            const int gm = m0 + r, gn = n0 + r, gk = k0 + kk;
            xs[kk][r] = (gm < M && gk < K) ? to_float(x[(size_t)gm * K + gk]) : 0.f;
            ws[kk][r] = (gn < N && gk < K) ? to_float(w[(size_t)gn * K + gk]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = xs[kk][tm * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = ws[kk][tn * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
        const int k_done = k0 + GK;
        if (k_done % G_CHUNK == 0 || k_done >= K) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) { group[i][j] += acc[i][j]; acc[i][j] = 0.f; }
        }
        if (k_done % G_GROUP == 0 || k_done >= K) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) { total[i][j] += group[i][j]; group[i][j] = 0.f; }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gm = m0 + tm * 4 + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int gn = n0 + tn * 4 + j;
            if (gn >= N) continue;
            float v = total[i][j];
            if (bias) v += to_float(bias[gn]);
            y[(size_t)gm * N + gn] = from_float<TY>(v);
        }
    }
}

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
template <typename F, int... I> __device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each(f, std::make_integer_sequence<int, N>{}); }

// 16 k more: lane l holds, of both operands, row l % 16 and the four k at 4 (l / 16); of the sums row (of x) l % 16 and the
// features 4 (l / 16) .. + 3.
__device__ __forceinline__ void multiply16(floatx4_t& acc, const floatx4_t& w, const floatx4_t& x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
}

// ---- large weights: a float32 number as three bfloat16 ones -----------------------------------------
// 24 bits are 8 + 8 + 8: p the number cut off after 8 bits (so that nothing overflows), q what is left rounded to 8, t what is left then, exactly from 2^-110 on (bfloat16
// ends at 2^-133).  Of the nine products of two numbers' parts the smallest, t t, is left out (2^-32 of the whole); the others are exact in float32.  The matrix cores cut a sum off
// where float32 instructions round it, so the largest products have a sum of their own, and the seven others, a 128th of it, another; the two are added at the end of a
// chunk.  Eight bfloat16 instructions stand for eight float32 ones of twice the time each, and their sums of 32 k at once round less often: error against
// 64 bits, 2-norm in 2^-24, K of 3584 and 18944, operands N(0, 1) 1.57 and 2.02 (the float32 instructions 3.61 and 3.82), all of one sign 0.83 and 1.18 (0.98 and 1.20), spread
// over twelve powers of ten 1.90 and 2.49 (2.92 and 3.15), rows with one value alone 0.42 and 0.42 (0.42 and 0.42; the largest 1.0 both ways), with one 10^8 times the others 1.64 and 2.27 (1.69 and
// 2.28).  Without q t and t q, and all in one sum, prompts took 0.88 of the time (300 rows of gate+up of the 7B shape 534 us and 607), but rows with one value had 0.67, the largest 3.9.
// Infinities have no parts (inf - inf), and numbers below 2^-110 lose up to 2^-133 of theirs, which is less than 2^-24 of a sum from 2^-64 on unless what they meet is beyond
// 2^30: a group's sum that is not finite, or smaller than that and not 0, is taken again with the float32 instructions, that one and no other, so that a
// result depends on its own rows of x and w alone.  (Sums of 0 stand, as rows of zeros are common: where all that a row meets are numbers below 2^-133, the result is 0.)
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
struct Parts { bf16x8_t p, q, t; };
__device__ __forceinline__ uint32_t high_halves(float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); }
__device__ __forceinline__ void split2(float a, float b, uint32_t& p, uint32_t& q, uint32_t& t) {
    p = high_halves(a, b);
    a -= __uint_as_float(__float_as_uint(a) & 0xffff0000u);
    b -= __uint_as_float(__float_as_uint(b) & 0xffff0000u);
    q = (uint32_t)float_to_bf16_bits(a) | (uint32_t)float_to_bf16_bits(b) << 16;
    a -= __uint_as_float(q << 16);
    b -= __uint_as_float(q & 0xffff0000u);
    t = high_halves(a, b);
}
__device__ __forceinline__ Parts split8(floatx4_t a, floatx4_t b) {
    u32x4_t p, q, t;
    uint32_t pp, qq, tt;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const floatx4_t v = i < 2 ? a : b;
        split2(v[2 * (i % 2)], v[2 * (i % 2) + 1], pp, qq, tt);
        p[i] = pp; q[i] = qq; t[i] = tt;
    }
    return {__builtin_bit_cast(bf16x8_t, p), __builtin_bit_cast(bf16x8_t, q), __builtin_bit_cast(bf16x8_t, t)};
}
// 32 k more: a lane holds, of both operands, row lane % 16 and the eight k at 8 (lane / 16); acc: the largest products, low: the others, the smallest first.
__device__ __forceinline__ void multiply32(floatx4_t& acc, floatx4_t& low, const Parts& w, const Parts& x) {
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.t, x.q, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.q, x.t, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.t, x.p, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p, x.t, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.q, x.q, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.q, x.p, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p, x.q, low, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.p, x.p, acc, 0, 0, 0);
}
__device__ __forceinline__ bool stands(float v) {
    const uint32_t twice = __float_as_uint(v) << 1;                     // (without its sign; 2^-64's exponent is 63, that of what is not finite 255)
    return twice == 0 || twice - (63u << 24) < 192u << 24;
}
__device__ __forceinline__ bool stand(floatx4_t v) { return stands(v[0]) && stands(v[1]) && stands(v[2]) && stands(v[3]); }
// The sums of a group (k_begin .. k_end) of 16 rows and 16 features by the float32 instructions, for a wave; xrow, wrow: the lane's rows.
__device__ __forceinline__ floatx4_t plain_group(const float* xrow, const float* wrow, int k_begin, int k_end, int k4) {
    floatx4_t group = {0.f, 0.f, 0.f, 0.f};
    for (int c0 = k_begin; c0 < k_end; c0 += G_CHUNK) {
        floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
        for (int k0 = c0; k0 < min(c0 + G_CHUNK, k_end); k0 += 16) {
            const floatx4_t none = {0.f, 0.f, 0.f, 0.f};
            const bool in = k0 + k4 < k_end;
            multiply16(acc, in ? *reinterpret_cast<const floatx4_t*>(wrow + k0 + k4) : none, in ? *reinterpret_cast<const floatx4_t*>(xrow + k0 + k4) : none);
        }
        group += acc;
    }
    return group;
}

// Up to 16 rows of x: a wave per (16 output features, one group of k).  With one group the result is finished here.
// Bound by the weights.  They come in stages of 64 k, 256 contiguous bytes of each of the 16 rows, by loads that end in LDS, three
// stages on their way while one is multiplied; a piece of 16 bytes lies at its number exclusive-or its row, so that the operands of 16
// rows meet all banks.  gate+up of the 7B shape (543 MB; products that large go by parts now, below), one row: 100 us (5.4 TB/s), eight rows 114; 131 and
// 141 with the operands loaded as the lanes need them, 64 bytes out of 16 rows a load, eight of those under way.
#define FEW_STAGES 4
__global__ __launch_bounds__(TQK_WAVE)
void gemm_few_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                          int M, int N, int K) {
    constexpr int NS = FEW_STAGES, U = 4;                               // 16 k a step, four steps a stage
    __shared__ __attribute__((aligned(1024))) float buf0[1024], buf1[1024], buf2[1024], buf3[1024];
    const int lane = threadIdx.x, r16 = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * 16;
    const int k_begin = blockIdx.y * G_GROUP, k_end = min(K, k_begin + G_GROUP), n_stage = (k_end - k_begin + 63) / 64;
    const float* xrow = x + (size_t)min(r16, M - 1) * K;                // rows past M repeat the last and are dropped
    // (rows past N and everything past the last row lie outside of the buffer: nothing is read there)
    const __amdgpu_buffer_rsrc_t w_mem = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, min(16, N - n0) * K * 4, 0x00020000);
    uint32_t w_at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 4 * j + g;
        w_at[j] = (uint32_t)row * (uint32_t)(K * 4) + ((r16 ^ row) * 16);
    }
    auto buf = [&](auto I) -> float* {
        constexpr int i = decltype(I)::value % NS;
        if constexpr (i == 0) return buf0; else if constexpr (i == 1) return buf1; else if constexpr (i == 2) return buf2; else return buf3;
    };
    floatx4_t xv[NS][U];
    auto load = [&](auto I, int stage) {
        const bool there = stage < n_stage;                             // (past the last stage: outside of the buffer, nothing is read)
        const int k0 = k_begin + (there ? stage * 64 : 0);
        const uint32_t nowhere = there ? 0u : 0x80000000u;              // (joined to the offsets, so that no branch lies here)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_mem, (lds_ptr_t)(buf(I) + j * 256), 16, (int)(w_at[j] | nowhere), k0 * 4, 0, 0);
#pragma unroll
        for (int u = 0; u < U; ++u) xv[decltype(I)::value % NS][u] = *reinterpret_cast<const floatx4_t*>(xrow + min(k0 + 16 * u + 4 * g, K - 4));
    };
    floatx4_t group = {0.f, 0.f, 0.f, 0.f}, acc = group;
    // (no branch in a stage: every stage issues its eight loads and multiplies, past the end what is nothing)
    auto multiply = [&](auto I, int stage) {
        const float* src = buf(I);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const u32x4_t wq = *reinterpret_cast<const u32x4_t*>(src + r16 * 64 + ((4 * u + g) ^ r16) * 4);
            const uint32_t in = k_begin + stage * 64 + 16 * u + 4 * g < k_end ? 0xffffffffu : 0u;       // past k_end both operands are nothing
            multiply16(acc, __builtin_bit_cast(floatx4_t, wq & in), __builtin_bit_cast(floatx4_t, __builtin_bit_cast(u32x4_t, xv[decltype(I)::value % NS][u]) & in));
        }
    };
    // The waits below count eight loads a stage in the stages' order.  Barriers keep the scheduler to it, and there is no test in front
    // of the loop (n_stage is at least 1): behind one the compiler had put all loads of x after all those of the weights.
    each<NS - 1>([&](auto S) {
        load(S, S);
        __builtin_amdgcn_sched_barrier(0);
    });
    int s0 = 0;
    do {
        each<NS>([&](auto S) {
            constexpr int h = decltype(S)::value;
            load(std::integral_constant<int, h + NS - 1>{}, s0 + h + NS - 1);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x0f70 | ((8 * (NS - 1)) & 15) | (((8 * (NS - 1)) >> 4) << 14));      // this stage's loads: eight of each later one may be under way
            __builtin_amdgcn_sched_barrier(0);
            multiply(S, s0 + h);
            if constexpr (h % 2 == 1) {
                group += acc;
                acc = floatx4_t{0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        s0 += NS;
    } while (s0 < n_stage);
    __builtin_amdgcn_s_waitcnt(0x0f70);                                 // nothing is on its way into LDS any more
    if (r16 >= M) return;
    const bool whole = gridDim.y == 1;
    float* dst = out + ((size_t)blockIdx.y * M + r16) * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + 4 * g + i;
        if (n < N) dst[n] = whole && bias ? group[i] + bias[n] : group[i];
    }
}

// The same by parts in bfloat16, for large weights.  What it spends beside its loads is taking numbers apart, 88 instructions for a stage's weights and as many for its x.
// ROWS: up to 4, 8 or 16 rows of x.  Of the 16 lanes that hold x's rows four (two) stand for one row where there are few, each takes a quarter (half) of the row's values apart,
// and the first gets the others' parts by turning the 16 lanes: 40 (56) instructions, and a quarter (half) of the loads; without the turning it takes 1.14, 1.08 and 1.02 of the time of
// one row, 4608, 3584 and 37888 features, K of 3584, 18944 and 3584.
// ONCE: the weights' loads say that they are read once (nt), as those of the bfloat16 kernels do: for a caller whose weights together are more than the caches hold and who reads each once a step
// (tqk_gemm_once).  Those sizes and 152064 features, with the kernel that adds up the groups, weights that no cache holds, us with and without: one row 16.0, 51, 93 and 335 (17.3, 55, 100 and
// 376: 6.5 TB/s in place of 5.8), 8 rows 17.9, 58, 105 and 428 (18.4, 62, 118 and 453); 8192 features, K of 2048, and the other way about, and 17920, K of 1536, one row 17.5, 18.3 and 26.1 (19.1, 20.0 and 28.1).
// Weights of 64 to 200 MB in all that the memory-side cache holds from one reading to the next lose by it: the first two of those sizes 16.5 and 18.2 (14.4 and 14.4), 16 rows 18.4 and 19.6 (16.2 and
// 16.3), 37888 features, K of 1024, 33.5 (30.2); 4608 and 3584 features, K of 3584, 14.9 and 12.6 (15.2 and 13.0); those of 4 to 32 MB each 0 to 2 %.
// TAIL: K is no multiple of 64.
template <bool TAIL, int ROWS, bool ONCE>
__global__ __launch_bounds__(TQK_WAVE)
void gemm_few_rows_apart_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                          int M, int N, int K) {
    constexpr int NS = FEW_STAGES, U = 4;                               // 16 k a step, four steps a stage
    __shared__ __attribute__((aligned(1024))) float buf0[1024], buf1[1024], buf2[1024], buf3[1024];
    const int lane = threadIdx.x, r16 = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * 16;
    const int k_begin = blockIdx.y * G_GROUP, k_end = min(K, k_begin + G_GROUP), n_stage = (k_end - k_begin + 63) / 64;
    const float* xrow = x + (size_t)min(r16 % ROWS, M - 1) * K;        // rows past M repeat the last and are dropped
    // (rows past N and everything past the last row lie outside of the buffer: nothing is read there)
    const __amdgpu_buffer_rsrc_t w_mem = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, min(16, N - n0) * K * 4, 0x00020000);
    uint32_t w_at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = 4 * j + g;
        w_at[j] = (uint32_t)row * (uint32_t)(K * 4) + ((r16 ^ row) * 16);
    }
    auto buf = [&](auto I) -> float* {
        constexpr int i = decltype(I)::value % NS;
        if constexpr (i == 0) return buf0; else if constexpr (i == 1) return buf1; else if constexpr (i == 2) return buf2; else return buf3;
    };
    constexpr int XU = ROWS / 4, LOADS = 4 + XU;
    floatx4_t xv[NS][XU];
    // where in a stage the lane's four k of part u of its operands lie
    auto place = [&](int u) { return 32 * (u / 2) + 8 * g + 4 * (u % 2); };
    auto x_place = [&](int u) { return place(r16 / ROWS * XU + u); };       // (of the x that the lane takes apart)
    auto load = [&](auto I, int stage) {
        const bool there = stage < n_stage;                             // (past the last stage: outside of the buffer, nothing is read)
        const int k0 = k_begin + (there ? stage * 64 : 0);
        const uint32_t nowhere = there ? 0u : 0x80000000u;              // (joined to the offsets, so that no branch lies here)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(w_mem, (lds_ptr_t)(buf(I) + j * 256), 16, (int)(w_at[j] | nowhere), k0 * 4, 0, ONCE ? 2 : 0);
#pragma unroll
        for (int u = 0; u < XU; ++u) xv[decltype(I)::value % NS][u] = *reinterpret_cast<const floatx4_t*>(xrow + min(k0 + x_place(u), K - 4));
    };
    floatx4_t group = {0.f, 0.f, 0.f, 0.f}, acc = group, low = group;
    // (no branch in a stage: every stage issues its loads and multiplies, past the end what is nothing)
    auto multiply = [&](auto I, int stage) {
        const float* src = buf(I);
        auto inside = [&](int at) { return (TAIL ? k_begin + stage * 64 + at < k_end : stage < n_stage) ? 0xffffffffu : 0u; };      // past k_end both operands are nothing
        auto masked = [&](floatx4_t v, uint32_t in) { return __builtin_bit_cast(floatx4_t, __builtin_bit_cast(u32x4_t, v) & in); };
        // (of a whole stage past it one of them alone: sums that are not finite are taken again anyway)
        floatx4_t wv[U], xs[XU];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            wv[u] = *reinterpret_cast<const floatx4_t*>(src + r16 * 64 + ((place(u) / 4) ^ r16) * 4);
            if (TAIL) wv[u] = masked(wv[u], inside(place(u)));
        }
#pragma unroll
        for (int u = 0; u < XU; ++u) xs[u] = masked(xv[decltype(I)::value % NS][u], inside(x_place(u)));
        Parts xp[2];
        auto turned = [&](auto ctrl, const Parts& from) {
            u32x4_t p = __builtin_bit_cast(u32x4_t, from.p), q = __builtin_bit_cast(u32x4_t, from.q), t = __builtin_bit_cast(u32x4_t, from.t);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)p[i], decltype(ctrl)::value, 0xf, 0xf, true);
                q[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)q[i], decltype(ctrl)::value, 0xf, 0xf, true);
                t[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t[i], decltype(ctrl)::value, 0xf, 0xf, true);
            }
            return Parts{__builtin_bit_cast(bf16x8_t, p), __builtin_bit_cast(bf16x8_t, q), __builtin_bit_cast(bf16x8_t, t)};
        };
        if constexpr (ROWS == 16) {
#pragma unroll
            for (int h = 0; h < 2; ++h) xp[h] = split8(xs[2 * h], xs[2 * h + 1]);
        } else if constexpr (ROWS == 8) {
            xp[0] = split8(xs[0], xs[1]);
            xp[1] = turned(std::integral_constant<int, 0x128>{}, xp[0]);                        // row_ror:8
        } else {
            // (own values first, then those of the lane four on (row_ror:12); the lanes eight on (row_ror:8) hold the other half so)
            uint32_t own[3][2];
            split2(xs[0][0], xs[0][1], own[0][0], own[1][0], own[2][0]);
            split2(xs[0][2], xs[0][3], own[0][1], own[1][1], own[2][1]);
            u32x4_t parts[3];
#pragma unroll
            for (int part = 0; part < 3; ++part)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    parts[part][i] = own[part][i];
                    parts[part][2 + i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own[part][i], 0x12c, 0xf, 0xf, true);
                }
            xp[0] = {__builtin_bit_cast(bf16x8_t, parts[0]), __builtin_bit_cast(bf16x8_t, parts[1]), __builtin_bit_cast(bf16x8_t, parts[2])};
            xp[1] = turned(std::integral_constant<int, 0x128>{}, xp[0]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) multiply32(acc, low, split8(wv[2 * h], wv[2 * h + 1]), xp[h]);
    };
    // The waits below count LOADS loads a stage in the stages' order.  Barriers keep the scheduler to it, and there is no test in front
    // of the loop (n_stage is at least 1): behind one the compiler had put all loads of x after all those of the weights.
    each<NS - 1>([&](auto S) {
        load(S, S);
        __builtin_amdgcn_sched_barrier(0);
    });
    int s0 = 0;
    do {
        each<NS>([&](auto S) {
            constexpr int h = decltype(S)::value;
            load(std::integral_constant<int, h + NS - 1>{}, s0 + h + NS - 1);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(0x0f70 | ((LOADS * (NS - 1)) & 15) | (((LOADS * (NS - 1)) >> 4) << 14));      // this stage's loads: those of each later one may be under way
            __builtin_amdgcn_sched_barrier(0);
            multiply(S, s0 + h);
            if constexpr (h % 2 == 1) {
                group += acc + low;
                acc = low = floatx4_t{0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        s0 += NS;
    } while (s0 < n_stage);
    __builtin_amdgcn_s_waitcnt(0x0f70);                                 // nothing is on its way into LDS any more
    if (__any(r16 < M && !stand(group))) {
        const floatx4_t plain = plain_group(x + (size_t)min(r16, M - 1) * K, w + (size_t)min(n0 + r16, N - 1) * K, k_begin, k_end, 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) group[i] = stands(group[i]) ? group[i] : plain[i];
    }
    if (r16 >= M) return;
    const bool whole = gridDim.y == 1;
    float* dst = out + ((size_t)blockIdx.y * M + r16) * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + 4 * g + i;
        if (n < N) dst[n] = whole && bias ? group[i] + bias[n] : group[i];
    }
}

// More rows: 64 rows by 64 features a block, each of four waves 32 by 32.  Stages of 32 k go through registers into LDS, two in turn;
// a row's 128 bytes lie 144 apart, so that the 16 rows of an operand meet all banks.  blockIdx.y: the block's share of the
// groups; with more than one share every group's sums go to scratch on their own.  Bound by the matrix cores (157 TFLOP/s in
// float32): gate+up of the 7B shape at 300 rows (products that large go by parts now, below) 750 us = 109 TFLOP/s (826 with the rows' tiles of some features far apart, 805 with loads one stage
// ahead, as a stage is hardly longer than a load takes, 855 with neither), and 2108 us through the FMA kernel above; down 465 us with the
// groups' sums written and added (495 with neither), 40 rows 206 and 108 (229 and 111).  Blocks of 160 rows by 64 features took 967 us
// for gate+up: fewer waves lose more than the bytes saved.
#define GM_LINE 36              // floats from row to row in LDS
__global__ __launch_bounds__(256)
void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                     int M, int N, int K, int groups_per_share) {
    __shared__ __attribute__((aligned(16))) float lds[2][2][GT * GM_LINE];     // [stage][x, w]
    const int tid = threadIdx.x, lane = tid % TQK_WAVE, wave = tid / TQK_WAVE;
    const int r16 = lane % 16, k4 = 4 * (lane / 16);
    // Blocks are dealt to the eight dies in turn: all rows' tiles of some features go to one die one after the other, so that the weights come out
    // of its second-level cache for all but the first.  37888 features, K of 3584, 300, 1024 and 4096 rows: 826, 2534 and 10307 us with neighbouring
    // blocks on one row of tiles, 752, 2276 and 9030 so.  Where the weights are small it hardly matters: 512 to 17920 features, 100 to 8192 rows within
    // 2 %, but for single sizes (3584 features and 2048 rows, 4096 and 4096: 4 and 5 % slower).  (Shares of K read other weights, so it is no loss that
    // a share's dealing begins at another die where the tiles are no multiple of eight.)
    const int tiles_m = (M + GT - 1) / GT, tiles_n = (N + GT - 1) / GT;
    int tm, tn;
    {
        const int n = tiles_m * tiles_n, die = blockIdx.x % 8, at = blockIdx.x / 8, each_die = n / 8, more = n % 8;
        const int id = die * each_die + min(die, more) + at;
        tm = id % tiles_m;
        tn = id / tiles_m;
    }
    const int m0 = tm * GT, n0 = tn * GT, wm = wave / 2 * 32, wn = wave % 2 * 32;
    const int k_begin = blockIdx.y * groups_per_share * G_GROUP, k_end = min(K, k_begin + groups_per_share * G_GROUP);
    const bool shared_out = gridDim.y > 1;
    // what a thread brings in: of rows tid / 8 and 32 + tid / 8 of both tiles the four k at 4 (tid % 8) (rows past the end repeat the last)
    const int sr = tid / 8, sk = 4 * (tid % 8);
    const float* src[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        src[0][i] = x + (size_t)min(m0 + sr + 32 * i, M - 1) * K;
        src[1][i] = w + (size_t)min(n0 + sr + 32 * i, N - 1) * K;
    }
    floatx4_t ahead[2][2][2];          // [stage % 2]: a stage's loads are issued two stages before it
    auto load = [&](int k0, int to) {
        const int k = min(k0 + sk, K - 4);          // past K: read from inside the row, zeros in its place
        const bool in = k0 + sk < K;
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                ahead[to][o][i] = *reinterpret_cast<const floatx4_t*>(src[o][i] + k);
                if (!in) ahead[to][o][i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            }
    };
    auto put = [&](int stage) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<floatx4_t*>(&lds[stage][o][(sr + 32 * i) * GM_LINE + sk]) = ahead[stage][o][i];
    };
    floatx4_t acc[2][2], group[2][2], total[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = group[a][b] = total[a][b] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto write = [&](float* y, const floatx4_t (&v)[2][2], bool with_bias) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int m = m0 + wm + 16 * a + r16;
            if (m >= M) continue;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int n = n0 + wn + 16 * b + k4 + i;
                    if (n < N) y[(size_t)m * N + n] = with_bias ? v[a][b][i] + bias[n] : v[a][b][i];
                }
        }
    };
    load(k_begin, 0);
    load(k_begin + 32, 1);
    put(0);
    __syncthreads();
    for (int c0 = k_begin; c0 < k_end; c0 += G_CHUNK) {
        // a chunk is four stages in a straight line (a last chunk that is not full meets zeros)
#pragma unroll
        for (int q = 0; q < G_CHUNK / 32; ++q) {
            const int stage = q % 2;
            load(c0 + 32 * (q + 2), stage);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                floatx4_t xv[2], wv[2];
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    xv[a] = *reinterpret_cast<const floatx4_t*>(&lds[stage][0][(wm + 16 * a + r16) * GM_LINE + 16 * h + k4]);
                    wv[a] = *reinterpret_cast<const floatx4_t*>(&lds[stage][1][(wn + 16 * a + r16) * GM_LINE + 16 * h + k4]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int a = 0; a < 2; ++a)
#pragma unroll
                        for (int b = 0; b < 2; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[b][i], xv[a][i], acc[a][b], 0, 0, 0);
            }
            if (q == G_CHUNK / 32 - 1) {
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) { group[a][b] += acc[a][b]; acc[a][b] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
            }
            put(stage ^ 1);
            __syncthreads();
        }
        const int done = c0 + G_CHUNK;
        if (done % G_GROUP == 0 || done >= k_end) {
            if (shared_out) write(out + (size_t)(c0 / G_GROUP) * M * N, group, false);
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) { total[a][b] += group[a][b]; group[a][b] = floatx4_t{0.f, 0.f, 0.f, 0.f}; }
        }
    }
    if (!shared_out) write(out, total, bias != nullptr);
}

// More rows against large weights, by parts in bfloat16: a block of four waves takes 16 RT rows by 64 FT features, each wave all rows of 16 FT.  A wave's weights come straight from
// memory to its own registers, which take them apart; x goes through LDS, taken apart once for the block (stages of 64 k, three parts a row of 128 bytes each, pieces of 16
// bytes at their number exclusive-or half their row, so that the 16 rows of an operand meet all banks; two stages in turn, one barrier each).  Loads are issued
// half a stage or a stage ahead of being taken apart, which happens beside the products of the half before.  Whole groups' sums wait in LDS too, a float4 of each thread's in turn, where
// the registers would cost a wave per SIMD.  Bound by the matrix cores' power and by what LDS delivers of x (12 pieces a wave for 64 products: two fifths of the time of those).  us, gate+up of the 7B
// shape, down, q/k/v and o at 300 rows: 607, 351, 103 and 86 (744, 463, 114 and 98 with the float32 instructions); 2000 rows of o 386 (441).  With six products in place of eight gate+up took 581, and of that: weights in
// whole lines in place of the matrix cores' order 0.96, not without LDS between; waves of 48 or 64 features, one to a SIMD, 1.15 and 1.23; numbers taken apart in front of the products 1.01.
#define GS_WAVES 4
template <int RT, int FT, bool TAIL>
__global__ __launch_bounds__(GS_WAVES * TQK_WAVE, 2)
void gemm_split_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                       int M, int N, int K, int groups_per_share) {
    constexpr int ROWS = 16 * RT, FEATURES = 16 * FT * GS_WAVES, THREADS = GS_WAVES * TQK_WAVE, XL = ROWS * 16 / THREADS;     // XL: what a thread brings in of x, in four k each
    __shared__ __attribute__((aligned(16))) char lds[2][3][ROWS * 128];
    __shared__ floatx4_t totals[FT * RT][THREADS];
    const int tid = threadIdx.x, lane = tid % TQK_WAVE, wave = tid / TQK_WAVE, r16 = lane % 16, g = lane / 16;
    const int tiles_m = (M + ROWS - 1) / ROWS, tiles_n = (N + FEATURES - 1) / FEATURES;
    int tm, tn;                                 // (blocks over the dies as in gemm_f32_kernel)
    {
        const int n = tiles_m * tiles_n, die = blockIdx.x % 8, at = blockIdx.x / 8, each_die = n / 8, more = n % 8;
        const int id = die * each_die + min(die, more) + at;
        tm = id % tiles_m;
        tn = id / tiles_m;
    }
    const int m0 = tm * ROWS, n0 = tn * FEATURES + wave * 16 * FT;
    const int k_begin = blockIdx.y * groups_per_share * G_GROUP, k_end = min(K, k_begin + groups_per_share * G_GROUP);
    const bool shared_out = gridDim.y > 1;
    const float* wrow[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) wrow[f] = w + (size_t)min(n0 + 16 * f + r16, N - 1) * K;
    const float* xsrc[XL];
    int xdst[XL];
    const int xk = 4 * (tid % 16);
#pragma unroll
    for (int i = 0; i < XL; ++i) {
        const int row = tid / 16 + i * (THREADS / 16);
        xsrc[i] = x + (size_t)min(m0 + row, M - 1) * K + xk;
        xdst[i] = row * 128 + (((xk / 8) ^ ((row >> 1) & 7)) * 16) + (xk & 4) * 2;
    }
    const floatx4_t none = {0.f, 0.f, 0.f, 0.f};
    floatx4_t wv[FT][4], xv[XL];
    // (past the last stage, and with TAIL past K, the row's last values are read; what lies past k_end counts as nothing when it is taken apart)
    auto load_w = [&](int k0, int h) {
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int u = 0; u < 2; ++u) wv[f][2 * h + u] = *reinterpret_cast<const floatx4_t*>(wrow[f] + min(k0 + 32 * h + 8 * g + 4 * u, K - 4));
    };
    auto load_x = [&](int k0, int h) {
#pragma unroll
        for (int i = h * XL / 2; i < (h + 1) * XL / 2; ++i) xv[i] = *reinterpret_cast<const floatx4_t*>(xsrc[i] + min(k0, K - 4 - xk));
    };
    auto put_x = [&](int k0, int to, int h) {
        const bool in = !TAIL || k0 + xk < k_end;
#pragma unroll
        for (int i = h * XL / 2; i < (h + 1) * XL / 2; ++i) {
            const floatx4_t v = in ? xv[i] : none;
            uint2 p, q, t;
            split2(v[0], v[1], p.x, q.x, t.x);
            split2(v[2], v[3], p.y, q.y, t.y);
            *reinterpret_cast<uint2*>(&lds[to][0][xdst[i]]) = p;
            *reinterpret_cast<uint2*>(&lds[to][1][xdst[i]]) = q;
            *reinterpret_cast<uint2*>(&lds[to][2][xdst[i]]) = t;
        }
    };
    floatx4_t acc[FT][RT], low[FT][RT], group[FT][RT];
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int a = 0; a < RT; ++a) {
            acc[f][a] = low[f][a] = group[f][a] = none;
            totals[f * RT + a][tid] = none;
        }
    auto write = [&](float* y, int f, int a, floatx4_t v, bool with_bias) {
        const int m = m0 + 16 * a + r16;
        if (m >= M) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + 16 * f + 4 * g + i;
            if (n < N) y[(size_t)m * N + n] = with_bias ? v[i] + bias[n] : v[i];
        }
    };
    Parts wp[FT], ahead[FT];                  // the weights' parts of the half stage at hand, and of the next one
    auto take_apart = [&](Parts (&to)[FT], int k0, int h) {
#pragma unroll
        for (int f = 0; f < FT; ++f) {
            const bool in0 = !TAIL || k0 + 32 * h + 8 * g < k_end, in1 = !TAIL || k0 + 32 * h + 8 * g + 4 < k_end;
            to[f] = split8(in0 ? wv[f][2 * h] : none, in1 ? wv[f][2 * h + 1] : none);
        }
    };
    load_x(k_begin, 0);
    load_x(k_begin, 1);
    load_w(k_begin, 0);
    load_w(k_begin, 1);
    put_x(k_begin, 0, 0);
    put_x(k_begin, 0, 1);
    load_x(k_begin + 64, 0);
    load_x(k_begin + 64, 1);
    take_apart(wp, k_begin, 0);
    load_w(k_begin + 64, 0);
    __syncthreads();
    for (int c0 = k_begin; c0 < k_end; c0 += G_CHUNK) {
#pragma unroll
        for (int stage = 0; stage < 2; ++stage) {
            const int k0 = c0 + 64 * stage;
            if (!TAIL && stage == 1 && k0 >= k_end) break;          // (K ends with half a chunk)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // the next half's weights and half of the next stage's x are taken apart beside this half's products
                take_apart(ahead, k0 + 64 * h, 1 - h);
                load_w(k0 + 64 + 64 * h, 1 - h);
                put_x(k0 + 64, stage ^ 1, h);                       // (what that part of LDS held has been multiplied: a barrier lies between)
                load_x(k0 + 128, h);
                Parts xp[RT];
#pragma unroll
                for (int a = 0; a < RT; ++a) {
                    const int row = 16 * a + r16, at = row * 128 + (((4 * h + g) ^ ((row >> 1) & 7)) * 16);
                    xp[a] = {*reinterpret_cast<const bf16x8_t*>(&lds[stage][0][at]), *reinterpret_cast<const bf16x8_t*>(&lds[stage][1][at]),
                             *reinterpret_cast<const bf16x8_t*>(&lds[stage][2][at])};
#pragma unroll
                    for (int f = 0; f < FT; ++f) multiply32(acc[f][a], low[f][a], wp[f], xp[a]);
                }
                // a product's instruction takes the matrix cores 16 cycles and the wave 4: three others beside each
                __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
                for (int a = 0; a < RT; ++a) {
#pragma unroll
                    for (int i = 0; i < 8 * FT; ++i) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                }
#pragma unroll
                for (int f = 0; f < FT; ++f) wp[f] = ahead[f];
            }
            __syncthreads();
        }
        const int done = c0 + G_CHUNK;
        const bool end = done % G_GROUP == 0 || done >= k_end;
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int a = 0; a < RT; ++a) {
                group[f][a] += acc[f][a] + low[f][a];
                acc[f][a] = low[f][a] = none;
            }
        if (!end) continue;
        bool all_stand = true;
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int a = 0; a < RT; ++a) all_stand = all_stand && stand(group[f][a]);
        uint32_t again = 0;                             // which of the lane's sums of the group do not stand
        static_assert(FT * RT * 4 <= 32, "a bit each");
        if (__any(!all_stand)) {
#pragma unroll
            for (int f = 0; f < FT; ++f)
#pragma unroll
                for (int a = 0; a < RT; ++a)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!stands(group[f][a][i])) { again |= 1u << (4 * (f * RT + a) + i); group[f][a][i] = 0.f; }
        }
#pragma unroll
        for (int f = 0; f < FT; ++f)
#pragma unroll
            for (int a = 0; a < RT; ++a) {
                if (shared_out) write(out + (size_t)(c0 / G_GROUP) * M * N, f, a, group[f][a], false);
                else totals[f * RT + a][tid] += group[f][a];
                group[f][a] = none;
            }
        if (__any(again != 0)) {
            const int g0 = c0 / G_GROUP * G_GROUP;
#pragma unroll 1
            for (int j = 0; j < FT * RT; ++j) {
                const uint32_t which = again >> (4 * j) & 15;
                if (!__any(which != 0)) continue;
                const int m = m0 + 16 * (j % RT) + r16, n = n0 + 16 * (j / RT);
                const floatx4_t plain = plain_group(x + (size_t)min(m, M - 1) * K, w + (size_t)min(n + r16, N - 1) * K, g0, min(done, k_end), 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (!(which >> i & 1)) continue;
                    if (!shared_out) totals[j][tid][i] += plain[i];
                    else if (m < M && n + 4 * g + i < N) out[(size_t)(c0 / G_GROUP) * M * N + (size_t)m * N + n + 4 * g + i] = plain[i];
                }
            }
        }
    }
    if (shared_out) return;
#pragma unroll
    for (int f = 0; f < FT; ++f)
#pragma unroll
        for (int a = 0; a < RT; ++a) write(out, f, a, totals[f * RT + a][tid], bias != nullptr);
}

// The groups' sums in their order.  Eight loads under way together: one after the other they were most of the time (19 groups of one row of 3584 5.6 -> 4.7 us).
__global__ void gemm_few_rows_sum_kernel(const float* __restrict__ group_sums, const float* __restrict__ bias,
                                         float* __restrict__ y, int n_groups, int M, int N) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * N) return;
    const size_t group = (size_t)M * N;
    const float* from = group_sums + i;
    float total = 0.f;
    int g = 0;
    for (; g + 8 <= n_groups; g += 8, from += 8 * group) {
        float sums[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) sums[u] = from[u * group];
#pragma unroll
        for (int u = 0; u < 8; ++u) total += sums[u];
    }
    // (what is left likewise: the last group again where there are fewer, not added)
    if (g < n_groups) {
        float sums[7];
#pragma unroll
        for (int u = 0; u < 7; ++u) sums[u] = from[min(u, n_groups - 1 - g) * group];
#pragma unroll
        for (int u = 0; u < 7; ++u) total = g + u < n_groups ? total + sums[u] : total;
    }
    if (bias) total += bias[i % N];
    y[i] = total;
}

static bool f32_case(int x_dtype, int w_dtype, const void* bias, int bias_dtype, int y_dtype, int K, const void* x, const void* w) {
    return K % 4 == 0 && x_dtype == TQK_F32 && w_dtype == TQK_F32 && y_dtype == TQK_F32 && (!bias || bias_dtype == TQK_F32) &&
           ((((uintptr_t)x) | ((uintptr_t)w)) & 15) == 0;
}

// Whether a product's numbers are taken apart: where its weights are large (4 MB).  Below it launches are what a product costs, and the kernel for a small model's
// whole step (small_step.hip) has the order of the float32 instructions.
extern "C" int tqk_gemm_takes_apart(int N, int K) { return (long long)N * K >= 1 << 20; }

// Tiles of 16 rows and of 16 features a wave of gemm_split_kernel takes, in blocks of four waves side by side: the largest that leaves every unit a block.  us with 64 rows by 128
// features everywhere, and so: 300 rows of 1536 x 1536 43 and 27, 64 and 24 rows of 3584 x 3584 43 and 31, 40 and 26, 24 of 37888 x 3584 178 and 150 (32, 36, 35 and 185 with the float32 instructions).
// 9 to 16 rows go there with one tile of each where that gives every unit two blocks (of whole groups): 16 rows of 37888 x 3584, 3584 x 18944, 152064 x 3584, 4608 x 3584 and 3584 x 3584
// 127, 62, 504, 23.3 and 21.0, through the kernel for few rows 143, 74, 538, 21.3 and 18.6 (138, 74, 538, 21.5 and 18.3 with the float32 instructions); 9 rows of the first and third 116 and 463, 119 and 461 (115 and 458).
struct SplitTile { int rows, features; };
static SplitTile split_tile(int M, int N, int K) {
    const int groups = (K + G_GROUP - 1) / G_GROUP;
    auto blocks = [&](SplitTile t) { return (long long)((M + 16 * t.rows - 1) / (16 * t.rows)) * ((N + 64 * t.features - 1) / (64 * t.features)) * groups; };
    if (M <= 16) return M > 8 && blocks({1, 1}) >= 512 ? SplitTile{1, 1} : SplitTile{0, 0};
    const SplitTile all[] = {{4, 2}, {2, 2}, {4, 1}, {2, 1}};
    for (const SplitTile& t : all)
        if ((t.rows == 2 || M > 32) && blocks(t) >= 256) return t;
    return {2, 1};
}

// How long blocks of `per` groups each (a last one of what is left) take for all tiles, in a single group's time: a unit holds two blocks, 512 are under way together, and 256 that are left
// have a unit each and take 0.6 of the time.
static double split_rounds(long long tiles, int groups, int per) {
    auto busy = [](long long blocks) { return blocks == 0 ? 0. : blocks <= 256 ? 0.6 : 1.; };
    const int rest = groups % per;
    const long long whole = tiles * (groups / per) / 512, left = tiles * (groups / per) % 512;
    if (rest == 0) return per * (whole + busy(left));
    // (the last ones begin beside those that are left of the others, and behind them where these leave too few places)
    if (tiles <= 512 - left) return per * whole + rest * busy(left + tiles) + (per - rest) * busy(left);
    return per * (whole + 1) + rest * busy(tiles - (512 - left));
}

// Into how many shares the groups are dealt for M rows: few rows, one a group; more, so that there are about four blocks a compute
// unit (one: 280 blocks of 300 x 3584 leave most units idle while a few do a second block), no more than there are groups.
// Products that take numbers apart: what sets the time is how many rounds of 512 blocks there are (split_rounds).  Short blocks leave less of a last round over, so every group is a share of its own,
// unless blocks that walk all of K come out ahead of that with the sums that they need not write and add up, or two groups a block take no more rounds, which saves a start and
// an end, where there is a full round of blocks without a tile's last group.  Below 400 tiles blocks of all of K leave a fifth of the places idle and were never the best.  From 512 tiles on, where two blocks a unit need no
// scratch, groups' sums take 128 MB of it at most (1000 rows of 4608 x 3584: 74 MB, 290 -> 265 us), and from 768 on none.
// us with two blocks a unit and so, weights that no cache holds, medians of ten turns: 300 and 1000 rows of 3584 x 18944 423 -> 351 and 1138 -> 993, 1000 of 1536 x 8960 284 -> 227, 500 of 4608 x 3584
// 178 -> 152, 64 of 37888 x 3584 203 -> 178; a group a block and two: 100, 128 and 256 rows of 3584 x 18944 180 -> 160, 183 -> 167 and 302 -> 293, 160 of 4096 x 11008 172 -> 161, 200 of 7168 x 5120
// 166 -> 161, 1000 of 1536 x 8960 234 -> 227.  317 sizes of 19 weights, 17 to 2048 rows: 1.003 of the best number's time (at most 1.11, 80 rows of 7168 x 5120), two blocks a
// unit 1.025 (at most 1.29).
extern "C" int tqk_gemm_f32_shares(int M, int N, int K) {
    const int groups = (K + G_GROUP - 1) / G_GROUP;
    if (M <= 16) return groups;
    if (tqk_gemm_takes_apart(N, K)) {
        const SplitTile t = split_tile(M, N, K);
        const long long tiles = (long long)((M + 16 * t.rows - 1) / (16 * t.rows)) * ((N + 64 * t.features - 1) / (64 * t.features));
        if (tiles >= 768 || (tiles >= 512 && (long long)groups * M * N * 4 > 128 << 20)) return 1;
        if (tiles < 400) return tiles * (groups - 1) >= 512 && split_rounds(tiles, groups, 2) <= split_rounds(tiles, groups, 1) ? (groups + 1) / 2 : groups;
        const double us = 8 + 39. * t.rows * t.features / 8;             // of a round of single groups
        return split_rounds(tiles, 1, 1) * (groups + 0.1) * us <= split_rounds(tiles, groups, 1) * 1.1 * us + 5 + (double)groups * M * N * 8 / 4.0e6 ? 1 : groups;
    }
    const long long tiles = (long long)((M + GT - 1) / GT) * ((N + GT - 1) / GT);
    const int want = (int)(tiles >= 1024 ? 1 : (1024 + tiles - 1) / tiles), per = (groups + want - 1) / want;
    return (groups + per - 1) / per;
}

/* Bytes of device scratch tqk_gemm wants for these sizes and dtypes (0: none). */
extern "C" size_t tqk_gemm_scratch_bytes(int x_dtype, int w_dtype, int bias_dtype, int y_dtype, int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || !f32_case(x_dtype, w_dtype, nullptr, bias_dtype, y_dtype, K, nullptr, nullptr) || tqk_gemm_f32_shares(M, N, K) == 1) return 0;
    return (size_t)((K + G_GROUP - 1) / G_GROUP) * M * N * sizeof(float);
}

template <typename TX, typename TW, typename TB>
static int launch_y(const void* x, const void* w, const void* bias, void* y, int y_dtype,
                    int M, int N, int K, hipStream_t s) {
    dim3 grid((N + GT - 1) / GT, (M + GT - 1) / GT);
    if (y_dtype == TQK_F32)
        gemm_generic_kernel<TX, TW, TB, float><<<grid, 256, 0, s>>>((const TX*)x, (const TW*)w, (const TB*)bias, (float*)y, M, N, K);
    else if (y_dtype == TQK_BF16)
        gemm_generic_kernel<TX, TW, TB, bf16_t><<<grid, 256, 0, s>>>((const TX*)x, (const TW*)w, (const TB*)bias, (bf16_t*)y, M, N, K);
    else
        return tqk_fail("tqk_gemm: unknown output dtype %d", y_dtype);
    return tqk_check_launch("tqk_gemm");
}

static int gemm(const void* x, int x_dtype, const void* w, int w_dtype, const void* bias, int bias_dtype, void* y, int y_dtype, int M, int N, int K, void* scratch, bool once, void* stream) {
    TQK_REQUIRE(x && w && y, "tqk_gemm: null pointer");
    TQK_REQUIRE(M >= 0 && N > 0 && K > 0, "tqk_gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    TQK_REQUIRE((M + GT - 1) / GT <= 65535, "tqk_gemm: M=%d is more than the grid takes", M);
    if (M == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (f32_case(x_dtype, w_dtype, bias, bias_dtype, y_dtype, K, x, w)) {
        const int groups = (K + G_GROUP - 1) / G_GROUP, shares = scratch ? tqk_gemm_f32_shares(M, N, K) : 1;       // (without scratch one block walks all of K)
        TQK_REQUIRE(groups <= 65535, "tqk_gemm: K=%d is more than the grid takes", K);
        const float *xf = (const float*)x, *wf = (const float*)w, *bf = (const float*)bias;
        float* out = shares > 1 ? (float*)scratch : (float*)y;
        const bool apart = tqk_gemm_takes_apart(N, K);
        const int per = (groups + shares - 1) / shares;
        SplitTile t = apart ? split_tile(M, N, K) : SplitTile{0, 0};
        if (apart && t.rows == 0 && shares < groups) t = {1, 1};             // (few rows without scratch: one block walks all of K)
        if (t.rows == 0 && M <= 16 && shares == groups) {
            const dim3 grid((N + 15) / 16, groups);
            if (!apart) gemm_few_rows_kernel<<<grid, TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K);
            else {
#define LAUNCH_ONCE(ROWS, ONCE) do { if (K % 64) gemm_few_rows_apart_kernel<true, ROWS, ONCE><<<grid, TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K); \
        else gemm_few_rows_apart_kernel<false, ROWS, ONCE><<<grid, TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K); } while (0)
#define LAUNCH(ROWS) do { if (once) LAUNCH_ONCE(ROWS, true); else LAUNCH_ONCE(ROWS, false); } while (0)
                if (M <= 4) LAUNCH(4);
                else if (M <= 8) LAUNCH(8);
                else LAUNCH(16);
#undef LAUNCH
#undef LAUNCH_ONCE
            }
        } else if (apart) {
            const dim3 grid(((N + 64 * t.features - 1) / (64 * t.features)) * ((M + 16 * t.rows - 1) / (16 * t.rows)), shares);
#define LAUNCH(RT, FT) do { if (K % 64) gemm_split_kernel<RT, FT, true><<<grid, GS_WAVES * TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K, per); \
        else gemm_split_kernel<RT, FT, false><<<grid, GS_WAVES * TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K, per); } while (0)
            if (t.rows == 1) LAUNCH(1, 1);
            else if (t.rows == 4) { if (t.features == 2) LAUNCH(4, 2); else LAUNCH(4, 1); }
            else if (t.features == 2) LAUNCH(2, 2);
            else LAUNCH(2, 1);
#undef LAUNCH
        } else gemm_f32_kernel<<<dim3(((N + GT - 1) / GT) * ((M + GT - 1) / GT), shares), 256, 0, s>>>(xf, wf, bf, out, M, N, K, (groups + shares - 1) / shares);
        if (tqk_check_launch("tqk_gemm float32")) return -1;
        if (shares == 1) return 0;
        const size_t total = (size_t)M * N;
        gemm_few_rows_sum_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>((const float*)scratch, bf, (float*)y, groups, M, N);
        return tqk_check_launch("tqk_gemm sum");
    }
    if (!bias) bias_dtype = w_dtype;
    const int code = x_dtype * 4 + w_dtype * 2 + bias_dtype;
    switch (code) {
        case 0: return launch_y<float, float, float>(x, w, bias, y, y_dtype, M, N, K, s);
        case 1: return launch_y<float, float, bf16_t>(x, w, bias, y, y_dtype, M, N, K, s);
        case 2: return launch_y<float, bf16_t, float>(x, w, bias, y, y_dtype, M, N, K, s);
        case 3: return launch_y<float, bf16_t, bf16_t>(x, w, bias, y, y_dtype, M, N, K, s);
        case 4: return launch_y<bf16_t, float, float>(x, w, bias, y, y_dtype, M, N, K, s);
        case 5: return launch_y<bf16_t, float, bf16_t>(x, w, bias, y, y_dtype, M, N, K, s);
        case 6: return launch_y<bf16_t, bf16_t, float>(x, w, bias, y, y_dtype, M, N, K, s);
        case 7: return launch_y<bf16_t, bf16_t, bf16_t>(x, w, bias, y, y_dtype, M, N, K, s);
    }
    return tqk_fail("tqk_gemm: unknown dtypes x=%d w=%d bias=%d", x_dtype, w_dtype, bias_dtype);
}

extern "C" int tqk_gemm(const void* x, int x_dtype, const void* w, int w_dtype, const void* bias,
                        int bias_dtype, void* y, int y_dtype, int M, int N, int K, void* scratch, void* stream) {
    return gemm(x, x_dtype, w, w_dtype, bias, bias_dtype, y, y_dtype, M, N, K, scratch, false, stream);
}

extern "C" int tqk_gemm_once(const void* x, int x_dtype, const void* w, int w_dtype, const void* bias,
                             int bias_dtype, void* y, int y_dtype, int M, int N, int K, void* scratch, void* stream) {
    return gemm(x, x_dtype, w, w_dtype, bias, bias_dtype, y, y_dtype, M, N, K, scratch, true, stream);
}
