// y[M,N] = x[M,K] w[N,K]^T (+ bias): the plain product of the float32 path, and of
// any dtype mix the fast kernels do not take.  The reference's linear layers are
// candle matmuls (src/models/turbo_generic.rs:68-91, 779-781).
//
// float32 throughout, K a multiple of 4 and operands at 16 bytes (every product of the float32 path of a usual model):
// v_mfma_f32_16x16x4_f32, whose products and sums are float32 ones (no reduced-precision mode of the matrix cores
// is used anywhere here).  Everything else: LDS-tiled, 64x64 outputs per block, 4x4 per thread, float32 FMA.
//
// The order of summation is fixed, and is the same for all numbers of rows, so that a result does
// not depend on M, on where a row stands in the batch, or on which kernel computed it: k is
// cut into chunks of 128 and groups of 8 chunks; a chunk is summed from zero, a group is the sum of its chunks in order,
// the result the sum of the groups in order (and then the bias).  Within a chunk the FMA kernel goes by increasing k; the
// matrix-core kernels take 16 k at a time, four instructions of which number i adds the k with k % 4 == i to what the ones
// before it left (a lane then reads its operands of all four as 16 contiguous bytes), with the same operands in the same
// registers whichever kernel it is.
//
// For up to 16 rows of x (decoding in the 32-bit path) the weights are the whole cost: a wave takes 16 output features and one
// group of k and streams their weights from memory into the operands' registers, 16 loads of a KB under way; groups beyond
// the first meet in a second kernel.  More rows: a block of four waves takes 64 rows by 64 features through LDS; where that gives
// few blocks they are also dealt out along the groups.  Measured at the 7B layers' sizes: see the kernels.
#include "common.h"
#include "tq_kernels.h"

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

// 16 k more: lane l holds, of both operands, row l % 16 and the four k at 4 (l / 16); of the sums row (of x) l % 16 and the
// features 4 (l / 16) .. + 3.
__device__ __forceinline__ void multiply16(floatx4_t& acc, const floatx4_t& w, const floatx4_t& x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i], x[i], acc, 0, 0, 0);
}

// Up to 16 rows of x: a wave per (16 output features, one group of k).  With one group the result is finished here.
// Bound by the weights, whose rows it takes 64 bytes at a time out of 16 of them: gate+up of the 7B shape (543 MB), one row, 124 us
// (4.4 TB/s; 141 with the loads marked read-once, since the other half of a line is the next load's).  With a feature a lane, each
// reading its own row, it was 131 us for one row, and every further row cost as much again in multiplications.
__global__ __launch_bounds__(TQK_WAVE)
void gemm_few_rows_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                          int M, int N, int K) {
    const int lane = threadIdx.x, r16 = lane % 16, k4 = 4 * (lane / 16);
    const int n0 = blockIdx.x * 16;
    const int k_begin = blockIdx.y * G_GROUP, k_end = min(K, k_begin + G_GROUP);
    const float* wrow = w + (size_t)min(n0 + r16, N - 1) * K;
    const float* xrow = x + (size_t)min(r16, M - 1) * K;          // rows past M repeat the last and are dropped
    floatx4_t group = {0.f, 0.f, 0.f, 0.f};
    constexpr int U = G_CHUNK / 16;                                     // a chunk's loads together, the next chunk's under way
    floatx4_t wv[2][U], xv[2][U];
    auto load = [&](int c0, floatx4_t (&wq)[U], floatx4_t (&xq)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(c0 + 16 * u + k4, K - 4);                 // (past the end: loaded from inside the row, not used)
            wq[u] = *reinterpret_cast<const floatx4_t*>(wrow + k);
            xq[u] = *reinterpret_cast<const floatx4_t*>(xrow + k);
        }
    };
    // (one straight line from the first product to the sum: where a branch lay between, the compiler let the sum read the last
    // register of a product that was still under way)
    auto add = [&](int c0, floatx4_t (&wq)[U], floatx4_t (&xq)[U]) {
        if (c0 + G_CHUNK > k_end) {                                     // a last chunk that is not full: zeros add nothing
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c0 + 16 * u + k4 >= k_end) wq[u] = xq[u] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        }
        floatx4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u) multiply16(acc, wq[u], xq[u]);
        group += acc;
    };
    load(k_begin, wv[0], xv[0]);
    for (int c0 = k_begin; c0 < k_end; c0 += 2 * G_CHUNK) {
        load(c0 + G_CHUNK, wv[1], xv[1]);
        __builtin_amdgcn_sched_barrier(0);
        add(c0, wv[0], xv[0]);
        if (c0 + G_CHUNK >= k_end) break;
        load(c0 + 2 * G_CHUNK, wv[0], xv[0]);
        __builtin_amdgcn_sched_barrier(0);
        add(c0 + G_CHUNK, wv[1], xv[1]);
    }
    if (r16 >= M) return;
    const bool whole = gridDim.y == 1;
    float* dst = out + ((size_t)blockIdx.y * M + r16) * N;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + k4 + i;
        if (n < N) dst[n] = whole && bias ? group[i] + bias[n] : group[i];
    }
}

// More rows: 64 rows by 64 features a block, each of four waves 32 by 32.  Stages of 32 k go through registers into LDS, two in turn;
// a row's 128 bytes lie 144 apart, so that the 16 rows of an operand meet all banks.  blockIdx.z: the block's share of the
// groups; with more than one share every group's sums go to scratch on their own.  Bound by the matrix cores (157 TFLOP/s in
// float32): gate+up of the 7B shape at 300 rows 836 us = 97 TFLOP/s, and 2108 us through the FMA kernel above; down 287 and 1663.
#define GM_LINE 36              // floats from row to row in LDS
__global__ __launch_bounds__(256)
void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ out,
                     int M, int N, int K, int groups_per_share) {
    __shared__ __attribute__((aligned(16))) float lds[2][2][GT * GM_LINE];     // [stage][x, w]
    const int tid = threadIdx.x, lane = tid % TQK_WAVE, wave = tid / TQK_WAVE;
    const int r16 = lane % 16, k4 = 4 * (lane / 16);
    const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT, wm = wave / 2 * 32, wn = wave % 2 * 32;
    const int k_begin = blockIdx.z * groups_per_share * G_GROUP, k_end = min(K, k_begin + groups_per_share * G_GROUP);
    const bool shared_out = gridDim.z > 1;
    // what a thread brings in: of rows tid / 8 and 32 + tid / 8 of both tiles the four k at 4 (tid % 8) (rows past the end repeat the last)
    const int sr = tid / 8, sk = 4 * (tid % 8);
    const float* src[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        src[0][i] = x + (size_t)min(m0 + sr + 32 * i, M - 1) * K;
        src[1][i] = w + (size_t)min(n0 + sr + 32 * i, N - 1) * K;
    }
    floatx4_t ahead[2][2];
    auto load = [&](int k0) {
        const int k = min(k0 + sk, K - 4);          // past K: read from inside the row, zeros in its place
        const bool in = k0 + sk < K;
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                ahead[o][i] = *reinterpret_cast<const floatx4_t*>(src[o][i] + k);
                if (!in) ahead[o][i] = floatx4_t{0.f, 0.f, 0.f, 0.f};
            }
    };
    auto put = [&](int stage) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<floatx4_t*>(&lds[stage][o][(sr + 32 * i) * GM_LINE + sk]) = ahead[o][i];
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
    load(k_begin);
    put(0);
    __syncthreads();
    for (int c0 = k_begin; c0 < k_end; c0 += G_CHUNK) {
        // a chunk is four stages in a straight line (a last chunk that is not full meets zeros)
#pragma unroll
        for (int q = 0; q < G_CHUNK / 32; ++q) {
            const int stage = q % 2;
            load(c0 + 32 * (q + 1));
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

__global__ void gemm_few_rows_sum_kernel(const float* __restrict__ group_sums, const float* __restrict__ bias,
                                         float* __restrict__ y, int n_groups, int M, int N) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * N) return;
    float total = 0.f;
    for (int g = 0; g < n_groups; ++g) total += group_sums[(size_t)g * M * N + i];
    if (bias) total += bias[i % N];
    y[i] = total;
}

static bool f32_case(int x_dtype, int w_dtype, const void* bias, int bias_dtype, int y_dtype, int K, const void* x, const void* w) {
    return K % 4 == 0 && x_dtype == TQK_F32 && w_dtype == TQK_F32 && y_dtype == TQK_F32 && (!bias || bias_dtype == TQK_F32) &&
           ((((uintptr_t)x) | ((uintptr_t)w)) & 15) == 0;
}

// Into how many shares the groups are dealt for M rows: few rows, one a group; more, so that there are about four blocks a compute
// unit (one: 280 blocks of 300 x 3584 leave most units idle while a few do a second block), no more than there are groups.
static int f32_shares(int M, int N, int K) {
    const int groups = (K + G_GROUP - 1) / G_GROUP;
    if (M <= 16) return groups;
    const long long tiles = (long long)((M + GT - 1) / GT) * ((N + GT - 1) / GT);
    const int want = (int)(tiles >= 1024 ? 1 : (1024 + tiles - 1) / tiles), per = (groups + want - 1) / want;
    return (groups + per - 1) / per;
}

/* Bytes of device scratch tqk_gemm wants for these sizes and dtypes (0: none). */
extern "C" size_t tqk_gemm_scratch_bytes(int x_dtype, int w_dtype, int bias_dtype, int y_dtype, int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || !f32_case(x_dtype, w_dtype, nullptr, bias_dtype, y_dtype, K, nullptr, nullptr) || f32_shares(M, N, K) == 1) return 0;
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

extern "C" int tqk_gemm(const void* x, int x_dtype, const void* w, int w_dtype, const void* bias,
                        int bias_dtype, void* y, int y_dtype, int M, int N, int K, void* scratch, void* stream) {
    TQK_REQUIRE(x && w && y, "tqk_gemm: null pointer");
    TQK_REQUIRE(M >= 0 && N > 0 && K > 0, "tqk_gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    TQK_REQUIRE((M + GT - 1) / GT <= 65535, "tqk_gemm: M=%d is more than the grid takes", M);
    if (M == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (f32_case(x_dtype, w_dtype, bias, bias_dtype, y_dtype, K, x, w)) {
        const int groups = (K + G_GROUP - 1) / G_GROUP, shares = scratch ? f32_shares(M, N, K) : 1;       // (without scratch one block walks all of K)
        TQK_REQUIRE(groups <= 65535, "tqk_gemm: K=%d is more than the grid takes", K);
        const float *xf = (const float*)x, *wf = (const float*)w, *bf = (const float*)bias;
        float* out = shares > 1 ? (float*)scratch : (float*)y;
        if (M <= 16 && shares == groups) gemm_few_rows_kernel<<<dim3((N + 15) / 16, groups), TQK_WAVE, 0, s>>>(xf, wf, bf, out, M, N, K);
        else gemm_f32_kernel<<<dim3((N + GT - 1) / GT, (M + GT - 1) / GT, shares), 256, 0, s>>>(xf, wf, bf, out, M, N, K, (groups + shares - 1) / shares);
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
