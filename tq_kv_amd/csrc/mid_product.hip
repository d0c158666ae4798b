// y[M,N] = x[M,K] w[N,K]^T for 17 to 128 rows (decoding steps of larger batches, the wanted rows
// of many prompts): bfloat16 in, MFMA, float32 accumulation.  The reference runs these products
// as candle matmuls (src/models/turbo_generic.rs:68-91).  At these M the product is still bound
// by the weight bytes, which are streamed from HBM once, straight into registers, from the copy
// packed in the lanes' order ([tile of 16 rows][K/32][lane][8 values], see skinny_fused.hip).
//
// With this many rows x is no longer small beside a tile of weights: every wave needs all of it.
// So a block is 3 to 8 waves that walk K together, each with its own tiles of 16 output features,
// and one or two more waves that do nothing but bring x in, 64 k a stage, into a ring in LDS with
// loads that end there (a load takes eight whole lines of 128 bytes, of eight rows; the 16-byte pieces
// of a row are exchanged within it so that the reads of 16 rows of one k step meet all banks once).
// What binds such a block is what a compute unit brings in, weights and x together: with x in whole
// lines 38 GB/s at 64 rows and 53 at 256, in pieces of 64 bytes of 16 rows, which is what the matrix
// cores' order asks for, 33 and 36 (a bare loop of such loads).  The waves that multiply count no load
// but their weights', 8 steps of 32 k ahead, and meet once a stage.  Against a kernel whose waves
// brought x in between their weights, through registers, us at 32, 64 and 128 rows: gate+up of the 7B
// shape 47, 54, 69 -> 44, 46, 55; down 24.9, 28.7, 40.0 -> 24.2, 26.3, 34.4; q/k/v 9.7, 11.3, 17.2 ->
// 8.8, 10.1, 14.5; o 8.4, 10.2, 13.9 -> 7.6, 8.6, 11.6; gate+up of the 1.5B shape 17.9, 22.8, 29.3 ->
// 12.8, 15.6, 21.6.  Measured and left: 2, 4, 6 and 12 steps of weights ahead (within 1 %), 4 and 8 stages
// of x (the same), counts in LDS in place of the barrier, so that the waves may run apart (2 to 15 % slower).
//
// v_mfma_f32_16x16x32_bf16: A = a tile of w (16 features x 32 k), B = 32 k x 16 rows of x, so
// D[n][m] is a tile of y^T: lane l holds row m = l%16 of its 16-row group and the four features
// 4*(l/16) .. +3, which it stores as one 8- or 16-byte piece.
//
// Where N alone gives too few blocks for the chip, K is split over blockIdx.y: each split writes
// its sums to scratch [split][M][N] and a second kernel adds them in split order and finishes
// (store, or the gate: silu(gate) * up of src/models/turbo_generic.rs:105-111).  The number of
// splits depends on the product's shape alone, never on M, so a row's result does not depend on
// the batch it is in.
#include "common.h"
#include "tq_kernels.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

enum { MID_STORE = 0, MID_GATED = 1 };
#define MID_CHUNK 128           // K is cut into multiples of it
#define MID_MIN_WAVES 4          // waves per block that multiply: in pieces or groups (mid_plan)
#define MID_MAX_WAVES 8
#define MID_LEAST_WAVES 3        // where K is whole (mid_waves)
#define MID_MAX_ROWS 128

struct MidArgs {
    const bf16_t* x;            // [M, K]
    const bf16_t* w;            // packed [tiles][K/32][64][8]
    void* y;                    // store: [M, N]; gated: [M, N/2] bfloat16
    float* partial;             // [splits][M][N] when the grid has splits
    int M, N, K, k_per_split;   // k_per_split: a multiple of MID_CHUNK
    int gate;                   // gated: which gate (TQK_GATE_*), with its limit and alpha
    float gate_limit, gate_alpha;
    int activated;              // store: the gate's function of the product itself is applied (act_value)
    int group_rows;             // store: features n of group n / group_rows read the rows of x + group * x_group_stride (0: one group)
    long long x_group_stride;
};

__device__ __forceinline__ uint2 pack4_bf16(float a, float b, float c, float d) {
    return make_uint2((uint32_t)float_to_bf16_bits(a) | ((uint32_t)float_to_bf16_bits(b) << 16),
                      (uint32_t)float_to_bf16_bits(c) | ((uint32_t)float_to_bf16_bits(d) << 16));
}

struct Gate { int kind; float limit, alpha; int activated; };
__device__ __forceinline__ float gate_times_up(const Gate& gate, float gate_sum, float up_sum) {
    const float g = to_float(from_float<bf16_t>(gate_sum)), up = to_float(from_float<bf16_t>(up_sum));
    return gate_value(gate.kind, gate.limit, gate.alpha, g, up);
}
__device__ __forceinline__ float finished(const Gate& gate, float sum) {
    return gate.activated ? act_value(gate.kind, gate.limit, gate.alpha, to_float(from_float<bf16_t>(sum))) : sum;
}

// What a wave does with its sums: acc[t][mt] holds row mt * 16 + lane % 16 and the four features 4 * (lane / 16) .. + 3 of tile t.
template <int MT, int TN, int EPI, typename TY>
__device__ __forceinline__ void mid_write(const MidArgs& p, floatx4_t (&acc)[TN][MT], int n_lo0, int n_out, int row, int kgrp) {
    const int nb = 4 * kgrp;
    if (gridDim.y > 1) {
        const bool vec = p.N % 4 == 0 && n_out % 4 == 0;           // the up rows' sums start at n_out
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int m = mt * 16 + row;
                const int n = EPI == MID_GATED ? t * n_out + n_lo0 + nb : n_lo0 + 16 * t + nb;
                const int n_lim = EPI == MID_GATED ? t * n_out + n_out : p.N;
                if (m >= p.M) continue;
                float* dst = p.partial + ((size_t)blockIdx.y * p.M + m) * p.N + n;
                if (vec && n + 3 < n_lim) { *reinterpret_cast<floatx4_t*>(dst) = acc[t][mt]; continue; }
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < n_lim) dst[r] = acc[t][mt][r];
            }
        return;
    }
    if constexpr (EPI == MID_STORE) {
        TY* y = (TY*)p.y;
        const bool vec = p.N % 4 == 0;
#pragma unroll
        for (int t = 0; t < TN; ++t)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int m = mt * 16 + row;
                const int n = n_lo0 + 16 * t + nb;
                if (m >= p.M) continue;
                TY* dst = y + (size_t)m * p.N + n;
                if (p.activated) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[t][mt][r] = finished(Gate{p.gate, p.gate_limit, p.gate_alpha, 1}, acc[t][mt][r]);
                }
                if (vec && n + 3 < p.N) {
                    if constexpr (sizeof(TY) == 4) *reinterpret_cast<floatx4_t*>(dst) = acc[t][mt];
                    else *reinterpret_cast<uint2*>(dst) = pack4_bf16(acc[t][mt][0], acc[t][mt][1], acc[t][mt][2], acc[t][mt][3]);
                    continue;
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < p.N) dst[r] = from_float<TY>(acc[t][mt][r]);
            }
    } else {
        bf16_t* y = (bf16_t*)p.y;
        const bool vec = n_out % 4 == 0;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = mt * 16 + row;
            const int n = n_lo0 + nb;
            if (m >= p.M) continue;
            float o[4];
            // (which gate is asked once, not for every value)
            if (p.gate == TQK_GATE_SILU) {
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = gate_times_up(Gate{TQK_GATE_SILU, 0.f, 1.f, 0}, acc[0][mt][r], acc[TN - 1][mt][r]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) o[r] = gate_times_up(Gate{p.gate, p.gate_limit, p.gate_alpha, 0}, acc[0][mt][r], acc[TN - 1][mt][r]);
            }
            bf16_t* dst = y + (size_t)m * n_out + n;
            if (vec && n + 3 < n_out) { *reinterpret_cast<uint2*>(dst) = pack4_bf16(o[0], o[1], o[2], o[3]); continue; }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < n_out) dst[r] = from_float<bf16_t>(o[r]);
        }
    }
}

// Stages of 64 k of x in LDS: as many as a wave's count of loads under way reaches, six at most.
constexpr int mid_stages(int mt, int xw) { return 2 * mt / xw > 15 ? 5 : 6; }

// MT: groups of 16 rows of x (2: up to 32 rows, 4: up to 64, 8: up to 128).  TN: tiles of 16 features per wave (gated: the gate tile and its up
// tile).  XW waves of the block bring x in and do nothing else; WAVES others at most multiply.
template <int MT, int TN, int EPI, typename TY, int XW, int WAVES>
__global__ __launch_bounds__((WAVES + XW) * TQK_WAVE)
void mid_product_kernel(const MidArgs p) {
    constexpr int NS = mid_stages(MT, XW), STAGE = MT * 2048, DMA = 2 * MT / XW;
    __shared__ __attribute__((aligned(1024))) char ring[NS * STAGE];        // [NS][rows][8 pieces of 16 bytes]
    const int lane = threadIdx.x % TQK_WAVE, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / TQK_WAVE);
    const int n_waves = blockDim.x / TQK_WAVE - XW;
    const int K = p.K;
    const int k_begin = blockIdx.y * p.k_per_split, n_step = min(K - k_begin, p.k_per_split) / 32, n_stage = (n_step + 1) / 2;
    if (wv >= n_waves) {
        const bf16_t* px = p.x + k_begin;
        if (EPI == MID_STORE && p.group_rows) px += (size_t)((int)blockIdx.x * n_waves * TN * 16 / p.group_rows) * p.x_group_stride;
        const __amdgpu_buffer_rsrc_t x_mem = __builtin_amdgcn_make_buffer_rsrc((void*)px, 0, 0x7fffffff, 0x00020000);
        const int xw = wv - n_waves;
        uint32_t x_at[DMA];
#pragma unroll
        for (int i = 0; i < DMA; ++i) {
            const int j = i * XW + xw;
            x_at[i] = (uint32_t)min(j * 8 + lane / 8, p.M - 1) * (uint32_t)(K * 2) + ((lane % 8) ^ ((4 * (j % 2) + lane / 16) % 8)) * 16;
        }
        auto load = [&](int stage) {
            char* to = ring + (stage % NS) * STAGE + xw * 1024;
            if (2 * stage + 1 == n_step) {          // half a stage is left: the other half's pieces are the same again, and not read
#pragma unroll
                for (int i = 0; i < DMA; ++i) x_at[i] -= (((lane % 8) ^ ((4 * ((i * XW + xw) % 2) + lane / 16) % 8)) & 4) * 16;
            }
#pragma unroll
            for (int i = 0; i < DMA; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(x_mem, (lds_ptr_t)(to + i * XW * 1024), 16, (int)x_at[i], stage * 128, 0, 0);
        };
        for (int s = 0; s < NS - 1 && s < n_stage; ++s) load(s);
        for (int s = 0; s < n_stage; ++s) {
            constexpr int left = (NS - 2) * DMA;
            static_assert(left < 64, "");
            if (s + NS - 1 <= n_stage) __builtin_amdgcn_s_waitcnt(0x0f70 | (left & 15) | ((left >> 4) << 14));
            else __builtin_amdgcn_s_waitcnt(0x0f70);
            __builtin_amdgcn_s_barrier();
            if (s + NS - 1 < n_stage) load(s + NS - 1);         // into the place of stage s - 1, which everybody has read
        }
        return;
    }

    const int row = lane % 16, kgrp = lane / 16;
    const int n_out = EPI == MID_GATED ? p.N / 2 : p.N;
    const int part_tiles = (n_out + 15) / 16;
    const int tile0 = (blockIdx.x * n_waves + wv) * (EPI == MID_GATED ? 1 : TN);
    const int n_lo0 = tile0 * 16;
    const size_t tile_size = (size_t)(K / 32) * 512;
    const bf16_t* wtile[TN];
#pragma unroll
    for (int t = 0; t < TN; ++t) {
        const int tile = EPI == MID_GATED ? t * part_tiles + min(tile0, part_tiles - 1) : min(tile0 + t, part_tiles - 1);
        wtile[t] = p.w + (size_t)tile * tile_size + (size_t)(k_begin / 32) * 512 + lane * 8;
    }
    floatx4_t acc[TN][MT];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    constexpr int WD = TN > 2 ? 4 : 8;              // steps of 32 k of weights under way
    bf16x8_t w[WD][TN];
    auto load_w = [&](int step, int t) {
        return __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(wtile[t] + (size_t)min(step, n_step - 1) * 512));      // read once
    };
#pragma unroll
    for (int s = 0; s < WD; ++s)
#pragma unroll
        for (int t = 0; t < TN; ++t) w[s][t] = load_w(s, t);

    const int at0 = row * 128 + (kgrp ^ (row / 2)) * 16, at1 = at0 ^ 64;
    const char* from = ring;
    auto stage = [&](int s, int h, bool last) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");              // what LDS holds has changed
        __builtin_amdgcn_sched_barrier(0);
        // (both steps' operands are asked for together where the registers hold them)
        constexpr bool BOTH = MT * TN < 16;
        bf16x8_t x[2][MT];
        auto read = [&](int u) __attribute__((always_inline)) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) x[u][mt] = *reinterpret_cast<const bf16x8_t*>(from + (u ? at1 : at0) + mt * 2048);
        };
        if (BOTH) {
            read(0);
            read(1);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (!BOTH) read(u);
            if (last && u == 1 && 2 * s + 1 == n_step) {         // K ends in the middle of the stage
                const bf16x8_t none = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) x[u][mt] = none;
#pragma unroll
                for (int t = 0; t < TN; ++t) w[2 * h + u][t] = none;
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int t = 0; t < TN; ++t) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 * h + u][t], x[u][mt], acc[t][mt], 0, 0, 0);
            if (!last) {
#pragma unroll
                for (int t = 0; t < TN; ++t) w[2 * h + u][t] = load_w(2 * s + u + WD, t);
            }
        }
        from = from == ring + (NS - 1) * STAGE ? ring : from + STAGE;
    };
    constexpr int H = WD / 2;
    int s = 0;
    for (; s + H <= n_step / 2; s += H) {
#pragma unroll
        for (int h = 0; h < H; ++h) stage(s + h, h, false);
    }
#pragma unroll
    for (int h = 0; h < H; ++h)
        if (s + h < n_stage) stage(s + h, h, true);
    mid_write<MT, TN, EPI, TY>(p, acc, n_lo0, n_out, row, kgrp);
}

// Adds the splits' sums in split order and finishes as the product kernel does without splits.
template <int EPI, typename TY>
__global__ void mid_finish_kernel(const float* __restrict__ partial, void* __restrict__ yv, int splits, int M, int N, Gate gate) {
    const int n_out = EPI == MID_GATED ? N / 2 : N;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * n_out) return;
    const int m = (int)(i / n_out), n = (int)(i % n_out);
    float a = 0.f, b = 0.f;
    for (int s = 0; s < splits; ++s) {
        const float* src = partial + ((size_t)s * M + m) * N;
        a += src[n];
        if (EPI == MID_GATED) b += src[n_out + n];
    }
    if (EPI == MID_GATED) ((bf16_t*)yv)[i] = from_float<bf16_t>(gate_times_up(gate, a, b));
    else ((TY*)yv)[i] = from_float<TY>(finished(gate, a));
}

// How a product is cut: pieces of K, from N and K alone (the order of a row's sums goes by them, and must not depend on the batch); and of products
// in pieces or in groups the tiles per wave and waves per block, too (mid_waves has those of the others).
struct MidPlan { int tn, waves, blocks, splits, k_per_split; };
#define MID_UNITS 256

static MidPlan mid_plan(int N, int K, bool gated) {
    MidPlan plan;
    const int n_out = gated ? N / 2 : N;
    const int tiles = (n_out + 15) / 16;
    // two tiles per wave halve the reads of x from LDS, but also the waves: only where many are left
    plan.tn = gated ? 2 : (tiles >= 8192 ? 2 : 1);
    const int items = gated ? tiles : (tiles + plan.tn - 1) / plan.tn;        // what a wave takes
    const int chunks = (K + MID_CHUNK - 1) / MID_CHUNK;
    plan.waves = MID_MAX_WAVES;
    plan.splits = 1;
    if (items >= MID_UNITS * MID_MIN_WAVES) {
        // enough for every unit.  Groups: the waves per block and rounds of blocks that leave the fewest units idle
        double best = 0.0;
        for (int rounds = 1; rounds <= 8; ++rounds) {
            int waves = (items + MID_UNITS * rounds - 1) / (MID_UNITS * rounds);
            if (waves > MID_MAX_WAVES) continue;
            if (waves < MID_MIN_WAVES) waves = MID_MIN_WAVES;
            const double used = (double)items / ((double)MID_UNITS * rounds * waves);
            if (used > best + 0.02) { best = used; plan.waves = waves; }
        }
        plan.blocks = (items + plan.waves - 1) / plan.waves;
    } else {
        // Few features: K cut so that there is about a block per unit, no piece shorter than 4 chunks; and as many
        // waves per block (8 down to 4) as leave the fewest units without a block.  A unit alone pulls a 256th of what
        // the memory gives, so a product that covers a fifth of the units runs at a fifth of the rate whatever its
        // waves do (a width of 1536 and K of 1536: 36 blocks of 8 waves, 72 of 4).
        double best = 0.0;
        for (int waves = MID_MAX_WAVES; waves >= MID_MIN_WAVES; --waves) {
            const int blocks = (items + waves - 1) / waves;
            int splits = MID_UNITS / blocks;
            if (splits > chunks / 4) splits = chunks / 4;
            if (splits < 1) splits = 1;
            const int total = blocks * splits, rounds = (total + MID_UNITS - 1) / MID_UNITS;
            const double covered = (double)total / ((double)rounds * MID_UNITS);
            if (waves == MID_MAX_WAVES || covered > best + 0.02) { best = covered; plan.waves = waves; plan.blocks = blocks; plan.splits = splits; }
        }
    }
    if (gated && plan.splits > 1) {
        // A gated product in pieces needs a kernel of its own to add them up and apply the gate (4 to 5 us); where the
        // blocks of the whole K already cover half the units, that costs more than the pieces gain.  The line is the one of a kernel whose
        // units pulled 34 GB/s, in blocks of four waves and more, of 6.5 TB/s that the memory gives, and stays where it was, since results' low bits go by
        // it.  Units pull about 55 GB/s today, x counted, and blocks may have three waves, so whole products are better over more sizes than it
        // says.  us whole and in pieces, 20, 64 and 128 rows, N of both parts: it takes 17920 x 1536 whole, 11.7, 14.3, 20.1 and 16.7, 23.6, 29.0; 22016 x
        // 4096 whole, 29.6, 32.8, 42.2 and 34.0, 39.2, 44.4; 4096 x 4096 in pieces, 19.2, 24.8, 34.6 and 15.6, 17.6, 21.4; 9728 x 8192 in pieces, 40.2, 50.0,
        // 67.4 and 32.3, 36.7, 42.3; but also 12288 x 2048 in pieces, 12.6, 15.8, 22.1 and 15.5, 20.9, 27.3, and 16384 x 4096, 24.3, 29.3, 39.0 and 37.5,
        // 43.2, 49.5.
        const double bytes = 2.0 * (double)N * (double)K;
        auto time_us = [&](int blocks) { return 4.0 + bytes / (1e6 * (blocks * 0.034 < 6.5 ? blocks * 0.034 : 6.5)); };
        double whole = 1e30;
        for (int waves = MID_MAX_WAVES; waves >= MID_MIN_WAVES; --waves) {
            const int blocks = (items + waves - 1) / waves;
            if (blocks <= MID_UNITS && time_us(blocks) < whole - 0.1) whole = time_us(blocks);
        }
        if (whole < time_us(plan.blocks * plan.splits) + 4.6) plan.splits = 1;
    }
    const int per = (chunks + plan.splits - 1) / plan.splits;
    plan.splits = (chunks + per - 1) / per;             // no empty piece
    plan.k_per_split = per * MID_CHUNK;
    return plan;
}

/* Into how many pieces the product's K is cut (1: none, no scratch is needed). */
extern "C" int tqk_mid_max_rows(void) { return MID_MAX_ROWS; }

extern "C" int tqk_mid_splits(int N, int K, int gated) {
    if (N <= 0 || K <= 0) return 1;
    return mid_plan(N, K, gated != 0).splits;
}

static size_t mid_scratch_bytes(int M, int N, int K, bool gated) {
    const int splits = tqk_mid_splits(N, K, gated);
    return splits > 1 && M > 0 ? (size_t)splits * M * N * sizeof(float) : 0;
}

template <int EPI, typename TY>
static int finish_mid(const MidArgs& a, const MidPlan& plan, bool finish, hipStream_t s) {
    if (tqk_check_launch("tqk_mid product")) return -1;
    if (plan.splits > 1 && finish) {
        const size_t total = (size_t)a.M * (EPI == MID_GATED ? a.N / 2 : a.N);
        mid_finish_kernel<EPI, TY><<<(unsigned)((total + 255) / 256), 256, 0, s>>>(a.partial, a.y, plan.splits, a.M, a.N, Gate{a.gate, a.gate_limit, a.gate_alpha, a.activated});
        return tqk_check_launch("tqk_mid finish");
    }
    return 0;
}

template <int MT, int TN, int EPI, typename TY, int WAVES>
static int launch_mid(const MidArgs& a, const MidPlan& plan, bool finish, hipStream_t s) {
    constexpr int XW = MT > 4 && WAVES == MID_MAX_WAVES ? 2 : 1;
    mid_product_kernel<MT, TN, EPI, TY, XW, WAVES><<<dim3(plan.blocks, plan.splits), (plan.waves + XW) * TQK_WAVE, 0, s>>>(a);
    return finish_mid<EPI, TY>(a, plan, finish, s);
}

// The most tiles a wave takes of a wide product, and with how many waves beside it at most: as many as the registers hold with x's rows.
template <int MT> struct MidWide { enum { tn = MT == 2 ? 5 : MT == 4 ? 6 : 3, waves = MT == 2 ? 8 : 7 }; };

// Tiles per wave and waves per block of a product whose K is whole (a sum's order does not depend on them).  A block brings in all of x beside
// its own weights, so what the busiest unit brings in is rounds of blocks times (tiles of a block + groups of rows of x), each 32 K bytes.
// us at 32, 64 and 128 rows, against two tiles a wave and as many waves as leave the fewest units idle: the 7B head 194, 231, 236 -> 172, 178,
// 219; the 1.5B one 89, 105, 115 -> 83, 91, 112; gate+up of the 1.5B shape (187 blocks of three waves for 140 of four) 15.7, 19.5, 25.9 ->
// 12.8, 15.6, 21.6.  Beyond that (us, weights that no cache holds):
//  - A round more than one costs its start and end, two tiles' worth: 128256 features, K of 4096, 20, 32 and 64 rows 183, 191 and 199 us in two rounds
//    of two tiles by eight waves, 157, 159 and 164 in one of five or six by six or seven.
//  - Blocks that lie a power of two from 256 KB on apart ask the same channels of memory at the same time, and up to 64 rows nothing hides it: K of 2048, 32000
//    features 28.5 and 30.3 us at 20 and 64 rows by eight waves (512 KB), 23.0 and 25.2 by five of two tiles; K of 1024, 64000 features 32.2 in 250
//    such blocks, 25.3 in 400 others.  At 128 rows 32.2 and 30.0, 38.9 and 36.0, K of 4096 and 32000 features 48.6 and 53.3: not counted there.
//  - More than two tiles a wave pay for themselves in long runs of K: 152064 features, 64 and 128 rows, K of 512 41.7 and 53.2 us with them, 37.8 and
//    48.4 without, K of 1024 64.5 and 77.8, 61.3 and 71.5; K of 2048 106.6 and 126.5, 110.5 and 121.8; K of 3584 174 and 212, 203 and 220.
static void mid_waves(MidPlan& plan, int N, int K, bool gated, int mt, int wide_tn, int wide_waves) {
    const int tiles = ((gated ? N / 2 : N) + 15) / 16;
    long long best = 1LL << 62;
    const int tns[3] = {1, 2, wide_tn};
    for (int i = 0; i < (gated ? 1 : K >= 1536 ? 3 : 2); ++i)
        for (int waves = MID_LEAST_WAVES; waves <= (i == 2 ? wide_waves : MID_MAX_WAVES); ++waves) {
            const int tn = gated ? 2 : tns[i];
            const int items = gated ? tiles : (tiles + tn - 1) / tn, blocks = (items + waves - 1) / waves, rounds = (blocks + MID_UNITS - 1) / MID_UNITS;
            const long long apart = (long long)waves * tn * K * 32;
            const bool same_channels = !gated && mt <= 4 && apart >= 256 * 1024 && (apart & (apart - 1)) == 0;
            const long long cost = (long long)rounds * (waves * tn * (same_channels ? 17 : 10) + mt * 10) + (gated ? 0 : (rounds - 1) * 20);
            if (cost < best) { best = cost; plan.tn = tn; plan.waves = waves; plan.blocks = blocks; }
        }
}

// The same for the rows that M falls among.
static void mid_waves(MidPlan& plan, int M, int N, int K, bool gated) {
    if (M > 64) mid_waves(plan, N, K, gated, 8, MidWide<8>::tn, MidWide<8>::waves);
    else if (M > 32) mid_waves(plan, N, K, gated, 4, MidWide<4>::tn, MidWide<4>::waves);
    else mid_waves(plan, N, K, gated, 2, MidWide<2>::tn, MidWide<2>::waves);
}

/* Which tile a product is given, for tests: 16 times the tiles a wave takes, plus the waves that multiply. */
extern "C" int tqk_mid_tile(int M, int N, int K, int gated) {
    if (M <= 0 || M > MID_MAX_ROWS || N <= 0 || K <= 0) return -1;
    MidPlan plan = mid_plan(N, K, gated != 0);
    if (plan.splits == 1) mid_waves(plan, M, N, K, gated != 0);
    return plan.tn * 16 + plan.waves;
}

template <int MT, int EPI, typename TY>
static int launch_rows(const MidArgs& a, MidPlan plan, bool finish, hipStream_t s) {
    constexpr int W = MID_MAX_WAVES;
    constexpr bool GATED = EPI == MID_GATED;
    using Wide = MidWide<MT>;
    if (plan.splits == 1 && !a.group_rows) mid_waves(plan, a.M, a.N, a.K, GATED);
    if (GATED || plan.tn == 2) return launch_mid<MT, 2, EPI, TY, W>(a, plan, finish, s);
    if constexpr (!GATED) {
        if (plan.tn == Wide::tn) return launch_mid<MT, Wide::tn, EPI, TY, Wide::waves>(a, plan, finish, s);
        return launch_mid<MT, 1, EPI, TY, W>(a, plan, finish, s);
    }
    return -1;
}

template <int EPI, typename TY>
static int launch_rows(const MidArgs& a, const MidPlan& plan, bool finish, hipStream_t s) {
    if (a.M > 64) return launch_rows<8, EPI, TY>(a, plan, finish, s);
    return a.M > 32 ? launch_rows<4, EPI, TY>(a, plan, finish, s) : launch_rows<2, EPI, TY>(a, plan, finish, s);
}

static int check_mid(const MidArgs& a, const void* scratch, bool gated, bool finish, const char* what) {
    TQK_REQUIRE(a.x && a.w, "%s: null pointer", what);
    TQK_REQUIRE(a.y || (!finish && tqk_mid_splits(a.N, a.K, gated) > 1), "%s: null output", what);
    TQK_REQUIRE(a.M >= 0 && a.M <= MID_MAX_ROWS, "%s: M=%d rows, this kernel takes at most %d", what, a.M, MID_MAX_ROWS);
    TQK_REQUIRE(a.N > 0 && a.K > 0 && a.K % 32 == 0, "%s: K=%d must be a positive multiple of 32 (N=%d)", what, a.K, a.N);
    TQK_REQUIRE(!gated || a.N % 2 == 0, "%s: odd N=%d", what, a.N);
    TQK_REQUIRE(((((uintptr_t)a.x) | ((uintptr_t)a.w) | ((uintptr_t)a.y) | ((uintptr_t)scratch)) & 15) == 0,
                "%s: x, w, y and scratch must be 16-byte aligned", what);
    TQK_REQUIRE(scratch || mid_scratch_bytes(a.M, a.N, a.K, gated) == 0, "%s: no scratch given", what);
    return 0;
}

/* y[M,N] = x w^T, M <= 128, w packed; scratch: float32 [tqk_mid_splits(N, K, 0)][M][N] where that
 * is more than 1.  finish == 0: with more than one piece the pieces' sums are left in scratch
 * (for tqk_add_rmsnorm_sums) and y is not written. */
extern "C" int tqk_mid_store(const void* x, const void* w_packed, void* y, int y_dtype, int M, int N, int K,
                             void* scratch, int finish, void* stream) {
    MidArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, y, (float*)scratch, M, N, K, 0, 0, 0.f, 1.f, 0, 0, 0};
    if (check_mid(a, scratch, false, finish != 0, "tqk_mid_store")) return -1;
    TQK_REQUIRE(y_dtype == TQK_F32 || y_dtype == TQK_BF16, "tqk_mid_store: unknown output dtype %d", y_dtype);
    if (M == 0) return 0;
    const MidPlan plan = mid_plan(N, K, false);
    a.k_per_split = plan.k_per_split;
    hipStream_t s = (hipStream_t)stream;
    return y_dtype == TQK_F32 ? launch_rows<MID_STORE, float>(a, plan, finish != 0, s)
                              : launch_rows<MID_STORE, bf16_t>(a, plan, finish != 0, s);
}

/* Several products in one launch: the rows n of w in groups of group_rows, group i taking x + i * x_group_stride; scratch as tqk_mid_store's for all
 * N rows.  Where tqk_mid_takes_groups (a block's features belong to one group). */
extern "C" int tqk_mid_takes_groups(int N, int K, int group_rows) {
    if (N <= 0 || K <= 0 || group_rows <= 0 || N % group_rows) return 0;
    const MidPlan plan = mid_plan(N, K, false);
    return group_rows % (plan.waves * plan.tn * 16) == 0;
}
extern "C" int tqk_mid_store_groups(const void* x, long long x_group_stride, int group_rows, const void* w_packed, void* y, int y_dtype, int M, int N, int K,
                                    void* scratch, void* stream) {
    MidArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, y, (float*)scratch, M, N, K, 0, 0, 0.f, 1.f, 0, group_rows, x_group_stride};
    if (check_mid(a, scratch, false, true, "tqk_mid_store_groups")) return -1;
    TQK_REQUIRE(y_dtype == TQK_F32 || y_dtype == TQK_BF16, "tqk_mid_store_groups: unknown output dtype %d", y_dtype);
    TQK_REQUIRE(tqk_mid_takes_groups(N, K, group_rows), "tqk_mid_store_groups: %d rows in groups of %d", N, group_rows);
    TQK_REQUIRE(x_group_stride % 8 == 0 && x_group_stride >= (long long)M * K, "tqk_mid_store_groups: the groups' rows of x overlap or are not aligned");
    if (M == 0) return 0;
    const MidPlan plan = mid_plan(N, K, false);
    a.k_per_split = plan.k_per_split;
    hipStream_t s = (hipStream_t)stream;
    return y_dtype == TQK_F32 ? launch_rows<MID_STORE, float>(a, plan, true, s) : launch_rows<MID_STORE, bf16_t>(a, plan, true, s);
}

/* y[M,N] = f(x w^T) in bfloat16, f a gate's function of one product (TQK_GATE_*: common.h). */
extern "C" int tqk_mid_store_act(const void* x, const void* w_packed, void* y, int M, int N, int K, void* scratch, int gate, float limit, float alpha,
                                 void* stream) {
    TQK_REQUIRE(gate >= 0 && gate < TQK_GATE_KINDS, "tqk_mid_store_act: unknown activation %d", gate);
    MidArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, y, (float*)scratch, M, N, K, 0, gate, limit, alpha, 1, 0, 0};
    if (check_mid(a, scratch, false, true, "tqk_mid_store_act")) return -1;
    if (M == 0) return 0;
    const MidPlan plan = mid_plan(N, K, false);
    a.k_per_split = plan.k_per_split;
    return launch_rows<MID_STORE, bf16_t>(a, plan, true, (hipStream_t)stream);
}

/* y[M, N/2] = silu(gate) * up, w = gate rows then up rows, packed in two parts. */
extern "C" int tqk_mid_gated(const void* x, const void* w_packed, void* y, int M, int N, int K, void* scratch, void* stream) {
    return tqk_mid_gated_act(x, w_packed, y, M, N, K, scratch, TQK_GATE_SILU, 0.f, 1.f, stream);
}

/* the same with another gate (TQK_GATE_*: common.h) */
extern "C" int tqk_mid_gated_act(const void* x, const void* w_packed, void* y, int M, int N, int K, void* scratch, int gate, float limit,
                                 float alpha, void* stream) {
    TQK_REQUIRE(gate >= 0 && gate < TQK_GATE_KINDS, "tqk_mid_gated: unknown gate %d", gate);
    MidArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, y, (float*)scratch, M, N, K, 0, gate, limit, alpha, 0, 0, 0};
    if (check_mid(a, scratch, true, true, "tqk_mid_gated")) return -1;
    if (M == 0) return 0;
    const MidPlan plan = mid_plan(N, K, true);
    a.k_per_split = plan.k_per_split;
    return launch_rows<MID_GATED, bf16_t>(a, plan, true, (hipStream_t)stream);
}
