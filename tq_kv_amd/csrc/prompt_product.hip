// y[M,N] = x[M,K] w[N,K]^T for many rows (prompts; more than the kernel for mid-sized steps takes): bfloat16 in, MFMA,
// float32 accumulation, the weight from the copy packed in the lanes' order ([tile of 16 rows][K/32][lane][8 values], see
// skinny_fused.hip).  The reference runs these products as candle matmuls (src/models/turbo_generic.rs:68-91).
//
// What binds it: with the model's values (not zeros) the matrix cores draw the card to its power limit at about
// 1.4 PFLOP/s; the same kernel on zeros, or without memory, runs at 1.6 and 2.1.  So the layout spends as little as it can
// beside the products themselves:
//
//  - A block is four waves side by side along the features, each with MT groups of 16 rows of x by NT tiles of 16
//    features, so a weight is needed by one wave alone: it comes straight into that wave's registers, 1 KB of contiguous
//    memory a load, WD steps of 32 k held, and never passes through LDS.  (With 32x32x16 instructions the same kernel
//    is 5 % slower: 1.16 against 1.23 PFLOP/s at 8000 x 18944 x 3584.)
//  - x is shared by the waves: stages of 64 k go from memory into LDS without passing through registers (loads that end in
//    LDS), four stages in turn, one barrier a stage.  A load takes eight whole 128-byte lines of x; the 16-byte pieces of a row
//    are exchanged within it (piece c of row r lies at c ^ ((r / 2) % 8)) so that the waves' reads of 16 rows of one k step meet
//    all banks once.  A wave reads its operands PD groups ahead, across the barrier too.
//  - WN = 5 with 15 groups of rows (240; in ten waves for up to 160, 192 and 256 rows, see five_wide): gated products of one such row of blocks and no more blocks than units, where what a compute unit
//    brings in binds and not the products: every block needs all of x, so few, even blocks count.  us at 129, 170, 232 rows against the best
//    tile of four waves: 18944 gated features (237 blocks of 80) x K of 3584 73, 73, 74 against 80, 84, 90; 17920 x 5120 100, 102, 104 against
//    115, 120, 127; 20480 x 3584 75, 78, 80 against 80, 84, 90; 16640 x 2048 43, 45, 46 against 42, 47, 51; 17920 x 1536 36, 39, 39 against
//    36, 38, 41.  With more blocks than units it loses (22016 x 4096 144, 144, 147 against 96, 100, 112), and from two rows of blocks on, too,
//    since a block alone on its unit has a lower rate (17920 x 1536, 440 rows: 38 against 34.5).  Products without a gate have too few blocks
//    of that height: with every number of pieces of K tried at 129 to 240 rows, q/k/v and o lose at all three Qwen2.5 shapes (7B, 232 rows:
//    25.0 against 18.9 and 23.5 against 15.8) and down at the 1.5B one (27 against 19); the other two are within 4 % (50.6 against 50.1, 85.6
//    against 89.3).  Ten waves: 18944 x 3584 at 129, 170 and 256 rows 74, 75 and 83 against 87 and 86 with 240 rows in five waves and 96 with the best tile of
//    four, 16640 x 2048 42, 46 and 49 against 50, 49 and 62, 17920 x 1536 35, 38 and 41 against 40, 39 and 44; at 232 rows the same as five.
//  - WM = 2: a second row of four waves on the next MT groups of rows, 256 rows a block, one block a compute unit; the two
//    waves of a column meet each other's weights in the first-level cache, and a unit brings in a third less than two blocks
//    of WM = 1 would.  Worth a little where K is long (8000 x 3584 x 18944: 861 us against 869), not where it is short (8000 x 37888 x 3584
//    without a gate 1585 against 1565; 8000 x 4608 x 3584, where blocks of that size do not go round evenly, 226 against 195).
//
// The waits are counted by hand where LDS is concerned (a wave knows how many loads it has issued since the stage it
// waits for) and by the compiler for the registers; each stage is an array of its own, so that the compiler can tell the
// stage being filled from the one being read.
//
// The epilogue turns 16 rows at a time through LDS, so that a store instruction writes whole lines (o, 2048 rows: 41 us against 45 with
// the 8 bytes a lane holds stored as they are), and applies a gate (silu(gate) * up of src/models/turbo_generic.rs:105-111) or
// an activation on the way.
//
// Against the library it replaces here (its own first choice for a shape, which is what a prompt of any length gets; in
// brackets the best of all its kernels, found by trying): 2048 rows of the 7B shape, us: gate+up 427 with the gate applied, against
// 522 (386) and 40 for the gate's kernel; down 223 against 365 (234); q/k/v 57 against 63 (64); o 41 against 55 (55).
#include "common.h"
#include "tq_kernels.h"

#include <type_traits>
#include <utility>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4_t;
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

enum { PROMPT_STORE = 0, PROMPT_GATED = 1, PROMPT_ACT = 2 };
#define PROMPT_STAGES 4
#define PROMPT_K 256            // k per turn of the loop: all stages once; K is cut into multiples of it

struct PromptArgs {
    const bf16_t* x;            // [M, K]
    const bf16_t* w;            // packed [tiles][K/32][64][8]; gated: the gate's tiles, then up's
    bf16_t* y;                  // store: [M, N]; gated: [M, N/2]
    float* sums;                // [splits][M][N] where K is cut, [M, N] where the result is wanted in float32; else null
    int M, N, K, k_per_split, tiles_m, tiles_n;
    int gate;                   // gated, activated: which gate (TQK_GATE_*), with its limit and alpha
    float gate_limit, gate_alpha;
};

template <typename F, int... I> __device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each(f, std::make_integer_sequence<int, N>{}); }

__device__ __forceinline__ uint2 pack4_bf16(const float (&v)[4]) {
    return make_uint2((uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16),
                      (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16));
}
__device__ __forceinline__ float rounded(float v) { return to_float(from_float<bf16_t>(v)); }

// The epilogue's last part: f of a value (gated: of a gate's and up's value), 16 rows at a time through LDS (`turn`, the wave's own), so that a
// store instruction writes whole lines.
template <int MT, int NT, int TW, typename F>
__device__ __forceinline__ void write_rows(const PromptArgs& p, const floatx4_t (&acc)[MT][NT], char* turn, int row0, int r16, int lane, int tile0,
                                           int part_tiles, int n_out, F&& f) {
    constexpr int LINE = TW * 32 + 16;              // bytes of a row in LDS: the wave's features and a gap that spreads the banks
    constexpr int PIECES = TW * 2;                  // of 16 bytes in a row
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            float o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = f(acc[m][TW == NT ? t : 2 * t][i], acc[m][TW == NT ? t : 2 * t + 1][i]);
            *reinterpret_cast<uint2*>(turn + r16 * LINE + t * 32 + lane / 16 * 8) = pack4_bf16(o);
        }
        // (a wave's own LDS operations are in order, and nobody else uses its rows)
#pragma unroll
        for (int i0 = 0; i0 < 16 * PIECES; i0 += TQK_WAVE) {
            const int i = i0 + lane, r = i / PIECES, c = i % PIECES, row = row0 + m * 16 + r;
            if (i < 16 * PIECES && row < p.M && tile0 + c / 2 < part_tiles)
                *reinterpret_cast<u32x4_t*>(p.y + (size_t)row * n_out + tile0 * 16 + c * 8) = *reinterpret_cast<const u32x4_t*>(turn + r * LINE + c * 16);
        }
    }
}

template <int MT, int NT, int WM, int WN, int EPI>
__global__ __launch_bounds__(TQK_WAVE * WN * WM, WM == 1 && WN == 4 ? 2 : 1)
void prompt_product_kernel(const PromptArgs p) {
    constexpr int NS = PROMPT_STAGES, WD = 4;
    constexpr int DMA = (2 * MT + WN - 1) / WN;     // loads of 1 KB by which a wave helps to bring in a stage
    constexpr int STAGE = WM * WN * DMA * 1024;     // bytes: [rows][8 pieces of 16 bytes]
    constexpr int PD = (2 * MT) % 4 == 0 ? 4 : (2 * MT) % 6 == 0 ? 6 : 5;          // operands read ahead; a divisor of a stage's groups
    static_assert((2 * MT) % PD == 0, "");
    constexpr int GROUPS = 2 * MT, SYNC = GROUPS - PD;
    constexpr int TW = EPI == PROMPT_GATED ? NT / 2 : NT;       // a wave's tiles of the output
    static_assert(NT <= MT && (EPI != PROMPT_GATED || NT % 2 == 0), "");
    __shared__ __attribute__((aligned(1024))) char buf0[STAGE], buf1[STAGE], buf2[STAGE], buf3[STAGE];
    const int lane = threadIdx.x % TQK_WAVE, wv = __builtin_amdgcn_readfirstlane(threadIdx.x / TQK_WAVE);
    const int wave = wv % WN, wm = wv / WN;
    const int r16 = lane % 16, K = p.K;

    // Blocks are dealt to the eight dies in turn: each die takes a run of tiles, rows fastest inside bands of 1024 rows, so
    // that the blocks a die runs at a time share both x and weights in its second-level cache.
    int tm, tn;
    {
        const int n = p.tiles_m * p.tiles_n, die = blockIdx.x % 8, at = blockIdx.x / 8, each_die = n / 8, more = n % 8;
        const int id = die * each_die + min(die, more) + at;
        constexpr int BAND = 8 / WM;
        const int band = id / (BAND * p.tiles_n), in = id % (BAND * p.tiles_n), rows = min(BAND, p.tiles_m - band * BAND);
        tm = band * BAND + in % rows;
        tn = in / rows;
    }
    const int k_begin = blockIdx.y * p.k_per_split, n_stage = min(K - k_begin, p.k_per_split) / 64;

    const int n_out = EPI == PROMPT_GATED ? p.N / 2 : p.N, part_tiles = n_out / 16;
    const int tile0 = (tn * WN + wave) * TW;
    // where the wave's tiles begin, in bytes (tiles past the end repeat the last one; their results are dropped)
    uint32_t w_at[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int tile = EPI == PROMPT_GATED ? (t % 2) * part_tiles + min(tile0 + t / 2, part_tiles - 1) : min(tile0 + t, part_tiles - 1);
        w_at[t] = ((uint32_t)tile * (uint32_t)(K / 32) + (uint32_t)(k_begin / 32)) * 1024u;
    }
    // the pieces of x a lane brings in: row 8 j + lane / 8 of the block's, piece (lane % 8) of its place in LDS; rows past M repeat the last
    uint32_t x_at[DMA];
    const char* x0 = (const char*)(p.x + (size_t)tm * (WM * MT * 16) * K + k_begin);
    {
        const int last = p.M - 1 - tm * (WM * MT * 16);
#pragma unroll
        for (int i = 0; i < DMA; ++i) {
            const int j = i * WN * WM + wv;
            x_at[i] = (uint32_t)min(j * 8 + lane / 8, last) * (uint32_t)(K * 2) + ((lane % 8) ^ ((4 * (j % 2) + lane / 16) % 8)) * 16;
        }
    }
    const __amdgpu_buffer_rsrc_t x_mem = __builtin_amdgcn_make_buffer_rsrc((void*)x0, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_mem = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, 0x7fffffff, 0x00020000);
    auto buf = [&](auto I) -> char* {
        constexpr int i = decltype(I)::value % NS;
        if constexpr (i == 0) return buf0; else if constexpr (i == 1) return buf1; else if constexpr (i == 2) return buf2; else return buf3;
    };
    // (past the last stage the last one is brought in again, into an array that is free, and not read: the count of loads stays)
    auto load_x = [&](auto I, int i, int stage) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_mem, (lds_ptr_t)(buf(I) + wv * 1024 + i * (1024 * WN * WM)), 16, (int)x_at[i], min(stage, n_stage - 1) * 128, 0, 0);
    };
    bf16x8_t w[WD][NT];
    auto load_w = [&](int step, int t, bf16x8_t& to) {
        to = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(w_mem, lane * 16, w_at[t] + min(step, 2 * n_stage - 1) * 1024, 0));
    };
    floatx4_t acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // a lane's place in a group of 16 rows: row r16, the piece of k step 0 or 1 of the stage
    const int at0 = wm * (MT * 2048) + r16 * 128 + ((lane / 16) ^ (r16 / 2)) * 16, at1 = at0 ^ 64;
    bf16x8_t xr[PD];
    each<NS - 1>([&](auto S) {
#pragma unroll
        for (int i = 0; i < DMA; ++i) load_x(S, i, S);
    });
#pragma unroll
    for (int s = 0; s < WD - 1; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t) load_w(s, t, w[s][t]);
    __builtin_amdgcn_s_waitcnt(0x0f70);             // vmcnt(0)
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int j = 0; j < PD; ++j) xr[j] = *reinterpret_cast<const bf16x8_t*>(buf0 + at0 + j * 2048);

    for (int s0 = 0; s0 < n_stage; s0 += NS) {
        each<NS>([&](auto H) {
            constexpr int h = decltype(H)::value;
            const int s = s0 + h;
            // a group: NT products with one operand of x; between groups the next operand is read and loads are issued
            each<GROUPS>([&](auto J) {
                constexpr int j = decltype(J)::value, m = j % MT, step = j / MT, q = j + PD;
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (j == SYNC) {
                    // The next stage's loads were issued behind this point two stages ago.  Since then the wave has issued a
                    // stage's loads of x and of weights, and what this stage has asked for so far: as many may be under way.
                    constexpr int here = (SYNC < NT ? SYNC : NT) + (SYNC > MT ? (SYNC - MT < NT ? SYNC - MT : NT) : 0);
                    constexpr int left = (NS - 3) * (DMA + 2 * NT) + here;
                    static_assert(left < 64, "");
                    __builtin_amdgcn_s_waitcnt(0x0f70 | (left & 15) | ((left >> 4) << 14));
                    __builtin_amdgcn_s_barrier();   // everybody's part of the next stage is there; the stage before this one is read
                }
                const bf16x8_t b = xr[j % PD];
                if constexpr (q < GROUPS) xr[j % PD] = *reinterpret_cast<const bf16x8_t*>(buf(H) + (q / MT ? at1 : at0) + (q % MT) * 2048);
                else xr[j % PD] = *reinterpret_cast<const bf16x8_t*>(buf(std::integral_constant<int, h + 1>{}) + at0 + (q - GROUPS) * 2048);
                if constexpr (m < NT) load_w(2 * s + step + WD - 1, m, w[(2 * h + step + WD - 1) % WD][m]);
                if constexpr (j >= SYNC) {
#pragma unroll
                    for (int i = (j - SYNC) * DMA / PD; i < (j - SYNC + 1) * DMA / PD; ++i) load_x(std::integral_constant<int, h + NS - 1>{}, i, s + NS - 1);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[(2 * h + step) % WD][t], b, acc[m][t], 0, 0, 0);
            });
        });
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);             // nothing is on its way into LDS any more, from any wave
    __builtin_amdgcn_s_barrier();

    // A product's D[feature][row]: a lane holds row r16 and the features 4 (lane / 16) .. + 3 of a tile.
    const int col = 4 * (lane / 16), row0 = (tm * WM + wm) * MT * 16;
    char* turn = (wv % 2 ? buf1 : buf0) + wv / 2 * 16 * (TW * 32 + 16);
    static_assert(16 * (TW * 32 + 16) * ((WN * WM + 1) / 2) <= STAGE, "");
    if constexpr (EPI != PROMPT_GATED) {
        if (p.sums) {
            float* y = p.sums + (size_t)blockIdx.y * p.M * p.N;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int row = row0 + m * 16 + r16;
#pragma unroll
                for (int t = 0; t < TW; ++t)
                    if (row < p.M && tile0 + t < part_tiles) *reinterpret_cast<floatx4_t*>(y + (size_t)row * p.N + (tile0 + t) * 16 + col) = acc[m][t];
            }
            return;
        }
    }
    // (which gate is asked once, not for every value: the usual one has a loop of its own)
    if constexpr (EPI == PROMPT_STORE) {
        write_rows<MT, NT, TW>(p, acc, turn, row0, r16, lane, tile0, part_tiles, n_out, [](float v, float) { return v; });
    } else if constexpr (EPI == PROMPT_ACT) {
        write_rows<MT, NT, TW>(p, acc, turn, row0, r16, lane, tile0, part_tiles, n_out,
                               [&](float v, float) { return act_value(p.gate, p.gate_limit, p.gate_alpha, rounded(v)); });
    } else if (p.gate == TQK_GATE_SILU) {
        write_rows<MT, NT, TW>(p, acc, turn, row0, r16, lane, tile0, part_tiles, n_out,
                               [](float g, float u) { return gate_value(TQK_GATE_SILU, 0.f, 1.f, rounded(g), rounded(u)); });
    } else {
        write_rows<MT, NT, TW>(p, acc, turn, row0, r16, lane, tile0, part_tiles, n_out,
                               [&](float g, float u) { return gate_value(p.gate, p.gate_limit, p.gate_alpha, rounded(g), rounded(u)); });
    }
}

// Adds the pieces of K up in order and finishes as the product's epilogue does without pieces.
template <typename TY>
__global__ void prompt_finish_kernel(const float* __restrict__ partial, TY* __restrict__ y, int splits, size_t n, int gate, float limit, float alpha,
                                     bool activated) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n) return;
    floatx4_t a = *reinterpret_cast<const floatx4_t*>(partial + i);
    for (int s = 1; s < splits; ++s) a += *reinterpret_cast<const floatx4_t*>(partial + (size_t)s * n + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) y[i + j] = from_float<TY>(activated ? act_value(gate, limit, alpha, rounded(a[j])) : a[j]);
}

// ---- which tile, and into how many pieces K is cut ----------------------------------------------------
// A block's time is its share of the products over the rate its tile reaches when every unit is busy, and units that hold one
// block more than the others set the time of all: time = ceil(blocks / 256) * rows * features * k / rate.  The rates are
// measured (8000 rows of the 7B products, corrected for the last round), relative to the best; smaller tiles bring more bytes in for
// a product.  The start and end of a block cost as much as 300 k; 600 for a gated block that has its unit to itself (wm = 2), since then
// nothing else runs on the unit while the gate is applied (8000 x 1536 x 17920 gated: 393 us against 350 with blocks of four waves;
// 37888 x 3584 1638 against 1539).  Cutting K adds the pieces' sums, written and read as float32.  Against all tiles tried one by one
// at 232, 300, 1024, 2048 and 8000 rows of the four 7B products the rule takes the fastest or one within 4 % of it, but for
// the gated product of 300 to 600 rows (within 10 %).  Elsewhere it can be further off: gated 24576 x 3072 and 22016 x 4096 at 170 rows
// 90 and 115 us, with another tile 78 and 100; o and q/k/v of the 1.5B shape, finished here, up to 2 us of 11 slower in pieces than whole.
struct PromptPlan { int config, splits, k_per_split; double us; };
struct PromptConfig { int mt, nt, wm, wn; double rate; };
static const PromptConfig CONFIGS[] = {
    {8, 4, 2, 4, 1.00}, {8, 4, 1, 4, 0.96}, {8, 3, 2, 4, 0.95}, {8, 3, 1, 4, 0.90}, {6, 4, 1, 4, 0.84},
    {8, 2, 1, 4, 0.78}, {5, 4, 1, 4, 0.72}, {4, 4, 1, 4, 0.66}, {5, 2, 1, 4, 0.58}, {15, 2, 1, 5, 0.79},     // (the last: five_wide)
};
#define PROMPT_CONFIGS ((int)(sizeof(CONFIGS) / sizeof(CONFIGS[0])))
#define PROMPT_UNITS 256
#define PROMPT_MAX_SPLITS 16

// The gated tile of five waves side by side has all rows in one block, as high as they are many: two rows of five waves for up to 160, 192 and 256, whose ten
// waves lie more evenly on the four SIMDs than five do (three and two against two and one), and one of five for up to 240, which brings weights in once.
static PromptConfig five_wide(int M) {
    if (M <= 160) return {5, 2, 2, 5, 0.62};
    if (M <= 192) return {6, 2, 2, 5, 0.72};
    if (M <= 240) return {15, 2, 1, 5, 0.79};
    return {8, 2, 2, 5, 0.84};
}

static PromptPlan prompt_plan(int M, int N, int K, bool gated) {
    PromptPlan best = {0, 1, K, 1e30};
    const long long turns = K / PROMPT_K;
    for (int i = 0; i < PROMPT_CONFIGS; ++i) {
        const PromptConfig c = CONFIGS[i].wn == 5 ? five_wide(M) : CONFIGS[i];
        if (gated && c.nt % 2) continue;
        if (c.wn == 5 && (!gated || M > 256)) continue;
        const long long rows = 16LL * c.mt * c.wm, width = 16LL * c.wn * (gated ? c.nt / 2 : c.nt), n_out = gated ? N / 2 : N;
        const long long tiles = ((M + rows - 1) / rows) * ((n_out + width - 1) / width);
        if (tiles > 0x7fffffffLL) continue;
        for (int splits = 1; splits <= (gated ? 1 : PROMPT_MAX_SPLITS) && splits <= turns; ++splits) {
            const long long per = (turns + splits - 1) / splits;
            if (per * (splits - 1) >= turns) continue;                                                // an empty piece
            const double rounds = (double)((tiles * splits + PROMPT_UNITS - 1) / PROMPT_UNITS);
            // (us: 256 units at the best tile's rate are 1.4 PFLOP/s)
            double us = rounds * (c.mt * c.nt * c.wm * c.wn / 4.0) / c.rate * (double)(per * PROMPT_K + (gated && c.wm == 2 && c.wn == 4 ? 600 : 300)) * 3.7e-4;
            if (splits > 1) us += (double)splits * M * N * 8.0 / 4.5e6;
            if (us < best.us) best = {i, splits, (int)(per * PROMPT_K), us};
        }
    }
    return best;
}

/* Whether the kernel takes a product of these sizes: K in whole turns of its loop, whole tiles of features, the packed weight within
 * what a 31-bit offset reaches (gated: N counts both parts' rows). */
extern "C" int tqk_prompt_takes(int M, int N, int K, int gated) {
    if (M <= 0 || N <= 0 || K <= 0 || K % PROMPT_K || N % (gated ? 32 : 16)) return 0;
    if ((long long)N * K * 2 > 0x7fffffffLL || 256LL * K * 2 > 0x7fffffffLL) return 0;
    return 1;
}

/* Into how many pieces the product's K is cut (1: none, no scratch is needed). */
extern "C" int tqk_prompt_splits(int M, int N, int K) { return tqk_prompt_takes(M, N, K, 0) ? prompt_plan(M, N, K, false).splits : 1; }

/* Whether a product that is taken is worth it where its pieces' sums are not left to another kernel; else the library is the faster one (its first
 * choice for a shape, us in replayed graphs, weights from memory).
 * Cut into pieces, the second kernel that adds them up takes 3.6 us and more: of 921 sizes (16 to 16384 features, K of 256 to 18944, 129 to 8000
 * rows) the 362 cut ones that the plan puts below 18 us with it are 1.17 times as slow as the library (200 x 512 x 4096 13.4 us against 8.3,
 * 129 x 128 x 2048 8.8 against 5.9), the 156 above 1.49 times as fast, the 403 whole ones 1.17 times; left to the next kernel cut ones are 1.49
 * times as fast, two of 520 slower.
 * A gate cannot be applied to pieces, so K is whole however few blocks there are: measured against what the same product without
 * the gate would take in pieces, and 5 us for a gate of its own.  Of 687 gated sizes those refused are 1.37 times as slow as the library with its gate's
 * kernel (200 x 64 x 8192 36 us against 13, 129 x 1024 x 8192 57 against 30), the others 1.33 times as fast; the factor 1.3 lies above
 * what the large products reach (1.16), which are to stay. */
extern "C" int tqk_prompt_pays(int M, int N, int K, int gated) {
    if (!tqk_prompt_takes(M, N, K, gated)) return 0;
    const PromptPlan plan = prompt_plan(M, N, K, gated != 0);
    if (!gated) return plan.splits == 1 || plan.us + 3.6 >= 18.0;
    return plan.us <= 1.3 * prompt_plan(M, N, K, false).us + 5.0;
}

/* Which tile the product takes (an index of the table above; -1: sizes that are not taken): for tests. */
extern "C" int tqk_prompt_tile(int M, int N, int K, int gated) { return tqk_prompt_takes(M, N, K, gated) ? prompt_plan(M, N, K, gated != 0).config : -1; }

template <int MT, int NT, int WM, int EPI, int WN = 4>
static void launch(const PromptArgs& a, int splits, hipStream_t s) {
    prompt_product_kernel<MT, NT, WM, WN, EPI><<<dim3(a.tiles_m * a.tiles_n, splits), TQK_WAVE * WN * WM, 0, s>>>(a);
}

template <int EPI>
static int launch_plan(PromptArgs a, const PromptPlan& plan, hipStream_t s) {
    const PromptConfig c = CONFIGS[plan.config].wn == 5 ? five_wide(a.M) : CONFIGS[plan.config];
    const int rows = 16 * c.mt * c.wm, width = 16 * c.wn * (EPI == PROMPT_GATED ? c.nt / 2 : c.nt), n_out = EPI == PROMPT_GATED ? a.N / 2 : a.N;
    a.tiles_m = (a.M + rows - 1) / rows;
    a.tiles_n = (n_out + width - 1) / width;
    a.k_per_split = plan.k_per_split;
    switch (plan.config) {
        case 0: launch<8, 4, 2, EPI>(a, plan.splits, s); break;
        case 1: launch<8, 4, 1, EPI>(a, plan.splits, s); break;
        case 2: if constexpr (EPI != PROMPT_GATED) launch<8, 3, 2, EPI>(a, plan.splits, s); break;
        case 3: if constexpr (EPI != PROMPT_GATED) launch<8, 3, 1, EPI>(a, plan.splits, s); break;
        case 4: launch<6, 4, 1, EPI>(a, plan.splits, s); break;
        case 5: launch<8, 2, 1, EPI>(a, plan.splits, s); break;
        case 6: launch<5, 4, 1, EPI>(a, plan.splits, s); break;
        case 7: launch<4, 4, 1, EPI>(a, plan.splits, s); break;
        case 8: launch<5, 2, 1, EPI>(a, plan.splits, s); break;
        default:
            if constexpr (EPI == PROMPT_GATED) {
                if (c.mt == 5) launch<5, 2, 2, EPI, 5>(a, plan.splits, s);
                else if (c.mt == 6) launch<6, 2, 2, EPI, 5>(a, plan.splits, s);
                else if (c.mt == 8) launch<8, 2, 2, EPI, 5>(a, plan.splits, s);
                else launch<15, 2, 1, EPI, 5>(a, plan.splits, s);
            }
            break;
    }
    return tqk_check_launch("tqk_prompt product");
}

static int check_prompt(const PromptArgs& a, const void* y, bool gated, const void* scratch, bool finish, const char* what) {
    TQK_REQUIRE(a.x && a.w, "%s: null pointer", what);
    TQK_REQUIRE(a.M >= 0, "%s: M=%d", what, a.M);
    if (a.M == 0) return 0;
    TQK_REQUIRE(tqk_prompt_takes(a.M, a.N, a.K, gated), "%s: sizes M=%d N=%d K=%d are not taken", what, a.M, a.N, a.K);
    TQK_REQUIRE(((((uintptr_t)a.x) | ((uintptr_t)a.w) | ((uintptr_t)y) | ((uintptr_t)scratch)) & 15) == 0, "%s: x, w, y and scratch must be 16-byte aligned", what);
    const int splits = gated ? 1 : tqk_prompt_splits(a.M, a.N, a.K);
    TQK_REQUIRE(y || (!finish && splits > 1), "%s: null output", what);
    TQK_REQUIRE(scratch || splits == 1, "%s: no scratch given", what);
    return 0;
}

static int prompt_store(PromptArgs a, bool activated, void* y, int y_dtype, float* scratch, bool finish, hipStream_t s) {
    const PromptPlan plan = prompt_plan(a.M, a.N, a.K, false);
    a.y = (bf16_t*)y;
    a.sums = plan.splits > 1 ? scratch : y_dtype == TQK_F32 ? (float*)y : nullptr;
    if (activated && plan.splits == 1 ? launch_plan<PROMPT_ACT>(a, plan, s) : launch_plan<PROMPT_STORE>(a, plan, s)) return -1;
    if (plan.splits == 1 || !finish) return 0;
    const size_t n = (size_t)a.M * a.N;
    const unsigned blocks = (unsigned)((n / 4 + 255) / 256);
    if (y_dtype == TQK_F32) prompt_finish_kernel<float><<<blocks, 256, 0, s>>>(scratch, (float*)y, plan.splits, n, a.gate, a.gate_limit, a.gate_alpha, activated);
    else prompt_finish_kernel<bf16_t><<<blocks, 256, 0, s>>>(scratch, (bf16_t*)y, plan.splits, n, a.gate, a.gate_limit, a.gate_alpha, activated);
    return tqk_check_launch("tqk_prompt finish");
}

/* y[M,N] = x w^T, w packed; scratch: float32 [tqk_prompt_splits(M, N, K)][M][N] where that is more than 1.  finish == 0: with more
 * than one piece the pieces' sums are left in scratch (for tqk_add_rmsnorm_sums, tqk_rope_store_sums) and y is not written. */
extern "C" int tqk_prompt_store(const void* x, const void* w_packed, void* y, int y_dtype, int M, int N, int K, void* scratch, int finish, void* stream) {
    const PromptArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, nullptr, nullptr, M, N, K, 0, 0, 0, 0, 0.f, 1.f};
    TQK_REQUIRE(y_dtype == TQK_F32 || y_dtype == TQK_BF16, "tqk_prompt_store: unknown output dtype %d", y_dtype);
    if (check_prompt(a, y, false, scratch, finish != 0, "tqk_prompt_store")) return -1;
    return M == 0 ? 0 : prompt_store(a, false, y, y_dtype, (float*)scratch, finish != 0, (hipStream_t)stream);
}

/* y[M,N] = f(x w^T) in bfloat16, f a gate's function of one product (TQK_GATE_*: common.h); scratch as tqk_prompt_store's. */
extern "C" int tqk_prompt_store_act(const void* x, const void* w_packed, void* y, int M, int N, int K, void* scratch, int gate, float limit, float alpha,
                                    void* stream) {
    TQK_REQUIRE(gate >= 0 && gate < TQK_GATE_KINDS, "tqk_prompt_store_act: unknown activation %d", gate);
    const PromptArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, nullptr, nullptr, M, N, K, 0, 0, 0, gate, limit, alpha};
    if (check_prompt(a, y, false, scratch, true, "tqk_prompt_store_act")) return -1;
    return M == 0 ? 0 : prompt_store(a, true, y, TQK_BF16, (float*)scratch, true, (hipStream_t)stream);
}

/* y[M, N/2] = gate(x wg^T, x wu^T) in bfloat16, w = gate rows then up rows, packed in two parts. */
extern "C" int tqk_prompt_gated_act(const void* x, const void* w_packed, void* y, int M, int N, int K, int gate, float limit, float alpha, void* stream) {
    TQK_REQUIRE(gate >= 0 && gate < TQK_GATE_KINDS, "tqk_prompt_gated_act: unknown gate %d", gate);
    const PromptArgs a = {(const bf16_t*)x, (const bf16_t*)w_packed, (bf16_t*)y, nullptr, M, N, K, 0, 0, 0, gate, limit, alpha};
    if (check_prompt(a, y, true, nullptr, true, "tqk_prompt_gated_act")) return -1;
    return M == 0 ? 0 : launch_plan<PROMPT_GATED>(a, prompt_plan(M, N, K, true), (hipStream_t)stream);
}
