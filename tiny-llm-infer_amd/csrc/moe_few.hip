// Routed experts for few rows (decode steps, bfloat16, up to 64 rows): two launches from the router's choice to the block's
// output, the shared expert taken along.
//
//   hidden:  hid[pair, f] = unit(x[row] . Wg_e[f], x[row] . Wu_e[f]) for every (row, chosen expert) pair, and the same of the
//            shared expert for every row
//   down:    part[j, row] = weight[row, j] (hid[row, j] . Wd_e) for the j-th expert of a row's choice, and behind them
//            part[top, row] = shared gate * (hid . Wd) of the shared expert; experts that hand their input on give weight * x.
//            The sum of the parts, in their order, is the block's output: whoever reads it adds them up.  Every part is written,
//            whichever experts a row names.
//
// Both are one kernel: a workgroup takes 32 rows of one expert's matrix (16 gate and 16 up rows of a gated one) and finds
// that expert's pairs of (row, place in the choice) itself, by looking through the choice: there is no sort.
//
// What bounds them is the reading of the chosen experts' matrices, and with so few bytes (a dozen experts of 8 to 25 MB)
// how many of their loads are in flight: k is dealt to the waves of a workgroup in steps of 128, as in gemm_skinny.hip.
// The tile-by-tile kernels of moe_grouped.hip give a wave all of k: 16 steps one after the other with one on its way.
// They stay for more rows, where an expert has several tiles and there are waves enough, and for more than 256 experts.
// Measured, 8 rows, 2 of 16 experts of width and hidden size 2,048, gated, a shared one of 4,096 (10 or 11 experts at work,
// 207 and 104 MB): hidden 43 -> 35 us with the shared expert's 8 us in it (5.9 TB/s), down 27 -> 20 us with its 6 us in it (5.2
// TB/s), sort (4.7 us) and sum of the parts (5.1 us) gone.  A down kernel of 16 columns of all experts at once, which needs no
// parts, has too few workgroups: 39 us.  Decode steps of four layers with 8 / 24 / 40 / 64 rows, width 2,048: 0.61 / 0.80 /
// 0.92 / 0.87 -> 0.47 / 0.58 / 0.69 / 0.69 ms; width 4,096 with 24 / 40 / 64 rows: 1.58 / 1.73 / 1.72 -> 1.26 / 1.54 / 1.56 ms.
//
// A row's result does not depend on the rows beside it: which wave takes which step of k depends on the sizes alone, and
// the sums of the waves are added in their order.
//
// Layout as in gemm_skinny.hip: A is a tile of W (16 outputs, blocks of 16 rows x 128 columns of 4 KiB), B the rows, a lane ends
// with four outputs of one row.
#include "common.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
union Pack16 {
    uint4 u;
    u32x4_t w;
    bf16x8 v;
};

__device__ __forceinline__ u32x4_t load16_once(const bf16_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
}

#define FEW_MAX_EXPERTS 256
#define FEW_MAX_ROWS 64

struct FewExperts {
    const bf16_t* x;             // [T, D]
    const int* ids;              // [T, top]: an id outside 0..E-1 is an expert that hands its input on
    const float* weights;        // [T, top] on the experts' outputs, or null
    const bf16_t *gate, *up, *down;          // [E] tiled [ff, D], [ff, D], [D, ff]; no gate matrices: null
    bf16_t* hid;                 // [T * top, ff]
    const bf16_t *s_gate, *s_up, *s_down;    // of the shared expert
    const float* s_weight;       // [T], or null: 1
    bf16_t* s_hid;               // [T, s_ff]
    float* part;                 // [top (+ 1), T, D]
    int handed_on;               // whether the choice may name experts that hand their input on
    long long s_step;            // elements between the shared expert's blocks of 16 hidden units
    int T, top, E, D, ff, s_ff;  // s_ff 0: no shared expert
    ExpertUnit unit;
    float s_limit;
};

// A wave's steps with the loads of the next DEPTH - 1 on their way: load(stage, n) and multiply(stage) for n = 0 .. count-1,
// no load under a branch in the main part (behind a branch the compiler waits for every load in flight).
template <int DEPTH, typename L, typename M>
__device__ __forceinline__ void in_steps(int count, L load, M multiply) {
    auto prologue = [&](auto self, auto INDEX) -> void {
        constexpr int I = decltype(INDEX)::value;
        if constexpr (I < DEPTH - 1) {
            if (I < count) load(std::integral_constant<int, I>{}, I);
            self(self, std::integral_constant<int, I + 1>{});
        }
    };
    auto round = [&](auto self, int i, auto INDEX, auto FULL_T) -> void {
        constexpr int I = decltype(INDEX)::value;
        constexpr bool FULL = decltype(FULL_T)::value;
        if constexpr (I < DEPTH) {
            if (FULL || i + I < count) {
                if (FULL || i + I + DEPTH - 1 < count) load(std::integral_constant<int, (I + DEPTH - 1) % DEPTH>{}, i + I + DEPTH - 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(std::integral_constant<int, I>{});
                __builtin_amdgcn_sched_barrier(0);
                self(self, i, std::integral_constant<int, I + 1>{}, FULL_T);
            }
        }
    };
    prologue(prologue, std::integral_constant<int, 0>{});
    int i = 0;
    for (; i + 2 * (DEPTH - 1) < count; i += DEPTH) round(round, i, std::integral_constant<int, 0>{}, std::true_type{});
    for (; i < count; i += DEPTH) round(round, i, std::integral_constant<int, 0>{}, std::false_type{});
}

#define FEW_GATED 0              // hidden units of gate and up rows
#define FEW_UP 1                 // hidden units of up rows alone
#define FEW_DOWN 2

// The pairs of an expert that found no slot, without the matrix cores: there are slots for as many pairs as rows, so these are
// only of choices that name an expert more than once in a row.  A wave a pair, a lane an output of the workgroup's two tiles
// `a` and `b` of W and one half of every 128 of k.
template <int KIND>
__device__ __forceinline__ void pairs_without_slot(const FewExperts& f, int e, int slots, const bf16_t* a, const bf16_t* b, int block, int K) {
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, waves = blockDim.x / 64;
    const bf16_t* w = lane % 32 < 16 ? a : b;
    for (int p = 0, n = 0; p < f.T * f.top; ++p) {
        if (f.ids[p] != e) continue;
        const int rank = n++;
        if (rank < slots || rank % waves != wave) continue;
        const bf16_t* x = KIND == FEW_DOWN ? f.hid + (size_t)p * K : f.x + (size_t)(p / f.top) * K;
        float s = 0.f;
        for (int i = 0; i < (K + 127) / 128 * 64; ++i) {             // (64 of 128 a step: c of two, j of four, eight in a row)
            const int kb = i / 64, c = lane / 32 * 2 + i / 32 % 2, j = i / 8 % 4, k = kb * 128 + c * 32 + i % 32;
            if (k < K) s = fmaf(bf16_to_f32(w[(size_t)kb * 2048 + j * 512 + (16 * c + lane % 16) * 8 + i % 8]), bf16_to_f32(x[k]), s);
        }
        s += __shfl_xor(s, 32, 64);
        const float other = __shfl_xor(s, 16, 64);
        const int unit = KIND == FEW_GATED ? block * 16 + lane % 16 : block * 32 + lane % 32;
        if (KIND == FEW_DOWN) {
            if (lane < 32 && unit < f.D)
                f.part[((size_t)(p % f.top) * f.T + p / f.top) * f.D + unit] = (f.weights ? f.weights[p] : 1.0f) * s;
        } else if (lane < (KIND == FEW_GATED ? 16 : 32) && unit < f.ff) {
            from_f32(f.hid + (size_t)p * f.ff + unit, KIND == FEW_GATED ? gated_unit(s, other, f.unit.limit, f.unit.slope) : act_of(f.unit.of_pair(p) * s, f.unit.kind));
        }
    }
}

// Blocks 0 .. s_blocks-1 are the shared expert's (FEW_DOWN: also of the experts that hand their input on); then `blocks` for each candidate expert: expert y where there are no more
// experts than pairs, else the expert of pair y, if no pair before it has the same.
template <int RB, int KIND>
__global__ void __launch_bounds__(256) moe_few_kernel(FewExperts f, int s_blocks, int blocks) {
    constexpr int WAVES = 4;
    constexpr bool GATED = KIND == FEW_GATED, DOWN = KIND == FEW_DOWN;
    __shared__ float red[WAVES][2 * RB][64][4];
    __shared__ int slots[WAVES][16 * RB];                   // the pair (of the shared expert: the row) of every slot
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);       // (in a scalar register)
    const int r = lane % 16, c = lane / 16;
    const bool shared = (int)blockIdx.x < s_blocks;
    const int block = shared ? blockIdx.x : (blockIdx.x - s_blocks) % blocks;
    const int P = f.T * f.top;
    int* mine = slots[wave];
    int e = 0, n = 0;                                        // the expert, and its number of pairs with a slot
    if (DOWN && shared && f.handed_on) {
        for (int i = threadIdx.x; i < P * 32; i += WAVES * 64) {
            const int p = i / 32, t = p / f.top, col = block * 32 + i % 32;
            if (col < f.D && (f.ids[p] < 0 || f.ids[p] >= f.E))
                f.part[((size_t)(p % f.top) * f.T + t) * f.D + col] = (f.weights ? f.weights[p] : 1.0f) * bf16_to_f32(f.x[(size_t)t * f.D + col]);
        }
    }
    if (DOWN && shared && f.s_ff == 0) return;
    if (shared) {
        n = f.T;
        for (int s = lane; s < 16 * RB; s += 64) mine[s] = min(s, f.T - 1);
    } else {
        const int y = (blockIdx.x - s_blocks) / blocks;
        e = f.E <= P ? y : f.ids[y];
        if (e < 0 || e >= f.E) return;                       // (the whole workgroup: all its waves see the same)
        for (int p0 = 0; p0 < P; p0 += 64) {
            const int p = p0 + lane;
            const bool match = p < P && f.ids[p] == e;
            const unsigned long long mask = __ballot(match);
            if (f.E > P && n == 0 && mask && p0 + __builtin_ctzll(mask) < y) return;
            const int rank = n + __popcll(mask & ((1ull << lane) - 1ull));
            if (match && rank < 16 * RB) mine[rank] = p;
            n += __popcll(mask);
        }
        if (n == 0) return;
        if (n > 16 * RB) {
            const int K = DOWN ? f.ff : f.D, kb = (K + 127) / 128, tiles = ((DOWN ? f.D : f.ff) + 15) / 16;
            const size_t expert = (size_t)e * tiles * kb * 2048, step = (size_t)kb * 2048;
            const bf16_t* u = (DOWN ? f.down : f.up) + expert;
            if (GATED) pairs_without_slot<KIND>(f, e, 16 * RB, f.gate + expert + block * step, u + block * step, block, K);
            else pairs_without_slot<KIND>(f, e, 16 * RB, u + 2 * block * step, u + min(2 * block + 1, tiles - 1) * step, block, K);
            n = 16 * RB;
        }
        wave_lds_sync();
        for (int s = lane; s < 16 * RB; s += 64)
            if (s >= n) mine[s] = mine[0];
    }
    wave_lds_sync();
    const int tiles = (n + 15) / 16;                         // of slots

    // the product's k and the rows of its matrix
    const int ff = shared ? f.s_ff : f.ff, K = DOWN ? ff : f.D, rows = DOWN ? f.D : ff;
    const int kblocks = (K + 127) / 128, all = (rows + 15) / 16;
    // the two tiles of W: gate and up rows of one block of hidden units, or the rows of two blocks
    const bf16_t* a_row[2];
    {
        const long long step = shared && !DOWN ? f.s_step : (long long)kblocks * 2048;
        const size_t expert = shared ? 0 : (size_t)e * all * kblocks * 2048;
        const bf16_t *g = shared ? f.s_gate : f.gate, *u = DOWN ? (shared ? f.s_down : f.down) : (shared ? f.s_up : f.up);
        if (GATED) {
            a_row[0] = g + expert + (size_t)block * step + lane * 8;
            a_row[1] = u + expert + (size_t)block * step + lane * 8;
        } else {
            a_row[0] = u + expert + (size_t)(2 * block) * step + lane * 8;
            a_row[1] = u + expert + (size_t)min(2 * block + 1, all - 1) * step + lane * 8;
        }
    }
    // Rows are read through a buffer descriptor, of which an offset past the end gives zeros: that is what lanes past the end
    // of k ask for.  (The tiles of W are zeros there, but a zero times whatever lies behind the row, or times an infinity that
    // stands in for it, need not be one.)
    const bf16_t* inputs = DOWN ? (shared ? f.s_hid : f.hid) : f.x;
    const auto buffer = __builtin_amdgcn_make_buffer_rsrc((void*)inputs, 0, (DOWN && !shared ? P : f.T) * K * 2, 0x00020000);
    int x_row[RB];                                            // in bytes
#pragma unroll
    for (int m = 0; m < RB; ++m) {
        const int slot = mine[m * 16 + r];
        x_row[m] = (DOWN || shared ? slot : slot / f.top) * K * 2;
    }

    f32x4 acc[2][RB];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < RB; ++m) acc[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
    Pack16 a[2][2][4], b[2][RB][4];
    auto load = [&](auto STAGE, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(STAGE)::value;
        const int kb = wave + i * WAVES;
#pragma unroll
        for (int m = 0; m < RB; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = kb * 128 + c * 32 + j * 8;
                b[S][m][j].w = __builtin_amdgcn_raw_buffer_load_b128(buffer, k < K ? x_row[m] + 2 * k : -16, 0, 0);
            }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) a[S][t][j].w = load16_once(a_row[t] + (size_t)kb * 2048 + j * 512);
    };
    auto multiply = [&](auto STAGE) __attribute__((always_inline)) {
        constexpr int S = decltype(STAGE)::value;
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int m = 0; m < RB; ++m)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[S][t][j].v, b[S][m][j].v, acc[t][m], 0, 0, 0);
    };
    in_steps<2>(wave < kblocks ? (kblocks - wave + WAVES - 1) / WAVES : 0, load, multiply);

#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < RB; ++m) *reinterpret_cast<f32x4*>(red[wave][t * RB + m][lane]) = acc[t][m];
    __syncthreads();
    // a tile of slots a wave
    if (wave >= RB || wave >= tiles) return;
    const int s = wave * 16 + r;
    if (s >= n) return;
    const int pair = mine[s];
    float v[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[t][i] = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) v[t][i] += red[w][t * RB + wave][lane][i];
        }
    bf16_t* row = (shared ? f.s_hid : f.hid) + (size_t)pair * ff;
    if constexpr (DOWN) {
        const float by = shared ? (f.s_weight ? f.s_weight[pair] : 1.0f) : f.weights ? f.weights[pair] : 1.0f;
        const int j = shared ? f.top : pair % f.top, t = shared ? pair : pair / f.top;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n0 = (2 * block + u) * 16 + c * 4;
            float y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = by * v[u][i];
            store4(f.part + ((size_t)j * f.T + t) * f.D + n0, y, f.D - n0, f.D % 4 == 0);
        }
    } else if (GATED) {
        const int n0 = block * 16 + c * 4;
        float h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = gated_unit(v[0][i], v[1][i], shared ? f.s_limit : f.unit.limit, f.unit.slope);
        store4(row + n0, h, ff - n0, ff % 4 == 0);
    } else {
        const float by = shared ? 1.0f : f.unit.of_pair(pair);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int n0 = (2 * block + t) * 16 + c * 4;
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = act_of(by * v[t][i], f.unit.kind);
            store4(row + n0, h, ff - n0, ff % 4 == 0);
        }
    }
}

// Whether the kernels above take these sizes.
extern "C" int tli_moe_few_takes(int T, int top, int E, int D, int ff) {
    return T > 0 && T <= FEW_MAX_ROWS && E > 0 && E <= FEW_MAX_EXPERTS && top > 0 && D > 0 && ff > 0 && D % 8 == 0 && ff % 8 == 0 &&
           (long long)T * D < 1 << 30 && (long long)T * top * ff < 1 << 30;       // (offsets into rows are 32 bits of bytes)
}

// gate_t, up_t, down_t as for tli_moe_grouped_bf16; hid [T * top, ff], s_hid [T, s_ff]: scratch; the shared expert (s_ff > 0): s_gate
// (act < 0) and s_up at the first block of 16 rows, blocks s_step elements apart, s_down tiled [D, s_ff].  part [top, T, D], one
// more with a shared expert: see the top of this file.
extern "C" int tli_moe_few_bf16(const void* x, const int* ids, const float* weights, const void* gate_t, const void* up_t,
                                const void* down_t, void* hid, const void* s_gate, const void* s_up, const void* s_down, long long s_step,
                                const float* s_weight, void* s_hid, float* part, int handed_on, int T, int top, int E, int D, int ff, int s_ff, float limit,
                                float slope, float s_limit, int act, int weight_on_input, void* stream) {
    if (T <= 0) return 0;
    if (!tli_moe_few_takes(T, top, E, D, ff) || s_ff < 0 || s_ff % 8 || (long long)T * s_ff >= 1 << 30)
        return tli_fail("moe_few: bad sizes (%d rows, %d of %d experts, width %d, %d and %d hidden units)", T, top, E, D, ff, s_ff);
    if (act >= TLI_ACT_KINDS || (act < 0 && (weight_on_input || !gate_t))) return tli_fail("moe_few: bad activation");
    if (s_ff && (!s_up || !s_down || !s_hid || s_step <= 0 || (act < 0 && (!s_gate || s_ff % 16)))) return tli_fail("moe_few: bad shared expert");
    if (((uintptr_t)x | (uintptr_t)gate_t | (uintptr_t)up_t | (uintptr_t)down_t | (uintptr_t)hid | (uintptr_t)s_gate | (uintptr_t)s_up |
         (uintptr_t)s_down | (uintptr_t)s_hid | (uintptr_t)part) & 15)
        return tli_fail("moe_few: operands must be 16-byte aligned");
    const FewExperts f{(const bf16_t*)x, ids, weight_on_input ? nullptr : weights, (const bf16_t*)gate_t, (const bf16_t*)up_t,
                       (const bf16_t*)down_t, (bf16_t*)hid, (const bf16_t*)s_gate, (const bf16_t*)s_up, (const bf16_t*)s_down, s_weight,
                       (bf16_t*)s_hid, part, handed_on, s_step, T, top, E, D, ff, s_ff,
                       ExpertUnit{act, limit, slope, weight_on_input ? weights : nullptr}, s_limit};
    hipStream_t s = (hipStream_t)stream;
    const int candidates = E < T * top ? E : T * top;
    const int units = act < 0 ? 16 : 32;
    const int s_blocks = (s_ff + units - 1) / units, blocks = (ff + units - 1) / units;
    const int d_blocks = (D + 31) / 32, d_s_blocks = s_ff || handed_on ? d_blocks : 0;
#define TLI_FEW(RB)                                                                                                          \
    if (act < 0) moe_few_kernel<RB, FEW_GATED><<<s_blocks + blocks * candidates, 256, 0, s>>>(f, s_blocks, blocks);          \
    else moe_few_kernel<RB, FEW_UP><<<s_blocks + blocks * candidates, 256, 0, s>>>(f, s_blocks, blocks);                    \
    moe_few_kernel<RB, FEW_DOWN><<<d_s_blocks + d_blocks * candidates, 256, 0, s>>>(f, d_s_blocks, d_blocks)
    if (T <= 16) { TLI_FEW(1); }
    else if (T <= 32) { TLI_FEW(2); }
    else { TLI_FEW(4); }
#undef TLI_FEW
    return tli_check_launch("moe_few");
}
