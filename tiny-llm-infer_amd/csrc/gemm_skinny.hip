// Matrix product for few rows (decode): y[M,N] = x[M,K] . W[N,K]^T, M <= 64,
// bfloat16 inputs, float32 accumulation on the matrix cores, bfloat16 or
// float32 output.  The work is streaming W from HBM once; everything is laid
// out so that each lane's global loads are 64 contiguous bytes of one W row and
// land directly in the MFMA operand registers (no LDS staging of W).
//
// The reference multiplies a single row with a hand GEMV and more rows with a
// library call (kernels/src/matmul_kernel_cuda.cu:72-91); this kernel covers
// both for up to 64 rows.
//
// v_mfma_f32_16x16x32_bf16 computes D[16x16] += A[16x32] B[32x16]; lane l holds
// A[l%16][(l/16)*8 .. +8], B[(l/16)*8 .. +8][l%16] and D[(l/16)*4 .. +4][l%16].
// Here A is a tile of W (16 output columns n), B is x^T (16 rows m), so a lane
// ends with y[m = l%16][n = (l/16)*4 .. +4].  The 32 k-slots of one MFMA may be
// any 32 values of k as long as A and B agree: lane group c = l/16 takes the 32
// consecutive k  [kb + 32c, kb + 32c + 32)  of a 128-wide step, 8 per MFMA.
//
// The rows of x of a step go through LDS where that pays (through_lds below), and where whole tiles of 16 columns leave half the
// compute units without one a workgroup takes half a tile (half_tiles).  Measured with 8 rows, cold weights, launches of a chain (straight
// into the operand registers, whole tiles, before): 2,048 columns into the residual of k 8,192 13.2 -> 9.8 us, of k 12,288 15.3 ->
// 12.6; 4,096 columns of k 4,096 9.0 -> 8.0, of k 12,288 19.9 -> 18.9; 24,576 of k 4,096 (gated) 31.6 -> 31.3.  A chain of launches
// costs 2.5 us each before the first byte; what is left goes by at 6.4 TB/s.
//
// A workgroup owns 16*RT output columns; its waves take the 128-wide k steps in
// turn and their partial sums are added through LDS in wave order, so the
// result does not depend on the launch.
//
// Two variants take the RMS norms of a decoder block into the products around them, so
// that a decode step needs no norm kernel between its products.  With h the float32
// residual, w the norm's weights and r = 1/sqrt(mean(h^2) + eps) of a row, the normed row
// is w*h*r, and (w*h*r) . W^T = r * ((w*h) . W^T): the scalar r can wait until after the
// product.
//   FUSE_RESIDUAL (output projections): h += x . W^T in float32, then the product writes
//       bfloat16(w*h) for the next product and, for every 16 columns, the rows' partial
//       sums of h^2.
//   FUSE_RSTD (the products that read normed rows): x is such a bfloat16(w*h); the rows'
//       partial sums are added in order, and the outputs are scaled by r (before the
//       SwiGLU of a gated matrix).
//   FUSE_SELF (a product that reads normed rows of another's outputs): x are the rows themselves; a wave rounds
//       w*x for its products, adds up the squares of what it reads, and the outputs are scaled by r.  A launch and a trip of the normed
//       rows through memory less.
// Sums, r and the residual are float32 (kernels/src/rmsnorm_kernel_cpu.cpp:27-43); the
// rounding to bfloat16 happens once, as for a separate norm, only before r is applied
// instead of after (a scalar factor does not change the relative rounding error).
#include "common.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any;     // four floats at any multiple of four bytes
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
union Pack16 {
    uint4 u;
    u32x4_t w;
    bf16x8 v;
};

// 16 bytes of a matrix that a step reads once, in the tiled layout (a load instruction of a
// wave takes 1 KiB in a row): a non-temporal load, so that the caches do not keep 16 GB of
// weights a step in place of the little that every kernel begins with (activations, norm
// weights, positions, block tables).  Measured at the Qwen3-8B shape: 3.37 -> 3.13 ms a step at
// batch 8, 13.8k -> 14.5k tokens/s at batch 64.  Not for loads that take a line in pieces:
// the key fragments of the decode attention as non-temporal loads made its step 3% slower.
__device__ __forceinline__ u32x4_t load16_once(const bf16_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
}

__device__ __forceinline__ uint4 load16_or_zero(const bf16_t* p, bool ok) {
    return ok ? *reinterpret_cast<const uint4*>(p) : make_uint4(0, 0, 0, 0);
}

#define FUSE_NONE 0
#define FUSE_RSTD 1
#define FUSE_RESIDUAL 2
#define FUSE_SELF 3

struct SkinnyFuse {
    const float* ssq_in;      // FUSE_RSTD: [parts_in][M] partial sums of squares of the rows of x's source
    int parts_in;
    float eps;
    float* resid;             // FUSE_RESIDUAL: [M][N] float32, updated in place
    const float* norm_w;      // [N] weights of the norm that follows; FUSE_SELF: [K] of the rows' own
    bf16_t* xw;               // [M][N] bfloat16(norm_w * resid)
    float* ssq_out;           // [ceil(N/16)][M]
    GateOut gate;             // of a gated matrix
    InputGroups inputs;
    OutUnit unit;             // of a product without a gate and norm
    int x_ld;                 // FUSE_SELF: elements between two rows of x
};

template <int RT, int MT, int WAVES, typename TO, bool TILED = false, bool GATED = false, int DEPTH = 2,
          int FUSE = FUSE_NONE, int XR = 0, bool WHOLE = false, bool HALF = false>
__global__ void __launch_bounds__(WAVES * 64)
gemm_skinny_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, TO* __restrict__ y,
                   int M, int N, int K, SkinnyFuse fuse) {
    static_assert(XR == 0 || MT == 1, "one tile of rows goes through LDS");
    // HALF: a workgroup takes half a tile, 8 columns (lanes of the other half repeat them), so that twice as many compute
    // units read a matrix of few rows
    static_assert(!HALF || (RT == 1 && MT == 1 && TILED && !GATED), "half a tile of a tiled matrix");
    constexpr int COLS = HALF ? 8 : 16 * RT;
    __shared__ float red[WAVES][RT * MT][64][4];
    __shared__ u32x4_t x_lds[XR ? WAVES : 1][16][16];            // a wave's rows of one step, chunk q of row r at q ^ r
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int r = lane % 16, c = lane / 16;
    const int n_base = blockIdx.x * COLS;
    if constexpr (FUSE == FUSE_NONE && TILED && !GATED) x += fuse.inputs.at(n_base);

    f32x4 acc[RT][MT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // Rows past the end read a valid row instead (w: row 0, x: the last row) and are
    // never stored, so that no load of the main loop is predicated.
    const bf16_t* w_row[RT];
    bool w_ok[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int n = n_base + t * 16 + r;
        w_ok[t] = n < N;
        w_row[t] = w + (size_t)(w_ok[t] ? n : 0) * K;
        // (past an odd number of tiles: the last one again; a gated matrix has pairs of them)
        const int tile = GATED || t == 0 ? blockIdx.x * RT + t : min((int)blockIdx.x * RT + t, (N - 1) / 16);
        if (TILED)   // blocks of 16 rows x 128 k = 4 KiB, stored [j][lane][8]: one load instruction
                     // of a wave reads 1 KiB in a row
            w_row[t] = HALF ? w + ((size_t)(blockIdx.x / 2) * ((K + 127) / 128)) * 2048 + (16 * c + 8 * (blockIdx.x % 2) + r % 8) * 8
                            : w + ((size_t)tile * ((K + 127) / 128)) * 2048 + lane * 8;
    }
    const bf16_t* x_row[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) x_row[m] = x + (size_t)min(m * 16 + r, M - 1) * (FUSE == FUSE_SELF ? fuse.x_ld : K);
    static_assert(FUSE != FUSE_SELF || (MT == 1 && TILED && !GATED && XR == 0), "rows that are normed on their way in");
    constexpr bool SELF = FUSE == FUSE_SELF;
    f32x4 own_w[SELF ? DEPTH : 1][SELF ? 8 : 1];               // the norm's weights of a step's 32 elements
    float own_ssq = 0.f;

    // Ring of DEPTH register stages: the loads of the next DEPTH-1 128-wide steps are in
    // flight while the MFMAs of the current one run, so a wave keeps up to
    // 4*(RT+MT)*(DEPTH-1) 16-byte loads in flight.  The main loop takes whole steps only
    // and none of its loads is under a branch: after a branch that may have issued loads
    // the compiler waits for all loads in flight, which would undo the prefetching.
    Pack16 a[DEPTH][RT][4], b[XR ? 1 : DEPTH][MT][4];
    // XR > 0: x goes through LDS.  A lane asks for 16 bytes of a row that its 15 neighbours go on with (a load instruction
    // takes four rows of 256 bytes), and the operands are read from LDS; straight into the operand registers every load
    // instruction takes 16 bytes from each of 64 places, which keeps the vector cache busy for longer than the weights do.
    u32x4_t x_step[XR ? DEPTH : 1][XR ? XR : 1];
    const bf16_t* x_piece[XR ? XR : 1];
#pragma unroll
    for (int i = 0; i < XR; ++i) x_piece[i] = x + (size_t)min(i * 4 + c, M - 1) * K + r * 8;
    auto load_step = [&](auto STAGE, int kb) {
        constexpr int S = decltype(STAGE)::value;
        const int k = kb + c * 32;
        // x first: it comes from L2 and loads complete in the order of issue
        if constexpr (XR > 0) {
#pragma unroll
            for (int i = 0; i < XR; ++i) x_step[S][i] = *reinterpret_cast<const u32x4_t*>(x_piece[i] + kb);
        } else {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    b[S][m][j].u = *reinterpret_cast<const uint4*>(x_row[m] + k + j * 8);
        }
        if constexpr (SELF) {
#pragma unroll
            for (int q = 0; q < 8; ++q) own_w[S][q] = *reinterpret_cast<const f32x4*>(fuse.norm_w + k + q * 4);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < RT; ++t)
                if (TILED)
                    a[S][t][j].w = load16_once(w_row[t] + (size_t)(kb / 128) * 2048 + j * 512);
                else
                    a[S][t][j].u = *reinterpret_cast<const uint4*>(w_row[t] + k + j * 8);
    };
    auto mma_step = [&](auto STAGE, auto DIRECT) {
        constexpr int S = decltype(STAGE)::value;
        constexpr int B = XR ? 0 : S;
        if constexpr (XR > 0 && !decltype(DIRECT)::value) {
            // (a wave's LDS instructions run in their order: no step overtakes the one before.  Rows from 4 XR on are
            // whatever lies there: they meet no other row's sums and are never stored)
#pragma unroll
            for (int i = 0; i < XR; ++i) x_lds[wave][i * 4 + c][r ^ (i * 4 + c)] = x_step[S][i];
            wave_lds_sync();
#pragma unroll
            for (int j = 0; j < 4; ++j) b[0][0][j].w = x_lds[wave][r][(4 * c + j) ^ r];
            wave_lds_sync();
        }
        if constexpr (SELF) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t two = b[S][0][j].w[e];
                    const float lo = __uint_as_float(two << 16), hi = __uint_as_float(two & 0xFFFF0000u);
                    own_ssq = fmaf(lo, lo, own_ssq);
                    own_ssq = fmaf(hi, hi, own_ssq);
                    b[S][0][j].w[e] = pack_bf16x2(lo * own_w[S][2 * j + e / 2][2 * (e % 2)], hi * own_w[S][2 * j + e / 2][2 * (e % 2) + 1]);
                }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[S][t][j].v, b[B][m][j].v,
                                                                        acc[t][m], 0, 0, 0);
        // keeps the scheduler from moving the loads of the next step (issued after this
        // in program order) ahead of these products, where they would have to be waited
        // for together with the operands used here
        __builtin_amdgcn_sched_barrier(0);
    };
    // this wave's whole steps: number i is at k = (wave + i*WAVES) * 128
    const int whole = K / 128;
    const int mine = wave < whole ? (whole - wave + WAVES - 1) / WAVES : 0;
    auto k_of = [&](int i) { return (wave + i * WAVES) * 128; };
    auto prologue = [&](auto self, auto INDEX) -> void {
        constexpr int I = decltype(INDEX)::value;
        if constexpr (I < DEPTH - 1) {
            if (I < mine) load_step(std::integral_constant<int, I>{}, k_of(I));
            self(self, std::integral_constant<int, I + 1>{});
        }
    };
    // a round: step i + I multiplies stage I after the load of step i + I + DEPTH - 1 went out
    auto round = [&](auto self, int i, auto INDEX, auto FULL_T) -> void {
        constexpr int I = decltype(INDEX)::value;
        constexpr bool FULL = decltype(FULL_T)::value;
        if constexpr (I < DEPTH) {
            if (FULL || i + I < mine) {
                if (FULL || i + I + DEPTH - 1 < mine)
                    load_step(std::integral_constant<int, (I + DEPTH - 1) % DEPTH>{}, k_of(i + I + DEPTH - 1));
                __builtin_amdgcn_sched_barrier(0);
                mma_step(std::integral_constant<int, I>{}, std::false_type{});
                self(self, i, std::integral_constant<int, I + 1>{}, FULL_T);
            }
        }
    };
    prologue(prologue, std::integral_constant<int, 0>{});
    // (asked for behind the first W fragments, needed only after the last)
    // FUSE_RSTD: the partial sums of squares are shared out over the waves and lane groups
    // (part p to wave (p / 4) % WAVES, lane group p % 4), asked for eight at a time without
    // a branch, and added up over the workgroup only after the main loop
    float ssq_mine[MT];
    if (FUSE == FUSE_RSTD) {
        constexpr int STEP = 4 * WAVES;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row = min(m * 16 + r, M - 1);
            float a = 0.f;
            for (int p0 = wave * 4 + c; p0 < fuse.parts_in; p0 += 8 * STEP) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int p = p0 + e * STEP;
                    v[e] = fuse.ssq_in[(size_t)min(p, fuse.parts_in - 1) * M + row] * (p < fuse.parts_in ? 1.f : 0.f);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) a += v[e];
            }
            ssq_mine[m] = quad_rows_sum(a);            // over the four lane groups
        }
    }
    float h_old[4] = {0.f, 0.f, 0.f, 0.f}, nw[4] = {0.f, 0.f, 0.f, 0.f};
    if (FUSE == FUSE_RESIDUAL) {
        static_assert(FUSE != FUSE_RESIDUAL || (MT == 1 && RT <= WAVES), "one tile a wave at most");
        {   // wave t < RT finishes tile t: its residual values and norm weights (the other
            // waves ask for the same as wave 0, which costs nothing and keeps the loads
            // free of branches; rows and columns past the end repeat the last)
            const int n0 = n_base + (wave < RT ? wave : 0) * 16 + (HALF ? c % 2 : c) * 4;
            if constexpr (WHOLE) {                     // rows of whole pieces of four columns: a load each
                const int col = min(n0, N - 4);
                const f32x4 h = *reinterpret_cast<const f32x4*>(fuse.resid + (size_t)min(r, M - 1) * N + col);
                const f32x4_any v = *reinterpret_cast<const f32x4_any*>(fuse.norm_w + col);
#pragma unroll
                for (int e = 0; e < 4; ++e) h_old[e] = h[e], nw[e] = v[e];
            } else
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = min(n0 + e, N - 1);
                h_old[e] = fuse.resid[(size_t)min(r, M - 1) * N + col];
                nw[e] = fuse.norm_w[col];
            }
        }
    }
    int i = 0;
    for (; i + 2 * (DEPTH - 1) < mine; i += DEPTH)
        round(round, i, std::integral_constant<int, 0>{}, std::true_type{});
    for (; i < mine; i += DEPTH)
        round(round, i, std::integral_constant<int, 0>{}, std::false_type{});
    // the last, partial step of k belongs to the wave whose turn it is; it comes after
    // that wave's whole steps, as it would in one loop over all steps
    if (K % 128 && wave == whole % WAVES) {
        const int k = whole * 128 + c * 32;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = k + j * 8 < K;
#pragma unroll
            for (int t = 0; t < RT; ++t)
                a[0][t][j].u = TILED ? *reinterpret_cast<const uint4*>(w_row[t] + (size_t)whole * 2048 + j * 512)
                                     : load16_or_zero(w_row[t] + k + j * 8, in);
#pragma unroll
            for (int m = 0; m < MT; ++m) b[0][m][j].u = load16_or_zero(x_row[m] + k + j * 8, in);
        }
        mma_step(std::integral_constant<int, 0>{}, std::true_type{});
    }

#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[wave][t * MT + m][lane][i] = acc[t][m][i];
    constexpr bool SCALED = FUSE == FUSE_RSTD || SELF;
    if constexpr (SELF) ssq_mine[0] = quad_rows_sum(own_ssq);
    __shared__ float ssq_red[SCALED ? WAVES : 1][MT][16];
    if (SCALED && c == 0) {
#pragma unroll
        for (int m = 0; m < MT; ++m) ssq_red[wave][m][r] = ssq_mine[m];
    }
    __syncthreads();
    float rstd[MT];
    if (SCALED) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float a = 0.f;
            for (int wv = 0; wv < WAVES; ++wv) a += ssq_red[wv][m][r];
            rstd[m] = 1.0f / sqrtf(a / (float)K + fuse.eps);
        }
    }
    if (GATED) {
        // row tiles come in pairs (gate rows, up rows of the same 16 outputs): the
        // epilogue writes silu(gate) * up, N/2 columns (kernels/src/swiglu_kernel_cpu.cpp:20-24)
        const int n_out = N / 2;
        for (int pair = wave; pair < (RT / 2) * MT; pair += WAVES) {
            const int tp = pair / MT, m = pair % MT;
            float g[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
            for (int wv = 0; wv < WAVES; ++wv)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    g[i] += red[wv][(2 * tp) * MT + m][lane][i];
                    u[i] += red[wv][(2 * tp + 1) * MT + m][lane][i];
                }
            const int row = m * 16 + r;
            const int n0 = (blockIdx.x * (RT / 2) + tp) * 16 + c * 4;
            if (FUSE == FUSE_RSTD) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    g[i] *= rstd[m];
                    u[i] *= rstd[m];
                }
            }
            if (row < M) {
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = gate_unit(g[i], u[i], fuse.gate);
                store4(y + (size_t)row * fuse.gate.ld + n0, o, n_out - n0, (fuse.gate.ld & 3) == 0);
            }
        }
        return;
    }
    // tiles are shared out over the waves; each sums the partials in wave order
    for (int tile = wave; tile < RT * MT; tile += WAVES) {
        const int t = tile / MT, m = tile % MT;
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        for (int wv = 0; wv < WAVES; ++wv)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += red[wv][tile][lane][i];
        const int row = HALF && c >= 2 ? M : m * 16 + r;       // (nothing is stored of what a half tile repeats)
        const int n0 = n_base + t * 16 + c * 4;
        if (FUSE == FUSE_RESIDUAL) {
            // (MT == 1 and tile == wave: the values asked for at the start are this tile's)
            float ssq = 0.f, h[4], hw[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h[i] = h_old[i] + s[i];
                hw[i] = nw[i] * h[i];
                if (row < M && n0 + i < N) ssq += h[i] * h[i];
            }
            if (row < M) {
                store4(fuse.resid + (size_t)row * N + n0, h, N - n0, (N & 3) == 0);
                store4(fuse.xw + (size_t)row * N + n0, hw, N - n0, (N & 3) == 0);
            }
            ssq = quad_rows_sum(ssq);                  // over the tile's 16 columns
            if (c == 0 && row < M && (HALF || RT == 1 || n_base + t * 16 < N)) fuse.ssq_out[(size_t)(blockIdx.x * RT + t) * M + row] = ssq;
            continue;
        }
        if (SCALED) {
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] *= rstd[m];
        }
        if (row < M) {
            if constexpr (FUSE == FUSE_NONE && TILED) fuse.unit.apply(s, row, n0, N - n0);
            store4(y + (size_t)row * N + n0, s, N - n0, (N & 3) == 0);
        }
    }
}

// Where the rows of x (up to 16) go through LDS.  It takes a fetch less of 64 places a load instruction and costs a trip through
// LDS in every step, which shows where a wave has few steps and where the matrix alone keeps the memory busy.  Cold weights,
// through LDS and straight into the operand registers, us:
//   into the residual: always.  4,096 columns of k 4,096, 16 rows 9.05 and 9.56; 2,048 of 2,048, 1 row 4.22 and 4.78.
//   half tiles: from k 1,024 on.  256 columns of k 4,096, 8 rows 4.94 and 5.77, of 1,024 2.94 and 3.22, of 512 2.62 and 2.67.
//   a tile a workgroup: 9 to 16 rows of k 1,024 and more.  4,096 columns normed, 16 rows of k 3,072 7.19 and 7.91, of 512 3.71 and
//   3.58; 8 rows of k 2,048 5.65 and 5.51, of 4,096 8.16 and 8.17.
//   two tiles: from k 4,096 on, and float outputs (the logits) from 9 rows on.  24,576 gated columns of k 4,096, 8 rows 31.4 and
//   31.7; 12,288 of 4,096 19.1 and 19.7, 16 rows of 2,048 13.0 and 12.5, of 512 6.77 and 5.65; 32,768 float columns, 8 rows of k
//   2,048 21.9 and 21.6, of 5,120 49.4 and 49.2, 16 rows 50.8 and 51.6.
static bool through_lds(int M, int K, bool two_tiles, bool half, bool float_out) {
    if (half) return K >= 1024;
    return two_tiles ? K >= 4096 && (M > 8 || !float_out) : M > 8 && K >= 1024;
}
// (four, eight or sixteen rows)
#define SKINNY_ROWS(M, LDS, LAUNCH)     \
    if (!(LDS)) { LAUNCH(0); }          \
    else if ((M) <= 4) { LAUNCH(1); }   \
    else if ((M) <= 8) { LAUNCH(2); }   \
    else { LAUNCH(4); }
#define SKINNY_ROWS_16(LDS, LAUNCH)     \
    if (!(LDS)) { LAUNCH(0); }          \
    else { LAUNCH(4); }

template <int RT, int MT, int WAVES>
static int launch_skinny(const bf16_t* x, const bf16_t* w, void* y, int M, int N, int K, int y_dtype,
                         int tiled, const GateOut& gate, const InputGroups& inputs, const OutUnit& unit, hipStream_t s, bool half = false) {
    SkinnyFuse plain{};
    plain.unit = unit;
    plain.gate = gate;
    plain.inputs = inputs;
    const int blocks = (N + 16 * RT - 1) / (16 * RT);
    constexpr bool CAN_HALF = RT == 1 && MT == 1;
    if constexpr (CAN_HALF) {
        if (half && tiled == 1) {
#define SKINNY_HALF(TO, XR) \
    gemm_skinny_kernel<1, 1, WAVES, TO, true, false, 2, FUSE_NONE, XR, false, true><<<(N + 7) / 8, WAVES * 64, 0, s>>>(x, w, (TO*)y, M, N, K, plain)
#define SKINNY_HALF_BF16(XR) SKINNY_HALF(bf16_t, XR)
#define SKINNY_HALF_F32(XR) SKINNY_HALF(float, XR)
            const bool lds = through_lds(M, K, false, true, false);
            if (y_dtype == TLI_BF16) SKINNY_ROWS(M, lds, SKINNY_HALF_BF16)
            else SKINNY_ROWS(M, lds, SKINNY_HALF_F32)
            return tli_check_launch("gemm_skinny");
        }
    }
#define SKINNY_LAUNCH(TO, TILED, GATED, XR) \
    gemm_skinny_kernel<RT, MT, WAVES, TO, TILED, GATED, 2, FUSE_NONE, XR><<<blocks, WAVES * 64, 0, s>>>(x, w, (TO*)y, M, N, K, plain)
#define SKINNY_GATED(XR) SKINNY_LAUNCH(bf16_t, true, true, XR)
#define SKINNY_BF16(XR) SKINNY_LAUNCH(bf16_t, true, false, XR)
#define SKINNY_F32(XR) SKINNY_LAUNCH(float, true, false, XR)
    if constexpr (MT == 1) {
        const bool lds = through_lds(M, K, RT == 2, false, y_dtype != TLI_BF16);
        if (tiled == 2) SKINNY_ROWS(M, lds, SKINNY_GATED)       // pairs of row tiles, silu(gate)*up written as bfloat16
        else if (tiled && y_dtype == TLI_BF16) {
            if constexpr (RT == 2) SKINNY_ROWS(M, lds, SKINNY_BF16)
            else SKINNY_ROWS_16(lds, SKINNY_BF16)
        } else if (tiled) SKINNY_ROWS_16(lds, SKINNY_F32)
        else if (y_dtype == TLI_BF16) SKINNY_LAUNCH(bf16_t, false, false, 0);
        else SKINNY_LAUNCH(float, false, false, 0);
    } else {
        if (tiled == 2) SKINNY_GATED(0);
        else if (tiled && y_dtype == TLI_BF16) SKINNY_BF16(0);
        else if (tiled) SKINNY_F32(0);
        else if (y_dtype == TLI_BF16) SKINNY_LAUNCH(bf16_t, false, false, 0);
        else SKINNY_LAUNCH(float, false, false, 0);
    }
    return tli_check_launch("gemm_skinny");
}

// Half tiles where whole ones leave half of the chip or more without a workgroup.  Cold weights, 8 rows, whole and half: 64
// columns of k 2,048 3.68 and 3.46 us, 256 of 4,096 5.16 and 4.64, 768 of 6,144 7.51 and 6.64; 1 and 16 rows gain as much.
// Not where k is shorter than the columns are many, or than two steps: 2,048 columns of k 512 2.97 and 3.06, normed 3.31 and
// 3.55, 256 of 128 2.14 and 2.26.  Into the residual only from 1,024 columns on (each half tile leaves sums of squares that the
// next product adds up), there of every k: 2,048 columns of k 256 3.41 and 3.21.
static bool half_tiles(int M, int N, int K, int tiled, bool into_residual) {
    if (M > 16 || tiled != 1 || (N + 15) / 16 > tli_compute_units() / 2) return false;
    return into_residual ? N >= 1024 && N % 4 == 0 : K >= N && K >= 256;
}

// The launch shape (row tiles * 10 + waves) of up to 16 rows.  One tile of 16 columns a workgroup while that gives no more than a workgroup a
// compute unit, two up to twice as many columns (x is read half as often), two by four waves from four times on.  In between two tiles and
// eight waves leave a second round of workgroups to a part of the chip, and smaller workgroups share it out better.  Cold weights, us,
// 28, 14, 18 and 24: 9,216 columns of k 2,048, 1 row 10.9, 9.6, 9.8 and 10.2, of 4,096 18.2, 16.9, 16.1 and 18.4; 11,264 columns, 6 rows 11.8,
// 10.6, 11.4 and 11.2, of 4,096 20.4, 18.7, 18.3 and 20.9, 16 rows 13.0, 12.5, 12.4 and 12.6; 12,288 12.5, 10.9, 12.3 and 11.6; 14,336
// columns, 6 rows 13.0, 13.0, 13.2 and 12.2, of 5,120 24 is 1.8% behind 28.  Gated products, whose tiles come in pairs, stay with 28: 24 is 1 to
// 4% behind.  Row-major matrices (tiled 0) stay with it outside 9 to 12 tiles for four compute units, 28 and the rule's other shape, us: 8,208 columns of k 5,120, 6
// and 16 rows 23.8, 23.6 and 28.2, 30.3; 9,216 26.8, 21.7 (1 row) and 33.6, 32.6; 12,288 30.8, 27.8 and 35.4, 35.6; 14,336 of 2,048 15.1, 15.4 and 17.5, 17.4.
static int wide_shape(int N, int K, int tiled) {
    const long tiles = (N + 15) / 16, units = tli_compute_units();
    const bool shorter = K < 4096, pairs = tiled == 2 || (tiled == 0 && (tiles < 2 * units + units / 4 || tiles > 3 * units));
    if (tiles <= units) return 18;
    if (tiles <= 2 * units || pairs || (tiles > 3 * units && !shorter)) return tiles < 4 * units ? 28 : 24;
    return tiles > 3 * units ? 24 : shorter ? 14 : 18;
}

template <int MT>
static int pick_skinny(const bf16_t* x, const bf16_t* w, void* y, int M, int N, int K, int y_dtype,
                       int tiled, const GateOut& gate, const InputGroups& inputs, const OutUnit& unit, hipStream_t s, int cfg) {
    // cfg 0: by shape.  Narrow outputs get one 16-column tile per workgroup so that
    // even N = 4096 gives 256 workgroups; wide outputs share x over two tiles.
    const long tiles = (N + 15) / 16;
    if (cfg == 0 && MT == 1) cfg = half_tiles(M, N, K, tiled, false) ? 8 : wide_shape(N, K, tiled);
    if (cfg == 0) cfg = tiles <= tli_compute_units() ? 18 : (tiles < 4 * tli_compute_units() ? 28 : 24);
    if (tiled == 2 && cfg < 20) cfg = 24;          // gated needs pairs of row tiles
    switch (cfg) {
        case 14: return launch_skinny<1, MT, 4>(x, w, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s);
        case 18: return launch_skinny<1, MT, 8>(x, w, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s);
        case 8: return launch_skinny<1, MT, 8>(x, w, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s, true);
        case 24: return launch_skinny<2, MT, 4>(x, w, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s);
        case 28: return launch_skinny<2, MT, 8>(x, w, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s);
        default: return tli_fail("gemm_skinny: unknown configuration %d", cfg);
    }
}

static int skinny(const void* x, const void* w, void* y, int M, int N, int K, int y_dtype, int tiled, int cfg, int act,
                  float act_scale, int y_ld, const InputGroups& inputs, const OutUnit& unit, void* stream) {
    const GateOut gate = gate_out(tiled == 2, act, act_scale, y_ld, N / 2);
    if (const char* fault = gate_out_fault(gate, N / 2)) return tli_fail("gemm_skinny: %s", fault);
    if (M <= 0 || N <= 0) return 0;
    if (M > 64) return tli_fail("gemm_skinny: %d rows, at most 64", M);
    if (K <= 0 || K % 8) return tli_fail("gemm_skinny: K = %d must be a positive multiple of 8", K);
    if (y_dtype != TLI_BF16 && y_dtype != TLI_F32) return tli_fail("gemm_skinny: bad output dtype %d", y_dtype);
    if (tiled < 0 || tiled > 2) return tli_fail("gemm_skinny: bad layout code %d", tiled);
    if (tiled == 2 && (N % 32 || y_dtype != TLI_BF16))
        return tli_fail("gemm_skinny: a gated product needs N %% 32 == 0 and bfloat16 output");
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) return tli_fail("gemm_skinny: operands must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* xp = (const bf16_t*)x;
    const bf16_t* wp = (const bf16_t*)w;
    switch ((M + 15) / 16) {
        case 1: return pick_skinny<1>(xp, wp, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s, cfg);
        case 2: return pick_skinny<2>(xp, wp, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s, cfg);
        case 3: return pick_skinny<3>(xp, wp, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s, cfg);
        default: return pick_skinny<4>(xp, wp, y, M, N, K, y_dtype, tiled, gate, inputs, unit, s, cfg);
    }
}

// y[M,N] = x[M,K] . W^T.  `tiled` = 0: w is W[N,K] row-major.  `tiled` = 1: w is the
// same matrix in blocks of 16 rows x 128 columns, zero-padded to whole blocks, stored
// [row block][column block][j = 0..3][lane = 16*c + r][8] with element
// W[16*row block + r][128*column block + 32*c + 8*j + e]: every load instruction of
// a wave then reads 1 KiB in a row.  `tiled` = 2: tiled, and the 16-row blocks alternate
// between a gate matrix and an up matrix (block 2t: gate rows 16t.., block 2t+1: up rows
// 16t..); N counts both, y is [M, N/2] bfloat16 = silu(x.gate^T) * (x.up^T).  cfg 0 picks the launch shape; other values
// (row tiles * 10 + waves) force one, for measurements.  act, act_scale, y_ld: the output of a gated product (common.h's
// GateOut: another activation than the silu, a factor, rows y_ld elements apart; y_ld 0: N/2).
extern "C" int tli_gemm_skinny_bf16(const void* x, const void* w, void* y, int M, int N, int K,
                                    int y_dtype, int tiled, int cfg, int act, float act_scale, int y_ld, void* stream) {
    return skinny(x, w, y, M, N, K, y_dtype, tiled, cfg, act, act_scale, y_ld, InputGroups{0, 0}, no_unit(), stream);
}

// The same, tiled and without a gate, of stacked matrices whose inputs differ (common.h's InputGroups; every in 32s).
extern "C" int tli_gemm_skinny_groups_bf16(const void* x, const void* w, void* y, int M, int N, int K, int y_dtype, int every,
                                           long long step, void* stream) {
    if (every <= 0 || every % 32 || step < (long long)M * K || step % 8) return tli_fail("gemm_skinny: bad input groups");
    return skinny(x, w, y, M, N, K, y_dtype, 1, 0, 0, 1.0f, 0, InputGroups{every, step}, no_unit(), stream);
}

// The same, tiled, without a gate and bfloat16, its outputs through common.h's OutUnit.
extern "C" int tli_gemm_skinny_unit_bf16(const void* x, const void* w, void* y, int M, int N, int K, int kind, const void* table,
                                         const int* ids, int width, int vocab, void* stream) {
    const OutUnit unit{kind, (const bf16_t*)table, ids, width, vocab};
    if (const char* fault = out_unit_fault(unit, N)) return tli_fail("gemm_skinny: %s", fault);
    return skinny(x, w, y, M, N, K, TLI_BF16, 1, 0, 0, 1.0f, 0, InputGroups{0, 0}, unit, stream);
}

template <int RT, int WAVES>
static int launch_skinny_fused(const bf16_t* x, const bf16_t* w, bf16_t* y, int M, int N, int K, int gated,
                               const SkinnyFuse& f, hipStream_t s, bool half = false) {
    const int blocks = (N + 16 * RT - 1) / (16 * RT);
#define SKINNY_FUSED(GATED, FUSE, XR, ...) \
    gemm_skinny_kernel<RT, 1, WAVES, bf16_t, true, GATED, 2, FUSE, XR, ##__VA_ARGS__><<<blocks, WAVES * 64, 0, s>>>(x, w, y, M, N, K, f)
#define SKINNY_RESIDUAL(XR) SKINNY_FUSED(false, FUSE_RESIDUAL, XR)
#define SKINNY_RESIDUAL_WHOLE(XR) SKINNY_FUSED(false, FUSE_RESIDUAL, XR, true)
#define SKINNY_RSTD_GATED(XR) SKINNY_FUSED(true, FUSE_RSTD, XR)
#define SKINNY_RSTD(XR) SKINNY_FUSED(false, FUSE_RSTD, XR)
#define SKINNY_RESIDUAL_HALF(XR) \
    gemm_skinny_kernel<1, 1, WAVES, bf16_t, true, false, 2, FUSE_RESIDUAL, XR, true, true><<<(N + 7) / 8, WAVES * 64, 0, s>>>(x, w, y, M, N, K, f)
#define SKINNY_RSTD_HALF(XR) \
    gemm_skinny_kernel<1, 1, WAVES, bf16_t, true, false, 2, FUSE_RSTD, XR, false, true><<<(N + 7) / 8, WAVES * 64, 0, s>>>(x, w, y, M, N, K, f)
    const bool lds = f.resid || through_lds(M, K, RT == 2, half, false);
    if constexpr (RT == 1) {
        if (half) {
            if (f.resid) SKINNY_ROWS(M, true, SKINNY_RESIDUAL_HALF)
            else SKINNY_ROWS(M, lds, SKINNY_RSTD_HALF)
            return tli_check_launch("gemm_skinny (norm taken in)");
        }
    }
    if (f.resid && N % 4 == 0) SKINNY_ROWS(M, true, SKINNY_RESIDUAL_WHOLE)
    else if (f.resid) SKINNY_ROWS(M, true, SKINNY_RESIDUAL)
    else if (gated) SKINNY_ROWS(M, lds, SKINNY_RSTD_GATED)
    else if constexpr (RT == 2) SKINNY_ROWS(M, lds, SKINNY_RSTD)
    else SKINNY_ROWS_16(lds, SKINNY_RSTD)
    return tli_check_launch("gemm_skinny (norm taken in)");
}

// The launch shape `cfg` of the product with a norm taken in (0: by the sizes), and whether it takes half tiles.
static int fused_shape(int M, int N, int K, int gated, bool into_residual, int cfg) {
    const long tiles = (N + 15) / 16;
    if (cfg == 0 && !into_residual) cfg = !gated && half_tiles(M, N, K, 1, false) ? 8 : wide_shape(N, K, gated ? 2 : 1);
    if (cfg == 0) cfg = half_tiles(M, N, K, 1, true) ? 8 : tiles <= tli_compute_units() ? 18 : (tiles < 4 * tli_compute_units() ? 28 : 24);
    return gated && cfg < 20 ? 24 : cfg;
}

// How many partial sums of squares a row has after a product into the residual: one for every 8 or 16 columns.
extern "C" int tli_gemm_skinny_parts(int M, int N, int cfg) { return fused_shape(M, N, 0, 0, true, cfg) == 8 ? (N + 7) / 8 : (N + 15) / 16; }

// The product with a norm taken in (see the top of this file), for up to 16 rows and W in the
// decode layout.  Either  resid != null:  resid[M,N] += x . W^T (float32), xw[M,N] =
// bfloat16(norm_w * resid), ssq_out[tli_gemm_skinny_parts(M, N, cfg)][M] = partial sums of resid^2 (y is not used);
// or  ssq_in != null:  y = (x . W^T) / sqrt(sum(ssq_in[parts_in][M]) / K + eps), through the
// SwiGLU of a gated matrix if `gated` (y then [M, N/2]).
extern "C" int tli_gemm_skinny_fused_bf16(const void* x, const void* w, void* y, int M, int N, int K, int gated,
                                          const float* ssq_in, int parts_in, float eps, float* resid,
                                          const float* norm_w, void* xw, float* ssq_out, int cfg, int act, float act_scale,
                                          int y_ld, void* stream) {
    const GateOut gate = gate_out(gated, act, act_scale, y_ld, N / 2);
    if (const char* fault = gate_out_fault(gate, N / 2)) return tli_fail("gemm_skinny: %s", fault);
    if (M <= 0 || N <= 0) return 0;
    if (M > 16) return tli_fail("gemm_skinny with a norm: %d rows, at most 16", M);
    if (K <= 0 || K % 8) return tli_fail("gemm_skinny: K = %d must be a positive multiple of 8", K);
    if ((resid != nullptr) == (ssq_in != nullptr))
        return tli_fail("gemm_skinny with a norm: give either the residual to add into or the sums of squares of x");
    if (resid && (gated || !norm_w || !xw || !ssq_out)) return tli_fail("gemm_skinny into the residual: missing arguments");
    if (ssq_in && (parts_in <= 0 || !y)) return tli_fail("gemm_skinny with sums of squares: missing arguments");
    if (gated && N % 32) return tli_fail("gemm_skinny: a gated product needs N %% 32 == 0");
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)resid | (uintptr_t)xw) & 15)
        return tli_fail("gemm_skinny: operands must be 16-byte aligned");
    const SkinnyFuse f{ssq_in, parts_in, eps, resid, norm_w, (bf16_t*)xw, ssq_out, gate};
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* xp = (const bf16_t*)x;
    const bf16_t* wp = (const bf16_t*)w;
    cfg = fused_shape(M, N, K, gated, resid != nullptr, cfg);
    if (cfg == 8 && resid && N % 4) return tli_fail("gemm_skinny: half tiles into a residual of %d columns (a multiple of 4)", N);
    switch (cfg) {
        case 14: return launch_skinny_fused<1, 4>(xp, wp, (bf16_t*)y, M, N, K, gated, f, s);
        case 18: return launch_skinny_fused<1, 8>(xp, wp, (bf16_t*)y, M, N, K, gated, f, s);
        case 8: return launch_skinny_fused<1, 8>(xp, wp, (bf16_t*)y, M, N, K, gated, f, s, true);
        case 24: return launch_skinny_fused<2, 4>(xp, wp, (bf16_t*)y, M, N, K, gated, f, s);
        case 28: return launch_skinny_fused<2, 8>(xp, wp, (bf16_t*)y, M, N, K, gated, f, s);
        default: return tli_fail("gemm_skinny: unknown configuration %d", cfg);
    }
}

// The same with float32 outputs (the logits of a step): y = (x . W^T) / sqrt(sum(ssq_in[parts_in][M]) / K + eps).  The launch shape is
// that of tli_gemm_skinny_bf16 with float32 outputs.  A decode step then has no pass for its last norm (8 rows of 4,096: 4.7 us).
// Last product, norm and head apart and so, us: 32,768 outputs of 4,096, 1 row 62.4 and 59.2, 8 rows 61.4 and 58.4, 16 rows 63.9 and 61.8; 151,936
// outputs 204.9 and 204.1, 204.4 and 203.2, 216.2 and 216.7; of 5,120 263.8 and 263.6, 261.3 and 262.1, 281.4 and 283.0.
template <int RT, int WAVES>
static int launch_skinny_normed_f32(const bf16_t* x, const bf16_t* w, float* y, int M, int N, int K, const SkinnyFuse& f, hipStream_t s,
                                    bool half = false) {
    const int blocks = (N + 16 * RT - 1) / (16 * RT);
    const bool lds = through_lds(M, K, RT == 2, half, true);
#define SKINNY_NORMED_F32(XR) \
    gemm_skinny_kernel<RT, 1, WAVES, float, true, false, 2, FUSE_RSTD, XR><<<blocks, WAVES * 64, 0, s>>>(x, w, y, M, N, K, f)
#define SKINNY_NORMED_F32_HALF(XR) \
    gemm_skinny_kernel<1, 1, WAVES, float, true, false, 2, FUSE_RSTD, XR, false, true><<<(N + 7) / 8, WAVES * 64, 0, s>>>(x, w, y, M, N, K, f)
    if constexpr (RT == 1) {
        if (half) {
            SKINNY_ROWS(M, lds, SKINNY_NORMED_F32_HALF)
            return tli_check_launch("gemm_skinny (norm taken in, float32)");
        }
    }
    SKINNY_ROWS_16(lds, SKINNY_NORMED_F32)
    return tli_check_launch("gemm_skinny (norm taken in, float32)");
}

extern "C" int tli_gemm_skinny_normed_f32(const void* x, const void* w, void* y, int M, int N, int K, const float* ssq_in, int parts_in,
                                          float eps, void* stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16) return tli_fail("gemm_skinny with a norm: %d rows, at most 16", M);
    if (K <= 0 || K % 8) return tli_fail("gemm_skinny: K = %d must be a positive multiple of 8", K);
    if (!ssq_in || parts_in <= 0 || !y) return tli_fail("gemm_skinny with sums of squares: missing arguments");
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) return tli_fail("gemm_skinny: operands must be 16-byte aligned");
    SkinnyFuse f{};
    f.ssq_in = ssq_in, f.parts_in = parts_in, f.eps = eps;
    const bf16_t *xp = (const bf16_t*)x, *wp = (const bf16_t*)w;
    hipStream_t s = (hipStream_t)stream;
    switch (fused_shape(M, N, K, 0, false, 0)) {
        case 8: return launch_skinny_normed_f32<1, 8>(xp, wp, (float*)y, M, N, K, f, s, true);
        case 14: return launch_skinny_normed_f32<1, 4>(xp, wp, (float*)y, M, N, K, f, s);
        case 18: return launch_skinny_normed_f32<1, 8>(xp, wp, (float*)y, M, N, K, f, s);
        case 28: return launch_skinny_normed_f32<2, 8>(xp, wp, (float*)y, M, N, K, f, s);
        default: return launch_skinny_normed_f32<2, 4>(xp, wp, (float*)y, M, N, K, f, s);
    }
}

// y[M,N] = norm(x) . W^T for rows that are part of wider ones: x [M, K], rows x_ld elements apart, the RMS norm over K with weights norm_w [K].
// Up to 16 rows, W in the decode layout, k in whole steps of 128.  Every workgroup reads all rows anyway and does their arithmetic again, 100 vector
// instructions a step beside loads that it waits for; the launch of norm_rows is saved.  Norm and product apart and so, in a recorded
// chain, us: 3,072 columns of k 1,024, 1 row 5.3 and 4.2, 8 rows 5.7 and 4.3, 16 rows 5.8 and 4.3; of 1,536, 8 rows 6.5 and 5.1; of 2,048, 8 rows 7.2 and
// 6.4.  The arithmetic is as long as the launch where a wave has more of it than W's loads hide: k beyond 2,048 (8 rows, k 4,096: 256 columns
// 7.8 and 8.9, 12,288 22.5 and 27.1) and, from more columns on than two tiles a compute unit, beyond 1,024 (12,288 of 2,048 13.4 and 14.5, of 1,024 9.1 and
// 8.8; 24,576 of 1,536 16.0 and 16.0).
extern "C" int tli_gemm_skinny_self_takes(int M, int N, int K) {
    return M > 0 && M <= 16 && N > 0 && K > 0 && K % 128 == 0 && (K <= 1024 || (K <= 2048 && (N + 15) / 16 <= 2 * tli_compute_units()));
}
extern "C" int tli_gemm_skinny_self_bf16(const void* x, int x_ld, const void* w, void* y, int M, int N, int K, const float* norm_w, float eps,
                                         void* stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 16) return tli_fail("gemm_skinny with a norm: %d rows, at most 16", M);
    if (K <= 0 || K % 128 || x_ld < K || x_ld % 8) return tli_fail("gemm_skinny with a norm of its own rows: K = %d, rows %d apart", K, x_ld);
    if (!norm_w || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)norm_w) & 15))
        return tli_fail("gemm_skinny: operands must be 16-byte aligned");
    SkinnyFuse f{};
    f.norm_w = norm_w, f.eps = eps, f.x_ld = x_ld;
    const bf16_t *xp = (const bf16_t*)x, *wp = (const bf16_t*)w;
    bf16_t* yp = (bf16_t*)y;
    hipStream_t s = (hipStream_t)stream;
#define SKINNY_SELF(RT, WAVES, HALF)                                                                                              \
    gemm_skinny_kernel<RT, 1, WAVES, bf16_t, true, false, 2, FUSE_SELF, 0, false, HALF>                                             \
        <<<(N + (HALF ? 8 : 16 * RT) - 1) / (HALF ? 8 : 16 * RT), WAVES * 64, 0, s>>>(xp, wp, yp, M, N, K, f)
    switch (fused_shape(M, N, K, 0, false, 0)) {
        case 8: SKINNY_SELF(1, 8, true); break;
        case 14: SKINNY_SELF(1, 4, false); break;
        case 18: SKINNY_SELF(1, 8, false); break;
        case 28: SKINNY_SELF(2, 8, false); break;
        default: SKINNY_SELF(2, 4, false); break;
    }
#undef SKINNY_SELF
    return tli_check_launch("gemm_skinny (norm of its own rows)");
}
