// Matrix product of the float32 path: y[M,N] = x[M,K] . W[N,K]^T, everything float32, on the matrix cores' float32
// instruction (v_mfma_f32_16x16x4_f32: float32 products and sums, 157 TFLOP/s against the vector units' same
// rate but with a sixteenth of the operand reads), W row-major as it is held.  K must be a multiple of 4.
//
// A row's result does not depend on the number of rows beside it: k goes to the eight waves of a workgroup in eight
// ranges that depend on K alone, every range is summed in the same order whatever the tiles, and the ranges are
// added in their order.
//
// What bounds it: for few rows the reading of W (4 bytes an element once, straight into the operand registers, no LDS:
// every wave owns its range of k, so nothing is read twice in a workgroup but x); from about 48 rows on the matrix cores.
// Lane l holds A[l%16][l/16], B[l/16][l%16], D[(l/16)*4 .. +4][l%16] of a 16 x 16 x 4 product.  The four k of a product may
// be any as long as A and B agree: lane group c = l/16 takes four k in a row, [kb + 4c, kb + 4c + 4), one 16-byte load that
// serves four products, so that a row of W is read in pieces of 64 bytes, the next piece by the next load.
//
// Measured with 1 to 5 rows at width 1,024 (the tiled kernel of the vector units in gemm_plain.hip, which walks k with one
// load in flight, before): q/k/v (6.3 MB) 156 -> 5.8 us, output and down projection (4.2 and 16.8 MB) 378 -> 9.8 us on
// average (5.2 where the reader adds the ranges' sums, see gemm_f32_ranges_kernel), gate/up with its activation (33.6 MB) 160 ->
// 10 us, the head (134 MB) 201 -> 29 us = 4.6 TB/s.  Error against float64 of the logits of four layers 2.9e-6 -> 1.1e-6.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define GF_RANGES 8

// acc[t][m] += the products of `count` steps of 16 k from step `first` on; w_row and x_row point at this lane's four k of step 0.
// U steps are asked for together, the next U while these are multiplied.
template <int RT, int MT, int U>
__device__ __forceinline__ void add_range(f32x4 (&acc)[RT][MT], const float* const (&w_row)[RT], const float* const (&x_row)[MT], int first,
                                          int count, int K, int c) {
    // the last step of k may be partial: it is left to the end, where loads are looked after one by one
    const int whole = min(count, max(0, K / 16 - first));
    const int batches = whole / U;

    f32x4 a[2][U][RT], b[2][U][MT];
    auto load = [&](int s, int batch) __attribute__((always_inline)) {
        const int kb = (first + batch * U) * 16;
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int m = 0; m < MT; ++m) b[s][u][m] = *reinterpret_cast<const f32x4*>(x_row[m] + kb + u * 16);
#pragma unroll
            for (int t = 0; t < RT; ++t) a[s][u][t] = *reinterpret_cast<const f32x4*>(w_row[t] + kb + u * 16);
        }
    };
    auto multiply = [&](int s, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][u][t][j], b[s][u][m][j], acc[t][m], 0, 0, 0);
    };
    auto multiply_all = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) multiply(s, u);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (batches > 0) {
        load(0, 0);
        int i = 0;
        for (; i + 2 < batches; i += 2) {
            load(1, i + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply_all(0);
            load(0, i + 2);
            __builtin_amdgcn_sched_barrier(0);
            multiply_all(1);
        }
        if (i + 1 < batches) {
            load(1, i + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply_all(0);
            multiply_all(1);
        } else {
            multiply_all(0);
        }
    }
    for (int s = batches * U; s < count; ++s) {
        const int k = (first + s) * 16;
        const bool in = k + c * 4 < K;                         // (K is a multiple of 4)
        const f32x4 zero = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < MT; ++m) b[0][0][m] = in ? *reinterpret_cast<const f32x4*>(x_row[m] + k) : zero;
#pragma unroll
        for (int t = 0; t < RT; ++t) a[0][0][t] = in ? *reinterpret_cast<const f32x4*>(w_row[t] + k) : zero;
        multiply(0, 0);
    }
}

// RT tiles of 16 rows of W and MT tiles of 16 rows of x a workgroup; U steps of 16 k are asked for together, the next U
// while these are multiplied.  GATED: W holds N gate rows, then N up rows; tiles come in pairs of both and y is
// act(gate) * up * scale.
// CT < 16 (one tile of W): a workgroup takes CT of a tile's 16 columns, its lanes of the others repeating them, so that a matrix
// of few rows is read by more compute units.
template <int RT, int MT, int U, bool GATED, int CT = 16>
__global__ void __launch_bounds__(GF_RANGES * 64)
gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ y, int M, int N, int K,
                GateOut gate) {
    constexpr int TOGETHER = GATED ? 2 : 1;                    // row tiles that are finished together
    __shared__ float red[GF_RANGES][TOGETHER * MT][64][4];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int r = lane % 16, c = lane / 16;
    static_assert(CT == 16 || RT == 1, "part of one tile");
    const int n_base = blockIdx.x * (CT == 16 ? 16 * RT / TOGETHER : CT), m_base = blockIdx.y * (16 * MT);

    f32x4 acc[RT][MT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = (f32x4){0.f, 0.f, 0.f, 0.f};

    // rows past the end read a valid one and are never stored
    const float* w_row[RT];
    const float* x_row[MT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int n = min(n_base + (t / TOGETHER) * 16 + r % CT, N - 1);
        w_row[t] = w + (size_t)(n + (GATED && (t & 1) ? N : 0)) * K + c * 4;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) x_row[m] = x + (size_t)min(m_base + m * 16 + r, M - 1) * K + c * 4;

    const int steps = (K + 15) / 16, each = (steps + GF_RANGES - 1) / GF_RANGES;
    const int first = min(wave * each, steps), count = min(steps - first, each);
    add_range<RT, MT, U>(acc, w_row, x_row, first, count, K, c);

#pragma unroll
    for (int t0 = 0; t0 < RT; t0 += TOGETHER) {
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < TOGETHER; ++t)
#pragma unroll
            for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(red[wave][t * MT + m][lane]) = acc[t0 + t][m];
        __syncthreads();
        if (wave < MT) {
            const int row = m_base + wave * 16 + r, n0 = n_base + (t0 / TOGETHER) * 16 + c * 4;
            float s[TOGETHER][4];
#pragma unroll
            for (int t = 0; t < TOGETHER; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    s[t][e] = 0.f;
                    for (int range = 0; range < GF_RANGES; ++range) s[t][e] += red[range][t * MT + wave][lane][e];
                }
            if (row < M && n0 < N && c * 4 < CT) {
                if constexpr (GATED) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[0][e] = gate_unit(s[0][e], s[1][e], gate);
                }
                const int ld = GATED ? gate.ld : N;
                store4(y + (size_t)row * ld + n0, s[0], N - n0, (ld & 3) == 0 && ((uintptr_t)y & 15) == 0);
            }
        }
    }
}

// The ranges' sums themselves, [range][M][N], for a reader that adds them in the ranges' order (the same bits as the kernel above): a wave
// a tile of 16 columns and range, GF_PART_WAVES tiles of a range a workgroup, whose waves share the pieces of x that they read.
// What it is for: 1,024 columns are 64 tiles, which the kernel above reaches all compute units with only by giving a workgroup a quarter of
// one, so that three quarters of its matrix instructions and loads repeat.  Here the tiles' eight ranges are 512 waves that repeat nothing,
// wait for no other wave, and have two batches of eight steps in flight, up to k of 2,048 all of their loads.  What bounds it: the launch and, up to
// there, one trip to memory; beyond, the loads follow behind the products: 4,096 k (four batches) 3.1 TB/s, a wave's 128 instructions of 32 cycles
// one after the other.
// Measured in a recorded chain, cold weights, us, with the norm that adds the sums against the kernel above and the norm: 5 rows, 1,024 columns of
// k 1,024 7.5 -> 6.0, of 4,096 15.5 -> 8.5; 16 rows 8.6 -> 6.3, 19.4 -> 9.5; 32 rows 10.8 -> 7.2, 26.8 -> 12.4; 1,536 of 1,024 alone 5.4 -> 4.1 (5 rows)
// and 8.8 -> 6.1 (32).  Non-temporal loads of W are no faster.
#define GF_PART_WAVES 2
template <int MT, int U>
__global__ void __launch_bounds__(GF_PART_WAVES * 64)
gemm_f32_ranges_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ parts, int M, int N, int K) {
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int r = lane % 16, c = lane / 16;
    const int n_base = (blockIdx.x * GF_PART_WAVES + wave) * 16, range = blockIdx.y;
    if (n_base >= N) return;
    f32x4 acc[1][MT];
    const float* w_row[1] = {w + (size_t)min(n_base + r, N - 1) * K + c * 4};       // rows past the end read a valid one and are never stored
    const float* x_row[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        acc[0][m] = (f32x4){0.f, 0.f, 0.f, 0.f};
        x_row[m] = x + (size_t)min(m * 16 + r, M - 1) * K + c * 4;
    }
    const int steps = (K + 15) / 16, each = (steps + GF_RANGES - 1) / GF_RANGES;
    const int first = min(range * each, steps), count = min(steps - first, each);
    add_range<1, MT, U>(acc, w_row, x_row, first, count, K, c);
    const int n0 = n_base + c * 4;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = m * 16 + r;
        if (row >= M || n0 >= N) continue;
        const float s[4] = {acc[0][m][0], acc[0][m][1], acc[0][m][2], acc[0][m][3]};
        store4(parts + ((size_t)range * M + row) * N + n0, s, N - n0, N % 4 == 0);
    }
}

template <int MT, int U, int CT>
static int launch_f32_part(const float* x, const float* w, float* y, int M, int N, int K, const GateOut& gate, hipStream_t s) {
    gemm_f32_kernel<1, MT, U, false, CT><<<dim3((N + CT - 1) / CT, (M + 16 * MT - 1) / (16 * MT)), GF_RANGES * 64, 0, s>>>(x, w, y, M, N, K, gate);
    return tli_check_launch("gemm_f32");
}

template <int RT, int MT, int U>
static int launch_f32(const float* x, const float* w, float* y, int M, int N, int K, const GateOut& gate, hipStream_t s) {
    constexpr int COLS = 16 * RT;
    const dim3 grid((N + (gate.on ? COLS / 2 : COLS) - 1) / (gate.on ? COLS / 2 : COLS), (M + 16 * MT - 1) / (16 * MT));
    if (grid.y > 65535) return tli_fail("gemm_f32: %d rows exceed the grid limit", M);
    if (gate.on) {
        if constexpr (RT > 1) gemm_f32_kernel<RT, MT, U, true><<<grid, GF_RANGES * 64, 0, s>>>(x, w, y, M, N, K, gate);
    } else {
        gemm_f32_kernel<RT, MT, U, false><<<grid, GF_RANGES * 64, 0, s>>>(x, w, y, M, N, K, gate);
    }
    return tli_check_launch("gemm_f32");
}

// y[M,N] = x[M,K] . w[N,K]^T in float32; gated: w is [2 N, K], gate rows before up rows, and y[M, y_ld] takes
// act(gate) * up * act_scale (y_ld 0: N).
extern "C" int tli_gemm_f32(const void* x, const void* w, void* y, int M, int N, int K, int gated, int act, float act_scale,
                            int y_ld, void* stream) {
    const GateOut gate = gate_out(gated, act, act_scale, y_ld, N);
    if (const char* fault = gate_out_fault(gate, N)) return tli_fail("gemm_f32: %s", fault);
    if (M <= 0 || N <= 0) return 0;
    if (K <= 0 || K % 4) return tli_fail("gemm_f32: K = %d must be a positive multiple of 4", K);
    if (((uintptr_t)x | (uintptr_t)w) & 15) return tli_fail("gemm_f32: operands must be 16-byte aligned");
    const float *xp = (const float*)x, *wp = (const float*)w;
    float* yp = (float*)y;
    hipStream_t s = (hipStream_t)stream;
    // Few rows: one tile of W a workgroup while that gives less than two workgroups a compute unit, two beyond (x is then
    // read half as often).  More than 32 rows: 32 outputs by 64 rows a workgroup where that is a workgroup a compute unit, else 16
    // by 64.  Cold weights, us, 32 and 16 outputs (the plain kernel): 64 rows, 1,024 columns of k 1,024 14.8 and 11.2 (143), 2,048 of
    // 6,144 96 and 57 (1,074), 32,768 of 1,024 58.6 and 77.7 (213); 256 rows, 2,048 of 2,048 30.8 and 37.7 (291), 6,144 of 4,096 184
    // and 214 (666), 1,536 of 1,024 (192 workgroups or 384) 15.2 and 20.3, but 33 rows, 6,144 of 4,096 (the same) 59.4 and 53.7; 512 rows, 4,096 gated of 1,024 108.5 (213); 2,048 rows, 2,048 of 6,144 737 and 842 (1,233) = 70 TFLOP/s.  64
    // outputs by 64 rows, whose registers leave a SIMD one wave, are nowhere faster: 2,048 rows, 2,048 of 6,144 738, 12,288 gated
    // of 4,096 at 64 rows 254 and with 32 outputs 170.
    const long tiles = ((long)(gated ? 2 : 1) * N + 15) / 16, units = tli_compute_units();
    // parts of a tile while that gives no more than a workgroup a compute unit (1,024 columns of k 4,096: 64 workgroups of
    // whole tiles, 256 of quarters: 16 decode steps of four layers of width 1,024 4.47 -> 4.19 ms)
    if (M <= 32 && !gated && tiles * 2 <= units) {
        const bool four = tiles * 4 <= units;
        if (M <= 16) return four ? launch_f32_part<1, 8, 4>(xp, wp, yp, M, N, K, gate, s) : launch_f32_part<1, 8, 8>(xp, wp, yp, M, N, K, gate, s);
        return four ? launch_f32_part<2, 4, 4>(xp, wp, yp, M, N, K, gate, s) : launch_f32_part<2, 4, 8>(xp, wp, yp, M, N, K, gate, s);
    }
    if (M <= 16) return tiles < 2 * units && !gated ? launch_f32<1, 1, 8>(xp, wp, yp, M, N, K, gate, s)
                                                    : launch_f32<2, 1, 4>(xp, wp, yp, M, N, K, gate, s);
    if (M <= 32) return tiles < 2 * units && !gated ? launch_f32<1, 2, 4>(xp, wp, yp, M, N, K, gate, s)
                                                    : launch_f32<2, 2, 4>(xp, wp, yp, M, N, K, gate, s);
    const long blocks = tiles * ((M + 63) / 64);
    if (blocks >= 2 * units || gated) return launch_f32<2, 4, 2>(xp, wp, yp, M, N, K, gate, s);
    return launch_f32<1, 4, 2>(xp, wp, yp, M, N, K, gate, s);
}

// How many planes of partial sums tli_gemm_f32_ranges leaves, or 0 where it does not take the product: up to 32 rows (more do not lie in a
// wave's registers beside W) and no more outputs than the kernel above gives parts of tiles for (with whole tiles the sums cost their
// reader more than they save: eight planes to read instead of one).
extern "C" int tli_gemm_f32_ranges_of(int M, int N) {
    return M > 0 && M <= 32 && N > 0 && ((long)N + 15) / 16 * 2 <= tli_compute_units() ? GF_RANGES : 0;
}

// Whether leaving the ranges' sums to the norm or the attention behind costs less than the whole product: not where k is short, as the reader has
// eight planes to read for one, nor where the eight ranges of a short k are not alike.  us, product and norm, whole and left, 1 and 32 rows: 1,024 columns of k 128 4.9, 5.1
// and 5.6, 5.8, of 256 5.2, 5.1 and 6.5, 6.1, of 1,024 7.5, 6.2 and 11.0, 7.5; 848 of k 392 5.7, 6.3 and 6.8, 7.5, 800 of 640 5% less; 2,048 of 512 6.7, 7.0 and 8.4, 8.9, of
// 1,024 7.5, 7.2 and 11.3, 9.9.  Rows that are no multiple of four are read element by element, which costs more of them: 250 of 256 6% less (1 row), 322 of 256
// 6% more, of 512 level, 893 of 512 7.7, 8.4 (1 row), of 1,024 5% less; 2,046 of 1,024 12% more, of 2,048 level.
extern "C" int tli_gemm_f32_ranges_pay(int N, int K) {
    if (N % 4) return K >= (N <= 256 ? 256 : N <= 512 ? 512 : N <= 1024 ? 1024 : 2048);
    if (N > 1024) return K >= 1024;
    return K >= (N > 512 && K % (16 * GF_RANGES) ? 640 : 256);
}

// parts[GF_RANGES][M][N]: y of tli_gemm_f32 is their sum in order, from zero.
extern "C" int tli_gemm_f32_ranges(const void* x, const void* w, void* parts, int M, int N, int K, void* stream) {
    if (!tli_gemm_f32_ranges_of(M, N)) return tli_fail("gemm_f32_ranges: %d rows of %d outputs are not taken", M, N);
    if (K <= 0 || K % 4) return tli_fail("gemm_f32_ranges: K = %d must be a positive multiple of 4", K);
    if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts) & 15) return tli_fail("gemm_f32_ranges: operands must be 16-byte aligned");
    const dim3 grid((unsigned)((N + 16 * GF_PART_WAVES - 1) / (16 * GF_PART_WAVES)), GF_RANGES);
    if (M <= 16) gemm_f32_ranges_kernel<1, 8><<<grid, GF_PART_WAVES * 64, 0, (hipStream_t)stream>>>((const float*)x, (const float*)w, (float*)parts, M, N, K);
    else gemm_f32_ranges_kernel<2, 8><<<grid, GF_PART_WAVES * 64, 0, (hipStream_t)stream>>>((const float*)x, (const float*)w, (float*)parts, M, N, K);
    return tli_check_launch("gemm_f32_ranges");
}
