// Attention over a latent vector a position: what stands before and behind the attention itself.
//
// prepare:        from the raw projections of a row (q of `heads` heads of dim + rot elements; the latent
//                 vector of `rank` elements and one key part of `rot` elements) the cache entry of the position,
//                 [RMS norm of the latent vector with its weight | the key part, turned], and the queries' own
//                 turned parts, written behind the place where their `rank` elements in the latent space go.
//                 The first rot_dims elements of a part are turned in pairs (i, i + rot_dims / 2).  One workgroup
//                 a row; float32 arithmetic.  Without a latent vector (a layer that reads another's) the queries only.
// head_products:  y[t, h, :] = W[h] x[t, h, :] for a matrix a head (float32 sums), with strides so that inputs
//                 and outputs may lie inside wider rows; times sigmoid(gate[t, h]) where gates are given.  Plain: any
//                 sizes and both types.
#include "common.h"

#define LP_THREADS 256

// One number a row and head that the head's output is multiplied by: the logistic function of logits that lie `ld`
// elements a row apart, or 1 without them.
template <typename T>
struct HeadGate {
    const T* z;
    int ld;
    __device__ __forceinline__ float of(int t, int h) const { return z ? 1.0f / (1.0f + expf(-to_f32(z[(size_t)t * ld + h]))) : 1.0f; }
};

template <typename T>
struct LatentRows {
    const T* q_in;
    int q_ld;
    const T* down_in;
    int down_ld;
    T *q_out, *cache;
    const int *positions, *seq_of_row, *tables;
    int table_width, page_size, num_pages, heads, dim, rot, rank, rot_dims;
    const float* norm_weight;
    float eps;
    const float *cos_t, *sin_t;
};

template <typename T>
__device__ __forceinline__ void latent_prepare_row(const LatentRows<T>& a, int row, float* red) {
    const int tid = threadIdx.x, half = a.rot_dims / 2, rot_dims = a.rot_dims, rot = a.rot, rank = a.rank, dim = a.dim;
    const T* src = a.q_in + (size_t)row * a.q_ld;
    const int pos = a.positions[row];
    const float* cs = a.cos_t + (size_t)pos * half;
    const float* sn = a.sin_t + (size_t)pos * half;
    const int key = rank + rot;
    // the queries' turned parts
    for (int i = tid; i < a.heads * rot; i += LP_THREADS) {
        const int h = i / rot, d = i % rot;
        const T* part = src + (size_t)h * (dim + rot) + dim;
        float v = to_f32(part[d]);
        if (d < half) v = rotate_first_half(v, to_f32(part[d + half]), cs[d], sn[d]);
        else if (d < rot_dims) v = rotate_second_half(v, to_f32(part[d - half]), cs[d - half], sn[d - half]);
        from_f32(a.q_out + ((size_t)row * a.heads + h) * key + rank + d, v);
    }
    if (!a.down_in) return;
    const int page = a.tables[(size_t)a.seq_of_row[row] * a.table_width + pos / a.page_size];
    const T* down = a.down_in + (size_t)row * a.down_ld;
    float ssq = 0.f;
    for (int d = tid; d < rank; d += LP_THREADS) {
        const float a = to_f32(down[d]);
        ssq = fmaf(a, a, ssq);
    }
    const float factor = 1.0f / sqrtf(block_sum(ssq, red) / (float)rank + a.eps);
    if (page < 0 || page >= a.num_pages) return;
    T* dst = a.cache + ((size_t)page * a.page_size + pos % a.page_size) * key;
    for (int d = tid; d < rank; d += LP_THREADS) {
        T r;
        from_f32(&r, to_f32(down[d]) * factor * a.norm_weight[d]);
        dst[d] = cache_value(r);
    }
    const T* part = down + rank;
    for (int d = tid; d < rot; d += LP_THREADS) {
        float v = to_f32(part[d]);
        if (d < half) v = rotate_first_half(v, to_f32(part[d + half]), cs[d], sn[d]);
        else if (d < rot_dims) v = rotate_second_half(v, to_f32(part[d - half]), cs[d - half], sn[d - half]);
        T r;
        from_f32(&r, v);
        dst[rank + d] = cache_value(r);
    }
}

template <typename T>
__global__ __launch_bounds__(LP_THREADS) void latent_prepare_kernel(LatentRows<T> a) {
    __shared__ float red[16];
    latent_prepare_row(a, blockIdx.x, red);
}

template <typename T>
__global__ __launch_bounds__(256) void head_products_plain_kernel(const T* __restrict__ x, long long x_row, long long x_head,
                                                                  const T* __restrict__ w, T* __restrict__ y, long long y_row,
                                                                  long long y_head, int N, int K, HeadGate<T> gate) {
    extern __shared__ float xs[];
    const int t = blockIdx.x, h = blockIdx.y;
    const T* xr = x + (size_t)t * x_row + (size_t)h * x_head;
    for (int k = threadIdx.x; k < K; k += blockDim.x) xs[k] = to_f32(xr[k]);
    __syncthreads();
    const int lane = threadIdx.x % TLI_WAVE, wave = threadIdx.x / TLI_WAVE, waves = blockDim.x / TLI_WAVE;
    for (int n = wave; n < N; n += waves) {
        const T* wr = w + ((size_t)h * N + n) * K;
        float a = 0.f;
        for (int k = lane; k < K; k += TLI_WAVE) a = fmaf(xs[k], to_f32(wr[k]), a);
        a = wave_sum(a);
        if (lane == 0) from_f32(y + (size_t)t * y_row + (size_t)h * y_head + n, a * gate.of(t, h));
    }
}

// q_in: rows q_ld elements apart, heads * (dim + rot) of each;  down_in: rows down_ld apart, latent (rank) | key part (rot),
// or null;  q_out [rows, heads, rank + rot] (only
// the last rot of every head are written);  cache [pages][slot][rank + rot];  cos_t, sin_t [positions, rot_dims / 2]
extern "C" int tli_latent_prepare(const void* q_in, int q_ld, const void* down_in, int down_ld, void* q_out, void* cache, const int* positions,
                                  const int* seq_of_row, const int* tables, int table_width, int page_size, int num_pages,
                                  int rows, int heads, int dim, int rot, int rank, int rot_dims, const float* norm_weight,
                                  float eps, const float* cos_t, const float* sin_t, int dtype, void* stream) {
    if (rows <= 0) return 0;
    if (heads <= 0 || dim <= 0 || rot <= 0 || rank <= 0 || rot_dims <= 0 || rot_dims % 2 || rot_dims > rot ||
        !q_in || q_ld < heads * (dim + rot) || (down_in && (down_ld < rank + rot || !norm_weight)))
        return tli_fail("latent_prepare: bad sizes");
    if (page_size <= 0 || table_width <= 0 || num_pages <= 0) return tli_fail("latent_prepare: bad cache geometry");
    hipStream_t s = (hipStream_t)stream;
#define LATENT_ROWS(T)                                                                                                                  \
    LatentRows<T>{(const T*)q_in, q_ld, (const T*)down_in, down_ld, (T*)q_out, (T*)cache, positions, seq_of_row, tables, table_width,   \
                  page_size, num_pages, heads, dim, rot, rank, rot_dims, norm_weight, eps, cos_t, sin_t}
    if (dtype == TLI_F32)
        latent_prepare_kernel<float><<<rows, LP_THREADS, 0, s>>>(LATENT_ROWS(float));
    else if (dtype == TLI_BF16)
        latent_prepare_kernel<bf16_t><<<rows, LP_THREADS, 0, s>>>(LATENT_ROWS(bf16_t));
    else
        return tli_fail("latent_prepare: unknown dtype %d", dtype);
    return tli_check_launch("latent_prepare");
}

// y[t, h, n] = sum_k x[t, h, k] w[h, n, k] (times sigmoid(gate[t * gate_ld + h]), if given);  x at x + t * x_row + h * x_head (elements), y likewise;  w [heads, N, K]
extern "C" int tli_head_products_plain(const void* x, long long x_row, long long x_head, const void* w, void* y, long long y_row,
                                       long long y_head, int rows, int heads, int N, int K, const void* gate, int gate_ld,
                                       int dtype, void* stream) {
    if (rows <= 0) return 0;
    if (heads <= 0 || heads > 65535 || N <= 0 || K <= 0 || K > 12288) return tli_fail("head_products: bad sizes");
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(rows, heads);
    if (dtype == TLI_F32)
        head_products_plain_kernel<float><<<grid, 256, (size_t)K * 4, s>>>((const float*)x, x_row, x_head, (const float*)w, (float*)y,
                                                                           y_row, y_head, N, K, HeadGate<float>{(const float*)gate, gate_ld});
    else if (dtype == TLI_BF16)
        head_products_plain_kernel<bf16_t><<<grid, 256, (size_t)K * 4, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)y,
                                                                            y_row, y_head, N, K, HeadGate<bf16_t>{(const bf16_t*)gate, gate_ld});
    else
        return tli_fail("head_products: unknown dtype %d", dtype);
    return tli_check_launch("head_products_plain");
}

// ---------------------------------------------------------------------------------------------------------------
// head_products on the matrix cores (bfloat16, N and K in sixteens): a workgroup of four waves takes 16 rows and one
// head; its waves share out the head's blocks of 16 outputs.  A is a block of W (16 outputs x 16 of k), B the rows'
// fragments, which a wave holds in registers for all its blocks (k up to 640), so a lane ends with four consecutive
// outputs of one row.  v_mfma_f32_16x16x16_bf16.
// ---------------------------------------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) short hp_bf16x4;
typedef __attribute__((ext_vector_type(4))) float hp_f32x4;
union HpFrag {
    uint2 u;
    hp_bf16x4 v;
};

// A wave takes RT tiles of 16 rows and walks all blocks of 16 outputs, two at a time with a sum each, so that a
// matrix instruction does not wait for the one before it; a block of W that it has fetched serves all its row tiles.
// (A workgroup's four waves fetch the same blocks of W one after the other: three of them find it in the cache.)
// EXACT: K is 16 KM (no condition left in the loop over k).
template <int KM, bool EXACT, int RT>
__device__ __forceinline__ void head_products_mfma(const bf16_t* __restrict__ x, long long x_row, long long x_head,
                                                   const bf16_t* __restrict__ w, bf16_t* __restrict__ y,
                                                   long long y_row, long long y_head, int T, int N, int K, HeadGate<bf16_t> gate, int shares) {
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int col = lane % 16, grp = lane / 16;
    const int t0 = (blockIdx.x * 4 + wave) * 16 * RT, h = blockIdx.y;
    if (t0 >= T) return;                                                // (the whole wave; no barriers in this kernel)
    const int nk = EXACT ? KM : K / 16;
    HpFrag xf[RT][KM];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int t = min(t0 + r * 16 + col, T - 1);                    // (rows past the end repeat the last; never stored)
        const bf16_t* xr = x + (size_t)t * x_row + (size_t)h * x_head;
#pragma unroll
        for (int j = 0; j < KM; ++j) {
            xf[r][j].u = make_uint2(0, 0);
            if (j < nk) xf[r][j].u = *reinterpret_cast<const uint2*>(xr + j * 16 + grp * 4);
        }
    }
    float by[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) by[r] = gate.of(min(t0 + r * 16 + col, T - 1), h);
    // (few rows: the blocks of outputs are shared out over blockIdx.z, an even number each)
    const int per_z = (((N / 16 + shares - 1) / shares) + 1) & ~1;
    const int nblocks = min(N / 16, (int)(blockIdx.z + 1) * per_z);
    for (int nb = blockIdx.z * per_z; nb < nblocks; nb += 2) {
        const bool two = nb + 1 < nblocks;
        const bf16_t* wr0 = w + ((size_t)h * N + nb * 16 + col) * K + grp * 4;
        const bf16_t* wr1 = two ? wr0 + (size_t)16 * K : wr0;
        hp_f32x4 acc0[RT], acc1[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) acc0[r] = acc1[r] = (hp_f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KM; ++j) {
            if (j < nk) {
                HpFrag a0, a1;
                a0.u = *reinterpret_cast<const uint2*>(wr0 + j * 16);
                a1.u = *reinterpret_cast<const uint2*>(wr1 + j * 16);
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    acc0[r] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0.v, xf[r][j].v, acc0[r], 0, 0, 0);
                    acc1[r] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a1.v, xf[r][j].v, acc1[r], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int t = t0 + r * 16 + col;
            if (t < T) {
                bf16_t* yr = y + (size_t)t * y_row + (size_t)h * y_head + grp * 4 + nb * 16;
                uint2 st;
                st.x = pack_bf16x2(acc0[r][0] * by[r], acc0[r][1] * by[r]);
                st.y = pack_bf16x2(acc0[r][2] * by[r], acc0[r][3] * by[r]);
                *reinterpret_cast<uint2*>(yr) = st;
                if (two) {
                    st.x = pack_bf16x2(acc1[r][0] * by[r], acc1[r][1] * by[r]);
                    st.y = pack_bf16x2(acc1[r][2] * by[r], acc1[r][3] * by[r]);
                    *reinterpret_cast<uint2*>(yr + 16) = st;
                }
            }
        }
    }
}

template <int KM, bool EXACT, int RT>
__global__ __launch_bounds__(256) void head_products_mfma_kernel(const bf16_t* __restrict__ x, long long x_row, long long x_head,
                                                                 const bf16_t* __restrict__ w, bf16_t* __restrict__ y,
                                                                 long long y_row, long long y_head, int T, int N, int K, HeadGate<bf16_t> gate) {
    head_products_mfma<KM, EXACT, RT>(x, x_row, x_head, w, y, y_row, y_head, T, N, K, gate, gridDim.z);
}

// Steps of few rows: the queries' products into the latent space and prepare, which touch nothing of each other's, as one launch: the
// first `shares` of gridDim.z multiply, the workgroups of the others prepare a row each (a row is a chain of fetches: 64 of them behind one
// another in a workgroup took 122 us).  8 rows of 16 heads, as part of a decode step: 6.1 and 4.2 us one behind the other, 6.0 together.
// The whole layer between its projections, 100 keys of 512 + 64, apart and together, us: 16 heads, 1 row 19.6 and 18.0, 8 rows 20.6 and
// 18.7, 64 rows 36.4 and 34.3; one head, 1 row 17.2 and 14.9, 64 rows 28.6 and 25.6.
template <int KM, bool EXACT>
__global__ __launch_bounds__(256) void latent_prepare_products_kernel(LatentRows<bf16_t> a, const bf16_t* __restrict__ w, int T, int shares) {
    __shared__ float red[16];
    const int key = a.rank + a.rot;
    if ((int)blockIdx.z >= shares) {
        const int row = ((blockIdx.z - shares) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        if (row < T) latent_prepare_row(a, row, red);
        return;
    }
    head_products_mfma<KM, EXACT, 1>(a.q_in, a.q_ld, a.dim + a.rot, w, a.q_out, (long long)a.heads * key, key, T, a.rank, a.dim,
                                     HeadGate<bf16_t>{nullptr, 0}, shares);
}

// Many rows, k of 64, 128, 256 or 512: the head's matrix comes through LDS.  A workgroup takes one head and 64 RT rows
// (a wave RT tiles of 16, their fragments in registers) and walks the outputs in chunks of 8192 elements of W (NB
// blocks of 16 outputs), which its 256 threads bring into one of two LDS buffers with 16-byte loads while the chunk
// before is multiplied; the waves read the blocks' fragments from there (rows of k + 8 elements: 8-byte reads without
// bank conflicts), each fragment serving the wave's RT row tiles, with two sums a row tile taking turns.
template <int KM, int RT>
__global__ __launch_bounds__(256) void head_products_lds_kernel(const bf16_t* __restrict__ x, long long x_row, long long x_head,
                                                                const bf16_t* __restrict__ w, bf16_t* __restrict__ y,
                                                                long long y_row, long long y_head, int T, int N, HeadGate<bf16_t> gate) {
    constexpr int K = KM * 16, LDW = K + 8, NB = 32 / KM, ROWS = NB * 16, PIECES = K / 8;
    __shared__ __align__(16) bf16_t wt[2][ROWS * LDW];
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int col = lane % 16, grp = lane / 16;
    const int t0 = (blockIdx.x * 4 + wave) * 16 * RT, h = blockIdx.y;
    HpFrag xf[RT][KM];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int t = min(t0 + r * 16 + col, T - 1);                    // (rows past the end repeat the last; never stored)
        const bf16_t* xr = x + (size_t)t * x_row + (size_t)h * x_head;
#pragma unroll
        for (int j = 0; j < KM; ++j) xf[r][j].u = *reinterpret_cast<const uint2*>(xr + j * 16 + grp * 4);
    }
    float by[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) by[r] = gate.of(min(t0 + r * 16 + col, T - 1), h);
    const bf16_t* wh = w + (size_t)h * N * K;
    const int chunks = (N + ROWS - 1) / ROWS;
    uint4 next[4];                                                      // ROWS * PIECES = 1024 pieces of 16 bytes a chunk
    auto fetch = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = i * 256 + tid;
            const int n = c * ROWS + idx / PIECES;
            next[i] = make_uint4(0, 0, 0, 0);
            if (n < N) next[i] = *reinterpret_cast<const uint4*>(wh + (size_t)n * K + (idx % PIECES) * 8);
        }
    };
    auto store = [&](bf16_t* buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = i * 256 + tid;
            *reinterpret_cast<uint4*>(buf + (idx / PIECES) * LDW + (idx % PIECES) * 8) = next[i];
        }
    };
    fetch(0);
    store(wt[0]);
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
        const bool more = c + 1 < chunks;
        if (more) fetch(c + 1);
        const bf16_t* buf = wt[c & 1];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            hp_f32x4 even[RT], odd[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) even[r] = odd[r] = (hp_f32x4){0.f, 0.f, 0.f, 0.f};
            const bf16_t* wr = buf + (nb * 16 + col) * LDW + grp * 4;
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                HpFrag a;
                a.u = *reinterpret_cast<const uint2*>(wr + j * 16);
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    if (j % 2)
                        odd[r] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.v, xf[r][j].v, odd[r], 0, 0, 0);
                    else
                        even[r] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.v, xf[r][j].v, even[r], 0, 0, 0);
                }
            }
            const int n0 = (c * NB + nb) * 16;
            if (n0 < N) {
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const int t = t0 + r * 16 + col;
                    if (t < T) {
                        uint2 st;
                        st.x = pack_bf16x2((even[r][0] + odd[r][0]) * by[r], (even[r][1] + odd[r][1]) * by[r]);
                        st.y = pack_bf16x2((even[r][2] + odd[r][2]) * by[r], (even[r][3] + odd[r][3]) * by[r]);
                        *reinterpret_cast<uint2*>(y + (size_t)t * y_row + (size_t)h * y_head + n0 + grp * 4) = st;
                    }
                }
            }
        }
        if (more) store(wt[(c + 1) & 1]);
        __syncthreads();                                // the next chunk is written; this one is read by all
    }
}

extern "C" int tli_head_products_mfma_takes(int N, int K, long long x_row, long long x_head, long long y_row, long long y_head) {
    return (N % 16 == 0 && K % 16 == 0 && N >= 16 && K >= 16 && K <= 640 && x_row % 4 == 0 && x_head % 4 == 0 &&
            y_row % 4 == 0 && y_head % 4 == 0) ? 1 : 0;
}

extern "C" int tli_head_products_mfma_bf16(const void* x, long long x_row, long long x_head, const void* w, void* y,
                                           long long y_row, long long y_head, int rows, int heads, int N, int K,
                                           const void* gate_z, int gate_ld, void* stream) {
    if (rows <= 0) return 0;
    if (heads <= 0 || heads > 65535 || !tli_head_products_mfma_takes(N, K, x_row, x_head, y_row, y_head))
        return tli_fail("head_products: the matrix-core kernel takes sizes in sixteens (k up to 640), not %d x %d", N, K);
    if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 7)) return tli_fail("head_products: operands must be 8-byte aligned");
    const HeadGate<bf16_t> gate{(const bf16_t*)gate_z, gate_ld};
    if (rows >= 1024 && (K == 64 || K == 128 || K == 256 || K == 512)) {
        const dim3 lgrid((rows + 127) / 128, heads);
        hipStream_t ls = (hipStream_t)stream;
#define HP_LDS(KM)                                                                                                       \
    head_products_lds_kernel<KM, 2><<<lgrid, 256, 0, ls>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)y, \
                                                           y_row, y_head, rows, N, gate)
        if (K == 64) HP_LDS(4);
        else if (K == 128) HP_LDS(8);
        else if (K == 256) HP_LDS(16);
        else HP_LDS(32);
#undef HP_LDS
        return tli_check_launch("head_products_lds");
    }
    // (many rows: a wave keeps 4 tiles of 16 rows, 2 where k is large, so that a block of W serves them all)
    const int rt = rows < 1024 ? 1 : (K <= 128 ? 4 : (K <= 512 ? 2 : 1));
    const int row_groups = (rows + 64 * rt - 1) / (64 * rt);
    int shares = 512 / (row_groups * heads);                           // enough workgroups for the chip
    shares = shares < 1 ? 1 : (shares > N / 32 ? (N / 32 < 1 ? 1 : N / 32) : shares);
    const dim3 grid(row_groups, heads, shares);
    hipStream_t s = (hipStream_t)stream;
#define HP_ONE(KM, EXACT, RT)                                                                                              \
    head_products_mfma_kernel<KM, EXACT, RT><<<grid, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)w, (bf16_t*)y, \
                                                                  y_row, y_head, rows, N, K, gate)
    if (K == 64) { if (rt == 4) HP_ONE(4, true, 4); else HP_ONE(4, true, 1); }
    else if (K == 128) { if (rt == 4) HP_ONE(8, true, 4); else HP_ONE(8, true, 1); }
    else if (K == 256) { if (rt == 2) HP_ONE(16, true, 2); else HP_ONE(16, true, 1); }
    else if (K == 512) { if (rt == 2) HP_ONE(32, true, 2); else HP_ONE(32, true, 1); }
    else if (K <= 128) { if (rt == 4) HP_ONE(8, false, 4); else HP_ONE(8, false, 1); }
    else if (K <= 512) { if (rt == 2) HP_ONE(32, false, 2); else HP_ONE(32, false, 1); }
    else HP_ONE(40, false, 1);
#undef HP_ONE
    return tli_check_launch("head_products_mfma");
}

// tli_latent_prepare and tli_head_products_mfma_bf16 of the queries with w_qk [heads, rank, dim] into q_out, bfloat16, for up to
// LPP_ROWS rows.
#define LPP_ROWS 64
extern "C" int tli_latent_prepare_products_bf16(const void* q_in, int q_ld, const void* down_in, int down_ld, void* q_out, void* cache,
                                                const int* positions, const int* seq_of_row, const int* tables, int table_width,
                                                int page_size, int num_pages, int rows, int heads, int dim, int rot, int rank,
                                                int rot_dims, const float* norm_weight, float eps, const float* cos_t,
                                                const float* sin_t, const void* w_qk, void* stream) {
    if (rows <= 0) return 0;
    if (heads <= 0 || heads > 65535 || dim <= 0 || rot <= 0 || rank <= 0 || rot_dims <= 0 || rot_dims % 2 || rot_dims > rot || rows > LPP_ROWS ||
        !q_in || q_ld < heads * (dim + rot) || (down_in && (down_ld < rank + rot || !norm_weight)))
        return tli_fail("latent_prepare_products: bad sizes");
    if (page_size <= 0 || table_width <= 0 || num_pages <= 0) return tli_fail("latent_prepare_products: bad cache geometry");
    const long long key = rank + rot;
    if (!tli_head_products_mfma_takes(rank, dim, q_ld, dim + rot, heads * key, key) || (((uintptr_t)q_in | (uintptr_t)w_qk | (uintptr_t)q_out) & 7))
        return tli_fail("latent_prepare_products: the products are not the matrix-core kernel's");
    const int row_groups = (rows + 63) / 64;
    int shares = 512 / (row_groups * heads);
    shares = shares < 1 ? 1 : (shares > rank / 32 ? (rank / 32 < 1 ? 1 : rank / 32) : shares);
    const int preparing = (rows + row_groups * heads - 1) / (row_groups * heads);        // (a workgroup a row: each is a chain of fetches)
    const dim3 grid(row_groups, heads, shares + preparing);
    hipStream_t s = (hipStream_t)stream;
    const LatentRows<bf16_t> a = LATENT_ROWS(bf16_t);
#define LPP_RUN(KM, EXACT) latent_prepare_products_kernel<KM, EXACT><<<grid, 256, 0, s>>>(a, (const bf16_t*)w_qk, rows, shares)
    if (dim == 64) LPP_RUN(4, true);
    else if (dim == 128) LPP_RUN(8, true);
    else if (dim == 256) LPP_RUN(16, true);
    else if (dim <= 128) LPP_RUN(8, false);
    else LPP_RUN(40, false);
#undef LPP_RUN
    return tli_check_launch("latent_prepare_products");
}
