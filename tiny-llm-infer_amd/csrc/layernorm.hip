// Residual add + layer norm without bias, for one or two weight vectors at once.
//
//   v = resid[r] + (d1[r] + d2[r])          (what the parts before still owe the residual; float32)
//   m = mean(v),  s = mean((v - m)^2)       (two passes: the variance is of the deviations)
//   out_a = (v - m) / sqrt(s + eps) * w_a   for a = 1 (and 2: two norms of the same row share m and s)
//
// With a row list only those rows are computed and the residual is left as it is.
//
// With a router (COLS > 0: 1,024 threads a row, bfloat16) the last output's row stays in LDS and the row's experts are chosen in the
// same launch (moe_route.h), whose weights come in while the row is normed.
#include "common.h"
#include "moe_route.h"

// What the parts owe may come as float32 partial sums [parts][total rows][n] in the place of rows of T (parts > 0): the row is
// their sum, rounded to T.  SUMS: whether either does; the kernels without them read their rows as before (8 rows of 5,120
// float32 4.34 us, and 4.68 with the question at every element).
struct OwedSums {
    const float* p[2];
    int parts[2];
    size_t step;                 // elements between two parts
};

template <typename T, bool SUMS>
struct Owed {
    const T *d1, *d2;            // at the row's first element
    OwedSums sums;
    size_t row;                  // the row's first element
    __device__ __forceinline__ bool has(int w) const { return (w ? d2 : d1) != nullptr || (SUMS && sums.parts[w] > 0); }
    __device__ __forceinline__ bool any() const { return has(0) || has(1); }
    __device__ __forceinline__ float part(int w, int i) const {
        if (!SUMS || sums.parts[w] == 0) return to_f32((w ? d2 : d1)[i]);
        float a = 0.f;
        for (int s = 0; s < sums.parts[w]; ++s) a += sums.p[w][s * sums.step + row + i];
        T t;
        from_f32(&t, a);
        return to_f32(t);
    }
    __device__ __forceinline__ float at(int i) const {
        float d = has(0) ? part(0, i) : 0.f;
        if (has(1)) d = has(0) ? d + part(1, i) : part(1, i);
        return d;
    }
};

template <typename T, bool SUMS>
__global__ void add_layernorm_kernel(float* __restrict__ resid, const T* __restrict__ d1, const T* __restrict__ d2, OwedSums sums,
                                     const float* __restrict__ w1, const float* __restrict__ w2,
                                     T* __restrict__ out1, T* __restrict__ out2, const int* __restrict__ rows,
                                     int n, float eps, int total_rows) {
    __shared__ float scratch[16];
    const int out_row = blockIdx.x;
    int r = rows ? rows[out_row] : out_row;
    if (r < 0 || r >= total_rows) r = 0;
    float* x = resid + (size_t)r * n;
    const Owed<T, SUMS> d{d1 ? d1 + (size_t)r * n : nullptr, d2 ? d2 + (size_t)r * n : nullptr, sums, (size_t)r * n};
    const bool update = rows == nullptr && d.any();
    const bool again = d.any() && !update;           // the sum is not stored: every pass makes it anew
    float sum = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float v = x[i];
        if (d.any()) v += d.at(i);
        if (update) x[i] = v;
        sum += v;
    }
    const float mean = block_sum(sum, scratch) / (float)n;
    float ss = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float v = x[i];
        if (again) v += d.at(i);
        ss += (v - mean) * (v - mean);
    }
    const float scale = 1.0f / sqrtf(block_sum(ss, scratch) / (float)n + eps);
    T* o1 = out1 + (size_t)out_row * n;
    T* o2 = out2 ? out2 + (size_t)out_row * n : nullptr;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        float v = x[i];
        if (again) v += d.at(i);
        const float z = (v - mean) * scale;
        from_f32(o1 + i, z * w1[i]);
        if (o2) from_f32(o2 + i, z * w2[i]);
    }
}

// The row in registers: n % 4 == 0 and n <= 4 * IT * blockDim.x, everything 16-byte aligned.
__device__ __forceinline__ void ln_load4(const float* p, float v[4]) {
    const float4 t = *reinterpret_cast<const float4*>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void ln_load4(const bf16_t* p, float v[4]) {
    const uint2 t = *reinterpret_cast<const uint2*>(p);
    v[0] = bf16_to_f32((bf16_t)(t.x & 0xffffu)); v[1] = bf16_to_f32((bf16_t)(t.x >> 16));
    v[2] = bf16_to_f32((bf16_t)(t.y & 0xffffu)); v[3] = bf16_to_f32((bf16_t)(t.y >> 16));
}
__device__ __forceinline__ void ln_store4(float* p, const float v[4]) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void ln_store4(bf16_t* p, const float v[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

// four elements of the sum of `parts` float32 parts, rounded to T
template <typename T>
__device__ __forceinline__ void ln_sum4(const float* p, int parts, size_t step, float v[4]) {
    v[0] = v[1] = v[2] = v[3] = 0.f;
    // (two parts on their way together)
    for (int s = 0; s < parts; s += 2) {
        float a[4], b[4] = {0.f, 0.f, 0.f, 0.f};
        ln_load4(p + s * step, a);
        if (s + 1 < parts) ln_load4(p + (s + 1) * step, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (v[e] + a[e]) + b[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        T t;
        from_f32(&t, v[e]);
        v[e] = to_f32(t);
    }
}

template <typename T, int IT, bool SUMS, int COLS = 0, int KI = 1>
__global__ void __launch_bounds__(1024) add_layernorm_vec_kernel(float* __restrict__ resid, const T* __restrict__ d1, const T* __restrict__ d2, OwedSums sums,
                                         const float* __restrict__ w1, const float* __restrict__ w2,
                                         T* __restrict__ out1, T* __restrict__ out2, const int* __restrict__ rows,
                                         int n, float eps, int total_rows, unsigned span, RouteArgs route) {
    static_assert(COLS == 0 || sizeof(T) == 2, "a router reads bfloat16 rows");
    __shared__ float scratch[16];
    __shared__ __align__(16) bf16_t row_lds[COLS > 0 ? 512 * KI : 1];
    __shared__ float s_lds[NORM_ROUTE_COLS + 1], c_lds[NORM_ROUTE_COLS];
    RouteRows<COLS, KI, NORM_ROUTE_THREADS / TLI_WAVE> router;
    const int out_row = blockIdx.x;
    int r = rows ? rows[out_row] : out_row;
    if (r < 0 || r >= total_rows) r = 0;
    float* x = resid + (size_t)r * n;
    const bool sums1 = SUMS && sums.parts[0] > 0, sums2 = SUMS && sums.parts[1] > 0, has1 = d1 || sums1, has2 = d2 || sums2;
    const bool update = rows == nullptr && (has1 || has2);
    // (Beside a router the norms' weights are asked for beside the row, which rows past 2,048 elements need: 8 rows of 4,096, 8 experts, 7.6 us
    // and behind the sums 7.8.  Else behind the sums: one norm of 8 rows of 2,048 3.28 us beside the row and 3.17, of 2,048 rows 9.5 and 9.1,
    // two norms of 8,192 rows of 4,096 91 and 86.)
    constexpr bool EARLY = COLS > 0;
    float v[IT][4], g1[IT][4], g2[IT][4];
    float sum = 0.f;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int i = (threadIdx.x + it * span) * 4;
        if (threadIdx.x < span && i < n) {
            ln_load4(x + i, v[it]);
            if constexpr (EARLY) {
                ln_load4(w1 + i, g1[it]);
                if (out2) ln_load4(w2 + i, g2[it]);
            }
            float a[4], b[4];
            if (sums1) ln_sum4<T>(sums.p[0] + (size_t)r * n + i, sums.parts[0], sums.step, a);
            else if (d1) ln_load4(d1 + (size_t)r * n + i, a);
            if (sums2) ln_sum4<T>(sums.p[1] + (size_t)r * n + i, sums.parts[1], sums.step, b);
            else if (d2) ln_load4(d2 + (size_t)r * n + i, b);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (has1 && has2) v[it][e] += a[e] + b[e];
                else if (has1) v[it][e] += a[e];
                else if (has2) v[it][e] += b[e];
                sum += v[it][e];
            }
            if (update) ln_store4(x + i, v[it]);
        }
    }
    if constexpr (COLS > 0) {
        router.fetch(route, n, threadIdx.x / TLI_WAVE, threadIdx.x % TLI_WAVE);
        if (threadIdx.x < route.E) c_lds[threadIdx.x] = route.correction ? route.correction[threadIdx.x] : 0.f;
    }
    const float mean = block_sum(sum, scratch) / (float)n;
    float ss = 0.f;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int i = (threadIdx.x + it * span) * 4;
        if (threadIdx.x < span && i < n) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[it][e] -= mean;
                ss += v[it][e] * v[it][e];
            }
        }
    }
    const float scale = 1.0f / sqrtf(block_sum(ss, scratch) / (float)n + eps);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int i = (threadIdx.x + it * span) * 4;
        if (threadIdx.x < span && i < n) {
            float o[4];
            if constexpr (!EARLY) ln_load4(w1 + i, g1[it]);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[it][e] * scale * g1[it][e];
            ln_store4(out1 + (size_t)out_row * n + i, o);
            if (out2) {
                if constexpr (!EARLY) ln_load4(w2 + i, g2[it]);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = v[it][e] * scale * g2[it][e];
                ln_store4(out2 + (size_t)out_row * n + i, o);
            }
            if constexpr (COLS > 0) ln_store4(row_lds + i, o);
        }
    }
    if constexpr (COLS > 0) {
        __syncthreads();
        router.route(route, row_lds, s_lds, c_lds, out_row, n, threadIdx.x / TLI_WAVE, threadIdx.x % TLI_WAVE);
    }
}

// Threads that share out a row: at least one quad each.
static int ln_threads(int quads) {
    int threads = 64;
    while (threads < 1024 && threads * 2 <= quads) threads *= 2;
    return threads;
}

template <typename T, bool SUMS>
static void launch_add_layernorm(float* resid, const void* d1, const void* d2, const OwedSums& sums, const float* w1, const float* w2,
                                 void* out1, void* out2, const int* rows, int out_rows, int total_rows, int n,
                                 float eps, hipStream_t s) {
    const uintptr_t all = (uintptr_t)resid | (uintptr_t)d1 | (uintptr_t)d2 | (uintptr_t)sums.p[0] | (uintptr_t)sums.p[1] | (uintptr_t)w1 | (uintptr_t)w2 |
                          (uintptr_t)out1 | (uintptr_t)out2;
    if (n % 4 == 0 && !(all & 15) && n <= 4 * 4 * 1024) {
        const int quads = n / 4, threads = ln_threads(quads);
        const int it = (quads + threads - 1) / threads;
#define TLI_LN(IT) hipLaunchKernelGGL((add_layernorm_vec_kernel<T, IT, SUMS>), dim3(out_rows), dim3(threads), 0, s, resid, \
                                      (const T*)d1, (const T*)d2, sums, w1, w2, (T*)out1, (T*)out2, rows, n, eps, total_rows, threads, RouteArgs{})
        if (it <= 1) TLI_LN(1);
        else if (it == 2) TLI_LN(2);
        else if (it == 3) TLI_LN(3);
        else TLI_LN(4);
#undef TLI_LN
        return;
    }
    hipLaunchKernelGGL((add_layernorm_kernel<T, SUMS>), dim3(out_rows), dim3(256), 0, s, resid, (const T*)d1, (const T*)d2, sums,
                       w1, w2, (T*)out1, (T*)out2, rows, n, eps, total_rows);
}

// d1, d2: rows of the dtype, or float32 partial sums [parts][total_rows][n] where parts1, parts2 > 0.
extern "C" int tli_add_layernorm(float* resid, const void* d1, int parts1, const void* d2, int parts2, const float* w1, const float* w2,
                                 void* out1, void* out2, const int* rows, int out_rows, int total_rows, int n,
                                 float eps, int dtype, void* stream) {
    if (out_rows <= 0) return 0;
    if (n <= 0) return tli_fail("add_layernorm: bad row size %d", n);
    if (parts1 < 0 || parts2 < 0) return tli_fail("add_layernorm: bad numbers of partial sums");
    const bool any = parts1 > 0 || parts2 > 0;
    const OwedSums sums{{parts1 > 0 ? (const float*)d1 : nullptr, parts2 > 0 ? (const float*)d2 : nullptr}, {d1 ? parts1 : 0, d2 ? parts2 : 0},
                        (size_t)total_rows * n};
    if (parts1 > 0) d1 = nullptr;
    if (parts2 > 0) d2 = nullptr;
    if (!w1 || !out1 || (out2 && !w2)) return tli_fail("add_layernorm: an output without its weight");
    hipStream_t s = (hipStream_t)stream;
#define TLI_LN_LAUNCH(T, SUMS) launch_add_layernorm<T, SUMS>(resid, d1, d2, sums, w1, w2, out1, out2, rows, out_rows, total_rows, n, eps, s)
    if (dtype == TLI_F32) {
        if (any) TLI_LN_LAUNCH(float, true);
        else TLI_LN_LAUNCH(float, false);
    } else if (dtype == TLI_BF16) {
        if (any) TLI_LN_LAUNCH(bf16_t, true);
        else TLI_LN_LAUNCH(bf16_t, false);
    } else {
        return tli_fail("add_layernorm: unknown dtype %d", dtype);
    }
#undef TLI_LN_LAUNCH
    return tli_check_launch("add_layernorm");
}

// The same for all rows in bfloat16, and the routed experts of the last output's rows (w2 and out2 null: the only one's): w_route
// [E (+ 1), n] and the rest as for tli_moe_router_bf16.  Takes what norm_route_takes says, everything 16-byte aligned; the same choice,
// weights and gates as that kernel's.
// A launch less a layer, which saves its start and the router's wait for rows that another launch wrote: 8 rows of 2,048, 16 experts and
// a shared gate, as part of a decode step, norm 4.8 us and router 6.5 before, 2.3 us less together now.
extern "C" int tli_add_layernorm_route_bf16(float* resid, const void* d1, int parts1, const void* d2, int parts2, const float* w1, const float* w2,
                                            void* out1, void* out2, int rows, int n, float eps, const void* w_route, int* ids, float* weights,
                                            float* shared_gate, int E, int top, int groups, int keep, float route_scale, int has_shared,
                                            int softmax_scores, int group_by_max, int normalize, const float* correction, void* stream) {
    if (rows <= 0) return 0;
    const RouteArgs route{(const bf16_t*)w_route, ids, weights, shared_gate, E, top, groups, keep, route_scale, has_shared, softmax_scores,
                          group_by_max, normalize, correction};
    if (const char* fault = route_fault(route)) return tli_fail("add_layernorm_route: %s", fault);
    if (!norm_route_takes(n, route.cols())) return tli_fail("add_layernorm_route: rows of %d, %d logits", n, route.cols());
    if (!w_route || !w1 || !out1 || (out2 && !w2) || parts1 < 0 || parts2 < 0) return tli_fail("add_layernorm_route: bad arguments");
    if (((uintptr_t)resid | (uintptr_t)d1 | (uintptr_t)d2 | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)out1 | (uintptr_t)out2 | (uintptr_t)w_route) & 15)
        return tli_fail("add_layernorm_route: operands must be 16-byte aligned");
    const OwedSums sums{{parts1 > 0 ? (const float*)d1 : nullptr, parts2 > 0 ? (const float*)d2 : nullptr}, {d1 ? parts1 : 0, d2 ? parts2 : 0},
                        (size_t)rows * n};
    const bool any = sums.parts[0] > 0 || sums.parts[1] > 0;
    if (sums.parts[0] > 0) d1 = nullptr;
    if (sums.parts[1] > 0) d2 = nullptr;
    const int span = ln_threads(n / 4);                      // (the threads that norm a row: as without a router)
#define TLI_LN_ROUTE(SUMS, COLS, KI, IT)                                                                                                \
    add_layernorm_vec_kernel<bf16_t, IT, SUMS, COLS, KI><<<rows, NORM_ROUTE_THREADS, 0, (hipStream_t)stream>>>(                         \
        resid, (const bf16_t*)d1, (const bf16_t*)d2, sums, w1, w2, (bf16_t*)out1, (bf16_t*)out2, nullptr, n, eps, rows, span, route)
#define TLI_LN_ROUTE_WIDTH(SUMS, COLS)                               \
    if (n <= 2048 && n / 4 <= span) TLI_LN_ROUTE(SUMS, COLS, 4, 1);  \
    else TLI_LN_ROUTE(SUMS, COLS, 8, 2);
#define TLI_LN_ROUTE_SUMS(SUMS)                                                                   \
    if (route.cols() <= NORM_ROUTE_THREADS / TLI_WAVE) { TLI_LN_ROUTE_WIDTH(SUMS, 1) }            \
    else { TLI_LN_ROUTE_WIDTH(SUMS, 2) }
    if (any) { TLI_LN_ROUTE_SUMS(true) }
    else { TLI_LN_ROUTE_SUMS(false) }
#undef TLI_LN_ROUTE_SUMS
#undef TLI_LN_ROUTE_WIDTH
#undef TLI_LN_ROUTE
    return tli_check_launch("add_layernorm_route");
}
