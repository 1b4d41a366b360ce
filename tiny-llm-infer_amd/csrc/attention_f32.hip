// Attention of the float32 path over the paged cache, a workgroup a (row, head): as attention_plain.hip, which walks 256 keys
// at a time with a key a thread and stays for what this kernel does not take (heads that are no multiple of 64, pages of fewer
// than four slots) and as its reference.
//
// The keys go to the four waves in blocks of 16, in turn; a wave keeps a running maximum, sum and output of its own, and the
// four are joined at the end.  In a block four lanes share a key (lane 16 c + j: quarter c of key j, 16 bytes a load), then a
// lane takes every 64th output element and the block's 16 values of it, four to a load.  What bounds a decode step's few short
// rows is the chain of loads of one block after the other, which is a quarter as long here and has all its loads in flight:
// 5 rows of up to 52 keys, 16 heads of 64: 15.9 -> 4.8 us, most of it the launch.  Longer rows and prompts, the plain kernel and
// this one (both with the 12 us of a launch from Python), 16 heads of 64 and 32 of 128: 1 row of 200 keys 44.9 -> 13.0 and 46.4 ->
// 12.9 us, of 4,000 850 -> 97 and 921 -> 148, of 16,000 3,535 -> 408 and 3,668 -> 578; 8 rows of 4,000 887 -> 104 and 929 -> 150; 64
// of 600 159 -> 35 and 525 -> 135; a prompt of 32 tokens 12.2 -> 12.2 and 14.8 -> 12.6, of 512 441 -> 109 and 1,297 -> 394, of 2,048
// 5.74 -> 1.46 and 19.6 -> 5.63 ms; heads of 192 and 256 1.04 to 5 times.
// The order of additions depends on the row's first and last key alone.
#include "gemm_reduce.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(4))) float f32x4;

#define AF_WAVES 4

// The projections of a decode step's rows, [planes][rows][(heads + 2 kv_heads) D] (planes > 1: partial sums), and what is done to them.
struct RawRows {
    const float* qkv;
    int planes;
    const float *q_norm_w, *k_norm_w;
    float q_eps, k_eps;
    const float *cos_table, *sin_table;
    int rotary_dim, table_positions;
    int write_cache;
};

// v[e] = sum_planes(at + 64 e, ..), every element's planes asked for before any is added: one trip to memory where one by one they are E.
template <int E>
__device__ __forceinline__ void sum_planes_of(float (&v)[E], const float* __restrict__ at, int planes, size_t plane) {
    if (planes == 1) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = at[e * 64];
        return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = 0.f;
    for (int s = 0; s < planes; s += 8) {
        float p[8][E];
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int e = 0; e < E; ++e) p[k][e] = at[(size_t)min(s + k, planes - 1) * plane + e * 64];
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = s + k < planes ? v[e] + p[k][e] : v[e];
    }
}

// x[D] in LDS: norm (weight `nw` or null) and rotation of a head that this wavefront takes from `src`, as qkv_to_cache_kernel does them.
template <int DH>
__device__ __forceinline__ void head_of_raw_row(float* x, const float* src, size_t plane, const RawRows& raw, const float* nw, float eps,
                                                const float* cos_row, const float* sin_row, int lane) {
    constexpr int D = DH * 64;
    float v[DH], w[DH], ss = 0.f;
#pragma unroll
    for (int e = 0; e < DH; ++e) w[e] = nw ? nw[e * 64 + lane] : 0.f;
    sum_planes_of(v, src + lane, raw.planes, plane);
#pragma unroll
    for (int e = 0; e < DH; ++e) ss = fmaf(v[e], v[e], ss);      // (written out: the sums of qkv_to_cache_kernel, bit for bit)
    if (nw) {
        const float scale = 1.0f / sqrtf(wave_sum(ss) / (float)D + eps);
#pragma unroll
        for (int e = 0; e < DH; ++e) v[e] = w[e] * v[e] * scale;
    }
#pragma unroll
    for (int e = 0; e < DH; ++e) x[e * 64 + lane] = v[e];
    if (!cos_row) return;
    wave_lds_sync();
    const int half = raw.rotary_dim / 2;
#pragma unroll
    for (int e = 0; e < DH; ++e) {
        const int i = e * 64 + lane;
        if (i < half) v[e] = rotate_first_half(v[e], x[i + half], cos_row[i], sin_row[i]);
        else if (i < raw.rotary_dim) v[e] = rotate_second_half(v[e], x[i - half], cos_row[i - half], sin_row[i - half]);
    }
    wave_lds_sync();
#pragma unroll
    for (int e = 0; e < DH; ++e) x[e * 64 + lane] = v[e];
}

// RAW: decode steps (one row a sequence) from the projections: every workgroup makes its query and its row's own key and value, the first
// head of a group writes these into the cache, and every head takes them from LDS, not from the cache, so that nothing waits for a store.
// The same bits as qkv_to_cache and the kernel without RAW, which is two launches and a trip of q through memory; most of either is launch and
// latency.  In a recorded chain, 16 heads of 64, projections as eight partial sums, us: 1 row of 30 keys 6.4 -> 4.9, 5 rows of 52 6.9 -> 5.4, 8 of
// 200 10.8 -> 9.5, 1 of 1,000 29.0 -> 27.4.
// APART: the one block with the row's own key apart from the loop, whose registers and order of loads what is done to it would change (RAW only).
template <int DH, bool RAW, bool APART>            // head_dim / 64
__global__ void __launch_bounds__(AF_WAVES * 64) attention_f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, float* __restrict__ k_cache, float* __restrict__ v_cache, RawRows raw,
    const int* __restrict__ positions, const int* __restrict__ seq_of_row, const int* __restrict__ tables, int table_width,
    int page_size, int num_pages, int heads, int kv_heads, float scale, int window) {
    constexpr int D = DH * 64;
    __shared__ __attribute__((aligned(16))) float p_s[AF_WAVES][16];
    __shared__ float m_s[AF_WAVES], l_s[AF_WAVES], o_s[AF_WAVES][D];
    const int row = blockIdx.x, head = blockIdx.y;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int j = lane % 16, c = lane / 16;
    const int g = head / (heads / kv_heads);
    const int pos = positions[row];
    const int* table = tables + (size_t)seq_of_row[row] * table_width;
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const size_t page_stride = (size_t)kv_heads * page_size * D;
    const float* k_head = k_cache + (size_t)g * page_size * D;
    const float* v_head = v_cache + (size_t)g * page_size * D;

    // this lane's quarter of the query: elements 16 i + 4 c .. + 4
    f32x4 qv[DH * 4];
    __shared__ __attribute__((aligned(16))) float own_s[RAW ? 3 : 1][RAW ? D : 4];      // RAW: the query, the row's own key and value
    const bool own = RAW && raw.write_cache;
    if constexpr (RAW) {
        const int width = (heads + 2 * kv_heads) * D;
        const float* src = raw.qkv + (size_t)row * width;
        const size_t plane = (size_t)gridDim.x * width;
        const bool turned = raw.cos_table && pos >= 0 && pos < raw.table_positions;
        const float* cos_row = turned ? raw.cos_table + (size_t)pos * (raw.rotary_dim / 2) : nullptr;
        const float* sin_row = turned ? raw.sin_table + (size_t)pos * (raw.rotary_dim / 2) : nullptr;
        const int page = own && head % (heads / kv_heads) == 0 ? table[pos / page_size] : -1;
        const bool store = page >= 0 && page < num_pages;
        if (wave == 0) head_of_raw_row<DH>(own_s[0], src + (size_t)head * D, plane, raw, raw.q_norm_w, raw.q_eps, cos_row, sin_row, lane);
        if (wave == 1 && own) {
            head_of_raw_row<DH>(own_s[1], src + (size_t)(heads + g) * D, plane, raw, raw.k_norm_w, raw.k_eps, cos_row, sin_row, lane);
            if (store)
#pragma unroll
                for (int e = 0; e < DH; ++e)                    // (a lane's own elements)
                    k_cache[(size_t)page * page_stride + ((size_t)g * page_size + pos % page_size) * D + e * 64 + lane] = own_s[1][e * 64 + lane];
        }
        if (wave == 2 && own) {
            float sums[DH];
            sum_planes_of(sums, src + (size_t)(heads + kv_heads + g) * D + lane, raw.planes, plane);
#pragma unroll
            for (int e = 0; e < DH; ++e) {
                const float v = cache_value(sums[e]);
                own_s[2][e * 64 + lane] = v;
                if (store) v_cache[(size_t)page * page_stride + ((size_t)g * D + e * 64 + lane) * page_size + pos % page_size] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < DH * 4; ++i) qv[i] = *reinterpret_cast<const f32x4*>(&own_s[0][i * 16 + c * 4]);
    } else {
        const float* q_row = q + ((size_t)row * heads + head) * D + c * 4;
#pragma unroll
        for (int i = 0; i < DH * 4; ++i) qv[i] = *reinterpret_cast<const f32x4*>(q_row + i * 16);
    }
    float m = -INFINITY, l = 0.f, o[DH];
#pragma unroll
    for (int i = 0; i < DH; ++i) o[i] = 0.f;
    auto page_of = [&](int t) { return t <= pos ? table[t / page_size] : -1; };

    // a block of 16 keys; OWN: RAW, and the row's own key may be among them
    auto block = [&](int base, auto OWN) __attribute__((always_inline)) {
        const int t = base + j;
        const int page = page_of(t);
        const bool seen = t >= lo && page >= 0 && page < num_pages;
        const float* kp = k_head + (size_t)(seen ? page : 0) * page_stride + (size_t)(t % page_size) * D + c * 4;
        f32x4 kv[DH * 4];
#pragma unroll
        for (int i = 0; i < DH * 4; ++i) kv[i] = *reinterpret_cast<const f32x4*>(kp + i * 16);
        // the values of the block: groups of four slots never straddle a page
        int v_page[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v_page[u] = page_of(base + 4 * u);
        f32x4 vv[DH][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool held = v_page[u] >= 0 && v_page[u] < num_pages;
            const float* vp = v_head + (size_t)(held ? v_page[u] : 0) * page_stride + (size_t)lane * page_size + (base + 4 * u) % page_size;
#pragma unroll
            for (int i = 0; i < DH; ++i) vv[i][u] = *reinterpret_cast<const f32x4*>(vp + (size_t)i * 64 * page_size);
        }
        if (decltype(OWN)::value && own && base + 16 > pos) {
            // the row's own slot, which another workgroup may be writing just now: what was read of it is not used
            if (t == pos)
#pragma unroll
                for (int i = 0; i < DH * 4; ++i) kv[i] = *reinterpret_cast<const f32x4*>(&own_s[RAW ? 1 : 0][(i * 16 + c * 4) % (RAW ? D : 4)]);
#pragma unroll
            for (int i = 0; i < DH; ++i) {
                const float mine = own_s[RAW ? 2 : 0][RAW ? i * 64 + lane : 0];
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < 4; ++e) vv[i][u][e] = base + 4 * u + e == pos ? mine : vv[i][u][e];
            }
        }
        f32x4 dot = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < DH * 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) dot[e] = fmaf(qv[i][e], kv[i][e], dot[e]);
        const float s = quad_rows_sum((dot[0] + dot[1]) + (dot[2] + dot[3])) * scale;
        const float score = seen ? s : -INFINITY;
        float top = score;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 16));
        if (!__any(score != -INFINITY)) return;                 // (nothing of this block counts: the same for the whole wave)
        // (a maximum passes NaNs over, the weights and their sum do not: a row with a NaN in it comes out as NaNs)
        const float m_new = fmaxf(m, top);
        const float p = !seen ? -0.f : score == -INFINITY ? 0.f : expf(score - m_new);
        const float corr = m == -INFINITY ? 0.f : expf(m - m_new);
        float sum = p;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 16);
        l = l * corr + sum;
        m = m_new;
        if (c == 0) p_s[wave][j] = p;
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < DH; ++i) o[i] *= corr;
        auto add = [&](auto WHOLE) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const f32x4 w = *reinterpret_cast<const f32x4*>(&p_s[wave][4 * u]);
#pragma unroll
                for (int i = 0; i < DH; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float next = fmaf(w[e], vv[i][u][e], o[i]);
                        o[i] = decltype(WHOLE)::value || __float_as_int(w[e]) >= 0 ? next : o[i];
                    }
            }
        };
        // what lies in a slot that is not this row's (its weight is -0) need not be a number, and 0 times it need not be 0
        if (__all(seen)) add(std::true_type{});
        else add(std::false_type{});
        wave_lds_sync();
    };
    int base = (lo / 16 + wave) * 16;
    for (; APART ? base + 16 <= pos : base <= pos; base += 16 * AF_WAVES) {
        if (RAW && !APART) block(base, std::true_type{});
        else block(base, std::false_type{});
    }
    if (APART && base <= pos) block(base, std::true_type{});
    if (lane == 0) {
        m_s[wave] = m;
        l_s[wave] = l;
    }
#pragma unroll
    for (int i = 0; i < DH; ++i) o_s[wave][i * 64 + lane] = o[i];
    __syncthreads();
    float best = m_s[0];
#pragma unroll
    for (int w = 1; w < AF_WAVES; ++w) best = fmaxf(best, m_s[w]);
    float total = 0.f, share[AF_WAVES];
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
        share[w] = m_s[w] == -INFINITY ? 0.f : expf(m_s[w] - best);
        total += l_s[w] * share[w];
    }
    const float inv = total > 0.f ? 1.0f / total : 0.f;
    for (int d = threadIdx.x; d < D; d += AF_WAVES * 64) {
        float y = 0.f;
#pragma unroll
        for (int w = 0; w < AF_WAVES; ++w) y = fmaf(share[w], o_s[w][d], y);
        out[((size_t)row * heads + head) * D + d] = y * inv;
    }
}

template <bool RAW>
static void launch_attention_f32(dim3 grid, const float* q, float* out, float* k_cache, float* v_cache, const RawRows& raw, const int* positions,
                                 const int* seq_of_row, const int* tables, int table_width, int page_size, int num_pages, int heads,
                                 int kv_heads, int head_dim, float scale, int window, hipStream_t s) {
#define TLI_AF(DH, APART)                                                                                                                  \
    attention_f32_kernel<DH, RAW, APART><<<grid, AF_WAVES * 64, 0, s>>>(q, out, k_cache, v_cache, raw, positions, seq_of_row, tables,        \
                                                                        table_width, page_size, num_pages, heads, kv_heads, scale, window)
    // The row's own key in the loop and apart, projections of k 1,024 included, us: 4 heads of 256, 1 row of 2,000 keys 137.5 and 118.5, 16 rows 128.2
    // and 113.8; 16 heads of 64 60.5 and 57.6, 63.9 and 60.7.  Heads of 128 are better off in the loop while there is no more than a workgroup a compute
    // unit, and worse from two on (attention alone; two launches, in the loop, apart): 32 heads, 8 rows of 700 keys 32.4, 28.0 and 30.1, of 4,000 148, 135 and
    // 147; 16 rows of 2,000 99.4, 102.5 and 96.3; 16 heads, 32 rows of 4,000 255, 263 and 250.
    switch (head_dim / 64) {
        case 1: TLI_AF(1, RAW); break;
        case 2:
            if (RAW && (long)grid.x * grid.y > tli_compute_units()) TLI_AF(2, RAW);
            else TLI_AF(2, false);
            break;
        case 3: TLI_AF(3, RAW); break;
        default: TLI_AF(4, RAW); break;
    }
#undef TLI_AF
}

extern "C" int tli_attention_f32_takes(int head_dim, int page_size) {
    return head_dim > 0 && head_dim % 64 == 0 && head_dim <= 256 && page_size >= 4 && page_size % 4 == 0;
}

// As tli_attention_plain, float32.
extern "C" int tli_attention_f32(const void* q, void* out, void* k_cache, void* v_cache, const int* positions,
                                 const int* seq_of_row, const int* tables, int table_width, int page_size, int num_pages, int rows,
                                 int heads, int kv_heads, int head_dim, float scale, int window, void* stream) {
    if (rows <= 0) return 0;
    if (!tli_attention_f32_takes(head_dim, page_size))
        return tli_fail("attention_f32: heads of %d (64, 128, 192, 256) or pages of %d slots are not taken", head_dim, page_size);
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || heads > 65535)
        return tli_fail("attention_f32: %d heads cannot be grouped over %d kv heads", heads, kv_heads);
    if (table_width <= 0 || num_pages <= 0) return tli_fail("attention_f32: bad cache geometry");
    if (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15) return tli_fail("attention_f32: operands must be 16-byte aligned");
    const dim3 grid(rows, heads);
    launch_attention_f32<false>(grid, (const float*)q, (float*)out, (float*)k_cache, (float*)v_cache, RawRows{}, positions, seq_of_row, tables,
                                table_width, page_size, num_pages, heads, kv_heads, head_dim, scale, window, (hipStream_t)stream);
    return tli_check_launch("attention_f32");
}

extern "C" int tli_qkv_to_cache(const void* qkv, int planes, void* q_out, void* k_cache, void* v_cache, const int* positions, const int* seq_of_row,
                                const int* tables, int table_width, int page_size, int num_pages, int rows, int heads, int kv_heads, int head_dim,
                                const float* q_norm_w, float q_eps, const float* k_norm_w, float k_eps, const float* cos_table,
                                const float* sin_table, int rotary_dim, int table_positions, int write_cache, int skip_values, int dtype, void* stream);

// Whether a decode step's rows of up to `keys` keys are sooner done in one launch from the projections than in two.  Every workgroup makes its own
// query and its group's key and value, and has more registers for it, so two launches are as good where the workgroups are many times what the chip
// holds and each has few keys, with heads of 256 any number of them; and, where no heads share a key, from 2 GB of keys and values on, which come from memory at its
// rate.  us, two launches and one: 512 rows of 20 keys, 32 heads of 64 43.1, 49.2, of 60 62.2, 62.7; 8 heads of 192 34.0, 35.7 and 55.2, 59.8, of 250 204, 199; 8 heads of 256
// 47.0, 53.2 and 80.0, 85.7, 16 of them with 500 keys 1,212, 1,234; 16 heads of 128 with a key each, 128 rows of 1,000 366, 380, of 300 128.5, 123.3.
// At the limits: 4,096 heads of rows of 64, 20 keys 14.6, 14.5, 50 keys 20.7, 18.8; of 128 23.6, 23.4 and 35.6, 33.6; 2,048 of 192 20.5, 19.8 and 28.9, 28.3; 1,536 of 256
// 20.3, 20.1 and 30.3, 28.3, 2,048 of 300 keys 128, 124.
extern "C" int tli_qkv_attention_f32_one(int rows, int heads, int kv_heads, int head_dim, int keys) {
    const long wgs = (long)rows * heads, units = tli_compute_units(), elements = wgs * head_dim;
    if (heads == kv_heads) return keys <= 128 || elements < 1024 * units || elements * keys < 1024 * 1024 * units;
    if (keys <= 128) return wgs <= (head_dim <= 128 ? 16 : head_dim <= 192 ? 8 : 6) * units;
    return head_dim <= 192 || wgs <= 8 * units;
}

// From the rows' projections qkv [planes][rows][(heads + 2 kv_heads) head_dim] (planes > 1: partial sums to be added) to the attention's output.
// `q` null: a decode step (one row a sequence) in one launch.  Else q [rows][heads * head_dim] takes the queries and it is tli_qkv_to_cache,
// then tli_attention_f32: a row of a portion also reads the keys of the rows before it.
extern "C" int tli_qkv_attention_f32(const void* qkv, int planes, void* q, void* out, void* k_cache, void* v_cache, const int* positions,
                                     const int* seq_of_row, const int* tables, int table_width, int page_size, int num_pages, int rows,
                                     int heads, int kv_heads, int head_dim, const float* q_norm_w, float q_eps, const float* k_norm_w,
                                     float k_eps, const float* cos_table, const float* sin_table, int rotary_dim, int table_positions,
                                     int write_cache, float scale, int window, void* stream) {
    if (rows <= 0) return 0;
    if (!tli_attention_f32_takes(head_dim, page_size))
        return tli_fail("qkv_attention_f32: heads of %d (64, 128, 192, 256) or pages of %d slots are not taken", head_dim, page_size);
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || heads > 65535)
        return tli_fail("qkv_attention_f32: %d heads cannot be grouped over %d kv heads", heads, kv_heads);
    if (table_width <= 0 || num_pages <= 0 || planes < 1) return tli_fail("qkv_attention_f32: bad cache geometry or planes");
    if ((cos_table == nullptr) != (sin_table == nullptr)) return tli_fail("qkv_attention_f32: cos without sin");
    if (cos_table && (rotary_dim <= 0 || rotary_dim % 2 || rotary_dim > head_dim))
        return tli_fail("qkv_attention_f32: rotary_dim %d must be even and at most head_dim %d", rotary_dim, head_dim);
    if (((uintptr_t)k_cache | (uintptr_t)v_cache) & 15) return tli_fail("qkv_attention_f32: the cache must be 16-byte aligned");
    if (q) {
        const int fault = tli_qkv_to_cache(qkv, planes, q, k_cache, v_cache, positions, seq_of_row, tables, table_width, page_size, num_pages, rows,
                                           heads, kv_heads, head_dim, q_norm_w, q_eps, k_norm_w, k_eps, cos_table, sin_table, rotary_dim,
                                           table_positions, write_cache, 0, TLI_F32, stream);
        return fault ? fault : tli_attention_f32(q, out, k_cache, v_cache, positions, seq_of_row, tables, table_width, page_size, num_pages, rows,
                                                 heads, kv_heads, head_dim, scale, window, stream);
    }
    const RawRows raw{(const float*)qkv, planes, q_norm_w, k_norm_w, q_eps, k_eps, cos_table, sin_table, rotary_dim, table_positions, write_cache};
    launch_attention_f32<true>(dim3(rows, heads), nullptr, (float*)out, (float*)k_cache, (float*)v_cache, raw, positions, seq_of_row, tables,
                               table_width, page_size, num_pages, heads, kv_heads, head_dim, scale, window, (hipStream_t)stream);
    return tli_check_launch("qkv_attention_f32");
}
