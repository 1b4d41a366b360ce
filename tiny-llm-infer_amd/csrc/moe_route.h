// The router of a row, where a workgroup has the row: the logits' choice by one wave (what is chosen: moe.hip), for the
// router's own kernel and for norms that a router reads.
#pragma once
#include "common.h"

#define MOE_MAX_TOP 32

struct RouteArgs {
    const bf16_t* w;             // [E (+ 1), n]: the router's rows, then the shared expert's gate; null: no router
    int* ids;                    // [rows, top]
    float* weights;              // [rows, top]
    float* shared_gate;          // [rows]
    int E, top, groups, keep;
    float scale;
    int has_shared, softmax_scores, group_by_max, normalize;
    const float* correction;     // [E] or null
    __host__ __device__ int cols() const { return E + (has_shared ? 1 : 0); }
};

static inline const char* route_fault(const RouteArgs& a) {
    if (a.E <= 0 || a.E > 2048 || a.top <= 0 || a.top > a.E || a.top > MOE_MAX_TOP || a.groups <= 0 || a.groups > 64 || a.E % a.groups ||
        a.keep <= 0 || a.keep > a.groups || (long long)a.keep * (a.E / a.groups) < a.top)
        return "bad sizes";
    if (!a.ids || !a.weights || (a.has_shared && !a.shared_gate)) return "missing outputs";
    return nullptr;
}

// What the choice goes by.  A score that is no number (a row with a NaN or an infinity in it) counts as the lowest: a NaN
// compares as neither larger nor smaller, the lanes of a choice would not agree on the largest, and an expert could be chosen
// twice.
__device__ __forceinline__ float choice_score(float v) { return v != v ? -INFINITY : v; }

// The largest of the lanes' values, ties to the lower index; every lane gets both.  (index < 0: the lane has none)
__device__ __forceinline__ void better_of(float& v, int& index, float ov, int oi) {
    if (oi >= 0 && (index < 0 || ov > v || (ov == v && oi < index))) v = ov, index = oi;
}
__device__ __forceinline__ void wave_best(float& v, int& index) {
    auto swapped = [&](const auto& a, const auto& b) {
        v = __uint_as_float(a[0]), index = (int)b[0];
        better_of(v, index, __uint_as_float(a[1]), (int)b[1]);
    };
    swapped(__builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false),
            __builtin_amdgcn_permlane32_swap((unsigned)index, (unsigned)index, false, false));
    swapped(__builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false),
            __builtin_amdgcn_permlane16_swap((unsigned)index, (unsigned)index, false, false));
    better_of(v, index, lane_xor8(v), __float_as_int(lane_xor8(__int_as_float(index))));
    better_of(v, index, lane_xor4(v), __float_as_int(lane_xor4(__int_as_float(index))));
    better_of(v, index, lane_xor2(v), __float_as_int(lane_xor2(__int_as_float(index))));
    better_of(v, index, lane_xor1(v), __float_as_int(lane_xor1(__int_as_float(index))));
}

// The choice of row t by one wave: s [E (+ 1)] holds the logits, c [E] the correction (or anything); both in LDS
__device__ __forceinline__ void route_choice(const RouteArgs& a, float* s, float* c, size_t t, int lane) {
    const int E = a.E, top = a.top, groups = a.groups, keep = a.keep;
    if (a.has_shared && lane == 0) a.shared_gate[t] = 1.0f / (1.0f + expf(-s[E]));
    if (a.softmax_scores) {
        float top_z = -INFINITY, sum = 0.f;
        for (int e = lane; e < E; e += TLI_WAVE) top_z = fmaxf(top_z, s[e]);
        top_z = wave_max(top_z);
        for (int e = lane; e < E; e += TLI_WAVE) {
            s[e] = expf(s[e] - top_z);
            sum += s[e];
        }
        sum = wave_sum(sum);
        for (int e = lane; e < E; e += TLI_WAVE) s[e] /= sum;
    } else {
        for (int e = lane; e < E; e += TLI_WAVE) s[e] = 1.0f / (1.0f + expf(-s[e]));
    }
    for (int e = lane; e < E; e += TLI_WAVE) c[e] = choice_score(a.correction ? s[e] + c[e] : s[e]);
    wave_lds_sync();
    const int per = E / groups;
    unsigned long long open = ~0ull;               // the `keep` best groups, a bit each (groups <= 64: one a lane)
    if (keep < groups) {
        open = 0ull;
        float g1 = -INFINITY, g2 = -INFINITY;      // the two largest of this lane's group
        if (lane < groups)
            for (int e = lane * per; e < (lane + 1) * per; ++e) {
                const float v = c[e];
                if (v > g1) { g2 = g1; g1 = v; }
                else if (v > g2) g2 = v;
            }
        const float score = (g2 > -INFINITY && !a.group_by_max) ? g1 + g2 : g1;
        for (int n = 0; n < keep; ++n) {
            float v = score;
            int g = lane < groups && !((open >> lane) & 1ull) ? lane : -1;
            wave_best(v, g);
            if (g >= 0) open |= 1ull << g;
        }
    }
    uint32_t taken = 0u;                           // of this lane's experts lane, lane + 64, .. (E <= 2048)
    float total = 0.f, mine = 0.f;                 // the weight of this lane's place in the choice (top <= 32)
    for (int n = 0; n < top; ++n) {
        float v = -INFINITY;
        int best = -1;
        for (int e = lane, k = 0; e < E; e += TLI_WAVE, ++k)
            if (!((taken >> k) & 1u) && ((open >> (e / per)) & 1ull) && (best < 0 || c[e] > v)) v = c[e], best = e;
        wave_best(v, best);
        if (best < 0) best = 0;                    // (not with sizes that the host lets through)
        if (best % TLI_WAVE == lane) taken |= 1u << (best / TLI_WAVE);
        total += s[best];
        if (lane == n) {
            mine = s[best];
            a.ids[t * top + n] = best;
        }
    }
    if (lane < top) a.weights[t * top + lane] = mine * (a.normalize ? a.scale / (total + 1e-20f) : a.scale);
}

// Norms that a router reads: the kernel that makes a row makes its logits and choice too.  A wave makes the logits
// wave, wave + WAVES, .. (COLS of them) of a row of up to 512 KI elements in LDS, from weights that it asked for before the
// row was there, with the sums in the order of moe_router_kernel.
template <int COLS, int KI, int WAVES>
struct RouteRows {
    static constexpr int HELD = COLS > 0 ? COLS : 1;
    uint4 v[HELD][KI];
    __device__ __forceinline__ void fetch(const RouteArgs& a, int n, int wave, int lane) {
#pragma unroll
        for (int j = 0; j < COLS; ++j) {
            const bf16_t* w = a.w + (size_t)min(wave + j * WAVES, a.cols() - 1) * n;   // (past the last row: the last one again, not kept)
#pragma unroll
            for (int i = 0; i < KI; ++i) {
                const int at = (i * TLI_WAVE + lane) * 8;
                v[j][i] = at < n ? *reinterpret_cast<const uint4*>(w + at) : make_uint4(0, 0, 0, 0);
            }
        }
    }
    // row: the row in LDS, complete; s [E + 1], c [E]: LDS of the choice, c holding the correction
    __device__ __forceinline__ void route(const RouteArgs& a, const bf16_t* row, float* s, float* c, size_t t, int n, int wave, int lane) {
        float sum[HELD];
#pragma unroll
        for (int j = 0; j < COLS; ++j) sum[j] = 0.f;
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int at = (i * TLI_WAVE + lane) * 8;
            const uint4 x = at < n ? *reinterpret_cast<const uint4*>(row + at) : make_uint4(0, 0, 0, 0);
            const uint32_t u[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int j = 0; j < COLS; ++j) {
                const uint32_t w[4] = {v[j][i].x, v[j][i].y, v[j][i].z, v[j][i].w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    sum[j] = fmaf(__uint_as_float(u[k] << 16), __uint_as_float(w[k] << 16), sum[j]);
                    sum[j] = fmaf(__uint_as_float(u[k] & 0xFFFF0000u), __uint_as_float(w[k] & 0xFFFF0000u), sum[j]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < COLS; ++j) {
            const float z = wave_sum(sum[j]);
            if (lane == 0 && wave + j * WAVES < a.cols()) s[wave + j * WAVES] = z;
        }
        __syncthreads();
        if (wave == 0) route_choice(a, s, c, t, lane);
    }
};

// What a norm with a router takes: up to 32 logits (two a wave of 1,024 threads), rows of up to 4,096 elements in 8s: the weights that a
// wave holds are 64 registers then, of the 128 a lane has with so many threads, and a third logit or a longer row does not fit
// beside the row.  With the router on its own and in the norm's launch, us, a shared gate beside the experts: rows of 512, 8 experts, 1 row
// 6.1 and 5.7 (layer norms), 6.2 and 5.7 (norm_add_norm), 128 rows 6.8 and 6.2, 6.9 and 6.2; rows of 4,096, 31 experts, 1 row 13.3 and 12.5,
// 13.5 and 12.7, 128 rows 14.7 and 13.5, 14.7 and 13.6.  (More than 128 rows are prompts' in the main: ROUTER_ROWS of kernels/ops.py.)
#define NORM_ROUTE_THREADS 1024
#define NORM_ROUTE_COLS 32
#define NORM_ROUTE_MAX 4096
static inline bool norm_route_takes(int n, int cols) { return n > 0 && n % 8 == 0 && n <= NORM_ROUTE_MAX && cols <= NORM_ROUTE_COLS; }
