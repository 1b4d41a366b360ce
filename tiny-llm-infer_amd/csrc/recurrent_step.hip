// Decode steps of the recurrent layers whose heads are normed one by one (retention.hip, mlstm.hip, wkv.hip): every sequence brings
// one row, and everything between the layer's products is one launch, a workgroup a (head, row).
//   retention:  q, k turned, k scaled; S <- c S + k v^T; o = S^T q; unit RMS; silu gate
//   mLSTM:      the two gates' logits (two dot products over the layer's input, which no other head shares), m, S <- a S +
//               b k v^T, n likewise, o = S^T q / (max(|n q|, exp(-m)) + 1e-6); RMS times the weight; logistic gate
//   wkv:        d = exp(-exp(W2 tanh(z) + w0)) a channel; o = (S + diag(u) k v^T)^T r; S <- diag(d) S + k v^T; RMS times the
//               weight; silu gate
// A column of S belongs to 16 lanes of a wave, a lane holding R elements of it (as in lightning.hip: pieces of up to four
// that lie side by side with the other lanes').  A workgroup takes 32 columns at a time (16 with 256 threads: step_wide says which) and
// asks for the row's own operands, then for the first GROUPS times as many columns, so that the state's bytes, which are nearly all
// that such a step moves, are on their way while the row's q, k, v and gates are made, and nothing of the row waits behind them.  256 threads
// that asked for the state first and for the decays' matrix after the row's tanh, and 512 in this order, 8 rows of 16 heads of
// 128 x 128 as part of a decode step: retention 9.8 us and 7.0, mLSTM 11.6 and 8.6, wkv 12.3 and 8.4.
#include "recurrence.h"
#include "row_gates.h"

__device__ __forceinline__ float rs_sum16(float v) {     // over the 16 lanes of a DPP row; every lane gets it
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));
    return v;
}

enum { STEP_RETENTION = 0, STEP_MEMORY = 1, STEP_WKV = 2 };

struct StepRows {                                        // what all kinds read and write
    const void* proj;                                    // [rows, ld]: q (H dk) | k (H dk) | v (H dv) | gate (H dv)
    int ld;
    void* out;                                           // rows out_ld elements apart, H dv of each
    int out_ld;
    float* state;                                        // [slots][H][OV][dk], OV = dv (retention) or dv + 1
    const int* seq_start;
    const int* slots;
    int rows, H, dk, dv;
    float eps, scale;                                    // of the norm; of the output
};

struct StepRetention {
    const int* positions;
    const float* decay;                                  // [H]
    const float* cos_table;                              // [table_positions, dims / 2] or null
    const float* sin_table;
    int dims, pairing, table_positions;
    float k_scale;
};

struct StepMemory {
    const void* x;                                       // [rows, n]: the layer's input
    const void* w;                                       // [2 H, n]: the gates' rows
    int n;
    RowFactor factor;                                    // of x
    const float* bias;                                   // [2 H]
    const float* weight;                                 // [H dv]
    float* m_state;                                      // [slots, H]
    float cap, q_scale;
};

struct StepTimeMix {
    const float* z;                                      // the decays' inner rows, before tanh: element i of row r at r z_row + i z_col
    long long z_row, z_col;
    const void* w2;                                      // [H dk, rank]
    const float* w0;                                     // [H dk]
    int rank;
    const float* u;                                      // [H, dk]
    const float* weight;                                 // [H dv]
};

// elements i .. i + 7 of a row of T where `eight`, else element i alone
template <typename T>
__device__ __forceinline__ float rs_dot8(const T* a, const T* b) {
    if constexpr (sizeof(T) == 2) {
        const uint4 x = *reinterpret_cast<const uint4*>(a), y = *reinterpret_cast<const uint4*>(b);
        const uint32_t u[4] = {x.x, x.y, x.z, x.w}, v[4] = {y.x, y.y, y.z, y.w};
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = fmaf(bf16_to_f32((bf16_t)(u[i] & 0xffffu)), bf16_to_f32((bf16_t)(v[i] & 0xffffu)), s);
            s = fmaf(bf16_to_f32((bf16_t)(u[i] >> 16)), bf16_to_f32((bf16_t)(v[i] >> 16)), s);
        }
        return s;
    } else {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) s = fmaf(a[i], b[i], s);
        return s;
    }
}

// T: of the projections; TO: of the output and the matrices
template <int KIND, int R, int THREADS, typename T, typename TO>
__global__ __launch_bounds__(THREADS) void recurrent_step_kernel(StepRows a, StepRetention ret, StepMemory mem, StepTimeMix mix) {
    constexpr bool MEMORY = KIND == STEP_MEMORY, WKV = KIND == STEP_WKV;
    constexpr int L = 16, DKP = L * R, NC = THREADS / L;
    constexpr int GROUPS = THREADS == 512 ? 4 : 8;                     // of NC columns, in flight together
    constexpr int VW = R % 4 == 0 ? 4 : R % 2 == 0 ? 2 : 1;
    extern __shared__ __align__(16) float rs_lds[];
    constexpr int WAVES = THREADS / TLI_WAVE;
    __shared__ float red[3 * WAVES < 16 ? 16 : 3 * WAVES];              // (block_sum asks for 16)
    const int h = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, sub = tid % L, jl = tid / L;
    const int dk = a.dk, dv = a.dv, H = a.H, OV = dv + (MEMORY ? 1 : 0);
    float* q_s = rs_lds;
    float* k_s = q_s + DKP;
    float* o_s = k_s + DKP;                                            // [OV]
    float* v_s = o_s + OV;                                             // [OV]
    float* d_s = v_s + OV;                                             // wkv: [DKP] decays,
    float* z_s = d_s + DKP;                                            // [rank]
    auto at = [&](int r) { return (r / VW) * (L * VW) + sub * VW + r % VW; };
    const int slot = a.slots[row];
    const bool fresh = a.seq_start[row] == 0;
    float* S_head = a.state + ((size_t)slot * H + h) * OV * dk;
    const bool whole = dk == DKP && dk % 4 == 0;
    float S[GROUPS][R], n[MEMORY ? R : 1];               // n: the mLSTM's normaliser, column dv, with the first 16 lanes
    auto load_column = [&](int j, auto& c) {
#pragma unroll
        for (int r = 0; r < R; ++r) c[r] = 0.f;
        if (fresh) return;
        const float* col = S_head + (size_t)j * dk;
        if (whole) {
#pragma unroll
            for (int r = 0; r < R; r += VW) {
                if constexpr (VW == 4) {
                    const float4 v = *reinterpret_cast<const float4*>(col + at(r));
                    c[r] = v.x, c[r + 1] = v.y, c[r + 2] = v.z, c[r + 3] = v.w;
                } else if constexpr (VW == 2) {
                    const float2 v = *reinterpret_cast<const float2*>(col + at(r));
                    c[r] = v.x, c[r + 1] = v.y;
                } else {
                    c[r] = col[at(r)];
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (at(r) < dk) c[r] = col[at(r)];
        }
    };
    auto store_column = [&](int j, const auto& c) {
        float* col = S_head + (size_t)j * dk;
        if (whole) {
#pragma unroll
            for (int r = 0; r < R; r += VW) {
                if constexpr (VW == 4) *reinterpret_cast<float4*>(col + at(r)) = make_float4(c[r], c[r + 1], c[r + 2], c[r + 3]);
                else if constexpr (VW == 2) *reinterpret_cast<float2*>(col + at(r)) = make_float2(c[r], c[r + 1]);
                else col[at(r)] = c[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (at(r) < dk) col[at(r)] = c[r];
        }
    };
    auto load = [&](int j0) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
            if (j0 + g * NC + jl < dv) load_column(j0 + g * NC + jl, S[g]);
    };
    // The row's operands first, into registers: an element of q or k a thread (2 DKP <= THREADS), one of v, of the gate and of the norm's
    // weights (more in rounds below), and what the kind needs.  Loads complete in the order of issue, so none of them waits for the
    // state, and the state is on its way while they are worked on.
    static_assert(2 * DKP <= THREADS, "an element of q or k a thread");
    const T* src = (const T*)a.proj + (size_t)row * a.ld;
    const T* q_src = src + (size_t)h * dk;
    const T* k_src = src + (size_t)(H + h) * dk;
    const T* v_src = src + (size_t)2 * H * dk + (size_t)h * dv;
    const T* g_src = src + (size_t)H * (2 * dk + dv) + (size_t)h * dv;
    const float* weight = MEMORY ? mem.weight + h * dv : WKV ? mix.weight + h * dv : nullptr;
    const bool is_k = tid >= DKP;
    const int own = is_k ? tid - DKP : tid;                            // this thread's element
    const bool owns = tid < 2 * DKP && own < dk;
    const T* own_src = is_k ? k_src : q_src;
    T qk_raw{}, other_raw{}, v_raw{}, g_raw{};
    float weight_raw = 1.f;
    if (owns) qk_raw = own_src[own];
    if (tid < dv) {
        v_raw = v_src[tid];
        g_raw = g_src[tid];
        if (MEMORY || WKV) weight_raw = weight[tid];
    }
    float keep = 0.f, floor_ = 0.f;
    float turn_cos = 1.f, turn_sin = 0.f;                              // retention: of this thread's element
    bool turned = false, second = false;
    constexpr int P = THREADS / DKP;                                // wkv: neighbouring threads that share out a channel's row of W2
    constexpr int HELD = P >= 16 ? 1 : P >= 8 ? 2 : 4;                 //      16-byte pieces of it that a thread holds
    const int channel = tid / P, part = tid % P;
    const TO* w2 = WKV ? (const TO*)mix.w2 + (size_t)(h * dk + min(channel, dk - 1)) * mix.rank : nullptr;
    const bool pieces = WKV && sizeof(TO) == 2 && mix.rank % 8 == 0;
    uint4 w2_raw[WKV ? HELD : 1];
    float z_raw = 0.f, w0_raw = 0.f, u_raw[WKV ? R : 1];
    float zi = 0.f, zf = 0.f, ss = 0.f, m0 = 0.f;                      // mLSTM: this thread's parts of the gates' sums
    float* m_slot = MEMORY ? mem.m_state + (size_t)slot * H + h : nullptr;
    if constexpr (WKV) {
        if (tid < mix.rank) z_raw = mix.z[row * mix.z_row + tid * mix.z_col];
        w0_raw = mix.w0[h * dk + min(channel, dk - 1)];
        if (pieces) {
#pragma unroll
            for (int e = 0; e < HELD; ++e) {
                const int i = (part + e * P) * 8;
                w2_raw[e] = i < mix.rank ? *reinterpret_cast<const uint4*>(w2 + i) : make_uint4(0, 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) u_raw[r] = at(r) < dk ? mix.u[h * dk + at(r)] : 0.f;
    } else if constexpr (MEMORY) {
        const T* x = (const T*)mem.x + (size_t)row * mem.n;
        const T* wi = (const T*)mem.w + (size_t)h * mem.n;
        const T* wf = (const T*)mem.w + (size_t)(H + h) * mem.n;
        if (mem.n % 8 == 0) {
            for (int i = tid * 8; i < mem.n; i += THREADS * 8) {
                zi += rs_dot8(x + i, wi + i);
                zf += rs_dot8(x + i, wf + i);
            }
        } else {
            for (int i = tid; i < mem.n; i += THREADS) {
                zi = fmaf(to_f32(x[i]), to_f32(wi[i]), zi);
                zf = fmaf(to_f32(x[i]), to_f32(wf[i]), zf);
            }
        }
        for (int p = tid; p < mem.factor.parts; p += THREADS) ss += mem.factor.ssq[(size_t)p * a.rows + row];
        if (!fresh) m0 = *m_slot;
    } else {
        keep = ret.decay[h];
        const int pos = ret.positions[row], half = ret.dims / 2;
        turned = owns && ret.cos_table && pos >= 0 && pos < ret.table_positions && own < ret.dims;
        if (turned) {
            second = ret.pairing ? (own & 1) : own >= half;
            const int pair = ret.pairing ? own / 2 : second ? own - half : own;
            other_raw = own_src[ret.pairing ? own ^ 1 : second ? own - half : own + half];
            turn_cos = ret.cos_table[(size_t)pos * half + pair];
            turn_sin = ret.sin_table[(size_t)pos * half + pair];
        }
    }
    if constexpr (MEMORY) {
        if (jl == 0) load_column(dv, n);
    }
    load(0);
    float x = to_f32(qk_raw);                                          // (zero past dk)
    float take = 1.f;
    if constexpr (WKV) {
        if (tid < mix.rank) z_s[tid] = tanhf(z_raw);
        for (int i = tid + THREADS; i < mix.rank; i += THREADS) z_s[i] = tanhf(mix.z[row * mix.z_row + i * mix.z_col]);
    } else if constexpr (MEMORY) {
        zi = wave_sum(zi), zf = wave_sum(zf), ss = wave_sum(ss);
        if (tid % TLI_WAVE == 0) red[tid / TLI_WAVE] = zi, red[WAVES + tid / TLI_WAVE] = zf, red[2 * WAVES + tid / TLI_WAVE] = ss;
        __syncthreads();                                               // (m0 is read by all as well)
        zi = zf = ss = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) zi += red[w], zf += red[WAVES + w], ss += red[2 * WAVES + w];
        if (mem.factor.parts > 0) {
            const float f = mem.factor.of_sum(ss);
            zi *= f, zf *= f;
        }
        const float gi = gate_capped(zi + mem.bias[h], mem.cap), gf = gate_log_sigmoid(gate_capped(zf + mem.bias[H + h], mem.cap));
        const float m = fmaxf(gf + m0, gi);
        keep = expf(gf + m0 - m);
        floor_ = expf(-m);
        take = expf(gi - m);
        if (tid == 0) *m_slot = m;
        if (!is_k) x *= mem.q_scale;
    } else {
        if (turned)
            x = second ? rotate_second_half(x, to_f32(other_raw), turn_cos, turn_sin) : rotate_first_half(x, to_f32(other_raw), turn_cos, turn_sin);
        if (is_k) x *= ret.k_scale;
    }
    if (tid < 2 * DKP) q_s[tid] = x;                                   // (k_s lies behind q_s)
    if (tid < dv) v_s[tid] = to_f32(v_raw) * take;
    for (int j = tid + THREADS; j < dv; j += THREADS) v_s[j] = to_f32(v_src[j]) * take;
    if (MEMORY && tid == 0) v_s[dv] = take;
    if constexpr (WKV) {
        __syncthreads();
        float acc = 0.f;
        if (pieces) {
            auto piece = [&](const uint4& raw, int i) {
                const uint32_t b[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc = fmaf(z_s[i + 2 * e], __uint_as_float(b[e] << 16), acc);
                    acc = fmaf(z_s[i + 2 * e + 1], __uint_as_float(b[e] & 0xFFFF0000u), acc);
                }
            };
#pragma unroll
            for (int e = 0; e < HELD; ++e)
                if ((part + e * P) * 8 < mix.rank) piece(w2_raw[e], (part + e * P) * 8);
            for (int i = (part + HELD * P) * 8; i < mix.rank; i += 8 * P) piece(*reinterpret_cast<const uint4*>(w2 + i), i);
        } else {
            for (int i = part; i < mix.rank; i += P) acc = fmaf(z_s[i], to_f32(w2[i]), acc);
        }
#pragma unroll
        for (int off = 1; off < P; off *= 2) acc += __shfl_xor(acc, off, TLI_WAVE);
        if (part == 0) d_s[channel] = channel < dk ? expf(-expf(acc + w0_raw)) : 0.f;
    }
    __syncthreads();
    float q[R], k[R];
#pragma unroll
    for (int r = 0; r < R; ++r) q[r] = q_s[at(r)], k[r] = k_s[at(r)];
    float d[WKV ? R : 1], bonus = 0.f;                   // wkv: the channels' decays; r diag(u) k
    if constexpr (WKV) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            d[r] = d_s[at(r)];
            bonus = fmaf(q[r] * u_raw[r], k[r], bonus);
        }
        bonus = rs_sum16(bonus);
    }
    auto walk = [&](int j, auto& c) {                    // (all 16 lanes of a column come here together, or none)
        const float v = v_s[j];
        float acc = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (WKV) {
                acc = fmaf(c[r], q[r], acc);
                c[r] = fmaf(d[r], c[r], k[r] * v);
            } else {
                c[r] = fmaf(keep, c[r], k[r] * v);
                acc = fmaf(c[r], q[r], acc);
            }
        }
        acc = rs_sum16(acc);
        if (sub == 0) o_s[j] = WKV ? fmaf(bonus, v, acc) : acc;
        store_column(j, c);
    };
    if constexpr (MEMORY) {
        if (jl == 0) walk(dv, n);
    }
    for (int j0 = 0; j0 < dv; j0 += GROUPS * NC) {
        if (j0 > 0) load(j0);
#pragma unroll
        for (int g = 0; g < GROUPS; ++g)
            if (j0 + g * NC + jl < dv) walk(j0 + g * NC + jl, S[g]);
    }
    __syncthreads();
    const float by = MEMORY ? 1.f / (fmaxf(fabsf(o_s[dv]), floor_) + 1e-6f) : 1.f;
    float sum = 0.f;
    for (int j = tid; j < dv; j += THREADS) {
        const float o = o_s[j] * by;
        sum = fmaf(o, o, sum);
    }
    const float factor = a.scale * by / sqrtf(block_sum(sum, red) / (float)dv + a.eps);
    TO* dst = (TO*)a.out + (size_t)row * a.out_ld + (size_t)h * dv;
    auto put = [&](int j, float z, float by_weight) {
        const float open = (MEMORY ? by_weight : WKV ? z * by_weight : z) / (1.f + expf(-z));
        from_f32(dst + j, o_s[j] * factor * open);
    };
    if (tid < dv) put(tid, to_f32(g_raw), weight_raw);
    for (int j = tid + THREADS; j < dv; j += THREADS) put(j, to_f32(g_src[j]), MEMORY || WKV ? weight[j] : 1.f);
}

// Threads of a workgroup: with 512 a head's step is the shorter chain, with 256 more heads' chains fit a compute unit side by side.
// 512 up to two workgroups of 512 a compute unit where a head has enough columns for them, one where not, none for heads of 16.
// us with 512 and 256 threads, retention, mLSTM and wkv: 16 heads of 128 x 128, 8 rows 5.8 and 7.5, 8.0 and 9.2, 7.6 and 9.2, 32 rows 10.6
// and 11.9, 13.1 and 14.0, 13.2 and 14.1, 64 rows 22.7 and 22.4, 25.9 and 22.8, 25.9 and 24.5; of 64 x 64, 32 rows 5.5 and 6.0, 7.9 and
// 8.0, 7.3 and 7.4, 64 rows 8.0 and 8.3, 11.8 and 10.7, 12.0 and 10.3; of 32 x 32, 16 rows 3.8 and 4.0, 5.8 and 5.8, 4.7 and 4.9, 32 rows
// 4.4 and 4.2, 6.9 and 6.2, 5.4 and 5.1; of 16 x 16, 8 rows level, 128 rows 7.7 and 5.6, 14.4 and 10.2, 10.1 and 7.6.  (256 threads that asked for the
// state first: level or 1 to 15% longer than the better of the two, but heads of 16 x 16 in 2,048 workgroups 9.2 and 6.6 for mLSTM and wkv.)
static bool step_wide(const StepRows& a) {
    return a.dk > 16 && (long long)a.H * a.rows <= ((long long)a.dk * a.dv >= 2048 ? 512 : 256);
}

template <int KIND, typename T, typename TO = T>
static int run_step(const StepRows& a, const StepRetention& ret, const StepMemory& mem, const StepTimeMix& mix, hipStream_t s) {
    int R = 1;
    while (16 * R < a.dk) R *= 2;
    const size_t lds = (size_t)(2 * 16 * R + 2 * (a.dv + 1) + (KIND == STEP_WKV ? 16 * R + mix.rank : 0)) * sizeof(float);
    if (lds > 65536) return tli_fail("recurrent_step: values of %d do not fit LDS", a.dv);
    const dim3 grid(a.H, a.rows);
    const bool wide = R > 8 || step_wide(a);
#define RS_RUN(R, THREADS) recurrent_step_kernel<KIND, R, THREADS, T, TO><<<grid, THREADS, lds, s>>>(a, ret, mem, mix)
#define RS_CASE(R) case R: if (wide) RS_RUN(R, 512); else RS_RUN(R, 256); break;
    switch (R) {
        RS_CASE(1) RS_CASE(2) RS_CASE(4) RS_CASE(8)
        case 16: RS_RUN(16, 512); break;
        default: return tli_fail("recurrent_step: keys of %d", a.dk);
    }
#undef RS_CASE
#undef RS_RUN
    return tli_check_launch("recurrent_step");
}

static const char* step_fault(const StepRows& a, int rows_need) {
    if (a.H <= 0 || a.H > 65535 || a.rows > 65535 || a.dk <= 0 || a.dk > TLI_RECURRENCE_MAX_DK || a.dv <= 0) return "bad sizes";
    if (a.ld < rows_need) return "the rows do not hold q, k, v and the gate";
    if (a.out_ld < a.H * a.dv) return "the output's rows overlap";
    if ((uintptr_t)a.state & 15) return "the state must be 16-byte aligned";
    return nullptr;
}

// proj: rows of ld elements, q (H dk) | k (H dk) | v (H dv) | gate (H dv) first; the rest as in retention.hip
extern "C" int tli_retention_step(const void* proj, int ld, const float* decay, float* state, void* out, int out_ld,
                                  const int* positions, const int* seq_start, const int* slots, const float* cos_table,
                                  const float* sin_table, int dims, int pairing, int table_positions, float k_scale, float eps,
                                  float scale, int rows, int H, int dk, int dv, int dtype, void* stream) {
    if (rows <= 0) return 0;
    const StepRows a{proj, ld, out, out_ld, state, seq_start, slots, rows, H, dk, dv, eps, scale};
    if (const char* fault = step_fault(a, 2 * H * (dk + dv))) return tli_fail("retention_step: %s", fault);
    if (cos_table && (dims <= 0 || dims % 2 || dims > dk)) return tli_fail("retention_step: %d turned elements of heads of %d", dims, dk);
    const StepRetention ret{positions, decay, cos_table, sin_table, dims, pairing, table_positions, k_scale};
    if (dtype == TLI_F32) return run_step<STEP_RETENTION, float>(a, ret, StepMemory{}, StepTimeMix{}, (hipStream_t)stream);
    if (dtype == TLI_BF16) return run_step<STEP_RETENTION, bf16_t>(a, ret, StepMemory{}, StepTimeMix{}, (hipStream_t)stream);
    return tli_fail("retention_step: unknown dtype %d", dtype);
}

// x: [rows, n] the layer's input (times the rows' factor where ssq is given: row_gates.h); w: [2 H, n]; the rest as in
// mlstm.hip
extern "C" int tli_mlstm_step(const void* proj, int ld, const void* x, const void* w, int n, const float* ssq, int parts, float x_eps,
                              const float* bias, float cap, float q_scale, const float* weight, float* m_state, float* state,
                              void* out, int out_ld, const int* seq_start, const int* slots, float eps, float scale, int rows,
                              int H, int dk, int dv, int dtype, void* stream) {
    if (rows <= 0) return 0;
    const StepRows a{proj, ld, out, out_ld, state, seq_start, slots, rows, H, dk, dv, eps, scale};
    if (const char* fault = step_fault(a, 2 * H * (dk + dv))) return tli_fail("mlstm_step: %s", fault);
    if (n <= 0 || !(cap > 0.f) || (ssq && parts <= 0)) return tli_fail("mlstm_step: bad gates");
    if (((uintptr_t)x | (uintptr_t)w) & 15) return tli_fail("mlstm_step: operands must be 16-byte aligned");
    const StepMemory mem{x, w, n, RowFactor{ssq, ssq ? parts : 0, rows, 1.0f / (float)n, x_eps}, bias, weight, m_state, cap, q_scale};
    if (dtype == TLI_F32) return run_step<STEP_MEMORY, float>(a, StepRetention{}, mem, StepTimeMix{}, (hipStream_t)stream);
    if (dtype == TLI_BF16) return run_step<STEP_MEMORY, bf16_t>(a, StepRetention{}, mem, StepTimeMix{}, (hipStream_t)stream);
    return tli_fail("mlstm_step: unknown dtype %d", dtype);
}

// proj: rows of ld elements of proj_dtype, r (H dk) | k (H dk) | v (H dv) | gate (H dv) first; z, w2, w0, rank: as for tli_wkv_decays
// (wkv.hip); u [H, dk]; weight [H dv]; state [slots][H][dv][dk]; out and w2 in `dtype` (proj_dtype: the same, or float32)
extern "C" int tli_wkv_step(const void* proj, int ld, int proj_dtype, const float* z, long long z_row, long long z_col, const void* w2,
                            const float* w0, int rank, const float* u, const float* weight, float* state, void* out, int out_ld,
                            const int* seq_start, const int* slots, float eps, int rows, int H, int dk, int dv, int dtype, void* stream) {
    if (rows <= 0) return 0;
    const StepRows a{proj, ld, out, out_ld, state, seq_start, slots, rows, H, dk, dv, eps, 1.0f};
    if (const char* fault = step_fault(a, 2 * H * (dk + dv))) return tli_fail("wkv_step: %s", fault);
    if (rank <= 0 || rank > 8192 || ((uintptr_t)w2 & 15)) return tli_fail("wkv_step: bad decays");
    const StepTimeMix mix{z, z_row, z_col, w2, w0, rank, u, weight};
    hipStream_t s = (hipStream_t)stream;
    if (dtype == TLI_F32 && proj_dtype == TLI_F32) return run_step<STEP_WKV, float>(a, StepRetention{}, StepMemory{}, mix, s);
    if (dtype == TLI_BF16 && proj_dtype == TLI_F32) return run_step<STEP_WKV, float, bf16_t>(a, StepRetention{}, StepMemory{}, mix, s);
    if (dtype == TLI_BF16 && proj_dtype == TLI_BF16) return run_step<STEP_WKV, bf16_t>(a, StepRetention{}, StepMemory{}, mix, s);
    return tli_fail("wkv_step: unknown dtypes %d, %d", proj_dtype, dtype);
}
