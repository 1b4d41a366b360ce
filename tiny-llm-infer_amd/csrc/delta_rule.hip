// The gated delta rule: a recurrent mixer with a matrix of state a head.
//
// Per row t of a sequence (G key heads of size dk, H value heads of size dv, value head h reads key
// head h / (H / G)), from the raw projections q, k, v [T, channels]:
//
//   prepare:     c  = silu(causal convolution over time, per channel, `taps` taps, zeros before position 0)
//                q' = unit(c_q) / sqrt(dk),  k' = unit(c_k),  unit(x) = x / sqrt(sum(x^2) + 1e-6),  v' = c_v
//                beta = sigmoid(b),  decay = exp(-exp(A_log) * softplus(a + dt_bias))
//   recurrence:  S <- decay S;  u = beta (v' - S^T k');  S <- S + k' u^T;  o = S^T q'
//   gated norm:  y = o / sqrt(mean(o^2) + eps) * w * silu(gate)         per head, over dv
//
// S is float32 [dk, dv] a head and lives in a slot of per-request state (in the order the recurrence
// kernel's lanes hold it, see there), as do the last taps - 1 raw rows that the convolution reads.  A sequence that starts at position 0 has no history: its slot is
// not read.  Everything after the projections is float32.
//
// The recurrence walks a sequence's rows one after the other.  Columns of S are independent, so a
// column belongs to 16 neighbouring lanes, each holding every 16th of its dk elements in registers; the
// two dot products of a row (k'.S and q'.S, both with the old S, since
// o = decay (q'.S_old) + (q'.k') u) are reduced over those lanes together.
#include "common.h"

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }

// ---------------------------------------------------------------------------------------------
// prepare: a workgroup takes one row and one piece of it: a key head (its q and k vectors: convolution,
// silu, unit vectors, their dot product; piece 0 also the row's beta and decay), or 256 channels of v
// ---------------------------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) delta_prepare_kernel(
    const T* __restrict__ proj, int ld, const float* __restrict__ conv_w, const T* __restrict__ kept,
    const float* __restrict__ ba, long long ba_row, long long ba_col, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, const int* __restrict__ positions, const int* __restrict__ seq_of_row,
    const int* __restrict__ row_start, const int* __restrict__ slots, float* __restrict__ qn, float* __restrict__ kn,
    float* __restrict__ vc, float* __restrict__ beta, float* __restrict__ decay, float* __restrict__ qk, int H, int G,
    int dk, int dv, int taps) {
    __shared__ float scratch[16];
    const int r = blockIdx.x, piece = blockIdx.y;
    const int seq = seq_of_row[r], pos = positions[r];
    const int in_step = r - row_start[seq];        // rows of this sequence that stand before r in the step
    const int qd = G * dk, C = 2 * qd + H * dv;
    const T* mine = kept ? kept + (size_t)slots[seq] * (taps - 1) * C : nullptr;
    auto conv_silu = [&](int c) {
        float acc = 0.f;
        for (int j = 0; j < taps; ++j) {
            const int back = taps - 1 - j;          // the tap's row lies this many positions before r
            if (back > pos) continue;               // before the sequence's first position: zero
            float x;
            if (back <= in_step) x = to_f32(proj[(size_t)(r - back) * ld + c]);
            else x = to_f32(mine[(size_t)(taps - 1 + in_step - back) * C + c]);
            acc = fmaf(conv_w[(size_t)j * C + c], x, acc);
        }
        return silu_f(acc);
    };
    if (piece >= G) {
        const int c = (piece - G) * 256 + threadIdx.x;
        if (c < H * dv) vc[(size_t)r * H * dv + c] = conv_silu(2 * qd + c);
        return;
    }
    const int i = threadIdx.x;                      // dk <= 256: an element of q and of k a thread
    const bool has = i < dk;
    const float q = has ? conv_silu(piece * dk + i) : 0.f;
    const float k = has ? conv_silu(qd + piece * dk + i) : 0.f;
    const float sq = block_sum(q * q, scratch), sk = block_sum(k * k, scratch);
    const float qu = q * (1.0f / sqrtf(sq + 1e-6f)) * (1.0f / sqrtf((float)dk));
    const float ku = k * (1.0f / sqrtf(sk + 1e-6f));
    const float dot = block_sum(qu * ku, scratch);
    if (has) {
        qn[(size_t)r * qd + (size_t)piece * dk + i] = qu;
        kn[(size_t)r * qd + (size_t)piece * dk + i] = ku;
    }
    if (i == 0) qk[(size_t)r * G + piece] = dot;
    if (piece == 0 && i < H) {
        const float b = ba[(size_t)r * ba_row + (size_t)i * ba_col];
        const float a = ba[(size_t)r * ba_row + (size_t)(H + i) * ba_col] + dt_bias[i];
        beta[(size_t)r * H + i] = 1.0f / (1.0f + expf(-b));
        const float sp = fmaxf(a, 0.f) + log1pf(expf(-fabsf(a)));
        decay[(size_t)r * H + i] = expf(-expf(a_log[i]) * sp);
    }
}

// The last taps - 1 raw rows of every sequence become its kept rows (oldest first).  Row j of the
// new kept rows is row n - (taps - 1) + j of the step's n rows, or, where that is negative, kept row
// n + j of before (zero for a sequence with no history): always a row further on than the one
// written, so the rows are moved in ascending order in place.
template <typename T>
__global__ void delta_conv_keep_kernel(const T* __restrict__ proj, int ld, T* __restrict__ kept,
                                       const int* __restrict__ row_start, const int* __restrict__ seq_start,
                                       const int* __restrict__ slots, int C, int taps) {
    const int seq = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const int r0 = row_start[seq], n = row_start[seq + 1] - r0;
    const bool fresh = seq_start[seq] == 0;
    T* mine = kept + (size_t)slots[seq] * (taps - 1) * C;
    for (int j = 0; j < taps - 1; ++j) {
        const int row = n - (taps - 1) + j;
        T x;
        if (row >= 0) x = proj[(size_t)(r0 + row) * ld + c];
        else if (fresh) from_f32(&x, 0.f);
        else x = mine[(size_t)(n + j) * C + c];
        mine[(size_t)j * C + c] = x;
    }
}

// ---------------------------------------------------------------------------------------------
// recurrence
// ---------------------------------------------------------------------------------------------
#define DELTA_LANES 16         // lanes that share a column of S: one row of 16 lanes, summed over with DPP moves
#define DELTA_COLS 16          // columns a workgroup of 256 threads walks

// Sum over the 16 lanes of a row, every lane gets it: neighbours, pairs (quad permutations), then the mirror
// image inside each half row and inside the row (by then the lanes of a quad, of a half row, hold the same).
__device__ __forceinline__ float row16_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));   // row_half_mirror
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));   // row_mirror
    return v;
}

template <int RPT>             // elements of a column a lane holds: dk <= 16 * RPT
__global__ __launch_bounds__(256) void delta_recurrence_kernel(
    const float* __restrict__ qn, const float* __restrict__ kn, const float* __restrict__ vc,
    const float* __restrict__ beta, const float* __restrict__ decay, const float* __restrict__ qk,
    float* __restrict__ state, float* __restrict__ out, const int* __restrict__ row_start,
    const int* __restrict__ seq_start, const int* __restrict__ slots, int H, int G, int dk, int dv) {
    // A sequence's rows pass through LDS in chunks of CT: the whole workgroup fetches a chunk with loads that
    // do not wait for each other (into registers, while the chunk before is worked on), so the walk along the
    // rows waits for LDS only.  In LDS an element i = part + 16 r of k or q lies at part * RPT + r: a lane's
    // share of a row is one run.
    constexpr int CT = RPT == 16 ? 16 : 32;      // rows a chunk (k and q of a chunk: 2 * CT * 16 RPT floats)
    constexpr int DKP = DELTA_LANES * RPT;
    constexpr int NK = CT * DKP / 256;           // elements of k (and of q) a thread fetches a chunk
    constexpr int NV = CT * DELTA_COLS / 256;    // of v
    __shared__ float ks[CT * DKP], qs[CT * DKP], vs[CT * DELTA_COLS], sc[3 * CT];
    const int seq = blockIdx.z, head = blockIdx.y;
    const int part = threadIdx.x % DELTA_LANES;
    const int local = threadIdx.x / DELTA_LANES;
    const int col_raw = blockIdx.x * DELTA_COLS + local;
    const bool live = col_raw < dv;
    const int col = live ? col_raw : dv - 1;
    const int kvh = head / (H / G);
    const int r0 = row_start[seq], r1 = row_start[seq + 1];
    const bool fresh = seq_start[seq] == 0;
    // The state of a slot: [head][block of 16 columns][r][column][part], element i = part + 16 r of a column: a
    // wave's 64 lanes read and write 64 floats in a row.  Elements past dk and columns past dv exist there too
    // (they stay 0: their k is 0, and the v of a column past dv is read as 0).
    float* mine = state + ((((size_t)slots[seq] * H + head) * gridDim.x + blockIdx.x) * RPT * DELTA_COLS + local) * DELTA_LANES + part;
    float S[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) S[r] = fresh ? 0.f : mine[(size_t)r * DELTA_COLS * DELTA_LANES];
    const size_t qd = (size_t)G * dk, vd = (size_t)H * dv;
    float pk[NK], pq[NK], pv[NV], ps = 0.f;
    auto fetch = [&](int c0) {                   // the chunk that starts at row c0, into registers
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            const int e = threadIdx.x + n * 256, t = e / DKP, i = e % DKP;
            const bool ok = c0 + t < r1 && i < dk;
            pk[n] = ok ? kn[(size_t)(c0 + t) * qd + (size_t)kvh * dk + i] : 0.f;
            pq[n] = ok ? qn[(size_t)(c0 + t) * qd + (size_t)kvh * dk + i] : 0.f;
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) {
            const int e = threadIdx.x + n * 256, t = e / DELTA_COLS, j = blockIdx.x * DELTA_COLS + e % DELTA_COLS;
            pv[n] = (c0 + t < r1 && j < dv) ? vc[(size_t)(c0 + t) * vd + (size_t)head * dv + j] : 0.f;
        }
        if (threadIdx.x < 3 * CT) {
            const int which = threadIdx.x / CT, t = threadIdx.x % CT;
            if (c0 + t < r1)
                ps = which == 0 ? beta[(size_t)(c0 + t) * H + head]
                                : which == 1 ? decay[(size_t)(c0 + t) * H + head] : qk[(size_t)(c0 + t) * G + kvh];
        }
    };
    if (r0 < r1) fetch(r0);
    for (int c0 = r0; c0 < r1; c0 += CT) {
        __syncthreads();                         // the chunk before has been walked
#pragma unroll
        for (int n = 0; n < NK; ++n) {
            const int e = threadIdx.x + n * 256, t = e / DKP, i = e % DKP;
            const int at = t * DKP + (i % DELTA_LANES) * RPT + i / DELTA_LANES;
            ks[at] = pk[n];
            qs[at] = pq[n];
        }
#pragma unroll
        for (int n = 0; n < NV; ++n) vs[threadIdx.x + n * 256] = pv[n];
        if (threadIdx.x < 3 * CT) sc[threadIdx.x] = ps;
        __syncthreads();
        if (c0 + CT < r1) fetch(c0 + CT);
        const int rows = min(CT, r1 - c0);
        // the row after the current one is read from LDS while the current one is worked on: two sets of
        // registers take turns, two rows a round of the loop
        auto read_row = [&](int t, float (&kx)[RPT], float (&qx)[RPT], float (&sx)[4]) {
            const float* kp = ks + t * DKP + part * RPT;
            const float* qp = qs + t * DKP + part * RPT;
#pragma unroll
            for (int r = 0; r < RPT; ++r) { kx[r] = kp[r]; qx[r] = qp[r]; }
            sx[0] = vs[t * DELTA_COLS + local];
            sx[1] = sc[t]; sx[2] = sc[CT + t]; sx[3] = sc[2 * CT + t];
        };
        auto walk_row = [&](int t, const float (&k)[RPT], const float (&q)[RPT], const float (&sx)[4]) {
            float d1[2] = {0.f, 0.f}, d2[2] = {0.f, 0.f};          // two sums each: shorter chains of dependent additions
#pragma unroll
            for (int r = 0; r < RPT; ++r) {
                d1[r & 1] = fmaf(k[r], S[r], d1[r & 1]);
                d2[r & 1] = fmaf(q[r], S[r], d2[r & 1]);
            }
            const float s1 = row16_sum(d1[0] + d1[1]), s2 = row16_sum(d2[0] + d2[1]);
            const float g0 = sx[2];
            const float u = sx[1] * (sx[0] - g0 * s1);
#pragma unroll
            for (int r = 0; r < RPT; ++r) S[r] = fmaf(k[r], u, g0 * S[r]);
            if (part == 0 && live) out[(size_t)(c0 + t) * vd + (size_t)head * dv + col] = fmaf(sx[3], u, g0 * s2);
        };
        float ka[RPT], qa[RPT], sa[4], kb[RPT], qb[RPT], sb[4];
        read_row(0, ka, qa, sa);
        int t = 0;
        for (; t + 1 < rows; t += 2) {
            read_row(t + 1, kb, qb, sb);
            walk_row(t, ka, qa, sa);
            read_row(min(t + 2, CT - 1), ka, qa, sa);
            walk_row(t + 1, kb, qb, sb);
        }
        if (t < rows) walk_row(t, ka, qa, sa);
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) mine[(size_t)r * DELTA_COLS * DELTA_LANES] = S[r];
}

// ---------------------------------------------------------------------------------------------
// gated norm of the heads' outputs: one wave a (row, head)
// ---------------------------------------------------------------------------------------------
template <typename T>
__global__ void gated_rmsnorm_kernel(const float* __restrict__ o, const T* __restrict__ gate, int gate_ld,
                                     const float* __restrict__ weight, T* __restrict__ out, int H, int dv, float eps,
                                     long long pairs) {
    const long long p = (long long)blockIdx.x * (blockDim.x / TLI_WAVE) + threadIdx.x / TLI_WAVE;
    if (p >= pairs) return;
    const int lane = threadIdx.x % TLI_WAVE;
    const long long row = p / H;
    const int h = (int)(p - row * H);
    const float* x = o + (size_t)p * dv;
    const T* gt = gate + (size_t)row * gate_ld + (size_t)h * dv;
    float ss = 0.f;
    for (int i = lane; i < dv; i += TLI_WAVE) ss += x[i] * x[i];
    ss = wave_sum(ss);
    const float scale = 1.0f / sqrtf(ss / (float)dv + eps);
    T* y = out + (size_t)p * dv;
    for (int i = lane; i < dv; i += TLI_WAVE) from_f32(y + i, x[i] * scale * weight[i] * silu_f(to_f32(gt[i])));
}

// ---------------------------------------------------------------------------------------------
// A decode step: every sequence brings one row, and everything between the layer's products is one launch, a workgroup a
// (head, row): the two gates' sums, the convolutions of the head's q, k and v, the recurrence and the gated norm (and a launch
// that moves the kept rows on: the q and k channels of a key head are read by H / G workgroups, so none of them may write them).
//
// What bounds such a step is not its bytes (64 KiB of state in and out a workgroup at 128 x 128) but the chain of fetches and
// launches, so the row's operands are asked for first (loads complete in the order of issue), then the whole state of the
// head, and the sums over the row are made while it is on its way.  8 rows, 16 heads of 128 x 128, 4 taps, width 2,048, as part of
// a decode step: five launches (the gates' product 6.7 us, prepare 7.4, kept rows 4.9, recurrence 8 to 11, norm 4.6) and these
// two: a step of four layers, two of them this one, 431 -> 400 us.
// ---------------------------------------------------------------------------------------------
#define DELTA_STEP_THREADS 512
#define DELTA_STEP_TAPS 8       // taps of a channel that are asked for together

struct DeltaStep {
    const bf16_t* proj;         // [rows, ld]: q (G dk) | k (G dk) | v (H dv) | gate (H dv)
    int ld;
    const bf16_t* x;            // [rows, n]: the layer's input
    const bf16_t* w_gates;      // [2 H, n]: b, then a
    int n;
    const float* conv_w;        // [taps, channels]
    const bf16_t* kept;         // [slots, taps - 1, channels]
    const float *a_log, *dt_bias, *weight;
    const int *positions, *slots;
    float* state;
    bf16_t* out;                // [rows, H dv]
    int H, G, dk, dv, taps;
    float eps;
};

template <int RPT>
__global__ __launch_bounds__(DELTA_STEP_THREADS) void delta_step_kernel(DeltaStep a) {
    constexpr int WAVES = DELTA_STEP_THREADS / TLI_WAVE;
    constexpr int TOGETHER = DELTA_STEP_THREADS / DELTA_LANES;           // columns walked side by side: two blocks
    constexpr int GROUPS = 4;                                            // of them, in flight together
    constexpr int DKP = DELTA_LANES * RPT;
    extern __shared__ float ds_lds[];
    __shared__ float red[2][WAVES];
    const int head = blockIdx.x, row = blockIdx.y, tid = threadIdx.x, lane = tid % TLI_WAVE, wave = tid / TLI_WAVE;
    const int part = tid % DELTA_LANES, local = tid / DELTA_LANES;
    const int dk = a.dk, dv = a.dv, H = a.H, kvh = head / (H / a.G), qd = a.G * dk, C = 2 * qd + H * dv;
    float* q_s = ds_lds;                                                 // [DKP], then k [DKP], v and o [dv]
    float* k_s = q_s + DKP;
    float* v_s = k_s + DKP;
    float* o_s = v_s + dv;
    const int slot = a.slots[row], pos = a.positions[row];
    const bool fresh = pos == 0;
    // the two gates' sums: every thread a part of both
    const bf16_t* xr = a.x + (size_t)row * a.n;
    const bf16_t* wb = a.w_gates + (size_t)head * a.n;
    const bf16_t* wa = a.w_gates + (size_t)(H + head) * a.n;
    float zb = 0.f, za = 0.f;
    for (int i = tid * 8; i < a.n; i += DELTA_STEP_THREADS * 8) {
        const uint4 xv = *reinterpret_cast<const uint4*>(xr + i), bv = *reinterpret_cast<const uint4*>(wb + i),
                    av = *reinterpret_cast<const uint4*>(wa + i);
        const uint32_t xu[4] = {xv.x, xv.y, xv.z, xv.w}, bu[4] = {bv.x, bv.y, bv.z, bv.w}, au[4] = {av.x, av.y, av.z, av.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float lo = __uint_as_float(xu[e] << 16), hi = __uint_as_float(xu[e] & 0xFFFF0000u);
            zb = fmaf(lo, __uint_as_float(bu[e] << 16), zb);
            zb = fmaf(hi, __uint_as_float(bu[e] & 0xFFFF0000u), zb);
            za = fmaf(lo, __uint_as_float(au[e] << 16), za);
            za = fmaf(hi, __uint_as_float(au[e] & 0xFFFF0000u), za);
        }
    }
    // the convolutions: a channel of q, k or v a thread and round
    const bf16_t* mine = a.kept ? a.kept + (size_t)slot * (a.taps - 1) * C : nullptr;
    for (int e = tid; e < 2 * DKP + dv; e += DELTA_STEP_THREADS) {
        const int i = e < 2 * DKP ? e % DKP : e - 2 * DKP;
        float value = 0.f;
        if (e >= 2 * DKP || i < dk) {
            const int c = e < DKP ? kvh * dk + i : e < 2 * DKP ? qd + kvh * dk + i : 2 * qd + head * dv + i;
            float acc = 0.f;
            for (int j0 = 0; j0 < a.taps; j0 += DELTA_STEP_TAPS) {
                float x[DELTA_STEP_TAPS], w[DELTA_STEP_TAPS];
#pragma unroll
                for (int j = 0; j < DELTA_STEP_TAPS; ++j) {
                    const int tap = j0 + j, back = a.taps - 1 - tap;     // the tap's row lies this many positions before
                    x[j] = w[j] = 0.f;
                    if (tap < a.taps && back <= pos) {
                        w[j] = a.conv_w[(size_t)tap * C + c];
                        x[j] = bf16_to_f32(back == 0 ? a.proj[(size_t)row * a.ld + c] : mine[(size_t)tap * C + c]);
                    }
                }
#pragma unroll
                for (int j = 0; j < DELTA_STEP_TAPS; ++j)
                    if (j0 + j < a.taps && a.taps - 1 - j0 - j <= pos) acc = fmaf(w[j], x[j], acc);
            }
            value = silu_f(acc);
        }
        q_s[e] = value;                                                  // (k and v lie behind q)
    }
    const int blocks = (dv + DELTA_COLS - 1) / DELTA_COLS;
    float* state = a.state + ((size_t)slot * H + head) * blocks * RPT * DELTA_COLS * DELTA_LANES + (local % DELTA_COLS) * DELTA_LANES + part;
    float S[GROUPS][RPT];
    auto at = [&](int col) { return state + (size_t)(col / DELTA_COLS) * RPT * DELTA_COLS * DELTA_LANES; };
    auto load = [&](int c0) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            const int col = c0 + g * TOGETHER + local;
            const bool there = !fresh && col < blocks * DELTA_COLS;
#pragma unroll
            for (int r = 0; r < RPT; ++r) S[g][r] = there ? at(col)[r * DELTA_COLS * DELTA_LANES] : 0.f;
        }
    };
    load(0);
    zb = wave_sum(zb), za = wave_sum(za);
    if (lane == 0) red[0][wave] = zb, red[1][wave] = za;
    __syncthreads();
    zb = za = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) zb += red[0][w], za += red[1][w];
    za += a.dt_bias[head];
    const float beta = 1.0f / (1.0f + expf(-zb));
    const float decay = expf(-expf(a.a_log[head]) * (fmaxf(za, 0.f) + log1pf(expf(-fabsf(za)))));
    // unit vectors and their product, every wave for itself (64 elements at a time, in their order, as delta_prepare_kernel adds them)
    float sq = 0.f, sk = 0.f, dot = 0.f;
#pragma unroll
    for (int i = 0; i < DKP; i += TLI_WAVE) {
        const float qe = i + lane < DKP ? q_s[i + lane] : 0.f, ke = i + lane < DKP ? k_s[i + lane] : 0.f;
        sq += wave_sum(qe * qe);
        sk += wave_sum(ke * ke);
    }
    const float q_unit = 1.0f / sqrtf(sq + 1e-6f), q_scale = 1.0f / sqrtf((float)dk), k_unit = 1.0f / sqrtf(sk + 1e-6f);
#pragma unroll
    for (int i = 0; i < DKP; i += TLI_WAVE) {
        const float qe = i + lane < DKP ? q_s[i + lane] * q_unit * q_scale : 0.f, ke = i + lane < DKP ? k_s[i + lane] * k_unit : 0.f;
        dot += wave_sum(qe * ke);
    }
    float q[RPT], k[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) q[r] = q_s[part + DELTA_LANES * r] * q_unit * q_scale, k[r] = k_s[part + DELTA_LANES * r] * k_unit;
    for (int c0 = 0; c0 < blocks * DELTA_COLS; c0 += GROUPS * TOGETHER) {
        if (c0 > 0) load(c0);
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) {
            const int col = c0 + g * TOGETHER + local;
            if (col >= blocks * DELTA_COLS) continue;                    // (the 16 lanes of a column alike)
            const float v = col < dv ? v_s[col] : 0.f;
            float d1[2] = {0.f, 0.f}, d2[2] = {0.f, 0.f};
#pragma unroll
            for (int r = 0; r < RPT; ++r) {
                d1[r & 1] = fmaf(k[r], S[g][r], d1[r & 1]);
                d2[r & 1] = fmaf(q[r], S[g][r], d2[r & 1]);
            }
            const float s1 = row16_sum(d1[0] + d1[1]), s2 = row16_sum(d2[0] + d2[1]);
            const float u = beta * (v - decay * s1);
#pragma unroll
            for (int r = 0; r < RPT; ++r) at(col)[r * DELTA_COLS * DELTA_LANES] = fmaf(k[r], u, decay * S[g][r]);
            if (part == 0 && col < dv) o_s[col] = fmaf(dot, u, decay * s2);
        }
    }
    __syncthreads();
    if (wave > 0) return;
    // the norm over the head's outputs (one wave, in the order of gated_rmsnorm_kernel)
    const bf16_t* gate = a.proj + (size_t)row * a.ld + C + (size_t)head * dv;
    float ss = 0.f;
    for (int i = lane; i < dv; i += TLI_WAVE) ss += o_s[i] * o_s[i];
    ss = wave_sum(ss);
    const float scale = 1.0f / sqrtf(ss / (float)dv + a.eps);
    bf16_t* y = a.out + ((size_t)row * H + head) * dv;
    for (int i = lane; i < dv; i += TLI_WAVE) from_f32(y + i, o_s[i] * scale * a.weight[i] * silu_f(to_f32(gate[i])));
}

// ---------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------
#define DELTA_MAX_DK 256

// proj: [T, ld] raw projections, channels q (G dk), k (G dk), v (H dv) first; conv_w: float32
// [taps, channels], oldest tap first; kept: [slots, taps - 1, channels] or null for one tap;
// ba: float32, b then a: number n of row t at t * ba_row + n * ba_col.  Outputs are float32: qn, kn [T, G dk], vc [T, H dv], beta, decay
// [T, H], qk [T, G].  `keep`: also move the kept rows on (after every row was read).
extern "C" int tli_delta_prepare(const void* proj, int ld, const float* conv_w, void* kept, const float* ba,
                                 long long ba_row, long long ba_col, const float* a_log, const float* dt_bias, const int* positions,
                                 const int* seq_of_row, const int* row_start, const int* seq_start, const int* slots,
                                 float* qn, float* kn, float* vc, float* beta, float* decay, float* qk, int T,
                                 int seqs, int H, int G, int dk, int dv, int taps, int dtype, void* stream) {
    if (T <= 0) return 0;
    if (H <= 0 || G <= 0 || H % G || dk <= 0 || dv <= 0 || taps <= 0)
        return tli_fail("delta_prepare: bad sizes (heads %d, key heads %d, dk %d, dv %d, taps %d)", H, G, dk, dv, taps);
    const int C = 2 * G * dk + H * dv;
    if (ld < C) return tli_fail("delta_prepare: rows of %d hold fewer than the %d channels", ld, C);
    if (taps > 1 && !kept) return tli_fail("delta_prepare: %d taps need the sequences' kept rows", taps);
    if (H > 256) return tli_fail("delta_prepare: at most 256 heads, got %d", H);
    if (dk > DELTA_MAX_DK) return tli_fail("delta_prepare: key heads of at most %d, got %d", DELTA_MAX_DK, dk);
    if (G + (H * dv + 255) / 256 > 65535) return tli_fail("delta_prepare: too many channels for one launch");
    const dim3 grid(T, G + (H * dv + 255) / 256);
    hipStream_t s = (hipStream_t)stream;
    if (dtype == TLI_F32) {
        hipLaunchKernelGGL((delta_prepare_kernel<float>), grid, dim3(256), 0, s, (const float*)proj, ld, conv_w,
                           (const float*)kept, ba, ba_row, ba_col, a_log, dt_bias, positions, seq_of_row, row_start, slots, qn, kn, vc,
                           beta, decay, qk, H, G, dk, dv, taps);
        if (taps > 1)
            hipLaunchKernelGGL((delta_conv_keep_kernel<float>), dim3((C + 255) / 256, seqs), dim3(256), 0, s,
                               (const float*)proj, ld, (float*)kept, row_start, seq_start, slots, C, taps);
    } else if (dtype == TLI_BF16) {
        hipLaunchKernelGGL((delta_prepare_kernel<bf16_t>), grid, dim3(256), 0, s, (const bf16_t*)proj, ld, conv_w,
                           (const bf16_t*)kept, ba, ba_row, ba_col, a_log, dt_bias, positions, seq_of_row, row_start, slots, qn, kn,
                           vc, beta, decay, qk, H, G, dk, dv, taps);
        if (taps > 1)
            hipLaunchKernelGGL((delta_conv_keep_kernel<bf16_t>), dim3((C + 255) / 256, seqs), dim3(256), 0, s,
                               (const bf16_t*)proj, ld, (bf16_t*)kept, row_start, seq_start, slots, C, taps);
    } else {
        return tli_fail("delta_prepare: unknown dtype %d", dtype);
    }
    return tli_check_launch("delta_prepare");
}

// Floats of state a head: columns in blocks of 16, key elements padded to 16 * RPT (RPT = 1, 2, 4, 8 or 16).
extern "C" int tli_delta_state_floats(int dk, int dv) {
    if (dk <= 0 || dv <= 0 || dk > DELTA_MAX_DK) return 0;
    const int rpt = dk <= 16 ? 1 : dk <= 32 ? 2 : dk <= 64 ? 4 : dk <= 128 ? 8 : 16;
    return ((dv + DELTA_COLS - 1) / DELTA_COLS) * rpt * DELTA_COLS * DELTA_LANES;
}

extern "C" int tli_delta_recurrence(const float* qn, const float* kn, const float* vc, const float* beta,
                                    const float* decay, const float* qk, float* state, float* out,
                                    const int* row_start, const int* seq_start, const int* slots, int seqs, int H,
                                    int G, int dk, int dv, void* stream) {
    if (seqs <= 0) return 0;
    if (H <= 0 || G <= 0 || H % G || dk <= 0 || dv <= 0 || dk > DELTA_MAX_DK)
        return tli_fail("delta_recurrence: bad sizes (heads %d, key heads %d, dk %d (at most %d), dv %d)", H, G, dk,
                        DELTA_MAX_DK, dv);
    if (H > 65535 || seqs > 65535) return tli_fail("delta_recurrence: too many heads or sequences for one launch");
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((dv + DELTA_COLS - 1) / DELTA_COLS, H, seqs);
#define TLI_DELTA(RPT) hipLaunchKernelGGL((delta_recurrence_kernel<RPT>), grid, dim3(256), 0, s, qn, kn, vc, beta, \
                                          decay, qk, state, out, row_start, seq_start, slots, H, G, dk, dv)
    if (dk <= 16) TLI_DELTA(1);
    else if (dk <= 32) TLI_DELTA(2);
    else if (dk <= 64) TLI_DELTA(4);
    else if (dk <= 128) TLI_DELTA(8);
    else TLI_DELTA(16);
#undef TLI_DELTA
    return tli_check_launch("delta_recurrence");
}

extern "C" int tli_gated_rmsnorm(const float* o, const void* gate, int gate_ld, const float* weight, void* out,
                                 int T, int H, int dv, float eps, int dtype, void* stream) {
    if (T <= 0) return 0;
    if (H <= 0 || dv <= 0 || gate_ld < H * dv) return tli_fail("gated_rmsnorm: bad sizes");
    hipStream_t s = (hipStream_t)stream;
    const long long pairs = (long long)T * H;
    const int blocks = (int)((pairs + 3) / 4);
    if (dtype == TLI_F32)
        hipLaunchKernelGGL((gated_rmsnorm_kernel<float>), dim3(blocks), dim3(256), 0, s, o, (const float*)gate, gate_ld,
                           weight, (float*)out, H, dv, eps, pairs);
    else if (dtype == TLI_BF16)
        hipLaunchKernelGGL((gated_rmsnorm_kernel<bf16_t>), dim3(blocks), dim3(256), 0, s, o, (const bf16_t*)gate,
                           gate_ld, weight, (bf16_t*)out, H, dv, eps, pairs);
    else
        return tli_fail("gated_rmsnorm: unknown dtype %d", dtype);
    return tli_check_launch("gated_rmsnorm");
}

// A decode step (one row a sequence) in bfloat16, from the projections to the gated norm's output [rows, H dv]: proj as for
// tli_delta_prepare with the output gate (H dv) behind the channels; x [rows, n], w_gates [2 H, n]; slots and positions per row;
// the kept rows are moved on.
extern "C" int tli_delta_step_bf16(const void* proj, int ld, const void* x, const void* w_gates, int n, const float* conv_w, void* kept,
                                   const float* a_log, const float* dt_bias, const float* weight, const int* positions,
                                   const int* row_start, const int* seq_start, const int* slots, float* state, void* out, int rows,
                                   int H, int G, int dk, int dv, int taps, float eps, void* stream) {
    if (rows <= 0) return 0;
    if (H <= 0 || G <= 0 || H % G || dk <= 0 || dv <= 0 || taps <= 0 || dk > DELTA_MAX_DK || H > 65535 || rows > 65535)
        return tli_fail("delta_step: bad sizes (heads %d, key heads %d, dk %d (at most %d), dv %d, taps %d, rows %d)", H, G, dk,
                        DELTA_MAX_DK, dv, taps, rows);
    const int C = 2 * G * dk + H * dv;
    if (ld < C + H * dv) return tli_fail("delta_step: rows of %d hold fewer than the %d channels and the gate", ld, C);
    if (taps > 1 && !kept) return tli_fail("delta_step: %d taps need the sequences' kept rows", taps);
    if (n <= 0 || n % 8 || (((uintptr_t)x | (uintptr_t)w_gates) & 15)) return tli_fail("delta_step: the gates' operands must be whole 16-byte pieces");
    const int rpt = dk <= 16 ? 1 : dk <= 32 ? 2 : dk <= 64 ? 4 : dk <= 128 ? 8 : 16;
    const size_t lds = (size_t)(2 * DELTA_LANES * rpt + 2 * dv) * sizeof(float);
    if (lds > 60 * 1024) return tli_fail("delta_step: values of %d do not fit LDS", dv);
    const DeltaStep a{(const bf16_t*)proj, ld, (const bf16_t*)x, (const bf16_t*)w_gates, n, conv_w, taps > 1 ? (const bf16_t*)kept : nullptr,
                      a_log, dt_bias, weight, positions, slots, state, (bf16_t*)out, H, G, dk, dv, taps, eps};
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(H, rows);
#define TLI_DELTA_STEP(RPT) case RPT: delta_step_kernel<RPT><<<grid, DELTA_STEP_THREADS, lds, s>>>(a); break
    switch (rpt) {
        TLI_DELTA_STEP(1);
        TLI_DELTA_STEP(2);
        TLI_DELTA_STEP(4);
        TLI_DELTA_STEP(8);
        default: delta_step_kernel<16><<<grid, DELTA_STEP_THREADS, lds, s>>>(a);
    }
#undef TLI_DELTA_STEP
    if (taps > 1)
        delta_conv_keep_kernel<bf16_t><<<dim3((C + 255) / 256, rows), 256, 0, s>>>((const bf16_t*)proj, ld, (bf16_t*)kept, row_start, seq_start,
                                                                                  slots, C, taps);
    return tli_check_launch("delta_step");
}
