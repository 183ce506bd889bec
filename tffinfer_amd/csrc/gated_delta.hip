// The gated delta rule: a linear recurrence whose state, a matrix S [key channel, value channel]
// per request and head, is decayed, corrected towards the token's value along the token's key,
// and read with the token's query:
//
//   S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
//
// with g_t = exp(-exp(A) softplus(a_t + dt)) and beta_t = sigmoid(b_t) per head, k_t a unit vector,
// q_t a unit vector times dim^(-1/2).  q, k, v come from a projection through a short causal
// convolution over time per channel and silu; the convolution's last taps - 1 inputs are part of
// the request's state, behind the heads' matrices.  Everything here is float32.
//
// A request's state row: [heads][value channel][key channel] (S transposed: the key channels of one
// value channel lie side by side, as the lanes that share the channel read them), then
// [taps - 1][channels] of the convolution's inputs, oldest first; channels are q (kv_heads x dim),
// k (kv_heads x dim), v (heads x vdim), in the projection's column order.
//
// tff_gdelta_prep:        per token: convolution + silu of q, k, v, unit vectors, beta and the decay.
// tff_gdelta_recurrence:  the recurrence over each request's tokens of the step; also leaves the
//                         convolution's last inputs in the state.
// tff_head_norm_silu_gate: out = o / sqrt(mean over the head of o^2 + eps) * w[channel] * silu(gate).
// tff_sigmoid_gate_heads: out = o * sigmoid(gate) * scale, heads of o a stride apart.
#include "head_norm.h"
#include "tffinfer_kernels.h"
#include <limits.h>

#define GD_MAX_TAPS 8
#define GD_FEW 4        // tokens a request up to which a step counts as decoding

__device__ __forceinline__ float gd_silu(float z) { return z / (1.0f + expf(-z)); }

// One wave per (token, unit); units: kv_heads q heads, kv_heads k heads, heads v heads, one for beta and decay.  The convolution's terms and
// the factor of a unit vector, which a whole row of the results shares, are kept in 64 bits until they are rounded once.
__global__ __launch_bounds__(64) void gdelta_prep_kernel(
    const float* __restrict__ proj, size_t ldp, const float* __restrict__ wconv, int taps,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias, const float* __restrict__ state,
    size_t state_row, size_t tail_off, const int32_t* __restrict__ token_req, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ state_slots, float* __restrict__ pre, int H, int G, int D, int E) {
    const int t = blockIdx.x, u = blockIdx.y, lane = threadIdx.x;
    const int C = 2 * G * D + H * E;
    const size_t ldq = (size_t)C + 2 * H;
    const float* row = proj + (size_t)t * ldp;
    float* out = pre + (size_t)t * ldq;
    if (u == 2 * G + H) {
        for (int h = lane; h < H; h += 64) {
            const float b = row[C + h], a = row[C + H + h] + dt_bias[h];
            const float sp = a > 20.f ? a : log1pf(expf(a));
            out[C + h] = 1.0f / (1.0f + expf(-b));
            out[C + H + h] = expf(-expf(a_log[h]) * sp);
        }
        return;
    }
    const int r = token_req[t];
    const int i = t - cu_tokens[r];               // the token's place in its request's portion
    const float* tail = state + (size_t)state_slots[r] * state_row + tail_off;
    int c0, n;
    if (u < 2 * G) { c0 = u * D; n = D; } else { c0 = 2 * G * D + (u - 2 * G) * E; n = E; }
    float ss = 0.f;
    for (int e = lane; e < n; e += 64) {
        const int c = c0 + e;
        double acc = 0.;
        for (int k = 0; k < taps; ++k) {
            const int s = i - (taps - 1) + k;     // the input's place in the portion; before it: the state's
            const float x = s >= 0 ? proj[(size_t)(t - (taps - 1) + k) * ldp + c] : tail[(size_t)(i + k) * C + c];
            acc = fma((double)wconv[(size_t)c * taps + k], (double)x, acc);
        }
        const float y = gd_silu((float)acc);
        out[c] = y;
        ss = fmaf(y, y, ss);
    }
    if (u < 2 * G) {
        ss = wave_sum(ss);
        const double f = 1.0 / sqrt(((double)ss + 1e-6) * (u < G ? (double)D : 1.0));
        __syncthreads();
        for (int e = lane; e < n; e += 64) out[c0 + e] = (float)((double)out[c0 + e] * f);      // (each lane rescales what it wrote)
    }
}

// The same for four taps and heads of whole float4, on rows of 16-byte alignment: LPT lanes share a head, four channels each, and a
// group of them takes a run of RUN tokens, so that an input row is read RUN + 3 times by RUN tokens instead of four times
// each, and the weights once a run.  A wave a token and head with 4-byte loads was bound by its instructions and by the turn of small
// blocks: 2,048 tokens of 8,192 channels (134 MB to move, 22 us at the rate of a large copy) 92 us, now 37.  The convolution's four terms
// and the factor of a unit vector, which a whole row of the results shares, are kept in 64 bits until they are rounded once.
// A run is one token below GD_RUNS_FROM tokens, where waves count for more; the sums are the same: 1, 8 and 48 tokens 6.4, 5.3 and
// 6.9 us before, 3.4, 4.4 and 5.4 now; 256 tokens 8.6 in runs of one, 11.9 in runs of four.
#define GD_RUNS_FROM 512
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gd_floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double gd_doublex4;

template <int LPT, int RUN>
__global__ __launch_bounds__(64) void gdelta_prep_runs_kernel(
    const float* __restrict__ proj, size_t ldp, const float* __restrict__ wconv, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, const float* __restrict__ state, size_t state_row, size_t tail_off,
    const int32_t* __restrict__ token_req, const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ state_slots,
    float* __restrict__ pre, int T, int H, int G, int D, int E) {
    constexpr int GROUPS = 64 / LPT;
    const int u = blockIdx.y, lane = threadIdx.x;
    const int C = 2 * G * D + H * E;
    const size_t ldq = (size_t)C + 2 * H;
    if (u == 2 * G + H) {
        const int first = blockIdx.x * GROUPS * RUN, count = min(GROUPS * RUN, T - first);
        for (int x = lane; x < count * H; x += 64) {
            const int t = first + x / H, h = x % H;
            const float* row = proj + (size_t)t * ldp;
            float* out = pre + (size_t)t * ldq;
            const float b = row[C + h], a = row[C + H + h] + dt_bias[h];
            const float sp = a > 20.f ? a : log1pf(expf(a));
            out[C + h] = 1.0f / (1.0f + expf(-b));
            out[C + H + h] = expf(-expf(a_log[h]) * sp);
        }
        return;
    }
    const int l = lane % LPT, t0 = (blockIdx.x * GROUPS + lane / LPT) * RUN;
    const int n = u < 2 * G ? D : E, c0 = u < 2 * G ? u * D : 2 * G * D + (u - 2 * G) * E;
    const bool live = 4 * l < n;
    const int c = c0 + (live ? 4 * l : 0);
    gd_floatx4 rows[RUN + 3];
#pragma unroll
    for (int q = 0; q < RUN + 3; ++q) {                 // (rows before the step and past it are read as its first and last and not used)
        const int t = min(max(t0 - 3 + q, 0), T - 1);
        rows[q] = *reinterpret_cast<const gd_floatx4*>(proj + (size_t)t * ldp + c);
    }
    gd_floatx4 w[4];                                       // by channel
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = *reinterpret_cast<const gd_floatx4*>(wconv + (size_t)(c + e) * 4);
#pragma unroll
    for (int q = 0; q < RUN; ++q) {
        const int t = min(t0 + q, T - 1);
        const int r = token_req[t], i = t - cu_tokens[r];  // the token's place in its request's portion
        gd_floatx4 x[4] = {rows[q], rows[q + 1], rows[q + 2], rows[q + 3]};
        if (i < 3) {                                       // inputs before the portion are the state's
            const float* tail = state + (size_t)state_slots[r] * state_row + tail_off;
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (i - 3 + k < 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[k][e] = tail[(size_t)(i + k) * C + c + e];
                }
        }
        gd_floatx4 y;
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            double acc = 0.;
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = fma((double)w[e][k], (double)x[k][e], acc);
            y[e] = gd_silu((float)acc);
            ss = fmaf(y[e], y[e], ss);
        }
        if (u < 2 * G) {
            ss = live ? ss : 0.f;
#pragma unroll
            for (int m = 1; m < LPT; m *= 2) ss += __shfl_xor(ss, m, 64);
            const double f = 1.0 / sqrt(((double)ss + 1e-6) * (u < G ? (double)D : 1.0));
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = (float)((double)y[e] * f);
        }
        if (live && t0 + q < T) *reinterpret_cast<gd_floatx4*>(pre + (size_t)t * ldq + c) = y;
    }
}

TFF_API int tff_gdelta_prep(const float* proj, size_t ldp, const float* wconv, int taps, const float* a_log,
                            const float* dt_bias, const float* state, size_t state_row, size_t tail_off,
                            const int32_t* token_req, const int32_t* cu_tokens, const int32_t* state_slots, float* pre,
                            int T, int H, int G, int D, int E, tff_stream_t stream) {
    TFF_REQUIRE(proj && wconv && a_log && dt_bias && state && token_req && cu_tokens && state_slots && pre,
                "gdelta_prep: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && G > 0 && H % G == 0 && D > 0 && E > 0 && taps >= 1 && taps <= GD_MAX_TAPS,
                "gdelta_prep: bad sizes heads=%d kv_heads=%d dim=%d vdim=%d taps=%d (taps up to %d)", H, G, D, E, taps,
                GD_MAX_TAPS);
    const size_t C = 2 * (size_t)G * D + (size_t)H * E;
    TFF_REQUIRE(ldp >= C + 2 * (size_t)H && tail_off + (size_t)(taps - 1) * C <= state_row,
                "gdelta_prep: rows of %zu or state rows of %zu are too short", ldp, state_row);
    TFF_REQUIRE(2 * G + H + 1 <= 65535, "gdelta_prep: too many heads");
    if (T == 0) return 0;
    const int widest = D > E ? D : E;
    if (taps == 4 && D % 4 == 0 && E % 4 == 0 && H % 2 == 0 && widest <= 256 && ldp % 4 == 0 && ((uintptr_t)proj % 16) == 0 &&
        ((uintptr_t)wconv % 16) == 0 && ((uintptr_t)pre % 16) == 0) {
#define GD_RUNS(LPT, RUN)                                                                                                     \
    gdelta_prep_runs_kernel<LPT, RUN><<<dim3((T + 64 / LPT * RUN - 1) / (64 / LPT * RUN), 2 * G + H + 1), 64, 0,               \
                                        (hipStream_t)stream>>>(proj, ldp, wconv, a_log, dt_bias, state, state_row, tail_off,   \
                                                               token_req, cu_tokens, state_slots, pre, T, H, G, D, E)
        if (T < GD_RUNS_FROM) {
            if (widest <= 64) GD_RUNS(16, 1);
            else if (widest <= 128) GD_RUNS(32, 1);
            else GD_RUNS(64, 1);
        } else if (widest <= 64) GD_RUNS(16, 4);
        else if (widest <= 128) GD_RUNS(32, 4);
        else GD_RUNS(64, 4);
#undef GD_RUNS
        return tff_check_launch("gdelta_prep_runs");
    }
    gdelta_prep_kernel<<<dim3(T, 2 * G + H + 1), 64, 0, (hipStream_t)stream>>>(
        proj, ldp, wconv, taps, a_log, dt_bias, state, state_row, tail_off, token_req, cu_tokens, state_slots, pre, H, G, D, E);
    return tff_check_launch("gdelta_prep");
}

// The convolution's last taps - 1 inputs go into the state: by the block of a head's first value channels, the
// head's value channels, and with the first head of a group its q and k.
__device__ __forceinline__ void gd_keep_inputs(const float* __restrict__ proj, size_t ldp, float* __restrict__ tail, int taps,
                                               int t0, int n, int h, int gk, int H, int G, int D, int E) {
    if (taps <= 1) return;
    const int C = 2 * G * D + H * E;
    const int own = (h % (H / G) == 0) ? 2 * D : 0;
    for (int x = threadIdx.x; x < E + own; x += blockDim.x) {
        const int c = x < E ? 2 * G * D + h * E + x : (x - E < D ? gk * D + x - E : (G + gk) * D + x - E - D);
        for (int i = 0; i < taps - 1; ++i) {            // ascending: what is read lies behind what was written
            const int src = n - (taps - 1) + i;
            tail[(size_t)i * C + c] = src >= 0 ? proj[(size_t)(t0 + src) * ldp + c] : tail[(size_t)(i + n) * C + c];
        }
    }
}

// One token of one value channel, on the row of sixteen lanes that shares the channel; lane s holds the key
// channels s, s + 16, ... of S, k and q.  The same additions in the same order wherever it is used, so that a
// sequence gives the same bits however it is cut into portions that are too short for chunks (below), whatever else a step holds.
template <int KPL>
__device__ __forceinline__ float gd_token(float (&S)[KPL], const float (&kk)[KPL], const float (&qq)[KPL], float v, float beta,
                                          float g) {
    float a = 0.f;
#pragma unroll
    for (int m = 0; m < KPL; ++m) a = fmaf(S[m], kk[m], a);
    a = row16_sum(a);
    const float u = beta * (v - g * a);
    float b = 0.f;
#pragma unroll
    for (int m = 0; m < KPL; ++m) {
        S[m] = fmaf(kk[m], u, g * S[m]);
        b = fmaf(S[m], qq[m], b);
    }
    return row16_sum(b);
}

// A portion of one head and sixteen value channels from j0 on, token by token, by a block of 256: no LDS and no barrier.  A row of
// sixteen lanes shares a value channel as above, but lane s takes the key channels s, s + 16, ...: a load or store of the state
// is sixteen neighbouring floats a row, and k and q come straight from the prepared rows.
template <int KPL>
__device__ __forceinline__ void gd_portion(const float* __restrict__ pre, int t0, int n, float* __restrict__ srow, float* __restrict__ o,
                                           int h, int gk, int H, int G, int D, int E, int j0) {
    const int tid = threadIdx.x, s = tid & 15, j = j0 + (tid >> 4), jc = min(j, E - 1);
    const int C = 2 * G * D + H * E;
    const size_t ldq = (size_t)C + 2 * H;
    float* sp = srow + ((size_t)h * E + jc) * D + s;
    const bool row_live = j < E;
    float S[KPL];
#pragma unroll
    for (int m = 0; m < KPL; ++m) S[m] = (row_live && s + 16 * m < D) ? sp[16 * m] : 0.f;
    for (int t = 0; t < n; ++t) {
        const float* p = pre + (size_t)(t0 + t) * ldq;
        const float* pk = p + (size_t)(G + gk) * D + s;
        const float* pq = p + (size_t)gk * D + s;
        float kk[KPL], qq[KPL];
#pragma unroll
        for (int m = 0; m < KPL; ++m) {
            const bool in = s + 16 * m < D;
            kk[m] = in ? pk[16 * m] : 0.f;
            qq[m] = in ? pq[16 * m] : 0.f;
        }
        const float v = p[2 * (size_t)G * D + (size_t)h * E + jc], beta = p[C + h], g = p[C + H + h];
        const float b = gd_token<KPL>(S, kk, qq, v, beta, g);
        if (s == 0 && row_live) o[(size_t)(t0 + t) * H * E + (size_t)h * E + j] = b;
    }
    if (row_live) {
#pragma unroll
        for (int m = 0; m < KPL; ++m)
            if (s + 16 * m < D) sp[16 * m] = S[m];
    }
}

// For steps in which every request brings a few tokens (decoding).
template <int KPL>
__global__ __launch_bounds__(256) void gdelta_recurrence_few_kernel(
    const float* __restrict__ pre, const float* __restrict__ proj, size_t ldp, float* __restrict__ state, size_t state_row,
    size_t tail_off, int taps, const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ state_slots,
    float* __restrict__ o, int H, int G, int D, int E, int below) {
    const int h = blockIdx.y, r = blockIdx.z, gk = h / (H / G);
    const int t0 = cu_tokens[r], n = cu_tokens[r + 1] - t0;
    if (n >= below) return;                                // (a portion for the kernels over chunks)
    float* srow = state + (size_t)state_slots[r] * state_row;
    gd_portion<KPL>(pre, t0, n, srow, o, h, gk, H, G, D, E, blockIdx.x * 16);
    if (blockIdx.x == 0) gd_keep_inputs(proj, ldp, srow + tail_off, taps, t0, n, h, gk, H, G, D, E);
}

// Block: sixteen value channels of one head of one request; a row of sixteen lanes shares a value channel, each
// lane the KPL key channels s, s + 16, ... of it (dim <= 16 KPL; the channels past dim are zero; in LDS a lane's
// channels of k and of q lie side by side).  The tokens of the portion pass in
// chunks of sixteen (eight for the widest heads): a chunk's k, q, its sixteen v, beta and decay are fetched into
// registers while the chunk before is worked through from LDS, so that no token waits for memory; the waves meet
// at the chunks' borders only.  Per token a lane does 4 KPL multiply-adds and two sums over its row:
//   a = S^T k (of the state before the token);   u = beta (v - g a);   S <- g S + k u;   o = S^T q.
// Only S runs from token to token; the read-out hangs off it, so with the loop unrolled by four a token's
// read-out, its store and the LDS reads of the tokens after it fill the waits of the next token's sum.
template <int KPL>
__global__ __launch_bounds__(256) void gdelta_recurrence_kernel(
    const float* __restrict__ pre, const float* __restrict__ proj, size_t ldp, float* __restrict__ state, size_t state_row,
    size_t tail_off, int taps, const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ state_slots,
    float* __restrict__ o, int H, int G, int D, int E, int below) {
    constexpr int DP = 16 * KPL;
    constexpr int GD_CHUNK = KPL >= 16 ? 8 : 16;           // (two chunks of the widest heads fill LDS otherwise)
    constexpr int ROWW = 2 * DP + 20;                      // k, q, sixteen v, beta, decay of a token; rows of 16 bytes
    constexpr int NLD = (GD_CHUNK * ROWW + 255) / 256;
    constexpr int VEC = KPL % 4 == 0 ? 4 : (KPL % 2 == 0 ? 2 : 1);
    __shared__ __attribute__((aligned(16))) float lds[2][GD_CHUNK * ROWW];
    const int h = blockIdx.y, r = blockIdx.z, j0 = blockIdx.x * 16;
    const int tid = threadIdx.x, s = tid & 15, j = j0 + (tid >> 4);
    const int C = 2 * G * D + H * E;
    const size_t ldq = (size_t)C + 2 * H;
    const int gk = h / (H / G);
    const int t0 = cu_tokens[r], n = cu_tokens[r + 1] - t0;
    if (n <= 0 || n >= below) return;                      // (the whole block: a request without tokens changes nothing; chunks)
    float* srow = state + (size_t)state_slots[r] * state_row;
    float S[KPL];
    float* sp = srow + ((size_t)h * E + min(j, E - 1)) * D + s;
#pragma unroll
    for (int m = 0; m < KPL; ++m) S[m] = (j < E && s + 16 * m < D) ? sp[16 * m] : 0.f;

    // (every element has one load at an address chosen without branches, so that the loads of a chunk are all in
    // flight together; what lies past the portion, dim or vdim reads the row's first element and is stored as zero.
    // Where an element comes from and where it goes in LDS does not change from chunk to chunk: found once.)
    float regs[NLD];
    unsigned rel[NLD], live = 0, cols = 0;
    int dst[NLD], tks[NLD];
#pragma unroll
    for (int x = 0; x < NLD; ++x) {
        const int e = x * 256 + tid;
        const int tk = e / ROWW, col = e - tk * ROWW;
        const int ck = col, cq = col - DP, cv = col - 2 * DP, cb = col - 2 * DP - 16;
        const bool isk = col < DP, isq = !isk && col < 2 * DP, isv = cv >= 0 && cv < 16, isb = cb >= 0 && cb < 2;
        const bool ok = tk < GD_CHUNK && ((isk && ck < D) || (isq && cq < D) || (isv && j0 + cv < E) || isb);
        const size_t at = isk ? (size_t)(G + gk) * D + ck
                        : isq ? (size_t)gk * D + cq
                        : isv ? 2 * (size_t)G * D + (size_t)h * E + j0 + cv
                              : (size_t)C + (size_t)cb * H + h;
        rel[x] = ok ? (unsigned)((size_t)tk * ldq + at) : 0u;
        cols |= ok ? 1u << x : 0u;
        tks[x] = tk;
        const int d = col < DP ? col : col - DP;                           // key channel d: lane d % 16, its place d / 16
        dst[x] = e < GD_CHUNK * ROWW ? tk * ROWW + (col < 2 * DP ? col - d + (d & 15) * KPL + (d >> 4) : col) : -1;
    }
    auto fetch = [&](int first) {
        const float* base = pre + (size_t)(t0 + first) * ldq;
        live = 0;
#pragma unroll
        for (int x = 0; x < NLD; ++x) {
            const bool ok = (cols >> x & 1u) && first + tks[x] < n;
            regs[x] = base[ok ? rel[x] : 0u];
            live |= ok ? 1u << x : 0u;
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int x = 0; x < NLD; ++x)
            if (dst[x] >= 0) lds[buf][dst[x]] = (live >> x & 1u) ? regs[x] : 0.f;
    };
    // a lane's KPL channels of a row of LDS, in reads of sixteen bytes where KPL allows
    auto take = [&](const float* p, float* dst) {
        if constexpr (VEC == 4) {
#pragma unroll
            for (int m = 0; m < KPL; m += 4) {
                const float4 x = *reinterpret_cast<const float4*>(p + m);
                dst[m] = x.x; dst[m + 1] = x.y; dst[m + 2] = x.z; dst[m + 3] = x.w;
            }
        } else if constexpr (VEC == 2) {
#pragma unroll
            for (int m = 0; m < KPL; m += 2) {
                const float2 x = *reinterpret_cast<const float2*>(p + m);
                dst[m] = x.x; dst[m + 1] = x.y;
            }
        } else {
#pragma unroll
            for (int m = 0; m < KPL; ++m) dst[m] = p[m];
        }
    };
    fetch(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    const bool writer = s == 0 && j < E;
    for (int first = 0; first < n; first += GD_CHUNK) {
        const bool more = first + GD_CHUNK < n;
        if (more) fetch(first + GD_CHUNK);
        const int cnt = min(GD_CHUNK, n - first);
        float* orow = o + (size_t)(t0 + first) * H * E + (size_t)h * E + min(j, E - 1);
#pragma unroll 4
        for (int tk = 0; tk < cnt; ++tk) {
            const float* L = lds[buf] + tk * ROWW;
            float kk[KPL], qq[KPL];
            take(L + s * KPL, kk);
            take(L + DP + s * KPL, qq);
            const float v = L[2 * DP + (tid >> 4)];
            const float2 bg = *reinterpret_cast<const float2*>(L + 2 * DP + 16);
            const float b = gd_token<KPL>(S, kk, qq, v, bg.x, bg.y);
            if (writer) orow[(size_t)tk * H * E] = b;
        }
        if (more) stash(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    if (j < E) {
#pragma unroll
        for (int m = 0; m < KPL; ++m)
            if (s + 16 * m < D) sp[16 * m] = S[m];
    }
    if (blockIdx.x == 0) gd_keep_inputs(proj, ldp, srow + tail_off, taps, t0, n, h, gk, H, G, D, E);
}

TFF_API int tff_gdelta_recurrence(const float* pre, const float* proj, size_t ldp, float* state, size_t state_row,
                                  size_t tail_off, int taps, const int32_t* cu_tokens, const int32_t* state_slots, float* o,
                                  int R, int H, int G, int D, int E, int max_tokens, int below, tff_stream_t stream) {
    TFF_REQUIRE(pre && proj && state && cu_tokens && state_slots && o, "gdelta_recurrence: null pointer");
    TFF_REQUIRE(R >= 0 && H > 0 && G > 0 && H % G == 0 && D > 0 && D <= 256 && E > 0 && taps >= 1 && taps <= GD_MAX_TAPS,
                "gdelta_recurrence: bad sizes heads=%d kv_heads=%d dim=%d vdim=%d taps=%d (dim up to 256, taps up to %d)", H, G, D,
                E, taps, GD_MAX_TAPS);
    const size_t C = 2 * (size_t)G * D + (size_t)H * E;
    TFF_REQUIRE(ldp >= C + 2 * (size_t)H && (size_t)H * E * D <= tail_off && tail_off + (size_t)(taps - 1) * C <= state_row,
                "gdelta_recurrence: rows of %zu or state rows of %zu are too short", ldp, state_row);
    TFF_REQUIRE(H <= 65535 && R <= 65535, "gdelta_recurrence: too many heads or requests");
    TFF_REQUIRE((C + 2 * (size_t)H) * 17 < ((size_t)1 << 31), "gdelta_recurrence: rows of %zu channels are too long", C);
    if (R == 0) return 0;
    if (below <= 0) below = INT_MAX;
    const dim3 grid((E + 15) / 16, H, R);
    hipStream_t s = (hipStream_t)stream;
    // (a request's tokens go one after the other: up to GD_FEW of them need no staging through LDS)
#define GD_LAUNCH(KPL)                                                                                                     \
    do {                                                                                                                   \
        if (max_tokens > 0 && max_tokens <= GD_FEW)                                                                        \
            gdelta_recurrence_few_kernel<KPL><<<grid, 256, 0, s>>>(pre, proj, ldp, state, state_row, tail_off, taps,        \
                                                                   cu_tokens, state_slots, o, H, G, D, E, below);          \
        else                                                                                                               \
            gdelta_recurrence_kernel<KPL><<<grid, 256, 0, s>>>(pre, proj, ldp, state, state_row, tail_off, taps, cu_tokens, \
                                                               state_slots, o, H, G, D, E, below);                         \
    } while (0)
    if (D <= 16) GD_LAUNCH(1);
    else if (D <= 32) GD_LAUNCH(2);
    else if (D <= 64) GD_LAUNCH(4);
    else if (D <= 128) GD_LAUNCH(8);
    else GD_LAUNCH(16);
#undef GD_LAUNCH
    return tff_check_launch("gdelta_recurrence");
}

// ------------------------------------------------- long portions: chunks of sixteen tokens ---
// For head sizes of 64, 128 and 256.  Each portion goes by its own length, so that a request's bits do not change with what else
// the step holds: portions of `from` tokens and more run here, shorter ones in the same step token by token.  Within a chunk that starts from S0, with G_t = g_0 .. g_t and P_ts = g_(s+1) .. g_t,
//
//   (I + L) U = B (V - diag(G) K S0),   L_ts = beta_t P_ts (k_t . k_s), s < t;      S_t = G_t S0 + sum over s <= t of P_ts k_s u_s^T
//   O = diag(G) Q S0 + A U,             A_ts = P_ts (q_t . k_s), s <= t
//
// so that a chunk is a handful of products on the float32 matrix cores (v_mfma_f32_16x16x4_f32) instead of sixteen steps that
// wait for one another.  The P are products, not quotients: a decay of zero is a factor like any other.  (I + L)^-1 B and A do not
// depend on S: gdelta_chunk_kernel forms them for all chunks at once, a wave per chunk and head (the inverse by forward
// substitution, a lane a column; its elements are beta_s k_t' (product of reflections) k_s, at most 1 in size).
// gdelta_scan_kernel walks the chunks of a request: a block per head and sixteen value channels, a wave a quarter of the key
// channels, whose part of S stays in its accumulators; the waves' parts of K S0 meet in LDS, one barrier a chunk (those of Q S0 once
// every four chunks, for which the waves then put one output together each), and the next chunks' operands are on their way
// meanwhile.  Accumulators are operands as they are: lane (column r, g) holds rows 4 g .. 4 g + 3 of a product, which is where the
// next product's MFMA j wants row 4 g + j.
// One token after the other took 0.25 us a token: 2,048 tokens of 32 heads of 128 x 128 in 540 us, now 21 + 188; with the preparation,
// 2,048 tokens of 4 heads of 64 x 64 438 / 129, four requests of 901, 700, 430 and 300 tokens 420 / 245.  Relative error against 64
// bits over 96 to 400 tokens, with the preparation (whose terms in 64 bits make up for more than the chunks' own roundings add), before /
// now: heads of 64 1.22e-7 / 1.08e-7, of 128 1.16e-7 / 1.00e-7, of 256 1.03e-7 / 0.95e-7; token by token now 1.07e-7, 0.96e-7, 0.89e-7.
//
// work: per chunk and head 16 x 16 of (I + L)^-1 B, 16 x 16 of A, 16 G, 16 P_15,s; the chunk that starts at token t of row r
// lies at place t / 16 + r.
#define GD_WORK 544


// From zero in two chains of eight terms, which meet at the end: half the wait and a smaller error.
__device__ __forceinline__ gd_floatx4 gd_mfma16(const float4& a, const gd_floatx4& b) {
    const gd_floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    gd_floatx4 x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], zero, 0, 0, 0);
    gd_floatx4 y = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], zero, 0, 0, 0);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], y, 0, 0, 0);
    return x + y;
}

// A block per place of the workspace and head, whatever the portions' lengths: a grid of the longest portion's chunks by requests
// was mostly blocks without work where one long portion met many decoding requests (2,048 tokens beside 47, 32 heads of 128 x 128:
// the whole recurrence 350 us, now 302).
__global__ __launch_bounds__(64) void gdelta_chunk_kernel(const float* __restrict__ pre, const int32_t* __restrict__ cu_tokens,
                                                          float* __restrict__ work, int R, int H, int G, int D, int E, int from) {
    __shared__ double sl[16][17];
    const int h = blockIdx.y, lane = threadIdx.x, c = lane & 15, g = lane >> 4;
    const int r = chunk_place_request(cu_tokens, R, blockIdx.x);
    const int t0 = cu_tokens[r], n = cu_tokens[r + 1] - t0, first = ((int)blockIdx.x - t0 / 16 - r) * 16;
    if (n < from || first >= n) return;
    const int C = 2 * G * D + H * E, gk = h / (H / G);
    const size_t ldq = (size_t)C + 2 * H;
    const int tok = first + c;                            // this lane's token as a row and as a column
    const float* row = pre + (size_t)(t0 + min(tok, n - 1)) * ldq;
    const float* kp = row + (size_t)(G + gk) * D + 4 * g;
    const float* qp = row + (size_t)gk * D + 4 * g;
    // (in 64 bits all of it, here and below: what is rounded here is rounded in whole rows of the results.
    // v_mfma_f64_16x16x4_f64 leaves lane (column c, g) the rows g + 4 i.)
    gd_doublex4 kk = {0., 0., 0., 0.}, qk = {0., 0., 0., 0.};
    for (int d = 0; d < D; d += 32) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const gd_floatx4 k4 = *reinterpret_cast<const gd_floatx4*>(kp + d + 16 * i), q4 = *reinterpret_cast<const gd_floatx4*>(qp + d + 16 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                kk = __builtin_amdgcn_mfma_f64_16x16x4f64((double)k4[e], (double)k4[e], kk, 0, 0, 0);      // k_t . k_s, s = c
                qk = __builtin_amdgcn_mfma_f64_16x16x4f64((double)q4[e], (double)k4[e], qk, 0, 0, 0);
            }
        }
    }
    // (tokens past the portion's end: beta 0, no decay)
    const float beta = tok < n ? row[C + h] : 0.f, dec = tok < n ? row[C + H + h] : 1.f;
    double p[4] = {1., 1., 1., 1.}, gt = 1., pe = 1.;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const double x = (double)__shfl(dec, j, 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] *= (j > c && j <= g + 4 * i) ? x : 1.;
        gt *= j <= c ? x : 1.;
        pe *= j > c ? x : 1.;
    }
    float* w = work + ((size_t)((t0 + first) / 16 + r) * H + h) * GD_WORK;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = g + 4 * i;
        const float bt = __shfl(beta, t, 64);
        sl[t][c] = c < t ? (double)bt * p[i] * kk[i] : 0.;
        w[256 + t * 16 + c] = c <= t ? (float)(p[i] * qk[i]) : 0.f;
    }
    __syncthreads();
    if (lane < 16) {
        double x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            double a = t == c ? 1. : 0.;
#pragma unroll
            for (int s = 0; s < t; ++s) a = fma(-sl[t][s], x[s], a);
            x[t] = a;
            w[t * 16 + c] = (float)(a * (double)beta);
        }
        w[512 + c] = (float)gt;
        w[528 + c] = (float)pe;
    }
}

// WV waves of NT tiles of 16 key channels each (D = 16 WV NT), NC groups of sixteen value channels.  Two groups a block where portions would
// wait for others' blocks (two blocks a CU are resident): the groups share a chunk's keys, queries and factors, so that the portions
// run side by side instead of in two rounds, and each fills the waits of the other's chain.  A chunk then takes 1.45 times as long, and
// its operands are asked for one chunk ahead (AHEAD + 1 sets of registers).  Four requests of 901, 848, 677 and 664
// tokens, 32 heads of 128 x 128, the recurrence with its preparation: 278 us with a group a block, with two 245; a single portion of 901 116 and 159.
template <int NT, int WV, int NC>
__global__ __launch_bounds__(64 * WV) void gdelta_scan_kernel(const float* __restrict__ pre, const float* __restrict__ proj, size_t ldp,
                                                          float* __restrict__ state, size_t state_row, size_t tail_off, int taps,
                                                          const int32_t* __restrict__ cu_tokens,
                                                          const int32_t* __restrict__ state_slots, const float* __restrict__ work,
                                                          float* __restrict__ o, int H, int G, int E, int from) {
    constexpr int D = 16 * WV * NT, AHEAD = NC == 1 ? 2 : 1;
    __shared__ gd_floatx4 px[2][NC][WV][64], py[2][NC][WV][WV][64];      // parts of K S0 by turns; of Q S0 by turns and chunk
    const int h = blockIdx.x, r = blockIdx.z, j0 = blockIdx.y * 16 * NC;      // (a head's blocks on one XCD: they read the same keys and queries)
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int t0 = cu_tokens[r], n = cu_tokens[r + 1] - t0;
    if (n < from) return;                                  // (the whole block: a portion for the token-by-token form)
    const int C = 2 * G * D + H * E, gk = h / (H / G);
    const size_t ldq = (size_t)C + 2 * H;
    float* srow = state + (size_t)state_slots[r] * state_row;
    bool live[NC];
    int j[NC];
    float* sp[NC];
    gd_floatx4 S[NC][NT];
#pragma unroll
    for (int w = 0; w < NC; ++w) {
        live[w] = j0 + 16 * w + c < E;
        j[w] = min(j0 + 16 * w + c, E - 1);
        sp[w] = srow + ((size_t)h * E + j[w]) * D + wv * 16 * NT + 4 * g;
#pragma unroll
        for (int m = 0; m < NT; ++m) S[w][m] = *reinterpret_cast<const gd_floatx4*>(sp[w] + 16 * m);
    }
    struct Ops {
        float4 k[NT], q[NT], inv, att, gt, pe;
        float kt[NT][4], v[NC][4];
    } x[AHEAD + 1];
    // Addresses are a uniform base and a lane's 32-bit offset that is the same for all chunks but the last, whose tokens past the
    // portion's end repeat its last one (their u is zero): with one wave to a SIMD address arithmetic is time.
    const unsigned wstep = (unsigned)H * GD_WORK * 4u, ld = (unsigned)ldq * 4u;
    const int chunks = (n + 15) / 16, last = n - 1 - 16 * (chunks - 1);
    const char* base = (const char*)(pre + (size_t)t0 * ldq);
    const char* wbase = (const char*)(work + ((size_t)(t0 / 16 + r) * H + h) * GD_WORK);
    const unsigned kcol = (unsigned)((G + gk) * D + wv * 16 * NT) * 4u, qcol = (unsigned)(gk * D + wv * 16 * NT) * 4u;
    unsigned vcol[NC];
#pragma unroll
    for (int w = 0; w < NC; ++w) vcol[w] = (unsigned)(2 * G * D + h * E + j[w]) * 4u;
    const unsigned in_w = (unsigned)(c * 16 + 4 * g) * 4u, in_g = (unsigned)(4 * g) * 4u;
    auto fetch = [&](int i, Ops& x) {
        const int most = i + 1 < chunks ? 15 : last;
        const char* b = base + (size_t)i * 16 * ld;
        const char* w = wbase + (size_t)i * wstep;
        const unsigned row = (unsigned)min(c, most) * ld + (unsigned)(4 * g) * 4u;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            x.k[m] = *reinterpret_cast<const float4*>(b + (row + kcol + 64u * m));
            x.q[m] = *reinterpret_cast<const float4*>(b + (row + qcol + 64u * m));
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const unsigned tr = (unsigned)min(4 * g + q, most) * ld;
#pragma unroll
            for (int u = 0; u < NC; ++u) x.v[u][q] = *reinterpret_cast<const float*>(b + (tr + vcol[u]));
#pragma unroll
            for (int m = 0; m < NT; ++m) x.kt[m][q] = *reinterpret_cast<const float*>(b + (tr + kcol + 64u * m + 4u * c));
        }
        x.inv = *reinterpret_cast<const float4*>(w + in_w);
        x.att = *reinterpret_cast<const float4*>(w + (in_w + 1024u));
        x.gt = *reinterpret_cast<const float4*>(w + (in_g + 2048u));
        x.pe = *reinterpret_cast<const float4*>(w + (in_g + 2112u));
    };
    // a chunk's operands are asked for ahead: one group's chunk takes less time than a load from far memory
    int i = 0;
    float* ocol = o + (size_t)t0 * H * E + (size_t)h * E;
    auto meet = [&](const gd_floatx4 (&p)[WV][64]) {       // the waves' parts, added as a tree
        gd_floatx4 v[WV];
#pragma unroll
        for (int w = 0; w < WV; ++w) v[w] = p[w][lane];
#pragma unroll
        for (int k = 1; k < WV; k *= 2)
#pragma unroll
            for (int w = 0; w < WV; w += 2 * k) v[w] = v[w] + v[w + k];
        return v[0];
    };
    // The outputs hang off the chain from chunk to chunk: each wave puts one of WV chunks' together once all of them are through.
    gd_floatx4 own_u[NC], own_gt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NC; ++w) own_u[w] = own_gt;
    float4 own_att = make_float4(0.f, 0.f, 0.f, 0.f);
    auto outputs = [&](int first) {
        const int mine = first + wv;
        if (mine >= chunks) return;
#pragma unroll
        for (int w = 0; w < NC; ++w) {
            const gd_floatx4 y = gd_mfma16(own_att, own_u[w]) + own_gt * meet(py[first / WV & 1][w][wv]);
            float* op = ocol + (size_t)(16 * mine + 4 * g) * H * E + j[w];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (live[w] && 16 * mine + 4 * g + q < n) op[(size_t)q * H * E] = y[q];
        }
    };
    auto chunk = [&](const Ops& now, Ops& ahead) {
        fetch(min(i + AHEAD, chunks - 1), ahead);      // (past the end the last one again: with a condition the wait for a chunk would be one for all)
        const int buf = i & 1;
        gd_floatx4 xw[NC];
#pragma unroll
        for (int w = 0; w < NC; ++w) {
            gd_floatx4 x = gd_mfma16(now.k[0], S[w][0]), y = gd_mfma16(now.q[0], S[w][0]);
#pragma unroll
            for (int m = 1; m < NT; ++m) {
                x = x + gd_mfma16(now.k[m], S[w][m]);
                y = y + gd_mfma16(now.q[m], S[w][m]);
            }
            px[buf][w][wv][lane] = x;
            py[i / WV & 1][w][i % WV][wv][lane] = y;
        }
        __syncthreads();          // (the other buffers were last read before this barrier)
#pragma unroll
        for (int w = 0; w < NC; ++w) xw[w] = meet(px[buf][w]);
        const gd_floatx4 gt = {now.gt.x, now.gt.y, now.gt.z, now.gt.w};
        const float gend = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(now.gt.w), 48));      // G_15: the whole chunk's decay
        gd_floatx4 u[NC];
#pragma unroll
        for (int w = 0; w < NC; ++w) {
            gd_floatx4 v = {now.v[w][0], now.v[w][1], now.v[w][2], now.v[w][3]};
            v = v - gt * xw[w];
            u[w] = gd_mfma16(now.inv, v);
        }
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            const float4 kt = make_float4(now.kt[m][0] * now.pe.x, now.kt[m][1] * now.pe.y, now.kt[m][2] * now.pe.z, now.kt[m][3] * now.pe.w);
#pragma unroll
            for (int w = 0; w < NC; ++w) {
                const gd_floatx4 add = gd_mfma16(kt, u[w]);
#pragma unroll
                for (int e = 0; e < 4; ++e) S[w][m][e] = fmaf(S[w][m][e], gend, add[e]);
            }
        }
        if (wv == i % WV) {
#pragma unroll
            for (int w = 0; w < NC; ++w) own_u[w] = u[w];
            own_gt = gt;
            own_att = now.att;
        }
        if (i % WV == WV - 1) outputs(i - (WV - 1));
        ++i;
    };
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) fetch(min(a, chunks - 1), x[a]);
    for (;;) {
        if constexpr (AHEAD == 2) {
            chunk(x[0], x[2]);
            if (i >= chunks) break;
            chunk(x[1], x[0]);
            if (i >= chunks) break;
            chunk(x[2], x[1]);
        } else {
            chunk(x[0], x[1]);
            if (i >= chunks) break;
            chunk(x[1], x[0]);
        }
        if (i >= chunks) break;
    }
    if (chunks % WV != 0) outputs(chunks - chunks % WV);
    // Where a u is not finite the zeros above the diagonals do not keep it from earlier tokens (0 x inf is not 0).  It is then in every
    // element of its channel of S for good: such a portion's sixteen channels are worked through once more token by token, from the
    // state that still stands.
#pragma unroll
    for (int w = 0; w < NC; ++w) {
        // (the block's vote in LDS that is there: two blocks of two groups take a CU's to the last byte)
        int* vote = reinterpret_cast<int*>(&px[0][0][0][0]);
        __syncthreads();
        if (tid == 0) *vote = 0;
        __syncthreads();
        if (!(fabsf(S[w][0][0]) < INFINITY)) *vote = 1;
        __syncthreads();
        if (*vote) {
            gd_portion<D / 16>(pre, t0, n, srow, o, h, gk, H, G, D, E, j0 + 16 * w);
        } else if (live[w]) {
#pragma unroll
            for (int m = 0; m < NT; ++m) *reinterpret_cast<gd_floatx4*>(sp[w] + 16 * m) = S[w][m];
        }
    }
    if (blockIdx.y == 0) gd_keep_inputs(proj, ldp, srow + tail_off, taps, t0, n, h, gk, H, G, D, E);
}

TFF_API size_t tff_gdelta_chunks_workspace_bytes(int T, int R, int H) { return ((size_t)T / 16 + R) * H * GD_WORK * sizeof(float); }

// (a lane's offset within sixteen rows of pre is 32 bits of bytes)
TFF_API int tff_gdelta_chunks_supported(int R, int H, int G, int D, int E, size_t state_row) {
    const size_t row = 2 * (size_t)G * D + (size_t)H * E + 2 * (size_t)H;
    return (D == 64 || D == 128 || D == 256) && E % 4 == 0 && H % 2 == 0 && state_row % 4 == 0 && H <= 65535 && R <= 65535 &&
           (E + 15) / 16 <= 65535 && row * 17 * sizeof(float) < ((size_t)1 << 32);
}

// As tff_gdelta_recurrence, in chunks, for the portions of `from` tokens and more.  groups: of sixteen value channels a block of the scan, 1,
// or 2 with heads of up to 128 (those of 256 keep one group: their state alone is eight tiles).  Every row's first 2 G D + H E + 2 H channels of pre are
// a multiple of four long, and pre, state and work are 16-byte aligned.
TFF_API int tff_gdelta_recurrence_chunks(const float* pre, const float* proj, size_t ldp, float* state, size_t state_row,
                                         size_t tail_off, int taps, const int32_t* cu_tokens, const int32_t* state_slots, float* work,
                                         float* o, int T, int R, int H, int G, int D, int E, int from, int groups, tff_stream_t stream) {
    TFF_REQUIRE(pre && proj && state && cu_tokens && state_slots && work && o, "gdelta_chunks: null pointer");
    TFF_REQUIRE(groups == 1 || (groups == 2 && D <= 128), "gdelta_chunks: %d groups of value channels a block, heads of %d", groups, D);
    TFF_REQUIRE(R >= 0 && H > 0 && G > 0 && H % G == 0 && E > 0 && taps >= 1 && taps <= GD_MAX_TAPS && T >= 0 && from > 0,
                "gdelta_chunks: bad sizes heads=%d kv_heads=%d vdim=%d taps=%d", H, G, E, taps);
    const size_t C = 2 * (size_t)G * D + (size_t)H * E;
    TFF_REQUIRE(tff_gdelta_chunks_supported(R, H, G, D, E, state_row), "gdelta_chunks: %d requests, %d and %d heads of %d x %d, state rows of %zu",
                R, H, G, D, E, state_row);
    TFF_REQUIRE(((uintptr_t)pre % 16) == 0 && ((uintptr_t)state % 16) == 0 && ((uintptr_t)work % 16) == 0,
                "gdelta_chunks: operands must be 16-byte aligned");
    TFF_REQUIRE(ldp >= C + 2 * (size_t)H && (size_t)H * E * D <= tail_off && tail_off + (size_t)(taps - 1) * C <= state_row,
                "gdelta_chunks: rows of %zu or state rows of %zu are too short", ldp, state_row);
    if (R == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    gdelta_chunk_kernel<<<dim3(T / 16 + R, H), 64, 0, s>>>(pre, cu_tokens, work, R, H, G, D, E, from);
    if (int rc = tff_check_launch("gdelta_chunk")) return rc;
#define GD_SCAN(NT, WV, NC)                                                                                                       \
    gdelta_scan_kernel<NT, WV, NC><<<dim3(H, (E + 16 * NC - 1) / (16 * NC), R), 64 * WV, 0, s>>>(                                    \
        pre, proj, ldp, state, state_row, tail_off, taps, cu_tokens, state_slots, work, o, H, G, E, from)
    if (D == 64 && groups == 2) GD_SCAN(1, 4, 2);
    else if (D == 64) GD_SCAN(1, 4, 1);
    else if (D == 128 && groups == 2) GD_SCAN(2, 4, 2);
    else if (D == 128) GD_SCAN(2, 4, 1);
    else GD_SCAN(4, 4, 1);
#undef GD_SCAN
    return tff_check_launch("gdelta_scan");
}

// One wave per (token, head): the head's E channels of o are divided by their root mean square, multiplied by
// w[channel] (one weight for all heads) and by silu(gate), and go to out[t * out_row + h * E + e].
template <typename TO>
__global__ __launch_bounds__(256) void head_norm_silu_gate_kernel(const float* __restrict__ o, const float* __restrict__ g,
                                                                  size_t g_row, const float* __restrict__ w, float eps,
                                                                  float scale, TO* __restrict__ out, size_t out_row,
                                                                  int pairs, int H, int E) {
    const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (id >= pairs) return;
    const int t = id / H, h = id % H;
    const float* orow = o + ((size_t)t * H + h) * E;
    float ss = 0.f;
    for (int e = lane; e < E; e += 64) ss = fmaf(orow[e], orow[e], ss);
    ss = wave_sum(ss);
    const float rr = scale / sqrtf(ss / (float)E + eps);
    const float* grow = g + (size_t)t * g_row + (size_t)h * E;
    for (int e = lane; e < E; e += 64)
        out[(size_t)t * out_row + (size_t)h * E + e] = from_f32<TO>(orow[e] * rr * w[e] * gd_silu(grow[e]));
}

TFF_API int tff_head_norm_silu_gate(const float* o, const float* g, size_t g_row, const float* w, float eps, float scale,
                                    void* out, size_t out_row, int T, int H, int E, int out_dtype, tff_stream_t stream) {
    TFF_REQUIRE(o && g && w && out, "head_norm_silu_gate: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && E > 0 && g_row >= (size_t)H * E && out_row >= (size_t)H * E, "head_norm_silu_gate: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int pairs = T * H;
    if (out_dtype == TFF_F32 ? launch_head_norm_gate(o, g, g_row, w, 0, eps, scale, (float*)out, out_row, pairs, H, E, s)
                             : out_dtype == TFF_BF16 && launch_head_norm_gate(o, g, g_row, w, 0, eps, scale, (bf16_t*)out, out_row, pairs, H, E, s))
        return tff_check_launch("head_norm_silu_gate");
    if (out_dtype == TFF_F32)
        head_norm_silu_gate_kernel<float><<<(pairs + 3) / 4, 256, 0, s>>>(o, g, g_row, w, eps, scale, (float*)out, out_row, pairs, H, E);
    else if (out_dtype == TFF_BF16)
        head_norm_silu_gate_kernel<bf16_t><<<(pairs + 3) / 4, 256, 0, s>>>(o, g, g_row, w, eps, scale, (bf16_t*)out, out_row, pairs, H, E);
    else
        return tff_fail("head_norm_silu_gate: unknown dtype %d", out_dtype);
    return tff_check_launch("head_norm_silu_gate");
}

// out[t * out_row + h * E + e] = o[t * o_row + h * o_head + e] * sigmoid(g[t * g_row + h * E + e]) * scale
template <typename T>
__global__ __launch_bounds__(256) void sigmoid_gate_heads_kernel(const T* __restrict__ o, size_t o_row, int o_head,
                                                                 const T* __restrict__ g, size_t g_row, float scale,
                                                                 T* __restrict__ out, size_t out_row, int HE, int E,
                                                                 size_t count) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= count) return;
    const size_t t = id / HE;
    const int c = (int)(id - t * HE), h = c / E, e = c - h * E;
    const float gz = to_f32(g[t * g_row + c]);
    out[t * out_row + c] = from_f32<T>(to_f32(o[t * o_row + (size_t)h * o_head + e]) * (scale / (1.0f + expf(-gz))));
}

// bfloat16, eight elements of a head a thread: 16-byte accesses.  us, an element a thread / this: 2,900 tokens of
// 32 heads of 128 30 / 15, 128 tokens 3.3 / 2.8; 48 tokens 2.5 / 2.6 and one 2.3 / 2.5, which stay with the kernel above.
__global__ __launch_bounds__(256) void sigmoid_gate_heads_vec_kernel(const bf16_t* __restrict__ o, size_t o_row, int o_head,
                                                                     const bf16_t* __restrict__ g, size_t g_row, float scale,
                                                                     bf16_t* __restrict__ out, size_t out_row, int HE, int E, size_t eighths) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= eighths) return;
    const size_t t = id / (unsigned)(HE >> 3);
    const int c = (int)(id - t * (HE >> 3)) * 8, h = c / E, e = c - h * E;
    union { uint4 u; bf16_t b[8]; } x, z, y;
    z.u = *reinterpret_cast<const uint4*>(g + t * g_row + c);
    x.u = *reinterpret_cast<const uint4*>(o + t * o_row + (size_t)h * o_head + e);
#pragma unroll
    for (int k = 0; k < 8; ++k) y.b[k] = (bf16_t)((float)x.b[k] * (scale / (1.0f + expf(-(float)z.b[k]))));
    *reinterpret_cast<uint4*>(out + t * out_row + c) = y.u;
}

TFF_API int tff_sigmoid_gate_heads(const void* o, size_t o_row, int o_head, const void* g, size_t g_row, float scale, void* out,
                                   size_t out_row, int T, int H, int E, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(o && g && out, "sigmoid_gate_heads: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && E > 0 && o_head >= E && o_row >= (size_t)H * o_head && g_row >= (size_t)H * E &&
                out_row >= (size_t)H * E, "sigmoid_gate_heads: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const size_t count = (size_t)T * H * E;
    // (up to 2^18 elements, 64 rows of 4,096, more blocks with fewer bytes each are through a little sooner)
    if (dtype == TFF_BF16 && count >= ((size_t)1 << 18) && E % 8 == 0 && o_row % 8 == 0 && o_head % 8 == 0 && g_row % 8 == 0 && out_row % 8 == 0 && ((uintptr_t)o % 16) == 0 &&
        ((uintptr_t)g % 16) == 0 && ((uintptr_t)out % 16) == 0) {
        sigmoid_gate_heads_vec_kernel<<<(unsigned)((count / 8 + 255) / 256), 256, 0, s>>>((const bf16_t*)o, o_row, o_head, (const bf16_t*)g, g_row,
                                                                                          scale, (bf16_t*)out, out_row, H * E, E, count / 8);
        return tff_check_launch("sigmoid_gate_heads");
    }
    const unsigned blocks = (unsigned)((count + 255) / 256);
    if (dtype == TFF_F32)
        sigmoid_gate_heads_kernel<float><<<blocks, 256, 0, s>>>((const float*)o, o_row, o_head, (const float*)g, g_row, scale,
                                                                (float*)out, out_row, H * E, E, count);
    else if (dtype == TFF_BF16)
        sigmoid_gate_heads_kernel<bf16_t><<<blocks, 256, 0, s>>>((const bf16_t*)o, o_row, o_head, (const bf16_t*)g, g_row, scale,
                                                                 (bf16_t*)out, out_row, H * E, E, count);
    else
        return tff_fail("sigmoid_gate_heads: unknown dtype %d", dtype);
    return tff_check_launch("sigmoid_gate_heads");
}
