// A linear recurrence with a matrix of state per head (time mixing in the manner of RWKV):
//
//   o_t = (S_{t-1} + diag(u) k_t v_t^T)^T r_t,      S_t = diag(w_t) S_{t-1} + k_t v_t^T,
//   w_t = exp(-exp(z_t + w0))                        (per head and key channel, float32)
//
// with S [key channel, value channel] per request and head in float32, carried from step to
// step in the request's state row.  The inputs of the projections are mixes of a token's row
// with the row of the token before it, whose last one is part of the state as well.
//
// tff_token_shift_mix: out[m, t, :] = x[t] + (x'[t] - x[t]) * mu[m], x' the row of the token
//   before t in the same request: the row above, or for the first token of a request's portion
//   the row that the state keeps (zeros for a request's first token).
// tff_wkv_recurrence: the recurrence over the tokens of each request's portion of `from` tokens and more but fewer than
//   `below`, one block per (head, request), a thread per value channel and slice of the key channels; the order of every
//   sum is fixed by the head size and the kernel's form alone, so a token's result does not depend on
//   how the tokens were cut into steps beyond rounding (`long_portions` picks the form for prompts, whose
//   sums run in another order than those of the form for single tokens).  The block of head 0 also
//   leaves the portion's last row of x in the state.
// tff_wkv_recurrence_chunks: the same in chunks of sixteen tokens on the float32 matrix cores, for heads of 64 and 128.
// Each portion takes the form that its own length asks for, so that a request's bits do not change with what else a step holds.
// tff_head_norm_gate: out = o / sqrt(mean over the head of o^2 + eps) * weight * silu(g).
// tff_tanh: out = tanh(in), float32 in, the activation type out.
#include "head_norm.h"
#include "tffinfer_kernels.h"
#include <limits.h>

template <typename TO>
__global__ __launch_bounds__(256) void token_shift_mix_kernel(
    const float* __restrict__ x, const float* __restrict__ state, size_t state_row, size_t prev_off,
    const float* __restrict__ mu, int M, const int32_t* __restrict__ token_req,
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ state_slots, TO* __restrict__ out, int T,
    int W) {
    const int t = blockIdx.x;
    const int r = token_req[t];
    const float* prev = (t == cu_tokens[r]) ? state + (size_t)state_slots[r] * state_row + prev_off
                                            : x + (size_t)(t - 1) * W;
    const float* xr = x + (size_t)t * W;
    const int c = blockIdx.y * 256 + threadIdx.x;      // (a block a token and 256 columns: few tokens still fill the GPU)
    if (c < W) {
        const float h = xr[c];
        const float d = prev[c] - h;
        for (int m = 0; m < M; ++m) out[((size_t)m * T + t) * W + c] = from_f32<TO>(h + d * mu[(size_t)m * W + c]);
    }
}

// The same, four columns a thread and TT tokens a block: a plane's row of mu is fetched for TT tokens, a token's row serves the next
// one as its predecessor, and every row of the block is asked for before the first is used.  us, a column a
// thread and a token a block / this: 2,900 tokens of 4,096 into five planes 47 / 28 (5.9 TB/s), 1,000 tokens 20 / 15.5, 128 tokens
// 4.1 / 3.7; 16 tokens and one 2.7 / 2.9, which stay with the kernel above.
template <typename TO, int TT>
__global__ __launch_bounds__(256) void token_shift_mix_vec_kernel(
    const float* __restrict__ x, const float* __restrict__ state, size_t state_row, size_t prev_off,
    const float* __restrict__ mu, int M, const int32_t* __restrict__ token_req,
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ state_slots, TO* __restrict__ out, int T, int W) {
    const int t0 = blockIdx.x * TT, c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= W) return;
    float4 h[TT], d[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) {
        const int t = min(t0 + i, T - 1), r = token_req[t];
        const float* prev = t == cu_tokens[r] ? state + (size_t)state_slots[r] * state_row + prev_off : x + (size_t)(t - 1) * W;
        h[i] = *reinterpret_cast<const float4*>(x + (size_t)t * W + c);
        d[i] = *reinterpret_cast<const float4*>(prev + c);
    }
#pragma unroll
    for (int i = 0; i < TT; ++i) d[i] = make_float4(d[i].x - h[i].x, d[i].y - h[i].y, d[i].z - h[i].z, d[i].w - h[i].w);
    for (int m = 0; m < M; ++m) {
        const float4 k = *reinterpret_cast<const float4*>(mu + (size_t)m * W + c);
#pragma unroll
        for (int i = 0; i < TT; ++i) {
            if (t0 + i >= T) break;
            const float y[4] = {h[i].x + d[i].x * k.x, h[i].y + d[i].y * k.y, h[i].z + d[i].z * k.z, h[i].w + d[i].w * k.w};
            TO* to = out + ((size_t)m * T + t0 + i) * W + c;
            if constexpr (sizeof(TO) == 4) {
                *reinterpret_cast<float4*>(to) = make_float4(y[0], y[1], y[2], y[3]);
            } else {
                union { bf16_t b[4]; uint2 u; } pk;
#pragma unroll
                for (int e = 0; e < 4; ++e) pk.b[e] = (bf16_t)y[e];
                *reinterpret_cast<uint2*>(to) = pk.u;
            }
        }
    }
}

TFF_API int tff_token_shift_mix(const float* x, const float* state, size_t state_row, size_t prev_off, const float* mu,
                                int M, const int32_t* token_req, const int32_t* cu_tokens, const int32_t* state_slots,
                                void* out, int T, int W, int out_dtype, tff_stream_t stream) {
    TFF_REQUIRE(x && state && mu && token_req && cu_tokens && state_slots && out, "token_shift_mix: null pointer");
    TFF_REQUIRE(T >= 0 && W > 0 && M > 0 && prev_off + (size_t)W <= state_row, "token_shift_mix: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    // (up to 2^18 elements, 64 rows of 4,096, more blocks with fewer bytes each are through a little sooner)
    if ((long)T * W >= (1L << 18) && W % 4 == 0 && state_row % 4 == 0 && prev_off % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)state % 16) == 0 && ((uintptr_t)mu % 16) == 0 &&
        ((uintptr_t)out % 16) == 0 && (out_dtype == TFF_F32 || out_dtype == TFF_BF16)) {
        // four tokens a block where that still leaves a few blocks a CU
        const int cols = (W + 1023) / 1024;
        const bool many = (long)T * cols >= 4096;
#define TFF_TSM(TO, TT)                                                                                                           \
    token_shift_mix_vec_kernel<TO, TT><<<dim3((T + TT - 1) / TT, cols), 256, 0, s>>>(x, state, state_row, prev_off, mu, M, token_req,  \
                                                                                    cu_tokens, state_slots, (TO*)out, T, W)
        if (out_dtype == TFF_F32) { if (many) TFF_TSM(float, 4); else TFF_TSM(float, 1); }
        else { if (many) TFF_TSM(bf16_t, 4); else TFF_TSM(bf16_t, 1); }
#undef TFF_TSM
        return tff_check_launch("token_shift_mix");
    }
    const dim3 grid(T, (W + 255) / 256);
    if (out_dtype == TFF_F32)
        token_shift_mix_kernel<float><<<grid, 256, 0, s>>>(x, state, state_row, prev_off, mu, M, token_req, cu_tokens,
                                                         state_slots, (float*)out, T, W);
    else if (out_dtype == TFF_BF16)
        token_shift_mix_kernel<bf16_t><<<grid, 256, 0, s>>>(x, state, state_row, prev_off, mu, M, token_req, cu_tokens,
                                                          state_slots, (bf16_t*)out, T, W);
    else
        return tff_fail("token_shift_mix: unknown dtype %d", out_dtype);
    return tff_check_launch("token_shift_mix");
}

#define WKV_MAX_D 128     // (a thread keeps a slice of a column of S in registers)
#define WKV_MAX_SLICES 4
#define WKV_CHUNK_ELEMS 1024   // tokens of a chunk x padded head size, at most
#define WKV_EPT 4              // elements of a chunk's array a thread fetches, at most

// KPT key channels a thread; ceil(D / KPT) <= 4 slices of the key channels; thread = slice * D + value channel.
// The tokens of a portion pass in chunks of up to 16: a chunk's r, k, w, v are fetched into registers while the
// chunk before it is worked through from LDS, so that no token waits for memory; within a chunk a token costs
// its multiply-adds, its slice of r, k, w in 16-byte LDS reads and one barrier (the slices' partial sums meet
// in LDS, in a buffer of the token's parity).  In LDS a token's channels lie Dp = slices * KPT apart, the
// channels past D zero, so that a slice needs no bounds.
template <int KPT>
__global__ __launch_bounds__(512) void wkv_recurrence_kernel(
    const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ z, size_t row, const float* __restrict__ w0, const float* __restrict__ u,
    float* __restrict__ state, size_t state_row, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ state_slots, float* __restrict__ o, int H, int D, const float* __restrict__ x, int W,
    size_t prev_off, int from, int below) {
    __shared__ __attribute__((aligned(16))) float buf[2][3][WKV_CHUNK_ELEMS];       // r, k, w of a chunk, [token][channel]
    __shared__ float bv[2][WKV_CHUNK_ELEMS];                                       // v of a chunk
    __shared__ float so[WKV_CHUNK_ELEMS];
    __shared__ float part[2][WKV_MAX_SLICES][WKV_MAX_D];
    const int h = blockIdx.x, req = blockIdx.y, tid = threadIdx.x, nt = blockDim.x;
    const int t0 = cu_tokens[req], t1 = cu_tokens[req + 1];
    if (t1 - t0 < from || t1 - t0 >= below) return;       // (the whole block: a portion of no tokens or of another form)
    const int slices = nt / D;
    const int Dp = slices * KPT;
    const int vi = tid % D, ks = tid / D;
    const int C = min(min(16, WKV_EPT * slices), WKV_CHUNK_ELEMS / Dp);      // tokens a chunk
    float* srow = state + (size_t)state_slots[req] * state_row;
    float* S = srow + (size_t)h * D * D;
    const size_t col = (size_t)h * D;
    float s[KPT], uu[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int kk = ks * KPT + i;
        s[i] = kk < D ? S[(size_t)kk * D + vi] : 0.f;
        uu[i] = kk < D ? u[col + kk] : 0.f;
    }
    for (int e = tid; e < 2 * 3 * WKV_CHUNK_ELEMS; e += nt) (&buf[0][0][0])[e] = 0.f;      // (the channels past D stay zero)
    float fr[WKV_EPT], fk[WKV_EPT], fz[WKV_EPT], fv[WKV_EPT];
    // a chunk's elements e = token * D + channel are dealt to the threads in strides of the block
    auto fetch = [&](int base) {
        const int n = min(C, t1 - base) * D;
#pragma unroll
        for (int i = 0; i < WKV_EPT; ++i) {
            const int e = tid + i * nt;
            if (e < n) {
                const size_t a = (size_t)(base + e / D) * row + col + e % D;
                fr[i] = r[a];
                fk[i] = k[a];
                fz[i] = z[a] + w0[col + e % D];
                fv[i] = v[a];
            }
        }
    };
    auto stage = [&](int base, int b) {
        const int n = min(C, t1 - base) * D;
#pragma unroll
        for (int i = 0; i < WKV_EPT; ++i) {
            const int e = tid + i * nt;
            if (e < n) {
                const int at = (e / D) * Dp + e % D;
                buf[b][0][at] = fr[i];
                buf[b][1][at] = fk[i];
                buf[b][2][at] = expf(-expf(fz[i]));
                bv[b][e] = fv[i];
            }
        }
    };
    fetch(t0);
    __syncthreads();
    stage(t0, 0);
    int b = 0;
    for (int base = t0; base < t1; base += C, b ^= 1) {
        const int n = min(C, t1 - base);
        __syncthreads();
        if (base + C < t1) fetch(base + C);
        for (int c = 0; c < n; ++c) {
            const float4* cr = reinterpret_cast<const float4*>(buf[b][0] + c * Dp + ks * KPT);
            const float4* ck = reinterpret_cast<const float4*>(buf[b][1] + c * Dp + ks * KPT);
            const float4* cw = reinterpret_cast<const float4*>(buf[b][2] + c * Dp + ks * KPT);
            const float vt = bv[b][c * D + vi];
            float acc = 0.f;
#pragma unroll
            for (int i = 0; i < KPT; i += 4) {
                const float4 r4 = cr[i >> 2], k4 = ck[i >> 2], w4 = cw[i >> 2];
                const float rr[4] = {r4.x, r4.y, r4.z, r4.w}, kk4[4] = {k4.x, k4.y, k4.z, k4.w},
                            ww[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float kv = kk4[j] * vt;
                    acc = fmaf(rr[j], fmaf(uu[i + j], kv, s[i + j]), acc);
                    s[i + j] = fmaf(ww[j], s[i + j], kv);
                }
            }
            part[c & 1][ks][vi] = acc;
            __syncthreads();
            if (ks == 0) {
                float sum = part[c & 1][0][vi];
                for (int p = 1; p < slices; ++p) sum += part[c & 1][p][vi];
                so[c * D + vi] = sum;
            }
        }
        __syncthreads();
        for (int e = tid; e < n * D; e += nt) o[(size_t)(base + e / D) * H * D + col + e % D] = so[e];
        if (base + C < t1) stage(base + C, b ^ 1);
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        const int kk = ks * KPT + i;
        if (kk < D) S[(size_t)kk * D + vi] = s[i];
    }
    if (h == 0 && x) {
        const float* last = x + (size_t)(t1 - 1) * W;
        for (int c = tid; c < W; c += nt) srow[prev_off + c] = last[c];
    }
}

// The same for head sizes that are multiples of 16 (D = 4 * KPT): a wave takes sixteen value channels, its four
// rows of sixteen lanes a quarter of the key channels each, and the quarters' partial sums meet through lane
// swaps: no barrier and no LDS between the tokens of a chunk, the waves run on their own.
template <int KPT>
__global__ __launch_bounds__(512) void wkv_recurrence_wave_kernel(
    const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ z, size_t row, const float* __restrict__ w0, const float* __restrict__ u,
    float* __restrict__ state, size_t state_row, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ state_slots, float* __restrict__ o, int H, const float* __restrict__ x, int W,
    size_t prev_off, int from, int below) {
    constexpr int D = 4 * KPT;
    constexpr int C = (WKV_CHUNK_ELEMS / D) < 16 ? (WKV_CHUNK_ELEMS / D) : 16;      // tokens a chunk
    constexpr int NT = 4 * D;                                                      // threads: D / 16 waves
    constexpr int EPT = (C * D + NT - 1) / NT;
    __shared__ __attribute__((aligned(16))) float buf[2][3][C * D];       // r, k, w of a chunk, [token][channel]
    __shared__ float bv[2][C * D];
    const int h = blockIdx.x, req = blockIdx.y, tid = threadIdx.x;
    const int t0 = cu_tokens[req], t1 = cu_tokens[req + 1];
    if (t1 - t0 < from || t1 - t0 >= below) return;       // (the whole block: a portion of no tokens or of another form)
    const int lane = tid & 63;
    const int ks = lane >> 4, vi = (tid >> 6) * 16 + (lane & 15);
    float* srow = state + (size_t)state_slots[req] * state_row;
    float* S = srow + (size_t)h * D * D;
    const size_t col = (size_t)h * D;
    float s[KPT], uu[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        s[i] = S[(size_t)(ks * KPT + i) * D + vi];
        uu[i] = u[col + ks * KPT + i];
    }
    float fr[EPT], fk[EPT], fz[EPT], fv[EPT];
    auto fetch = [&](int base) {
        const int n = min(C, t1 - base) * D;
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                const size_t a = (size_t)(base + e / D) * row + col + e % D;
                fr[i] = r[a];
                fk[i] = k[a];
                fz[i] = z[a] + w0[col + e % D];
                fv[i] = v[a];
            }
        }
    };
    auto stage = [&](int base, int b) {
        const int n = min(C, t1 - base) * D;
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = tid + i * NT;
            if (e < n) {
                buf[b][0][e] = fr[i];
                buf[b][1][e] = fk[i];
                buf[b][2][e] = expf(-expf(fz[i]));
                bv[b][e] = fv[i];
            }
        }
    };
    fetch(t0);
    stage(t0, 0);
    int b = 0;
    for (int base = t0; base < t1; base += C, b ^= 1) {
        const int n = min(C, t1 - base);
        __syncthreads();
        if (base + C < t1) fetch(base + C);
        for (int c = 0; c < n; ++c) {
            const float4* cr = reinterpret_cast<const float4*>(buf[b][0] + c * D + ks * KPT);
            const float4* ck = reinterpret_cast<const float4*>(buf[b][1] + c * D + ks * KPT);
            const float4* cw = reinterpret_cast<const float4*>(buf[b][2] + c * D + ks * KPT);
            const float vt = bv[b][c * D + vi];
            float acc = 0.f;
#pragma unroll
            for (int i = 0; i < KPT; i += 4) {
                const float4 r4 = cr[i >> 2], k4 = ck[i >> 2], w4 = cw[i >> 2];
                const float rr[4] = {r4.x, r4.y, r4.z, r4.w}, kk4[4] = {k4.x, k4.y, k4.z, k4.w},
                            ww[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float kv = kk4[j] * vt;
                    acc = fmaf(rr[j], fmaf(uu[i + j], kv, s[i + j]), acc);
                    s[i + j] = fmaf(ww[j], s[i + j], kv);
                }
            }
            acc = rows_sum(acc);        // (quarter 0 + quarter 1) + (quarter 2 + quarter 3), in every lane
            if (ks == 0) o[(size_t)(base + c) * H * D + col + vi] = acc;
        }
        // (the other buffer was last read before this pass's barrier)
        if (base + C < t1) stage(base + C, b ^ 1);
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) S[(size_t)(ks * KPT + i) * D + vi] = s[i];
    if (h == 0 && x) {
        const float* last = x + (size_t)(t1 - 1) * W;
        for (int c = tid; c < W; c += NT) srow[prev_off + c] = last[c];
    }
}

// For long portions (prompts) of heads of 64 or 128 channels (D = 16 * KPT): a token's cost is what bounds a
// prompt, since its tokens go one after the other.  Here a row of sixteen lanes shares a value channel, each
// lane KPT key channels, so a token is KPT steps of four instructions and a sum over the row; a block of four
// waves takes sixteen value channels of a head, D / 16 blocks a head.
template <int KPT>
__global__ __launch_bounds__(256) void wkv_recurrence_rows_kernel(
    const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ z, size_t row, const float* __restrict__ w0, const float* __restrict__ u,
    float* __restrict__ state, size_t state_row, const int32_t* __restrict__ cu_tokens,
    const int32_t* __restrict__ state_slots, float* __restrict__ o, int H, const float* __restrict__ x, int W,
    size_t prev_off, int from, int below) {
    constexpr int D = 16 * KPT;
    constexpr int C = WKV_CHUNK_ELEMS / D;         // tokens a chunk: 16 or 8
    constexpr int NT = 256;
    constexpr int EPT = C * D / NT;                // 4
    constexpr int Q = KPT / 4;
    __shared__ __attribute__((aligned(16))) float buf[2][3][C * D];       // r, k, w of a chunk, [token][channel]
    __shared__ float bv[2][C * 16];                                        // v of the block's sixteen channels
    const int h = blockIdx.x, req = blockIdx.y, tid = threadIdx.x;
    const int t0 = cu_tokens[req], t1 = cu_tokens[req + 1];
    if (t1 - t0 < from || t1 - t0 >= below) return;       // (the whole block: a portion of no tokens or of another form)
    const int lane = tid & 63;
    const int ks = lane & 15, vl = (tid >> 6) * 4 + (lane >> 4), vi = blockIdx.z * 16 + vl;
    float* srow = state + (size_t)state_slots[req] * state_row;
    float* S = srow + (size_t)h * D * D;
    const size_t col = (size_t)h * D;
    float s[KPT], uu[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
        s[i] = S[(size_t)(ks * KPT + i) * D + vi];
        uu[i] = u[col + ks * KPT + i];
    }
    float fr[EPT], fk[EPT], fz[EPT], fv = 0.f;
    auto fetch = [&](int base) {
        const int n = min(C, t1 - base);
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = tid + i * NT;
            if (e < n * D) {
                const size_t a = (size_t)(base + e / D) * row + col + e % D;
                fr[i] = r[a];
                fk[i] = k[a];
                fz[i] = z[a] + w0[col + e % D];
            }
        }
        if (tid < n * 16) fv = v[(size_t)(base + tid / 16) * row + col + blockIdx.z * 16 + tid % 16];
    };
    auto stage = [&](int base, int b) {
        const int n = min(C, t1 - base);
#pragma unroll
        for (int i = 0; i < EPT; ++i) {
            const int e = tid + i * NT;
            if (e < n * D) {
                buf[b][0][e] = fr[i];
                buf[b][1][e] = fk[i];
                buf[b][2][e] = expf(-expf(fz[i]));
            }
        }
        if (tid < n * 16) bv[b][tid] = fv;
    };
    fetch(t0);
    stage(t0, 0);
    int b = 0;
    for (int base = t0; base < t1; base += C, b ^= 1) {
        const int n = min(C, t1 - base);
        __syncthreads();
        if (base + C < t1) fetch(base + C);
        // (unrolled by four: only s runs from token to token, one multiply-add an element; the sums over the rows,
        // the stores and the LDS reads of neighbouring tokens overlap)
        float* orow = o + (size_t)base * H * D + col + vi;
#pragma unroll 4
        for (int c = 0; c < n; ++c) {
            const float4* cr = reinterpret_cast<const float4*>(buf[b][0] + c * D + ks * KPT);
            const float4* ck = reinterpret_cast<const float4*>(buf[b][1] + c * D + ks * KPT);
            const float4* cw = reinterpret_cast<const float4*>(buf[b][2] + c * D + ks * KPT);
            const float vt = bv[b][c * 16 + vl];
            float acc = 0.f;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float4 r4 = cr[q], k4 = ck[q], w4 = cw[q];
                const float rr[4] = {r4.x, r4.y, r4.z, r4.w}, kk4[4] = {k4.x, k4.y, k4.z, k4.w},
                            ww[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float kv = kk4[j] * vt;
                    acc = fmaf(rr[j], fmaf(uu[4 * q + j], kv, s[4 * q + j]), acc);
                    s[4 * q + j] = fmaf(ww[j], s[4 * q + j], kv);
                }
            }
            acc = row16_sum(acc);
            if (ks == 0) orow[(size_t)c * H * D] = acc;
        }
        // (the other buffer was last read before this pass's barrier)
        if (base + C < t1) stage(base + C, b ^ 1);
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) S[(size_t)(ks * KPT + i) * D + vi] = s[i];
    if (h == 0 && blockIdx.z == 0 && x) {
        const float* last = x + (size_t)(t1 - 1) * W;
        for (int c = tid; c < W; c += NT) srow[prev_off + c] = last[c];
    }
}

TFF_API int tff_wkv_recurrence(const float* r, const float* k, const float* v, const float* z, size_t row, const float* w0,
                               const float* u, float* state, size_t state_row, const int32_t* cu_tokens,
                               const int32_t* state_slots, float* o, int R, int H, int D, const float* x, int W,
                               size_t prev_off, int long_portions, int from, int below, tff_stream_t stream) {
    TFF_REQUIRE(r && k && v && z && w0 && u && state && cu_tokens && state_slots && o, "wkv_recurrence: null pointer");
    TFF_REQUIRE(R >= 0 && H > 0 && D > 0 && D <= WKV_MAX_D, "wkv_recurrence: %d heads of %d (up to %d)", H, D, WKV_MAX_D);
    TFF_REQUIRE(row >= (size_t)H * D && (size_t)H * D * D <= state_row && (!x || prev_off + (size_t)W <= state_row),
                "wkv_recurrence: rows of %zu, state rows of %zu do not hold %d heads of %d", row, state_row, H, D);
    TFF_REQUIRE(from > 0, "wkv_recurrence: portions from %d tokens on", from);
    if (R == 0) return 0;
    if (below <= 0) below = INT_MAX;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(H, R);
#define WKV_LAUNCH(KPT)                                                                                              \
    wkv_recurrence_kernel<KPT><<<grid, D * ((D + KPT - 1) / KPT), 0, s>>>(r, k, v, z, row, w0, u, state, state_row, \
                                                                           cu_tokens, state_slots, o, H, D, x, W, prev_off, from, below)
#define WKV_WAVES(KPT)                                                                                             \
    wkv_recurrence_wave_kernel<KPT><<<grid, 16 * KPT, 0, s>>>(r, k, v, z, row, w0, u, state, state_row, cu_tokens, \
                                                              state_slots, o, H, x, W, prev_off, from, below)
    if (long_portions && (D == 64 || D == 128)) {
        const dim3 grid3(H, R, D / 16);
        if (D == 64)
            wkv_recurrence_rows_kernel<4><<<grid3, 256, 0, s>>>(r, k, v, z, row, w0, u, state, state_row, cu_tokens,
                                                                state_slots, o, H, x, W, prev_off, from, below);
        else
            wkv_recurrence_rows_kernel<8><<<grid3, 256, 0, s>>>(r, k, v, z, row, w0, u, state, state_row, cu_tokens,
                                                                state_slots, o, H, x, W, prev_off, from, below);
    } else if (D % 16 == 0) {
        switch (D / 4) {
            case 4: WKV_WAVES(4); break;
            case 8: WKV_WAVES(8); break;
            case 12: WKV_WAVES(12); break;
            case 16: WKV_WAVES(16); break;
            case 20: WKV_WAVES(20); break;
            case 24: WKV_WAVES(24); break;
            case 28: WKV_WAVES(28); break;
            default: WKV_WAVES(32); break;
        }
    } else if (D <= 64) WKV_LAUNCH(16);
    else WKV_LAUNCH(32);
#undef WKV_WAVES
#undef WKV_LAUNCH
    return tff_check_launch("wkv_recurrence");
}

// ------------------------------------------------- portions in chunks of sixteen tokens ---
// For heads of 64 and 128.  Within a chunk that starts from S0, with F_t = w_0 .. w_(t-1) and P_ts = w_(s+1) .. w_(t-1) per key channel,
//
//   o_t = S0^T (F_t r_t) + sum over s < t of (sum over i of r_t[i] P_ts[i] k_s[i]) v_s + (sum over i of r_t[i] u[i] k_t[i]) v_t
//   S  <- diag(w_0 .. w_15) S0 + sum over s of (w_(s+1) .. w_15 k_s) v_s^T
//
// No factor is a quotient (a running product of decays underflows): all are products of up to fifteen decays, formed where they are
// used.  wkv_chunk_kernel works out what does not depend on S, a wave per chunk and head (lane (token, quarter of every sixteen channels);
// the sums over channels for all pairs of tokens, walking s down from t while the product grows by one decay a step).
// wkv_scan_kernel carries S through a request's chunks with products on the float32 matrix cores: a block per head and sixteen value
// channels, a wave a quarter of the key channels with its part of S in its accumulators; the waves' parts of an output meet
// in LDS.  S itself waits for one multiply-add a chunk.
// A token after the other took 0.25 - 0.28 us a token, however wide the GPU: us, called from Python, before / now for 1,500 tokens of 64
// heads of 64 374 / 92 (chunks 41, scan 47), of 16 heads of 128 652 / 110, of 4 heads of 64 297 / 62; four portions of 901, 700, 430 and
// 300 tokens 280 / 129.  Relative error of the outputs against 64 bits 8.7e-8 / 6.7e-8 (heads of 128: 9.5e-8 / 6.8e-8).
//
// work: per chunk and head 16 rows of F_t r_t, 16 of w_(s+1) .. w_15 k_s, 16 x 16 weights of v, the chunk's decays; the chunk that
// starts at token t of row r lies at place t / 16 + r.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float wkv_floatx4;

// from zero in two chains of eight terms that meet at the end: half the wait and a smaller error
__device__ __forceinline__ wkv_floatx4 wkv_mfma16(const wkv_floatx4& a, const wkv_floatx4& b) {
    const wkv_floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    wkv_floatx4 x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0], b[0], zero, 0, 0, 0);
    wkv_floatx4 y = __builtin_amdgcn_mfma_f32_16x16x4f32(a[2], b[2], zero, 0, 0, 0);
    x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[1], b[1], x, 0, 0, 0);
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(a[3], b[3], y, 0, 0, 0);
    return x + y;
}
constexpr int wkv_work(int D) { return 33 * D + 256; }

// A block per place of the workspace and head (heads fastest), whatever the portions' lengths: a grid of the longest portion's chunks by
// requests was mostly blocks without work where one long portion met many decoding requests (2,048 tokens beside 47, 64 heads of
// 64: the whole recurrence 250 us, now 167).
template <int D>
__global__ __launch_bounds__(64) void wkv_chunk_kernel(const float* __restrict__ r, const float* __restrict__ k,
                                                       const float* __restrict__ z, size_t row, const float* __restrict__ w0,
                                                       const float* __restrict__ u, const int32_t* __restrict__ cu_tokens,
                                                       float* __restrict__ work, int R, int H, int from) {
    constexpr int M = D / 16, LDR = D + 4;
    __shared__ __attribute__((aligned(16))) float ks[16 * LDR], ws[16 * LDR];
    const int place = blockIdx.x / H, h = blockIdx.x - place * H, lane = threadIdx.x, c = lane & 15, g = lane >> 4;
    const int req = chunk_place_request(cu_tokens, R, place);
    const int t0 = cu_tokens[req], n = cu_tokens[req + 1] - t0, first = (place - t0 / 16 - req) * 16;
    if (n < from || first >= n) return;
    const bool live = first + c < n;                      // (tokens past the portion's end: no key, no decay)
    const size_t at = (size_t)(t0 + min(first + c, n - 1)) * row + (size_t)h * D + 4 * g;
    const float* up = u + (size_t)h * D + 4 * g;
    const float* bp = w0 + (size_t)h * D + 4 * g;
    wkv_floatx4 x[M], kk[M], w[M];
    double own = 0.;                                      // r u k of the token itself
#pragma unroll
    for (int m = 0; m < M; ++m) {
        x[m] = *reinterpret_cast<const wkv_floatx4*>(r + at + 16 * m);
        kk[m] = *reinterpret_cast<const wkv_floatx4*>(k + at + 16 * m);
        w[m] = *reinterpret_cast<const wkv_floatx4*>(z + at + 16 * m);
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const wkv_floatx4 b = *reinterpret_cast<const wkv_floatx4*>(bp + 16 * m), uu = *reinterpret_cast<const wkv_floatx4*>(up + 16 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            w[m][e] = live ? expf(-expf(w[m][e] + b[e])) : 1.f;
            kk[m][e] = live ? kk[m][e] : 0.f;
            own = fma((double)x[m][e] * (double)uu[e], (double)kk[m][e], own);
        }
        *reinterpret_cast<wkv_floatx4*>(ks + c * LDR + 16 * m + 4 * g) = kk[m];
        *reinterpret_cast<wkv_floatx4*>(ws + c * LDR + 16 * m + 4 * g) = w[m];
    }
    __syncthreads();
    float* wp = work + ((size_t)((t0 + first) / 16 + req) * H + h) * wkv_work(D);
    auto quarters = [](double a) {                        // the sum over the four lanes of a token
        a += __shfl_xor(a, 16, 64);
        return a + __shfl_xor(a, 32, 64);
    };
    own = quarters(own);
    wkv_floatx4 att = {0.f, 0.f, 0.f, 0.f};
    // (products and sums in 64 bits: up to fifteen roundings of a product would be seen in the results)
    double p[M][4];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[m][e] = (double)x[m][e];
#pragma unroll
    for (int s = 15; s >= 0; --s) {
        double a = 0.;
        if (s < c) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const wkv_floatx4 y = *reinterpret_cast<const wkv_floatx4*>(ks + s * LDR + 16 * m + 4 * g);
                const wkv_floatx4 d = *reinterpret_cast<const wkv_floatx4*>(ws + s * LDR + 16 * m + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a = fma(p[m][e], (double)y[e], a);
                    p[m][e] *= (double)d[e];
                }
            }
        }
        a = quarters(a);
        if (s >> 2 == g) att[s & 3] = s < c ? (float)a : (s == c ? (float)own : 0.f);
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {                         // (p is r times all decays before its token by now)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[m][e] = (float)p[m][e];
        *reinterpret_cast<wkv_floatx4*>(wp + c * D + 16 * m + 4 * g) = x[m];
    }
    *reinterpret_cast<wkv_floatx4*>(wp + 32 * D + c * 16 + 4 * g) = att;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) p[m][e] = 1.;
#pragma unroll
    for (int j = 15; j > 0; --j)
        if (j > c) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const wkv_floatx4 d = *reinterpret_cast<const wkv_floatx4*>(ws + j * LDR + 16 * m + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) p[m][e] *= (double)d[e];
            }
        }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        wkv_floatx4 end;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            end[e] = (float)((double)w[m][e] * p[m][e]);
            kk[m][e] = (float)((double)kk[m][e] * p[m][e]);
        }
        *reinterpret_cast<wkv_floatx4*>(wp + 16 * D + c * D + 16 * m + 4 * g) = kk[m];
        if (c == 0) *reinterpret_cast<wkv_floatx4*>(wp + 32 * D + 256 + 16 * m + 4 * g) = end;
    }
}

// A portion of one head and sixteen value channels from j0 on, token by token, by a block of 256: as wkv_recurrence_rows_kernel,
// without its way through LDS.
template <int KPT>
__device__ __forceinline__ void wkv_portion(const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v,
                                            const float* __restrict__ z, size_t row, const float* __restrict__ w0,
                                            const float* __restrict__ u, int t0, int n, float* __restrict__ S, float* __restrict__ o,
                                            int h, int H, int j0) {
    constexpr int D = 16 * KPT;
    const int ks = threadIdx.x & 15, vi = j0 + (int)(threadIdx.x >> 4);
    const size_t col = (size_t)h * D + ks * KPT;
    float s[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) s[i] = S[(size_t)(ks * KPT + i) * D + vi];
    for (int t = t0; t < t0 + n; ++t) {
        const size_t a = (size_t)t * row;
        const float vt = v[a + (size_t)h * D + vi];
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < KPT; ++i) {
            const float kv = k[a + col + i] * vt;
            acc = fmaf(r[a + col + i], fmaf(u[col + i], kv, s[i]), acc);
            s[i] = fmaf(expf(-expf(z[a + col + i] + w0[col + i])), s[i], kv);
        }
        acc = row16_sum(acc);
        if (ks == 0) o[(size_t)t * H * D + (size_t)h * D + vi] = acc;
    }
#pragma unroll
    for (int i = 0; i < KPT; ++i) S[(size_t)(ks * KPT + i) * D + vi] = s[i];
}

// Four waves of NT tiles of 16 key channels (D = 64 NT).  Four chunks between two barriers: after the barrier each wave has one
// chunk's output to put together, so that no wave waits for another's.
template <int NT>
__global__ __launch_bounds__(256) void wkv_scan_kernel(const float* __restrict__ r, const float* __restrict__ k,
                                                       const float* __restrict__ v, const float* __restrict__ z, size_t row,
                                                       const float* __restrict__ w0, const float* __restrict__ u,
                                                       float* __restrict__ state, size_t state_row,
                                                       const int32_t* __restrict__ cu_tokens,
                                                       const int32_t* __restrict__ state_slots, const float* __restrict__ work,
                                                       float* __restrict__ o, int H, const float* __restrict__ x, int W, size_t prev_off, int from) {
    constexpr int D = 64 * NT;
    __shared__ wkv_floatx4 part[2][4][4][64];              // by turns, chunk, wave
    const int h = blockIdx.x, req = blockIdx.z, j0 = blockIdx.y * 16;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int t0 = cu_tokens[req], n = cu_tokens[req + 1] - t0;
    if (n < from) return;
    float* srow = state + (size_t)state_slots[req] * state_row;
    float* sp = srow + (size_t)h * D * D + (size_t)(wv * 16 * NT + 4 * g) * D + j0 + c;
    wkv_floatx4 S[NT];
#pragma unroll
    for (int m = 0; m < NT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[m][i] = sp[(size_t)(16 * m + i) * D];
    struct Ops {
        wkv_floatx4 r[NT], kt[NT], w[NT], v;
    } ops[4];
    // Addresses are a uniform base and a lane's 32-bit offset that is the same for all chunks but the last, whose tokens past the
    // portion's end repeat its last one (their keys are zero).
    const int chunks = (n + 15) / 16, last = n - 1 - 16 * (chunks - 1);
    const char* wbase = (const char*)(work + ((size_t)(t0 / 16 + req) * H + h) * wkv_work(D));
    const size_t wstep = (size_t)H * wkv_work(D) * 4;
    const char* vbase = (const char*)(v + (size_t)t0 * row + (size_t)h * D + j0);
    const unsigned ldv = (unsigned)row * 4u;
    const unsigned in_r = (unsigned)(c * D + 4 * g + wv * 16 * NT) * 4u, in_k = (unsigned)(16 * D + 4 * g * D + c + wv * 16 * NT) * 4u;
    const unsigned in_w = (unsigned)(32 * D + 256 + 4 * g + wv * 16 * NT) * 4u, in_a = (unsigned)(32 * D + c * 16 + 4 * g) * 4u;
    auto fetch = [&](int i, Ops& q) {
        const int most = i + 1 < chunks ? 15 : last;
        const char* w = wbase + (size_t)i * wstep;
        const char* vp = vbase + (size_t)i * 16 * ldv;
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            q.r[m] = *reinterpret_cast<const wkv_floatx4*>(w + (in_r + 64u * m));
            q.w[m] = *reinterpret_cast<const wkv_floatx4*>(w + (in_w + 64u * m));
#pragma unroll
            for (int e = 0; e < 4; ++e) q.kt[m][e] = *reinterpret_cast<const float*>(w + (in_k + (unsigned)(e * D + 16 * m) * 4u));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            q.v[e] = *reinterpret_cast<const float*>(vp + ((unsigned)min(4 * g + e, most) * ldv + (unsigned)c * 4u));
    };
#pragma unroll
    for (int a = 0; a < 4; ++a) fetch(min(a, chunks - 1), ops[a]);
    int buf = 0;
    for (int first = 0; first < chunks; first += 4, buf ^= 1) {
        const int mine = first + wv;
        const wkv_floatx4 att = *reinterpret_cast<const wkv_floatx4*>(wbase + (size_t)min(mine, chunks - 1) * wstep + in_a);
        wkv_floatx4 vm = ops[0].v;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            Ops& now = ops[a];
            if (a > 0 && wv == a) vm = now.v;
            if (first + a < chunks) {
                wkv_floatx4 y = wkv_mfma16(now.r[0], S[0]);
#pragma unroll
                for (int m = 1; m < NT; ++m) y = y + wkv_mfma16(now.r[m], S[m]);
#pragma unroll
                for (int m = 0; m < NT; ++m) {
                    const wkv_floatx4 add = wkv_mfma16(now.kt[m], now.v);
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[m][e] = fmaf(S[m][e], now.w[m][e], add[e]);
                }
                part[buf][a][wv][lane] = y;
            }
            fetch(min(first + 4 + a, chunks - 1), now);   // (past the end the last one again: a condition would make the waits exact for neither)
        }
        __syncthreads();                                  // (the other buffer was last read before this barrier)
        if (mine < chunks) {
            wkv_floatx4 y = (part[buf][wv][0][lane] + part[buf][wv][1][lane]) + (part[buf][wv][2][lane] + part[buf][wv][3][lane]);
            y = wkv_mfma16(att, vm) + y;
            float* op = o + (size_t)(t0 + 16 * mine + 4 * g) * H * D + (size_t)h * D + j0 + c;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (16 * mine + 4 * g + q < n) op[(size_t)q * H * D] = y[q];
        }
    }
    // A value that is not finite meets the zero weights of earlier tokens of its chunk (0 x inf is not 0).  It is then in every element of
    // its channel of S for good: such a portion's sixteen channels are worked through once more token by token, from the state
    // that still stands.
    if (__syncthreads_or(!(fabsf(S[0][0]) < INFINITY))) {
        wkv_portion<D / 16>(r, k, v, z, row, w0, u, t0, n, srow + (size_t)h * D * D, o, h, H, j0);
    } else {
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) sp[(size_t)(16 * m + e) * D] = S[m][e];
    }
    if (h == 0 && blockIdx.y == 0 && x) {
        const float* lastx = x + (size_t)(t0 + n - 1) * W;
        for (int e = tid; e < W; e += 256) srow[prev_off + e] = lastx[e];
    }
}

TFF_API size_t tff_wkv_chunks_workspace_bytes(int T, int R, int H, int D) {
    return ((size_t)T / 16 + R) * H * wkv_work(D) * sizeof(float);
}

// (a lane's offset within sixteen rows is 32 bits of bytes)
TFF_API int tff_wkv_chunks_supported(int T, int R, int H, int D, size_t row) {
    return (D == 64 || D == 128) && row % 4 == 0 && row < ((size_t)1 << 25) && R <= 65535 && ((size_t)T / 16 + R) * H < ((size_t)1 << 31);
}

// As tff_wkv_recurrence, for heads of 64 and 128 and portions of `from` tokens and more; row a multiple of 4 and r, k, z, w0, u and
// work 16-byte aligned.
TFF_API int tff_wkv_recurrence_chunks(const float* r, const float* k, const float* v, const float* z, size_t row, const float* w0,
                                      const float* u, float* state, size_t state_row, const int32_t* cu_tokens,
                                      const int32_t* state_slots, float* work, float* o, int T, int R, int H, int D, const float* x,
                                      int W, size_t prev_off, int from, tff_stream_t stream) {
    TFF_REQUIRE(r && k && v && z && w0 && u && state && cu_tokens && state_slots && work && o, "wkv_chunks: null pointer");
    TFF_REQUIRE(R >= 0 && T >= 0 && H > 0 && from > 0 && tff_wkv_chunks_supported(T, R, H, D, row),
                "wkv_chunks: %d requests of %d tokens, %d heads of %d (64 or 128), rows of %zu", R, T, H, D, row);
    TFF_REQUIRE(row >= (size_t)H * D && (size_t)H * D * D <= state_row && (!x || prev_off + (size_t)W <= state_row),
                "wkv_chunks: rows of %zu, state rows of %zu do not hold %d heads of %d", row, state_row, H, D);
    TFF_REQUIRE(((uintptr_t)r % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)z % 16) == 0 && ((uintptr_t)w0 % 16) == 0 &&
                ((uintptr_t)u % 16) == 0 && ((uintptr_t)work % 16) == 0, "wkv_chunks: operands must be 16-byte aligned");
    if (R == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(H, D / 16, R);
    const unsigned pieces = (unsigned)((T / 16 + R) * H);
    if (D == 64) wkv_chunk_kernel<64><<<pieces, 64, 0, s>>>(r, k, z, row, w0, u, cu_tokens, work, R, H, from);
    else wkv_chunk_kernel<128><<<pieces, 64, 0, s>>>(r, k, z, row, w0, u, cu_tokens, work, R, H, from);
    if (int rc = tff_check_launch("wkv_chunk")) return rc;
    if (D == 64) wkv_scan_kernel<1><<<grid, 256, 0, s>>>(r, k, v, z, row, w0, u, state, state_row, cu_tokens, state_slots, work, o, H, x, W, prev_off, from);
    else wkv_scan_kernel<2><<<grid, 256, 0, s>>>(r, k, v, z, row, w0, u, state, state_row, cu_tokens, state_slots, work, o, H, x, W, prev_off, from);
    return tff_check_launch("wkv_scan");
}

template <typename TO>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ o, const float* __restrict__ g,
                                                             size_t g_row, const float* __restrict__ nw, float eps,
                                                             TO* __restrict__ out, int pairs, int H, int D) {
    const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (id >= pairs) return;
    const int t = id / H, h = id % H;
    const float* orow = o + ((size_t)t * H + h) * D;
    float ss = 0.f;
    for (int e = lane; e < D; e += 64) ss = fmaf(orow[e], orow[e], ss);
    ss = wave_sum(ss);
    const float rr = 1.0f / sqrtf(ss / (float)D + eps);
    const float* grow = g + (size_t)t * g_row + (size_t)h * D;
    for (int e = lane; e < D; e += 64) {
        const float gz = grow[e];
        const float gate = gz / (1.0f + expf(-gz));
        out[((size_t)t * H + h) * D + e] = from_f32<TO>(orow[e] * rr * nw[h * D + e] * gate);
    }
}

TFF_API int tff_head_norm_gate(const float* o, const float* g, size_t g_row, const float* nw, float eps, void* out, int T,
                               int H, int D, int out_dtype, tff_stream_t stream) {
    TFF_REQUIRE(o && g && nw && out, "head_norm_gate: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && D > 0 && g_row >= (size_t)H * D, "head_norm_gate: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int pairs = T * H;
    if (out_dtype == TFF_F32 ? launch_head_norm_gate(o, g, g_row, nw, D, eps, 1.0f, (float*)out, (size_t)H * D, pairs, H, D, s)
                             : out_dtype == TFF_BF16 && launch_head_norm_gate(o, g, g_row, nw, D, eps, 1.0f, (bf16_t*)out, (size_t)H * D, pairs, H, D, s))
        return tff_check_launch("head_norm_gate");
    if (out_dtype == TFF_F32)
        head_norm_gate_kernel<float><<<(pairs + 3) / 4, 256, 0, s>>>(o, g, g_row, nw, eps, (float*)out, pairs, H, D);
    else if (out_dtype == TFF_BF16)
        head_norm_gate_kernel<bf16_t><<<(pairs + 3) / 4, 256, 0, s>>>(o, g, g_row, nw, eps, (bf16_t*)out, pairs, H, D);
    else
        return tff_fail("head_norm_gate: unknown dtype %d", out_dtype);
    return tff_check_launch("head_norm_gate");
}

template <typename TO>
__global__ __launch_bounds__(256) void tanh_kernel(const float* __restrict__ in, TO* __restrict__ out, size_t count) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) out[i] = from_f32<TO>(tanhf(in[i]));
}

TFF_API int tff_tanh(const float* in, void* out, size_t count, int out_dtype, tff_stream_t stream) {
    TFF_REQUIRE(in && out, "tanh: null pointer");
    if (count == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const unsigned blocks = (unsigned)((count + 255) / 256);
    if (out_dtype == TFF_F32)
        tanh_kernel<float><<<blocks, 256, 0, s>>>(in, (float*)out, count);
    else if (out_dtype == TFF_BF16)
        tanh_kernel<bf16_t><<<blocks, 256, 0, s>>>(in, (bf16_t*)out, count);
    else
        return tff_fail("tanh: unknown dtype %d", out_dtype);
    return tff_check_launch("tanh");
}
