// A feed-forward made of many small experts of which every token uses a few.
//
// tff_route_topk:   z = Wr h in float32 (or given: a product that ran before), s = sigmoid(z); the `top` experts with the largest
//                   s + bias are chosen (the lowest index among equals), their weights are
//                   s / (sum of the chosen s + 1e-20): the bias moves the choice only.  With `softmax`,
//                   s = softmax(z) over all experts and the weights are the chosen s as they are.
//                   With `groups`, E / groups neighbours form a group whose score is the sum of its two
//                   largest s + bias, and only experts of the best `keep` groups can be chosen.  The weights
//                   are multiplied by `scale`.  With `shared`, z has one row more, whose sigmoid goes there (the
//                   weight of an expert that every token uses).
// tff_experts_gate_up: for every (token, chosen expert): g = min(Wg h, limit),
//                   u = clamp(Wu h, -limit, limit), y = g * sigmoid(act_alpha * g) * (u + up_offset)
//                   (limit = infinity, act_alpha = 1, up_offset = 0: silu(g) * u).
// tff_experts_down: out[t] = sum over the token's experts, in the order they were chosen, of
//                   weight * (Wd y), float32.
//
// Experts numbered E and beyond have no matrices: such an expert hands its input on, f_e = h.
//
// The two expert kernels give every (token, expert) pair waves of its own that stream the
// expert's rows once: what a step of few tokens is bound by.  Each output element is one
// wave's dot product in a fixed order of k, so a token's result does not depend on what else
// the step holds.  Expert weights lie [experts, out, in], row-major, rows ldw elements apart (ldw >= in:
// rows a power of two of bytes apart all come through one memory channel, so the loader puts a
// little room behind each).
#include "common.h"
#include "mfma_tiles.h"
#include "tffinfer_kernels.h"
#include <math.h>
#include <type_traits>

// dot product of two rows of K elements by one wave (lanes stride through k, then a tree)
template <typename TA, typename TB>
__device__ __forceinline__ float wave_dot(const TA* __restrict__ a, const TB* __restrict__ b, int K, int lane) {
    float acc = 0.f;
    for (int k = lane; k < K; k += 64) acc = fmaf(to_f32(a[k]), to_f32(b[k]), acc);
    return wave_sum(acc);
}
// Dot products of one bfloat16 row with R others at once (K a multiple of 8, rows 16-byte aligned): eight elements a lane
// and load, U loads of each row asked for before the first is used.  A lane adds its elements in ascending order, whatever R and U.
template <int R, int U>
__device__ __forceinline__ void wave_dots8(const bf16_t* __restrict__ a, const bf16_t* const (&b)[R], int K, int lane, float (&acc)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    for (int k = lane * 8; k < K; k += 512 * U) {
        union P { uint4 u; bf16_t h[8]; };
        P x[U], y[R][U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + 512 * u < K) {
                x[u].u = *reinterpret_cast<const uint4*>(a + k + 512 * u);
#pragma unroll
                for (int r = 0; r < R; ++r) y[r][u].u = *reinterpret_cast<const uint4*>(b[r] + k + 512 * u);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (k + 512 * u < K) {
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[r] = fmaf((float)x[u].h[j], (float)y[r][u].h[j], acc[r]);
            }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);
}
#define RT_MAX_E 1024

// One block of RT_WAVES waves per token.  logits != null: z is given (a product that ran before);
// else the waves compute it, each its share of the experts, 16 bytes a lane and load.
#define RT_WAVES 8

template <typename T>
__global__ __launch_bounds__(64 * RT_WAVES) void route_topk_kernel(const T* __restrict__ h, int h_row,
                                                                   const float* __restrict__ Wr,
                                                                   const float* __restrict__ logits,
                                                                   const float* __restrict__ bias, int width, int E,
                                                                   int top, int softmax, int groups, int keep, float scale,
                                                                   float* __restrict__ shared, int32_t* __restrict__ idx,
                                                                   float* __restrict__ wts) {
    __shared__ float s_all[RT_MAX_E + 1];
    __shared__ float c_all[RT_MAX_E];
    __shared__ float g_all[RT_MAX_E];       // a group's score; of the chosen groups -infinity
    __shared__ int chosen[64];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int rows = E + (shared ? 1 : 0);
    if (logits) {
        for (int e = threadIdx.x; e < rows; e += blockDim.x) s_all[e] = logits[(size_t)t * rows + e];
    } else {
        const T* hr = h + (size_t)t * h_row;
        for (int e = wv; e < rows; e += RT_WAVES) {
            const float z = wave_dot(hr, Wr + (size_t)e * width, width, lane);
            if (lane == 0) s_all[e] = z;
        }
    }
    __syncthreads();
    if (wv > 0) return;
    // (one wave from here on: LDS works through its accesses in order)
    if (softmax == 1) {
        // s = exp(z - max) / sum over all experts, the sum in the order of the lanes' strides and a tree
        float mx = -INFINITY;
        for (int e = lane; e < E; e += 64) mx = fmaxf(mx, s_all[e]);
        mx = wave_max(mx);
        float den = 0.f;
        for (int e = lane; e < E; e += 64) {
            const float x = expf(s_all[e] - mx);
            s_all[e] = x;
            den += x;
        }
        den = wave_sum(den);
        for (int e = lane; e < E; e += 64) {
            const float s = s_all[e] / den;
            s_all[e] = s;
            c_all[e] = s + (bias ? bias[e] : 0.f);
        }
    } else {
        for (int e = lane; e < E; e += 64) {
            const float s = 1.0f / (1.0f + expf(-s_all[e]));
            s_all[e] = s;
            c_all[e] = s + (bias ? bias[e] : 0.f);
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    // the first of the largest of n numbers in LDS
    auto largest = [&](const float* v, int n) {
        float best = -INFINITY;
        int bi = 0x7fffffff;
        for (int e = lane; e < n; e += 64) {
            const float c = v[e];
            if (c > best) { best = c; bi = e; }      // (ascending e: the first of equals stays)
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
        }
        return min(bi, n - 1);
    };
    if (keep < groups) {
        const int size = E / groups;
        for (int g = lane; g < groups; g += 64) {
            float a = -INFINITY, b = -INFINITY;      // the two largest
            for (int j = 0; j < size; ++j) {
                const float c = c_all[g * size + j];
                b = fmaxf(b, fminf(a, c));
                a = fmaxf(a, c);
            }
            g_all[g] = size > 1 ? a + b : a;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
        for (int k = 0; k < keep; ++k) {
            const int g = largest(g_all, groups);
            if (lane == 0) g_all[g] = -INFINITY;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
        }
        for (int e = lane; e < E; e += 64)
            if (g_all[e / size] != -INFINITY) c_all[e] = -INFINITY;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
    float sum = 0.f;
    for (int k = 0; k < top; ++k) {
        const int bi = largest(c_all, E);
        // (one wave from here on: LDS works through its accesses in order)
        if (lane == 0) {
            idx[(size_t)t * top + k] = bi;
            chosen[k] = bi;
            c_all[bi] = -INFINITY;
        }
        sum += s_all[bi];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
    const float inv = softmax ? 1.0f : 1.0f / (sum + 1e-20f);      // (mode 2: sigmoid scores as they are)
    if (lane < top) wts[(size_t)t * top + lane] = s_all[chosen[lane]] * inv * scale;
    if (shared && lane == 0) shared[t] = 1.0f / (1.0f + expf(-s_all[E]));
}

TFF_API int tff_route_topk(const void* h, int h_row, const float* Wr, const float* logits, const float* bias, int T,
                           int width, int E, int top, int softmax, int groups, int keep, float scale, float* shared, int32_t* idx,
                           float* wts, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(idx && wts && (logits || (h && Wr)), "route_topk: null pointer");
    TFF_REQUIRE(T >= 0 && (logits || (width > 0 && h_row >= width)), "route_topk: bad sizes T=%d width=%d row=%d", T, width, h_row);
    TFF_REQUIRE(E > 0 && E <= RT_MAX_E && top > 0 && top <= E && top <= 64,
                "route_topk: %d of %d experts (up to 64 of up to %d)", top, E, RT_MAX_E);
    TFF_REQUIRE(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (E / groups),
                "route_topk: %d of %d experts from %d of %d groups", top, E, keep, groups);
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == TFF_F32)
        route_topk_kernel<float><<<T, 64 * RT_WAVES, 0, s>>>((const float*)h, h_row, Wr, logits, bias, width, E, top, softmax,
                                                                groups, keep, scale, shared, idx, wts);
    else if (dtype == TFF_BF16)
        route_topk_kernel<bf16_t><<<T, 64 * RT_WAVES, 0, s>>>((const bf16_t*)h, h_row, Wr, logits, bias, width, E, top, softmax,
                                                                groups, keep, scale, shared, idx, wts);
    else
        return tff_fail("route_topk: unknown dtype %d", dtype);
    return tff_check_launch("route_topk");
}

// Experts by a table over the token ids instead of a router: idx[t, k] = table[ids[t], k], each with the weight
// 1 / top.  An id or an expert outside its range is brought into it (a launch never reads outside a table).
__global__ __launch_bounds__(256) void route_by_table_kernel(const int32_t* __restrict__ table, const int32_t* __restrict__ ids,
                                                             int pairs, int V, int top, int E, int32_t* __restrict__ idx,
                                                             float* __restrict__ wts) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= pairs) return;
    const int t = p / top, k = p - t * top;
    const int id = min(max(ids[t], 0), V - 1);
    idx[p] = min(max(table[(size_t)id * top + k], 0), E - 1);
    wts[p] = 1.0f / (float)top;
}

TFF_API int tff_route_by_table(const int32_t* table, const int32_t* ids, int T, int V, int top, int E, int32_t* idx,
                               float* wts, tff_stream_t stream) {
    TFF_REQUIRE(table && ids && idx && wts, "route_by_table: null pointer");
    TFF_REQUIRE(T >= 0 && V > 0 && top > 0 && E > 0, "route_by_table: bad sizes T=%d V=%d top=%d E=%d", T, V, top, E);
    if (T == 0) return 0;
    route_by_table_kernel<<<(T * top + 255) / 256, 256, 0, (hipStream_t)stream>>>(table, ids, T * top, V, top, E, idx, wts);
    return tff_check_launch("route_by_table");
}

#define EX_WAVES 4
#define EX_PER_WAVE 4      // outputs a wave works through
// Few pairs leave the SIMDs with a wave or two: then a wave takes half as many gated outputs, and a token's experts are dealt to waves of their own
// (experts_down_shared_kernel).  us, one token, four experts of 4,096 x 1,536 19.1 + 12.7 / 17.5 + 10.6, two of 2,048 x 1,024 6.6 + 5.4 / 5.3 + 4.7,
// two tokens of the latter 8.0 + 6.2 / 7.2 + 5.6; three tokens of the former 48.2 + 24.7 / 45.4 + 26.4, four 61.7 + 31.8 / 61.1 + 34.0.
#define EX_FEW_OUTPUTS 18432      // gated outputs up to which it is so
#define EX_FEW_DOWN 4096          // results

// What bounds a step of one token is how many loads are in flight: a wave asks for two pieces of four weight rows at a time (two
// outputs' gate and up rows, or four outputs' down rows).  A row after the other on waves of eight outputs, one token of four
// experts of 4,096 x 1,536 took 74 + 64 us, now 21 + 14 (4.8 and 3.7 TB/s); eight tokens 117 + 83, now 112 + 60.  Longer
// pieces (four loads of each row) or eight outputs a wave: 5 to 60 % slower at one token, within 3 % at eight.
template <typename T>
__global__ __launch_bounds__(64 * EX_WAVES) void experts_gate_up_kernel(
    const T* __restrict__ h, int h_row, const T* __restrict__ Wg, const T* __restrict__ Wu,
    const int32_t* __restrict__ idx, int top, int width, int ff, int ldw, float limit, float act_alpha, float up_offset,
    const float* __restrict__ in_wts, T* __restrict__ y, int E, int per_wave) {
    // Wg null: experts without a gate, y = max(Wu h, 0)^2.  in_wts: the pair's weight multiplies what goes into the
    // expert, W (w h) = w (W h): both products times w before clamps and activation.
    const int pair = blockIdx.x;                  // token * top + k
    const int t = pair / top;
    const int e = idx[pair];
    if (e >= E) return;                           // (an expert without matrices)
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const T* hr = h + (size_t)t * h_row;
    const T* wg = Wg ? Wg + (size_t)e * ff * ldw : nullptr;
    const T* wu = Wu + (size_t)e * ff * ldw;
    const bool vec = sizeof(T) == 2 && width % 8 == 0 && ldw % 8 == 0 && h_row % 8 == 0 && ((uintptr_t)h % 16) == 0 &&
                     ((uintptr_t)Wg % 16) == 0 && ((uintptr_t)Wu % 16) == 0;
    const float win = in_wts ? in_wts[pair] : 1.0f;
    const int f0 = (blockIdx.y * EX_WAVES + wv) * per_wave, f1 = min(ff, f0 + per_wave);
    auto finish = [&](int f, float g, float u) {
        u *= win;
        if (!wg) {
            u = fmaxf(u, 0.f);
            y[(size_t)pair * ff + f] = from_f32<T>(u * u);
            return;
        }
        g = fminf(g * win, limit);
        u = fminf(fmaxf(u, -limit), limit);
        y[(size_t)pair * ff + f] = from_f32<T>(g * (1.0f / (1.0f + expf(-act_alpha * g))) * (u + up_offset));
    };
    if constexpr (sizeof(T) == 2) {
        if (vec) {
            if (wg) {
                for (int f = f0; f < f1; f += 2) {
                    const int g = min(f + 1, ff - 1);
                    const T* const rows[4] = {wg + (size_t)f * ldw, wg + (size_t)g * ldw, wu + (size_t)f * ldw, wu + (size_t)g * ldw};
                    float d[4];
                    wave_dots8<4, 2>(hr, rows, width, lane, d);
                    if (lane == 0) {
                        finish(f, d[0], d[2]);
                        if (f + 1 < f1) finish(f + 1, d[1], d[3]);
                    }
                }
            } else {
                for (int f = f0; f < f1; f += 4) {
                    const T* const rows[4] = {wu + (size_t)f * ldw, wu + (size_t)min(f + 1, ff - 1) * ldw,
                                              wu + (size_t)min(f + 2, ff - 1) * ldw, wu + (size_t)min(f + 3, ff - 1) * ldw};
                    float d[4];
                    wave_dots8<4, 2>(hr, rows, width, lane, d);
                    if (lane == 0) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (f + i < f1) finish(f + i, 0.f, d[i]);
                    }
                }
            }
            return;
        }
    }
    for (int f = f0; f < f1; ++f) {
        const float u = wave_dot(hr, wu + (size_t)f * ldw, width, lane);
        const float g = wg ? wave_dot(hr, wg + (size_t)f * ldw, width, lane) : 0.f;
        if (lane == 0) finish(f, g, u);
    }
}

template <typename T>
__global__ __launch_bounds__(64 * EX_WAVES) void experts_down_kernel(
    const T* __restrict__ y, const T* __restrict__ Wd, const int32_t* __restrict__ idx, const float* __restrict__ wts,
    int top, int width, int ff, int ldw, float* __restrict__ out, int E, const T* __restrict__ h, int h_row) {
    const int t = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool vec = sizeof(T) == 2 && ff % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)Wd % 16) == 0;
    const int n0 = (blockIdx.y * EX_WAVES + wv) * EX_PER_WAVE, n1 = min(width, n0 + EX_PER_WAVE);
    for (int n = n0; n < n1; n += 4) {
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < top; ++k) {
            const int e = idx[(size_t)t * top + k];
            const float w = wts ? wts[(size_t)t * top + k] : 1.0f;
            const T* yr = y + ((size_t)t * top + k) * ff;
            float d[4];
            if (e >= E) {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[i] = to_f32(h[(size_t)t * h_row + min(n + i, width - 1)]);
            } else {
                const T* const wd = Wd + (size_t)e * width * ldw;
                const T* const rows[4] = {wd + (size_t)n * ldw, wd + (size_t)min(n + 1, width - 1) * ldw,
                                          wd + (size_t)min(n + 2, width - 1) * ldw, wd + (size_t)min(n + 3, width - 1) * ldw};
                bool done = false;
                if constexpr (sizeof(T) == 2) {
                    if (vec) {
                        wave_dots8<4, 2>(yr, rows, ff, lane, d);
                        done = true;
                    }
                }
                if (!done) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) d[i] = wave_dot(yr, rows[i], ff, lane);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = fmaf(w, d[i], acc[i]);
        }
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (n + i < n1) out[(size_t)t * width + n + i] = acc[i];
        }
    }
}

// The same with a wave for every expert of a token: SHARE waves take the experts of the same four outputs in turn, and the first of them adds
// their sums up, in the order of k as above.
template <int SHARE>
__global__ __launch_bounds__(64 * EX_WAVES * SHARE) void experts_down_shared_kernel(
    const bf16_t* __restrict__ y, const bf16_t* __restrict__ Wd, const int32_t* __restrict__ idx, const float* __restrict__ wts,
    int top, int width, int ff, int ldw, float* __restrict__ out, int E, const bf16_t* __restrict__ h, int h_row) {
    __shared__ float4 sums[SHARE][EX_WAVES];
    __shared__ float weights[SHARE][EX_WAVES];
    const int t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = wave % EX_WAVES, share = wave / EX_WAVES;
    const int n = (blockIdx.y * EX_WAVES + g) * 4;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < top; k0 += SHARE) {
        const int k = k0 + share;
        if (k < top && n < width) {
            const int e = idx[(size_t)t * top + k];
            const float w = wts ? wts[(size_t)t * top + k] : 1.0f;
            float d[4];
            if (e >= E) {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[i] = to_f32(h[(size_t)t * h_row + min(n + i, width - 1)]);
            } else {
                const bf16_t* const wd = Wd + (size_t)e * width * ldw;
                const bf16_t* const rows[4] = {wd + (size_t)n * ldw, wd + (size_t)min(n + 1, width - 1) * ldw,
                                               wd + (size_t)min(n + 2, width - 1) * ldw, wd + (size_t)min(n + 3, width - 1) * ldw};
                wave_dots8<4, 2>(y + ((size_t)t * top + k) * ff, rows, ff, lane, d);
            }
            if (lane == 0) {
                sums[share][g] = make_float4(d[0], d[1], d[2], d[3]);
                weights[share][g] = w;
            }
        }
        __syncthreads();
        if (share == 0) {
            const int here = min(SHARE, top - k0);
#pragma unroll
            for (int s = 0; s < SHARE; ++s)
                if (s < here) {
                    const float4 d = sums[s][g];
                    const float w = weights[s][g];
                    acc[0] = fmaf(w, d.x, acc[0]), acc[1] = fmaf(w, d.y, acc[1]);
                    acc[2] = fmaf(w, d.z, acc[2]), acc[3] = fmaf(w, d.w, acc[3]);
                }
        }
        if (k0 + SHARE < top) __syncthreads();
    }
    if (share == 0 && lane == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n + i < width) out[(size_t)t * width + n + i] = acc[i];
    }
}

TFF_API int tff_experts_gate_up(const void* h, int h_row, const void* Wg, const void* Wu, const int32_t* idx, int T,
                                int top, int E, int width, int ff, int ldw, float limit, float act_alpha, float up_offset,
                                const float* in_wts, void* y,
                                int dtype, tff_stream_t stream) {
    TFF_REQUIRE(h && Wu && idx && y, "experts_gate_up: null pointer");
    TFF_REQUIRE(T >= 0 && top > 0 && E > 0 && width > 0 && ff > 0 && h_row >= width && ldw >= width,
                "experts_gate_up: bad sizes T=%d top=%d width=%d ff=%d", T, top, width, ff);
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int per_wave = Wg && (long)T * top * ff <= EX_FEW_OUTPUTS ? EX_PER_WAVE / 2 : EX_PER_WAVE;
    const dim3 grid(T * top, (ff + EX_WAVES * per_wave - 1) / (EX_WAVES * per_wave));
    TFF_REQUIRE(grid.y <= 65535, "experts_gate_up: too many outputs");
    if (dtype == TFF_F32)
        experts_gate_up_kernel<float><<<grid, 64 * EX_WAVES, 0, s>>>((const float*)h, h_row, (const float*)Wg, (const float*)Wu,
                                                                    idx, top, width, ff, ldw, limit, act_alpha, up_offset, in_wts, (float*)y, E, per_wave);
    else if (dtype == TFF_BF16)
        experts_gate_up_kernel<bf16_t><<<grid, 64 * EX_WAVES, 0, s>>>((const bf16_t*)h, h_row, (const bf16_t*)Wg,
                                                                     (const bf16_t*)Wu, idx, top, width, ff, ldw, limit,
                                                                     act_alpha, up_offset, in_wts, (bf16_t*)y, E, per_wave);
    else
        return tff_fail("experts_gate_up: unknown dtype %d", dtype);
    return tff_check_launch("experts_gate_up");
}

// h [T, width], rows h_row apart (may be null where every expert has matrices): what experts from number E on hand on.
TFF_API int tff_experts_down(const void* y, const void* Wd, const int32_t* idx, const float* wts, int T, int top, int E,
                             int width, int ff, int ldw, const void* h, int h_row, int identity, float* out, int dtype,
                             tff_stream_t stream) {
    TFF_REQUIRE(y && Wd && idx && out, "experts_down: null pointer");      // (wts null: every pair counts 1)
    TFF_REQUIRE(identity == 0 || (h && h_row >= width), "experts_down: experts without matrices need the rows they hand on");
    TFF_REQUIRE(T >= 0 && top > 0 && E > 0 && width > 0 && ff > 0 && ldw >= ff, "experts_down: bad sizes T=%d top=%d width=%d ff=%d",
                T, top, width, ff);
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(T, (width + EX_WAVES * EX_PER_WAVE - 1) / (EX_WAVES * EX_PER_WAVE));
    TFF_REQUIRE(grid.y <= 65535, "experts_down: too many outputs");
    if (dtype == TFF_F32)
        experts_down_kernel<float><<<grid, 64 * EX_WAVES, 0, s>>>((const float*)y, (const float*)Wd, idx, wts, top, width, ff, ldw, out, E, (const float*)h, h_row);
    else if (dtype == TFF_BF16 && top > 1 && (long)T * width <= EX_FEW_DOWN && ff % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)Wd % 16) == 0) {
        if (top > 2)
            experts_down_shared_kernel<4><<<grid, 64 * EX_WAVES * 4, 0, s>>>((const bf16_t*)y, (const bf16_t*)Wd, idx, wts, top, width, ff, ldw, out, E, (const bf16_t*)h, h_row);
        else
            experts_down_shared_kernel<2><<<grid, 64 * EX_WAVES * 2, 0, s>>>((const bf16_t*)y, (const bf16_t*)Wd, idx, wts, top, width, ff, ldw, out, E, (const bf16_t*)h, h_row);
    } else if (dtype == TFF_BF16)
        experts_down_kernel<bf16_t><<<grid, 64 * EX_WAVES, 0, s>>>((const bf16_t*)y, (const bf16_t*)Wd, idx, wts, top, width, ff, ldw, out, E, (const bf16_t*)h, h_row);
    else
        return tff_fail("experts_down: unknown dtype %d", dtype);
    return tff_check_launch("experts_down");
}

// ------------------------------------------------------------- many tokens: by expert ---
// With many tokens a step the (token, expert) pairs are dealt to their experts first: every
// expert's pairs fill tiles of `rows` pairs (64, or 128 where the experts have a few hundred pairs
// each; an expert's last tile is padded), so that a tile's rows share the expert's matrices and the
// products run on the matrix cores.  A pair's row is computed from the pair alone, k ascending,
// whatever tile and place it lands in: the result does not depend on what else the step holds, nor
// on the order the pairs were dealt in.
//
// experts_sort_kernel:  tile_expert[tile] = (expert, its first tile, how many tiles it has, 0), tile_rows[tile * rows + i] =
//                       pair (token * top + k) or -1, num_tiles[0]; one block.  At most pairs / rows + E tiles.
// experts_tiles_kernel: the two products per tile.  The down product writes
//                       out[k][t][:] = wts[t][k] * Wd y: `top` planes that the norm after the
//                       feed-forward adds up in the order of k.

__global__ __launch_bounds__(1024) void experts_sort_kernel(const int32_t* __restrict__ idx, int pairs, int E,
                                                            int rows, int4* __restrict__ tile_expert,
                                                            int32_t* __restrict__ tile_rows,
                                                            int32_t* __restrict__ num_tiles) {
    __shared__ int count[RT_MAX_E];
    __shared__ int first[RT_MAX_E + 1];     // an expert's first tile
    const int tid = threadIdx.x;
    for (int e = tid; e < E; e += blockDim.x) count[e] = 0;
    __syncthreads();
    for (int p = tid; p < pairs; p += blockDim.x)
        if (idx[p] < E) atomicAdd(&count[idx[p]], 1);       // (experts without matrices have no tiles)
    __syncthreads();
    if (tid == 0) {
        int t = 0;
        for (int e = 0; e < E; ++e) {
            first[e] = t;
            t += (count[e] + rows - 1) / rows;
        }
        first[E] = t;
        num_tiles[0] = t;
    }
    __syncthreads();
    const int tiles = first[E];
    for (int e = tid; e < E; e += blockDim.x) {
        for (int t = first[e]; t < first[e + 1]; ++t) tile_expert[t] = make_int4(e, first[e], first[e + 1] - first[e], 0);
        count[e] = 0;
    }
    for (int i = tid; i < tiles * rows; i += blockDim.x) tile_rows[i] = -1;
    __syncthreads();
    for (int p = tid; p < pairs; p += blockDim.x) {
        const int e = idx[p];
        if (e >= E) continue;
        const int at = atomicAdd(&count[e], 1);
        tile_rows[first[e] * rows + at] = p;
    }
}

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 ex_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ex_floatx4;

__device__ __forceinline__ ex_bf16x8 ex_load8(const bf16_t* p, bool ok) {
    union { uint4 u; ex_bf16x8 v; } x;
    x.u = ok ? *reinterpret_cast<const uint4*>(p) : make_uint4(0, 0, 0, 0);
    return x.v;
}

// One kernel for both products.  Block: one tile of 64 or 128 pairs x 128 weight rows, four waves side by
// side, each all pairs x 32 weight rows (eight or sixteen accumulators).  GATE_UP: a wave's 32 weight rows
// are 16 outputs of the gate and the same 16 of the up projection; else 32 outputs of the down
// projection.  K goes in steps of 64.  The pairs' rows, which all four waves need, pass through LDS
// (global -> registers while the step before is computed, then registers -> LDS; a fragment of 16
// rows x 32 k lies there as a wave reads it, lane l's eight elements at l * 16 bytes); a wave's own
// weight rows go straight from memory into its MFMA operands, one step ahead: LDS bandwidth is what
// bounds a block of few waves, and the weight is two thirds of the operands.
// C[w][pair] += W[w][k] a[pair][k]: lane (pair = lane & 15, kg = lane >> 4) ends up with weight rows
// kg * 4 .. + 3 of its pair.  k ascends for every pair alike, whatever tile and place the pair was
// dealt to.
#define EXT_KSTEP 64

// What a block of the experts' products works on.  Blocks go to the eight XCDs in turn by their number, each XCD with an L2 of its own;
// of the (tile, column block) pairs in order each XCD takes an eighth, so that none is without work.  The order is an expert after the
// other, of an expert EX_GROUP tiles at a time, of these all column blocks, tiles fastest: the 32 blocks that an XCD runs at a time are
// then one or two experts' whole products, whose weight rows come from memory once for the group's tiles and whose pairs' rows meet in L2
// for the column blocks.  (A column block of all experts after the other, which stood here, shared the weight's rows as well but fetched
// the pairs' rows once more for every column block.  us for both products, so / now: 32 experts, four a token, 4,096 x 1,536 gated,
// 2,048 tokens 573 / 560, 4,000 tokens 852 / 817; 2,048 x 1,536, 4,500 tokens 519 / 494; 64 to 150 tokens within 1 %.)
// The pair's number in that order, or -1 for a block without one.
__host__ __device__ __forceinline__ int ex_block(unsigned block, int tiles, int col_blocks) {
    const int all = tiles * col_blocks, share = (all + 7) >> 3, at = (int)(block >> 3), id = (int)(block & 7) * share + at;
    return at < share && id < all ? id : -1;
}
#define EX_GROUP 8
// The tile and column block of pair `id`; `t` is the entry of tile id / col_blocks, which belongs to the same expert.
__host__ __device__ __forceinline__ void ex_place(int id, int col_blocks, int4 t, int& tile, int& col_block) {
    const int in = id - t.y * col_blocks, group = in / (EX_GROUP * col_blocks);
    const int rest = in - group * EX_GROUP * col_blocks, left = t.z - group * EX_GROUP, n = left < EX_GROUP ? left : EX_GROUP;
    col_block = rest / n;
    tile = t.y + group * EX_GROUP + rest - col_block * n;
}
// For tests: tile * col_blocks + column block of pair `id` of an expert whose `n` tiles begin at `first`.
TFF_API int tff_experts_place(int id, int col_blocks, int first, int n) {
    int4 t;
    t.x = 0; t.y = first; t.z = n; t.w = 0;
    int tile, col_block;
    ex_place(id, col_blocks, t, tile, col_block);
    return tile * col_blocks + col_block;
}
TFF_API int tff_experts_block(int block, int tiles, int col_blocks) { return ex_block((unsigned)block, tiles, col_blocks); }

// MODE 0: the down product; 1: gate and up; 2: up alone, y = max(Wu h, 0)^2 (a wave's 32 weight rows are 32 outputs).
template <int MODE, int AFR>
__global__ __launch_bounds__(256) void experts_tiles_kernel(
    const bf16_t* __restrict__ a_rows, int a_row, const bf16_t* __restrict__ W0, const bf16_t* __restrict__ W1,
    const int4* __restrict__ tile_expert, const int32_t* __restrict__ tile_rows,
    const int32_t* __restrict__ num_tiles, const float* __restrict__ wts, int T, int top, int K, int N,
    float limit, float act_alpha, float up_offset, bf16_t* __restrict__ y, float* __restrict__ out, int col_blocks,
    int ldw, int weight_input) {
    // weight_input: a pair's weight multiplies what goes into its expert (both first products, before clamps
    // and activation: W (w h) = w (W h)) and the second product counts 1
    constexpr bool GATE_UP = MODE == 1;
    constexpr int ROWS = AFR * 16;       // pairs of a tile: 64, or 128 where the experts have many pairs each
    __shared__ __attribute__((aligned(16))) bf16_t lds[2 * AFR * 512];      // two sub-steps of AFR fragments
    const int tiles = num_tiles[0], id = ex_block(blockIdx.x, tiles, col_blocks);
    if (id < 0) return;
    const int4 of = tile_expert[id / col_blocks];
    int tile, col_block;
    ex_place(id, col_blocks, of, tile, col_block);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = lane & 15, kg = lane >> 4;
    const int e = of.x;
    const int c0 = col_block * (GATE_UP ? 64 : 128) + wv * (GATE_UP ? 16 : 32);     // the wave's first output
    // the pairs' rows: 2 AFR fragments a step (AFR of 16 pairs, two sub-steps of 32 k), AFR / 2 a wave
    constexpr int AU = AFR / 2;
    const bf16_t* asrc[AU];
    bool aok[AU];
#pragma unroll
    for (int i = 0; i < AU; ++i) {
        const int fs = i * 4 + wv, sub = fs / AFR, frag = fs % AFR;
        const int pair = tile_rows[tile * ROWS + frag * 16 + r];
        aok[i] = pair >= 0;
        asrc[i] = a_rows + (size_t)(MODE != 0 ? max(pair, 0) / top : max(pair, 0)) * a_row + sub * 32 + kg * 8;
    }
    // the wave's weight rows: two fragments
    const bf16_t* wsrc[2];
    bool wok[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = GATE_UP ? c0 + r : c0 + j * 16 + r;
        wok[j] = n < N;
        wsrc[j] = ((GATE_UP && j == 1) ? W1 : W0) + ((size_t)e * N + min(n, N - 1)) * ldw + kg * 8;
    }
    ex_floatx4 acc[2][AFR];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < AFR; ++i) acc[j][i] = ex_floatx4{0.f, 0.f, 0.f, 0.f};
    uint4 areg[AU];
    ex_bf16x8 wreg[2][2];        // [sub][fragment] of the step that is fetched
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < AU; ++i) {
            const int sub = (i * 4 + wv) / AFR;
            const bool in = aok[i] && k0 + sub * 32 + kg * 8 < K;
            areg[i] = in ? *reinterpret_cast<const uint4*>(asrc[i] + k0) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int j = 0; j < 2; ++j) wreg[sub][j] = ex_load8(wsrc[j] + k0 + sub * 32, wok[j] && k0 + sub * 32 + kg * 8 < K);
    };
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += EXT_KSTEP) {
        __syncthreads();            // the step before is read
#pragma unroll
        for (int i = 0; i < AU; ++i) *reinterpret_cast<uint4*>(lds + (size_t)(i * 4 + wv) * 512 + lane * 8) = areg[i];
        ex_bf16x8 wnow[2][2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int j = 0; j < 2; ++j) wnow[sub][j] = wreg[sub][j];
        __syncthreads();
        if (k0 + EXT_KSTEP < K) fetch(k0 + EXT_KSTEP);      // travels while this step is computed
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            ex_bf16x8 av[AFR];
#pragma unroll
            for (int i = 0; i < AFR; ++i)
                av[i] = *reinterpret_cast<const ex_bf16x8*>(lds + (size_t)(sub * AFR + i) * 512 + lane * 8);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < AFR; ++i)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wnow[sub][j], av[i], acc[j][i], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < AFR; ++i) {
        const int pair = tile_rows[tile * ROWS + i * 16 + r];
        const float win = (MODE != 0 && weight_input && pair >= 0) ? wts[pair] : 1.0f;
        if (GATE_UP) {
            const float g4[4] = {acc[0][i][0], acc[0][i][1], acc[0][i][2], acc[0][i][3]};
            const float u4[4] = {acc[1][i][0], acc[1][i][1], acc[1][i][2], acc[1][i][3]};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int f = c0 + kg * 4 + c;
                if (pair >= 0 && f < N) {
                    const float gv = fminf(g4[c] * win, limit);
                    const float uv = fminf(fmaxf(u4[c] * win, -limit), limit);
                    y[(size_t)pair * N + f] = (bf16_t)(gv * (1.0f / (1.0f + expf(-act_alpha * gv))) * (uv + up_offset));
                }
            }
        } else if (MODE == 2) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float v4[4] = {acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int n = c0 + j * 16 + kg * 4 + c;
                    const float u = fmaxf(v4[c] * win, 0.f);
                    if (pair >= 0 && n < N) y[(size_t)pair * N + n] = (bf16_t)(u * u);
                }
            }
        } else {
            const int p = max(pair, 0), t = p / top, k = p - t * top;
            const float w = weight_input ? 1.0f : wts[p];
            float* o = out + ((size_t)k * T + t) * N;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float v4[4] = {acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int n = c0 + j * 16 + kg * 4 + c;
                    if (pair >= 0 && n < N) o[n] = w * v4[c];
                }
            }
        }
    }
}

// The same products for inner sizes in units of 64: both operands pass through LDS as whole cache lines, four waves, one to
// a SIMD, with the LDS reads of the next 32 k and the copies of later units between the MFMAs of the present ones.  Block:
// BM = 16 WTM WGM pairs x BN = 64 WTN / WGM weight rows.  What bounds the kernel above is the number of requests to L2 (operands as
// 64-byte pieces of rows, 64 flops a byte on its 128 x 128 tile) and the waits between its barriers, which nothing overlaps.
// Here a unit of 64 k is copied eight rows x 128 bytes at a time (lane i of a copy lands at byte 16 i and fetches row i / 8,
// chunk (i % 8) ^ (i / 8), so that an operand's sixteen rows come back from different banks), the pairs' rows through
// the tile's list; NS units lie in LDS, two are on their way.  GATE_UP: the tile's groups of 16 weight rows are gate
// and up in turn, so a lane holds both sums of its outputs.  k ascends in steps of 32 for every pair as above: the same bits.
// A unit's operands have all been read, and have arrived (lgkmcnt 0), before the barrier in the middle of its work, and at once the first half of
// the copies of the unit three behind it goes into its slot, the second half during the first half of the next unit's work.  At
// the barrier in the middle of unit u every wave's copies of unit u + 1 have landed: all but the CP that it issued since.  So a copy has from one
// unit's work to two to arrive in (with unit u + 2 copied during unit u, as it was, from a half to one and a half).  us a product of 32
// experts, 4,096 x 3,072, that / this: 256 pairs an expert 233 / 224, 300 330 / 296, 384 351 / 324; 8,192 pairs of one expert, whose rows the caches
// hold, 160 / 163.  The last unit's second half issues no copies (the results go through its slot) and stands behind the loop: with a choice
// between the two inside it, the compiler moved accumulators about right behind MFMAs whose wait states it does not know.
// A block that works on one pair of tile and column block spends 10 to 15 us of its 40 to 75 on what nothing overlaps: three loads that wait for
// each other, the first units on their way, the results' way out.  So the launch has a block a CU, and a block goes on to its next
// pair: that one's list of rows travels during the first units of the present pair, its first two units of operands during the
// last three, and the results leave through the third slot while they land.
// us for both products, a pair a block / now: 32 experts, four a token, 4,096 x 1,536 gated, 2,048 tokens 560 / 537 (576 TFLOP/s; some 720
// with the tiles' padding), 4,000 tokens 817 / 783; 4,096 x 3,072 without a gate, 2,919 tokens 776 / 739; 2,048 x 1,536 gated, 4,500 tokens
// 494 / 462; 16 experts, two a token, 2,048 x 1,024, 2,000 tokens 121 / 101; 150 tokens of the first within 2 % (the weight's stream).
#define EXL_CHAIN 5      // units of K from which a block may go on to another pair: its list is there before its first copies
template <int MODE, int WGM, int WTM, int WTN>
__global__ __launch_bounds__(256) void experts_lines_kernel(
    const bf16_t* __restrict__ a_rows, int a_row, const bf16_t* __restrict__ W0, const bf16_t* __restrict__ W1,
    const int4* __restrict__ tile_expert, const int32_t* __restrict__ tile_rows, const int32_t* __restrict__ num_tiles,
    const float* __restrict__ wts, int T, int top, int K, int N, float limit, float act_alpha, float up_offset,
    bf16_t* __restrict__ y, float* __restrict__ out, int col_blocks, int ldw, int weight_input) {
    constexpr int NW = 4, NS = 3, WGN = NW / WGM;
    constexpr int BM = WGM * WTM * 16, BN = WGN * WTN * 16;
    constexpr int LPA = BM / 8 / NW, LPW = BN / 8 / NW, CP = LPA + LPW;      // a wave's copies of a unit
    constexpr unsigned A_BYTES = BM * 128u, UNIT = (BM + BN) * 128u;
    constexpr int NMF = WTM * WTN, RPM = NMF / (WTM + WTN), CPM = NMF / (CP / 2);
    static_assert(RPM >= 1 && CPM >= 1 && CP % 2 == 0 && LPA >= 1, "the MFMAs of a k-tile hide its reads and copies");
    constexpr unsigned LIST = NS * UNIT;                // behind the units: each wave's lists of pairs, this tile's and the next one's
    static_assert(LIST + NW * 2048 <= 160 * 1024 && BM * 4 <= 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) char smem[LIST + NW * 2048];
    const int tiles = num_tiles[0];
    unsigned block = blockIdx.x;
    int id = ex_block(block, tiles, col_blocks);
    if (id < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = WGM == 2 ? wave >> 1 : 0, wn = WGM == 2 ? wave & 1 : wave;
    const int fr = lane & 15, fg = lane >> 4;
    int4 of = tile_expert[id / col_blocks];
    int tile, col_block;
    ex_place(id, col_blocks, of, tile, col_block);

    // what a wave copies of a unit: the pairs' rows, eight at a time, and the weight's
    const unsigned smem_addr = (unsigned)(size_t)(lds_ptr_t)smem;
    const unsigned chunk = (unsigned)(((lane & 7) ^ (lane >> 3)) * 16);
    unsigned off[CP];
    unsigned long long base[3];
    base[0] = (unsigned long long)a_rows;
    auto weight_rows = [&]() {
        base[1] = (unsigned long long)(W0 + (size_t)of.x * N * ldw);
        base[2] = MODE == 1 ? (unsigned long long)(W1 + (size_t)of.x * N * ldw) : base[1];
#pragma unroll
        for (int c = 0; c < LPW; ++c) {
            const int r0 = (wave + NW * c) * 8, grp = r0 >> 4, in = (r0 & 15) + (lane >> 3);
            const int n = col_block * (MODE == 1 ? BN / 2 : BN) + (MODE == 1 ? grp >> 1 : grp) * 16 + in;
            off[LPA + c] = (unsigned)min(n, N - 1) * (unsigned)ldw * 2u + chunk;
        }
    };
    auto pair_row = [&](int p) {     // (a place without a pair repeats pair 0, nobody reads it)
        p = max(p, 0);
        return (unsigned)(MODE != 0 ? p / top : p) * (unsigned)a_row * 2u + chunk;
    };
    // a tile's list into the wave's buffer `to`: the lanes past its end repeat it
    auto copy_list = [&](int of_tile, unsigned to) {
        copy16_to_lds_sbase((unsigned long long)(tile_rows + (size_t)of_tile * BM), (unsigned)(lane * 16) & (BM * 4 - 1),
                            smem_addr + LIST + (unsigned)wave * 2048u + to);
    };
    unsigned list = 0;                                // the present tile's list
#pragma unroll
    for (int c = 0; c < LPA; ++c) off[c] = pair_row(tile_rows[(size_t)tile * BM + (wave + NW * c) * 8 + (lane >> 3)]);
    weight_rows();
    copy_list(tile, list);
    const int nu = K >> 6;
    int u_next = 0;                                   // the unit to copy next
    unsigned long long k_off = 0;
    unsigned ws = 0;                                  // its slot
#define EXL_COPY(c)                                                                                                 \
    {                                                                                                               \
        const int which = (c) < LPA ? 0 : (MODE == 1 && (((wave + NW * ((c) - LPA)) >> 1) & 1)) ? 2 : 1;             \
        copy16_to_lds_sbase(base[which] + k_off, off[c],                                                            \
                            smem_addr + ws + ((c) < LPA ? 0u : A_BYTES) + (unsigned)(wave + NW * ((c) < LPA ? (c) : (c) - LPA)) * 1024u); \
    }
#define EXL_ISSUED()                                                                                                \
    {                                                                                                               \
        if (u_next + 1 < nu) { ++u_next; k_off += 128ull; }                                                         \
        ws = ws + UNIT == NS * UNIT ? 0u : ws + UNIT;                                                               \
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int c = 0; c < CP; ++c) EXL_COPY(c)
        EXL_ISSUED()                                  // (past the end of K the last unit once more)
    }
#pragma unroll
    for (int c = 0; c < CP / 2; ++c) EXL_COPY(c)
    // a lane's 16 bytes of an operand: row fr of 16, chunk h * 4 + fg of the row's 8
    unsigned rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) rd[h] = (unsigned)(fr >> 3) * 1024u + (unsigned)(((fr & 7) * 8 + ((h * 4 + fg) ^ (fr & 7))) * 16);
    const unsigned a_rd = (unsigned)(wm * WTM) * 2048u, w_rd = A_BYTES + (unsigned)(wn * WTN) * 2048u;
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(CP + CP / 2));
    __syncthreads();
    bf16x8 fw[2][WTN], fa[2][WTM];
#pragma unroll
    for (int i = 0; i < WTN; ++i) fw[0][i] = *reinterpret_cast<const bf16x8*>(smem + w_rd + rd[0] + i * 2048);
#pragma unroll
    for (int j = 0; j < WTM; ++j) fa[0][j] = *reinterpret_cast<const bf16x8*>(smem + a_rd + rd[0] + j * 2048);
    unsigned rs = 0;                                  // the slot that the next operands are read from
#define EXL_TILE(h, COPIES)                                                                                         \
    {                                                                                                               \
        if (h) {                                                                                                    \
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                                      \
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(CP));                                                              \
            asm volatile("s_barrier" ::: "memory");                                                                 \
            rs = rs + UNIT == NS * UNIT ? 0u : rs + UNIT;                                                           \
        }                                                                                                           \
        const char* na = smem + rs + a_rd + rd[(h) ^ 1];                                                            \
        const char* nw = smem + rs + w_rd + rd[(h) ^ 1];                                                            \
        _Pragma("unroll") for (int i = 0; i < WTN; ++i)                                                             \
            _Pragma("unroll") for (int j = 0; j < WTM; ++j) {                                                       \
                const int q = i * WTM + j;                                                                          \
                mfma_acc(acc[i][j], fw[h][i], fa[h][j]);                                                            \
                if (q % RPM == RPM - 1 && q / RPM < WTN + WTM) {                                                    \
                    const int x = q / RPM;                                                                          \
                    if (x < WTM) fa[(h) ^ 1][x < WTM ? x : 0] = *reinterpret_cast<const bf16x8*>(na + x * 2048);    \
                    else fw[(h) ^ 1][x >= WTM ? x - WTM : 0] = *reinterpret_cast<const bf16x8*>(nw + (x - WTM) * 2048); \
                }                                                                                                   \
                if ((COPIES) && q % CPM == CPM - 1 && q / CPM < CP / 2) EXL_COPY(((h) ^ 1) * (CP / 2) + q / CPM)     \
            }                                                                                                       \
    }
    floatx4 acc[WTN][WTM];
    for (;;) {
        const int c0 = col_block * (MODE == 1 ? BN / 2 : BN);           // the pair's first output
        block += gridDim.x;
        const int next = nu >= EXL_CHAIN ? ex_block(block, tiles, col_blocks) : -1;
        if (next >= 0) {
            of = tile_expert[next / col_blocks];
            ex_place(next, col_blocks, of, tile, col_block);
        }
#pragma unroll
        for (int i = 0; i < WTN; ++i)
#pragma unroll
            for (int j = 0; j < WTM; ++j) {
                acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                asm volatile("" : "+a"(acc[i][j]));
            }
        asm volatile("s_nop 7");
        EXL_TILE(0, true)
        EXL_ISSUED()
        if (next >= 0) copy_list(tile, list ^ 1024u);                  // here since the barrier of unit 1
        for (int u = 1; u < nu; ++u) {
            EXL_TILE(1, true)
            EXL_TILE(0, true)
            EXL_ISSUED()
            if (next >= 0 && u == nu - 3) {                             // the coming copies are the next pair's
                const int32_t* in_list = reinterpret_cast<const int32_t*>(smem + LIST + wave * 2048 + (list ^ 1024u));
#pragma unroll
                for (int c = 0; c < LPA; ++c) off[c] = pair_row(in_list[(wave + NW * c) * 8 + (lane >> 3)]);
                weight_rows();
                u_next = 0;
                k_off = 0;
            }
        }
        EXL_TILE(1, false)                                              // (the results go through the last unit's slot)
        // The last MFMAs have written.  The unit that was worked on last has left its slot (its last operands had arrived before the barrier in
        // its middle), and the next pair's first two units are in the other two or on their way: the results go through that slot, a
        // part of it for each wave, so that its stores are whole pieces of a pair's row.
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        typedef typename std::conditional<MODE == 0, float, bf16_t>::type TO;
        constexpr int OW = MODE == 1 ? WTN / 2 : WTN, EL = 16 / (int)sizeof(TO);
        constexpr int RB = OW * 16 * (int)sizeof(TO), RBP = RB + 16, LPR = RB / 16, RPI = 64 / LPR;
        constexpr int REGION = (int)(UNIT / NW) & ~1023;
        constexpr int JS = WTM * 16 * RBP <= REGION ? WTM : WTM / 2 * 16 * RBP <= REGION ? WTM / 2 : 1;      // groups of 16 pairs at a time
        static_assert(JS * 16 * RBP <= REGION && WTM % JS == 0 && LPR <= 64 && (LPR & (LPR - 1)) == 0 && 16 % RPI == 0, "the wave's part holds its results");
        char* region = smem + ws + wave * REGION;
        const int32_t* pairs = reinterpret_cast<const int32_t*>(smem + LIST + wave * 2048 + list) + wm * WTM * 16;
        const int ln = w4_lane(), r = ln & 15, g = ln >> 4;
        const int srow = ln / LPR, sch = ln % LPR, n = c0 + wn * OW * 16 + sch * EL;
#pragma unroll
        for (int j0 = 0; j0 < WTM; j0 += JS) {
#pragma unroll
            for (int j = j0; j < j0 + JS; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                float w = 1.0f;
                if (MODE == 0 ? !weight_input : weight_input != 0) {
                    const int p = pairs[j * 16 + r];
                    w = p >= 0 ? wts[p] : 0.f;
                }
#pragma unroll
                for (int i = 0; i < OW; ++i) {
                    char* dst = region + ((j - j0) * 16 + r) * RBP + (i * 16 + g * 4) * (int)sizeof(TO);
                    float v[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if constexpr (MODE == 1) {
                            const float gv = fminf(acc[2 * i][j][c] * w, limit);
                            const float uv = fminf(fmaxf(acc[2 * i + 1][j][c] * w, -limit), limit);
                            v[c] = gv * (1.0f / (1.0f + expf(-act_alpha * gv))) * (uv + up_offset);
                        } else if constexpr (MODE == 2) {
                            const float u = fmaxf(acc[i][j][c] * w, 0.f);
                            v[c] = u * u;
                        } else {
                            v[c] = w * acc[i][j][c];
                        }
                    }
                    if constexpr (sizeof(TO) == 4) {
                        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                    } else {
                        union { bf16_t h[4]; uint2 u; } pk;
#pragma unroll
                        for (int c = 0; c < 4; ++c) pk.h[c] = (bf16_t)v[c];
                        *reinterpret_cast<uint2*>(dst) = pk.u;
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (other lanes' results, as another type)
#pragma unroll 4
            for (int t = 0; t < JS * 16 / RPI; ++t) {
                const int row = t * RPI + srow, p = pairs[j0 * 16 + row];
                const uint4 v = *reinterpret_cast<const uint4*>(region + row * RBP + sch * 16);
                if (p < 0 || n >= N) continue;                // (N is a multiple of 8: a piece is whole or not there)
                if constexpr (MODE == 0) *reinterpret_cast<uint4*>(out + ((size_t)(p % top) * T + p / top) * N + n) = v;
                else *reinterpret_cast<uint4*>(y + (size_t)p * N + n) = v;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        if (next < 0) break;
        asm volatile("s_barrier" ::: "memory");       // every wave has left the slot: the next unit's copies go there
        list ^= 1024u;
#pragma unroll
        for (int c = 0; c < CP / 2; ++c) EXL_COPY(c)
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));         // the copies past the end must not outlive the block
#undef EXL_TILE
#undef EXL_COPY
#undef EXL_ISSUED
}

// The planes of the pairs whose expert has no matrices: out[k][t][:] = wts[t][k] * h[t][:].
__global__ __launch_bounds__(256) void experts_identity_kernel(const bf16_t* __restrict__ h, int h_row,
                                                               const int32_t* __restrict__ idx, const float* __restrict__ wts,
                                                               int T, int top, int E, int width, float* __restrict__ out) {
    const int p = blockIdx.x;
    if (idx[p] < E) return;
    const int t = p / top, k = p - t * top;
    const float w = wts[p];
    float* o = out + ((size_t)k * T + t) * width;
    for (int e = threadIdx.x * 4; e < width; e += 1024) {       // (width is a multiple of 8 here)
        union { uint2 u; bf16_t b[4]; } x;
        x.u = *reinterpret_cast<const uint2*>(h + (size_t)t * h_row + e);
        *reinterpret_cast<float4*>(o + e) = make_float4(w * (float)x.b[0], w * (float)x.b[1], w * (float)x.b[2], w * (float)x.b[3]);
    }
}

TFF_API int tff_experts_tiles_supported(int width, int ff, int h_row) {
    return width % 8 == 0 && ff % 8 == 0 && h_row % 8 == 0;
}

// h [T, width] bfloat16; workspace: tile_expert [max_tiles * 4] (16-byte aligned), tile_rows [max_tiles * 128], num_tiles [1] (int32),
// y [T * top, ff] bfloat16; out float32 [top, T, width].  max_tiles >= T * top / 64 + E.
TFF_API int tff_experts_by_tiles(const void* h, int h_row, const void* Wg, const void* Wu, const void* Wd,
                                 const int32_t* idx, const float* wts, int T, int top, int E, int width, int ff,
                                 int ldw_in, int ldw_down, float limit, float act_alpha, float up_offset, int32_t* tile_expert,
                                 int32_t* tile_rows, int32_t* num_tiles, int max_tiles, void* y, float* out,
                                 int weight_input, int identity, tff_stream_t stream) {
    TFF_REQUIRE(h && Wu && Wd && idx && wts && tile_expert && tile_rows && num_tiles && y && out,
                "experts_by_tiles: null pointer");
    TFF_REQUIRE(T >= 0 && top > 0 && E > 0 && E <= RT_MAX_E && width > 0 && ff > 0 && h_row >= width,
                "experts_by_tiles: bad sizes T=%d top=%d E=%d width=%d ff=%d", T, top, E, width, ff);
    TFF_REQUIRE(tff_experts_tiles_supported(width, ff, h_row) && ldw_in % 8 == 0 && ldw_down % 8 == 0 && ldw_in >= width &&
                ldw_down >= ff, "experts_by_tiles: width %d, ff %d, rows of %d and the weights' rows of %d and %d must be "
                "multiples of 8", width, ff, h_row, ldw_in, ldw_down);
    TFF_REQUIRE(((uintptr_t)h % 16) == 0 && ((uintptr_t)Wg % 16) == 0 && ((uintptr_t)Wu % 16) == 0 &&
                ((uintptr_t)Wd % 16) == 0 && ((uintptr_t)y % 16) == 0 && ((uintptr_t)tile_expert % 16) == 0 && ((uintptr_t)tile_rows % 16) == 0,
                "experts_by_tiles: operands must be 16-byte aligned");
    TFF_REQUIRE((long)T * top < (1L << 31) && max_tiles <= (1 << 20) && max_tiles >= (long)T * top / 64 + E,
                "experts_by_tiles: %d tiles do not hold %d x %d pairs of %d experts", max_tiles, T, top, E);
    // Inner sizes in units of 64 run on whole cache lines, the others on 64-byte pieces.  (A lane's offset into the rows is 32 bits.)
    const size_t limit32 = (size_t)1 << 32;
    const bool h_near = (size_t)T * h_row * 2 < limit32, y_near = (size_t)T * top * ff * 2 < limit32;
    const bool lines_up = width % 64 == 0 && h_near && (size_t)ff * ldw_in * 2 < limit32;
    const bool lines_down = ff % 64 == 0 && y_near && (size_t)width * ldw_down * 2 < limit32;
    // Tiles of 128 or of 64 pairs.  On 64-byte pieces: 128 where an expert has a few hundred pairs on average (every weight element
    // fetched serves twice the flops; the padding of an expert's last tile costs more with fewer).  On whole lines a block is
    // alone on its CU and a tile of 128 takes some 1.12 times as long as one of 64 (up to there both are their weight's stream), so
    // what counts is how often the blocks go round the CUs.  us, 64 / 128: 32 experts, four a token, 4,096 x 1,536, 150 tokens 244 / 265,
    // 512 tokens 318 / 288, 1,000 tokens 413 / 376; 16 experts, two a token, 2,048 x 1,024, 700 tokens 68 / 80, 1,000 tokens 114 / 83.
    const int cus = tff_device_cus();
    bool tall = (long)T * top >= 192L * E;
    if (lines_up && lines_down) {
        const double n = (double)T * top / E;
        const int cb_up = (ff + (Wg ? 127 : 255)) / (Wg ? 128 : 256), cb_down = (width + 255) / 256;
        double cost[2];
        for (int i = 0; i < 2; ++i) {
            const double tiles = E * fmax(1.0, n / (64 << i) + 0.5);      // (half of an expert's last tile is padding on average)
            cost[i] = ceil(tiles * cb_up / cus) * width + ceil(tiles * cb_down / cus) * ff;
        }
        tall = cost[1] * 1.12 < cost[0];
    }
    const int rows = tall ? 128 : 64;
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (identity > 0) {
        experts_identity_kernel<<<T * top, 256, 0, s>>>((const bf16_t*)h, h_row, idx, wts, T, top, E, width, out);
        if (int rc0 = tff_check_launch("experts_identity")) return rc0;
    }
    experts_sort_kernel<<<1, 1024, 0, s>>>(idx, T * top, E, rows, (int4*)tile_expert, tile_rows, num_tiles);
    int rc = tff_check_launch("experts_sort");
    if (rc) return rc;
    const int up_mode = Wg ? 1 : 2;
    const bf16_t *w0 = (const bf16_t*)(Wg ? Wg : Wu), *w1 = (const bf16_t*)(Wg ? Wu : nullptr);
#define EX_ARGS_UP (const bf16_t*)h, h_row, w0, w1, (const int4*)tile_expert, tile_rows, num_tiles, wts, T, top, width, ff, limit, act_alpha, \
                   up_offset, (bf16_t*)y, nullptr, cb, ldw_in, weight_input
#define EX_ARGS_DOWN (const bf16_t*)y, ff, (const bf16_t*)Wd, nullptr, (const int4*)tile_expert, tile_rows, num_tiles, wts, T, top, ff, width, limit, \
                     act_alpha, up_offset, nullptr, out, cb, ldw_down, weight_input
#define EX_GRID (unsigned)(((long)cb * max_tiles + 7) / 8 * 8)
// (one block a CU, which goes on from pair to pair; each pair a block of its own where K has too few units for that)
#define EXL_GRID(MODE) (((MODE) == 0 ? ff : width) / 64 < EXL_CHAIN ? EX_GRID : EX_GRID < most ? EX_GRID : most)
#define EX_LINES(MODE, ...)                                                                                \
    do {                                                                                                   \
        if (tall) experts_lines_kernel<MODE, 2, 4, 8><<<EXL_GRID(MODE), 256, 0, s>>>(__VA_ARGS__);         \
        else experts_lines_kernel<MODE, 1, 4, 4><<<EXL_GRID(MODE), 256, 0, s>>>(__VA_ARGS__);              \
    } while (0)
#define EX_TILES(MODE, ...)                                                                                \
    do {                                                                                                   \
        if (tall) experts_tiles_kernel<MODE, 8><<<EX_GRID, 256, 0, s>>>(__VA_ARGS__);                      \
        else experts_tiles_kernel<MODE, 4><<<EX_GRID, 256, 0, s>>>(__VA_ARGS__);                           \
    } while (0)
    const unsigned most = (unsigned)(cus < 8 ? 8 : cus / 8 * 8);      // (a multiple of the XCDs, which the blocks' numbering deals them to)
    {
        const int out_cols = (lines_up ? 256 : 128) / (Wg ? 2 : 1), cb = (ff + out_cols - 1) / out_cols;
        if (lines_up && up_mode == 1) EX_LINES(1, EX_ARGS_UP);
        else if (lines_up) EX_LINES(2, EX_ARGS_UP);
        else if (up_mode == 1) EX_TILES(1, EX_ARGS_UP);
        else EX_TILES(2, EX_ARGS_UP);
        rc = tff_check_launch("experts_gate_up_tiles");
        if (rc) return rc;
    }
    const int cb = (width + (lines_down ? 255 : 127)) / (lines_down ? 256 : 128);
    if (lines_down) EX_LINES(0, EX_ARGS_DOWN);
    else EX_TILES(0, EX_ARGS_DOWN);
#undef EX_ARGS_UP
#undef EX_ARGS_DOWN
#undef EX_GRID
#undef EXL_GRID
#undef EX_LINES
#undef EX_TILES
    return tff_check_launch("experts_down_tiles");
}
