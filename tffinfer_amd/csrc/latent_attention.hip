// Latent attention: what stands around the paged attention kernels when keys and values are
// kept as one low-rank latent vector per token.
//
// Per token the cache holds c (kv_rank elements, RMS-normed) and one rotated key part kr
// (rot elements) that all heads share.  With the up-projections taken to the query's side,
//   score_h(i, j) = (Wuk_h^T q_h^nope)(i) . c(j) + q_h^rot(i) . kr(j)
//   out_h(i)      = Wuv_h (sum_j p_h(i, j) c(j))
// the attention itself is attention with ONE key head of size kv_rank + rot whose values are
// the first kv_rank elements of its keys, which the paged kernels of this library run as they
// are: a key page row is [c | kr | 0 ..] up to the padded head size Dp, the (transposed) value
// page holds c in its first kv_rank rows and zeros below.
//
// tff_latent_kv_store:  c = rmsnorm(x[:rank]) * w, kr = rotate(x[rank:]) into the token's slot; where the
//                       queries pass a latent vector too, its RMS norm in the same launch.
// tff_head_linear:      out[t, h, :N] = W[h] x[t, h, :K]  (W [H, N, K]), per head, with
//                       an optional sigmoid gate on the result and an optional tail of the
//                       input row that is rotated by the token's position (either pairing) and copied behind
//                       the product (the query's rotated part), zeros up to pad_to.
//                       bfloat16 on the matrix cores where rows are 16-byte aligned.
#include "mfma_tiles.h"
#include "tffinfer_kernels.h"

// Element e of the rotated part (rot elements at x, the first rot_dims of them rotated) after the rotation
// by the position's angles cs [pair][cos, sin]: pairing 0 turns (i, i + rot_dims / 2), 1 turns (2i, 2i + 1);
// the pair (u, w) becomes (u c - w s, w c + u s).
template <typename T>
__device__ __forceinline__ float latent_rotated(const T* __restrict__ x, int e, int rot_dims, int pairing,
                                                const float* __restrict__ cs) {
    const float v = to_f32(x[e]);
    if (!cs || e >= rot_dims) return v;
    int i, other;
    bool first;
    if (pairing == 0) {
        const int half = rot_dims >> 1;
        first = e < half;
        i = first ? e : e - half;
        other = first ? e + half : e - half;
    } else {
        first = !(e & 1);
        i = e >> 1;
        other = e ^ 1;
    }
    const float o = to_f32(x[other]), c = cs[2 * i], s = cs[2 * i + 1];
    return first ? fmaf(v, c, -(o * s)) : fmaf(v, c, o * s);
}

// A token's key side: x's latent part normed and its rotated part into the token's slot; by all threads of the block.
template <typename T, typename TC>
__device__ __forceinline__ void latent_store_token(const T* __restrict__ xr, int t, int rank, int rot, int rot_dims, int pairing,
                                                   const float* __restrict__ norm_w, float eps, const float* __restrict__ cos_sin, int max_pos,
                                                   const int32_t* __restrict__ positions, int slot, TC* __restrict__ k_cache,
                                                   TC* __restrict__ v_cache, int page_size, int Dp, float* red) {
    const int tid = threadIdx.x;
    float ss = 0.f;
    for (int e = tid; e < rank; e += blockDim.x) {
        const float v = to_f32(xr[e]);
        ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, red);
    const float rr = 1.0f / sqrtf(ss / (float)rank + eps);
    const int page = slot / page_size, off = slot - page * page_size;
    TC* kr = k_cache + ((size_t)page * page_size + off) * Dp;
    TC* vr = v_cache + (size_t)page * Dp * page_size + off;
    for (int e = tid; e < rank; e += blockDim.x) {
        const TC c = from_f32<TC>(to_f32(xr[e]) * rr * norm_w[e]);
        kr[e] = c;
        vr[(size_t)e * page_size] = c;
    }
    int pos = positions[t];
    pos = min(max(pos, 0), max_pos - 1);
    const float* cs = cos_sin ? cos_sin + (size_t)pos * rot_dims : nullptr;   // [pair][cos, sin]
    for (int e = tid; e < Dp - rank; e += blockDim.x)
        kr[rank + e] = from_f32<TC>(e < rot ? latent_rotated<T>(xr + rank, e, rot_dims, pairing, cs) : 0.f);
}

// One block a token.  xq (may be null): the query's latent vector, q_rank elements, whose RMS norm times
// q_norm_w goes to q_out.  x (may be null: a layer that reads another layer's cache): the key side.
template <typename T, typename TC>
__global__ __launch_bounds__(256) void latent_kv_store_kernel(
    const T* __restrict__ x, int x_stride, int rank, int rot, int rot_dims, int pairing,
    const float* __restrict__ norm_w, float eps, const float* __restrict__ cos_sin, int max_pos,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ slots, TC* __restrict__ k_cache,
    TC* __restrict__ v_cache, int page_size, int Dp, const T* __restrict__ xq, int xq_stride, int q_rank,
    const float* __restrict__ q_norm_w, TC* __restrict__ q_out, int q_out_stride) {
    __shared__ float red[17];
    const int t = blockIdx.x, tid = threadIdx.x;
    if (xq) {
        const T* qr = xq + (size_t)t * xq_stride;
        float qs = 0.f;
        for (int e = tid; e < q_rank; e += blockDim.x) {
            const float v = to_f32(qr[e]);
            qs = fmaf(v, v, qs);
        }
        qs = block_sum(qs, red);
        const float rq = 1.0f / sqrtf(qs / (float)q_rank + eps);
        for (int e = tid; e < q_rank; e += blockDim.x)
            q_out[(size_t)t * q_out_stride + e] = from_f32<TC>(to_f32(qr[e]) * rq * q_norm_w[e]);
    }
    if (!x) return;
    const int slot = slots[t];
    if (slot < 0) return;      // (the whole block: a token that writes no key)
    latent_store_token<T, TC>(x + (size_t)t * x_stride, t, rank, rot, rot_dims, pairing, norm_w, eps, cos_sin, max_pos, positions, slot, k_cache,
                              v_cache, page_size, Dp, red);
}

TFF_API int tff_latent_kv_store(const void* x, int x_stride, int T, int rank, int rot, int rot_dims, int pairing,
                                const float* norm_w, float eps, const float* cos_sin, int max_pos,
                                const int32_t* positions, const int32_t* slots, void* k_cache, void* v_cache,
                                int page_size, int num_pages, int Dp, const void* xq, int xq_stride, int q_rank,
                                const float* q_norm_w, void* q_out, int q_out_stride, int dtype, int cache_dtype,
                                tff_stream_t stream) {
    TFF_REQUIRE(x || xq, "latent_kv_store: neither a key side nor a query side");
    TFF_REQUIRE(!x || (norm_w && positions && slots && k_cache && v_cache), "latent_kv_store: null pointer");
    TFF_REQUIRE(!x || (T >= 0 && rank > 0 && rot >= 0 && Dp >= rank + rot && x_stride >= rank + rot),
                "latent_kv_store: bad sizes rank=%d rot=%d padded=%d stride=%d", rank, rot, Dp, x_stride);
    TFF_REQUIRE(!x || (rot_dims >= 0 && rot_dims <= rot && rot_dims % 2 == 0 && (rot_dims == 0 || (cos_sin && max_pos > 0)) &&
                       (pairing == 0 || pairing == 1)),
                "latent_kv_store: %d rotated dimensions of %d need an even count and a table", rot_dims, rot);
    TFF_REQUIRE(!x || (page_size > 0 && num_pages > 0), "latent_kv_store: bad cache geometry");
    TFF_REQUIRE(!xq || (q_rank > 0 && xq_stride >= q_rank && q_norm_w && q_out && q_out_stride >= q_rank),
                "latent_kv_store: the query's latent vector of %d needs a weight and a place to go", q_rank);
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
#define TFF_LKS(TI, TCC)                                                                                              \
    latent_kv_store_kernel<TI, TCC><<<T, 256, 0, s>>>((const TI*)x, x_stride, rank, rot, rot_dims, pairing, norm_w, eps, \
                                                      rot_dims ? cos_sin : nullptr, max_pos, positions, slots,        \
                                                      (TCC*)k_cache, (TCC*)v_cache, page_size, Dp, (const TI*)xq,     \
                                                      xq_stride, q_rank, q_norm_w, (TCC*)q_out, q_out_stride)
    if (dtype == TFF_F32 && cache_dtype == TFF_F32)
        TFF_LKS(float, float);
    else if (dtype == TFF_BF16 && cache_dtype == TFF_BF16)
        TFF_LKS(bf16_t, bf16_t);
    else if (dtype == TFF_F32 && cache_dtype == TFF_BF16)
        TFF_LKS(float, bf16_t);
    else
        return tff_fail("latent_kv_store: rows of type %d for a cache of type %d", dtype, cache_dtype);
#undef TFF_LKS
    return tff_check_launch("latent_kv_store");
}

// ---------------------------------------------------------------- per-head products ---
// The general kernel (float32, and bfloat16 rows that are not 16-byte aligned): one block per
// (TT tokens, head, 256 output columns).  The block's input rows go to LDS as float32, KC
// elements at a time; thread n walks k along its row W[h][n][:], adding into TT accumulators,
// k ascending for every token whatever the batch.
#define HL_TT 8
#define HL_KC 128

struct HeadLinearTail {
    int tail;            // elements of the input row behind the K multiplied ones that are copied behind the product
    int rot_dims;        // of which the first rot_dims are rotated
    int pairing;         // 0: pairs (i, i + rot_dims / 2), 1: pairs (2i, 2i + 1)
    int pad_to;          // the output's head is filled with zeros up to this many elements
    int max_pos;
    const float* cos_sin;          // [position][pair][cos, sin], rot_dims / 2 pairs
    const int32_t* positions;      // per token
};

// The tail of the input heads of tokens t0 .. t0 + nt - 1 of head h, rotated and copied behind the
// N products, zeros up to pad_to; by all threads of the block.
template <typename T>
__device__ __forceinline__ void head_tail(const T* __restrict__ x, int x_row, int x_head, T* __restrict__ out,
                                          int out_row, int out_head, int t0, int nt, int h, int K, int N,
                                          const HeadLinearTail tl) {
    const int extra = tl.pad_to - N;
    for (int i = threadIdx.x; i < nt * extra; i += blockDim.x) {
        const int tt = i / extra, e = i - tt * extra;
        const T* xr = x + (size_t)(t0 + tt) * x_row + (size_t)h * x_head + K;
        float v = 0.f;
        if (e < tl.tail) {
            if (e < tl.rot_dims) {
                const int pos = min(max(tl.positions[t0 + tt], 0), tl.max_pos - 1);
                v = latent_rotated<T>(xr, e, tl.rot_dims, tl.pairing, tl.cos_sin + (size_t)pos * tl.rot_dims);
            } else {
                v = to_f32(xr[e]);
            }
        }
        out[(size_t)(t0 + tt) * out_row + (size_t)h * out_head + N + e] = from_f32<T>(v);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void head_linear_kernel(
    const T* __restrict__ x, int x_row, int x_head, const T* __restrict__ Wt, T* __restrict__ out, int out_row,
    int out_head, int Tn, int K, int N, const T* __restrict__ gate, int gate_row, HeadLinearTail tl) {
    __shared__ float xs[HL_TT][HL_KC];
    const int t0 = blockIdx.x * HL_TT, h = blockIdx.y, tid = threadIdx.x;
    const int n = blockIdx.z * 256 + tid;
    const int nt = min(HL_TT, Tn - t0);
    const T* W = Wt + ((size_t)h * N + min(n, N - 1)) * K;      // the thread's row
    float acc[HL_TT];
#pragma unroll
    for (int i = 0; i < HL_TT; ++i) acc[i] = 0.f;
    for (int k0 = 0; k0 < K; k0 += HL_KC) {
        const int kc = min(HL_KC, K - k0);
        __syncthreads();
        for (int i = tid; i < HL_TT * HL_KC; i += 256) {
            const int tt = i / HL_KC, k = i - tt * HL_KC;
            xs[tt][k] = (tt < nt && k < kc) ? to_f32(x[(size_t)(t0 + tt) * x_row + (size_t)h * x_head + k0 + k]) : 0.f;
        }
        __syncthreads();
        if (n < N) {
            for (int k = 0; k < kc; ++k) {
                const float w = to_f32(W[k0 + k]);
#pragma unroll
                for (int i = 0; i < HL_TT; ++i) acc[i] = fmaf(xs[i][k], w, acc[i]);
            }
        }
    }
    if (n < N) {
#pragma unroll
        for (int i = 0; i < HL_TT; ++i) {
            if (i >= nt) break;
            float v = acc[i];
            if (gate) {
                const float gz = to_f32(gate[(size_t)(t0 + i) * gate_row + (size_t)h * N + n]);
                v *= 1.0f / (1.0f + expf(-gz));
            }
            out[(size_t)(t0 + i) * out_row + (size_t)h * out_head + n] = from_f32<T>(v);
        }
    }
    if (blockIdx.z == 0 && tl.pad_to > N) head_tail<T>(x, x_row, x_head, out, out_row, out_head, t0, nt, h, K, N, tl);
}

// The same by whole pieces of eight elements, where sizes and addresses allow it.
__device__ __forceinline__ void head_tail_vec(const bf16_t* __restrict__ x, int x_row, int x_head, bf16_t* __restrict__ out,
                                              int out_row, int out_head, int t0, int nt, int h, int K, int N, const HeadLinearTail tl) {
    union Eight { uint4 u; bf16_t b[8]; };
    const int pieces = (tl.pad_to - N) >> 3;
    for (int i = threadIdx.x; i < nt * pieces; i += blockDim.x) {
        const int tt = i / pieces, e = (i - tt * pieces) * 8, t = t0 + tt;
        const bf16_t* xr = x + (size_t)t * x_row + (size_t)h * x_head + K;
        Eight v;
        v.u = make_uint4(0, 0, 0, 0);
        if (e < tl.tail) v.u = *reinterpret_cast<const uint4*>(xr + e);
        if (e < tl.rot_dims) {
            const int pos = min(max(tl.positions[t], 0), tl.max_pos - 1), half = tl.rot_dims >> 1;
            const float* cs = tl.cos_sin + (size_t)pos * tl.rot_dims;
            float c[16];
            if (tl.pairing == 1) {
                reinterpret_cast<float4*>(c)[0] = *reinterpret_cast<const float4*>(cs + e);
                reinterpret_cast<float4*>(c)[1] = *reinterpret_cast<const float4*>(cs + e + 4);
                Eight y;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float a = (float)v.b[k], o = (float)v.b[k ^ 1], co = c[k & 6], si = c[(k & 6) + 1];
                    y.b[k] = (bf16_t)(!(k & 1) ? fmaf(a, co, -(o * si)) : fmaf(a, co, o * si));
                }
                v = y;
            } else {
                const bool first = e < half;
                const int i0 = first ? e : e - half;
                Eight w, y;
                w.u = *reinterpret_cast<const uint4*>(xr + (first ? e + half : e - half));
#pragma unroll
                for (int k = 0; k < 4; ++k) reinterpret_cast<float4*>(c)[k] = *reinterpret_cast<const float4*>(cs + 2 * i0 + 4 * k);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float a = (float)v.b[k], o = (float)w.b[k], co = c[2 * k], si = c[2 * k + 1];
                    y.b[k] = (bf16_t)(first ? fmaf(a, co, -(o * si)) : fmaf(a, co, o * si));
                }
                v = y;
            }
        }
        *reinterpret_cast<uint4*>(out + (size_t)t * out_row + (size_t)h * out_head + N + e) = v.u;
    }
}

// bfloat16 on the matrix cores, any inner size.  Block: 64 tokens of one head, two waves of 32 tokens each for every second run of 64
// outputs; a wave asks for four k-steps of both operands at a time (24 loads), straight into the operands, and its results leave
// through LDS as whole pieces of 16 bytes.  C[n][t] += W[n][k] x[t][k]: W's rows are the first operand's rows, so lane (t = lane & 15,
// kg = lane >> 4) holds outputs n = kg * 4 .. + 3 of token t for each of the 4 x 2 tiles.  k ascends in steps of 32 for every token
// whatever the batch.
// VEC: output rows, heads, N and the tail's sizes are multiples of eight elements at 16-byte aligned addresses, and the gate's rows
// of four at 8-byte aligned ones; else the results go out one by one.  `runs`: runs of 64 outputs of a block.
template <bool VEC>
__global__ __launch_bounds__(256, 2) void head_linear_mfma_kernel(
    const bf16_t* __restrict__ x, int x_row, int x_head, const bf16_t* __restrict__ W, bf16_t* __restrict__ out,
    int out_row, int out_head, int Tn, int K, int N, const bf16_t* __restrict__ gate, int gate_row,
    HeadLinearTail tl, int runs) {
    constexpr int RB = 64 * 2 + 16, KS = 4;       // bytes of a staged row of 64 outputs; k-steps asked for at a time
    __shared__ __attribute__((aligned(16))) char staged[VEC ? 4 * 32 * RB : 16];
    union Eight { uint4 u; bf16x8 v; };
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, r = lane & 15, kg = lane >> 4;
    const int h = blockIdx.x, tb = blockIdx.y * 64, t0 = tb + (wv & 1) * 32;
    const int n_end = min(N, (int)(blockIdx.z + 1) * runs * 64);
    const bf16_t* xp[2];
    bool xok[2];        // (a lane whose row does not exist does not ask: the address unit takes a cycle for each lane that does)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        xok[i] = t0 + i * 16 + r < Tn;
        xp[i] = x + (size_t)min(t0 + i * 16 + r, Tn - 1) * x_row + (size_t)h * x_head;
    }
    if (t0 < Tn)        // (a wave's condition: the MFMAs below run for whole waves; outputs past the end repeat the last one)
        for (int n0 = (blockIdx.z * runs + (wv >> 1)) * 64; n0 < n_end; n0 += 128) {
            const bf16_t* wp[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) wp[j] = W + ((size_t)h * N + min(n0 + j * 16 + r, N - 1)) * K;
            union Four { uint2 u; bf16_t b[4]; } gz[4][2];
            if (VEC && gate) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        gz[j][i].u = xok[i] ? *reinterpret_cast<const uint2*>(gate + (size_t)(t0 + i * 16 + r) * gate_row + (size_t)h * N +
                                                                              min(n0 + j * 16 + kg * 4, N - 4))
                                            : make_uint2(0, 0);
            }
            floatx4 acc[4][2];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
            int k0 = 0;
            for (; k0 + KS * 32 <= K; k0 += KS * 32) {
                Eight a[KS][4], b[KS][2];
#pragma unroll
                for (int q = 0; q < KS; ++q) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) a[q][j].u = *reinterpret_cast<const uint4*>(wp[j] + k0 + q * 32 + kg * 8);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                        b[q][i].u = xok[i] ? *reinterpret_cast<const uint4*>(xp[i] + k0 + q * 32 + kg * 8) : make_uint4(0, 0, 0, 0);
                }
#pragma unroll
                for (int q = 0; q < KS; ++q)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[q][j].v, b[q][i].v, acc[j][i], 0, 0, 0);
            }
            for (; k0 < K; k0 += 32) {       // (K is a multiple of 8: a lane's eight elements exist together)
                const bool kok = k0 + kg * 8 < K;
                const int k = min(k0 + kg * 8, K - 8);
                Eight a[4], b[2];
#pragma unroll
                for (int j = 0; j < 4; ++j) a[j].u = *reinterpret_cast<const uint4*>(wp[j] + k);
#pragma unroll
                for (int i = 0; i < 2; ++i) b[i].u = *reinterpret_cast<const uint4*>(xp[i] + k);
#pragma unroll
                for (int j = 0; j < 4; ++j) a[j].u = kok ? a[j].u : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 2; ++i) b[i].u = kok ? b[i].u : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j].v, b[i].v, acc[j][i], 0, 0, 0);
            }
            char* region = staged + (VEC ? wv * 32 * RB : 0);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int t = t0 + i * 16 + r;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float v4[4] = {acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]};
                    if constexpr (VEC) {
                        Four p;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            p.b[e] = (bf16_t)(gate ? v4[e] * (1.0f / (1.0f + expf(-(float)gz[j][i].b[e]))) : v4[e]);
                        *reinterpret_cast<uint2*>(region + (i * 16 + r) * RB + (j * 16 + kg * 4) * 2) = p.u;
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int n = n0 + j * 16 + kg * 4 + e;
                            if (t < Tn && n < N) {
                                float v = v4[e];
                                if (gate) v *= 1.0f / (1.0f + expf(-(float)gate[(size_t)t * gate_row + (size_t)h * N + n]));
                                out[(size_t)t * out_row + (size_t)h * out_head + n] = (bf16_t)v;
                            }
                        }
                    }
                }
            }
            if constexpr (VEC) {             // (the wave's own part: its LDS operations come in order)
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                const int n = n0 + (lane & 7) * 8;
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const int row = p * 8 + (lane >> 3), t = t0 + row;
                    const uint4 v = *reinterpret_cast<const uint4*>(region + row * RB + (lane & 7) * 16);
                    if (t < Tn && n < N) *reinterpret_cast<uint4*>(out + (size_t)t * out_row + (size_t)h * out_head + n) = v;
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            }
        }
    if (blockIdx.z == 0 && tl.pad_to > N) {
        if constexpr (VEC) head_tail_vec(x, x_row, x_head, out, out_row, out_head, tb, min(64, Tn - tb), h, K, N, tl);
        else head_tail<bf16_t>(x, x_row, x_head, out, out_row, out_head, tb, min(64, Tn - tb), h, K, N, tl);
    }
}

// The same for inner sizes of one to four units of 64: through LDS as whole cache lines.  In the kernel
// above sixteen lanes of a load lie in sixteen rows, which costs the address unit a cycle a lane: 95 cycles a load, whatever the
// caches give.  Block: 64 tokens of one head and `runs` runs of 64 outputs, four waves of 32 tokens x 32 outputs.  The tokens' rows are
// copied once (eight rows x 128 bytes a copy, lane i takes chunk (i % 8) ^ (i / 8) of row i / 8, so that an operand's sixteen
// rows come back from different banks), a run's rows of W while the run before goes out.  The same order of k: the same bits.
// What bounds it is the rows going in and out, 60 MB for 2,048 tokens of 32 heads; with few tokens two latencies to memory.
// us, the kernel above as it was with results one by one / now: heads of 128 with a rotated tail of 64 into 256 elements, 1, 100, 2,048 and
// 8,192 tokens 4.5 / 3.5, 18.7 / 4.2, 56 / 19, 171 / 63; of 256 into 128 with a gate 7.2 / 4.4, 16.4 / 5.0, 52 / 23, 257 / 87.
// STORE: the launch writes the tokens' keys too (TffLatentStore, bfloat16): the blocks behind the heads', four tokens each.  The products
// and the keys come from the same projection and wait for nothing of each other; a launch costs a decode step some 5 us.
#define HL_STORE_TOKENS 4
template <bool STORE>
__global__ __launch_bounds__(256) void head_linear_lines_kernel(
    const bf16_t* __restrict__ x, int x_row, int x_head, const bf16_t* __restrict__ W, bf16_t* __restrict__ out,
    int out_row, int out_head, int Tn, int K, int N, const bf16_t* __restrict__ gate, int gate_row,
    HeadLinearTail tl, int runs, int H, const TffLatentStore st) {
    constexpr int RB = 32 * 2 + 16;               // bytes of a wave's staged row
    __shared__ __attribute__((aligned(16))) char staged[4 * 32 * RB];
    if constexpr (STORE) {
        if ((int)blockIdx.x >= H) {
            if (blockIdx.z) return;
            for (int i = 0; i < HL_STORE_TOKENS; ++i) {
                const int t = blockIdx.y * 64 + ((int)blockIdx.x - H) * HL_STORE_TOKENS + i;
                if (t >= Tn) return;
                const int slot = st.slots[t];
                if (slot >= 0)                    // (the whole block)
                    latent_store_token<bf16_t, bf16_t>((const bf16_t*)st.x + (size_t)t * st.x_stride, t, st.rank, st.rot, st.rot_dims, st.pairing,
                                                       st.norm_w, st.eps, st.rot_dims ? st.cos_sin : nullptr, st.max_pos, st.positions, slot,
                                                       (bf16_t*)st.k_cache, (bf16_t*)st.v_cache, st.page_size, st.Dp, reinterpret_cast<float*>(staged));
            }
            return;
        }
    }
    extern __shared__ __attribute__((aligned(1024))) char tiles[];       // the tokens' units, then the run's: 8 KB each
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, kg = lane >> 4;
    const int h = blockIdx.x, tb = blockIdx.y * 64, units = K >> 6;
    const int wm = wv & 1, wn = wv >> 1;
    const int n_first = blockIdx.z * runs * 64, n_end = min(N, n_first + runs * 64);
    const unsigned x_lds = (unsigned)(size_t)(lds_ptr_t)tiles, w_lds = x_lds + (unsigned)units * 8192u;
    const unsigned chunk = (unsigned)(((lane & 7) ^ (lane >> 3)) * 16);
    // a wave's copies of a unit: rows 16 wv .. + 15 of both operands
    unsigned xo[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) xo[c] = (unsigned)min(wv * 16 + c * 8 + (lane >> 3), Tn - 1 - tb) * (unsigned)x_row * 2u + chunk;
    const unsigned long long xb = (unsigned long long)(x + (size_t)tb * x_row + (size_t)h * x_head);
    for (int u = 0; u < units; ++u)
#pragma unroll
        for (int c = 0; c < 2; ++c) copy16_to_lds_sbase(xb + (unsigned)u * 128u, xo[c], x_lds + (unsigned)u * 8192u + (unsigned)(wv * 2 + c) * 1024u);
    auto copy_run = [&](int n0) {
        const unsigned long long wb = (unsigned long long)(W + ((size_t)h * N + n0) * K);
        for (int u = 0; u < units; ++u)
#pragma unroll
            for (int c = 0; c < 2; ++c)
                copy16_to_lds_sbase(wb + (unsigned)u * 128u, (unsigned)min(wv * 16 + c * 8 + (lane >> 3), N - 1 - n0) * (unsigned)K * 2u + chunk,
                                    w_lds + (unsigned)u * 8192u + (unsigned)(wv * 2 + c) * 1024u);
    };
    copy_run(n_first);
    unsigned rd[2];               // a lane's 16 bytes of an operand: row r of 16, chunk half * 4 + kg of the row's 8
#pragma unroll
    for (int q = 0; q < 2; ++q) rd[q] = (unsigned)(r >> 3) * 1024u + (unsigned)(((r & 7) * 8 + ((q * 4 + kg) ^ (r & 7))) * 16);
    const char* xt = tiles + wm * 4096;
    const char* wt = tiles + units * 8192 + wn * 4096;
    char* region = staged + wv * 32 * RB;
    for (int n0 = n_first; n0 < n_end; n0 += 64) {
        union Four { uint2 u; bf16_t b[4]; } gz[2][2];
        if (gate) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    gz[j][i].u = *reinterpret_cast<const uint2*>(gate + (size_t)min(tb + wm * 32 + i * 16 + r, Tn - 1) * gate_row + (size_t)h * N +
                                                                 min(n0 + wn * 32 + j * 16 + kg * 4, N - 4));
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __syncthreads();
        floatx4 acc[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
        for (int u = 0; u < units; ++u)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                bf16x8 a[2], b[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) a[j] = *reinterpret_cast<const bf16x8*>(wt + u * 8192 + j * 2048 + rd[q]);
#pragma unroll
                for (int i = 0; i < 2; ++i) b[i] = *reinterpret_cast<const bf16x8*>(xt + u * 8192 + i * 2048 + rd[q]);
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], b[i], acc[j][i], 0, 0, 0);
            }
        __syncthreads();                             // the run's rows have been read
        if (n0 + 64 < n_end) copy_run(n0 + 64);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                Four p;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = acc[j][i][e];
                    p.b[e] = (bf16_t)(gate ? v * (1.0f / (1.0f + expf(-(float)gz[j][i].b[e]))) : v);
                }
                *reinterpret_cast<uint2*>(region + (i * 16 + r) * RB + (j * 16 + kg * 4) * 2) = p.u;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (the wave's own part)
        const int n = n0 + wn * 32 + (lane & 3) * 8;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int row = p * 16 + (lane >> 2), t = tb + wm * 32 + row;
            const uint4 v = *reinterpret_cast<const uint4*>(region + row * RB + (lane & 3) * 16);
            if (t < Tn && n < N) *reinterpret_cast<uint4*>(out + (size_t)t * out_row + (size_t)h * out_head + n) = v;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if (blockIdx.z == 0 && tl.pad_to > N) head_tail_vec(x, x_row, x_head, out, out_row, out_head, tb, min(64, Tn - tb), h, K, N, tl);
}

TFF_API int tff_head_linear(const void* x, int x_row, int x_head, const void* Wt, void* out, int out_row, int out_head,
                            int T, int H, int K, int N, const void* gate, int gate_row, int tail, int rot_dims,
                            int pairing, int pad_to, const float* cos_sin, int max_pos, const int32_t* positions, int dtype,
                            const TffLatentStore* store, tff_stream_t stream) {
    TFF_REQUIRE(x && Wt && out, "head_linear: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && K > 0 && N > 0 && H <= 65535, "head_linear: bad sizes T=%d H=%d K=%d N=%d", T, H, K, N);
    TFF_REQUIRE(x_head >= K + tail && x_row >= (H - 1) * x_head + K + tail,
                "head_linear: input rows of %d with heads %d apart do not hold %d heads of %d + %d", x_row, x_head, H, K, tail);
    const int width = pad_to > N ? pad_to : N;
    TFF_REQUIRE(tail >= 0 && width >= N + tail && out_head >= width && out_row >= (H - 1) * out_head + width,
                "head_linear: output rows of %d with heads %d apart do not hold %d heads of %d", out_row, out_head, H, width);
    TFF_REQUIRE(rot_dims >= 0 && rot_dims <= tail && rot_dims % 2 == 0 && (rot_dims == 0 || (cos_sin && positions && max_pos > 0)) &&
                (pairing == 0 || pairing == 1),
                "head_linear: %d rotated dimensions of a tail of %d need an even count, a table and positions", rot_dims, tail);
    TFF_REQUIRE(!gate || gate_row >= H * N, "head_linear: gate rows of %d hold fewer than %d", gate_row, H * N);
    if (T == 0) return 0;
    auto keys_apart = [&]() {
        return tff_latent_kv_store(store->x, store->x_stride, T, store->rank, store->rot, store->rot_dims, store->pairing, store->norm_w, store->eps,
                                   store->cos_sin, store->max_pos, store->positions, store->slots, store->k_cache, store->v_cache, store->page_size,
                                   store->num_pages, store->Dp, nullptr, 0, 0, nullptr, nullptr, 0, store->dtype, store->cache_dtype, stream);
    };
    if (store) {        // (checked here as there)
        TFF_REQUIRE(store->x && store->norm_w && store->positions && store->slots && store->k_cache && store->v_cache, "head_linear: a null pointer among the keys'");
        TFF_REQUIRE(store->rank > 0 && store->rot >= 0 && store->Dp >= store->rank + store->rot && store->x_stride >= store->rank + store->rot &&
                    store->rot_dims >= 0 && store->rot_dims <= store->rot && store->rot_dims % 2 == 0 &&
                    (store->rot_dims == 0 || (store->cos_sin && store->max_pos > 0)) && (store->pairing == 0 || store->pairing == 1) &&
                    store->page_size > 0 && store->num_pages > 0, "head_linear: bad sizes of the keys");
    }
    hipStream_t s = (hipStream_t)stream;
    const HeadLinearTail tl{tail, rot_dims, pairing, pad_to, max_pos, cos_sin, positions};
    const dim3 grid((T + HL_TT - 1) / HL_TT, H, (N + 255) / 256);
    if (store && dtype != TFF_BF16)
        if (int rc = keys_apart()) return rc;
    if (dtype == TFF_F32)
        head_linear_kernel<float><<<grid, 256, 0, s>>>((const float*)x, x_row, x_head, (const float*)Wt, (float*)out, out_row,
                                                       out_head, T, K, N, (const float*)gate, gate_row, tl);
    else if (dtype == TFF_BF16) {
        const bool aligned = K % 8 == 0 && x_row % 8 == 0 && x_head % 8 == 0 && ((uintptr_t)x % 16) == 0 &&
                             ((uintptr_t)Wt % 16) == 0;
        if (aligned) {
            // whole pieces: of the results and the tail eight elements, of the gate four (its row of a head starts at h * N)
            const int extra = pad_to > N ? pad_to - N : 0;
            const bool vec = N % 8 == 0 && out_row % 8 == 0 && out_head % 8 == 0 && ((uintptr_t)out % 16) == 0 && extra % 8 == 0 && tail % 8 == 0 &&
                             rot_dims % (pairing == 0 ? 16 : 8) == 0 && ((uintptr_t)cos_sin % 16) == 0 &&
                             (!gate || (gate_row % 4 == 0 && ((uintptr_t)gate % 8) == 0));
            // A block has all of a head's outputs where that fills the chip (the tokens' rows are read once), else one run of 64: a step
            // of few tokens is two latencies to memory and what the address units of the CUs in use take for its loads.
            const int all = (N + 63) / 64, runs = (long)((T + 63) / 64) * H >= 512 ? all : 1;
            const dim3 mg(H, (T + 63) / 64, (all + runs - 1) / runs);
#define TFF_HL(VEC)                                                                                                              \
    head_linear_mfma_kernel<VEC><<<mg, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)Wt, (bf16_t*)out, out_row,     \
                                                    out_head, T, K, N, (const bf16_t*)gate, gate_row, tl, runs)
#define TFF_HL_LINES(STORE, GRID, KEYS)                                                                                            \
    head_linear_lines_kernel<STORE><<<GRID, 256, (unsigned)K * 256u, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)Wt, (bf16_t*)out, \
                                                                          out_row, out_head, T, K, N, (const bf16_t*)gate, gate_row, tl, runs, H, KEYS)
            if (vec && K % 64 == 0 && K <= 256) {
                if (store && store->dtype == TFF_BF16 && store->cache_dtype == TFF_BF16) {
                    const int per_tile = (T < 64 ? T : 64), columns = (per_tile + HL_STORE_TOKENS - 1) / HL_STORE_TOKENS;
                    TFF_HL_LINES(true, dim3(mg.x + columns, mg.y, mg.z), *store);
                    return tff_check_launch("head_linear");
                }
                if (store)
                    if (int rc = keys_apart()) return rc;
                TFF_HL_LINES(false, mg, TffLatentStore{});
                return tff_check_launch("head_linear");
            }
#undef TFF_HL_LINES
            if (store)
                if (int rc = keys_apart()) return rc;
            store = nullptr;
            if (vec) TFF_HL(true);
            else TFF_HL(false);
#undef TFF_HL
        }
        else {
            if (store)
                if (int rc = keys_apart()) return rc;
            head_linear_kernel<bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)x, x_row, x_head, (const bf16_t*)Wt, (bf16_t*)out,
                                                            out_row, out_head, T, K, N, (const bf16_t*)gate, gate_row, tl);
        }
    }
    else
        return tff_fail("head_linear: unknown dtype %d", dtype);
    return tff_check_launch("head_linear");
}
