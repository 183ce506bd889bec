// What stands around the paged attention kernels in a grouped attention whose queries carry a temperature that grows
// with the position and whose window has the mean keys of whole blocks of tokens before it.
//
// tff_grouped_qkv_store:  from the joint projection (float32): biases, an RMS norm over all of a token's q (and of its k)
//                         at once, rotation of q and k, the temperature on q, q laid out with the cache's head size, the
//                         token's key and value into its slot.
// tff_pool_keys:          for every token of the step that ends a block of P tokens: the means of the block's P keys and
//                         values, as the pages hold them, into the block's slot.
// tff_gate_heads:         a head's output times one gate per head and a scale, heads brought together.
#include "common.h"
#include "tffinfer_kernels.h"

struct GroupedRot {
    const float* cs;     // the position's [pair][cos, sin], or null
    int dims;            // rotated elements of a head (even)
    int pairing;         // 0: (i, i + dims/2), 1: (2i, 2i+1)
};

// Elements of a head come two by two: place p < dims / 2 is the p-th pair that turns, the others two neighbours behind
// the turned part.  f(element, its value): elements from D to P - 1 are zeros.
template <typename V, typename F>
__device__ __forceinline__ void grouped_pair(int p, int D, const GroupedRot r, V value, F f) {
    const int half = r.cs ? r.dims >> 1 : 0;
    if (p < half) {
        const int i = r.pairing == 0 ? p : 2 * p, j = r.pairing == 0 ? p + half : 2 * p + 1;
        const float u = value(i), w = value(j), c = r.cs[2 * p], s = r.cs[2 * p + 1];
        // the pair (u, w) becomes (u c - w s, w c + u s)
        f(i, fmaf(u, c, -(w * s)));
        f(j, fmaf(w, c, u * s));
    } else {
        const int i = 2 * p;
        f(i, i < D ? value(i) : 0.f);
        f(i + 1, i + 1 < D ? value(i + 1) : 0.f);
    }
}

// What happens to the projections before rotation.
struct GroupedPre {
    const float* bias;                 // [H D + G D + G E] in the projection's column order, or null
    const float *q_norm, *k_norm;      // [H D], [G D]: RMS norms over the whole of q and of k, or null
    float eps;
};

// Blocks (token, y): y < q_blocks works through `per_q` query heads; the others through `per_kv` kv heads each: their key
// and value rows into the token's slot.  Elements past a head's own size are zeros.  With a norm every block forms the
// sum of squares it needs by itself, always in the same order (its threads are as many whatever the step).
#define GQ_THREADS 128
#define GQ_WIDE 512      // threads with a norm, and where few tokens wait for one another's loads
#define GQ_HEADS 8

// 1 / sqrt(mean over x[0 .. n) of (x + bias)^2 + eps), the result in every thread of the block
template <int NT>
__device__ __forceinline__ float grouped_rms(const float* __restrict__ x, const float* __restrict__ bias, int n, float eps, bool vec,
                                             float* red) {
    float ss = 0.f;
    if (vec) {
#pragma unroll 8
        for (int c = threadIdx.x * 4; c < n; c += NT * 4) {
            float4 v = *reinterpret_cast<const float4*>(x + c);
            if (bias) {
                const float4 b = *reinterpret_cast<const float4*>(bias + c);
                v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
            }
            ss = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss))));
        }
    } else {
        for (int c = threadIdx.x; c < n; c += NT) {
            const float v = x[c] + (bias ? bias[c] : 0.f);
            ss = fmaf(v, v, ss);
        }
    }
    ss = rows_sum(row16_sum(ss));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) ss += red[i];
    return 1.0f / sqrtf(ss / (float)n + eps);
}

template <typename TC, int NT>
__global__ __launch_bounds__(NT) void grouped_qkv_store_kernel(
    const float* __restrict__ proj, size_t row, const float* __restrict__ cos_sin, int rot_dims, int pairing, int max_pos,
    float temp_coef, int temp_every, const GroupedPre pre, const int32_t* __restrict__ positions, const int32_t* __restrict__ slots,
    TC* __restrict__ q_out, TC* __restrict__ k_cache, TC* __restrict__ v_cache, int page_size, int H, int G, int D, int E, int P,
    int q_blocks, int per_q, int per_kv, int vec) {
    __shared__ float red[NT / 64];
    const int t = blockIdx.x, y = blockIdx.y, tid = threadIdx.x;
    const float* x = proj + (size_t)t * row;
    const int pos = max(positions[t], 0), tpos = min(pos, max(max_pos - 1, 0));
    const GroupedRot rot{(cos_sin && rot_dims) ? cos_sin + (size_t)tpos * rot_dims : nullptr, rot_dims, pairing};
    const int half = P >> 1;                 // places of a head
    if (y < q_blocks) {
        const float temp = temp_coef != 0.f ? 1.0f + temp_coef * logf((float)((pos + 1) / temp_every + 1)) : 1.0f;
        const float rr = pre.q_norm ? grouped_rms<NT>(x, pre.bias, H * D, pre.eps, vec, red) : 1.0f;
        TC* qo = q_out + (size_t)t * H * P;
        const int h0 = y * per_q, count = (min(H, h0 + per_q) - h0) * half;
        for (int idx = tid; idx < count; idx += NT) {
            const int h = h0 + idx / half, p = idx % half, c0 = h * D;
            TC* const qh = qo + (size_t)h * P;
            grouped_pair(p, D, rot,
                [&](int e) {
                    float v = x[c0 + e];
                    if (pre.bias) v += pre.bias[c0 + e];
                    return pre.q_norm ? v * rr * pre.q_norm[c0 + e] : v;
                },
                [&](int e, float v) { qh[e] = from_f32<TC>(v * temp); });
        }
        return;
    }
    const int slot = slots[t];
    if (slot < 0) return;      // (the whole block: a token that writes no key)
    const int page = slot / page_size, off = slot - page * page_size;
    const size_t ck = (size_t)H * D;
    const float* xk = x + ck;
    const float* bk = pre.bias ? pre.bias + ck : nullptr;
    const float rr = pre.k_norm ? grouped_rms<NT>(xk, bk, G * D, pre.eps, vec, red) : 1.0f;
    const int g0 = (y - q_blocks) * per_kv, groups = min(G, g0 + per_kv) - g0;
    for (int idx = tid; idx < groups * half; idx += NT) {
        const int g = g0 + idx / half, p = idx % half, c0 = g * D;
        TC* const kd = k_cache + (((size_t)page * G + g) * page_size + off) * P;
        grouped_pair(p, D, rot,
            [&](int e) {
                float v = xk[c0 + e];
                if (bk) v += bk[c0 + e];
                return pre.k_norm ? v * rr * pre.k_norm[c0 + e] : v;
            },
            [&](int e, float v) { kd[e] = from_f32<TC>(v); });
    }
    for (int idx = tid; idx < groups * P; idx += NT) {
        const int g = g0 + idx / P, e = idx % P;
        const size_t cv = ck + (size_t)G * D + (size_t)g * E + e;
        TC* const vd = v_cache + ((size_t)page * G + g) * P * page_size + off;
        vd[(size_t)e * page_size] = from_f32<TC>(e < E ? x[cv] + (pre.bias ? pre.bias[cv] : 0.f) : 0.f);
    }
}

// The same for steps of many tokens in bfloat16 whose heads are of one size in units of eight and turn as a whole, in either pairing, or
// not at all: a thread has four neighbouring elements of either half of a head, 16 bytes a load, and the values go to their transposed pages eight
// tokens at a time, 16 bytes a store, in blocks of their own (the grid's rows from qk_rows on).  One value of a token is two bytes
// of a line that its neighbours' blocks write too, on other XCDs.  The same sums in the same order: the same bits.
// us, an element a thread and load / now: 4,500 tokens of 32 + 8 + 8 heads of 128 65 / 45, with norms over all of q and k 74 / 60;
// 1,500 tokens 24 / 17 and 30 / 23.
template <int NT>
__global__ __launch_bounds__(NT) void grouped_qkv_store_vec_kernel(
    const float* __restrict__ proj, size_t row, const float* __restrict__ cos_sin, int pairing, int max_pos, float temp_coef, int temp_every,
    const GroupedPre pre, const int32_t* __restrict__ positions, const int32_t* __restrict__ slots, bf16_t* __restrict__ q_out,
    bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache, int page_size, int T, int H, int G, int D, int q_blocks, int per_q,
    int qk_rows, int per_kv) {
    __shared__ float red[NT / 64];
    __shared__ __attribute__((aligned(16))) bf16_t tile[8][256 + 8];
    __shared__ int vslots[8];
    const int tid = threadIdx.x, y = blockIdx.y;
    if (y >= qk_rows) {                     // values: eight tokens and one kv head
        const long item = (long)(y - qk_rows) * T + blockIdx.x;
        if (item >= (long)((T + 7) / 8) * G) return;
        const int t0 = (int)(item / G) * 8, g = (int)(item % G), ppr = D >> 2;
        if (tid < 8) vslots[tid] = t0 + tid < T ? slots[t0 + tid] : -1;
        const size_t cv = (size_t)H * D + (size_t)G * D + (size_t)g * D;
        for (int i = tid; i < 8 * ppr; i += NT) {
            const int tk = i / ppr, e = (i - tk * ppr) * 4;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (t0 + tk < T) v = *reinterpret_cast<const float4*>(proj + (size_t)(t0 + tk) * row + cv + e);
            if (pre.bias) {
                const float4 b = *reinterpret_cast<const float4*>(pre.bias + cv + e);
                v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
            }
            tile[tk][e] = (bf16_t)v.x; tile[tk][e + 1] = (bf16_t)v.y; tile[tk][e + 2] = (bf16_t)v.z; tile[tk][e + 3] = (bf16_t)v.w;
        }
        __syncthreads();
        const int s0 = vslots[0];
        bool run = s0 >= 0 && (s0 & 7) == 0 && page_size % 8 == 0;
#pragma unroll
        for (int i = 1; i < 8; ++i) run = run && vslots[i] == s0 + i;
        for (int e = tid; e < D; e += NT) {
            if (run) {
                union { uint4 u; bf16_t h[8]; } pk;
#pragma unroll
                for (int i = 0; i < 8; ++i) pk.h[i] = tile[i][e];
                *reinterpret_cast<uint4*>(v_cache + (((size_t)(s0 / page_size) * G + g) * D + e) * page_size + s0 % page_size) = pk.u;
            } else {
                for (int i = 0; i < 8; ++i)
                    if (vslots[i] >= 0) v_cache[(((size_t)(vslots[i] / page_size) * G + g) * D + e) * page_size + vslots[i] % page_size] = tile[i][e];
            }
        }
        return;
    }
    const int t = blockIdx.x, half = D >> 1, pieces = D >> 3;
    const bool is_q = y < q_blocks;
    const int slot = is_q ? 0 : slots[t];
    const int pos = max(positions[t], 0), tpos = min(pos, max(max_pos - 1, 0));
    if (slot < 0) return;      // (the whole block: a token that writes no key)
    const size_t c0 = is_q ? 0 : (size_t)H * D;
    const float* x = proj + (size_t)t * row + c0;
    const float* bias = pre.bias ? pre.bias + c0 : nullptr;
    const float* nw = is_q ? pre.q_norm : pre.k_norm;
    const int heads = is_q ? H : G, first = is_q ? y * per_q : (y - q_blocks) * per_kv, count = min(heads, first + (is_q ? per_q : per_kv)) - first;
    const float temp = is_q && temp_coef != 0.f ? 1.0f + temp_coef * logf((float)((pos + 1) / temp_every + 1)) : 1.0f;
    const float rr = nw ? grouped_rms<NT>(x, bias, heads * D, pre.eps, 1, red) : 1.0f;
    const float* cs = cos_sin ? cos_sin + (size_t)tpos * D : nullptr;
    bf16_t* const to = is_q ? q_out + (size_t)t * H * D : k_cache + (((size_t)(slot / page_size) * G) * page_size + slot % page_size) * D;
    const size_t step = is_q ? (size_t)D : (size_t)page_size * D;
    for (int idx = tid; idx < count * pieces; idx += NT) {
        const int h = first + idx / pieces, p = (idx % pieces) * 4, e = h * D + p;
        float u[4], w[4], c[8];
        auto take = [&](float* v, int at) {
            *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(x + at);
            if (bias) {
                const float4 b = *reinterpret_cast<const float4*>(bias + at);
                v[0] += b.x; v[1] += b.y; v[2] += b.z; v[3] += b.w;
            }
            if (nw) {
                const float4 n = *reinterpret_cast<const float4*>(nw + at);
                v[0] = v[0] * rr * n.x; v[1] = v[1] * rr * n.y; v[2] = v[2] * rr * n.z; v[3] = v[3] * rr * n.w;
            }
        };
        if (cs) {
            // (cosine and sine of the piece's four pairs, or of its two pairs in the first half and of the two in the second)
            *reinterpret_cast<float4*>(c) = *reinterpret_cast<const float4*>(pairing == 0 ? cs + 2 * p : cs + p);
            *reinterpret_cast<float4*>(c + 4) = *reinterpret_cast<const float4*>(pairing == 0 ? cs + 2 * p + 4 : cs + half + p);
        }
        take(u, e);
        take(w, e + half);
        union { uint2 v; bf16_t b[4]; } a, b;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float yu = u[k], yw = w[k];
            if (cs && pairing == 0) {
                yu = fmaf(u[k], c[2 * k], -(w[k] * c[2 * k + 1]));
                yw = fmaf(w[k], c[2 * k], u[k] * c[2 * k + 1]);
            } else if (cs) {
                const int j = k & 2;
                yu = !(k & 1) ? fmaf(u[k], c[j], -(u[k ^ 1] * c[j + 1])) : fmaf(u[k], c[j], u[k ^ 1] * c[j + 1]);
                yw = !(k & 1) ? fmaf(w[k], c[4 + j], -(w[k ^ 1] * c[4 + j + 1])) : fmaf(w[k], c[4 + j], w[k ^ 1] * c[4 + j + 1]);
            }
            a.b[k] = (bf16_t)(is_q ? yu * temp : yu);
            b.b[k] = (bf16_t)(is_q ? yw * temp : yw);
        }
        bf16_t* const o = to + (size_t)h * step + p;
        *reinterpret_cast<uint2*>(o) = a.v;
        *reinterpret_cast<uint2*>(o + half) = b.v;
    }
}

TFF_API int tff_grouped_qkv_store(const float* proj, size_t row, const float* cos_sin, int rot_dims, int pairing, int max_pos,
                                  float temp_coef, int temp_every, const float* bias, const float* q_norm, const float* k_norm,
                                  float norm_eps, const int32_t* positions, const int32_t* slots, void* q_out, void* k_cache,
                                  void* v_cache, int page_size, int num_pages, int T, int H, int G, int D, int E, int P, int store,
                                  int dtype, tff_stream_t stream) {
    TFF_REQUIRE(proj && positions && q_out && (!store || (slots && k_cache && v_cache)), "grouped_qkv_store: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && G > 0 && H % G == 0 && D > 0 && E > 0 && P >= D && P >= E && temp_every > 0,
                "grouped_qkv_store: bad sizes H=%d G=%d D=%d E=%d P=%d", H, G, D, E, P);
    TFF_REQUIRE(P % 2 == 0, "grouped_qkv_store: a cache head of %d elements must be even", P);
    TFF_REQUIRE(row >= (size_t)H * D + (store ? (size_t)G * (D + E) : 0), "grouped_qkv_store: rows of %zu are too short", row);
    TFF_REQUIRE(rot_dims >= 0 && rot_dims <= D && rot_dims % 2 == 0 && (rot_dims == 0 || (cos_sin && max_pos > 0)) &&
                (pairing == 0 || pairing == 1), "grouped_qkv_store: %d rotated elements of a head of %d need an even count and a table", rot_dims, D);
    TFF_REQUIRE(page_size > 0 && num_pages > 0, "grouped_qkv_store: bad cache geometry");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    // (with a norm over all heads, many tokens fill the GPU with a block each for q and for k: nothing is summed twice)
    const bool whole = (q_norm || k_norm) && T >= 128;
    const int per_q = whole ? H : GQ_HEADS, per_kv = whole ? G : 1;
    const int q_blocks = (H + per_q - 1) / per_q, kv_blocks = store ? (G + per_kv - 1) / per_kv : 0;
    const int vec = D % 4 == 0 && row % 4 == 0 && ((uintptr_t)proj % 16) == 0 && ((uintptr_t)bias % 16) == 0;
    TFF_REQUIRE(q_blocks + kv_blocks <= 65535, "grouped_qkv_store: too many heads");
    const dim3 grid(T, q_blocks + kv_blocks);
    const bool wide = q_norm || k_norm || T < 128;
    auto ok16 = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
    // Heads of 128 and more; of 64 and more with norms, or once their rows are some megabytes: smaller ones are a few pieces a head, and
    // the lanes that share a head's index arithmetic are fewer.  us, an element a thread / pieces: 16 + 4 + 4 heads of 64, 1,000 tokens 6.7 / 7.2,
    // 3,000 15.1 / 14.8, with norms 1,000 9.8 / 9.4; 20 + 20 + 20 of 40, 3,000 41 / 45, with norms 34 / 44.
    const bool pays = D >= 128 || (D >= 64 && (wide || (long)T * (H + 2 * G) * D >= (1L << 22)));
    if (pays && T >= 128 && store && dtype == TFF_BF16 && vec && D == E && D == P && D % 8 == 0 && D <= 256 && ok16(q_norm) && ok16(k_norm) && ok16(cos_sin) &&
        ok16(q_out) && ok16(k_cache) && ok16(v_cache) && (rot_dims == 0 || rot_dims == D)) {
        const int qk_rows = q_blocks + kv_blocks, v_rows = (int)(((long)((T + 7) / 8) * G + T - 1) / T);      // (the values' blocks fill whole rows of the grid)
        const dim3 vgrid(T, qk_rows + v_rows);
#define GQ_VEC(NT)                                                                                                                  \
    grouped_qkv_store_vec_kernel<NT><<<vgrid, NT, 0, s>>>(proj, row, rot_dims ? cos_sin : nullptr, pairing, max_pos, temp_coef, temp_every, \
                                                          GroupedPre{bias, q_norm, k_norm, norm_eps}, positions, slots, (bf16_t*)q_out, \
                                                          (bf16_t*)k_cache, (bf16_t*)v_cache, page_size, T, H, G, D, q_blocks, per_q,    \
                                                          qk_rows, per_kv)
        if (wide) GQ_VEC(GQ_WIDE);
        else GQ_VEC(GQ_THREADS);
#undef GQ_VEC
        return tff_check_launch("grouped_qkv_store");
    }
#define GQ_LAUNCH(TC, NT)                                                                                                      \
    grouped_qkv_store_kernel<TC, NT><<<grid, NT, 0, s>>>(proj, row, cos_sin, rot_dims, pairing, max_pos, temp_coef, temp_every, \
                                                         GroupedPre{bias, q_norm, k_norm, norm_eps}, positions, slots, (TC*)q_out, \
                                                         (TC*)k_cache, (TC*)v_cache, page_size, H, G, D, E, P, q_blocks, per_q, per_kv, vec)
    if (dtype == TFF_F32 && wide) GQ_LAUNCH(float, GQ_WIDE);
    else if (dtype == TFF_F32) GQ_LAUNCH(float, GQ_THREADS);
    else if (dtype == TFF_BF16 && wide) GQ_LAUNCH(bf16_t, GQ_WIDE);
    else if (dtype == TFF_BF16) GQ_LAUNCH(bf16_t, GQ_THREADS);
    else return tff_fail("grouped_qkv_store: unknown dtype %d", dtype);
#undef GQ_LAUNCH
    return tff_check_launch("grouped_qkv_store");
}

// Blocks (token, kv head); the tokens are those that `tokens` lists, or all of the step's, of which those that end no
// block leave at once.  The sum runs over the block's tokens in their order; a thread takes elements tid, tid + 128, ...
// Where the tokens' keys and values lie is worked out by the threads side by side, PK_RUN tokens at a time.
#define PK_THREADS 128
#define PK_RUN 64

template <typename TC>
__global__ __launch_bounds__(PK_THREADS) void pool_keys_kernel(TC* __restrict__ k_cache, TC* __restrict__ v_cache,
                                                               const int32_t* __restrict__ block_tables, int bt_stride,
                                                               const int32_t* __restrict__ pool_tables, int pt_stride,
                                                               const int32_t* __restrict__ token_req,
                                                               const int32_t* __restrict__ positions,
                                                               const int32_t* __restrict__ slots,
                                                               const int32_t* __restrict__ tokens, int page_size, int pool, int G,
                                                               int d) {
    __shared__ size_t koff[PK_RUN], voff[PK_RUN];
    const int t = tokens ? tokens[blockIdx.x] : (int)blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
    const int pos = positions[t];
    if (slots[t] < 0 || (pos + 1) % pool) return;      // (the whole block)
    const int r = token_req[t], blk = pos / pool, first = pos + 1 - pool;
    const int32_t* bt = block_tables + (size_t)r * bt_stride;
    const int dpage = pool_tables[(size_t)r * pt_stride + blk / page_size], dslot = blk % page_size;
    const float f = 1.0f / (float)pool;
    const size_t dhead = ((size_t)dpage * G + g) * page_size * d;
    for (int e0 = 0; e0 < d; e0 += PK_THREADS) {
        const int e = min(e0 + tid, d - 1);
        float ks = 0.f, vs = 0.f;
        for (int i0 = 0; i0 < pool; i0 += PK_RUN) {
            const int cnt = min(PK_RUN, pool - i0);
            if (i0 || e0) __syncthreads();             // the run before is read
            if (tid < cnt) {
                const int j = first + i0 + tid, slot = j % page_size;
                const size_t head = ((size_t)bt[j / page_size] * G + g) * page_size * d;
                koff[tid] = head + (size_t)slot * d;
                voff[tid] = head + slot;
            }
            __syncthreads();
#pragma unroll 8
            for (int i = 0; i < cnt; ++i) {
                ks += to_f32(k_cache[koff[i] + e]);
                vs += to_f32(v_cache[voff[i] + (size_t)e * page_size]);
            }
        }
        if (e0 + tid < d) {
            k_cache[dhead + (size_t)dslot * d + e] = from_f32<TC>(ks * f);
            v_cache[dhead + (size_t)e * page_size + dslot] = from_f32<TC>(vs * f);
        }
    }
}

TFF_API int tff_pool_keys(void* k_cache, void* v_cache, const int32_t* block_tables, int bt_stride, const int32_t* pool_tables,
                          int pt_stride, const int32_t* token_req, const int32_t* positions, const int32_t* slots,
                          const int32_t* tokens, int page_size, int num_pages, int pool, int T, int G, int d, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(k_cache && v_cache && block_tables && pool_tables && token_req && positions && slots, "pool_keys: null pointer");
    TFF_REQUIRE(T >= 0 && G > 0 && G <= 65535 && d > 0 && pool > 0 && page_size > 0 && num_pages > 0 && bt_stride > 0 && pt_stride > 0,
                "pool_keys: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(T, G);
    if (dtype == TFF_F32)
        pool_keys_kernel<float><<<grid, PK_THREADS, 0, s>>>((float*)k_cache, (float*)v_cache, block_tables, bt_stride, pool_tables, pt_stride,
                                                            token_req, positions, slots, tokens, page_size, pool, G, d);
    else if (dtype == TFF_BF16)
        pool_keys_kernel<bf16_t><<<grid, PK_THREADS, 0, s>>>((bf16_t*)k_cache, (bf16_t*)v_cache, block_tables, bt_stride, pool_tables,
                                                             pt_stride, token_req, positions, slots, tokens, page_size, pool, G, d);
    else
        return tff_fail("pool_keys: unknown dtype %d", dtype);
    return tff_check_launch("pool_keys");
}

// out[t, h E + e] = o[t, h P + e] * sigmoid(g[t, h]) * scale      (g null: no gate); rows of out out_row apart
template <typename T>
__global__ __launch_bounds__(256) void gate_heads_kernel(const T* __restrict__ o, size_t o_row, int P, const float* __restrict__ g,
                                                         size_t g_row, float scale, T* __restrict__ out, size_t out_row, int HE, int E,
                                                         size_t count) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= count) return;
    const size_t t = id / HE;
    const int c = (int)(id - t * HE), h = c / E, e = c - h * E;
    const float f = g ? scale / (1.0f + expf(-g[t * g_row + h])) : scale;
    out[t * out_row + c] = from_f32<T>(to_f32(o[t * o_row + (size_t)h * P + e]) * f);
}

// The same, eight neighbouring elements a thread (E, P and the rows' strides multiples of 8).
__global__ __launch_bounds__(256) void gate_heads8_kernel(const bf16_t* __restrict__ o, size_t o_row, int P, const float* __restrict__ g,
                                                          size_t g_row, float scale, bf16_t* __restrict__ out, size_t out_row, int HE8,
                                                          int E8, size_t count) {
    const size_t id = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= count) return;
    const size_t t = id / HE8;
    const int c = (int)(id - t * HE8), h = c / E8, e = c - h * E8;
    const float f = g ? scale / (1.0f + expf(-g[t * g_row + h])) : scale;
    union { uint4 u; bf16_t b[8]; } x;
    x.u = *reinterpret_cast<const uint4*>(o + t * o_row + (size_t)h * P + e * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) x.b[i] = (bf16_t)((float)x.b[i] * f);
    *reinterpret_cast<uint4*>(out + t * out_row + (size_t)c * 8) = x.u;
}

TFF_API int tff_gate_heads(const void* o, size_t o_row, int P, const float* g, size_t g_row, float scale, void* out, size_t out_row,
                           int T, int H, int E, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(o && out, "gate_heads: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && E > 0 && P >= E && o_row >= (size_t)H * P && out_row >= (size_t)H * E && (!g || g_row >= (size_t)H),
                "gate_heads: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const size_t count = (size_t)T * H * E;
    const unsigned blocks = (unsigned)((count + 255) / 256);
    if (dtype == TFF_BF16 && E % 8 == 0 && P % 8 == 0 && o_row % 8 == 0 && out_row % 8 == 0 && ((uintptr_t)o % 16) == 0 &&
        ((uintptr_t)out % 16) == 0) {
        gate_heads8_kernel<<<(unsigned)((count / 8 + 255) / 256), 256, 0, s>>>((const bf16_t*)o, o_row, P, g, g_row, scale, (bf16_t*)out,
                                                                               out_row, H * E / 8, E / 8, count / 8);
        return tff_check_launch("gate_heads");
    }
    if (dtype == TFF_F32)
        gate_heads_kernel<float><<<blocks, 256, 0, s>>>((const float*)o, o_row, P, g, g_row, scale, (float*)out, out_row, H * E, E, count);
    else if (dtype == TFF_BF16)
        gate_heads_kernel<bf16_t><<<blocks, 256, 0, s>>>((const bf16_t*)o, o_row, P, g, g_row, scale, (bf16_t*)out, out_row, H * E, E, count);
    else
        return tff_fail("gate_heads: unknown dtype %d", dtype);
    return tff_check_launch("gate_heads");
}
