// Attention whose heads exchange their scores before the softmax, over the paged cache:
//
//   s_g(i, j) = cap * tanh(scale * q_g(i) . k_g(j) / cap)  [cap > 0]  + bias[min(i - j, rows - 1), g]
//   s'_h(i, j) = sum_g mix[h, g] * s_g(i, j)                         [mix given]
//   visible: j <= i and (i - j < window or j < keep_first)           [window > 0; else all j <= i]
//   p_h(i, j) = exp(s'_h) / (sink + sum over visible j of exp(s'_h))  (sink = 1: a key of score 0 without a value)
//   out_h(i) = sum_j p_h(i, j) v(j)
//
// Query head g reads kv head g / (H / G).  Scores, bias, mixing and softmax are float32.  Keys lie
// in pages [kv head, slot, element], values transposed [kv head, element, slot].
//
// tff_qk_bias_norm_store: q and k rows from one projection [T, (H + G) * D] (float32) get their biases;
//   q is divided by its root mean square over the head and written out; k goes into the token's slot
//   twice: as projected into the value page, divided by its root mean square into the key page.
// tff_mixed_attention: one block per query token (and split of its keys), all heads; keys in tiles of 64 (32 on the matrix
//   cores) whose borders are multiples of their size from the sequence's start, so a query's sums are formed in the same
//   order in every step that computes it with the same number of splits; a step of few tokens splits each
//   token's tiles over several blocks and a second kernel puts them together.
#include "common.h"
#include "tffinfer_kernels.h"

template <typename TC>
__global__ __launch_bounds__(256) void qk_bias_norm_store_kernel(
    const float* __restrict__ qk, size_t row, const float* __restrict__ qb, const float* __restrict__ kb, float eps,
    TC* __restrict__ q_out, TC* __restrict__ k_cache, TC* __restrict__ v_cache,
    const int32_t* __restrict__ slot_mapping, int page_size, int pairs, int H, int G, int D) {
    const int id = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (id >= pairs) return;
    const int t = id / (H + G), head = id % (H + G);
    const float* src = qk + (size_t)t * row + (size_t)head * D;
    const float* bias = head < H ? (qb ? qb + (size_t)head * D : nullptr) : (kb ? kb + (size_t)(head - H) * D : nullptr);
    float ss = 0.f;
    for (int e = lane; e < D; e += 64) {
        const float a = src[e] + (bias ? bias[e] : 0.f);
        ss = fmaf(a, a, ss);
    }
    ss = wave_sum(ss);
    const float rr = 1.0f / sqrtf(ss / (float)D + eps);
    if (head < H) {
        TC* dst = q_out + ((size_t)t * H + head) * D;
        for (int e = lane; e < D; e += 64) dst[e] = from_f32<TC>((src[e] + (bias ? bias[e] : 0.f)) * rr);
        return;
    }
    const int slot = slot_mapping[t];
    if (slot < 0) return;
    const int g = head - H, page = slot / page_size, off = slot % page_size;
    TC* kd = k_cache + (((size_t)page * G + g) * page_size + off) * D;
    TC* vd = v_cache + ((size_t)page * G + g) * D * page_size + off;
    for (int e = lane; e < D; e += 64) {
        const float a = src[e] + (bias ? bias[e] : 0.f);
        kd[e] = from_f32<TC>(a * rr);
        vd[(size_t)e * page_size] = from_f32<TC>(a);
    }
}

TFF_API int tff_qk_bias_norm_store(const float* qk, size_t row, const float* qb, const float* kb, float eps, void* q_out,
                                   void* k_cache, void* v_cache, const int32_t* slot_mapping, int page_size, int T, int H,
                                   int G, int D, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(qk && q_out && k_cache && v_cache && slot_mapping, "qk_bias_norm_store: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && G > 0 && D > 0 && page_size > 0 && row >= (size_t)(H + G) * D,
                "qk_bias_norm_store: bad sizes");
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int pairs = T * (H + G);
    if (dtype == TFF_F32)
        qk_bias_norm_store_kernel<float><<<(pairs + 3) / 4, 256, 0, s>>>(qk, row, qb, kb, eps, (float*)q_out, (float*)k_cache,
                                                                         (float*)v_cache, slot_mapping, page_size, pairs, H, G, D);
    else if (dtype == TFF_BF16)
        qk_bias_norm_store_kernel<bf16_t><<<(pairs + 3) / 4, 256, 0, s>>>(qk, row, qb, kb, eps, (bf16_t*)q_out,
                                                                          (bf16_t*)k_cache, (bf16_t*)v_cache, slot_mapping,
                                                                          page_size, pairs, H, G, D);
    else
        return tff_fail("qk_bias_norm_store: unknown dtype %d", dtype);
    return tff_check_launch("qk_bias_norm_store");
}

#define MA_TK 64        // keys a tile: one a lane where a wave takes a head's scores
#define MA_THREADS 512   // eight waves: two a SIMD, so that LDS and lane-swap latencies of one hide behind the other
#define MA_WAVES 8

// eight consecutive elements as floats
__device__ __forceinline__ void ma_load8(const float* p, float* f) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
}
__device__ __forceinline__ void ma_load8(const bf16_t* p, float* f) {
    union { uint4 u; bf16_t h[8]; } pk;
    pk.u = *reinterpret_cast<const uint4*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = (float)pk.h[i];
}

// A token's visible keys lie in two ranges: the first tokens that are kept (those that the window does not
// hold anyway), [0, a_hi), and the window, [lo, pos].  Their tiles are numbered through: first those of
// the first range, then those of the second, each starting at a multiple of the tile's size.
template <int TK>
struct MaTiles {
    int a_hi, lo, hi, n_a, jt_b, n;
    __device__ MaTiles(int pos, int window, int keep_first) {
        lo = window > 0 ? max(0, pos - window + 1) : 0;
        a_hi = min(keep_first, lo);
        hi = pos + 1;
        n_a = (a_hi + TK - 1) / TK;
        jt_b = (lo / TK) * TK;
        n = n_a + (pos - jt_b) / TK + 1;
    }
};

// One block per (token, split of the token's tiles).  With one split the block writes the token's result;
// with more it leaves, per head, its running maximum, its sum and the unnormalised weighted values for
// mixed_attention_merge_kernel (the sink's term is then the merge's to add).
// Eight consecutive elements as they come from memory; several are asked for before the first is used, so that
// a thread waits for memory once per group and not once per load.
template <typename TC> struct MaRaw;
template <> struct MaRaw<bf16_t> {
    uint4 u;
    __device__ __forceinline__ void load(const bf16_t* p) { u = *reinterpret_cast<const uint4*>(p); }
    __device__ __forceinline__ void zero() { u = make_uint4(0, 0, 0, 0); }
    __device__ __forceinline__ void get(float* f) const {
        union { uint4 u; bf16_t h[8]; } pk;
        pk.u = u;
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = (float)pk.h[i];
    }
};
template <> struct MaRaw<float> {
    float4 a, b;
    __device__ __forceinline__ void load(const float* p) {
        a = *reinterpret_cast<const float4*>(p);
        b = *reinterpret_cast<const float4*>(p + 4);
    }
    __device__ __forceinline__ void zero() { a = make_float4(0, 0, 0, 0); b = a; }
    __device__ __forceinline__ void get(float* f) const {
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
};

#define MA_AHEAD 4      // key rows a wave asks for before it multiplies the first
#define MA_RUNS 4       // runs of 8 values a thread asks for before it multiplies the first

template <typename TC, int ACC>
__global__ __launch_bounds__(MA_THREADS) void mixed_attention_kernel(
    const TC* __restrict__ q, const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int bt_width, const int32_t* __restrict__ token_req,
    const int32_t* __restrict__ positions, const float* __restrict__ bias, int bias_rows,
    const float* __restrict__ mix, float scale, float cap, int window, int keep_first, int sink,
    TC* __restrict__ out, int H, int G, int D, int page_size, int tiles_per_split, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
    extern __shared__ float lds[];
    float* q_s = lds;                       // [H][D]
    float* s_raw = q_s + H * D;             // [H][TK]
    float* p_s = s_raw + H * MA_TK;         // [H][TK]
    float* mix_s = p_s + H * MA_TK;         // [H][H] (if mix)
    float* m_s = mix_s + (mix ? H * H : 0); // [H]
    float* l_s = m_s + H;
    float* c_s = l_s + H;
    // per run of 8 keys of a tile: its page and its place in the page; two sets, by the tile's parity (a wave may
    // be at the next tile's products while another still weighs this tile's values)
    int* chunk_s = reinterpret_cast<int*>(c_s + H);      // [2][2][TK / 8]
    const int t = blockIdx.x, split = blockIdx.y, nsplit = gridDim.y;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int pos = positions[t];
    const int32_t* table = block_tables + (size_t)token_req[t] * bt_width;
    const int rep = H / G, HD = H * D;
    const bool own_sink = sink && nsplit == 1;
    for (int i = tid; i < HD; i += MA_THREADS) q_s[i] = to_f32(q[(size_t)t * HD + i]);
    if (mix)
        for (int i = tid; i < H * H; i += MA_THREADS) mix_s[i] = mix[i];
    for (int i = tid; i < H; i += MA_THREADS) {
        m_s[i] = own_sink ? 0.f : -INFINITY;
        l_s[i] = own_sink ? 1.f : 0.f;
    }
    float acc[ACC];
#pragma unroll
    for (int n = 0; n < ACC; ++n) acc[n] = 0.f;
    __syncthreads();
    const MaTiles<MA_TK> tiles(pos, window, keep_first);
    const int i_lo = nsplit == 1 ? 0 : split * tiles_per_split;
    const int i_hi = split == nsplit - 1 ? tiles.n : min(tiles.n, i_lo + tiles_per_split);      // (the last split takes what is left)
    // lanes of a key: a key's row of D elements is read by D / 8 neighbouring lanes, 16 bytes each (where D / 8
    // is a power of two up to 64), so that a wave's load covers whole rows; else a lane reads a key's whole row
    const int lpk = D / 8;
    const bool rows_by_lanes = D % 8 == 0 && lpk <= 64 && (lpk & (lpk - 1)) == 0;
    const int lpk_shift = 31 - __clz(max(lpk, 1));
    const size_t page_elems = (size_t)G * D * page_size;
    for (int ti = i_lo; ti < i_hi; ++ti) {
        const bool first = ti < tiles.n_a;
        const int jt = first ? ti * MA_TK : tiles.jt_b + (ti - tiles.n_a) * MA_TK;
        const int r_lo = first ? 0 : tiles.lo, r_hi = first ? tiles.a_hi : tiles.hi;
        int* chunk = chunk_s + (ti & 1) * (MA_TK / 4);
        if (tid < MA_TK / 8) {
            const int j = jt + tid * 8;
            chunk[tid] = j < r_hi ? table[j / page_size] : 0;       // (no page is looked up past the token's own)
            chunk[MA_TK / 8 + tid] = j % page_size;
        }
        // products of all heads' queries with the tile's keys
        if (rows_by_lanes) {
            const int kpi = 64 >> lpk_shift;           // keys a wave takes at a time
            const int kl = lane >> lpk_shift, dl = lane & (lpk - 1);
            const int its = G << lpk_shift;            // (MA_TK / kpi = lpk rounds a kv head)
            for (int it0 = wv; it0 < its; it0 += MA_WAVES * MA_AHEAD) {
                MaRaw<TC> rows[MA_AHEAD];
#pragma unroll
                for (int a = 0; a < MA_AHEAD; ++a) {
                    const int it = it0 + a * MA_WAVES;
                    const int kvh = it >> lpk_shift, j = jt + (it & (lpk - 1)) * kpi + kl;
                    rows[a].zero();
                    if (it < its && j >= r_lo && j < r_hi) {
                        const int page = table[j / page_size], off = j % page_size;
                        rows[a].load(k_cache + (((size_t)page * G + kvh) * page_size + off) * D + dl * 8);
                    }
                }
#pragma unroll
                for (int a = 0; a < MA_AHEAD; ++a) {
                    const int it = it0 + a * MA_WAVES;
                    if (it >= its) break;
                    const int kvh = it >> lpk_shift, key = (it & (lpk - 1)) * kpi + kl;
                    float kf[8];
                    rows[a].get(kf);
                    for (int g = kvh * rep; g < (kvh + 1) * rep; ++g) {
                        const float4* q4 = reinterpret_cast<const float4*>(q_s + g * D + dl * 8);
                        const float4 qa = q4[0], qb = q4[1];
                        float dot = qa.x * kf[0];
                        dot = fmaf(qa.y, kf[1], dot); dot = fmaf(qa.z, kf[2], dot); dot = fmaf(qa.w, kf[3], dot);
                        dot = fmaf(qb.x, kf[4], dot); dot = fmaf(qb.y, kf[5], dot); dot = fmaf(qb.z, kf[6], dot);
                        dot = fmaf(qb.w, kf[7], dot);
                        for (int o = 1; o < lpk; o <<= 1) dot += __shfl_xor(dot, o, 64);
                        if (dl == 0) s_raw[g * MA_TK + key] = dot;
                    }
                }
            }
        } else {
            const int j = jt + lane;
            const bool vis = j >= r_lo && j < r_hi;
            if (vis) {
                const int page = table[j / page_size], off = j % page_size;
                for (int g = wv; g < H; g += MA_WAVES) {
                    const TC* kr = k_cache + (((size_t)page * G + g / rep) * page_size + off) * D;
                    const float* qg = q_s + g * D;
                    float dot = 0.f;
                    for (int d = 0; d < D; ++d) dot = fmaf(qg[d], to_f32(kr[d]), dot);
                    s_raw[g * MA_TK + lane] = dot;
                }
            } else {
                for (int g = wv; g < H; g += MA_WAVES) s_raw[g * MA_TK + lane] = 0.f;
            }
        }
        __syncthreads();
        // scale, soft cap and the bias of the distance: a lane a key, a wave a head at a time
        {
            const int j = jt + lane;
            const bool vis = j >= r_lo && j < r_hi;
            const int dist = min(pos - j, bias_rows - 1);
            for (int g = wv; g < H; g += MA_WAVES) {
                float sc = 0.f;
                if (vis) {
                    sc = s_raw[g * MA_TK + lane] * scale;
                    if (cap > 0.f) sc = cap * tanhf(sc / cap);
                    if (bias) sc += bias[(size_t)dist * H + g];
                }
                s_raw[g * MA_TK + lane] = sc;
            }
        }
        __syncthreads();
        // the heads' scores mixed; the running maximum and sum of each head, a wave a head
        {
            const int j = jt + lane;
            const bool vis = j >= r_lo && j < r_hi;
            for (int h = wv; h < H; h += MA_WAVES) {
                float sc;
                if (mix) {
                    sc = 0.f;
                    for (int g = 0; g < H; ++g) sc = fmaf(mix_s[h * H + g], s_raw[g * MA_TK + lane], sc);
                } else {
                    sc = s_raw[h * MA_TK + lane];
                }
                if (!vis) sc = -INFINITY;
                const float m_old = m_s[h];
                const float m_new = fmaxf(m_old, wave_max(sc));
                float p = 0.f, corr = 1.f;
                if (m_new > -INFINITY) {
                    p = vis ? expf(sc - m_new) : 0.f;
                    corr = expf(m_old - m_new);
                }
                const float l_new = l_s[h] * corr + wave_sum(p);
                p_s[h * MA_TK + lane] = p;
                if (lane == 0) {
                    m_s[h] = m_new;
                    l_s[h] = l_new;
                    c_s[h] = corr;
                }
            }
        }
        __syncthreads();
        // weighted values: thread -> (head, element) pairs; the tile's runs of 8 keys are asked for four at a time
        {
            const int c_lo = (max(jt, r_lo) - jt) >> 3, c_hi = (min(jt + MA_TK, r_hi) - jt + 7) >> 3;
#pragma unroll
            for (int n = 0; n < ACC; ++n) {
                const int idx = tid + n * MA_THREADS;
                if (idx < HD) {
                    const int h = idx / D;
                    const int voff = ((h / rep) * D + idx % D) * page_size;      // (kv head, element) in a value page
                    float a = acc[n] * c_s[h];
                    const float* ph = p_s + h * MA_TK;
#pragma unroll
                    for (int c0 = 0; c0 < MA_TK / 8; c0 += MA_RUNS) {
                        MaRaw<TC> runs[MA_RUNS];
#pragma unroll
                        for (int c = 0; c < MA_RUNS; ++c) {
                            runs[c].zero();
                            if (c0 + c >= c_lo && c0 + c < c_hi)        // (pages hold a multiple of 8 tokens)
                                runs[c].load(v_cache + (size_t)chunk[c0 + c] * page_elems + chunk[MA_TK / 8 + c0 + c] + voff);
                        }
#pragma unroll
                        for (int c = 0; c < MA_RUNS; ++c) {
                            float vf[8];
                            runs[c].get(vf);
#pragma unroll
                            for (int i = 0; i < 8; ++i) a = fmaf(ph[(c0 + c) * 8 + i], vf[i], a);
                        }
                    }
                    acc[n] = a;
                }
            }
        }
        // (the next tile's scores go to s_raw, which nobody reads any more; its barrier stands
        // between these reads of p_s and the next writes)
    }
    __syncthreads();
    if (nsplit == 1) {
#pragma unroll
        for (int n = 0; n < ACC; ++n) {
            const int idx = tid + n * MA_THREADS;
            if (idx < HD) {
                const float l = l_s[idx / D];
                out[(size_t)t * HD + idx] = from_f32<TC>(l > 0.f ? acc[n] / l : 0.f);
            }
        }
        return;
    }
    if (i_lo < i_hi) {                                   // (the merge reads nothing of a split without tiles)
        float* po = part_o + ((size_t)t * nsplit + split) * HD;
#pragma unroll
        for (int n = 0; n < ACC; ++n) {
            const int idx = tid + n * MA_THREADS;
            if (idx < HD) po[idx] = acc[n];
        }
    }
    float* pm = part_ml + ((size_t)t * nsplit + split) * 2 * H;
    for (int i = tid; i < H; i += MA_THREADS) {
        pm[i] = m_s[i];
        pm[H + i] = l_s[i];
    }
}

// The splits of a token's keys put together: M = max of the maxima (and 0, the sink's score),
// L = [sink] e^-M + sum_s l_s e^(m_s - M), out = sum_s o_s e^(m_s - M) / L.  A block per (token, head), WAVES waves that
// take the splits in turn, MA_MERGE of them asked for at once: one after the other, a split's loads cost a round trip to
// memory each (17 splits: 24 us, so 5).  The order of the additions goes by the number of splits alone.
#define MA_MERGE 8
template <typename TC, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void mixed_attention_merge_kernel(const float* __restrict__ part_o,
                                                                           const float* __restrict__ part_ml, int nsplit,
                                                                           int sink, TC* __restrict__ out, int H, int D) {
    __shared__ float sums[WAVES][64];
    const int t = blockIdx.x / H, h = blockIdx.x % H, HD = H * D;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const float* pm = part_ml + (size_t)t * nsplit * 2 * H + h;
    const float* po = part_o + (size_t)t * nsplit * HD + (size_t)h * D;
    float M = sink ? 0.f : -INFINITY;
    for (int s = lane; s < nsplit; s += 64) M = fmaxf(M, pm[(size_t)s * 2 * H]);
    M = wave_max(M);
    float L = 0.f;
    for (int s = lane; s < nsplit; s += 64) {
        const float m = pm[(size_t)s * 2 * H];
        if (m > -INFINITY) L = fmaf(pm[(size_t)s * 2 * H + H], expf(m - M), L);
    }
    L = wave_sum(L) + (sink ? expf(-M) : 0.f);
    for (int e0 = 0; e0 < D; e0 += 64) {
        const int e = min(e0 + lane, D - 1);
        float a = 0.f;
        for (int s0 = wv; s0 < nsplit; s0 += WAVES * MA_MERGE) {
            float m[MA_MERGE], o[MA_MERGE];
#pragma unroll
            for (int i = 0; i < MA_MERGE; ++i) {
                const int s = min(s0 + i * WAVES, nsplit - 1);
                m[i] = pm[(size_t)s * 2 * H];
                o[i] = po[(size_t)s * HD + e];
            }
#pragma unroll
            for (int i = 0; i < MA_MERGE; ++i)               // (a split without visible keys has left no values)
                if (s0 + i * WAVES < nsplit && m[i] > -INFINITY) a = fmaf(o[i], expf(m[i] - M), a);
        }
        if (WAVES > 1) {
            __syncthreads();
            sums[wv][lane] = a;
            __syncthreads();
            a = sums[0][lane];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) a += sums[w][lane];
        }
        if (wv == 0 && e0 + lane < D) out[(size_t)t * HD + (size_t)h * D + e] = from_f32<TC>(L > 0.f ? a / L : 0.f);
    }
}

// The same for the up to MA_MERGE splits of a prompt's tokens: D / 4 lanes a (token, head), 16 bytes a lane and load, several heads a
// wave and four waves a block.  A wave and block of its own for each head of 1,500 tokens are 48,000 blocks, which are placed no
// faster than some 50 us, whatever they read.  The values are added in the same order.  us, a block a head / now: 1,500 tokens of
// 32 heads of 128 57 / 13.
template <typename TC, int LPH>
__global__ __launch_bounds__(256) void mixed_attention_merge_vec_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                        int nsplit, int sink, TC* __restrict__ out, int pairs, int H) {
    constexpr int D = LPH * 4;
    const int lane = threadIdx.x & 63, e = (lane % LPH) * 4;
    const int id = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / LPH) + lane / LPH;
    if (id >= pairs) return;
    const int t = id / H, h = id - t * H, HD = H * D;
    const float* pm = part_ml + (size_t)t * nsplit * 2 * H + h;
    const float* po = part_o + (size_t)t * nsplit * HD + (size_t)h * D + e;
    float m[MA_MERGE], l[MA_MERGE];
    float4 o[MA_MERGE];
#pragma unroll
    for (int s = 0; s < MA_MERGE; ++s) {
        m[s] = -INFINITY;
        l[s] = 0.f;
        o[s] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (s < nsplit) {
            m[s] = pm[(size_t)s * 2 * H];
            l[s] = pm[(size_t)s * 2 * H + H];
            o[s] = *reinterpret_cast<const float4*>(po + (size_t)s * HD);
        }
    }
    float M = sink ? 0.f : -INFINITY;
#pragma unroll
    for (int s = 0; s < MA_MERGE; ++s) M = fmaxf(M, m[s]);
    float L = sink ? expf(-M) : 0.f;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < MA_MERGE; ++s)
        if (m[s] > -INFINITY) {                          // (a split without visible keys has left no values)
            const float f = expf(m[s] - M);
            L = fmaf(l[s], f, L);
            a.x = fmaf(o[s].x, f, a.x); a.y = fmaf(o[s].y, f, a.y); a.z = fmaf(o[s].z, f, a.z); a.w = fmaf(o[s].w, f, a.w);
        }
    const float4 y = L > 0.f ? make_float4(a.x / L, a.y / L, a.z / L, a.w / L) : make_float4(0.f, 0.f, 0.f, 0.f);
    TC* to = out + (size_t)t * HD + (size_t)h * D + e;
    if constexpr (sizeof(TC) == 4) {
        *reinterpret_cast<float4*>(to) = y;
    } else {
        union { bf16_t b[4]; uint2 u; } pk;
        pk.b[0] = (bf16_t)y.x; pk.b[1] = (bf16_t)y.y; pk.b[2] = (bf16_t)y.z; pk.b[3] = (bf16_t)y.w;
        *reinterpret_cast<uint2*>(to) = pk.u;
    }
}

// (a wave does for the splits of a prompt's blocks, eight at most; a step of few tokens has many splits and few blocks)
template <typename TC>
static int ma_merge(const float* part_o, const float* part_ml, int splits, int sink, void* out, int T, int H, int D, hipStream_t s) {
    if (splits <= MA_MERGE && D >= 16 && D <= 256 && (D & (D - 1)) == 0 && ((uintptr_t)part_o % 16) == 0 && ((uintptr_t)out % 16) == 0) {
        const int pairs = T * H, per = 1024 / D;             // heads a block
        const unsigned blocks = (unsigned)((pairs + per - 1) / per);
#define MA_MERGE_VEC(L) mixed_attention_merge_vec_kernel<TC, L><<<blocks, 256, 0, s>>>(part_o, part_ml, splits, sink, (TC*)out, pairs, H)
        if (D == 16) MA_MERGE_VEC(4);
        else if (D == 32) MA_MERGE_VEC(8);
        else if (D == 64) MA_MERGE_VEC(16);
        else if (D == 128) MA_MERGE_VEC(32);
        else MA_MERGE_VEC(64);
#undef MA_MERGE_VEC
        return tff_check_launch("mixed_attention_merge");
    }
    if (splits <= MA_MERGE)
        mixed_attention_merge_kernel<TC, 1><<<T * H, 64, 0, s>>>(part_o, part_ml, splits, sink, (TC*)out, H, D);
    else
        mixed_attention_merge_kernel<TC, 4><<<T * H, 256, 0, s>>>(part_o, part_ml, splits, sink, (TC*)out, H, D);
    return tff_check_launch("mixed_attention_merge");
}

// ---- bfloat16 on the matrix cores ----
//
// Both kernels below share three steps a tile of keys (borders at multiples of its size from the sequence's start):
//   1. S_g = Q_g K^T per head g: bf16 MFMA 16x16x32 over the head's elements, operands straight from memory (lane (row,
//      quarter) holds 8 consecutive elements of its row); scale and cap on the accumulators; float32 scores to LDS.
//   2. The heads mixed: float32 MFMA 16x16x4, rows the mixed heads, columns sixteen keys of one query, so that a head's
//      keys lie in the sixteen lanes of a row: mask, running maximum and sum follow in registers.
//   3. O_h += P_h V: bf16 MFMA 16x16x32 over 32 keys, values from the transposed pages.
// A wave has the heads of one kv head where it can, so that no other wave fetches that kv head's keys and values.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 ma_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ma_floatx4;

// maximum over the sixteen lanes of a row, in all of them
__device__ __forceinline__ float row16_max(float v) {
#define MA_DPP(x, ctrl) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xF, 0xF, true))
    v = fmaxf(v, MA_DPP(v, 0xB1));       // quad_perm [1, 0, 3, 2]
    v = fmaxf(v, MA_DPP(v, 0x4E));       // quad_perm [2, 3, 0, 1]
    v = fmaxf(v, MA_DPP(v, 0x141));      // row_half_mirror
    v = fmaxf(v, MA_DPP(v, 0x140));      // row_mirror
#undef MA_DPP
    return v;
}

// tanh without branches, by the method of Cephes' tanhf (S. Moshier): up to 0.625 x + x^3 p(x^2), with p fitted here to tanh's relative error
// (4e-9), above it 1 - 2 / (e^2|x| + 1); what is lost in the exponent's argument and in the sum goes into the reciprocal's correction.  At most
// 1.12 units in the last place from 64 bits, 0.33 in the mean between 0.625 and 1 where it is worst (the library's tanhf: 1.36 and 0.34),
// in some 25 instructions instead of 70.  Beyond 20 it is one; NaN stays NaN.
__device__ __forceinline__ float ma_tanh(float x) {
    const float a = fabsf(x), z = x * x;
    float p = fmaf(-0.005704986397176981f, z, 0.02063908614218235f);
    p = fmaf(p, z, -0.05373971536755562f);
    p = fmaf(p, z, 0.13331441581249237f);
    p = fmaf(p, z, -0.3333328068256378f);
    const float small = fmaf(a, z * p, a);
    const float b = a > 20.f ? 20.f : a, hi = b * 2.8853900817779268f;
    const float e = __builtin_amdgcn_exp2f(hi), d = e + 1.f, r = __builtin_amdgcn_rcpf(d);
    const float tail = fmaf(e * 0.6931471805599453f, fmaf(b, 2.8853900817779268f, -hi), e - (d - 1.f));
    const float big = fmaf(-2.f, fmaf(fmaf(-tail, r, fmaf(-d, r, 1.f)), r, r), 1.f);
    return copysignf(a < 0.625f ? small : big, x);
}
// e^x for x <= 0 (NaN stays NaN): the rounding of x / ln 2 goes into a factor of its own.
__device__ __forceinline__ float ma_exp(float x) {
    x = x < -200.f ? -200.f : x;
    const float hi = x * 1.4426950408889634f;
    const float lo = fmaf(x, 1.4426950408889634f, -hi) + x * 1.9259629911266175e-8f;
    const float e = __builtin_amdgcn_exp2f(hi);
    return fmaf(e, lo * 0.6931471805599453f, e);
}

// Eight values of keys j .. j + 7 with those outside [lo, hi) as zero: a slot that holds no visible key holds anything, and
// its weight of zero does not make a product with a NaN vanish.
__device__ __forceinline__ ma_bf16x8 ma_visible(ma_bf16x8 v, int j, int lo, int hi) {
    if (j < lo || j + 8 > hi) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = j + i >= lo && j + i < hi ? v[i] : (bf16_t)0.f;
    }
    return v;
}

// Eight values with those that are not finite as zero.
__device__ __forceinline__ ma_bf16x8 ma_finite(ma_bf16x8 v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = fabsf((float)v[i]) < INFINITY ? v[i] : (bf16_t)0.f;
    return v;
}

#define Q16_THREADS 512
#define Q16_WAVES 8
#define Q16_TK 64        // keys a tile
#define Q16_DIST 80      // distances between a tile's keys and the block's queries (79), in blocks of sixteen

// Prompts: a block takes up to 16 consecutive tokens of one request (a work item: first token, count) and all heads.
// The results and a tile's operands fill the registers and the scores LDS, hence one block of eight waves a CU with 64 keys a
// tile: the scores of
// 16 queries, 32 heads and 64 keys are 128 KB of LDS, a barrier is paid once in 64 keys, and a lane of step 2 holds four
// neighbouring keys (column c of the mixing's product kb is key 4 c + kb), so that scores and weights go through LDS in
// pieces of 16 and 8 bytes.  Scores lie as [query][head][key], a row's pieces moved by the query (Q16_PIECE), since step 1
// writes sixteen queries of one head and step 2 reads four heads of one query at a time.  A query's weights (bfloat16)
// replace its own scores: the same wave reads the ones and writes the others.  The biases are mixed once a tile, by
// distance, and are what the mixing's products start from: straight from the table, a head's biases of a tile are a cache
// line each.  32 heads of 128 on 8 kv heads under a window of 1,024, us a call with its merge, against tiles of 16 keys mixed
// by the vector unit: 300 tokens 86 -> 44, 1,500 659 -> 269, 4,000 1,261 -> 456; 16 heads, 1,500 tokens 259 -> 155.  What is
// left is half the fetching of queries and keys, a third the softmax.
#define Q16_PIECE(p, qq) ((p) ^ ((qq) & 7))
// (one head, one run of keys after the other: worked on at once, they take more registers than there are beside the results)
#define Q16_IN_TURN __builtin_amdgcn_sched_barrier(0)
#define LOG2E 1.4426950408889634f

// the larger of two, a NaN passed over (fmaxf quiets every operand first, an instruction each)
__device__ __forceinline__ float ma_max(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }

// ONE_KV: a wave's heads have one kv head, whose keys and values it fetches once.
template <int HPW, int EB, bool ONE_KV>
__global__ __launch_bounds__(Q16_THREADS) void mixed_attention_q16_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int bt_width, const int32_t* __restrict__ token_req,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ work, const float* __restrict__ bias,
    int bias_rows, const float* __restrict__ mix, float scale, float cap, int window, int keep_first, int sink,
    bf16_t* __restrict__ out, int H, int G, int page_size, int tiles_per_split, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
    constexpr int D = EB * 16, KC = D / 32, HP = HPW * Q16_WAVES, HB = HPW == 4 ? 2 : 1, KS = HP / 4;
    constexpr int BROW = HB * 16 + 4;
    __shared__ __attribute__((aligned(16))) float s_s[16 * HP * Q16_TK];
    __shared__ __attribute__((aligned(16))) float bias_s[Q16_DIST * BROW];          // [distance][mixed head]
    __shared__ __attribute__((aligned(16))) float m_s[16 * HP], l_s[16 * HP];       // [query][head]
    __shared__ __attribute__((aligned(16))) float c_s[HP * 16];                     // [head][query]
    __shared__ float mix_s[HB * KS * 64];
    const int t0 = work[2 * blockIdx.x], n = work[2 * blockIdx.x + 1];
    const int split = blockIdx.y, nsplit = gridDim.y;
    const bool own_sink = sink && nsplit == 1;       // (with several splits the merge adds the sink's term)
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, g4 = lane >> 4;
    const int pos0 = positions[t0], pos_last = pos0 + n - 1;
    const int32_t* table = block_tables + (size_t)token_req[t0] * bt_width;
    const int rep = H / G, HD = H * D;
    const float scale_in = cap > 0.f ? scale / cap : scale;
    for (int i = tid; i < 16 * HP; i += Q16_THREADS) {
        m_s[i] = own_sink ? 0.f : -INFINITY;
        l_s[i] = own_sink ? 1.f : 0.f;
    }
    if (H < HP)                                      // rows of no head: their weight in the mixing is zero, they are too
        for (int i = tid; i < 16 * (HP - H) * Q16_TK; i += Q16_THREADS) {
            const int qq = i / ((HP - H) * Q16_TK), r = i % ((HP - H) * Q16_TK);
            s_s[(qq * HP + H) * Q16_TK + r] = 0.f;
        }
    // the mixing's left operands, mixed head (row) by head (a lane's quarter and the step), as step 2 asks for them
    for (int i = tid; i < HB * KS * 64; i += Q16_THREADS) {
        const int h = i / (KS * 64) * 16 + (i & 15), g = (i / 64) % KS * 4 + (i >> 4 & 3);
        mix_s[i] = mix && h < H && g < H ? mix[h * H + g] : 0.f;
    }
    ma_floatx4 oacc[HPW][EB];
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh)
#pragma unroll
        for (int eb = 0; eb < EB; ++eb) oacc[hh][eb] = ma_floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16_t* qrow = q + (size_t)(t0 + min(col, n - 1)) * HD + g4 * 8;
    const size_t page_elems = (size_t)G * D * page_size;
    const int lo_first = window > 0 ? max(0, pos0 - window + 1) : 0;
    const int lo_last = window > 0 ? max(0, pos_last - window + 1) : 0;
    const int h_lo = wv * HPW;
    __syncthreads();

    auto tile = [&](int jt) {
        // (what follows from the lane and the wave is worked out again in every tile: kept, it costs the registers the values need)
        int ln = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        asm volatile("" : "+v"(ln), "+s"(w));
        const int lane = ln & 63, wv = w & 7, col = lane & 15, g4 = lane >> 4, h_lo = wv * HPW;
        // sixteen keys that some query sees (no page is looked up for others), and where they lie
        auto on = [&](int j0) { return j0 <= pos_last && (window <= 0 || j0 + 15 >= lo_first || j0 < keep_first); };
        auto base = [&](int j0) { return on(j0) ? (size_t)table[j0 / page_size] * page_elems : 0; };
        // 1. scores
        if (bias && wv < Q16_DIST / 16) {                     // sixteen distances a wave
            const int dl = wv * 16 + col;
            const float* brow = bias + (size_t)min(max(pos0 - jt - (Q16_TK - 1) + dl, 0), bias_rows - 1) * H;
            ma_floatx4 mb[HB];
#pragma unroll
            for (int hb = 0; hb < HB; ++hb) mb[hb] = ma_floatx4{0.f, 0.f, 0.f, 0.f};
            if (mix) {
                float b[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) b[ks] = ks * 4 + g4 < H ? brow[ks * 4 + g4] : 0.f;
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int hb = 0; hb < HB; ++hb) mb[hb] = __builtin_amdgcn_mfma_f32_16x16x4f32(mix_s[(hb * KS + ks) * 64 + lane], b[ks], mb[hb], 0, 0, 0);
            } else {
#pragma unroll
                for (int hb = 0; hb < HB; ++hb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) mb[hb][i] = brow[min(hb * 16 + g4 * 4 + i, H - 1)];
            }
#pragma unroll
            for (int hb = 0; hb < HB; ++hb) *reinterpret_cast<ma_floatx4*>(bias_s + dl * BROW + hb * 16 + g4 * 4) = mb[hb];
        }
        {
            int ln2 = lane;
            asm volatile("" : "+v"(ln2));
            const int col = ln2 & 15, g4 = ln2 >> 4 & 3;
            ma_bf16x8 kf[4][KC], qf[KC];
#pragma unroll
            for (int hh = 0; hh < HPW; ++hh) {
                const int h = h_lo + hh;
                if (h < H) {
                    if (hh == 0 || !ONE_KV) {
#pragma unroll
                        for (int kb = 0; kb < 4; ++kb) {
                            const int j0 = jt + kb * 16;
                            const bf16_t* krow = k_cache + base(j0) + ((size_t)(h / rep) * page_size + j0 % page_size + col) * D + g4 * 8;
                            if (on(j0)) {
#pragma unroll
                                for (int kc = 0; kc < KC; ++kc) kf[kb][kc] = *reinterpret_cast<const ma_bf16x8*>(krow + kc * 32);
                            }
                        }
                    }
                    // (a tile's keys are held and the queries fetched once: all blocks' queries of an XCD fill its L2)
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc) qf[kc] = *reinterpret_cast<const ma_bf16x8*>(qrow + h * D + kc * 32);
#pragma unroll
                    for (int kb = 0; kb < 4; ++kb) {
                        if (!on(jt + kb * 16)) continue;
                        ma_floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int kc = 0; kc < KC; ++kc) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][kc], qf[kc], acc, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; ++i)          // (key g4 * 4 + i, query col)
                            acc[i] = cap > 0.f ? cap * ma_tanh(acc[i] * scale_in) : acc[i] * scale_in;
                        *reinterpret_cast<ma_floatx4*>(s_s + (col * HP + h) * Q16_TK + Q16_PIECE(kb * 4 + g4, col) * 4) = acc;
                    }
                }
            }
        }
        __syncthreads();
        // 2. two queries a wave: lane (quarter g4, col) has mixed heads hb * 16 + g4 * 4 + i of keys kb * 16 + col
#pragma unroll 1
        for (int q2 = 0; q2 < 2; ++q2) {
            int ln2 = lane;
            asm volatile("" : "+v"(ln2));
            const int lane = ln2 & 63, col = lane & 15, g4 = lane >> 4;
            const int qq = wv * 2 + q2, posq = pos0 + qq;
            if (qq >= n) {                                    // (a query that the block does not have: weights of zero)
                uint4* z = reinterpret_cast<uint4*>(s_s + qq * HP * Q16_TK);
                for (int i = lane; i < HP * Q16_TK / 8; i += 64) z[i] = make_uint4(0, 0, 0, 0);
                for (int i = lane; i < HP; i += 64) c_s[i * 16 + qq] = 1.f;
                continue;
            }
            // lane (quarter g4, col): mixed heads hb * 16 + g4 * 4 + i of keys 4 col + kb
            ma_floatx4 sm[4][HB];
            const float* scores = s_s + qq * HP * Q16_TK + Q16_PIECE(col, qq) * 4;
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int hb = 0; hb < HB; ++hb)
                    sm[kb][hb] = bias ? *reinterpret_cast<const ma_floatx4*>(bias_s + (qq + Q16_TK - 1 - col * 4 - kb) * BROW + hb * 16 + g4 * 4)
                                      : ma_floatx4{0.f, 0.f, 0.f, 0.f};
            if (mix) {
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const ma_floatx4 b = *reinterpret_cast<const ma_floatx4*>(scores + (ks * 4 + g4) * Q16_TK);
#pragma unroll
                    for (int hb = 0; hb < HB; ++hb) {
                        const float a = mix_s[(hb * KS + ks) * 64 + lane];
#pragma unroll
                        for (int kb = 0; kb < 4; ++kb) sm[kb][hb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[kb], sm[kb][hb], 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int hb = 0; hb < HB; ++hb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const ma_floatx4 b = *reinterpret_cast<const ma_floatx4*>(scores + min(hb * 16 + g4 * 4 + i, HP - 1) * Q16_TK);
#pragma unroll
                        for (int kb = 0; kb < 4; ++kb) sm[kb][hb][i] += b[kb];
                    }
            }
            asm volatile("" ::: "memory");                    // (the weights go where these scores were)
            const int j_last = jt + Q16_TK - 1;
            if (!(j_last <= posq && (window <= 0 || posq - jt < window || j_last < keep_first))) {
#pragma unroll
                for (int kb = 0; kb < 4; ++kb) {
                    const int j = jt + col * 4 + kb;
                    const bool vis = j <= posq && (window <= 0 || posq - j < window || j < keep_first);
#pragma unroll
                    for (int hb = 0; hb < HB; ++hb)
#pragma unroll
                        for (int i = 0; i < 4; ++i) sm[kb][hb][i] = vis ? sm[kb][hb][i] : -INFINITY;
                }
            }
#pragma unroll
            for (int hb = 0; hb < HB; ++hb) {
                const int h0 = hb * 16 + g4 * 4;
                if (h0 < HP) {
                    const ma_floatx4 m_old = *reinterpret_cast<const ma_floatx4*>(m_s + qq * HP + h0);
                    ma_floatx4 l = *reinterpret_cast<const ma_floatx4*>(l_s + qq * HP + h0), m_new;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        Q16_IN_TURN;
                        const float mx = row16_max(ma_max(ma_max(ma_max(sm[0][hb][i], sm[1][hb][i]), ma_max(sm[2][hb][i], sm[3][hb][i])), m_old[i]));
                        // (nothing visible yet: weights of zero.  Differences are what is scaled: a maximum of its own scaled would be
                        // rounded, so that results kept from tile to tile drift, and the lowest number there is would overflow)
                        const float from = mx > -INFINITY ? mx : 0.f;
                        union { bf16_t h[4]; uint2 u; } p;
                        float sum = 0.f;
#pragma unroll
                        for (int kb = 0; kb < 4; ++kb) {
                            // (the sum takes the weights as the product will see them)
                            p.h[kb] = (bf16_t)__builtin_amdgcn_exp2f((sm[kb][hb][i] - from) * LOG2E);
                            sum += (float)p.h[kb];
                        }
                        *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(s_s + qq * HP * Q16_TK) + (h0 + i) * Q16_TK
                                                  + Q16_PIECE(col >> 1, qq) * 8 + (col & 1) * 4) = p.u;
                        const float corr = __builtin_amdgcn_exp2f((m_old[i] - from) * LOG2E);
                        m_new[i] = mx;
                        l[i] = fmaf(l[i], corr, row16_sum(sum));
                        if (col == 0) c_s[(h0 + i) * 16 + qq] = corr;
                    }
                    if (col == 0) {
                        *reinterpret_cast<ma_floatx4*>(m_s + qq * HP + h0) = m_new;
                        *reinterpret_cast<ma_floatx4*>(l_s + qq * HP + h0) = l;
                    }
                }
            }
        }
        __syncthreads();
        // 3. weighted values; where the wave's heads share a kv head its values are fetched once for all of them
        const bool on_first = on(jt) || on(jt + 16);
#pragma unroll 1
        for (int kk = 0; kk < 2; ++kk) {
            const bool on2[2] = {on(jt + kk * 32), on(jt + kk * 32 + 16)};
            if (!on2[0] && !on2[1]) continue;
            int ln2 = lane;
            asm volatile("" : "+v"(ln2));
            const int col = ln2 & 15, g4 = ln2 >> 4 & 3;
            const int j = jt + kk * 32 + g4 * 8;              // the lane's eight keys
            const bool live = g4 < 2 ? on2[0] : on2[1];
            const size_t vbase = (g4 < 2 ? base(jt + kk * 32) : base(jt + kk * 32 + 16)) + (size_t)col * page_size + j % page_size;
            const ma_bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
            ma_bf16x8 vb[EB];
#pragma unroll
            for (int hh = 0; hh < HPW; ++hh) {
                const int h = h_lo + hh;
                if (h < H) {
                    if (hh == 0 || !ONE_KV) {
                        const bf16_t* vhead = v_cache + vbase + (size_t)(h / rep) * D * page_size;
#pragma unroll
                        for (int e = 0; e < EB; ++e) vb[e] = live ? *reinterpret_cast<const ma_bf16x8*>(vhead + (size_t)e * 16 * page_size) : zero;
                        if (jt + kk * 32 + 32 > pos_last + 1) {
#pragma unroll
                            for (int e = 0; e < EB; ++e) vb[e] = ma_visible(vb[e], j, 0, pos_last + 1);
                        }
                    }
                    const ma_bf16x8 pa = *reinterpret_cast<const ma_bf16x8*>(reinterpret_cast<const bf16_t*>(s_s + col * HP * Q16_TK) + h * Q16_TK
                                                                              + Q16_PIECE(kk * 4 + g4, col) * 8);
                    if (kk == 0 || !on_first) {
                        const float4 cr = *reinterpret_cast<const float4*>(c_s + h * 16 + g4 * 4);
#pragma unroll
                        for (int e = 0; e < EB; ++e) {
                            oacc[hh][e][0] *= cr.x;
                            oacc[hh][e][1] *= cr.y;
                            oacc[hh][e][2] *= cr.z;
                            oacc[hh][e][3] *= cr.w;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < EB; ++e) oacc[hh][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, vb[e], oacc[hh][e], 0, 0, 0);
                    Q16_IN_TURN;
                }
            }
        }
        __syncthreads();
    };

    // the block's tiles, numbered through: those of the kept first tokens before the windows, then the windows'
    const int jt_b = lo_first / Q16_TK * Q16_TK;
    const int n_a = (min(min(keep_first, lo_last), jt_b) + Q16_TK - 1) / Q16_TK;
    const int tiles = n_a + (pos_last - jt_b) / Q16_TK + 1;
    const int i_lo = nsplit == 1 ? 0 : split * tiles_per_split;
    const int i_hi = split == nsplit - 1 ? tiles : min(tiles, i_lo + tiles_per_split);      // (the last split takes what is left)
    for (int ti = i_lo; ti < i_hi; ++ti) tile(ti < n_a ? ti * Q16_TK : jt_b + (ti - n_a) * Q16_TK);
#pragma unroll
    for (int hh = 0; hh < HPW; ++hh) {
        const int h = h_lo + hh;
        if (h < H) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int qq = g4 * 4 + i;
                if (qq < n) {
                    if (nsplit == 1) {
                        const float l = l_s[qq * HP + h];
                        const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
                        for (int eb = 0; eb < EB; ++eb)
                            out[(size_t)(t0 + qq) * HD + h * D + eb * 16 + col] = (bf16_t)(oacc[hh][eb][i] * inv);
                    } else if (i_lo < i_hi) {                 // (the merge reads nothing of a split without tiles)
                        float* po = part_o + ((size_t)(t0 + qq) * nsplit + split) * HD + h * D + col;
#pragma unroll
                        for (int eb = 0; eb < EB; ++eb) po[eb * 16] = oacc[hh][eb][i];
                    }
                }
            }
        }
    }
    if (nsplit > 1) {
        // (maximum and sum per head and query, in the merge's layout: [token][split][maxima of the heads | sums])
        const int h = tid >> 4, qq = tid & 15;
        if (h < H && qq < n) {
            float* pm = part_ml + ((size_t)(t0 + qq) * nsplit + split) * 2 * H;
            pm[h] = m_s[qq * HP + h];
            pm[H + h] = l_s[qq * HP + h];
        }
    }
}

#define FEW_TK 32        // keys a tile of a block with one token: the contraction of one MFMA over the values

// Decoding and short portions: a block per token and split of its keys, eight waves, each the kv heads wv, wv + 8, ...
// What bounds it is latency (a token's 1,000 keys are 4 MB, read in under a microsecond by all CUs), so a tile is as small as
// the values' MFMA allows and spread over as many blocks, and its keys and values are all asked for at once.  A kv
// head's query heads are the columns of the scores' product and the rows of the values'.  The weights stay exact: a float32
// weight is the sum of three bfloat16 (8 + 8 + 8 bits), and each takes an MFMA of its own.  32 heads of 128 on 8 kv heads, window
// 1,024, us a call with its merge, against products by the vector unit: one token of 1,500 79 -> 16, six 91 -> 18, 48 273 -> 69;
// of 60 keys 60 -> 12.
template <int GPW, int EB>
__global__ __launch_bounds__(Q16_THREADS) void mixed_attention_few_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int bt_width, const int32_t* __restrict__ token_req,
    const int32_t* __restrict__ positions, const float* __restrict__ bias, int bias_rows,
    const float* __restrict__ mix, float scale, float cap, int window, int keep_first, int sink,
    bf16_t* __restrict__ out, int H, int G, int page_size, int tiles_per_split, float* __restrict__ part_o,
    float* __restrict__ part_ml) {
    constexpr int D = EB * 16, KC = D / 32, SROW = FEW_TK + 16;     // (four heads' rows of a step of the mixing lie in different banks)
    __shared__ __attribute__((aligned(16))) float s_s[32 * SROW];
    __shared__ __attribute__((aligned(16))) bf16_t p_s[3][32 * FEW_TK];
    __shared__ float m_s[32], l_s[32], c_s[32];
    __shared__ int again;
    const int t = blockIdx.x, split = blockIdx.y, nsplit = gridDim.y;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 15, g4 = lane >> 4;
    const int pos = positions[t], rep = H / G, HD = H * D;
    const float scale_in = cap > 0.f ? scale / cap : scale;
    const int32_t* table = block_tables + (size_t)token_req[t] * bt_width;
    const bool own_sink = sink && nsplit == 1;
    const MaTiles<FEW_TK> tiles(pos, window, keep_first);
    const int i_lo = nsplit == 1 ? 0 : split * tiles_per_split;
    const int i_hi = split == nsplit - 1 ? tiles.n : min(tiles.n, i_lo + tiles_per_split);      // (the last split takes what is left)
    for (int i = tid; i < (32 - H) * SROW; i += Q16_THREADS) s_s[H * SROW + i] = 0.f;      // rows of no head
    const size_t page_elems = (size_t)G * D * page_size;
    float mixf[8];
    if (wv < 2) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const int h = wv * 16 + col, g = ks * 4 + g4;
            mixf[ks] = mix && h < H && g < H ? mix[h * H + g] : 0.f;
        }
    }
    ma_floatx4 oacc[GPW][EB];
    const ma_bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    if (tid == 0) again = 0;
    // finite_only: the weights' second and third terms meet values that are not finite as zero (below)
    for (bool finite_only = false;; finite_only = true) {
        if (tid < 32) {
            m_s[tid] = own_sink ? 0.f : -INFINITY;
            l_s[tid] = own_sink ? 1.f : 0.f;
        }
#pragma unroll
        for (int gg = 0; gg < GPW; ++gg)
#pragma unroll
            for (int eb = 0; eb < EB; ++eb) oacc[gg][eb] = ma_floatx4{0.f, 0.f, 0.f, 0.f};
        __syncthreads();
        for (int ti = i_lo; ti < i_hi; ++ti) {
            const bool first = ti < tiles.n_a;
            const int jt = first ? ti * FEW_TK : tiles.jt_b + (ti - tiles.n_a) * FEW_TK;
            const int r_lo = first ? 0 : tiles.lo, r_hi = first ? tiles.a_hi : tiles.hi;
            // the lane's places: keys jt + col and jt + 16 + col for the scores, jt + g4 * 8 and the seven after it for the values
            // (no page is looked up for keys the token does not see)
            const int j8 = jt + g4 * 8;
            const bool live = j8 < r_hi && j8 + 8 > r_lo;
            const size_t vbase = live ? (size_t)table[j8 / page_size] * page_elems + j8 % page_size + (size_t)col * page_size : 0;
            size_t kbase[2];
            bool kon[2];
#pragma unroll
            for (int k2 = 0; k2 < 2; ++k2) {
                const int j = jt + k2 * 16 + col;
                kon[k2] = j >= r_lo && j < r_hi;
                kbase[k2] = kon[k2] ? (size_t)table[j / page_size] * page_elems + (size_t)(j % page_size) * D + g4 * 8 : 0;
            }
            ma_bf16x8 vb[GPW == 1 ? EB : 1];
#pragma unroll 1
            for (int gg = 0; gg < GPW; ++gg) {
                const int kvh = wv + gg * Q16_WAVES;
                if (kvh < G) {
                    ma_bf16x8 kf[2][KC], qf[KC];
                    const int h = kvh * rep + col;
#pragma unroll
                    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
                        for (int kc = 0; kc < KC; ++kc)
                            kf[k2][kc] = kon[k2] ? *reinterpret_cast<const ma_bf16x8*>(k_cache + kbase[k2] + (size_t)kvh * page_size * D + kc * 32) : zero;
#pragma unroll
                    for (int kc = 0; kc < KC; ++kc)
                        qf[kc] = col < rep ? *reinterpret_cast<const ma_bf16x8*>(q + (size_t)t * HD + (size_t)h * D + kc * 32 + g4 * 8) : zero;
                    float bf[2][4];
#pragma unroll
                    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            bf[k2][i] = bias && col < rep ? bias[(size_t)min(max(pos - (jt + k2 * 16 + g4 * 4 + i), 0), bias_rows - 1) * H + h] : 0.f;
                    if (GPW == 1) {
#pragma unroll
                        for (int e = 0; e < (GPW == 1 ? EB : 1); ++e)
                            vb[e] = live ? *reinterpret_cast<const ma_bf16x8*>(v_cache + vbase + ((size_t)kvh * D + e * 16) * page_size) : zero;
                    }
#pragma unroll
                    for (int k2 = 0; k2 < 2; ++k2) {
                        ma_floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int kc = 0; kc < KC; ++kc) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[k2][kc], qf[kc], acc, 0, 0, 0);
                        if (col < rep) {                          // (keys g4 * 4 + i, head col)
                            float sc[4];
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                sc[i] = acc[i] * scale_in;
                                if (cap > 0.f) sc[i] = cap * ma_tanh(sc[i]);
                                sc[i] += bf[k2][i];
                            }
                            *reinterpret_cast<float4*>(s_s + h * SROW + k2 * 16 + g4 * 4) = make_float4(sc[0], sc[1], sc[2], sc[3]);
                        }
                    }
                }
            }
            __syncthreads();
            if (wv < 2 && wv * 16 < H) {                          // sixteen mixed heads a wave: lane (quarter g4, col) has wv * 16 + g4 * 4 + i of keys col, 16 + col
                ma_floatx4 sm[2];
                bool vis[2];
#pragma unroll
                for (int k2 = 0; k2 < 2; ++k2) {
                    const int j = jt + k2 * 16 + col;
                    vis[k2] = j >= r_lo && j < r_hi;
                    sm[k2] = ma_floatx4{0.f, 0.f, 0.f, 0.f};
                    if (mix) {
#pragma unroll
                        for (int ks = 0; ks < 8; ++ks)
                            sm[k2] = __builtin_amdgcn_mfma_f32_16x16x4f32(mixf[ks], s_s[(ks * 4 + g4) * SROW + k2 * 16 + col], sm[k2], 0, 0, 0);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) sm[k2][i] = s_s[(wv * 16 + g4 * 4 + i) * SROW + k2 * 16 + col];
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int h = wv * 16 + g4 * 4 + i;
                    const float m_old = m_s[h];
                    float mx = m_old;
#pragma unroll
                    for (int k2 = 0; k2 < 2; ++k2)
                        if (vis[k2]) mx = fmaxf(mx, sm[k2][i]);
                    mx = row16_max(mx);
                    const float corr = mx > -INFINITY ? expf(m_old - mx) : 1.f;
                    const float from = mx > -INFINITY ? mx : 0.f;      // (no key has a weight yet: weights of zero)
                    float sum = 0.f;
#pragma unroll
                    for (int k2 = 0; k2 < 2; ++k2) {
                        const float p = vis[k2] ? ma_exp(sm[k2][i] - from) : 0.f;
                        sum += p;
                        const bf16_t p1 = (bf16_t)p;
                        const float r1 = p - (float)p1;
                        const bf16_t p2 = (bf16_t)r1;
                        const int at = h * FEW_TK + k2 * 16 + col;
                        p_s[0][at] = p1;
                        p_s[1][at] = p2;
                        p_s[2][at] = (bf16_t)(r1 - (float)p2);
                    }
                    sum = row16_sum(sum);
                    if (col == 0) {
                        m_s[h] = mx;
                        l_s[h] = l_s[h] * corr + sum;
                        c_s[h] = corr;
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int gg = 0; gg < GPW; ++gg) {
                const int kvh = wv + gg * Q16_WAVES;
                if (kvh < G) {
                    ma_bf16x8 pa[3];
#pragma unroll
                    for (int s = 0; s < 3; ++s)
                        pa[s] = col < rep ? *reinterpret_cast<const ma_bf16x8*>(&p_s[s][(kvh * rep + col) * FEW_TK + g4 * 8]) : zero;
                    float cr[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) cr[i] = g4 * 4 + i < rep ? c_s[kvh * rep + g4 * 4 + i] : 1.f;
#pragma unroll
                    for (int e = 0; e < EB; ++e) {
                        ma_bf16x8 v = GPW == 1 ? vb[GPW == 1 ? e : 0]
                                               : (live ? *reinterpret_cast<const ma_bf16x8*>(v_cache + vbase + ((size_t)kvh * D + e * 16) * page_size) : zero);
                        v = ma_visible(v, j8, r_lo, r_hi);
#pragma unroll
                        for (int i = 0; i < 4; ++i) oacc[gg][e][i] *= cr[i];
                        const ma_bf16x8 vf = finite_only ? ma_finite(v) : v;
#pragma unroll
                        for (int s = 2; s >= 0; --s) oacc[gg][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[s], s ? vf : v, oacc[gg][e], 0, 0, 0);
                    }
                }
            }
            // (the next tile's scores go to s_s, which nobody reads any more; its first barrier stands between these reads of
            // p_s and c_s and their next writes)
        }
        // A term of zero or of the other sign makes NaN of an infinite value, whose product with the whole weight is infinite.  Values
        // are seldom infinite, so that is looked for in the results, and the block's keys are then worked through once more.
        float sum = 0.f;
#pragma unroll
        for (int gg = 0; gg < GPW; ++gg)
#pragma unroll
            for (int eb = 0; eb < EB; ++eb)
#pragma unroll
                for (int i = 0; i < 4; ++i) sum = fmaf(0.f, oacc[gg][eb][i], sum);
        if (sum != 0.f) again = 1;
        __syncthreads();
        if (!again || finite_only) break;
    }
#pragma unroll
    for (int gg = 0; gg < GPW; ++gg) {
        const int kvh = wv + gg * Q16_WAVES;
        if (kvh < G) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = g4 * 4 + i, h = kvh * rep + row;
                if (row < rep) {
                    if (nsplit == 1) {
                        const float l = l_s[h];
#pragma unroll
                        for (int e = 0; e < EB; ++e)
                            out[(size_t)t * HD + (size_t)h * D + e * 16 + col] = (bf16_t)(l > 0.f ? oacc[gg][e][i] / l : 0.f);
                    } else if (i_lo < i_hi) {                 // (the merge reads nothing of a split without tiles)
                        float* po = part_o + ((size_t)t * nsplit + split) * HD + (size_t)h * D + col;
#pragma unroll
                        for (int e = 0; e < EB; ++e) po[e * 16] = oacc[gg][e][i];
                    }
                }
            }
        }
    }
    if (nsplit > 1 && tid < H) {
        float* pm = part_ml + ((size_t)t * nsplit + split) * 2 * H;
        pm[tid] = m_s[tid];
        pm[H + tid] = l_s[tid];
    }
}

// bfloat16, up to 32 heads of 32, 64 or 128 elements, pages of a multiple of 16 tokens.
TFF_API int tff_mixed_attention_q16_supported(int H, int D, int page_size, int has_mix) {
    (void)has_mix;
    return H > 0 && H <= 32 && (D == 32 || D == 64 || D == 128) && page_size % 16 == 0;
}

// work: int32 [items][2] = (first token of the step, count <= 16), the tokens of an item consecutive tokens of one
// request; every one of the step's T tokens lies in one item.  splits > 1: an item's tiles of 64 keys are dealt to
// `splits` blocks, tiles_per_split each, and merged as tff_mixed_attention's are (the same workspace size).
TFF_API int tff_mixed_attention_q16(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                                    int bt_width, const int32_t* token_req, const int32_t* positions, const int32_t* work,
                                    int items, const float* bias, int bias_rows, const float* mix, float scale, float cap,
                                    int window, int keep_first, int sink, void* out, int T, int H, int G, int D,
                                    int page_size, int splits, int tiles_per_split, float* workspace, tff_stream_t stream) {
    TFF_REQUIRE(q && k_cache && v_cache && block_tables && token_req && positions && work && out,
                "mixed_attention_q16: null pointer");
    TFF_REQUIRE(splits >= 1 && splits <= 65535 && (splits == 1 || (tiles_per_split >= 1 && workspace)),
                "mixed_attention_q16: %d splits of %d tiles", splits, tiles_per_split);
    TFF_REQUIRE(G > 0 && H % G == 0 && bt_width > 0 && tff_mixed_attention_q16_supported(H, D, page_size, mix != nullptr),
                "mixed_attention_q16: %d heads of %d on %d kv heads, pages of %d", H, D, G, page_size);
    TFF_REQUIRE(!bias || bias_rows > 0, "mixed_attention_q16: a bias table without rows");
    TFF_REQUIRE(window >= 0 && keep_first >= 0 && items >= 0, "mixed_attention_q16: negative sizes");
    if (items == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int hpw = (H + Q16_WAVES - 1) / Q16_WAVES;
    float* part_o = workspace;
    float* part_ml = workspace ? workspace + (size_t)T * splits * H * D : nullptr;
#define Q16_LAUNCH(HPW, EB, ONE)                                                                                     \
    mixed_attention_q16_kernel<HPW, EB, ONE><<<dim3(items, splits), Q16_THREADS, 0, s>>>(                              \
        (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_width, token_req,       \
        positions, work, bias, bias_rows, mix, scale, cap, window, keep_first, sink, (bf16_t*)out, H, G, page_size, \
        tiles_per_split, part_o, part_ml)
#define Q16_BY_EB(HPW, ONE)                   \
    do {                                      \
        if (D == 32) Q16_LAUNCH(HPW, 2, ONE); \
        else if (D == 64) Q16_LAUNCH(HPW, 4, ONE); \
        else Q16_LAUNCH(HPW, 8, ONE);         \
    } while (0)
    const int rep = H / G;
    if (hpw <= 1) Q16_BY_EB(1, true);
    else if (hpw <= 2 && rep % 2 == 0) Q16_BY_EB(2, true);
    else if (hpw <= 2) Q16_BY_EB(2, false);
    else if (rep % 4 == 0) Q16_BY_EB(4, true);
    else Q16_BY_EB(4, false);
#undef Q16_BY_EB
#undef Q16_LAUNCH
    int rc = tff_check_launch("mixed_attention_q16");
    if (rc || splits <= 1) return rc;
    return ma_merge<bf16_t>(part_o, part_ml, splits, sink, out, T, H, D, s);
}

static size_t ma_lds_bytes(int H, int D, bool mix) {
    return sizeof(float) * ((size_t)H * D + 2 * (size_t)H * MA_TK + (mix ? (size_t)H * H : 0) + 3 * (size_t)H + MA_TK / 2);
}

TFF_API int tff_mixed_attention_supported(int H, int D, int has_mix) {
    return H > 0 && D > 0 && (size_t)H * D <= 8 * MA_THREADS && ma_lds_bytes(H, D, has_mix != 0) <= 64 * 1024;
}

// Floats of workspace that `splits` splits of T tokens need (0 for one split).
TFF_API size_t tff_mixed_attention_workspace_bytes(int T, int H, int D, int splits) {
    return splits <= 1 ? 0 : sizeof(float) * (size_t)T * splits * ((size_t)H * D + 2 * (size_t)H);
}

template <typename TC>
static int ma_launch(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables, int bt_width,
                     const int32_t* token_req, const int32_t* positions, const float* bias, int bias_rows, const float* mix,
                     float scale, float cap, int window, int keep_first, int sink, void* out, int T, int H, int G, int D,
                     int page_size, int splits, int tiles_per_split, float* ws, hipStream_t s) {
    const size_t lds = ma_lds_bytes(H, D, mix != nullptr);
    const int per = (H * D + MA_THREADS - 1) / MA_THREADS;
    float* part_o = ws;
    float* part_ml = ws ? ws + (size_t)T * splits * H * D : nullptr;
    const dim3 grid(T, splits);
#define MA_LAUNCH(ACC)                                                                                                   \
    mixed_attention_kernel<TC, ACC><<<grid, MA_THREADS, lds, s>>>((const TC*)q, (const TC*)k_cache, (const TC*)v_cache,   \
                                                                   block_tables, bt_width, token_req, positions, bias,   \
                                                                   bias_rows, mix, scale, cap, window, keep_first, sink, \
                                                                   (TC*)out, H, G, D, page_size, tiles_per_split, part_o, \
                                                                   part_ml)
    if (per <= 1) MA_LAUNCH(1);
    else if (per <= 2) MA_LAUNCH(2);
    else if (per <= 4) MA_LAUNCH(4);
    else MA_LAUNCH(8);
#undef MA_LAUNCH
    int rc = tff_check_launch("mixed_attention");
    if (rc || splits <= 1) return rc;
    return ma_merge<TC>(part_o, part_ml, splits, sink, out, T, H, D, s);
}

// Whether a step of few tokens runs on the matrix cores: bfloat16, up to 32 heads of 32, 64 or 128, up to 16 on a kv head,
// and pages of a multiple of 8 tokens; not more than 16 kv heads of 128 (the results of four of them a wave leave no registers).
static bool ma_few(int H, int G, int D, int page_size, int dtype) {
    return dtype == TFF_BF16 && H > 0 && H <= 32 && G > 0 && H / G <= 16 && (D == 32 || D == 64 || D == 128) && page_size % 8 == 0 &&
           (G + Q16_WAVES - 1) / Q16_WAVES * D <= 256;
}

TFF_API int tff_mixed_attention_tile(int H, int G, int D, int page_size, int dtype) {
    return ma_few(H, G, D, page_size, dtype) ? FEW_TK : MA_TK;
}

static int ma_few_launch(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables, int bt_width,
                         const int32_t* token_req, const int32_t* positions, const float* bias, int bias_rows, const float* mix,
                         float scale, float cap, int window, int keep_first, int sink, void* out, int T, int H, int G, int D,
                         int page_size, int splits, int tiles_per_split, float* ws, hipStream_t s) {
    float* part_o = ws;
    float* part_ml = ws ? ws + (size_t)T * splits * H * D : nullptr;
    const int gpw = (G + Q16_WAVES - 1) / Q16_WAVES;
#define FEW_LAUNCH(GPW, EB)                                                                                              \
    mixed_attention_few_kernel<GPW, EB><<<dim3(T, splits), Q16_THREADS, 0, s>>>(                                         \
        (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables, bt_width, token_req, positions,  \
        bias, bias_rows, mix, scale, cap, window, keep_first, sink, (bf16_t*)out, H, G, page_size, tiles_per_split,      \
        part_o, part_ml)
#define FEW_BY_EB(GPW)                   \
    do {                                 \
        if (D == 32) FEW_LAUNCH(GPW, 2); \
        else if (D == 64) FEW_LAUNCH(GPW, 4); \
        else FEW_LAUNCH(GPW, 8);         \
    } while (0)
    if (gpw <= 1) FEW_BY_EB(1);
    else if (gpw <= 2) FEW_BY_EB(2);
    else if (D == 32) FEW_LAUNCH(4, 2);
    else FEW_LAUNCH(4, 4);
#undef FEW_BY_EB
#undef FEW_LAUNCH
    int rc = tff_check_launch("mixed_attention");
    if (rc || splits <= 1) return rc;
    return ma_merge<bf16_t>(part_o, part_ml, splits, sink, out, T, H, D, s);
}

TFF_API int tff_mixed_attention(const void* q, const void* k_cache, const void* v_cache, const int32_t* block_tables,
                                int bt_width, const int32_t* token_req, const int32_t* positions, const float* bias,
                                int bias_rows, const float* mix, float scale, float cap, int window, int keep_first,
                                int sink, void* out, int T, int H, int G, int D, int page_size, int splits,
                                int tiles_per_split, float* workspace, int dtype, tff_stream_t stream) {
    TFF_REQUIRE(q && k_cache && v_cache && block_tables && token_req && positions && out, "mixed_attention: null pointer");
    TFF_REQUIRE(T >= 0 && G > 0 && H % G == 0 && bt_width > 0 && page_size > 0 && page_size % 8 == 0,
                "mixed_attention: %d heads on %d kv heads, pages of %d", H, G, page_size);
    TFF_REQUIRE(tff_mixed_attention_supported(H, D, mix != nullptr), "mixed_attention: %d heads of %d do not fit a block", H, D);
    TFF_REQUIRE(!bias || bias_rows > 0, "mixed_attention: a bias table without rows");
    TFF_REQUIRE(window >= 0 && keep_first >= 0, "mixed_attention: negative window");
    TFF_REQUIRE(splits >= 1 && splits <= 65535 && (splits == 1 || (tiles_per_split >= 1 && workspace)),
                "mixed_attention: %d splits of %d tiles", splits, tiles_per_split);
    if (T == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (ma_few(H, G, D, page_size, dtype))
        return ma_few_launch(q, k_cache, v_cache, block_tables, bt_width, token_req, positions, bias, bias_rows, mix, scale, cap,
                             window, keep_first, sink, out, T, H, G, D, page_size, splits, tiles_per_split, workspace, s);
    if (dtype == TFF_F32)
        return ma_launch<float>(q, k_cache, v_cache, block_tables, bt_width, token_req, positions, bias, bias_rows, mix,
                                scale, cap, window, keep_first, sink, out, T, H, G, D, page_size, splits, tiles_per_split,
                                workspace, s);
    if (dtype == TFF_BF16)
        return ma_launch<bf16_t>(q, k_cache, v_cache, block_tables, bt_width, token_req, positions, bias, bias_rows, mix,
                                 scale, cap, window, keep_first, sink, out, T, H, G, D, page_size, splits, tiles_per_split,
                                 workspace, s);
    return tff_fail("mixed_attention: unknown dtype %d", dtype);
}
