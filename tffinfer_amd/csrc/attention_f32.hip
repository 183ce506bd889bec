// Attention over the paged cache in float32 on the float32 matrix cores (v_mfma_f32_16x16x4_f32), for head sizes that
// are multiples of 16 up to 128, 192 and 256, and pages of a power of two of at least four tokens: the path of the
// 32-bit model.  Other sizes, and keys of blocks before a window, run on the general kernel (attention_generic.hip).
//
// A column is a (token, q head of the kv head's group) pair of one request, numbered token * G + head.  A wave takes
// 16 NC columns; per step of 32 keys
//   S^T = K Q^T      lane (column = l % 16, g = l / 16) gets the scores of keys 4 g .. 4 g + 3 of sixteen;
//   softmax          running maximum m and sum l per column (two lane swaps a step), scores scaled after the product,
//                    capped (c tanh(s / c)) if a cap is given, then masked: lo <= key <= position;
//   O^T += V^T P^T   the probabilities lie in the registers as the MFMA wants them, the values come transposed from
//                    their page, [element][slot]: four keys of an element are one 16-byte load.
// Keys and values go from memory straight into the MFMA operands.  With sinks, e^(sink - m) is one more term of the
// denominator.
//
// The order of a column's sums is fixed by its position, the window and the head size alone: step number i (keys 32 i ..
// 32 i + 31 of the request) belongs to part i % PARTS, a part is one chain in ascending order, and the parts are folded in
// ascending order (keys that a column does not see add exact zeros, wherever the tile's walk begins).  No multiply-add is
// left to the compiler's choice.  So a token's result is the same bits alone or beside others, as part of any portion, and in
// every form: a block of 16 columns whose waves share the parts, so that short prompts and decode steps fill the chip, or a block
// of 128 columns with four waves of 32, each of which goes through all parts, so that neighbouring columns walk the same keys and
// the CU's cache serves them.
// What bounds it: the matrix cores and the operands' way from L2 for prompts (2,048 tokens of 32 heads of 128 on 8 kv heads
// 410 us = 84 TFLOP/s; the general kernel, a wave a token and head on the vector units, 43,960 us), the chain of a step for
// few keys (two requests of 400 tokens decoding 20 us, 207 before; 401 + 230 tokens of 16 heads 32 us, 1,193 before).
#include "common.h"
#include "tffinfer_kernels.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float af_floatx4;

__device__ __forceinline__ af_floatx4 af_mfma16(const float4& a, const float4& b, af_floatx4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
}

// The value of key j, zero if it lies outside of what the tile sees or is not finite, which `odd` then notes.
__device__ __forceinline__ float af_finite(float v, int j, int lo, int hi, bool& odd) {
    const bool in = j >= lo && j <= hi, fine = fabsf(v) < INFINITY;
    odd |= in && !fine;
    return in && fine ? v : 0.f;
}
// A value that is not finite as a number whose sums over up to 255 values tell how many of which kind there were, and what
// such a sum stands for.
__device__ __forceinline__ float af_kind(float v) { return v == INFINITY ? 1.f : v == -INFINITY ? 256.f : v != v ? 65536.f : 0.f; }
__device__ __forceinline__ float af_sum_of_kinds(int n) {
    const bool up = n & 255, down = n >> 8 & 255;
    return n >> 16 || (up && down) ? __builtin_nanf("") : up ? INFINITY : down ? -INFINITY : 0.f;
}

// WAVES waves; SHARED: all with the same columns, each with PARTS / WAVES parts of the keys, else with columns of their own and all parts.
template <int DF, int NC, int WAVES, bool SHARED, int PARTS>
__global__ __launch_bounds__(64 * WAVES, 2) void attention_f32_kernel(
    const float* __restrict__ q, int q_stride, float* __restrict__ out, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, const int32_t* __restrict__ block_tables, int bt_stride,
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ start_pos, const int32_t* __restrict__ work, int items,
    int tiles, int nq, int nkv, int ps_shift, int window, float scale, const float* __restrict__ sinks, float softcap) {
#pragma clang fp contract(off)
    constexpr int D = 16 * DF;
    static_assert((PARTS & (PARTS - 1)) == 0 && PARTS % WAVES == 0, "a step's part is its number's last bits");
    __shared__ af_floatx4 red_o[WAVES * NC * DF][64];
    __shared__ float red_ml[SHARED ? WAVES * NC : 1][2][16];
    // heads fastest: the blocks of one kv head meet on one XCD when there are eight; the last columns, which see most
    // keys, first
    const int g_kv = blockIdx.x % nkv, item = items - 1 - (int)(blockIdx.x / nkv);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, wq = SHARED ? 0 : wv, r = lane & 15, g = lane >> 4;
    const int G = nq / nkv, ps = 1 << ps_shift;
    const int row = work ? work[2 * item] : item / tiles;
    const int c0 = (work ? work[2 * item + 1] : item % tiles * 16) + wq * 16 * NC;
    const int t0 = cu_tokens[row], ncol = (cu_tokens[row + 1] - t0) * G, p0 = start_pos[row];
    if (ncol <= 0) return;                                // (the whole block: a row without tokens)
    const int32_t* bt = block_tables + (size_t)row * bt_stride;
    const bool any = c0 < ncol;
    // the wave's columns; those past the last one repeat it
    int pos[NC], lo[NC];
    float4 qf[NC][DF];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = min(c0 + c * 16 + r, ncol - 1);
        const int tok = col / G, head = g_kv * G + col - tok * G;
        pos[c] = p0 + tok;
        lo[c] = window > 0 ? max(0, pos[c] - window + 1) : 0;
        const float* qp = q + (size_t)(t0 + tok) * q_stride + (size_t)head * D + 4 * g;
#pragma unroll
        for (int s = 0; s < DF; ++s) qf[c][s] = *reinterpret_cast<const float4*>(qp + 16 * s);
    }
    const int first_pos = p0 + c0 / G, last_pos = p0 + (min(c0 + 16 * NC, ncol) - 1) / G;
    const int lo_min = window > 0 ? max(0, first_pos - window + 1) : 0;
    const int lo_max = window > 0 ? max(0, last_pos - window + 1) : 0;
    float m[NC], l[NC];
    af_floatx4 o[NC][DF];
    // one part of the keys, and the sums over the four lanes of a column
    auto walk = [&](int part) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            m[c] = -INFINITY;
            l[c] = 0.f;
#pragma unroll
            for (int s = 0; s < DF; ++s) o[c][s] = af_floatx4{0.f, 0.f, 0.f, 0.f};
        }
        const int first = lo_min >> 5, begin = 32 * (first + ((part - first) & (PARTS - 1)));
        bool odd = false;
        for (int k = begin; k <= last_pos; k += 32 * PARTS) {
            af_floatx4 sc[NC][2];
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const int key = min(max(k + 16 * f + r, lo_min), last_pos);      // (no page outside of what some column sees is looked up)
                const float* kp = k_cache + (((size_t)bt[key >> ps_shift] * nkv + g_kv) * ps + (key & (ps - 1))) * D + 4 * g;
                float4 kf[DF];
#pragma unroll
                for (int s = 0; s < DF; ++s) kf[s] = *reinterpret_cast<const float4*>(kp + 16 * s);
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    sc[c][f] = af_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < DF; ++s) sc[c][f] = af_mfma16(kf[s], qf[c][s], sc[c][f]);
                }
            }
            const bool edge = k < lo_max || k + 31 > first_pos;       // some column does not see all of the step
            float4 p[NC][2];
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                float s[8], mx = -INFINITY;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    s[i] = sc[c][i >> 2][i & 3] * scale;
                    if (softcap > 0.f) s[i] = softcap * tanhf(s[i] / softcap);
                    if (edge) {
                        const int key = k + 16 * (i >> 2) + 4 * g + (i & 3);
                        if (key < lo[c] || key > pos[c]) s[i] = -INFINITY;
                    }
                    mx = fmaxf(mx, s[i]);
                }
                const float m_new = fmaxf(m[c], rows_max(mx));
                const float ref = m_new == -INFINITY ? 0.f : m_new;   // (a column that has seen no key yet)
                const float corr = expf(m[c] - ref);
                m[c] = m_new;
                float sum = 0.f, e[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    e[i] = expf(s[i] - ref);
                    sum += e[i];
                }
                l[c] = fmaf(l[c], corr, sum);        // (the four lanes of a column add theirs at the end)
#pragma unroll
                for (int x = 0; x < DF; ++x) o[c][x] = o[c][x] * corr;
                p[c][0] = make_float4(e[0], e[1], e[2], e[3]);
                p[c][1] = make_float4(e[4], e[5], e[6], e[7]);
            }
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const int quad = k + 16 * f + 4 * g, key = min(max(quad, lo_min & ~3), last_pos & ~3);
                const float* vp = v_cache + ((size_t)bt[key >> ps_shift] * nkv + g_kv) * ps * D + (key & (ps - 1)) + (size_t)r * ps;
                float4 vf[DF];
#pragma unroll
                for (int s = 0; s < DF; ++s) vf[s] = *reinterpret_cast<const float4*>(vp + (size_t)16 * s * ps);
                if (edge) {
                    // Slots that hold nothing of the request's may hold anything, and 0 x NaN is not 0; nor may a value that is not
                    // finite reach the columns that do not see its token.  Such values are left out, and follow below.
#pragma unroll
                    for (int s = 0; s < DF; ++s) {
                        vf[s].x = af_finite(vf[s].x, quad + 0, lo_min, last_pos, odd);
                        vf[s].y = af_finite(vf[s].y, quad + 1, lo_min, last_pos, odd);
                        vf[s].z = af_finite(vf[s].z, quad + 2, lo_min, last_pos, odd);
                        vf[s].w = af_finite(vf[s].w, quad + 3, lo_min, last_pos, odd);
                    }
                }
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int s = 0; s < DF; ++s) o[c][s] = af_mfma16(vf[s], p[c][f], o[c][s]);
            }
        }
        if (__any(odd)) {        // what the values that were left out amount to for the columns that see them, their number by kind
#pragma unroll 1
            for (int k = begin; k <= last_pos; k += 32 * PARTS) {
                if (!(k < lo_max || k + 31 > first_pos)) continue;
#pragma unroll 1
                for (int f = 0; f < 2; ++f) {
                    const int quad = k + 16 * f + 4 * g, key = min(max(quad, lo_min & ~3), last_pos & ~3);
                    const float* vp = v_cache + ((size_t)bt[key >> ps_shift] * nkv + g_kv) * ps * D + (key & (ps - 1)) + (size_t)r * ps;
#pragma unroll
                    for (int s = 0; s < DF; ++s) {
                        const float4 v = *reinterpret_cast<const float4*>(vp + (size_t)16 * s * ps);
#pragma unroll
                        for (int c = 0; c < NC; ++c) {
                            auto sees = [&](int j) { return j >= lo[c] && j <= pos[c] ? 1.f : 0.f; };
                            const af_floatx4 n = af_mfma16(make_float4(af_kind(v.x), af_kind(v.y), af_kind(v.z), af_kind(v.w)),
                                                           make_float4(sees(quad), sees(quad + 1), sees(quad + 2), sees(quad + 3)),
                                                           af_floatx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                            for (int i = 0; i < 4; ++i) o[c][s][i] += af_sum_of_kinds((int)n[i]);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) l[c] = rows_sum(l[c]);
    };
    // (M, L, T) takes one more part in: all by the column's maximum so far
    auto fold = [](float& M, float& L, float m, float l, float& a, float& b) {
        const float to = fmaxf(M, m), ref = to == -INFINITY ? 0.f : to;
        a = expf(M - ref);
        b = expf(m - ref);
        L = fmaf(L, a, l * b);
        M = to;
    };
    auto add = [](const af_floatx4& T, float a, const af_floatx4& o, float b) {
        return af_floatx4{fmaf(T[0], a, o[0] * b), fmaf(T[1], a, o[1] * b), fmaf(T[2], a, o[2] * b), fmaf(T[3], a, o[3] * b)};
    };
    // (a column has seen its own key by now, so M is a number)
    auto finish = [&](int c, int s, const af_floatx4& T, float M, float L) {
        const int col = c0 + c * 16 + r;
        if (col >= ncol) return;
        const int tok = col / G, head = g_kv * G + col - tok * G;
        const float inv = 1.0f / (sinks ? L + expf(sinks[head] - M) : L);
        *reinterpret_cast<float4*>(out + ((size_t)(t0 + tok) * nq + head) * D + 16 * s + 4 * g) =
            make_float4(T[0] * inv, T[1] * inv, T[2] * inv, T[3] * inv);
    };
    const af_floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!SHARED) {
        if (!any) return;
        float M[NC], L[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            M[c] = -INFINITY;
            L[c] = 0.f;
#pragma unroll
            for (int s = 0; s < DF; ++s) red_o[(wq * NC + c) * DF + s][lane] = zero;      // (the wave's own)
        }
#pragma unroll 1
        for (int part = 0; part < PARTS; ++part) {
            __builtin_amdgcn_sched_barrier(0);      // (what the fold needs has no registers during the walk)
            walk(part);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                float a, b;
                fold(M[c], L[c], m[c], l[c], a, b);
#pragma unroll
                for (int s = 0; s < DF; ++s) {
                    af_floatx4& T = red_o[(wq * NC + c) * DF + s][lane];
                    T = add(T, a, o[c][s], b);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int s = 0; s < DF; ++s) finish(c, s, red_o[(wq * NC + c) * DF + s][lane], M[c], L[c]);
    } else {
        constexpr int OWN = (DF + WAVES - 1) / WAVES;       // groups of 16 elements a wave folds: wv, wv + WAVES, ...
        af_floatx4 T[NC][OWN];
        float M[NC], L[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            M[c] = -INFINITY;
            L[c] = 0.f;
#pragma unroll
            for (int s = 0; s < OWN; ++s) T[c][s] = zero;
        }
        auto fold_all = [&] {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int w = 0; w < WAVES; ++w) {
                    float a, b;
                    fold(M[c], L[c], red_ml[w * NC + c][0][r], red_ml[w * NC + c][1][r], a, b);
#pragma unroll
                    for (int s = 0; s < OWN; ++s)
                        if (wv + s * WAVES < DF) T[c][s] = add(T[c][s], a, red_o[(w * NC + c) * DF + wv + s * WAVES][lane], b);
                }
        };
#pragma unroll 1
        for (int first = 0; first < PARTS; first += WAVES) {
            walk(first + wv);
            if (first) {                                   // (the waves meet when all have walked, not in between)
                __syncthreads();
                fold_all();
                __syncthreads();
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (g == 0) {
                    red_ml[wv * NC + c][0][r] = m[c];
                    red_ml[wv * NC + c][1][r] = l[c];
                }
#pragma unroll
                for (int s = 0; s < DF; ++s) red_o[(wv * NC + c) * DF + s][lane] = o[c][s];
            }
        }
        __syncthreads();
        fold_all();
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int s = 0; s < OWN; ++s)
                if (wv + s * WAVES < DF) finish(c, wv + s * WAVES, T[c][s], M[c], L[c]);
    }
}

TFF_API int tff_attention_f32_supported(int d, int page_size) {
    const bool size = (d > 0 && d <= 128 && d % 16 == 0) || d == 192 || d == 256;
    return size && page_size >= 4 && (page_size & (page_size - 1)) == 0;
}

// work: int32 [items, 2] (row, first column) of tiles of `cols` columns, or null: every row has `tiles` tiles from column
// 0 on, items = rows * tiles.  cols 16: the block's waves share a tile's parts of the keys; 128: 4 waves of 32 columns each.
TFF_API int tff_attention_f32(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache,
                              const int32_t* block_tables, int bt_stride, const int32_t* cu_tokens, const int32_t* start_pos,
                              const int32_t* work, int items, int tiles, int cols, int nq, int nkv, int d, int page_size,
                              int num_pages, int window, float scale, const float* sinks, float softcap, tff_stream_t stream) {
    TFF_REQUIRE(q && out && k_cache && v_cache && block_tables && cu_tokens && start_pos, "attention_f32: null pointer");
    TFF_REQUIRE(tff_attention_f32_supported(d, page_size), "attention_f32: head size %d on pages of %d tokens", d, page_size);
    TFF_REQUIRE(nq > 0 && nkv > 0 && nq % nkv == 0, "attention_f32: %d query heads are not a multiple of %d key heads", nq, nkv);
    TFF_REQUIRE(num_pages > 0 && bt_stride > 0 && window >= 0 && q_stride >= nq * d && q_stride % 4 == 0,
                "attention_f32: bad geometry pages=%d table stride=%d window=%d query rows of %d", num_pages, bt_stride, window, q_stride);
    TFF_REQUIRE(((uintptr_t)q % 16) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)k_cache % 16) == 0 &&
                ((uintptr_t)v_cache % 16) == 0, "attention_f32: operands must be 16-byte aligned");
    TFF_REQUIRE(items >= 0 && (work || tiles > 0) && (long)items * nkv < (1L << 31), "attention_f32: bad work");
    TFF_REQUIRE(cols == 16 || (cols == 128 && work && d <= 128), "attention_f32: tiles of %d columns of %d", cols, d);
    if (items == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int shift = __builtin_ctz(page_size);
    // Eight waves for a tile's eight parts while the blocks do not go round the CUs twice, else four that take two parts
    // each (half the LDS, a third block on a CU).  us on eight / four: 47 requests of 100 to 2,900 tokens decoding beside a portion
    // of 64 (504 blocks) 134 / 189, 600 tokens of 8 heads of 48 (304) 16.0 / 17.7, 401 + 230 tokens (632) 33.6 / 31.7, 2,048 tokens under a
    // window of 256 (4,096) 227 / 146.
    const bool few = items * nkv < 512;
#define AF_LAUNCH(DF, NC, WAVES, SHARED, PARTS)                                                                            \
    attention_f32_kernel<DF, NC, WAVES, SHARED, PARTS><<<items * nkv, 64 * WAVES, 0, s>>>(                                 \
        (const float*)q, q_stride, (float*)out, (const float*)k_cache, (const float*)v_cache, block_tables, bt_stride,      \
        cu_tokens, start_pos, work, items, tiles, nq, nkv, shift, window, scale, sinks, softcap)
#define AF_SIZE(DF)                                         \
    case DF:                                                \
        if (cols == 128) AF_LAUNCH(DF, 2, 4, false, 8);     \
        else if (few) AF_LAUNCH(DF, 1, 8, true, 8);         \
        else AF_LAUNCH(DF, 1, 4, true, 8);                  \
        break
    switch (d / 16) {
        AF_SIZE(1);
        AF_SIZE(2);
        AF_SIZE(3);
        AF_SIZE(4);
        AF_SIZE(5);
        AF_SIZE(6);
        AF_SIZE(7);
        AF_SIZE(8);
        case 12: AF_LAUNCH(12, 1, 4, true, 4); break;
        default: AF_LAUNCH(16, 1, 4, true, 4); break;
    }
#undef AF_SIZE
#undef AF_LAUNCH
    return tff_check_launch("attention_f32");
}
