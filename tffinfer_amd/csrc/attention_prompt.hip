// bfloat16 attention of prompt portions over the paged cache: the blocks that attention_mfma.hip gives long portions,
// for large heads without a cap on the scores and without pooled blocks of keys, on four waves of several column tiles.
// (Reference: src/kernel/cuda/paged_flash_attention.cu:855-1055.)  Columns, operand orders, the softmax on raw scores and
// the merge of key groups are those of that file; what differs is what bounds it.
//
// With a column tile (16 columns) a wave every MFMA wants an operand of 1 KB from LDS, and LDS gives a CU 128 bytes a
// cycle: eight waves' slices of 32 keys take 1,024 cycles there, 512 on the matrix cores.  So a wave works on NQT
// column tiles and every fragment it reads feeds NQT MFMAs; the accumulators (in the accumulation registers, and the
// queries beside them) then leave room for one wave a SIMD, and what two waves would do for each other the wave does
// itself.  In step s its MFMAs are P(s-1) . V(s-1) and Q . K(s+1), none of which waits for the softmax of slice s that
// stands between them: 64 MFMAs of sixteen cycles beside some 140 instructions of four and 32 exponentials of sixteen.
// The fragments of K(s+1) are read from LDS behind the first half of the MFMAs, those of V(s) behind the second.
//
// What is left to bound it is the issue of that one wave, so the softmax has neither a maximum nor a rescaling: the
// reference of a column's exponentials is the largest score of its first slice, and float32 holds what the others exceed
// it by: sums and outputs are of the size 2^(largest - reference), without any loss of precision up to 2^50 and values up
// to 2^77.  Where a column's sum turns out below 2^-50, or a group's part of it beyond 2^50, or an output is no finite
// number, the block goes over the item's keys once more for the largest score of every column and then repeats the item
// against that.  The bound is for two groups, whose references differ: what a group brings to their merge is scaled by
// 2^-126 at least or is zero, so that of sums up to 2^50 no more than 2^-76 is lost of one that must be 2^-50.
// Values that are not finite reach columns that do not see them (0 . inf is no number), and with them the test, which sends the
// item into its second pass: there a wave takes values that none of its columns sees as zeros.
//
// us, the blocks of eight waves / these, 32 query and 8 key heads of 128: 512 tokens 19.3 / 17.5, 901 27.8 / 23.9, 2,048 60.0 / 50.5,
// 4,096 207 / 141, 16,384 2,610 / 1,793 (0.84 / 1.23 PFLOP/s); 3,001 and 1,700 tokens of 16 and 4 heads in a window of 1,024
// 63.9 / 46; a head size of 256, 32 heads on one, 2,048 tokens in a window of 1,024: 104 / 77.  With a running maximum, its
// test and the rescaling in every step 16,384 tokens took 2,003.
#include <type_traits>
#include <utility>

#include "common.h"
#include "mfma_tiles.h"
#include "tffinfer_kernels.h"

#define ATTN_PROMPT_PAGES 2048

namespace {

// The three MFMAs of a step: scores from zero, scores on, outputs.  As instructions, so that scores stay in the vector
// registers and queries and outputs in the accumulation registers.
__device__ __forceinline__ void mfma_score0(floatx4& s, const bf16x8& k, const bf16x8& q) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(k), "a"(q));
}
__device__ __forceinline__ void mfma_score(floatx4& s, const bf16x8& k, const bf16x8& q) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(k), "a"(q));
}
// 16 bytes a lane into LDS at lds + PLUS, from OFF bytes behind g (the instruction adds them to both addresses)
template <int OFF, int PLUS>
__device__ __forceinline__ void copy16_at(unsigned long long g, unsigned lds) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off offset:%2"
                 : : "s"(lds), "v"(g), "i"(OFF), "i"(PLUS - OFF) : "memory", "m0", "scc");
}

// f(0), f(1), ... f(N - 1), each with its number as a constant
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_each(f, std::make_integer_sequence<int, N>{});
}

template <int DT, int NQT, int KGRP>
__global__ __launch_bounds__(256, 1) void attn_prompt_kernel(
    const bf16_t* __restrict__ q, int q_stride, bf16_t* __restrict__ out, const bf16_t* __restrict__ k_cache,
    const bf16_t* __restrict__ v_cache, const int32_t* __restrict__ block_tables, int bt_stride,
    const int32_t* __restrict__ cu_tokens, const int32_t* __restrict__ start_pos, const int32_t* __restrict__ work,
    const int32_t* __restrict__ block_items, int nq, int nkv, int page_size, int page_shift, int window, float scale,
    const float* __restrict__ sinks) {
    constexpr int D = DT * 16, KS = D / 32, KFR = 2 * KS, VFR = DT;      // 1 KB fragments of a slice
    static_assert(DT % 2 == 0, "whole steps of 32 elements");
    constexpr int NW = 4 / KGRP;                      // waves along the columns; KGRP groups take every KGRP-th slice
    constexpr int NR = KGRP == 1 ? 4 : 3;             // slices of K and of V in LDS
    constexpr int KC = KFR * KGRP / 4, VC = VFR * KGRP / 4, CPI = KC + VC;      // a wave's copies a step
    static_assert(KS % KC == 0 || KC == KS, "a wave's fragments of K are those of one tile of keys");
    constexpr unsigned K_SLOT = KGRP * KFR * 1024u, V_SLOT = KGRP * VFR * 1024u, V_BASE = NR * K_SLOT;
    constexpr int NPV = DT * NQT, NQK = KFR * NQT, NP = NQT * 4;      // MFMAs of the two halves, pairs of scores a lane
    static_assert(NPV == 32 && NQK == 32 && 4 + 3 * NP <= 62, "a step's schedule");
    constexpr float NO_KEY = 1e30f, SUM_MIN = 0x1p-50f, SUM_MAX = 0x1p50f;
    static_assert(KGRP == 1 || V_BASE + NR * V_SLOT >= NW * NQT * (DT * 1024u + 512u), "the merge borrows the slices' place");
    __shared__ __attribute__((aligned(1024))) char smem[V_BASE + NR * V_SLOT];
    __shared__ int32_t pages[ATTN_PROMPT_PAGES];      // starts of pages in units of 16 bytes
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wcol = wave % NW, kgi = wave / NW;      // this wave's columns and key group
    const int qc = lane & 15, kg = lane >> 4;
    const int g = blockIdx.y, G = nq / nkv;
    // what this wave copies: of group c_sub's slice the fragments of K from c_wi * KC on and the value tiles from c_wi * VC on
    const int c_sub = wave / NW, c_wi = wave % NW;
    const int c_kt = c_wi * KC / KS, c_ks = c_wi * KC % KS;
    const int c_key = (qc >> 2) * 8 + c_kt * 4 + (qc & 3);
    const unsigned c_koff = (unsigned)(c_ks * 4 + kg), c_voff = (unsigned)((c_wi * VC * 16 + qc) * page_size) >> 3;
    const unsigned lds0 = (unsigned)(size_t)(lds_ptr_t)smem;
    const unsigned k_to = lds0 + (unsigned)c_sub * KFR * 1024u + (unsigned)(c_wi * KC) * 1024u;
    const unsigned v_to = lds0 + V_BASE + (unsigned)c_sub * VFR * 1024u + (unsigned)(c_wi * VC) * 1024u;
    const unsigned long long kbase = (unsigned long long)(k_cache + (size_t)g * page_size * D);
    const unsigned long long vbase = (unsigned long long)(v_cache + (size_t)g * D * page_size);
    const uint32_t page_units = (uint32_t)nkv * page_size * (D / 8);
    const unsigned v_step = (unsigned)page_size * 32u;                   // bytes from a value tile to the next
    const float sl2 = scale * 1.44269504088896f;

    const int it_begin = block_items ? block_items[blockIdx.x] : (int)(gridDim.x - 1 - blockIdx.x);
    const int it_end = block_items ? block_items[blockIdx.x + 1] : it_begin + 1;
    if (it_begin >= it_end) return;
    // an item's place, queries and first pages, asked for before the item before it is stored
    int f_r, f_bcol0, f_tok0, f_ncols, f_P, f_page;
    bf16x8 qf[NQT][KS];
    auto fetch = [&](int item) {
        f_r = work[2 * item];
        f_bcol0 = work[2 * item + 1];
        f_tok0 = cu_tokens[f_r];
        f_ncols = (cu_tokens[f_r + 1] - f_tok0) * G;
        f_P = start_pos[f_r];
        const int kmin = window > 0 ? max(0, f_P + f_bcol0 / G - window + 1) : 0;
        const int kmax = f_P + (min(f_bcol0 + NW * NQT * 16, f_ncols) - 1) / G;
        f_page = block_tables[(size_t)f_r * bt_stride + min(((kmin / 32 * 32) >> page_shift) + tid, kmax >> page_shift)];
#pragma unroll
        for (int t = 0; t < NQT; ++t) {
            const int c = min(f_bcol0 + wcol * (NQT * 16) + t * 16 + qc, f_ncols - 1), tl = c / G;
            const bf16_t* qp = q + (size_t)(f_tok0 + tl) * q_stride + (size_t)(g * G + (c - tl * G)) * D;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) qf[t][ks] = *reinterpret_cast<const bf16x8*>(qp + ks * 32 + kg * 8);
        }
    };
    fetch(it_begin);
    for (int item = it_begin; item < it_end; ++item) {
        if (item > it_begin) __syncthreads();         // the last item's slices and pages are read
        const int r = f_r, bcol0 = f_bcol0, tok0 = f_tok0, ncols = f_ncols, P = f_P, first_page = f_page;
        const int32_t* bt = block_tables + (size_t)r * bt_stride;
        const int col0 = bcol0 + wcol * (NQT * 16);
        // (a column past the last one repeats it: nothing of it is stored)
        int c_pos[NQT], c_lo[NQT];
        int w_min, w_lo;                              // the wave's first column's last key, its last column's first
#pragma unroll
        for (int t = 0; t < NQT; ++t) {
            c_pos[t] = P + min(col0 + t * 16 + qc, ncols - 1) / G;
            c_lo[t] = window > 0 ? max(0, c_pos[t] - window + 1) : 0;
        }
        w_min = P + min(col0, ncols - 1) / G;
        w_lo = window > 0 ? max(0, P + min(col0 + NQT * 16 - 1, ncols - 1) / G - window + 1) : 0;
        w_min = __builtin_amdgcn_readfirstlane(w_min);
        w_lo = __builtin_amdgcn_readfirstlane(w_lo);
        const int kmin = window > 0 ? max(0, P + bcol0 / G - window + 1) : 0;
        const int kmax = P + (min(bcol0 + NW * NQT * 16, ncols) - 1) / G;
        const int kb0 = (kmin / 32) * 32, nsteps = (kmax - kb0) / 32 + 1;
        const int seg_steps = max(KGRP, ((((ATTN_PROMPT_PAGES - 1) * page_size) >> 5) / KGRP) * KGRP);

        floatx4 o[NQT][DT], sc[2][NQT][2];
        bf16x8 pf[2][NQT], kf[KFR], vf[VFR];
        float neg_ref[NQT], l_run[NQT];      // minus a column's reference in the exponent's units, the sum against it
#pragma unroll
        for (int t = 0; t < NQT; ++t) {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+a"(qf[t][ks]));      // (waited for here: the compiler does not see the copies)
        }
        // scores of a slice whose first key is kb: minus infinity where a column does not see the key (past the last slice it sees none)
        auto mask = [&](floatx4 (&x)[NQT][2], int kb) {
#pragma unroll
            for (int t = 0; t < NQT; ++t) {
                const unsigned from = (unsigned)(kb + kg * 8 - c_lo[t]), span = (unsigned)(c_pos[t] - c_lo[t]);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[t][e >> 2][e & 3] = from + (unsigned)e <= span ? x[t][e >> 2][e & 3] : -INFINITY;
                asm volatile("" : "+v"(x[t][0]), "+v"(x[t][1]));      // (here, in the branch)
            }
        };
        // (the scores' MFMAs have written: named one by one, or the compiler, which does not know them for MFMAs, reads them before)
        auto settle = [&](floatx4 (&x)[NQT][2]) {
            asm volatile("s_nop 15");
#pragma unroll
            for (int t = 0; t < NQT; ++t) asm volatile("" : "+v"(x[t][0]), "+v"(x[t][1]));
        };
        auto largest = [&](const floatx4 (&x)[2]) {
            float m = fmaxf(x[0][0], x[1][0]);
#pragma unroll
            for (int e = 1; e < 4; ++e) m = fmaxf(m, fmaxf(x[0][e], x[1][e]));
            return m;
        };

        // a slice's values of keys that none of the wave's columns sees become zeros
        auto hide = [&](int kb) {
            const int w_from = __builtin_amdgcn_readfirstlane(c_lo[0]), w_to = __builtin_amdgcn_readlane(c_pos[NQT - 1], 15);
            const unsigned from = (unsigned)(kb + kg * 8 - w_from), span = (unsigned)(w_to - w_from);
            unsigned seen[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                seen[i] = (from + 2u * i <= span ? 0xffffu : 0u) | (from + 2u * i + 1u <= span ? 0xffff0000u : 0u);
#pragma unroll
            for (int dt = 0; dt < VFR; ++dt) {
                union { bf16x8 f; unsigned u[4]; } x;
                x.f = vf[dt];
#pragma unroll
                for (int i = 0; i < 4; ++i) x.u[i] &= seen[i];
                vf[dt] = x.f;
                asm volatile("" : "+v"(vf[dt]));
            }
            asm volatile("s_nop 1");      // (what a vector instruction has written an MFMA may read two instructions later: the compiler does not know these for MFMAs)
        };

        // the columns' references for the second pass: the largest score of all of the group's slices
        auto against_largest = [&]() {
            float top[NQT];
#pragma unroll
            for (int t = 0; t < NQT; ++t) top[t] = -INFINITY;
            for (int sl = kgi; sl < nsteps; sl += KGRP) {
                const int kb = kb0 + sl * 32;
                floatx4 x[NQT][2];
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    const int j = min(kb + (qc >> 2) * 8 + kt * 4 + (qc & 3), kmax);
                    const bf16_t* kp = k_cache + (size_t)g * page_size * D + (size_t)bt[j >> page_shift] * nkv * page_size * D
                                       + (size_t)(j & (page_size - 1)) * D + kg * 8;
                    bf16x8 k[KS];
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks) k[ks] = *reinterpret_cast<const bf16x8*>(kp + ks * 32);
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                        for (int t = 0; t < NQT; ++t) {
                            if (ks == 0) mfma_score0(x[t][kt], k[ks], qf[t][ks]);
                            else mfma_score(x[t][kt], k[ks], qf[t][ks]);
                        }
                }
                settle(x);
                mask(x, kb);
#pragma unroll
                for (int t = 0; t < NQT; ++t) top[t] = fmaxf(top[t], largest(x[t]));
            }
#pragma unroll
            for (int t = 0; t < NQT; ++t) {
                const float m = rows_max(top[t]);
                neg_ref[t] = m == -INFINITY ? NO_KEY : -m * sl2;
            }
        };

        // the copies of a segment's step x: a lane's key, past the last one that once more, and its page (keys count from the segment's first page)
        int seg0 = 0, seg1 = 0, key0 = 0, k_end = 0, v_end = 0;
        auto k_key = [&](int x) { return key0 + (x * KGRP + c_sub) * 32 + c_key; };
        auto v_key = [&](int x) { return key0 + (x * KGRP + c_sub) * 32 + kg * 8; };
        auto page_of = [&](int j) { return (uint32_t)pages[j >> page_shift]; };
        auto k_at = [&](uint32_t page, int j) {
            return kbase + ((unsigned long long)(page + (uint32_t)((j & (page_size - 1)) * (D / 8)) + c_koff) << 4);
        };
        auto v_at = [&](uint32_t page, int j) {
            return vbase + ((unsigned long long)(page + (uint32_t)((j & (page_size - 1)) >> 3) + c_voff) << 4);
        };
        static_assert(KC <= 4 && VC <= 4, "a wave's copies");
        auto copies_k = [&](auto C, unsigned long long at, unsigned to) {
            constexpr int c = decltype(C)::value;
            copy16_at<c * 64, c * 1024>(at, to);
        };
        auto copies_v = [&](auto C, unsigned long long& at, unsigned to) {
            constexpr int c = decltype(C)::value;
            copy16_at<0, c * 1024>(at, to);
            if constexpr (c + 1 < VC) at += v_step;
        };

        for (int pass = 0;; ++pass) {
#pragma unroll
            for (int t = 0; t < NQT; ++t) {
                l_run[t] = 0.f;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    o[t][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
                    asm volatile("" : "+a"(o[t][dt]));
                }
            }
            for (seg0 = 0; seg0 < nsteps; seg0 += seg_steps) {
                seg1 = min(nsteps, seg0 + seg_steps);
                if (seg0 > 0 || pass > 0) {
                    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));      // the segment before: its copies have landed, its slices and pages are read
                    __syncthreads();
                }
                {
                    const int first = kb0 + seg0 * 32, last = min(kmax, kb0 + seg1 * 32 - 1), pg0 = first >> page_shift;
                    key0 = first - (pg0 << page_shift);
                    k_end = last - (pg0 << page_shift);
                    v_end = (k_end >> 3) << 3;      // (pages hold a multiple of 8 tokens)
                    if (seg0 == 0 && tid <= k_end >> page_shift) pages[tid] = (int32_t)((uint32_t)first_page * page_units);
                    for (int i = seg0 == 0 ? tid + 256 : tid; i <= k_end >> page_shift; i += 256)
                        pages[i] = (int32_t)((uint32_t)bt[pg0 + i] * page_units);
                }
                __syncthreads();
                // step x issues K(x + NR) and V(x + NR - 1): the steps -NR .. -1
#pragma unroll
                for (int x = 0; x < NR; ++x) {
                    int j = min(k_key(x), k_end);
                    const unsigned long long ka = k_at(page_of(j), j);
                    static_for<KC>([&](auto C) { copies_k(C, ka, k_to + x * K_SLOT); });
                    if (x > 0) {
                        j = min(v_key(x - 1), v_end);
                        unsigned long long va = v_at(page_of(j), j);
                        static_for<VC>([&](auto C) { copies_v(C, va, v_to + (x - 1) * V_SLOT); });
                    }
                }
                const int nsup = (seg1 - seg0 + KGRP - 1) / KGRP;
                __builtin_amdgcn_s_waitcnt(vmcnt_imm((NR - 1) * CPI));
                __syncthreads();
                // K(0) against the queries, and nothing yet to multiply values with
                {
                    const char* ks_ = smem + kgi * KFR * 1024 + lane * 16;
#pragma unroll
                    for (int f = 0; f < KFR; ++f) kf[f] = *reinterpret_cast<const bf16x8*>(ks_ + f * 1024);
#pragma unroll
                    for (int f = 0; f < KFR; ++f)
#pragma unroll
                        for (int t = 0; t < NQT; ++t) {
                            if (f < 2) mfma_score0(sc[0][t][f & 1], kf[(f & 1) * KS + (f >> 1)], qf[t][f >> 1]);
                            else mfma_score(sc[0][t][f & 1], kf[(f & 1) * KS + (f >> 1)], qf[t][f >> 1]);
                        }
                    if (seg0 == 0 && pass == 0) {      // the columns' references
                        settle(sc[0]);
#pragma unroll
                        for (int t = 0; t < NQT; ++t) {
                            // Keys that a column's window has passed count here: what matters is the scores' size.  Those that every column's
                            // has passed do not: their pages may be given back, and then the table has another request's in their place.
                            const unsigned from = kgi < seg1 ? (unsigned)(kb0 + kgi * 32 + kg * 8 - kmin) : 0x40000000u, span = (unsigned)(c_pos[t] - kmin);
                            float m = -INFINITY;
#pragma unroll
                            for (int e = 0; e < 8; ++e) m = from + (unsigned)e <= span ? fmaxf(m, sc[0][t][e >> 2][e & 3]) : m;
                            m = rows_max(m);
                            neg_ref[t] = m == -INFINITY ? NO_KEY : -m * sl2;
                        }
                    }
                    const uint4 zero = make_uint4(0, 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < NQT; ++t) pf[1][t] = *reinterpret_cast<const bf16x8*>(&zero);
#pragma unroll
                    for (int dt = 0; dt < VFR; ++dt) vf[dt] = *reinterpret_cast<const bf16x8*>(&zero);
                }
                unsigned k_rd = K_SLOT, v_rd = 0;                             // K(s + 1), V(s)
                unsigned k_wr = k_to, v_wr = v_to + (NR - 1) * V_SLOT;        // where K(s + NR), V(s + NR - 1) go
                int k_next = k_key(NR), v_next = v_key(NR - 1);               // and which keys those are
                // the steps whose slices lie within every column's keys
                const int full0 = max(0, (w_lo - kb0 + 31) / 32 - seg0 - kgi + KGRP - 1) / KGRP;
                const int full1 = min((w_min - 31 - kb0 >= 0 ? (w_min - 31 - kb0) / 32 + 1 : 0), seg1) - seg0 - kgi;
                const unsigned full = (unsigned)max(0, (full1 > 0 ? (full1 + KGRP - 1) / KGRP : 0) - full0);
                // the first key of the group's slice of step s; past the segment's last slice one that no column sees
                auto group_slice = [&](int s) { return seg0 + s * KGRP + kgi < seg1 ? kb0 + (seg0 + s * KGRP + kgi) * 32 : 0x40000000; };
                auto step = [&](auto H, int s) {
                    constexpr int h = decltype(H)::value;
                    __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((NR - 2) * CPI));
                    asm volatile("s_barrier\n\ts_nop 7" ::: "memory");        // (the scores' last MFMAs have written before a vector instruction reads them)
                    const char* ksrc = smem + k_rd + kgi * KFR * 1024 + lane * 16;
                    const char* vsrc = smem + V_BASE + v_rd + kgi * VFR * 1024 + lane * 16;
                    float tmp0 = 0.f, tmp1 = 0.f;
                    uint32_t pk = 0, pv = 0;
                    int jk = 0, jv = 0;
                    unsigned long long ka = 0, va = 0;
                    if (pass > 0) hide(group_slice(s - 1));
                    static_for<NPV + NQK>([&](auto slot) {
                        constexpr int n = decltype(slot)::value;
                        if constexpr (n < NPV) {
                            mfma_acc(o[n % NQT][n / NQT], vf[n / NQT], pf[h ^ 1][n % NQT]);
                        } else {
                            constexpr int f = (n - NPV) / NQT, t = n % NQT, kt = f & 1, ks = f >> 1;
                            if constexpr (ks == 0) mfma_score0(sc[h ^ 1][t][kt], kf[kt * KS + ks], qf[t][ks]);
                            else mfma_score(sc[h ^ 1][t][kt], kf[kt * KS + ks], qf[t][ks]);
                        }
                        // fragments: K(s + 1) in the order of their use, then V(s)
                        if constexpr (n < NPV && n % (NPV / KFR) == 0) {
                            constexpr int f = n / (NPV / KFR), fr = (f & 1) * KS + (f >> 1);
                            kf[fr] = *reinterpret_cast<const bf16x8*>(ksrc + fr * 1024);
                        }
                        if constexpr (n >= NPV && n < NPV + VFR * (VFR > 8 ? 1 : 2) && (VFR > 8 || n % 2 == 0)) {
                            constexpr int dt = (n - NPV) / (VFR > 8 ? 1 : 2);
                            vf[dt] = *reinterpret_cast<const bf16x8*>(vsrc + dt * 1024);
                        }
                        // the softmax of slice s
                        if constexpr (n == 3) if ((unsigned)(s - full0) >= full) mask(sc[h], group_slice(s));
                        if constexpr (n >= 4 && n < 4 + 3 * NP) {
                            constexpr int p = (n - 4) / 3, t = p / 4, e = (p % 4) * 2;
                            if constexpr ((n - 4) % 3 == 0) {
                                tmp0 = fmaf(sc[h][t][e >> 2][e & 3], sl2, neg_ref[t]);
                                tmp1 = fmaf(sc[h][t][e >> 2][(e & 3) + 1], sl2, neg_ref[t]);
                                tmp0 = __builtin_amdgcn_exp2f(tmp0);            // 2^-inf = 0 for masked scores
                            } else if constexpr ((n - 4) % 3 == 1) {
                                tmp1 = __builtin_amdgcn_exp2f(tmp1);
                                l_run[t] += tmp0;
                            } else {
                                l_run[t] += tmp1;
                                pf[h][t][e] = (bf16_t)tmp0;
                                pf[h][t][e + 1] = (bf16_t)tmp1;
                            }
                        }
                        // the copies of later slices
                        if constexpr (n == 5) jk = min(k_next, k_end);
                        if constexpr (n == 6) pk = page_of(jk);
                        if constexpr (n == 8) jv = min(v_next, v_end);
                        if constexpr (n == 9) pv = page_of(jv);
                        if constexpr (n == 11) k_next += KGRP * 32;
                        if constexpr (n == 12) v_next += KGRP * 32;
                        if constexpr (n == 33) ka = k_at(pk, jk);
                        if constexpr (n == 35) va = v_at(pv, jv);
                        if constexpr (n >= 36 && n < 36 + 3 * CPI && n % 3 == 0) {
                            constexpr int c = (n - 36) / 3;
                            if constexpr (c < KC) copies_k(std::integral_constant<int, c < KC ? c : 0>{}, ka, k_wr);
                            else copies_v(std::integral_constant<int, c < KC ? 0 : c - KC>{}, va, v_wr);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    // (worked out here: the compiler would move the softmax out of the MFMAs, behind the next step's branch: 16,384 tokens 1,885 / 1,940)
#pragma unroll
                    for (int t = 0; t < NQT; ++t) asm volatile("" : "+v"(pf[h][t]), "+v"(l_run[t]));
                    k_wr = k_to + k_rd;
                    v_wr = v_to + v_rd;
                    k_rd = ring_next<K_SLOT, NR * K_SLOT>(k_rd);
                    v_rd = ring_next<V_SLOT, NR * V_SLOT>(v_rd);
                };
                // (in pairs, whose second step may have nothing: with an end in between the compiler carries the accumulators from one set of
                // registers to another in every step)
                for (int s = 0; s < nsup; s += 2) {
                    step(std::integral_constant<int, 0>{}, s);
                    step(std::integral_constant<int, 1>{}, s + 1);
                }
                // the values of the segment's last slice
                if (pass > 0) hide(group_slice((nsup + 1) / 2 * 2 - 1));
#pragma unroll
                for (int n = 0; n < NPV; ++n) mfma_acc(o[n % NQT][n / NQT], vf[n / NQT], pf[1][n % NQT]);
            }
            asm volatile("s_nop 15\n\ts_nop 15");       // (the outputs' last MFMAs have written)
#pragma unroll
            for (int t = 0; t < NQT; ++t)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) asm volatile("" : "+a"(o[t][dt]));
            __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm(0));      // the copies past the end must not outlive the block

            // With two groups each one finishes half of the column tiles: it hands the other's references, sums and outputs over through
            // the slices' place.
            static_assert(KGRP <= 2 && NQT % KGRP == 0, "two groups at most");
            float* mo = reinterpret_cast<float*>(smem) + wcol * NQT * (DT * 256 + 128) + lane * 4;
            bool again = false;      // a column whose sums leave float32's comfortable range: the whole block once more
#pragma unroll
            for (int t = 0; t < NQT; ++t) again |= !(l_run[t] <= SUM_MAX);      // (a lane's part of its group's; zero without a key)
            auto give = [&](auto FROM) {
#pragma unroll
                for (int t = decltype(FROM)::value; t < decltype(FROM)::value + NQT / KGRP; ++t) {
                    float* m = mo + t * (DT * 256 + 128);
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
                        *reinterpret_cast<float4*>(m + dt * 256) = make_float4(o[t][dt][0], o[t][dt][1], o[t][dt][2], o[t][dt][3]);
                    *reinterpret_cast<float2*>(m + DT * 256 - lane * 2) = make_float2(neg_ref[t], l_run[t]);
                }
            };
            auto finish = [&](auto FROM) {
#pragma unroll
                for (int t = decltype(FROM)::value; t < decltype(FROM)::value + NQT / KGRP; ++t) {
                    if constexpr (KGRP > 1) {
                        const float* m = mo + t * (DT * 256 + 128);
                        const float2 other = *reinterpret_cast<const float2*>(m + DT * 256 - lane * 2);
                        const float n = fminf(neg_ref[t], other.x);
                        const float a1 = __builtin_amdgcn_exp2f(n - neg_ref[t]), a2 = __builtin_amdgcn_exp2f(n - other.x);
                        l_run[t] = l_run[t] * a1 + other.y * a2;
                        neg_ref[t] = n;
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) {
                            const float4 o2 = *reinterpret_cast<const float4*>(m + dt * 256);
                            o[t][dt][0] = o[t][dt][0] * a1 + o2.x * a2;
                            o[t][dt][1] = o[t][dt][1] * a1 + o2.y * a2;
                            o[t][dt][2] = o[t][dt][2] * a1 + o2.z * a2;
                            o[t][dt][3] = o[t][dt][3] * a1 + o2.w * a2;
                        }
                    }
                    l_run[t] = rows_sum(l_run[t]);
                    float all = 0.f;      // infinite or no number where one of the outputs is
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) all += (o[t][dt][0] + o[t][dt][1]) + (o[t][dt][2] + o[t][dt][3]);
                    again |= !(l_run[t] >= SUM_MIN) || !(fabsf(all) < INFINITY);
                }
            };
            if constexpr (KGRP > 1) {
                __syncthreads();
                if (kgi == 0) give(std::integral_constant<int, NQT / 2>{});
                else give(std::integral_constant<int, 0>{});
                __syncthreads();
                if (kgi == 0) finish(std::integral_constant<int, 0>{});
                else finish(std::integral_constant<int, NQT / 2>{});
            } else {
                finish(std::integral_constant<int, 0>{});
            }
            if (!__syncthreads_or(again) || pass > 0) break;
            against_largest();
        }
        if (item + 1 < it_end) fetch(item + 1);
        auto store = [&](auto FROM) {
#pragma unroll
            for (int t = decltype(FROM)::value; t < decltype(FROM)::value + NQT / KGRP; ++t) {
                const int c = col0 + t * 16 + qc;
                if (c >= ncols) continue;
                const int tl = c / G, head = g * G + (c - tl * G);
                float l = l_run[t], by = 1.f;
                if (sinks) {      // (against the larger of the two references: the sink may lie far above every score)
                    const float z = sinks[head] * 1.4426950408889634f, m = fmaxf(z, -neg_ref[t]);
                    by = __builtin_amdgcn_exp2f(-neg_ref[t] - m);
                    l = l * by + __builtin_amdgcn_exp2f(z - m);
                }
                const float inv = by / l;
                bf16_t* op = out + ((size_t)(tok0 + tl) * nq + head) * D;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    union { bf16_t h[4]; uint2 u; } pk;
#pragma unroll
                    for (int i = 0; i < 4; ++i) pk.h[i] = (bf16_t)(o[t][dt][i] * inv);
                    *reinterpret_cast<uint2*>(op + dt * 16 + kg * 4) = pk.u;
                }
            }
        };
        constexpr int SECOND = KGRP == 2 ? NQT / 2 : 0;
        if (KGRP == 2 && kgi > 0) store(std::integral_constant<int, SECOND>{});
        else store(std::integral_constant<int, 0>{});
    }
}

}  // namespace

TFF_API int tff_attention_prompt_cols(int d, int key_groups) {
    return d == 128 && key_groups == 1 ? 256 : (d == 128 && key_groups == 2) || (d == 256 && key_groups == 1) ? 128 : 0;
}

TFF_API int tff_attention_prompt(const void* q, int q_stride, void* out, const void* k_cache, const void* v_cache,
                                 const int32_t* block_tables, int bt_stride, const int32_t* cu_tokens, const int32_t* start_pos,
                                 const int32_t* work, int num_work, const int32_t* block_items, int num_blocks, int key_groups,
                                 int nq, int nkv, int d, int page_size, int num_pages, int window, float scale, const float* sinks,
                                 tff_stream_t stream) {
    TFF_REQUIRE(q && out && k_cache && v_cache && block_tables && cu_tokens && start_pos && work, "attention_prompt: null pointer");
    TFF_REQUIRE(nq > 0 && nkv > 0 && nkv <= 65535 && nq % nkv == 0, "attention_prompt: %d query heads are not a multiple of %d key heads", nq, nkv);
    TFF_REQUIRE(tff_attention_prompt_cols(d, key_groups) > 0, "attention_prompt: head size %d with %d key groups", d, key_groups);
    TFF_REQUIRE(page_size >= 8 && (page_size & (page_size - 1)) == 0, "attention_prompt: pages of %d tokens", page_size);
    TFF_REQUIRE((long)nkv * page_size * d < (1L << 31) && (long)num_pages * nkv * page_size * d / 8 < (1L << 32),
                "attention_prompt: a cache of %d pages of %d x %d x %d elements is too large", num_pages, nkv, page_size, d);
    TFF_REQUIRE(q_stride >= nq * d && q_stride % 8 == 0 && ((uintptr_t)q % 16) == 0, "attention_prompt: query rows must be 16-byte aligned (stride %d)", q_stride);
    TFF_REQUIRE(((uintptr_t)out % 8) == 0 && ((uintptr_t)k_cache % 16) == 0 && ((uintptr_t)v_cache % 16) == 0, "attention_prompt: unaligned tensors");
    TFF_REQUIRE(bt_stride > 0 && num_pages > 0 && window >= 0, "attention_prompt: bad geometry");
    if (!block_items) num_blocks = num_work;
    TFF_REQUIRE(num_blocks >= 0 && num_blocks <= num_work, "attention_prompt: %d blocks for %d work items", num_blocks, num_work);
    if (num_blocks == 0) return 0;
    int page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
    const dim3 grid(num_blocks, nkv);
    hipStream_t s = (hipStream_t)stream;
#define TFF_PROMPT(...)                                                                                                   \
    attn_prompt_kernel<__VA_ARGS__><<<grid, 256, 0, s>>>((const bf16_t*)q, q_stride, (bf16_t*)out, (const bf16_t*)k_cache, \
                                                         (const bf16_t*)v_cache, block_tables, bt_stride, cu_tokens,      \
                                                         start_pos, work, block_items, nq, nkv, page_size, page_shift,    \
                                                         window, scale, sinks)
    if (d == 256) TFF_PROMPT(16, 2, 1);
    else if (key_groups == 2) TFF_PROMPT(8, 4, 2);
    else TFF_PROMPT(8, 4, 1);
#undef TFF_PROMPT
    return tff_check_launch("attention_prompt");
}
