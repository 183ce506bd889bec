// What the bfloat16 products share: loads, stores, the gated activation, what a product takes besides its operands.
#pragma once
#include <type_traits>

#include "common.h"
#include "mfma_tiles.h"

__device__ __forceinline__ uint4 ld16(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }
// The same of a weight that one block reads; ONCE: and that nobody asks for again before it has left the caches.
template <bool ONCE>
__device__ __forceinline__ uint4 ld16_weight(const bf16_t* p) {
    if constexpr (!ONCE) return ld16(p);
    typedef __attribute__((__vector_size__(16))) unsigned once_t;
    const once_t v = __builtin_nontemporal_load(reinterpret_cast<const once_t*>(p));
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ bf16x8 as_frag(const uint4& v) { return *reinterpret_cast<const bf16x8*>(&v); }

template <typename TC>
__device__ __forceinline__ void store4(TC* dst, const floatx4& v, int n, int N, bool vec) {
    if (vec) {  // n % 4 == 0 and N % 4 == 0: the four columns exist
        if constexpr (sizeof(TC) == 4) {
            *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
            // (one value of four, not four put together in memory: the compiler took those apart, and joined the last number's store with the one
            // below, three stores of a lane for one; 685 rows of 17,256 x 120 27.8 us that way, 14.6 this way)
            typedef __attribute__((__vector_size__(4 * sizeof(bf16_t)))) __bf16 bf16x4;
            *reinterpret_cast<bf16x4*>(dst) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) dst[e] = from_f32<TC>(v[e]);
    }
}

// What a product takes besides its operands: a bias (float32, in the order of W's rows, ceil16(N) numbers) or null,
// and how a gated product joins gate and up.
struct GemmEpilogue {
    const float* bias;
    GluAct act;
};
// And what some kernels of their own take beside that (in the arguments of all, it changed the schedule of most: gate and up of 2,048 columns
// and 3 rows 11.8 / 12.3 us).
// unary: what becomes of a result that is not gated (unary_activation), where the streaming kernel or the sum over a split K's
// parts stores it.  plane_cols > 0: several products in one launch.  W's rows are theirs one after the other, plane_cols each; the
// columns of plane p take their rows from A + p * a_step, and C holds the planes [p][M][plane_cols].
struct GemmExtra : GemmEpilogue {
    int unary;
    int plane_cols;
    size_t a_step;
};
// And what only the launches ask.  once: no cache holds the weight from one call to the next (see the streaming kernel's note).
struct GemmCall : GemmExtra {
    int once;
};

// GLU: the 16-row groups of W alternate between a gate and an up projection
// (group 2p gate, group 2p+1 up); the epilogue writes act(gate, up), N / 2 columns: silu(gate) * up, or in the form
// with constants g sigmoid(alpha g) (u + up_offset), g = min(gate, limit), u = clamp(up, -limit, limit).
__device__ __forceinline__ floatx4 glu4(const floatx4& g, const floatx4& u, const GluAct& act) {
    floatx4 o;
    if (act.plain) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = g[e] / (1.0f + __expf(-g[e])) * u[e];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float a = fminf(g[e], act.limit), b = fminf(fmaxf(u[e], -act.limit), act.limit);
            o[e] = a / (1.0f + __expf(-act.alpha * a)) * (b + act.up_offset);
        }
    }
    return o;
}

// Four neighbouring numbers of a bias in the order of W's rows (16 NB of them), for a lane's four columns from n
// on; columns past the end, whose results are never stored, take the last ones.
__device__ __forceinline__ floatx4 bias4(const float* __restrict__ bias, int n, int NB) {
    const float4 b = *reinterpret_cast<const float4*>(bias + min(n, NB * 16 - 4));
    return floatx4{b.x, b.y, b.z, b.w};
}

// ---- up to 16 rows: the streaming kernel (gemm_few_rows.hip) ----
// An RMS norm between two such products costs a kernel of a few microseconds for a few rows.
// Its per-row factor commutes with the product that follows it, so the two products take the
// norm between them (EPI):
//   2, the product before the norm (float32 result): its epilogue adds its result to the
//      residual stream in place, writes the sum times the norm's weight as the bfloat16 input
//      of the next product, *without* the factor rsqrt(mean of squares + eps), and leaves the
//      sum of squares of its 16 columns of every row in ss_out[row][row group];
//   1, the product after the norm: adds up the sums of squares of a row, in a fixed order, and
//      multiplies its float32 accumulators by the row's factor before anything else is done
//      to them.
// The sum of squares is over the float32 residual stream, as in the norm's own kernel.
//   3, the product before a norm that has no statistics (tanh(alpha v) w + b element by element): its
//      epilogue adds its result to the residual stream in place and writes the norm of the sum as the
//      bfloat16 input of the next product, whole: there is no factor to leave to anyone.
struct FewRowsFuse {
    const float* ss_in;     // EPI 1: [16][ss_stride] sums of squares, ss_count of them a row
    int ss_stride, ss_count;
    float inv_dim, eps;     // 1 / row length of the normalised tensor
    float* resid;           // EPI 2: [M, N] float32, updated in place
    const float* norm_w;    // [N]
    bf16_t* x_out;          // [M, N]
    float* ss_out;          // [16][ss_out_stride]
    int ss_out_stride;
    const float* bias;      // EPI 3: [N], and the scalar inside the tanh
    float alpha;
};
// epi: 0 a plain or gated product, else as above.
int tff_gemm_few_rows(int epi, const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall& ex, int c_dtype, int glu_out, hipStream_t s,
                      const FewRowsFuse& fz);
