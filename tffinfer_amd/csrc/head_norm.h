// A recurrence's output per head: o / sqrt(mean over the head of o^2 + eps) * scale * weight * silu(gate), 16 bytes a lane and load.
#pragma once
#include "common.h"

// LPH = D / 4 lanes a head, 64 / LPH heads a wave; `pairs` (token, head) pairs; head h's weight starts at w + h * w_step.
// What bounds it is its rows (ten bytes an element).  A wave a head with four bytes a lane had too few bytes in flight:
// us, that / now: 2,900 tokens of 64 heads of 64 51 / 20 (6.1 TB/s), of 32 heads of 128 35 / 21; one token 2.5 / 2.4.
template <int LPH, typename TO>
__global__ __launch_bounds__(256) void head_norm_gate_vec_kernel(const float* __restrict__ o, const float* __restrict__ g, size_t g_row,
                                                                 const float* __restrict__ w, int w_step, float eps, float scale,
                                                                 TO* __restrict__ out, size_t out_row, int pairs, int H) {
    constexpr int D = LPH * 4, HPW = 64 / LPH;
    const int lane = threadIdx.x & 63, e = (lane % LPH) * 4;
    const int id = (blockIdx.x * 4 + (threadIdx.x >> 6)) * HPW + lane / LPH, p = min(id, pairs - 1);
    const int t = p / H, h = p - t * H;
    const float4 x = *reinterpret_cast<const float4*>(o + (size_t)p * D + e);
    const float4 z = *reinterpret_cast<const float4*>(g + (size_t)t * g_row + (size_t)h * D + e);
    const float4 c = *reinterpret_cast<const float4*>(w + (size_t)h * w_step + e);
    float ss = fmaf(x.x, x.x, fmaf(x.y, x.y, fmaf(x.z, x.z, x.w * x.w)));
#pragma unroll
    for (int s = LPH / 2; s > 0; s >>= 1) ss += __shfl_xor(ss, s, 64);
    const float rr = scale / sqrtf(ss / (float)D + eps);
    const float y[4] = {x.x * rr * c.x * (z.x / (1.0f + expf(-z.x))), x.y * rr * c.y * (z.y / (1.0f + expf(-z.y))),
                        x.z * rr * c.z * (z.z / (1.0f + expf(-z.z))), x.w * rr * c.w * (z.w / (1.0f + expf(-z.w)))};
    if (id >= pairs) return;
    TO* to = out + (size_t)t * out_row + (size_t)h * D + e;
    if constexpr (sizeof(TO) == 4) {
        *reinterpret_cast<float4*>(to) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
        union { bf16_t b[4]; uint2 u; } pk;
#pragma unroll
        for (int k = 0; k < 4; ++k) pk.b[k] = (bf16_t)y[k];
        *reinterpret_cast<uint2*>(to) = pk.u;
    }
}

// Heads of 16 to 256 elements in powers of two on 16-byte aligned rows; false: the caller's general kernel.
template <typename TO>
static bool launch_head_norm_gate(const float* o, const float* g, size_t g_row, const float* w, int w_step, float eps, float scale, TO* out,
                                  size_t out_row, int pairs, int H, int D, hipStream_t s) {
    if (D < 16 || D > 256 || (D & (D - 1)) || g_row % 4 || out_row % 4 || ((uintptr_t)o % 16) || ((uintptr_t)g % 16) || ((uintptr_t)w % 16) ||
        ((uintptr_t)out % 16))
        return false;
    const unsigned blocks = (unsigned)((pairs + 1024 / D - 1) / (1024 / D));       // four waves of 256 / D heads
#define TFF_HN(L) head_norm_gate_vec_kernel<L, TO><<<blocks, 256, 0, s>>>(o, g, g_row, w, w_step, eps, scale, out, out_row, pairs, H)
    switch (D) {
        case 16: TFF_HN(4); break;
        case 32: TFF_HN(8); break;
        case 64: TFF_HN(16); break;
        case 128: TFF_HN(32); break;
        default: TFF_HN(64); break;
    }
#undef TFF_HN
    return true;
}
