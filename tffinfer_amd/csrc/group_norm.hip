// Norms on a sublayer's OUTPUT and sums over the depth of the model.
//
// tff_group_rmsnorm_add: a row of `delta` (a sublayer's output, perhaps as `planes` partial sums,
//   `plane` elements apart, added up first in their order) is cut into `groups` equal consecutive
//   parts; each part is divided by its own sqrt(mean(part^2) + eps); the whole is multiplied by w.
//   With `resid` the result is added into that row of the float32 residual stream, and `out`
//   (optional) gets the new row in the activation type.  Without `resid` the result itself goes to
//   `out`; `rows` (optional) then names the rows of `delta` to take (the rows whose logits are
//   wanted).  Sums, means, roots and products in float32.
// tff_depth_average: hist[n - 1] <- x;  x <- sum_{j < n} coef[j] * hist[j] (j ascending), with
//   hist [depths, T, W] the outputs of the embedding and of the layers so far; `out` (optional)
//   gets x in the activation type.
// tff_scale_rows: x <- alpha * x on float32 rows.
#include "common.h"
#include "tffinfer_kernels.h"

#define GN_THREADS 256

// One block per (row, group); GN_ITS x 256 elements of a group pass through memory once: 2048 at most.  Bound by latency for few
// rows and by memory for many: element by element the planes are added one load after the other, and weight and stream asked for after
// the sum over the group.  EARLY: all loads under way first, the same sums in the same order; us without / with: 2 rows of 4096 in one
// group 8.2 / 5.7, in four with four planes 5.1 / 3.8, 8 rows of 6000 14.1 / 10.4, 400 rows of 8192 24.8 / 16.5, 1,500 rows of 4096 in eight
// groups 25.0 / 19.9, in two with eight planes 52.6 / 50.1.
// DEPTH: the new row is a level of the sum over depth, which takes its place in the stream and goes to `out` (tff_depth_average in the same
// launch): the levels before do not wait for the norm, and the stream is not written and read in between.  For groups that pass through memory
// once (tff_group_depth_in_norm).
struct GroupDepth {
    float* hist;
    const float* coef;
    size_t level;
    int n;
};
template <typename TO, int GN_ITS, bool EARLY, bool DEPTH>
__global__ __launch_bounds__(GN_THREADS) void group_rmsnorm_add_kernel(
    float* __restrict__ resid, const float* __restrict__ delta, int planes, size_t plane,
    const int32_t* __restrict__ rows, const float* __restrict__ w, int groups, float eps,
    TO* __restrict__ out, int H, const GroupDepth dp) {
    __shared__ float red[17];
    const int r = blockIdx.x / groups, g = blockIdx.x % groups, tid = threadIdx.x;
    const int src = rows ? rows[r] : r;
    const int Hg = H / groups, base = g * Hg;
    const float* dl = delta + (size_t)src * H + base;
    float* x = resid ? resid + (size_t)r * H + base : nullptr;
    TO* o = out ? out + (size_t)r * H + base : nullptr;
    const float* wg = w + base;
    auto term = [&](int j) {
        float d = dl[j];
        for (int p = 1; p < planes; ++p) d += dl[p * plane + j];
        return d;
    };
    // (all loads of the row, what the sum is multiplied with and added to included, are on their way before the first is waited for;
    // past the row's end its last element again)
    float cache[GN_ITS], wr[GN_ITS], xr[GN_ITS];
#pragma unroll
    for (int it = 0; it < GN_ITS; ++it) {
        const int j = min(tid + it * GN_THREADS, Hg - 1);
        cache[it] = EARLY ? dl[j] : term(j);
        wr[it] = EARLY ? wg[j] : 0.f;
        xr[it] = EARLY && x ? x[j] : 0.f;
    }
    if constexpr (EARLY) {
#pragma unroll 4
        for (int p = 1; p < planes; ++p)
#pragma unroll
            for (int it = 0; it < GN_ITS; ++it) cache[it] += dl[p * plane + min(tid + it * GN_THREADS, Hg - 1)];
    }
    float* const hist = DEPTH ? dp.hist + (size_t)r * H + base : nullptr;
    float acc[DEPTH ? GN_ITS : 1];
    if constexpr (DEPTH) {
#pragma unroll
        for (int it = 0; it < GN_ITS; ++it) acc[it] = 0.f;
#pragma unroll 2
        for (int l = 0; l + 1 < dp.n; ++l) {
            const float c = dp.coef[l];
#pragma unroll
            for (int it = 0; it < GN_ITS; ++it) acc[it] = fmaf(c, hist[l * dp.level + min(tid + it * GN_THREADS, Hg - 1)], acc[it]);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int it = 0; it < GN_ITS; ++it)
        if (tid + it * GN_THREADS < Hg) ss = fmaf(cache[it], cache[it], ss);
    for (int j = tid + GN_ITS * GN_THREADS; j < Hg; j += GN_THREADS) {
        const float d = term(j);
        ss = fmaf(d, d, ss);
    }
    ss = block_sum(ss, red);
    const float rr = 1.0f / sqrtf(ss / (float)Hg + eps);
    auto emit = [&](int j, float d, float weight, float before, float levels) {
        float y = d * rr * weight;
        if (x) {
            y += before;
            if constexpr (DEPTH) {
                hist[(dp.n - 1) * dp.level + j] = y;
                y = fmaf(dp.coef[dp.n - 1], y, levels);
            }
            x[j] = y;
        }
        if (o) o[j] = from_f32<TO>(y);
    };
#pragma unroll
    for (int it = 0; it < GN_ITS; ++it) {
        const int j = tid + it * GN_THREADS;
        if (j < Hg) emit(j, cache[it], EARLY ? wr[it] : wg[j], EARLY ? xr[it] : x ? x[j] : 0.f, DEPTH ? acc[it] : 0.f);
    }
    if constexpr (!DEPTH)
        for (int j = tid + GN_ITS * GN_THREADS; j < Hg; j += GN_THREADS) emit(j, term(j), wg[j], x ? x[j] : 0.f, 0.f);
}

template <bool DEPTH>
static int group_norm_launch(float* resid, const float* delta, int planes, size_t plane, const int32_t* rows, const float* w, int groups,
                             float eps, void* out, int n, int H, int out_dtype, const GroupDepth dp, tff_stream_t stream) {
    TFF_REQUIRE(delta && w && (resid || out), "group_rmsnorm_add: null pointer");
    TFF_REQUIRE(n >= 0 && H > 0 && groups > 0 && H % groups == 0, "group_rmsnorm_add: rows of %d in %d groups", H, groups);
    TFF_REQUIRE(planes >= 1 && !(rows && (resid || planes > 1)), "group_rmsnorm_add: bad combination of operands");
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const int Hg = H / groups;
    // The early loads of groups over 1024 take 117 registers, four blocks to a CU instead of eight: worth it while the blocks are there
    // at once (1,024), and where neither a tail behind 2048 elements nor many planes keep the memory busy.  us late / early: 1,000 rows of
    // 4096 13.9 / 12.5, 1,100 rows 14.3 / 19.4, with eight planes 60.2 / 56.7 and 60.6 / 87.8; 1,000 rows of 4096 in two groups with eight
    // planes 31.5 / 35.9, with two 16.7 / 15.1.
    const bool early = (long)n * groups <= 1024 || (Hg <= 8 * GN_THREADS && planes <= 4);
#define GN_LAUNCH(T, ITS, EARLY) \
    group_rmsnorm_add_kernel<T, ITS, EARLY, DEPTH><<<n * groups, GN_THREADS, 0, s>>>(resid, delta, planes, plane, rows, w, groups, eps, (T*)out, H, dp)
#define GN_BY_SIZE(T)                                           \
    do {                                                        \
        if (Hg <= GN_THREADS) GN_LAUNCH(T, 1, true);            \
        else if (Hg <= 2 * GN_THREADS) GN_LAUNCH(T, 2, true);   \
        else if (Hg <= 4 * GN_THREADS) GN_LAUNCH(T, 4, true);   \
        else if (early) GN_LAUNCH(T, 8, true);                  \
        else GN_LAUNCH(T, 8, false);                            \
    } while (0)
    if (!out || out_dtype == TFF_F32) GN_BY_SIZE(float);
    else if (out_dtype == TFF_BF16) GN_BY_SIZE(bf16_t);
    else
        return tff_fail("group_rmsnorm_add: unknown dtype %d", out_dtype);
#undef GN_BY_SIZE
#undef GN_LAUNCH
    return tff_check_launch("group_rmsnorm_add");
}
TFF_API int tff_group_rmsnorm_add(float* resid, const float* delta, int planes, size_t plane, const int32_t* rows,
                                  const float* w, int groups, float eps, void* out, int n, int H, int out_dtype,
                                  tff_stream_t stream) {
    return group_norm_launch<false>(resid, delta, planes, plane, rows, w, groups, eps, out, n, H, out_dtype, GroupDepth{}, stream);
}
template <typename TO>
__global__ __launch_bounds__(256) void depth_average_kernel(float* __restrict__ hist, size_t level, int n,
                                                            const float* __restrict__ coef, float* __restrict__ x,
                                                            TO* __restrict__ out, size_t count, int whole) {
    // bound by memory, and for few rows by the levels' latency: 2 rows of 4096 over 6 levels 5.0 us element by element, 2.6 now; 1,500 rows
    // over 12 levels (one more read, three written) 103 / 62, over 3 40 / 21
    // four elements a thread; `count` is a multiple of 4 or the tail goes one by one
    const size_t i4 = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i4 >= count) return;
    if (whole) {                                           // (the same sums, eight levels' loads of 16 bytes in flight)
        const float4 v = *reinterpret_cast<const float4*>(x + i4);
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
        for (int j = 0; j + 1 < n; ++j) {
            const float c = coef[j];
            const float4 h = *reinterpret_cast<const float4*>(hist + (size_t)j * level + i4);
            acc.x = fmaf(c, h.x, acc.x);
            acc.y = fmaf(c, h.y, acc.y);
            acc.z = fmaf(c, h.z, acc.z);
            acc.w = fmaf(c, h.w, acc.w);
        }
        const float cl = coef[n - 1];
        *reinterpret_cast<float4*>(hist + (size_t)(n - 1) * level + i4) = v;
        const float4 y = make_float4(fmaf(cl, v.x, acc.x), fmaf(cl, v.y, acc.y), fmaf(cl, v.z, acc.z), fmaf(cl, v.w, acc.w));
        *reinterpret_cast<float4*>(x + i4) = y;
        if (out) {
            out[i4] = from_f32<TO>(y.x);
            out[i4 + 1] = from_f32<TO>(y.y);
            out[i4 + 2] = from_f32<TO>(y.z);
            out[i4 + 3] = from_f32<TO>(y.w);
        }
        return;
    }
    const int m = (int)((count - i4) < 4 ? (count - i4) : 4);
    float v[4], acc[4];
    for (int e = 0; e < m; ++e) {
        v[e] = x[i4 + e];
        acc[e] = 0.f;
    }
    for (int j = 0; j + 1 < n; ++j) {
        const float c = coef[j];
        const float* hj = hist + (size_t)j * level + i4;
        for (int e = 0; e < m; ++e) acc[e] = fmaf(c, hj[e], acc[e]);
    }
    const float cl = coef[n - 1];
    float* hl = hist + (size_t)(n - 1) * level + i4;
    for (int e = 0; e < m; ++e) {
        hl[e] = v[e];
        const float y = fmaf(cl, v[e], acc[e]);
        x[i4 + e] = y;
        if (out) out[i4 + e] = from_f32<TO>(y);
    }
}

TFF_API int tff_depth_average(float* hist, size_t level, int n, const float* coef, float* x, void* out, size_t count,
                              int out_dtype, tff_stream_t stream) {
    TFF_REQUIRE(hist && coef && x, "depth_average: null pointer");
    TFF_REQUIRE(n >= 1 && level >= count, "depth_average: %d levels of %zu for %zu elements", n, level, count);
    if (count == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const unsigned blocks = (unsigned)((count + 1023) / 1024);
    const int whole = count % 4 == 0 && level % 4 == 0 && ((uintptr_t)hist % 16) == 0 && ((uintptr_t)x % 16) == 0;
    if (!out || out_dtype == TFF_F32)
        depth_average_kernel<float><<<blocks, 256, 0, s>>>(hist, level, n, coef, x, (float*)out, count, whole);
    else if (out_dtype == TFF_BF16)
        depth_average_kernel<bf16_t><<<blocks, 256, 0, s>>>(hist, level, n, coef, x, (bf16_t*)out, count, whole);
    else
        return tff_fail("depth_average: unknown dtype %d", out_dtype);
    return tff_check_launch("depth_average");
}

// Whether the sum over depth goes with the norm.  Not for groups that a block reads more than once, whose elements past the first 2,048 would
// take a load a level one after the other; nor, for few blocks, over many levels: a block asks for two levels at a time, the sum by
// itself for eight.  us, two launches / one, rows of 4,096 in two groups: one row, 4, 7, 12 and 33 levels 5.6 / 4.9, 5.9 / 5.3, 5.8 / 6.0 and 6.2 / 9.0;
// 48 rows, 12 and 20 levels 6.7 / 6.3 and 6.9 / 7.4; 128 rows, 20 and 33 12.6 / 11.4 and 16.3 / 15.2; 1,500 rows, 33 186 / 172; in one group, one row,
// 7 and 33 levels 8.9 / 12.6 and 9.2 / 36.
TFF_API int tff_group_depth_in_norm(int n, int H, int groups, int levels) {
    const long blocks = (long)n * groups;
    return H / groups <= 8 * GN_THREADS && (levels <= (blocks < 64 ? 10 : blocks < 256 ? 12 : 20) || blocks >= 512);
}
TFF_API int tff_group_rmsnorm_add_depth(float* resid, const float* delta, int planes, size_t plane, const float* w, int groups, float eps,
                                        float* hist, size_t level, int levels, const float* coef, void* out, int n, int H, int out_dtype,
                                        tff_stream_t stream) {
    TFF_REQUIRE(resid && hist && coef && levels >= 1 && level >= (size_t)n * H, "group_rmsnorm_add_depth: %d levels, %zu apart, of %d rows of %d", levels,
                level, n, H);
    TFF_REQUIRE(n >= 0 && H > 0 && groups > 0 && H % groups == 0, "group_rmsnorm_add_depth: rows of %d in %d groups", H, groups);
    if (tff_group_depth_in_norm(n, H, groups, levels))
        return group_norm_launch<true>(resid, delta, planes, plane, nullptr, w, groups, eps, out, n, H, out_dtype, GroupDepth{hist, coef, level, levels}, stream);
    if (int rc = group_norm_launch<false>(resid, delta, planes, plane, nullptr, w, groups, eps, nullptr, n, H, TFF_F32, GroupDepth{}, stream)) return rc;
    return tff_depth_average(hist, level, levels, coef, resid, out, (size_t)n * H, out_dtype, stream);
}

__global__ __launch_bounds__(256) void scale_rows_kernel(float* __restrict__ x, float alpha, size_t count) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < count) x[i] *= alpha;
}

TFF_API int tff_scale_rows(float* x, float alpha, size_t count, tff_stream_t stream) {
    TFF_REQUIRE(x, "scale_rows: null pointer");
    if (count == 0) return 0;
    scale_rows_kernel<<<(unsigned)((count + 255) / 256), 256, 0, (hipStream_t)stream>>>(x, alpha, count);
    return tff_check_launch("scale_rows");
}
