// The bfloat16 product of up to 16 rows (decoding: a row a live request): a stream of the weight from HBM into the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16), float32 accumulation; the weight's layout is gemm_bf16.hip's.
//
// A block owns 16 R columns of the result (R row groups of W) for the whole of K.  Its KSPLIT waves take units of 128 k in turn, so that what a
// block reads is one run of memory (runs of a wave's own, a power of two apart, met in the same channels: gated 8,192 x 8,192 26.6 / 22.9 us,
// 24,576 x 4,096 on four waves 40 / 34); each wave reads its fragments of W straight from global memory into MFMA operands, DEPTH units in flight from its
// first to its last: a fragment's registers are loaded again as soon as its MFMAs are issued.  Partial sums meet in LDS and are added in a
// fixed order.  What bounds it is the stream: how soon it begins, how many bytes are in flight, and what else the load units have to fetch.
//
// * The rows of A.  An MFMA's second operand is 16 columns by 32 k, and with few rows most of it is repetition: fetched as such, the rows took as
//   many requests as W, sixteen pieces of 64 bytes beside W's eight lines.  A load of MP = 4 or 8 rows brings 4 or 2 k-steps at once instead:
//   lane (c, g) of it holds row c % MP of step c / MP.  The MFMA of step s then has the right sums in the columns c with c / MP = s, and sums that nobody
//   reads in the others; each of the four steps of a unit has an accumulator of its own, and a wave picks its columns' when its units end.  16
//   rows take two loads of eight, and two MFMAs a step, of which there are plenty.  Every load is eight whole lines.
// * The order of a sum is the same whatever MP, DEPTH and R are: within a wave the steps s, s + 4 KSPLIT, .. of its units, then (s0 + s2) + (s1 + s3), then
//   the waves in turn.  A row's bits hang on KSPLIT alone.
// * The factors of rows that lack their norm's (EPI 1) are added up by all waves, a row or two each, while the first fragments of W travel.
//
// us in a graph of such products over weights that no cache holds, before (sixteen columns of A a fragment, groups of 4 to 32 steps waited for together) /
// now, rows 1, 8, 16: 4,096 x 1,024 after a norm 4.1, 4.4, 4.8 / 3.5, 3.7, 4.1; 1,024 x 3,072 before a norm 5.4, 6.2, 8.0 / 4.3, 5.2, 6.3;
// 6,144 x 4,096 12.6, 14.1, 17.7 / 10.0, 10.8, 12.2; 4,096 x 12,288 18.7, 22.3, 28.5 / 17.7, 18.2, 21.3; gated 12,288 x 2,048 14.5, 15.4, 17.3 / 10.6,
// 11.3, 13.3, 24,576 x 4,096 35.7, 36.1, 38.9 (tiles) / 33.3, 32.7, 34.5 (6.1 TB/s).
//
// Where the caller says that no cache holds the weight from one call to the next (once: a model's weights are more than the 256 MB behind the
// L2), its loads say that nobody asks for the line again (nt): the caches then keep the rows of A and do not write lines about
// that nothing will hit.  us, four decode steps of 8 requests on 8 layers of the 8B shape 4,300 / 4,057, a prompt of 96 tokens and 15
// decode steps of the 0.6B shape 18,700 / 17,800; the head of 151,936 columns, 3 rows, 200 / 177 (7.0 TB/s).
// Weights that do fit lose by it: four of 5,120 x 5,120 (210 MB) in turn, 8 rows, 10.6 / 15.8 us, 24 of 4,096 x 1,024, one row, 3.4 / 3.7.
// The four-wave kernel has the same where it reads a weight once (launch_w4).
// Weights that others read too (several row tiles), or in pieces of 64 bytes (float32 rows, 8,030 -> 8,200), lose by it.
#include "gemm_bf16.h"
#include "tffinfer_kernels.h"

// MORE: several products in one launch, or an activation of the result (GemmExtra).  Kernels of their own: the tests for them and the registers
// of the activations cost every plain product 0.2 us.
// Sixteen rows of a gate and its up group with one unit in flight are at the 256 registers that two waves a SIMD have, on either side of them by what the
// epilogue takes; the compiler has to stay below (16 rows without factors, 25,728 x 2,056 with one wave a SIMD 29.6 us, with two 24.1; four rows more
// than eight cost 0.2 us).
template <int MP, bool GLU, int DEPTH, int KSPLIT>
constexpr int few_rows_waves() { return MP == 16 && GLU && DEPTH == 1 && KSPLIT <= 4 ? 2 : 1; }

template <int MP, int R, int DEPTH, int KSPLIT, bool GLU, int EPI, bool MORE, bool ONCE>
__global__ __launch_bounds__(64 * KSPLIT, (few_rows_waves<MP, GLU, DEPTH, KSPLIT>())) void gemm_bf16_few_rows_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wp, void* __restrict__ C, int c_float32, int M, int N, int K, int lda, int KB, int n_out,
    const FewRowsFuse fz, const typename std::conditional<MORE, GemmExtra, GemmEpilogue>::type ex) {
    static_assert(MP == 4 || MP == 8 || MP == 16, "rows a load packs");
    static_assert(DEPTH == 1 || DEPTH == 2, "the ends of the stream are written for one unit in flight and for two");
    static_assert(!GLU || R == 2, "a gate and its up group are a wave's");
    static_assert(EPI < 2 || !GLU, "the product before a norm has a plain float32 result");
    static_assert(!MORE || (EPI == 0 && !GLU), "planes and activations are for plain products");
    constexpr int H = MP == 16 ? 2 : 1;                  // halves of the rows, a load and an MFMA each
    constexpr int AL = MP == 4 ? 1 : 2;                  // loads of a half's rows a unit
    __shared__ floatx4 part[KSPLIT][R][64];
    __shared__ float row_factor[EPI == 1 ? 16 : 1];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int NB = (N + 15) / 16;
    const int nb0 = blockIdx.x * R;
    int ldc = GLU ? n_out : N;
    size_t c_base = 0;
    if constexpr (MORE) {
        if (ex.plane_cols) {      // (a wave's columns are one plane's; C as its column 0 of row 0 would lie)
            const size_t plane = (size_t)(min(nb0, NB - 1) * 16 / ex.plane_cols);
            A += plane * ex.a_step;
            c_base = plane * (size_t)(M - 1) * ex.plane_cols;
            ldc = ex.plane_cols;
        }
    }
    // (the result's type is looked at where it is stored: a kernel for each would be another hundred)
    auto store = [&](size_t at, const floatx4& v, int n, int cols) {
        if (c_float32) store4<float>((float*)C + at, v, n, cols, (ldc % 4) == 0);
        else store4<bf16_t>((bf16_t*)C + at, v, n, cols, (ldc % 4) == 0);
    };

    // What the epilogue needs from memory is asked for first, so that it has arrived long before the stream of W ends.
    float4 resid_in[R], normw_in[R], bias_in[R];
#pragma unroll
    for (int r = 0; r < R; ++r) resid_in[r] = normw_in[r] = bias_in[r] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (wave == 0) {
        if constexpr (EPI >= 2) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int n = (nb0 + r) * 16 + fg * 4;
                if (fr < M && n < N) {
                    resid_in[r] = *reinterpret_cast<const float4*>(fz.resid + (size_t)fr * N + n);
                    normw_in[r] = *reinterpret_cast<const float4*>(fz.norm_w + n);
                    if constexpr (EPI == 3) bias_in[r] = *reinterpret_cast<const float4*>(fz.bias + n);
                }
            }
        } else if (ex.bias) {
#pragma unroll
            for (int r = 0; r < R; ++r) bias_in[r] = *reinterpret_cast<const float4*>(ex.bias + min((nb0 + r) * 16 + fg * 4, NB * 16 - 4));
        }
    }
    // EPI 1: the sums of squares of rows wave, wave + KSPLIT, .. : the first 256 of each row are asked for here
    constexpr int SR = EPI == 1 ? (MP + KSPLIT - 1) / KSPLIT : 1;
    float4 ssv[SR];
    if constexpr (EPI == 1) {
#pragma unroll
        for (int i = 0; i < SR; ++i) {
            const int row = wave + i * KSPLIT;
            ssv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (row < M && lane * 4 < (fz.ss_count & ~3)) ssv[i] = *reinterpret_cast<const float4*>(fz.ss_in + (size_t)row * fz.ss_stride + lane * 4);
        }
    }

    // Units of 128 k are dealt to the waves in turn.  Row groups past the end of W and rows past the end of A repeat the last.
    const int units = (KB + 3) >> 2;
    const int count = (units - wave + KSPLIT - 1) / KSPLIT;        // (0: a wave without work)
    auto unit = [&](int i) { return wave + i * KSPLIT; };
    const bf16_t* wgroup[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wgroup[r] = Wp + (size_t)min(nb0 + r, NB - 1) * KB * 512;
    const int packed = MP == 4 ? fr & 3 : fr & 7;        // the row of a half, and the step of a load, that this lane's column holds
    const int step_of = MP == 4 ? fr >> 2 : fr >> 3;
    const bf16_t* arow[H];
#pragma unroll
    for (int h = 0; h < H; ++h) arow[h] = A + (size_t)min(h * 8 + packed, M - 1) * lda;
    const int lane_k = step_of * 32 + fg * 8;

    floatx4 acc[R][H][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
            for (int s = 0; s < 4; ++s) acc[r][h][s] = floatx4{0.f, 0.f, 0.f, 0.f};

    uint4 rw[DEPTH][R][4], ra[DEPTH][H][AL];
    // (a unit that W or A end in: steps and k past the end load the last ones and are not used)
    auto load_w = [&](int slot, int u, int s) {
#pragma unroll
        for (int r = 0; r < R; ++r) rw[slot][r][s] = ld16_weight<ONCE>(wgroup[r] + (size_t)min(u * 4 + s, KB - 1) * 512 + lane * 8);
    };
    auto load_a = [&](int slot, int u, int j) {
        const int k = min(u * 128 + j * 64 + lane_k, K - 8);
#pragma unroll
        for (int h = 0; h < H; ++h) ra[slot][h][j] = ld16(arow[h] + k);
    };
    auto load_unit = [&](int slot, int u) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            load_w(slot, u, s);
            if (s % (4 / AL) == 0) load_a(slot, u, s / (4 / AL));
        }
    };
    auto step = [&](int slot, int s) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int h = 0; h < H; ++h)
                acc[r][h][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(rw[slot][r][s]), as_frag(ra[slot][h][s / (4 / AL)]), acc[r][h][s], 0, 0, 0);
    };
    // unit u of a slot; its registers are loaded with unit `next` step by step
    auto use = [&](int slot, int u, int next, auto REFILL) {
        constexpr bool refill = decltype(REFILL)::value;
        if (!refill && u * 128 + 128 > K) {              // (the last unit of all: nothing is loaded behind it)
#pragma unroll
            for (int j = 0; j < AL; ++j)
                if (u * 128 + j * 64 + lane_k >= K)
#pragma unroll
                    for (int h = 0; h < H; ++h) ra[slot][h][j] = make_uint4(0, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < 4; ++s)
                if (u * 4 + s < KB) step(slot, s);
            return;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            step(slot, s);
            if constexpr (refill) {
                load_w(slot, next, s);
                if (s % (4 / AL) == 4 / AL - 1) load_a(slot, next, s / (4 / AL));
            }
        }
    };
    constexpr auto refill = std::true_type{};
    constexpr auto drain = std::false_type{};
    // the factors: while the first fragments travel
    auto factors = [&]() {
        if constexpr (EPI == 1) {
#pragma unroll
            for (int i = 0; i < SR; ++i) {
                const int row = wave + i * KSPLIT;
                if (row >= M) break;
                const float* sp = fz.ss_in + (size_t)row * fz.ss_stride;
                const int vec_end = fz.ss_count & ~3;
                float s = (ssv[i].x + ssv[i].y) + (ssv[i].z + ssv[i].w);
                for (int j = 256 + lane * 4; j < vec_end; j += 256) {
                    const float4 v = *reinterpret_cast<const float4*>(sp + j);
                    s += (v.x + v.y) + (v.z + v.w);
                }
                if (lane < fz.ss_count - vec_end) s += sp[vec_end + lane];
                s = rows_sum(row16_sum(s));
                if (lane == 0) row_factor[row] = rsqrtf(s * fz.inv_dim + fz.eps);
            }
        }
    };
    if (count >= DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) load_unit(d, unit(d));
        factors();
        int i = 0;                                       // (slot d holds unit i + d)
        for (; i + 2 * DEPTH <= count; i += DEPTH)
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) use(d, unit(i + d), unit(i + d + DEPTH), refill);
        const int more = count - i - DEPTH;              // units that are not loaded yet, fewer than DEPTH
        auto end = [&](auto MORE_UNITS) {
            constexpr int m = decltype(MORE_UNITS)::value;
#pragma unroll
            for (int d = 0; d < m; ++d) use(d, unit(i + d), unit(i + d + DEPTH), refill);
#pragma unroll
            for (int d = m; d < DEPTH; ++d) use(d, unit(i + d), 0, drain);
#pragma unroll
            for (int d = 0; d < m; ++d) use(d, unit(i + d + DEPTH), 0, drain);
        };
        if (more == 0) end(std::integral_constant<int, 0>{});
        if constexpr (DEPTH > 1) { if (more == 1) end(std::integral_constant<int, 1>{}); }
    } else {
        auto all = [&](auto UNITS) {
            constexpr int m = decltype(UNITS)::value;
#pragma unroll
            for (int d = 0; d < m; ++d) load_unit(d, unit(d));
            factors();
#pragma unroll
            for (int d = 0; d < m; ++d) use(d, unit(d), 0, drain);
        };
        if (count <= 0) factors();
        if constexpr (DEPTH > 1) { if (count == 1) all(std::integral_constant<int, 1>{}); }
    }

    // The steps' sums of the columns that hold them, row fr's in lane fr of a row of sixteen lanes.
    floatx4 sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#define TFF_ROR(x, n) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + (n), 0xF, 0xF, true))
            if constexpr (MP == 4) {
                const float lo = step_of & 1 ? acc[r][0][1][e] : acc[r][0][0][e], hi = step_of & 1 ? acc[r][0][3][e] : acc[r][0][2][e];
                float v = step_of & 2 ? hi : lo;
                v += TFF_ROR(v, 8);                      // steps 0 and 2, 1 and 3
                sum[r][e] = v + TFF_ROR(v, 4);
            } else {
                float v[H];
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    v[h] = step_of ? acc[r][h][1][e] + acc[r][h][3][e] : acc[r][h][0][e] + acc[r][h][2][e];
                    v[h] += TFF_ROR(v[h], 8);
                }
                sum[r][e] = H == 2 && fr >= 8 ? v[H - 1] : v[0];
            }
#undef TFF_ROR
        }
    }
    if constexpr (KSPLIT > 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) part[wave][r][lane] = sum[r];
    }
    if constexpr (KSPLIT > 1 || EPI == 1) __syncthreads();
    if (wave != 0) return;      // the first wave adds up, in the order of K
    if constexpr (KSPLIT > 1) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int w = 1; w < KSPLIT; ++w) {
                const floatx4 p = part[w][r][lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[r][e] += p[e];
            }
    }
    const int m = fr;
    if constexpr (EPI == 1) {
        const float f = row_factor[min(m, M - 1)];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[r][e] *= f;
    } else if constexpr (EPI == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            sum[r][0] += bias_in[r].x; sum[r][1] += bias_in[r].y; sum[r][2] += bias_in[r].z; sum[r][3] += bias_in[r].w;
        }
    }
    if constexpr (GLU) {
        const int n = (nb0 >> 1) * 16 + fg * 4;
        if (m < M && n < n_out) store((size_t)m * ldc + n, glu4(sum[0], sum[1], ex.act), n, n_out);
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            floatx4 v = sum[r];
            const int n = (nb0 + r) * 16 + fg * 4;
            if constexpr (EPI == 2) {
                // N is a multiple of 4 here: four columns are in or out together
                float ss = 0.f;
                if (m < M && n < N) {
                    const float4 s = make_float4(resid_in[r].x + v[0], resid_in[r].y + v[1], resid_in[r].z + v[2], resid_in[r].w + v[3]);
                    *reinterpret_cast<float4*>(fz.resid + (size_t)m * N + n) = s;
                    union { bf16_t h[4]; uint2 u; } pk;
                    pk.h[0] = (bf16_t)(s.x * normw_in[r].x);
                    pk.h[1] = (bf16_t)(s.y * normw_in[r].y);
                    pk.h[2] = (bf16_t)(s.z * normw_in[r].z);
                    pk.h[3] = (bf16_t)(s.w * normw_in[r].w);
                    *reinterpret_cast<uint2*>(fz.x_out + (size_t)m * N + n) = pk.u;
                    ss = fmaf(s.x, s.x, fmaf(s.y, s.y, fmaf(s.z, s.z, s.w * s.w)));
                }
                ss += __shfl_xor(ss, 16, 64);
                ss += __shfl_xor(ss, 32, 64);
                if (fg == 0 && nb0 + r < NB) fz.ss_out[(size_t)fr * fz.ss_out_stride + nb0 + r] = ss;
            } else if constexpr (EPI == 3) {
                if (m < M && n < N) {
                    const float4 s = make_float4(resid_in[r].x + v[0], resid_in[r].y + v[1], resid_in[r].z + v[2], resid_in[r].w + v[3]);
                    *reinterpret_cast<float4*>(fz.resid + (size_t)m * N + n) = s;
                    union { bf16_t h[4]; uint2 u; } pk;
                    pk.h[0] = (bf16_t)fmaf(tanhf(fz.alpha * s.x), normw_in[r].x, bias_in[r].x);
                    pk.h[1] = (bf16_t)fmaf(tanhf(fz.alpha * s.y), normw_in[r].y, bias_in[r].y);
                    pk.h[2] = (bf16_t)fmaf(tanhf(fz.alpha * s.z), normw_in[r].z, bias_in[r].z);
                    pk.h[3] = (bf16_t)fmaf(tanhf(fz.alpha * s.w), normw_in[r].w, bias_in[r].w);
                    *reinterpret_cast<uint2*>(fz.x_out + (size_t)m * N + n) = pk.u;
                }
            } else if (m < M && n < N) {
                if constexpr (MORE) {
                    if (ex.unary) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = unary_activation(v[e], ex.unary);
                    }
                }
                store(c_base + (size_t)m * ldc + n, v, n, N);
            }
        }
    }
}

template <int MP, int R, int DEPTH, int KSPLIT, bool GLU, int EPI>
static int launch_few_rows(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall& ex, int c_dtype, int n_out, hipStream_t s,
                           const FewRowsFuse& fz) {
    const int KB = (K + 31) / 32;
    const dim3 grid(((N + 15) / 16 + R - 1) / R);
    auto launch = [&](auto ONCE) {
        constexpr bool once = decltype(ONCE)::value;
        if constexpr (EPI == 0 && !GLU) {
            if (ex.plane_cols || ex.unary) {
                gemm_bf16_few_rows_kernel<MP, R, DEPTH, KSPLIT, false, 0, true, once><<<grid, 64 * KSPLIT, 0, s>>>(A, Wp, C, c_dtype == TFF_F32, M, N, K, lda, KB, n_out, fz, ex);
                return;
            }
        }
        gemm_bf16_few_rows_kernel<MP, R, DEPTH, KSPLIT, GLU, EPI, false, once><<<grid, 64 * KSPLIT, 0, s>>>(A, Wp, C, c_dtype == TFF_F32, M, N, K, lda, KB, n_out, fz, ex);
    };
    if (ex.once) launch(std::true_type{});
    else launch(std::false_type{});
    return tff_check_launch("gemm_bf16_few_rows");
}

// Row groups a block, units in flight and waves, by the columns, K and the rows.  How many waves share K goes by the columns and K alone (but for
// wide gated weights, see there).  Fitted to 300 products of 192 to 12,288 k and 256 to 34,816 columns, rows 2, 8 and 16, and, where K is short or the
// weight gated, to 14,600 of 64 to 12,000 k and 64 to 60,000 columns; us beside the rules.
// With a short K and many columns the blocks are many and their work little: a CU goes through them as fast as its registers hold waves with work, so
// that no more waves share K than it has units for (12 rows, 59,520 x 64 on four waves 13.0, on one 5.9; 16 rows, 55,040 x 152 13.7 and 7.5, on four
// waves and on two 16,384 x 512 7.0 and 5.6).
template <int MP, int EPI>
static int few_rows_for(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall& ex, int c_dtype, int glu_out, hipStream_t s,
                        const FewRowsFuse& fz) {
#define TFF_FEW(R, DEPTH, KSPLIT, GLU) return launch_few_rows<MP, R, DEPTH, KSPLIT, GLU, EPI>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz)
    const int cus = tff_device_cus(), nb = (N + 15) / 16;
    if (glu_out > 0) {
        if constexpr (EPI < 2) {
            // A pair of groups a CU or less: a block has to keep its CU's share of the stream in flight alone.  (Two units of sixteen rows are
            // more registers than eight waves have: spilled, 2,560 k took twice as long.)  With the rows' factors to add up, eight waves also for a short K.
            if (nb <= 2 * cus) {
                if (EPI == 0 && K <= 512) TFF_FEW(2, 2, 2, true);
                if constexpr (MP < 16) TFF_FEW(2, 2, 8, true);
                else TFF_FEW(2, 1, 8, true);
            }
            // Two waves: 16 rows, 12,800 x 264 gated 5.3 on eight, 4.8 on two; after a norm 7.9 and 7.0.
            if (nb <= 4 * cus) TFF_FEW(2, 2, 2, true);
            // Eight waves of a short K have a unit or none: 18,432 x 1,024, 2 / 8 / 16 rows, two waves 9.1 / 9.4 / 10.6, eight 9.4 / 9.8 / 13.7.
            if (K < 2048) TFF_FEW(2, 1, 2, true);
            // More, and more than eight rows: blocks of four waves, of which a CU holds more at sixteen rows' registers (34,816 x 5,120, 16 rows,
            // four waves 68.5, eight 73.4; 2 rows 59.2, 57.4).
            if constexpr (MP < 16) TFF_FEW(2, 1, 8, true);
            else TFF_FEW(2, 1, 4, true);
        } else {
            return tff_fail("gemm: a gated product does not come before a norm");
        }
    } else {
        // A group a CU or less: as above (2,048 x 12,288, 2 rows, eight waves 12.1, four 12.8).
        if (nb <= cus) {
            if (EPI != 1 && K <= 256) TFF_FEW(1, 2, 2, false);
            TFF_FEW(1, 2, 8, false);
        }
        // (up to two groups a CU the rows' factors are what a block of few waves waits for)
        if (nb <= 4 * cus) {
            if (K <= 1024 && (EPI != 1 || nb > 2 * cus)) TFF_FEW(1, 2, 2, false);
        } else if (K <= 896) {
            if constexpr (EPI == 1) TFF_FEW(1, 2, 2, false);
            else TFF_FEW(1, 2, 1, false);
        }
        // A few groups a CU: two groups a block, which then all run at once and fetch the rows for two (6,144 x 12,288, 16 rows, 30.9,
        // one group a block 36.8); up to four rows there is little to fetch, and one group a block begins sooner (25.6 and 26.4).
        if constexpr (MP == 4) {
            if (nb < 2 * cus) TFF_FEW(1, 1, 4, false);
        } else {
            // sixteen rows are as many bytes from L2 as a group's columns are from HBM: two groups also for the widest weights
            // (24,576 x 8,192 65.8, one group 73.6; 12,288 x 4,096 22.9 and 20.8)
            const bool two = MP == 8 ? nb * 4 <= cus * 7 : nb <= 2 * cus || (nb >= 6 * cus && K >= 2560);
            if (two) TFF_FEW(2, 2, 4, false);
        }
        TFF_FEW(1, 2, 4, false);
    }
#undef TFF_FEW
}

template <int EPI>
static int few_rows_of(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall& ex, int c_dtype, int glu_out, hipStream_t s,
                       const FewRowsFuse& fz) {
    if (M <= 4) return few_rows_for<4, EPI>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz);
    if (M <= 8) return few_rows_for<8, EPI>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz);
    return few_rows_for<16, EPI>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz);
}

int tff_gemm_few_rows(int epi, const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall& ex, int c_dtype, int glu_out, hipStream_t s,
                      const FewRowsFuse& fz) {
    TFF_REQUIRE(M >= 1 && M <= 16, "gemm: %d rows for the kernel of up to 16", M);
    TFF_REQUIRE(!(glu_out > 0 && (ex.plane_cols || ex.unary)), "gemm: planes or an activation of a gated product");
    if (epi == 0) return few_rows_of<0>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz);
    if (epi == 1) return few_rows_of<1>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, fz);
    if (epi == 2) return few_rows_of<2>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, fz);
    return few_rows_of<3>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, fz);
}
