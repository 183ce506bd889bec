// float32 matrix product C = A . W^T on the float32 matrix cores (v_mfma_f32_16x16x4_f32: whole float32 operands,
// products and sums; gfx950 has no shortened float32 mode that could slip in).
//
// The order of a sum is fixed by K alone: K is cut into up to eight parts of one length (a multiple of 32), a part is
// one chain of MFMAs in ascending groups of 16 k, and the parts are added in ascending order.  Both kernels keep to it,
// so a row's result is the same bits however many other rows the step holds.
//
// gemm_f32_rows_kernel, up to 16 rows, and 17 to 64 where the model below finds it faster: a block per 16 weight rows, a wave per part of K; what bounds it is the weight's
//   stream.  The weight goes straight into the MFMA operands (lane l of a wave holds four k of row l % 16: sixteen
//   pieces of 64 bytes a load), no staging and one barrier.  Every block fetches all of A's rows, so the time grows
//   by 0.2 us a row of K = 2,048.
// gemm_f32_tiles_kernel, otherwise: 2 x 2 waves of 32 or 64 x 64 elements, k-steps of 32 staged through LDS in two
//   buffers, the next step's loads in flight during the MFMAs.  A wave of 64 x 64 reads 8 KB of LDS for 64 MFMAs of
//   32 cycles, so the matrix cores bound it.
//
// The reference's own float32 product is a 128x128x16 SIMT kernel (src/kernel/cuda/mat_mul.cu:149-518).
#include "common.h"
#include "tffinfer_kernels.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf_floatx4;

// Four k of a row, zeros past K or for a row that is not there.  VEC: K, the rows' stride and the operands'
// addresses are multiples of 16 bytes; else element by element.
template <bool VEC>
__device__ __forceinline__ float4 gf_load4(const float* __restrict__ row, int k, int K, bool live) {
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (VEC) {
        if (live && k < K) x = *reinterpret_cast<const float4*>(row + k);
    } else if (live) {
        if (k + 0 < K) x.x = row[k + 0];
        if (k + 1 < K) x.y = row[k + 1];
        if (k + 2 < K) x.z = row[k + 2];
        if (k + 3 < K) x.w = row[k + 3];
    }
    return x;
}

// C += W[16 rows][16 k] A[16 rows][16 k]^T, lane (row = lane % 16, g = lane / 16) holding k = 4 g .. 4 g + 3 of its row;
// lane (m = lane % 16, g) ends up with weight rows 4 g .. 4 g + 3 of A's row m.
__device__ __forceinline__ gf_floatx4 gf_mfma16(const float4& w, const float4& a, gf_floatx4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, a.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, a.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(w.z, a.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(w.w, a.w, c, 0, 0, 0);
}

__device__ __forceinline__ void gf_store4(float* __restrict__ C, int m, int n, int M, int N, bool vec, gf_floatx4 x) {
    if (m >= M) return;
    float* p = C + (size_t)m * N + n;
    if (vec && n + 3 < N) {
        *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < N) p[i] = x[i];
}

#define GF_PARTS 8       // parts of K, at most
#define GF_AHEAD 8       // loads of 16 k a wave asks for before it multiplies

template <int MT, bool VEC>
__global__ __launch_bounds__(64 * GF_PARTS) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                      float* __restrict__ C, int M, int N, int K, int lda,
                                                                      int part_len, int store_vec) {
    __shared__ gf_floatx4 red[GF_PARTS][MT][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, parts = blockDim.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const float* wrow = W + (size_t)min(n0 + r, N - 1) * K;
    const bool wlive = n0 + r < N;
    gf_floatx4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = gf_floatx4{0.f, 0.f, 0.f, 0.f};
    const int k1 = min(K, (wv + 1) * part_len);
    for (int k = wv * part_len; k < k1; k += 16 * GF_AHEAD) {
        float4 w[GF_AHEAD];
#pragma unroll
        for (int i = 0; i < GF_AHEAD; ++i) w[i] = gf_load4<VEC>(wrow, k + 16 * i + 4 * g, k1, wlive);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int row = m * 16 + r;
            const float* arow = A + (size_t)min(row, M - 1) * lda;
            float4 a[GF_AHEAD];
#pragma unroll
            for (int i = 0; i < GF_AHEAD; ++i) a[i] = gf_load4<VEC>(arow, k + 16 * i + 4 * g, k1, row < M);
#pragma unroll
            for (int i = 0; i < GF_AHEAD; ++i) acc[m] = gf_mfma16(w[i], a[i], acc[m]);
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) red[wv][m][lane] = acc[m];
    __syncthreads();
    for (int m = wv; m < MT; m += parts) {
        gf_floatx4 t = {0.f, 0.f, 0.f, 0.f};
        for (int p = 0; p < parts; ++p) t = t + red[p][m][lane];
        gf_store4(C, m * 16 + r, n0 + 4 * g, M, N, store_vec, t);
    }
}

#define GF_BK 32

// Block: 32 MF rows of A x 32 NF weight rows, four waves of 16 MF x 16 NF.  A k-step lies in LDS as rows of 32 k, the
// 16-byte piece c of row r at place c ^ (r / 2 % 8): a wave's read of four k of sixteen rows, and a row's eight
// neighbouring writes, meet every bank once.
// AHEAD k-steps are on their way from memory in registers: the smaller a wave's part of the tile, the less of a load's
// time one step of its MFMAs covers.
template <int MF, int NF, int AHEAD, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_f32_tiles_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K, int lda, int part_len,
    int store_vec, int tiles_m, int tiles) {
    constexpr int BM = 32 * MF, BN = 32 * NF, LD = MF + NF;
    __shared__ __attribute__((aligned(16))) float lds[2][(BM + BN) * GF_BK];
    // blocks go to the eight XCDs in turn by their number: each takes a run of neighbouring tiles, row tiles fastest, so
    // that a weight tile is fetched into one L2
    const int share = (tiles + 7) / 8, id = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= share || id >= tiles) return;
    const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = lane & 15, g = lane >> 4;
    const int wm = (wv & 1) * 16 * MF, wn = (wv >> 1) * 16 * NF;
    const int lr = tid >> 3, lc = tid & 7;
    const float* src[LD];
    bool live[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const int row = lr + 32 * i;
        if (i < MF) {
            live[i] = m0 + row < M;
            src[i] = A + (size_t)min(m0 + row, M - 1) * lda;
        } else {
            live[i] = n0 + row - BM < N;
            src[i] = W + (size_t)min(n0 + row - BM, N - 1) * K;
        }
    }
    const int wplace = (lc ^ (lr >> 1 & 7)) * 4;          // (32 i rows further the swizzle is the same)
    gf_floatx4 acc[NF][MF], tot[NF][MF];
#pragma unroll
    for (int n = 0; n < NF; ++n)
#pragma unroll
        for (int m = 0; m < MF; ++m) acc[n][m] = tot[n][m] = gf_floatx4{0.f, 0.f, 0.f, 0.f};
    float4 reg[AHEAD][LD];
#pragma unroll
    for (int d = 0; d < AHEAD; ++d)
#pragma unroll
        for (int i = 0; i < LD; ++i) reg[d][i] = gf_load4<VEC>(src[i], d * GF_BK + lc * 4, K, live[i]);
    const int swz = r >> 1 & 7;
    int left = part_len;                                  // k of the present part that are still to come
    int buf = 0;
    for (int kk = 0; kk < K; kk += GF_BK * AHEAD) {
#pragma unroll
        for (int d = 0; d < AHEAD; ++d) {
            const int k0 = kk + d * GF_BK;
            if (AHEAD > 1 && k0 >= K) break;
            float* const here = lds[buf];
#pragma unroll
            for (int i = 0; i < LD; ++i) *reinterpret_cast<float4*>(here + (lr + 32 * i) * GF_BK + wplace) = reg[d][i];
            __syncthreads();      // (the other buffer was read before the barrier of the step before this one's)
#pragma unroll
            for (int i = 0; i < LD; ++i) reg[d][i] = gf_load4<VEC>(src[i], k0 + GF_BK * AHEAD + lc * 4, K, live[i]);
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                const int place = ((sub * 4 + g) ^ swz) * 4;
                float4 a[MF], w[NF];
#pragma unroll
                for (int m = 0; m < MF; ++m) a[m] = *reinterpret_cast<const float4*>(here + (wm + m * 16 + r) * GF_BK + place);
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    w[n] = *reinterpret_cast<const float4*>(here + (BM + wn + n * 16 + r) * GF_BK + place);
                // (each j walks all the accumulators, so that no MFMA waits for the one before it)
#define GF_STEP(j)                                                                                                     \
    _Pragma("unroll") for (int n = 0; n < NF; ++n) _Pragma("unroll") for (int m = 0; m < MF; ++m) acc[n][m] =          \
        __builtin_amdgcn_mfma_f32_16x16x4f32(w[n].j, a[m].j, acc[n][m], 0, 0, 0)
                GF_STEP(x);
                GF_STEP(y);
                GF_STEP(z);
                GF_STEP(w);
#undef GF_STEP
            }
            buf ^= 1;
            left -= GF_BK;
            if (left == 0 || k0 + GF_BK >= K) {
                left = part_len;
#pragma unroll
                for (int n = 0; n < NF; ++n)
#pragma unroll
                    for (int m = 0; m < MF; ++m) {
                        tot[n][m] = tot[n][m] + acc[n][m];
                        acc[n][m] = gf_floatx4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NF; ++n)
#pragma unroll
        for (int m = 0; m < MF; ++m) gf_store4(C, m0 + wm + m * 16 + r, n0 + wn + n * 16 + 4 * g, M, N, store_vec, tot[n][m]);
}

// Which kernel and tile: a launch takes as long as its busiest CU, that is, with n = ceil(blocks / 256) blocks of one tile,
// 20 + slope n us at K = 2,048 (a lone block waits for its operands, further blocks on the CU fill its waits); the slopes
// are fitted to 90 measured cases (N of 1,024 to 12,288, 65 to 1,400 rows).  us at 4,096 x 2,048 on tiles of 128 x 128 /
// 64 x 128 / 64 x 64 / 32 x 64 / 32 x 32: 128 rows 153 / 92 / 57 / 43 / 39, 301 rows 154 / 94 / 90 / 78 / 74, 602 rows
// 156 / 155 / 128 / 130 / 140, 1,400 rows 275 / 237 / 248 / 265 / 302.  The rows kernel takes 8 + N / 4,096 (6 + 0.22 M):
// up to 64 rows 26 us at N = 4,096 and 70 at 12,288, where the tiles take 53.
// Against the kernel on the vector units that stood here (64 x 64 x 16, whatever M), us before / now, K = 2,048: N = 4,096
// 2 rows 214 / 13, 64 rows 252 / 26, 602 rows 406 / 128; N = 12,288 2 rows 212 / 27, 602 rows 888 / 276; N = 151,936 2 rows
// 952 / 238 (5.2 TB/s).  The relative error against 64 bits went from 8.1e-7 to 2.9e-7.
template <bool VEC>
static int gemm_f32_for(const float* A, const float* W, float* C, int M, int N, int K, int lda, int store_vec, hipStream_t s) {
    const int part_len = 32 * ((K + 32 * GF_PARTS - 1) / (32 * GF_PARTS));
    auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    TFF_REQUIRE(tiles(32, 32) < (1L << 28), "gemm: too many tiles for M=%d N=%d", M, N);
    static const struct { int bm, bn; double slope; } sizes[5] = {{128, 128, 125}, {64, 128, 70}, {64, 64, 34.5}, {32, 64, 19.5}, {32, 32, 11}};
    int best = 0;
    double cost = 0;
    for (int i = 0; i < 5; ++i) {
        const double c = 20 + sizes[i].slope * (double)((tiles(sizes[i].bm, sizes[i].bn) + 255) / 256);
        if (i == 0 || c < cost) { best = i; cost = c; }
    }
    if (M <= 16 || (M <= 64 && 8 + N / 4096.0 * (6 + 0.22 * M) <= cost)) {
        const int waves = (K + part_len - 1) / part_len, mt = (M + 15) / 16, blocks = (N + 15) / 16;
#define GF_ROWS(MT) gemm_f32_rows_kernel<MT, VEC><<<blocks, 64 * waves, 0, s>>>(A, W, C, M, N, K, lda, part_len, store_vec)
        if (mt == 1) GF_ROWS(1);
        else if (mt == 2) GF_ROWS(2);
        else if (mt == 3) GF_ROWS(3);
        else GF_ROWS(4);
#undef GF_ROWS
        return tff_check_launch("gemm_f32_rows");
    }
#define GF_TILES(MF, NF, AH)                                                                                          \
    do {                                                                                                              \
        const int tm = (M + 32 * MF - 1) / (32 * MF), t = (int)tiles(32 * MF, 32 * NF);                               \
        gemm_f32_tiles_kernel<MF, NF, AH, VEC>                                                                        \
            <<<(t + 7) / 8 * 8, 256, 0, s>>>(A, W, C, M, N, K, lda, part_len, store_vec, tm, t);                      \
    } while (0)
    switch (best) {
        case 0: GF_TILES(4, 4, 1); break;
        case 1: GF_TILES(2, 4, 2); break;
        case 2: GF_TILES(2, 2, 3); break;
        case 3: GF_TILES(1, 2, 4); break;
        default: GF_TILES(1, 1, 4); break;
    }
#undef GF_TILES
    return tff_check_launch("gemm_f32_tiles");
}

int tff_gemm_f32(const float* A, const float* W, void* C, int M, int N, int K, int lda,
                 int c_dtype, hipStream_t s) {
    if (c_dtype != TFF_F32) return tff_fail("gemm: a float32 product writes float32, not type %d", c_dtype);
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0;
    const int store_vec = N % 4 == 0 && ((uintptr_t)C % 16) == 0;
    return vec ? gemm_f32_for<true>(A, W, (float*)C, M, N, K, lda, store_vec, s)
               : gemm_f32_for<false>(A, W, (float*)C, M, N, K, lda, store_vec, s);
}
