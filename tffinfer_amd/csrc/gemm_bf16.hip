// bfloat16 matrix product C = A . W^T on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_bf16), float32 accumulation.  Replaces the reference's
// SIMT products (src/kernel/cuda/quant/quant_q_8_0_mat_mul.cu:338-447,
// src/kernel/cuda/mat_mul.cu:149-518) with a design for 64-wide waves.
//
// Weights are kept in *fragment order*: W [N, K] is cut into tiles of 16 rows
// by 32 k, and each tile is stored as the 1 KB an MFMA operand is, lane after
// lane: element (n, k) lies at
//     ((n / 16) * (Kp / 32) + k / 32) * 512 + (((k % 32) / 8) * 16 + n % 16) * 8 + k % 8
// with N and K padded to multiples of 16 and 32 by zeros.  A wave fetches an
// operand with one fully contiguous 1 KB load (measured: a quarter more of
// the HBM bandwidth than 16 rows x 64 bytes of a row-major matrix), and a tile
// staged in LDS in the same order is read back without bank conflicts.
// Activations A [M, K] stay row-major.  The W tile is the MFMA's first operand,
// so a lane ends up with 4 consecutive output columns of one row.
#include "gemm_bf16.h"
#include "tffinfer_kernels.h"

// ------------------------------------------------------- tiled, async copy ---
// Block tile (WGM*WTM*16) x (WGN*WTN*16) x (32 KPS) on WGM x WGN waves, each wave
// WTM x WTN MFMA tiles.  Both operands are staged in LDS in fragment order; the
// padding of W to 32 k holds zeros, so k past the end of A only has to be
// readable: what it multiplies is zero.  The copies global -> LDS are done by
// the load unit itself (global_load_lds_dwordx4: every lane's 16 bytes land at
// LDS base + lane * 16, which is exactly fragment order), so no register and no
// LDS store instruction is spent on staging, and STAGES - 1 tiles are in flight
// while one is worked on.
// A wave waits for its own copies of the tile it is about to read
// (s_waitcnt vmcnt), the barrier that follows makes the other waves' visible.
typedef const __attribute__((address_space(1))) void* glb_ptr_t;
template <int WGM, int WGN, int WTM, int WTN, int STAGES, bool GLU, typename TC, int KPS = 2, bool EARLY = false>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_bf16_async_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wp, TC* __restrict__ C, int M, int N,
    int K, int lda, int KB, int n_out, float* __restrict__ part, const GemmEpilogue ex) {
    const float* __restrict__ const bias = ex.bias;
    // WGM x WGN waves, each WTM x WTN MFMA tiles of 16 x 16
    constexpr int NW = WGM * WGN;
    constexpr int BM = WGM * WTM * 16, BN = WGN * WTN * 16;
    constexpr int AF = BM / 16 * KPS, WF = BN / 16 * KPS;   // fragments per operand tile (KPS k-steps of 32)
    constexpr int FR = AF + WF;                          // fragments per stage, 1 KB each
    // copies a wave issues per tile: fragment wave + NW j is copy j of a wave; where the fragments
    // do not go round evenly the last waves copy the last fragment once more (same bytes to the
    // same place), so that every wave has the same number of copies in flight
    constexpr int LPW = (FR + NW - 1) / NW;
    static_assert((STAGES - 2) * LPW < 64, "vmcnt has 6 bits");
    __shared__ __attribute__((aligned(1024))) bf16_t smem[STAGES * FR * 512];
    const int tid = threadIdx.x;
    // (the wave's index as a scalar: what follows from it, the fragments it copies and where they
    // land in LDS, is then worked out by the scalar unit)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int fr = lane & 15, fg = lane >> 4;
    // Blocks are handed to the eight XCDs in turn, and each XCD has an L2 of its own: block b
    // of the launch runs on XCD b % 8.  Row tiles are taken in groups of eight; within a group
    // the tiles are numbered column tile by column tile, and XCD x works through the x-th
    // eighth of that sequence one after the other: with 32 blocks of an XCD in flight these are
    // four column tiles by eight row tiles, a tile of W is fetched into one L2 only (two at the
    // seam of two eighths) and the (smaller) A is what every L2 holds.  A full group gives
    // every XCD exactly TN tiles whatever TN is; only the last, smaller group pads the launch.
    const int TM = (M + BM - 1) / BM, TN = (N + BN - 1) / BN;
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
    const int full = (TM >> 3) * TN;           // blocks an XCD runs for the full groups
    int grp, grp_rows, j;
    if (seq < full) {
        grp = seq / TN;
        grp_rows = 8;
        j = xcd * TN + (seq - grp * TN);
    } else {
        grp = TM >> 3;
        grp_rows = TM & 7;
        const int per = (grp_rows * TN + 7) >> 3;
        j = xcd * per + (seq - full);
        if (seq - full >= per || j >= grp_rows * TN) return;   // the launch is padded to eight equal shares
    }
    const int tn = j / grp_rows, tm = grp * 8 + j % grp_rows;
    const int m0 = tm * BM, n0 = tn * BN;
    const int NB = (N + 15) / 16;
    const int nk = (K + 32 * KPS - 1) / (32 * KPS);
    // With gridDim.z > 1 the blocks of one tile split K among them and leave partial sums in
    // part[z][M][N], which a second kernel adds up in a fixed order.
    const int kt_per = (nk + (int)gridDim.z - 1) / (int)gridDim.z;
    const int kt0 = (int)blockIdx.z * kt_per;
    const int kt1 = min(nk, kt0 + kt_per);

    floatx4 acc[WTN][WTM];
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
        for (int j = 0; j < WTM; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (bias && blockIdx.z == 0) {
#pragma unroll
        for (int i = 0; i < WTN; ++i) {
            const floatx4 b = bias4(bias, n0 + (wn * WTN + i) * 16 + fg * 4, NB);
#pragma unroll
            for (int j = 0; j < WTM; ++j) acc[i][j] = b;
        }
    }

    // this wave's copies: fragments f = wave + NW j of a stage; f < AF is of A, else of W
    const bf16_t* src[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int f = min(wave + NW * j, FR - 1);
        if (f < AF) {
            const int row = min(m0 + (f / KPS) * 16 + fr, M - 1);   // rows past the end repeat the last
            src[j] = A + (size_t)row * lda;
        } else {
            const int nb = min(n0 / 16 + (f - AF) / KPS, NB - 1);
            src[j] = Wp + (size_t)nb * KB * 512 + lane * 8;
        }
    }
    // Tiles past the end are copied too (as the last tile, into stages nobody reads any more):
    // then the number of copies in flight is the same in every iteration and one constant wait
    // covers them all.
#define TFF_ISSUE_TILE(tile)                                                                       \
    {                                                                                              \
        const int kt_ = min((tile), nk - 1);                                                       \
        const int st_ = ((tile) - kt0) % STAGES;                                                   \
        _Pragma("unroll") for (int j = 0; j < LPW; ++j) {                                          \
            const int f = min(wave + NW * j, FR - 1);                                               \
            const bf16_t* g_;                                                                      \
            if (f < AF) g_ = src[j] + min((kt_ * KPS + f % KPS) * 32 + fg * 8, K - 8);                 \
            else g_ = src[j] + (size_t)min(KPS * kt_ + (f - AF) % KPS, KB - 1) * 512;                  \
            copy16_to_lds(g_, smem + (st_ * FR + f) * 512);                                        \
        }                                                                                          \
    }

#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t) TFF_ISSUE_TILE(kt0 + t)
    if constexpr (EARLY) {
        // The barrier stands between a tile's LDS reads and its MFMAs: a wave arrives with its
        // operands on the way, and when the barrier opens every wave can start its MFMAs at once
        // (with the barrier before the reads, all waves read at the same time and the matrix
        // cores wait for the first operands after every barrier).  The barrier of tile kt makes
        // tile kt + 1 visible, so the copies have to be one tile further ahead.
        static_assert(KPS == 1 && STAGES >= 3, "one k-step a tile, three stages or more");
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * LPW));
        __syncthreads();
        for (int kt = kt0; kt < kt1; ++kt) {
            const bf16_t* st = smem + ((kt - kt0) % STAGES) * FR * 512;
            bf16x8 fw[WTN], fa[WTM];
#pragma unroll
            for (int i = 0; i < WTN; ++i)
                fw[i] = *reinterpret_cast<const bf16x8*>(st + (AF + wn * WTN + i) * 512 + lane * 8);
#pragma unroll
            for (int j = 0; j < WTM; ++j)
                fa[j] = *reinterpret_cast<const bf16x8*>(st + (wm * WTM + j) * 512 + lane * 8);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 3) * LPW));   // this wave's part of tile kt + 1 is in
            asm volatile("s_barrier" ::: "memory");
            TFF_ISSUE_TILE(kt + STAGES - 1)                              // into the stage of tile kt - 1
            if (kt < KB) {
#pragma unroll
                for (int i = 0; i < WTN; ++i)
#pragma unroll
                    for (int j = 0; j < WTM; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i], fa[j], acc[i][j], 0, 0, 0);
            }
        }
    } else
    for (int kt = kt0; kt < kt1; ++kt) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((STAGES - 2) * LPW));   // this wave's part of tile kt is in
        __syncthreads();                                             // ... and everybody else's
        TFF_ISSUE_TILE(kt + STAGES - 1)                              // into the stage read last iteration
        const bf16_t* st = smem + ((kt - kt0) % STAGES) * FR * 512;
#pragma unroll
        for (int ks = 0; ks < KPS; ++ks) {
            if (KPS * kt + ks < KB) {   // k-steps past the end of K are not in W
                bf16x8 fw[WTN], fa[WTM];
#pragma unroll
                for (int i = 0; i < WTN; ++i)
                    fw[i] = *reinterpret_cast<const bf16x8*>(st + (AF + (wn * WTN + i) * KPS + ks) * 512 + lane * 8);
#pragma unroll
                for (int j = 0; j < WTM; ++j)
                    fa[j] = *reinterpret_cast<const bf16x8*>(st + ((wm * WTM + j) * KPS + ks) * 512 + lane * 8);
#pragma unroll
                for (int i = 0; i < WTN; ++i)
#pragma unroll
                    for (int j = 0; j < WTM; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i], fa[j], acc[i][j], 0, 0, 0);
            }
        }
    }
#undef TFF_ISSUE_TILE
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));   // the copies past the end must not outlive the block

    if (part) {   // partial sums over this block's share of K, columns as W has them
        float* P = part + (size_t)blockIdx.z * M * N;
        const bool vec = (N % 4) == 0;
#pragma unroll
        for (int i = 0; i < WTN; ++i) {
            const int n = n0 + (wn * WTN + i) * 16 + fg * 4;
#pragma unroll
            for (int j = 0; j < WTM; ++j) {
                const int m = m0 + (wm * WTM + j) * 16 + fr;
                if (m < M && n < N) store4<float>(P + (size_t)m * N + n, acc[i][j], n, N, vec);
            }
        }
        return;
    }
    if constexpr (GLU) {
        static_assert(WTN % 2 == 0, "gate and up groups come in pairs");
        const bool vec = (n_out % 4) == 0;
#pragma unroll
        for (int i = 0; i < WTN; i += 2) {
            const int n = (n0 + (wn * WTN + i) * 16) / 2 + fg * 4;
#pragma unroll
            for (int j = 0; j < WTM; ++j) {
                const int m = m0 + (wm * WTM + j) * 16 + fr;
                if (m < M && n < n_out)
                    store4<TC>(C + (size_t)m * n_out + n, glu4(acc[i][j], acc[i + 1][j], ex.act), n, n_out, vec);
            }
        }
    } else {
        const bool vec = (N % 4) == 0;
#pragma unroll
        for (int i = 0; i < WTN; ++i) {
            const int n = n0 + (wn * WTN + i) * 16 + fg * 4;
#pragma unroll
            for (int j = 0; j < WTM; ++j) {
                const int m = m0 + (wm * WTM + j) * 16 + fr;
                if (m < M && n < N) store4<TC>(C + (size_t)m * N + n, acc[i][j], n, N, vec);
            }
        }
    }
}

// Adds up the partial sums part[s][M][N] of a product whose blocks split K, s = 0, 1, ... in
// turn, and writes C; with GLU, columns come as gate and up groups of 16 in turn and
// C[m][j] = silu(gate) * up.  One thread makes four neighbouring outputs.
template <bool GLU, typename TC, bool UNARY>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, int S,
                                                                  int M, int N, TC* __restrict__ C,
                                                                  int n_out, GluAct act, int unary) {
    const int per_row = (n_out + 3) / 4;
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)M * per_row) return;
    const int m = (int)(idx / per_row), j = (int)(idx % per_row) * 4;
    const size_t plane = (size_t)M * N;
    floatx4 a = floatx4{0.f, 0.f, 0.f, 0.f}, b = a;
    if constexpr (GLU) {
        const int c = (j >> 4) * 32 + (j & 15);   // N is a multiple of 32 here: whole float4s
        const float* p = part + (size_t)m * N + c;
        for (int s = 0; s < S; ++s, p += plane) {
            const float4 g = *reinterpret_cast<const float4*>(p);
            const float4 u = *reinterpret_cast<const float4*>(p + 16);
            a[0] += g.x; a[1] += g.y; a[2] += g.z; a[3] += g.w;
            b[0] += u.x; b[1] += u.y; b[2] += u.z; b[3] += u.w;
        }
        a = glu4(a, b, act);
    } else {
        const float* p = part + (size_t)m * N + j;
        const bool vec = (N % 4) == 0;
        for (int s = 0; s < S; ++s, p += plane) {
            if (vec) {
                const float4 v = *reinterpret_cast<const float4*>(p);
                a[0] += v.x; a[1] += v.y; a[2] += v.z; a[3] += v.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (j + e < N) a[e] += p[e];
            }
        }
        if constexpr (UNARY) {
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = unary_activation(a[e], unary);
        }
    }
    store4<TC>(C + (size_t)m * n_out + j, a, j, n_out, (n_out % 4) == 0);
}

template <bool GLU>
static int launch_reduce(const float* part, int S, int M, int N, void* C, int n_out, const GemmExtra& ex, int c_dtype, hipStream_t s) {
    const int blocks = (int)(((long)M * ((n_out + 3) / 4) + 255) / 256);
#define TFF_REDUCE(TC, UNARY) gemm_splitk_reduce_kernel<GLU, TC, UNARY><<<blocks, 256, 0, s>>>(part, S, M, N, (TC*)C, n_out, ex.act, ex.unary)
    if constexpr (!GLU) {
        if (ex.unary) {
            if (c_dtype == TFF_F32) TFF_REDUCE(float, true);
            else TFF_REDUCE(bf16_t, true);
            return tff_check_launch("gemm_splitk_reduce");
        }
    }
    if (c_dtype == TFF_F32) TFF_REDUCE(float, false);
    else TFF_REDUCE(bf16_t, false);
#undef TFF_REDUCE
    return tff_check_launch("gemm_splitk_reduce");
}

// splits > 1: the blocks of a tile split K among them; part holds splits * M * N floats
template <int WGM, int WGN, int WTM, int WTN, int STAGES, bool GLU = false, int KPS = 2, bool EARLY = false>
static int launch_async_g(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda,
                          const GemmCall ex, int c_dtype, int n_out, hipStream_t s, int splits = 1, float* part = nullptr,
                          bool reduce = true) {
    const int KB = (K + 31) / 32;
    constexpr int BM = WGM * WTM * 16, BN = WGN * WTN * 16;
    if (splits <= 1 || !part) { splits = 1; part = nullptr; }
    const long TM = (M + BM - 1) / BM, TN = (N + BN - 1) / BN;
    const long tiles = 8 * ((TM / 8) * TN + ((TM % 8) * TN + 7) / 8);   // eight equal shares, see the kernel
    TFF_REQUIRE(tiles < (1L << 31), "gemm: too many tiles for M=%d N=%d", M, N);
    const dim3 grid((unsigned)tiles, 1, splits);
    if (c_dtype == TFF_F32)
        gemm_bf16_async_kernel<WGM, WGN, WTM, WTN, STAGES, GLU, float, KPS, EARLY>
            <<<grid, 64 * WGM * WGN, 0, s>>>(A, Wp, (float*)C, M, N, K, lda, KB, n_out, part, ex);
    else
        gemm_bf16_async_kernel<WGM, WGN, WTM, WTN, STAGES, GLU, bf16_t, KPS, EARLY>
            <<<grid, 64 * WGM * WGN, 0, s>>>(A, Wp, (bf16_t*)C, M, N, K, lda, KB, n_out, part, ex);
    if (int rc = tff_check_launch("gemm_bf16_async")) return rc;
    if (splits > 1 && reduce) {
        return launch_reduce<GLU>(part, splits, M, N, C, GLU ? n_out : N, ex, c_dtype, s);
    }
    return 0;
}

// ------------------------------------------- four waves, whole cache lines ---
// Block tile 256 or 192 x (32 WTN) on 2 x 2 waves (or 128 or 96 x (64 WTN) on 1 x 4, for products of few rows,
// whose time is the weight's stream: all four waves then read the same rows of A), one wave to a
// SIMD, each wave 8 or 6 x WTN MFMA tiles: half the LDS reads per MFMA of sixteen waves of 64 x 64.  With one wave to a SIMD nothing overlaps unless
// the wave interleaves it itself: the fragments of k-tile t + 1 are read from LDS into a second set
// of registers, and the copies of later tiles are issued, between the MFMAs of k-tile t.
//
// What bounds this product is the number of requests to L2, not their bytes: a row-major A read 32 k
// at a time is 64 bytes a row, half a cache line a request.  So A is copied 64 k at a time, eight
// rows x 128 bytes a copy (a unit of two k-tiles, NA = 3 of them in LDS), W 32 k at a time as it is
// packed (NWS k-tiles in LDS).  Within a copy's 1 KB lane i lands at byte 16 i; it fetches row
// i / 8, 16-byte chunk (i % 8) ^ (i / 8), so that the sixteen rows an MFMA operand is made of are
// read back from different banks.
// In k-tile t (32 k) a wave copies half of A unit u + 3 (t = 2 u + 1 the first, t = 2 u + 2 the second half) and W tile
// t + NWS: into the slots of the unit and tile whose fragments were last read in tile t - 1 or before.  Every wave waits
// for its own reads before the barrier at the start of t, which makes those slots free; the last quarter of a tile's
// MFMAs has no reads (of tiles of eight MFMAs and more), so that wait seldom lasts.  At the start of t it needs W tile t + 1 and the A unit of
// t + 1, issued in tiles t - NWS + 1 and t - 3 at the latest.  Copies complete in the order issued, so the wait is by count.
//
// What bounds the loop of one wave a SIMD is the issue of what stands between the MFMAs: a wave issues an instruction
// every four cycles and an MFMA takes sixteen, so three others fit behind each and the fourth leaves the matrix core
// idle.  With a 64-bit address a copy that each walks k, its LDS address and the ring's bookkeeping a tile took 1,340
// cycles (no copies at all: 1,093, whatever the clock; a tile of the same reads and MFMAs whose copies do not walk: 1,180).
// So all copies of an operand share one address, the lane's part of it in a register that never changes; a copy is an
// s_add into M0 before an MFMA and the load after it; and what moves the rings and addresses on is dealt over the gaps
// behind a tile's last copies: 1,110 cycles.  The clock falls with the idle cycles (1.80 -> 1.72 GHz: the power limit), so
// the time falls by less: us before / now, 2,048 rows of the 8B shape: QKV 77.0 / 72.9, O 57.8 / 53.0, gate+up 299 / 284,
// down 159 / 145; 16,384 rows, gate+up 2,343 / 2,221; 600 rows of 2,048: O 16.0 / 15.2, gate+up 32.5 / 29.3.
// Before its first tile a block sets its accumulators while the first copies are on their way (set twice before and behind
// them, 512 instructions, a product of 600 rows of 6,144 took 27.9 us, now 26.7; 16,384 rows, gate+up 2,221 / 2,213).
// K a multiple of 64; a split of K takes whole units.
// A wave's 128 rows x OW column groups of results go out through LDS, so that a store instruction
// writes whole rows instead of 16 rows x 8 or 16 bytes: a lane leaves its four columns of a row in
// the wave's own region of LDS (rows padded by 16 bytes against bank conflicts) and takes 16 bytes
// of a row back.  Only this wave touches the region, LDS works through a wave's accesses in order,
// so no barrier is needed within; RC of the 8 row groups go through at a time, as many as the
// region holds.  A store instruction takes 64 / LPR rows, LPR lanes to a row (the power of two that
// holds a row's 16-byte pieces; the lanes beyond them idle), so that the address of a lane's store
// is that of its last one plus a constant.  vec: the rows of the result are a multiple of 16 bytes
// long, the 16 bytes are one store; otherwise they go out element by element (slow, and rare: a
// width that is no multiple of 8).  This is the kernel's only way out for its results on purpose:
// with a second one beside it the compiler converts accumulators for both before the branch, runs
// out of registers and spills, and a kernel that uses scratch memory pays some 15 us at its launch.
template <int OW, int REGION, typename TO, int WTM = 8, typename F>
__device__ __forceinline__ void w4_store_rows(char* region, F val, TO* out, size_t ld, int m_base, int n_base,
                                              int M, int ncols, int lane, bool vec) {
    constexpr int E = 16 / (int)sizeof(TO);           // columns in 16 bytes
    constexpr int RB = OW * 16 * (int)sizeof(TO), RBP = RB + 16, CPR = RB / 16;
    constexpr int LPR = CPR <= 4 ? 4 : CPR <= 8 ? 8 : CPR <= 16 ? 16 : 32;   // lanes a row
    static_assert(CPR <= LPR, "a row's pieces fit its lanes");
    constexpr int RPI = 64 / LPR;                     // rows a store instruction
    constexpr int RC = WTM * 16 * RBP <= REGION ? WTM : WTM / 2;   // row groups that go through the region at a time
    static_assert(RC >= 1 && RC * 16 * RBP <= REGION, "the wave's region of LDS holds half its row groups at least");
    const int fr = lane & 15, fg = lane >> 4;
    const int srow = lane / LPR, sch = lane % LPR;    // this lane's row of an instruction's, and its piece
    const int n = n_base + sch * E;
    const bool mine = sch < CPR && n < ncols;
    const char* src = region + srow * RBP + sch * 16;
#pragma unroll
    for (int p = 0; p < WTM / RC; ++p) {
#pragma unroll
        for (int jj = 0; jj < RC; ++jj) {
            __builtin_amdgcn_sched_barrier(0);   // a row group at a time: all accumulators converted at once do not fit the registers
#pragma unroll
            for (int i = 0; i < OW; ++i) {
                const floatx4 v = val(i, p * RC + jj);
                char* dst = region + (jj * 16 + fr) * RBP + (i * 16 + fg * 4) * (int)sizeof(TO);
                if constexpr (sizeof(TO) == 4) {
                    *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
                    union { bf16_t h[4]; uint2 u; } pk;
#pragma unroll
                    for (int e = 0; e < 4; ++e) pk.h[e] = (bf16_t)v[e];
                    *reinterpret_cast<uint2*>(dst) = pk.u;
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        int m = m_base + p * RC * 16 + srow;
        TO* dst = out + (size_t)m * ld + n;
        if (vec) {   // (the branch outside the loop: its reads of LDS are then issued together, not one per store)
#pragma unroll
            for (int t = 0; t < RC * 16 / RPI; ++t) {
                const uint4 v = *reinterpret_cast<const uint4*>(src + t * RPI * RBP);
                if (mine && m < M) *reinterpret_cast<uint4*>(dst) = v;
                m += RPI;
                dst += (size_t)RPI * ld;
            }
        } else {
            for (int t = 0; t < RC * 16 / RPI; ++t) {
                union { uint4 u; TO e[E]; } v;
                v.u = *reinterpret_cast<const uint4*>(src + t * RPI * RBP);
                if (mine && m < M) {
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        if (n + e < ncols) dst[e] = v.e[e];
                }
                m += RPI;
                dst += (size_t)RPI * ld;
            }
        }
    }
}

// Which tile a block works on.  Blocks go to the eight XCDs in turn by their number, and an XCD's 32 CUs share an L2 that holds a
// stretch of k of the tile rows and columns they work on at a time: so those should be few, and every XCD should get as many
// tiles.  The tile rows are cut into bands of w4_band of them (up to 1,024 rows of A), a band's tiles numbered column after column; as many bands as
// hold 256 tiles at least go together, and an XCD takes an eighth of their tiles, one after the other: 4 x 8 tiles of 256 rows at a time.
// (Eight tile rows of every column to an XCD, whatever their number, were 32 x 1 tiles of a result 1,024 wide: every XCD
// read all of A.  us before / now: 7,376 rows of 1,024 x 3,072 on tiles of 256 x 128 55 / 40,
// 4,700 of 2,048 x 2,048 37.4 / 35.9, 16,384 of 4,096 x 12,288 1,070 / 1,041, of 24,576 x 4,096 2,198 / 2,177.)
template <int BM>
constexpr int w4_band() { return BM >= 192 ? 4 : 8; }
template <int BM>
__host__ __device__ inline int w4_rows_together(int TN) {
    const int band = w4_band<BM>() * TN;
    return w4_band<BM>() * ((256 + band - 1) / band);
}
template <int BM>
__host__ __device__ inline long w4_blocks(long TM, long TN) {
    const long rows = w4_rows_together<BM>((int)TN), full = TM / rows, rest = TM - full * rows;
    return 8 * (full * ((rows * TN + 7) / 8) + (rest * TN + 7) / 8);
}
template <int BM>
__device__ __forceinline__ bool w4_place(unsigned block, int TM, int TN, int& tm, int& tn) {
    constexpr int BAND = w4_band<BM>();
    const int xcd = block & 7, seq = block >> 3;
    if (TM <= BAND) {      // (one band: the same with one division, which few rows' products notice)
        const int mine = (TM * TN + 7) >> 3, j = xcd * mine + seq;
        if (seq >= mine || j >= TM * TN) return false;
        tn = j / TM;
        tm = j - tn * TM;
        return true;
    }
    const int together = w4_rows_together<BM>(TN), share = (together * TN + 7) >> 3;
    const int at = min(seq / share, TM / together);
    const int first = at * together, rows = min(together, TM - first);
    const int mine = (rows * TN + 7) >> 3, i = seq - at * share, j = xcd * mine + i;
    if (i >= mine || j >= rows * TN) return false;
    const int band = j / (BAND * TN), in = j - band * BAND * TN, high = min(BAND, rows - band * BAND);
    tn = in / high;
    tm = first + band * BAND + (in - tn * high);
    return true;
}

// SCALE: A's rows (up to 16 of them) still lack the factor of the RMS norm they went through; the
// factor, rsqrt(sum of the row's sums of squares / dim + eps), is applied to the accumulators.
struct W4Scale {
    const float* ss;        // [16][stride] sums of squares, count of them a row
    int stride, count;
    float inv_dim, eps;
};
// PLANES: several products in one launch (GemmExtra).  A kernel of its own: a test of plane_cols in every product cost those of a short
// prompt up to 1.5 % (gate+up of 560 rows 34.5 / 35.0 us).
// ONCE: the block reads its columns of W alone, and no later call finds them in a cache (see launch_w4).
template <int WTN, int NWS, bool GLU, typename TC, int WGM = 2, bool SCALE = false, int WTM = 8, bool PLANES = false, bool ONCE = false>
__global__ __launch_bounds__(256) void gemm_bf16_w4_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wp, TC* __restrict__ C, int M, int N,
    int K, int lda, int KB, int n_out, W4Scale sc,
    const typename std::conditional<PLANES, GemmExtra, GemmEpilogue>::type ex) {
    const float* __restrict__ const bias = ex.bias;
    static_assert(!SCALE || WGM == 1, "rows that lack their norm's factor: up to 16, one row tile");
    // WGM: waves along the rows, 2 (a block tile of 256 rows, two waves side by side) or 1 (128 rows, four side by side)
    // WTM: row groups of 16 a wave, 8 or 6 (a block tile of 192 or 96 rows), or with the waves side by side 4 or 2 (of 64 or 32 rows)
    constexpr int NW = 4, NA = 3, WGN = NW / WGM;
    static_assert(WGM == 1 || WGM == 2, "four waves as 2 x 2 or 1 x 4");
    static_assert(WTM == 8 || WTM == 6 || (WGM == 1 && (WTM == 4 || WTM == 2)), "few rows a wave only with the waves side by side");
    constexpr int BM = WGM * WTM * 16, BN = WGN * WTN * 16;
    constexpr int WF = BN / 16;                       // W fragments a k-tile, 1 KB each
    static_assert(WF % NW == 0, "every wave copies as many fragments of W");
    constexpr int ACP = BM / 8;                       // A copies a unit, 1 KB each
    constexpr int LPA = ACP / NW, LPW = WF / NW;
    constexpr int NMF = WTM * WTN;                    // MFMAs a k-tile
    constexpr int RPM = NMF * 3 / 4 / (WTM + WTN) > 0 ? NMF * 3 / 4 / (WTM + WTN) : 1;   // a read after every RPM MFMAs
    constexpr int LPA_O = (LPA + 1) / 2, LPA_E = LPA / 2;   // copies of A in an odd and an even k-tile
    constexpr int CPM = (NMF - 4) / (LPA_O + LPW) > 0 ? (NMF - 4) / (LPA_O + LPW) : 1;   // a copy with every CPM-th MFMA
    static_assert(NWS == 4 || NWS == 5, "the waits below are written for four or five tiles ahead");
    static_assert(RPM * (WTM + WTN) <= NMF, "a tile's MFMAs hold the reads of the next");
    constexpr int UP0 = NMF >= 8 ? NMF - 4 : NMF - 1, UP1 = NMF >= 8 ? NMF - 3 : NMF - 1;   // the gaps that move rings and addresses on
    constexpr int UP2 = NMF >= 8 ? NMF - 2 : NMF - 1, UP3 = NMF - 1;
    static_assert(RPM >= 1 && CPM * (LPA_O + LPW) <= UP1, "not enough MFMAs to hide the reads and copies");
    constexpr unsigned A_UNIT = ACP * 1024u, W_TILE = WF * 1024u, W_BASE = NA * A_UNIT;
    static_assert(W_BASE + NWS * W_TILE <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) char smem[W_BASE + NWS * W_TILE];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = WGM == 2 ? wave >> 1 : 0, wn = WGM == 2 ? wave & 1 : wave;
    const int fr = lane & 15, fg = lane >> 4;
    const int TM = (M + BM - 1) / BM, TN = (N + BN - 1) / BN;
    int tm, tn;
    if (!w4_place<BM>(blockIdx.x, TM, TN, tm, tn)) return;
    const int m0 = tm * BM, n0 = tn * BN;
    const int NB = (N + 15) / 16;
    if constexpr (PLANES) {   // (a tile's columns are one plane's; C as its column 0 of row 0 would lie)
        const size_t plane = (size_t)(n0 / ex.plane_cols);
        A += plane * ex.a_step;
        C += plane * (size_t)(M - 1) * ex.plane_cols;
    }
    const int nu = KB / 2;                            // units of 64 k
    const int u_per = (nu + (int)gridDim.z - 1) / (int)gridDim.z;
    const int u0 = (int)blockIdx.z * u_per;
    const int u1 = min(nu, u0 + u_per);
    const int kt0 = 2 * u0, kt1 = 2 * u1;

    floatx4 start[WTN];      // what the accumulators start from
#pragma unroll
    for (int i = 0; i < WTN; ++i) start[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (bias && blockIdx.z == 0) {
#pragma unroll
        for (int i = 0; i < WTN; ++i) start[i] = bias4(bias, n0 + (wn * WTN + i) * 16 + fg * 4, NB);
#pragma unroll
        for (int i = 0; i < WTN; ++i) asm volatile("" : "+v"(start[i]));      // (here, before the copies, which the compiler does not see)
    }
    // (a lane's results are four columns of row fr of each row group: of row fr itself in the first,
    // the only one that counts with up to 16 rows; the four lanes of a row share out its sums)
    float row_ss = 0.f;
    if constexpr (SCALE) {
        // (16 bytes a load, eight loads asked for before the first is added: one trip to memory for rows of up to 8,192 elements)
        const float* sp = sc.ss + (size_t)fr * sc.stride;
        const int vec_end = sc.count & ~3;
        for (int j0 = fg * 4; j0 < vec_end; j0 += 16 * 8) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = j0 + 16 * u < vec_end ? *reinterpret_cast<const float4*>(sp + j0 + 16 * u) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int u = 0; u < 8; ++u) row_ss += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        }
        if (fg == 0)
            for (int j = vec_end; j < sc.count; ++j) row_ss += sp[j];
    }

    // this wave's copies: of an A unit the copies wave + 4 c, of a W tile the fragments wave + 4 c; a lane's bytes from the operand's address on
    const unsigned long long a0 = (unsigned long long)(A + (size_t)m0 * lda + (size_t)kt0 * 32);
    const unsigned long long w0 = (unsigned long long)(Wp + ((size_t)(n0 / 16) * KB + kt0) * 512);
    unsigned aoff[LPA], woff[LPW];
#pragma unroll
    for (int c = 0; c < LPA; ++c)
        aoff[c] = (unsigned)(min(m0 + (wave + NW * c) * 8 + (lane >> 3), M - 1) - m0) * (unsigned)lda * 2u + (unsigned)(((lane & 7) ^ (lane >> 3)) * 16);
#pragma unroll
    for (int c = 0; c < LPW; ++c)
        woff[c] = (unsigned)(min(n0 / 16 + wave + NW * c, NB - 1) - n0 / 16) * (unsigned)KB * 1024u + (unsigned)lane * 16u;
    const unsigned lds_wave = (unsigned)(size_t)(lds_ptr_t)smem + (unsigned)wave * 1024u;
    floatx4 acc[WTN][WTM];
    auto start_acc = [&]() {
#pragma unroll
        for (int i = 0; i < WTN; ++i)
#pragma unroll
            for (int jj = 0; jj < WTM; ++jj) {
                acc[i][jj] = start[i];
                asm volatile("" : "+a"(acc[i][jj]));
            }
    };
    if (u0 < u1) {   // (a part of a split K that holds no unit only stores its zeros)
        // copies past the end repeat the last unit or tile, so that the counts in flight stay the same
        const unsigned a_end = (unsigned)(u1 - u0 - 1) * 128u, w_end = (unsigned)(kt1 - kt0 - 1) * 1024u;
        // the tiles before the first, in the order of the loop: t = -5 .. -1
#pragma unroll
        for (int t = -5; t < 0; ++t) {
            const int u = (t + 5) / 2;                    // unit 0 in tiles -5 and -4, 1 in -3 and -2, the first half of 2 in -1
#pragma unroll
            for (int c = (t & 1) ? 0 : LPA_O; c < ((t & 1) ? LPA_O : LPA); ++c)
                copy16_to_lds_sbase(a0 + min((unsigned)u * 128u, a_end), aoff[c], lds_wave + (unsigned)u * A_UNIT + (unsigned)c * 4096u);
            if (t + NWS >= 0) {
#pragma unroll
                for (int c = 0; c < LPW; ++c)
                    copy16_to_lds_sbase<ONCE>(w0 + min((unsigned)(t + NWS) * 1024u, w_end), woff[c],
                                        lds_wave + W_BASE + (unsigned)(t + NWS) * W_TILE + (unsigned)c * 4096u);
            }
        }
        unsigned a_ko = min(2u * 128u, a_end), w_ko = min((unsigned)NWS * 1024u, w_end);   // the unit and tile copied next, in bytes of k
        unsigned long long a_at = a0 + a_ko, w_at = w0 + w_ko;
        unsigned a_to = lds_wave + 2u * A_UNIT, w_to = lds_wave;   // where they go
        // what may still be in flight at the start of tile t: the copies of the last two tiles, of three where W is that far ahead
        constexpr int ODD = LPA_O + LPW, EVEN = LPA_E + LPW;
        constexpr int FLY_E = NWS == 5 ? 2 * ODD + EVEN : ODD + EVEN;   // t even: t - 1 is odd
        constexpr int FLY_O = ODD + EVEN;
        // a lane's 16 bytes of an A operand: row fr of 16, chunk h * 4 + fg of the row's 8
        unsigned a_rd[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            a_rd[h] = (unsigned)(wm * WTM * 2 + (fr >> 3)) * 1024u + (unsigned)(((fr & 7) * 8 + ((h * 4 + fg) ^ (fr & 7))) * 16);
        const unsigned w_rd = W_BASE + (unsigned)(wn * WTN) * 1024u + lane * 16;
        unsigned a_rs = 0, w_rs = W_TILE;                 // slots of the tile whose fragments are read next (kt0 + 1)
        start_acc();      // (while the first copies are on their way)
        // before the first tile: A unit u0 and W tile kt0, issued in tile -4 at the latest
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * ODD + EVEN));
        __syncthreads();
        bf16x8 fw[2][WTN], fa[2][WTM];
#pragma unroll
        for (int i = 0; i < WTN; ++i) fw[0][i] = *reinterpret_cast<const bf16x8*>(smem + w_rd + i * 1024);
#pragma unroll
        for (int jj = 0; jj < WTM; ++jj) fa[0][jj] = *reinterpret_cast<const bf16x8*>(smem + a_rd[0] + jj * 2048);

        // a k-tile's MFMAs with the LDS reads of the next tile and the copies of later ones between them
        const char* a_src = smem + a_rd[1];
        const char* w_src = smem + w_rd + w_rs;
#define W4_TILE(h)                                                                                  \
        {                                                                                           \
            constexpr int NA_C = (h) ? LPA_O : LPA_E, A_C0 = (h) ? 0 : LPA_O, NC = NA_C + LPW;      \
            __builtin_amdgcn_s_waitcnt(vmcnt_lgkm0_imm((h) ? FLY_O : FLY_E));                       \
            asm volatile("s_barrier" ::: "memory");                                                 \
            _Pragma("unroll") for (int i = 0; i < WTN; ++i)                                         \
                _Pragma("unroll") for (int jj = 0; jj < WTM; ++jj) {                                \
                    const int q = i * WTM + jj;                                                     \
                    const int cp = q % CPM == CPM - 1 && q / CPM < NC ? q / CPM : -1;               \
                    if (cp >= 0 && cp < NA_C)                                                       \
                        mfma_acc_copy(acc[i][jj], fw[h][i], fa[h][jj], a_to, (unsigned)(A_C0 + cp) * 4096u, aoff[cp >= 0 && cp < NA_C ? A_C0 + cp : 0], a_at); \
                    else if (cp >= 0)                                                               \
                        mfma_acc_copy<ONCE>(acc[i][jj], fw[h][i], fa[h][jj], w_to, W_BASE + (unsigned)(cp - NA_C) * 4096u, woff[cp >= NA_C ? cp - NA_C : 0], w_at); \
                    else mfma_acc(acc[i][jj], fw[h][i], fa[h][jj]);                                 \
                    if (q % RPM == RPM - 1 && q / RPM < WTN + WTM) {                                \
                        const int rd = q / RPM;                                                     \
                        if (rd < WTM) fa[(h) ^ 1][rd < WTM ? rd : 0] = *reinterpret_cast<const bf16x8*>(a_src + rd * 2048); \
                        else fw[(h) ^ 1][rd >= WTM ? rd - WTM : 0] = *reinterpret_cast<const bf16x8*>(w_src + (rd - WTM) * 1024); \
                    }                                                                               \
                    if (q == UP0) w_ko = step_to(w_ko, 1024u, w_end);                           \
                    if (q == UP1) { w_at = w0 + w_ko; w_to = lds_wave + w_rs; }                 \
                    if (q == UP2) w_rs = ring_next<W_TILE, NWS * W_TILE>(w_rs);                 \
                    if ((h) == 0 && q == UP1) a_ko = step_to(a_ko, 128u, a_end);                \
                    if ((h) == 0 && q == UP2) { a_at = a0 + a_ko; a_to = lds_wave + a_rs; }     \
                    if ((h) == 0 && q == UP3) a_rs = ring_next<A_UNIT, NA * A_UNIT>(a_rs);      \
                }                                                                                   \
            a_src = smem + a_rs + a_rd[h];                                                          \
            w_src = smem + w_rs + w_rd;                                                             \
        }
        // tile 2 u reads its successor from its own unit, tile 2 u + 1 from the next: a_rs moves on after an even tile
        for (int kt = kt0; kt < kt1; kt += 2) {
            W4_TILE(0)
            W4_TILE(1)
        }
    } else {
        start_acc();
    }
#undef W4_TILE
    // every copy has landed and every read of LDS has come back, in every wave: LDS is free for the results
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");   // (and the last MFMAs have written their accumulators)
    __syncthreads();
    constexpr int REGION = (int)((W_BASE + NWS * W_TILE) / 4) & ~1023;
    char* region = smem + wave * REGION;
    const int mw = m0 + wm * WTM * 16;                // the wave's first row
    constexpr int E = 16 / (int)sizeof(TC);
    const int lane_out = w4_lane();
    float rs = 1.f;
    if constexpr (SCALE) {
        row_ss += __shfl_xor(row_ss, 16, 64);
        row_ss += __shfl_xor(row_ss, 32, 64);
        rs = rsqrtf(row_ss * sc.inv_dim + sc.eps);
    }
    auto scaled = [&](const floatx4& v) {
        if constexpr (SCALE) return floatx4{v[0] * rs, v[1] * rs, v[2] * rs, v[3] * rs};
        else return v;
    };
    if constexpr (GLU) {
        static_assert(WTN % 2 == 0, "gate and up groups come in pairs");
        w4_store_rows<WTN / 2, REGION, TC, WTM>(region, [&](int i, int jj) { return glu4(scaled(acc[2 * i][jj]), scaled(acc[2 * i + 1][jj]), ex.act); },
                                           C, (size_t)n_out, mw, (n0 + wn * WTN * 16) / 2, M, n_out, lane_out,
                                           n_out % E == 0);
    } else {
        // (partial sums of a split K: plane blockIdx.z of the launcher's float32 workspace, which it passes as C)
        int ldc = N;
        if constexpr (PLANES) ldc = ex.plane_cols;
        TC* out = PLANES ? C : C + (size_t)blockIdx.z * M * N;
        w4_store_rows<WTN, REGION, TC, WTM>(region, [&](int i, int jj) { return scaled(acc[i][jj]); }, out, (size_t)ldc, mw,
                                       n0 + wn * WTN * 16, M, N, lane_out, ldc % E == 0);
    }
}

// Whether a tile's offsets fit (see launch_far).
static bool w4_reaches(int rows, int cols, int K, int lda) {
    return (size_t)(rows - 1) * lda * 2 + 128 < (1ull << 32) && (size_t)(cols / 16) * (K / 32) * 1024 < (1ull << 32);
}

// splits > 1: the blocks of a tile split K among them in units of 64; part holds splits * M * N floats
template <int WTN, int NWS, bool GLU = false, int WGM = 2, bool SCALE = false, int WTM = 8>
static int launch_w4(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall ex, int c_dtype,
                     int n_out, hipStream_t s, int splits = 1, float* part = nullptr, bool reduce = true,
                     W4Scale sc = W4Scale{nullptr, 0, 0, 0.f, 0.f}) {
    TFF_REQUIRE(!SCALE || (M <= 16 && sc.ss && (splits <= 1 || !part)),
                "gemm: rows that lack their norm's factor: up to 16 of them and K in one part");
    TFF_REQUIRE(K % 64 == 0, "gemm: the four-wave tiles take K in units of 64, not K=%d", K);
    const int KB = K / 32;
    constexpr int BM = 16 * WTM * WGM, BN = (4 / WGM) * WTN * 16;
    if (splits <= 1 || !part) { splits = 1; part = nullptr; }
    TFF_REQUIRE(splits <= KB / 2, "gemm: %d parts of %d units of K", splits, KB / 2);
    const long TM = (M + BM - 1) / BM, TN = (N + BN - 1) / BN;
    const long tiles = w4_blocks<BM>(TM, TN);   // eight equal shares
    TFF_REQUIRE(tiles < (1L << 31), "gemm: too many tiles for M=%d N=%d", M, N);
    TFF_REQUIRE(w4_reaches(BM, BN, K, lda), "gemm: rows of %d elements at a stride of %d are too long", K, lda);
    const dim3 grid((unsigned)tiles, 1, splits);
    // the blocks of a split K leave plain float32 sums, plane by plane; a gate is applied when they are added up
    if (ex.plane_cols) {
        if constexpr (!GLU && !SCALE) {
            TFF_REQUIRE(splits == 1 && c_dtype == TFF_F32 && ex.plane_cols % BN == 0, "gemm: planes of %d columns on tiles of %d", ex.plane_cols, BN);
            gemm_bf16_w4_kernel<WTN, NWS, false, float, WGM, false, WTM, true><<<grid, 256, 0, s>>>(A, Wp, (float*)C, M, N, K, lda, KB, n_out, sc, ex);
            return tff_check_launch("gemm_bf16_w4");
        } else {
            return tff_fail("gemm: planes of a gated or scaled product");
        }
    }
    auto launch = [&](auto ONCE) {
        constexpr bool once = decltype(ONCE)::value;
        if (splits > 1)
            gemm_bf16_w4_kernel<WTN, NWS, false, float, WGM, false, WTM><<<grid, 256, 0, s>>>(A, Wp, part, M, N, K, lda, KB, 0, sc, ex);
        else if (c_dtype == TFF_F32)
            gemm_bf16_w4_kernel<WTN, NWS, GLU, float, WGM, SCALE, WTM, false, once><<<grid, 256, 0, s>>>(A, Wp, (float*)C, M, N, K, lda, KB, n_out, sc, ex);
        else
            gemm_bf16_w4_kernel<WTN, NWS, GLU, bf16_t, WGM, SCALE, WTM, false, once><<<grid, 256, 0, s>>>(A, Wp, (bf16_t*)C, M, N, K, lda, KB, n_out, sc, ex);
    };
    // A weight that one block reads, K in one part: 40 and 100 rows of 24,576 x 4,096 38.0 / 35.6 and 43.9 / 40.7 us, 17 rows of 151,936
    // 218 / 192 (plain loads / once), on one tile of 256 rows 200 of 24,576 x 4,096, gated, 61.3 / 58.5, of 34,816 x 5,120 105.7 / 102.9.  The short
    // streams of a split K lose by it: 100 rows of 4,096 x 4,096 16.3 / 19.4, 128 of 7,168 x 5,120 24.8 / 27.8.
    if (ex.once && TM == 1 && splits == 1) launch(std::true_type{});
    else launch(std::false_type{});
    if (int rc = tff_check_launch("gemm_bf16_w4")) return rc;
    if (splits > 1 && reduce) {
        return launch_reduce<GLU>(part, splits, M, N, C, GLU ? n_out : N, ex, c_dtype, s);
    }
    return 0;
}

// ------------------------------------------------- few rows, no workspace ---
// 17 to 64 rows whose plan splits K, where the caller brings no room for the parts' sums: a block owns 32 rows of W for the whole of K, its
// eight waves split K in contiguous runs, UNROLL k-steps of loads each before the first is used, and their sums meet in LDS in a fixed order.
template <int MT, int UNROLL, typename TC>
__global__ __launch_bounds__(512) void gemm_bf16_row_tiles_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ Wp, TC* __restrict__ C, int M, int N, int K,
                                                                  int lda, int KB, const GemmEpilogue ex) {
    constexpr int R = 2, KSPLIT = 8;
    __shared__ floatx4 part[KSPLIT][R * MT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int fr = lane & 15, fg = lane >> 4;
    const int NB = (N + 15) / 16;
    const int nb0 = blockIdx.x * R;
    floatx4 acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const floatx4 b = ex.bias && wave == 0 ? bias4(ex.bias, (nb0 + r) * 16 + fg * 4, NB) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = b;
    }
    const int per = (KB + KSPLIT - 1) / KSPLIT;
    int s0 = wave * per;
    const int s_end = min(KB, s0 + per);
    // Row groups past the end of W and rows past the end of A repeat the last: their results are never stored.
    const bf16_t* wfrag[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wfrag[r] = Wp + (size_t)min(nb0 + r, NB - 1) * KB * 512 + lane * 8;
    const bf16_t* arow[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) arow[t] = A + (size_t)min(t * 16 + fr, M - 1) * lda;
    const int full_end = min(s_end, K / 32);   // steps below K / 32 have all their 32 k in A
    for (; s0 + UNROLL <= full_end; s0 += UNROLL) {
        uint4 rw[UNROLL][R], ra[UNROLL][MT];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
#pragma unroll
            for (int r = 0; r < R; ++r) rw[u][r] = ld16(wfrag[r] + (size_t)(s0 + u) * 512);
#pragma unroll
            for (int t = 0; t < MT; ++t) ra[u][t] = ld16(arow[t] + (s0 + u) * 32 + fg * 8);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(rw[u][r]), as_frag(ra[u][t]), acc[r][t], 0, 0, 0);
    }
    // what is left, a step at a time; in the last step of K some k may not exist in A
    for (; s0 < s_end; ++s0) {
        const int k = s0 * 32 + fg * 8;
        const bool kok = k < K;
        uint4 rw[R], ra[MT];
#pragma unroll
        for (int r = 0; r < R; ++r) rw[r] = ld16(wfrag[r] + (size_t)s0 * 512);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint4 v = ld16(arow[t] + (kok ? k : 0));
            ra[t] = kok ? v : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(rw[r]), as_frag(ra[t]), acc[r][t], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[wave][r * MT + t][lane] = acc[r][t];
    __syncthreads();
    if (wave != 0) return;      // the first wave adds up
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            floatx4 v = part[0][r * MT + t][lane];
#pragma unroll
            for (int w = 1; w < KSPLIT; ++w) {
                const floatx4 p = part[w][r * MT + t][lane];
                v[0] += p[0]; v[1] += p[1]; v[2] += p[2]; v[3] += p[3];
            }
            const int n = (nb0 + r) * 16 + fg * 4, m = t * 16 + fr;
            if (m < M && n < N) store4<TC>(C + (size_t)m * N + n, v, n, N, (N % 4) == 0);
        }
}

template <int MT>
static int launch_row_tiles(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmEpilogue& ex, int c_dtype, hipStream_t s) {
    const dim3 grid(((N + 15) / 16 + 1) / 2);
    if (c_dtype == TFF_F32) gemm_bf16_row_tiles_kernel<MT, 4, float><<<grid, 512, 0, s>>>(A, Wp, (float*)C, M, N, K, lda, (K + 31) / 32, ex);
    else gemm_bf16_row_tiles_kernel<MT, 4, bf16_t><<<grid, 512, 0, s>>>(A, Wp, (bf16_t*)C, M, N, K, lda, (K + 31) / 32, ex);
    return tff_check_launch("gemm_bf16_row_tiles");
}

// The tiled product's plan for M > 16: which tile, and into how many parts the blocks of a
// tile split K, by a small cost model (see plan_for).  With K in units of 64: the four-wave
// kernel's tiles of 256 and 192 rows (256, 192 or 128 columns), of 128 (384, 256 or 128 columns) and 96 rows (128) and,
// up to 64 and 32 rows, of 64 and 32 rows (256 or 128 columns), and from 65 to 512 rows also
// 64 x 128 with several row tiles; otherwise the sixteen-wave kernel's tiles.
struct GemmPlan { int tile; int bn; int splits; };   // tile = rows of a block tile
// Up to 16 rows, not gated: more groups of 16 columns than CUs, but at most 1.6 times as many.
static bool little_more_groups_than_cus(int N) {
    const int nb = (N + 15) / 16, cus = tff_device_cus();
    return nb > cus && nb * 10 <= cus * 16;
}
// One row tile of 32 rows, K in one part: the width (128 or 256 columns) that plan_for's model prices lowest.
static int plan_rows32(int N, int K) {
    const double CUS = (double)tff_device_cus();
    const int widths[2] = {128, 256};
    const double rates[2] = {1.3e6, 1.4e6};
    int best = 256;
    double best_t = 1e30;
    for (int i = 0; i < 2; ++i) {
        const double blocks = (double)((N + widths[i] - 1) / widths[i]);
        const double bw = fmin(6.0e4, 7.72e6 / fmin(blocks, CUS));
        const double unit = fmax(2.0 * 32 * widths[i] * 64.0 / rates[i], widths[i] * 128.0 / bw);
        const double t = ceil(blocks / CUS) * (K / 64.0 * unit + 3.0);
        if (t < best_t) { best_t = t; best = widths[i]; }
    }
    return best;
}

// Up to 16 rows, gated: the streaming kernel's time grows with the rows, from nine on by a tenth; that of the four-wave kernel's tiles of 32 rows, K in
// one part, does not, and hangs on how their blocks go round the CUs: ahead where they fill three quarters of one round, behind with fewer, and in
// a second round.  us at 8 / 9 / 16 rows after a norm, streaming against tiles, and the tiles: 51,200 x 5,120 79.5 / 83.4 / 90.3 against 79.5, 200;
// 28,672 x 8,192 71.3 / 75.2 / 78.7 against 75, 224; 27,648 x 5,120 46.1 / 49.0 / 53.2 against 47.5, 216; 24,576 x 4,096 31.7 / 37.6 / 34.1 against 36,
// 192; 34,816 x 5,120 56.9 / 60.6 / 65.6 against 65, 136; 22,016 x 8,192 54.3 / 59.9 / 60.2 against 62.5, 172; 8,192 x 12,288 33.4 / 34.3 / 35.9 against
// 83, 64.  11,000 products of 2e7 to 5e8 elements and 2 to 16 rows: 0.5 % from the better one on average.  (The largest weights are on tiles with any rows:
// within 2 % there.)
static bool few_rows_gated_on_tiles(int M, int N, int K) {
    const double w = (double)N * K;
    if (K % 64 != 0 || !(w >= 2.4e8 || (M >= 9 && w >= 4e7))) return false;
    const int bn = plan_rows32(N, K), cus = tff_device_cus(), blocks = (N + bn - 1) / bn;
    return blocks <= cus && blocks * 4 >= cus * 3;
}

// plane > 0: the columns of several products, so many each; a tile takes columns of one of them, and K is not split.
// unary: an activation follows, in the kernel that adds up the parts, which one part then has as well (200 rows of 18,432 x 4,096, a squared relu: in
// one part, as without it, 63 us, in two 54).  Where K is split the activation sees float32 sums: its constants stay as they were when the
// others were fitted again, so that no size loses them.
static GemmPlan plan_for(int M, int N, int K, bool glu, bool keep, int plane = 0, bool unary = false) {
    const double CUS = (double)tff_device_cus();
    // Up to 16 rows: the streaming kernel.  Not where the caller takes partial sums anyway, the groups of 16 columns go badly round the CUs and the
    // weight is large: those rows are on tiles that split K, with the norm in a kernel of its own.  These lines were drawn beside a streaming
    // kernel that took a third longer, and are not where the two meet now: with the norm and the next product, streaming against tiles,
    // us at 9 / 16 rows, 5,120 x 17,408 43 / 49 against 56; 2,560 x 20,480 30 / 37 against 39; 12,800 x 22,528 at 16 rows 149 against 122.
    if (M <= 16 && glu && few_rows_gated_on_tiles(M, N, K)) return {32, plan_rows32(N, K), 1};
    if (M <= 16 && plane) return {0, 0, 1};
    if (M <= 16) {
        const int nb = (N + 15) / 16;
        const double fill = (double)nb / (ceil(nb / CUS) * CUS);
        if (glu || !keep || fill >= 0.8 || (double)N * K < 40e6) return {0, 0, 1};
        if (little_more_groups_than_cus(N) && (M <= 8 || (double)N * K < 45e6)) return {0, 0, 1};
    }
    const int nk = (K + 63) / 64;
    if (K % 64 == 0) {
        // The four-wave kernel's tiles (256 or 192 rows on 2 x 2 waves, 128 or 96 rows on 1 x 4) and, up to 512 rows,
        // its 64 x 128, two blocks to a CU.  A block goes through its part of K in
        // units of 64; a unit takes what its MFMAs take at the tile's rate or what its columns of W take
        // to arrive, whichever is longer: a block's share of the HBM stream, at most what one CU pulls.
        // Blocks go round the CUs of an XCD, which takes an eighth of the tiles in all their parts: 42 tiles in six parts are 252 blocks, but on some
        // XCDs 36 for 32 CUs, a second round (160 rows of 8,064 x 14,144 104 us, in four parts 69; 411 rows of 10,496 x 13,120, 82 tiles in three parts, 201,
        // in two 133).  Each round ends with the pipeline filled and the tile stored.  The constants are
        // fitted to products of the 0.6B to 14B shapes and of the other designs, every tile with
        // 1 .. 8 parts timed on an MI355X (weights in turn that no cache holds, rows from five places), in five pieces:
        // * Results of one kernel or of the sum over the parts, more than 64 rows: 4,347 products of 65 .. 16,500 rows.  The pick is 0.8 % from the best
        //   candidate on average; against the tiles of 256, 128 and 64 rows alone 0.988 of the time (513 to 1,500 rows 0.967), and in 2 of 100 slower by
        //   more than 3 % (in 4 of 100 with constants whose stream's bound was half as high again as a copy's rate: gated, 68 rows of 24,576 x 4,096
        //   43.4 / 51.2 us, 145 rows 53.0 / 56.1).
        // * Sums kept for a norm, more than 64 rows, no more columns than K: 3,875 products of 65 .. 16,500 rows, each timed with the norm behind it: 1.0 % from
        //   the best, 0.972 of the time of the tiles of 256, 128 and 64 rows by their constants, in 2 of 100 slower by more than 3 %.  The norm reads the
        //   parts one after the other, 0.3 us each beside their bytes (116 rows of 2,048 x 2,048: four parts 10.9, eight 12.7).
        // * Before an activation, more than 64 rows: an older fit of results (see above).
        // * Kept sums of more columns than K, which no model's product into its stream has: constants of an older fit.
        // * Up to 64 rows the four waves side by side take 64 or 32 rows: a product of so few rows is its
        //   weight's stream, and a block that does not work through 128 rows for 32 asks for its next
        //   columns sooner (3 to 10 % less time than the tiles of 128 rows and the sixteen-wave kernel's
        //   64 x 128 on the four products of the three shapes at 17 to 64 rows; their rates fitted to
        //   those 88 cases stand for that, the pick 0.5 % from the best on average, 5 % at worst).
        // Tiles of 192 and 96 rows are finer steps between the others: blocks that fill the CUs, or less padding.  They take K from 1,024 on and whole
        // columns of tiles, which the products they are fitted to have; not one row tile of few rows, whose time is the weight's stream (161 rows of 34,816 x 5,120
        // gated 91 on 256 x 192, 101 on 192 x 256); up to 384 rows only where they pad less than tiles of 128, if
        // the sums are not kept; and beyond 2,048 rows K in one part (2,210 of 4,096 x 18,432 257 on 256 x 192, 335 on 192 x 128 in two).
        // From 1,500 rows on they have to be 2 % ahead: large products are bound by the power the card allows, of which a smaller tile's reads take more
        // (slower than the tiles before by more than 2 %: 2 of 100 such products without this margin, 0.7 with it).
        // Three and six parts are for kept sums of 129 to 1,024 rows: beyond, the parts' traffic grows and the rounds are many.  Beyond 2,048 rows kept parts that
        // are more than the caches hold are not cut further (but few columns are: 2,219 rows of 128 x 15,424 in eight parts 25.9, in two 48.6).
        // The kernel that adds up results' parts costs 3.5 us beside its bytes, 2.3 where it also joins gate and up (68 rows of 4,096 x 1,024 in one part 7.4,
        // in four 9.9; 600 gated rows of 512 x 1,088 in two parts rather than one).
        // A rate is in flops a microsecond of a CU; ends: us that a block's first fetch and storing its tile take.  Of results, of kept sums, before an activation, of the
        // older fit's, up to 64 rows.
        struct Cand { int bm, bn, slots; double rate, ends, rate_kept, ends_kept, rate_act, ends_act, rate_wide, rate_few; };
        static const Cand cands[15] = {
            {256, 256, 1, 7.58e6, 0.93, 8.16e6, 1.72, 8.43e6, 1.02, 6.45e6, 0}, {256, 192, 1, 7.34e6, 1.07, 7.76e6, 2.57, 7.65e6, 1.04, 6.10e6, 0},
            {256, 128, 1, 6.25e6, 1.10, 6.86e6, 1.45, 6.20e6, 0.95, 5.42e6, 0}, {192, 256, 1, 7.33e6, 0.85, 7.70e6, 1.66, 0, 0, 0, 0},
            {192, 192, 1, 6.83e6, 1.61, 5.95e6, 1.92, 0, 0, 0, 0}, {192, 128, 1, 5.72e6, 0.48, 5.27e6, 0.67, 0, 0, 0, 0},
            {128, 384, 1, 6.48e6, 0.98, 7.05e6, 3.67, 10.6e6, 1.76, 6.49e6, 3.24e6}, {128, 256, 1, 6.05e6, 1.38, 7.00e6, 0.40, 6.18e6, 0.96, 5.38e6, 4.61e6},
            {128, 128, 1, 4.37e6, 0.64, 5.30e6, 0.92, 4.41e6, 0.61, 3.56e6, 3.45e6}, {96, 128, 1, 3.70e6, 1.01, 4.12e6, 0.40, 0, 0, 0, 0},
            {64, 256, 1, 0, 0, 0, 0, 0, 0, 0, 2.4e6}, {64, 128, 1, 0, 0, 0, 0, 0, 0, 0, 2.0e6},
            {32, 256, 1, 0, 0, 0, 0, 0, 0, 0, 1.4e6}, {32, 128, 1, 0, 0, 0, 0, 0, 0, 0, 1.3e6},
            {64, 128, 2, 2.70e6, 0.15, 5.29e6, 0.08, 2.67e6, 0.12, 2.48e6, 0}};
        const bool few = M <= 64, wide = keep && !few && N > K, kept = keep && !few && !wide, act = unary && !few;
        // bytes a microsecond of all CUs together (as a bound it is high: what the stream costs beside MFMAs is in the tiles' rates) and of one alone
        const double HBM = few ? 7.72e6 : wide ? 8.18e6 : kept ? 10.6e6 : act ? 9.41e6 : 6.99e6;
        const double CU_MAX = few ? 6.0e4 : wide ? 6.54e4 : act ? 6.04e4 : 4.98e4;
        GemmPlan best = {128, 128, 1};
        double best_t = 1e30;
        for (const Cand& c : cands) {
            const bool between = c.bm == 192 || c.bm == 96;
            if (c.bm == 256 && M <= 64) continue;
            if (between) {
                if (few || wide || unary || K < 1024 || N % c.bn || M <= (c.bm == 192 ? 192 : 128)) continue;
                if (!kept && M <= 384 && (M + c.bm - 1) / c.bm * c.bm >= (M + 127) / 128 * 128) continue;
            }
            if (c.slots == 1 && c.bm <= 64 && M > c.bm) continue;         // (four waves side by side: one row tile)
            if (c.slots == 2 && (M <= 64 || M > 512)) continue;            // (64 x 128 with several row tiles)
            if (plane % c.bn) continue;
            for (int S = 1; S <= (plane ? 1 : (glu && M > 64) ? 2 : 8); S += S < 4 ? 1 : 2) {
                if (S > 1 && nk / S < 4) break;
                if (S % 3 == 0 && !(kept && M > 128 && M <= 1024)) continue;
                const double plane_bytes = (double)M * N * 4.0;
                if (S > (between ? 1 : 2) && kept && M > 2048 && S * plane_bytes > 32e6) break;
                const double blocks = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * S;
                const double mine = ceil(blocks / S / 8.0) * S, xcd = CUS / 8.0;      // an XCD's blocks, and its CUs
                const double rounds = ceil(mine / (xcd * c.slots)), at_once = fmin(blocks, CUS * c.slots);
                double rate = kept ? c.rate_kept : act ? c.rate_act : c.rate, ends = kept ? c.ends_kept : act ? c.ends_act : c.ends, units = (nk + S - 1) / S;
                double streams = ceil((double)N / c.bn) * S;              // (row tiles fetch a column tile's weight once between them)
                double share = c.slots == 2 && mine > xcd ? (kept ? 3.52 : act ? 1.77 : 1.91) : 1.0;     // blocks that share a CU's MFMAs, and each other's waits
                if (few || wide) {
                    rate = few ? c.rate_few : c.rate_wide;
                    ends = few ? 3.0 : 1.29 + 2.55 * (c.bm * c.bn / 65536.0);
                    units = (double)nk / S;
                    streams = at_once;
                    share = fmin((double)c.slots, ceil(blocks / CUS));
                }
                const double bw = fmin(CU_MAX, HBM / fmin(at_once, streams));
                const double unit = fmax(2.0 * c.bm * c.bn * 64.0 * share / rate, c.bn * 128.0 / bw);
                double t = rounds * (units * unit + ends);
                // the partial sums: written, read and added by a second kernel, or (kept) read by the
                // consumer in place of one plane
                // (from the caches as long as they are some 32 MB)
                if (S > 1 && keep) t += (S - 1.0) * (plane_bytes / (few || (kept && S * plane_bytes <= 32e6) ? 4e6 : kept ? 2.56e6 : 1.97e6) + (kept ? 0.3 : 0.0));
                else if (S > 1 || unary) t += S * plane_bytes / (few ? 2.54e6 : act ? 2.21e6 : 2.2e6) + (few ? 2.7 : glu ? 2.28 : act ? 3.0 : 3.45);
                if (between && M >= 1500) t *= 1.02;
                if (t < best_t) { best_t = t; best = {c.bm, c.bn, S}; }
            }
        }
        return best;
    }
    if (M <= 64) {
        // A stream of W: a CU pulls a block's k-tile of 64 (16 KB) in some 0.63 us whatever else
        // runs, blocks go round the 256 CUs, and the most loaded CU sets the time.  Splitting K
        // evens the load out (272 blocks are two rounds for 16 CUs and one for the rest; 1,088
        // quarters are five rounds against 4.25) at the price of the partial sums' traffic and
        // of some 4 us that a block spends before its first and after its last k-tile (two
        // blocks of a CU overlap theirs).
        const long blocks = (N + 127) / 128;
        int best_s = 1;
        double best_t = 1e30;
        for (int S = 1; S <= 8; S *= 2) {
            if (S > 1 && nk / S < 4) break;
            double t = ceil(blocks * S / CUS) * ceil((double)nk / S) * 0.63 + ceil(blocks * S / (2.0 * CUS)) * 4.0 + 1.0;
            if (S > 1) t += keep ? (S - 1.0) * M * N * 4.0 / 4e6 : (double)S * M * N * 8.0 / 4e6 + 3.0;
            if (t < best_t) { best_t = t; best_s = S; }
        }
        return {64, 128, best_s};
    }
    // K in no units of 64, more than 64 rows: the sixteen-wave kernel's tiles.  rate: flops a microsecond
    // that a CU sustains on blocks of this tile; slots: blocks a CU holds.
    struct Cand { int bm, bn, slots; double rate; };
    static const Cand cands_w16[5] = {{256, 256, 1, 5.2e6}, {256, 192, 1, 4.4e6}, {128, 256, 1, 3.6e6},
                                      {128, 128, 1, 2.6e6}, {64, 128, 2, 2.2e6}};
    GemmPlan best = {256, 256, 1};
    double best_t = 1e30;
    for (const Cand& c : cands_w16) {
        for (int S = 1; S <= (glu ? 2 : 8); S *= 2) {
            // gate and up groups come in pairs, an even number a wave: three a wave of the sixteen do not do
            if (glu && c.bn == 192) break;
            if (S > 1 && nk / S < 8) break;
            const double blocks = (double)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * S;
            const double rounds = ceil(blocks / (CUS * c.slots));
            // a round: the blocks' work at the tile's rate plus some 3 us to fill the pipeline and
            // store the tile; a last round that fills part of the machine takes as long as a full one
            const double round_us = 2.0 * c.bm * c.bn * ((double)K / S) * c.slots / c.rate + 3.0;
            double t = round_us * rounds + 3.0;
            // the partial sums: written, read and added by a second kernel, or (kept) read by the
            // consumer in place of one plane
            if (S > 1) t += keep ? (S - 1.0) * M * N * 4.0 / 4e6 : (double)S * M * N * 4.0 / 3e6 + 3.0;
            if (t < best_t) { best_t = t; best = {c.bm, c.bn, S}; }
        }
    }
    return best;
}

// A product in one part before an activation (tff_gemm_unary) leaves float32 sums, which the sum's kernel reads, as long as their
// traffic, twice that of sums in bfloat16, is little beside the product's own work, which grows with K: wherever splitting K in two is
// not far behind either.  us, bfloat16 and a kernel over it / float32, gelu: 50 rows of 18,432 x 4,096 36.6 / 37.3, 122 46.4 / 48.7, 234 61.6 / 63.8,
// 102 of 9,216 x 2,048 16.0 / 16.1; past the line 1,500 rows of 9,216 x 2,048 would be 62 / 69, and the activation is a kernel over
// the product's own type.  In the tiles' epilogue the exact gelu takes longer than in a kernel of its own, one wave a SIMD with
// nothing beside it: 200 rows of 18,432 68, 2,048 rows 300 for 262.
static bool unary_in_float32(const GemmPlan& p, int M, int N, int K) {
    if (p.tile == 0 || p.splits > 1 || K % 64) return false;
    return (long)M * N <= (K < 6144 ? 1150L : 3300L) * K;
}

TFF_API size_t tff_gemm_workspace_bytes(int M, int N, int K, int ab_dtype, int glu, int keep_partials) {
    if (ab_dtype != TFF_BF16 || M <= 0 || N <= 0 || K <= 0) return 0;
    const GemmPlan p = plan_for(M, N, K, glu != 0, keep_partials != 0);
    return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

// For tests and tuning: the plan's tile (rows x columns) and number of parts.
TFF_API int tff_gemm_plan(int M, int N, int K, int glu, int keep_partials, int* tile_rows, int* tile_cols,
                          int* splits) {
    const GemmPlan p = plan_for(M, N, K, glu != 0, keep_partials != 0);
    if (tile_rows) *tile_rows = p.tile;
    if (tile_cols) *tile_cols = p.bn;
    if (splits) *splits = p.splits;
    return 0;
}

// The four-wave tiles address a block's rows and its columns of W by 32-bit offsets.  Rows or a stride too long for a plan's tile (256 rows
// 8.4 million elements apart, K of 11 million on 192 columns) go to the sixteen-wave kernel, which has 64 bits a copy, K in as many parts.
template <bool GLU>
static int launch_far(const GemmPlan& plan, const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda, const GemmCall ex, int c_dtype,
                      int n_out, hipStream_t s, float* part, bool reduce) {
    TFF_REQUIRE((size_t)15 * lda * 2 + 128 < (1ull << 32), "gemm: row stride %d too large", lda);
    if (plan.tile <= 64) return launch_async_g<2, 2, 2, 4, 3, GLU>(A, Wp, C, M, N, K, lda, ex, c_dtype, n_out, s, plan.splits, part, reduce);
    if (plan.tile <= 128 && plan.bn == 128)
        return launch_async_g<2, 2, 4, 4, 3, GLU>(A, Wp, C, M, N, K, lda, ex, c_dtype, n_out, s, plan.splits, part, reduce);
    if (plan.tile <= 128) return launch_async_g<2, 4, 4, 4, 3, GLU>(A, Wp, C, M, N, K, lda, ex, c_dtype, n_out, s, plan.splits, part, reduce);
    return launch_async_g<4, 4, 4, 4, 5, GLU, 1, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, n_out, s, plan.splits, part, reduce);
}

// A product by its plan (planned_splits: the parts it would have with room for their sums).
static int run_plan(const GemmPlan& plan, int planned_splits, bool far, const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda,
                    const GemmCall ex, int c_dtype, int glu_out, float* workspace, bool red, hipStream_t s) {
    const int S = plan.splits;
    if (glu_out > 0) {
        TFF_REQUIRE(N % 32 == 0 && glu_out <= N / 2 && glu_out > N / 2 - 16,
                    "gemm: a gated weight of %d rows does not fit %d output columns", N, glu_out);
        if (plan.tile == 0) return tff_gemm_few_rows(0, A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, FewRowsFuse{});
        if (far) return launch_far<true>(plan, A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, workspace, true);
        if (plan.tile <= 64 && K % 64 == 0) {                // the four waves side by side on 64 or 32 rows
            if (plan.tile == 32 && plan.bn == 128) return launch_w4<2, 5, true, 1, false, 2>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            if (plan.tile == 32) return launch_w4<4, 5, true, 1, false, 2>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            if (plan.bn == 128) return launch_w4<2, 5, true, 1, false, 4>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            return launch_w4<4, 5, true, 1, false, 4>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
        }
        if (plan.tile == 64)
            return launch_async_g<2, 2, 2, 4, 3, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
        if (K % 64 == 0) {
            if (plan.tile == 128) {
                if (plan.bn == 128) return launch_w4<2, 5, true, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
                if (plan.bn == 256) return launch_w4<4, 5, true, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
                return launch_w4<6, 4, true, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            }
            if (plan.tile == 192) {
                if (plan.bn == 128) return launch_w4<4, 5, true, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
                if (plan.bn == 192) return launch_w4<6, 5, true, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
                return launch_w4<8, 5, true, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            }
            if (plan.tile == 96) return launch_w4<2, 5, true, 1, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            if (plan.bn == 128) return launch_w4<4, 5, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            if (plan.bn == 192) return launch_w4<6, 5, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
            return launch_w4<8, 4, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
        }
        if (plan.tile == 128 && plan.bn == 128)
            return launch_async_g<2, 2, 4, 4, 3, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
        if (plan.tile == 128)
            return launch_async_g<2, 4, 4, 4, 3, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
        return launch_async_g<4, 4, 4, 4, 5, true, 1, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, s, S, workspace);
    }
    if (plan.tile == 0) return tff_gemm_few_rows(0, A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, FewRowsFuse{});
    if (plan.tile == 64 || plan.tile == 32) {
        // few columns and no room for partial sums: the streaming kernel, whose blocks split K
        // among their waves
        if (S == 1 && planned_splits > 1 && M <= 64) {
            if (M <= 32) return launch_row_tiles<2>(A, Wp, C, M, N, K, lda, ex, c_dtype, s);
            return launch_row_tiles<4>(A, Wp, C, M, N, K, lda, ex, c_dtype, s);
        }
        if (far) return launch_far<false>(plan, A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, workspace, red);
        if (K % 64 == 0) {                                   // the four waves side by side on 64 or 32 rows
            if (plan.tile == 32 && plan.bn == 128) return launch_w4<2, 5, false, 1, false, 2>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            if (plan.tile == 32) return launch_w4<4, 5, false, 1, false, 2>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            if (plan.bn == 128) return launch_w4<2, 5, false, 1, false, 4>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            return launch_w4<4, 5, false, 1, false, 4>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        }
        return launch_async_g<2, 2, 2, 4, 3>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
    }
    if (far) return launch_far<false>(plan, A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, workspace, red);
    if (K % 64 == 0) {
        if (plan.tile == 128) {
            if (plan.bn == 128) return launch_w4<2, 5, false, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            if (plan.bn == 256) return launch_w4<4, 5, false, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            return launch_w4<6, 4, false, 1>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        }
        if (plan.tile == 192) {
            if (plan.bn == 128) return launch_w4<4, 5, false, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            if (plan.bn == 192) return launch_w4<6, 5, false, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
            return launch_w4<8, 5, false, 2, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        }
        if (plan.tile == 96) return launch_w4<2, 5, false, 1, false, 6>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        if (plan.bn == 128) return launch_w4<4, 5>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        if (plan.bn == 192) return launch_w4<6, 5>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
        return launch_w4<8, 4>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
    }
    if (plan.tile == 128 && plan.bn == 128)
        return launch_async_g<2, 2, 4, 4, 3>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
    if (plan.tile == 128)
        return launch_async_g<2, 4, 4, 4, 3>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
    if (plan.bn == 192)
        return launch_async_g<4, 4, 4, 3, 5, false, 1, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
    return launch_async_g<4, 4, 4, 4, 5, false, 1, true>(A, Wp, C, M, N, K, lda, ex, c_dtype, 0, s, S, workspace, red);
}

// glu_out > 0: W holds gate and up groups in turn (N = 2 * ceil16(glu_out) rows) and C is
// [M, glu_out] = silu(gate) * up.  workspace: room for partial sums (tff_gemm_workspace_bytes);
// with less the blocks do not split K.
// bias (may be null): ceil16(N) float32 numbers in the order of W's rows, added to the product (before the gate's
// activation): the accumulators start from them (of a split K, the first part's).
// keep_partials: where the plan splits K, the partial sums stay in the workspace
// ([splits, M, N] float32) for the caller to add up, and C is not written.
int tff_gemm_bf16(const bf16_t* A, const bf16_t* Wp, void* C, int M, int N, int K, int lda,
                  const GemmCall ex, int c_dtype, int glu_out, float* workspace, size_t workspace_bytes,
                  int keep_partials, hipStream_t s) {
    TFF_REQUIRE(K % 8 == 0 && lda % 8 == 0,
                "gemm: the bfloat16 product needs the inner size (K=%d, row stride %d) to be a multiple of 8",
                K, lda);
    TFF_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)Wp % 16) == 0 && ((uintptr_t)C % 16) == 0,
                "gemm: operands must be 16-byte aligned");
    TFF_REQUIRE(c_dtype == TFF_F32 || c_dtype == TFF_BF16, "gemm: unknown output type %d", c_dtype);
    GemmPlan plan = plan_for(M, N, K, glu_out > 0, keep_partials != 0, ex.plane_cols, ex.unary != 0);
    const int planned_splits = plan.splits;
    if (!workspace || workspace_bytes < (size_t)plan.splits * M * N * sizeof(float)) plan.splits = 1;
    const bool far = plan.tile > 0 && K % 64 == 0 && !w4_reaches(plan.tile, plan.bn, K, lda);
    if (far && ex.plane_cols) {      // (one product after the other)
        GemmCall one = ex;
        one.plane_cols = 0;
        const size_t w_plane = (size_t)(ex.plane_cols / 16) * (K / 32) * 512;
        for (int p = 0; p < N / ex.plane_cols; ++p)
            if (int rc = tff_gemm_bf16(A + p * ex.a_step, Wp + p * w_plane, (float*)C + (size_t)p * M * ex.plane_cols, M, ex.plane_cols, K, lda, one,
                                       c_dtype, 0, nullptr, 0, 0, s)) return rc;
        return 0;
    }
    if (ex.unary && glu_out == 0 && !keep_partials && planned_splits == 1 && unary_in_float32(plan, M, N, K) && workspace &&
        workspace_bytes >= (size_t)M * N * sizeof(float)) {
        // K in one part, whose float32 results the sum's kernel takes as the only plane
        GemmCall plain = ex;
        plain.unary = 0;
        if (int rc = run_plan(plan, 1, far, A, Wp, workspace, M, N, K, lda, plain, TFF_F32, 0, nullptr, true, s)) return rc;
        return launch_reduce<false>(workspace, 1, M, N, C, N, ex, c_dtype, s);
    }
    TFF_REQUIRE(!ex.unary || (glu_out == 0 && !keep_partials && (plan.tile == 0 || plan.splits > 1)),
                "gemm: an activation is applied by the streaming kernel or to the sum over the parts of K");
    TFF_REQUIRE(!keep_partials || (glu_out == 0 && c_dtype == TFF_F32),
                "gemm: partial sums are kept for a plain float32 result only");
    return run_plan(plan, planned_splits, far, A, Wp, C, M, N, K, lda, ex, c_dtype, glu_out, workspace, !keep_partials, s);
}

// ---- the norm between two products of up to 16 rows, taken into them ----
static int check_fused_operands(const char* what, const void* A, const void* Wp, int M, int N, int K, int lda) {
    TFF_REQUIRE(A && Wp, "%s: null pointer", what);
    TFF_REQUIRE(M >= 1 && M <= 16 && N > 0 && K > 0 && lda >= K, "%s: bad sizes M=%d N=%d K=%d lda=%d (1 to 16 rows)",
                what, M, N, K, lda);
    TFF_REQUIRE(K % 8 == 0 && lda % 8 == 0, "%s: the inner size (K=%d, row stride %d) must be a multiple of 8", what,
                K, lda);
    TFF_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)Wp % 16) == 0, "%s: operands must be 16-byte aligned", what);
    return 0;
}

// resid[M, N] += A . W^T (bfloat16 A and packed W, float32 sums); x_out[M, N] = bfloat16 of the new
// resid times norm_w[N]; ss_out[m][g] (16 rows of ss_stride floats, ss_stride >= ceil(N / 16)) =
// sum of squares of the new resid over columns 16 g .. 16 g + 15 of row m.  N a multiple of 8.
TFF_API int tff_gemm_residual_prenorm(const void* A, const void* Wp, int M, int N, int K, int lda, float* resid,
                                      const float* norm_w, void* x_out, float* ss_out, int ss_stride,
                                      int w_once, tff_stream_t stream) {
    if (int rc = check_fused_operands("gemm_residual_prenorm", A, Wp, M, N, K, lda)) return rc;
    TFF_REQUIRE(resid && norm_w && x_out && ss_out, "gemm_residual_prenorm: null pointer");
    TFF_REQUIRE(N % 8 == 0 && ss_stride >= (N + 15) / 16, "gemm_residual_prenorm: N=%d must be a multiple of 8 and "
                "ss_out needs %d floats a row, has %d", N, (N + 15) / 16, ss_stride);
    TFF_REQUIRE(((uintptr_t)resid % 16) == 0 && ((uintptr_t)norm_w % 16) == 0 && ((uintptr_t)x_out % 8) == 0,
                "gemm_residual_prenorm: operands must be 16-byte aligned");
    FewRowsFuse fz{nullptr, 0, 0, 0.f, 0.f, resid, norm_w, (bf16_t*)x_out, ss_out, ss_stride, nullptr, 0.f};
    return tff_gemm_few_rows(2, (const bf16_t*)A, (const bf16_t*)Wp, resid, M, N, K, lda, GemmCall{{{nullptr, glu_act(__builtin_inff(), 1.0f, 0.0f)}, 0, 0, 0}, w_once}, TFF_F32, 0, (hipStream_t)stream, fz);
}

// resid[M, N] += A . W^T (bfloat16 A and packed W, float32 sums); x_out[M, N] = bfloat16 of
// tanh(alpha * resid) * norm_w + bias over the new resid: the norm without statistics in the epilogue of the
// product before it.  Up to 16 rows; N a multiple of 8.
TFF_API int tff_gemm_residual_dyt(const void* A, const void* Wp, int M, int N, int K, int lda, float* resid, float alpha,
                                  const float* norm_w, const float* bias, void* x_out, int w_once, tff_stream_t stream) {
    if (int rc = check_fused_operands("gemm_residual_dyt", A, Wp, M, N, K, lda)) return rc;
    TFF_REQUIRE(resid && norm_w && bias && x_out, "gemm_residual_dyt: null pointer");
    TFF_REQUIRE(N % 8 == 0, "gemm_residual_dyt: N=%d must be a multiple of 8", N);
    TFF_REQUIRE(((uintptr_t)resid % 16) == 0 && ((uintptr_t)norm_w % 16) == 0 && ((uintptr_t)bias % 16) == 0 &&
                ((uintptr_t)x_out % 8) == 0, "gemm_residual_dyt: operands must be 16-byte aligned");
    FewRowsFuse fz{nullptr, 0, 0, 0.f, 0.f, resid, norm_w, (bf16_t*)x_out, nullptr, 0, bias, alpha};
    return tff_gemm_few_rows(3, (const bf16_t*)A, (const bf16_t*)Wp, resid, M, N, K, lda, GemmCall{{{nullptr, glu_act(__builtin_inff(), 1.0f, 0.0f)}, 0, 0, 0}, w_once}, TFF_F32, 0, (hipStream_t)stream, fz);
}

// C = rstd[m] * (A . W^T) with rstd[m] = rsqrt(sum_g ss[m][g] / dim + eps), g < ss_count: the product
// after tff_gemm_residual_prenorm (A = its x_out, ss = its ss_out, dim = its N).  glu_out as in tff_gemm.
TFF_API int tff_gemm_row_scaled(const void* A, const void* Wp, void* C, int M, int N, int K, int lda, int c_dtype,
                                int glu_out, const float* ss, int ss_stride, int ss_count, int dim, float eps,
                                float glu_limit, float glu_alpha, float glu_up_offset, int w_once, tff_stream_t stream) {
    const GemmCall ex{{{nullptr, glu_act(glu_limit, glu_alpha, glu_up_offset)}, 0, 0, 0}, w_once};
    if (int rc = check_fused_operands("gemm_row_scaled", A, Wp, M, N, K, lda)) return rc;
    TFF_REQUIRE(C && ss && ((uintptr_t)C % 16) == 0 && ((uintptr_t)ss % 16) == 0, "gemm_row_scaled: null or unaligned pointer");
    TFF_REQUIRE(c_dtype == TFF_F32 || c_dtype == TFF_BF16, "gemm_row_scaled: unknown output type %d", c_dtype);
    TFF_REQUIRE(ss_count > 0 && ss_stride >= ss_count && ss_stride % 4 == 0 && dim > 0,
                "gemm_row_scaled: %d sums of squares a row, %d apart (a multiple of 4), over %d elements", ss_count,
                ss_stride, dim);
    if (glu_out > 0)
        TFF_REQUIRE(N % 32 == 0 && glu_out <= N / 2 && glu_out > N / 2 - 16,
                    "gemm_row_scaled: a gated weight of %d rows does not fit %d output columns", N, glu_out);
    // (the four-wave kernel's tiles of 32 rows take the rows' factors into their epilogue too)
    if (glu_out > 0 && few_rows_gated_on_tiles(M, N, K) && w4_reaches(32, plan_rows32(N, K), K, lda)) {
        const W4Scale sc{ss, ss_stride, ss_count, 1.0f / (float)dim, eps};
        const bf16_t* a = (const bf16_t*)A;
        const bf16_t* w = (const bf16_t*)Wp;
        hipStream_t s = (hipStream_t)stream;
        if (plan_rows32(N, K) == 128)
            return launch_w4<2, 5, true, 1, true, 2>(a, w, C, M, N, K, lda, ex, c_dtype, glu_out, s, 1, nullptr, true, sc);
        return launch_w4<4, 5, true, 1, true, 2>(a, w, C, M, N, K, lda, ex, c_dtype, glu_out, s, 1, nullptr, true, sc);
    }
    FewRowsFuse fz{ss, ss_stride, ss_count, 1.0f / (float)dim, eps, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0.f};
    return tff_gemm_few_rows(1, (const bf16_t*)A, (const bf16_t*)Wp, C, M, N, K, lda, ex, c_dtype, glu_out, (hipStream_t)stream, fz);
}

int tff_gemm_f32(const float* A, const float* W, void* C, int M, int N, int K, int lda,
                 int c_dtype, hipStream_t s);

TFF_API int tff_gemm(const void* A, const void* W, void* C, int M, int N, int K, int lda,
                     int ab_dtype, int c_dtype, int w_packed, int glu_out, const float* bias, float glu_limit,
                     float glu_alpha, float glu_up_offset, void* workspace, size_t workspace_bytes, int keep_partials,
                     int w_once, tff_stream_t stream) {
    TFF_REQUIRE(A && W && C, "gemm: null pointer");
    TFF_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm: bad sizes M=%d N=%d K=%d lda=%d", M, N, K, lda);
    if (M == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    if (ab_dtype == TFF_F32) {
        TFF_REQUIRE(!w_packed && glu_out == 0 && !keep_partials && !bias,
                    "gemm: the float32 product takes a plain row-major weight, no bias and keeps no partial sums");
        return tff_gemm_f32((const float*)A, (const float*)W, C, M, N, K, lda, c_dtype, s);
    }
    if (ab_dtype == TFF_BF16) {
        TFF_REQUIRE(w_packed, "gemm: the bfloat16 product takes a weight in fragment order");
        TFF_REQUIRE(((uintptr_t)workspace % 16) == 0, "gemm: the workspace must be 16-byte aligned");
        TFF_REQUIRE(((uintptr_t)bias % 16) == 0, "gemm: the bias must be 16-byte aligned");
        return tff_gemm_bf16((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda,
                             GemmCall{{{bias, glu_act(glu_limit, glu_alpha, glu_up_offset)}, 0, 0, 0}, w_once}, c_dtype, glu_out,
                             (float*)workspace, workspace ? workspace_bytes : 0, keep_partials, s);
    }
    return tff_fail("gemm: unknown operand type %d", ab_dtype);
}

// C = act(A . W^T), act one of unary_activation's kinds, where the product's plan lets a kernel apply it to float32 sums: the streaming
// kernel, or the sum over the parts of a split K, which may be one (unary_in_float32).  Else 0 there, and the activation is a kernel of its own.
TFF_API int tff_gemm_takes_unary(int M, int N, int K) {
    const GemmPlan p = plan_for(M, N, K, false, false, 0, true);
    return p.tile == 0 || p.splits > 1 || unary_in_float32(p, M, N, K);
}
// Room for its float32 sums.
TFF_API size_t tff_gemm_unary_workspace_bytes(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const GemmPlan p = plan_for(M, N, K, false, false, 0, true);
    return p.splits > 1 || unary_in_float32(p, M, N, K) ? (size_t)p.splits * M * N * sizeof(float) : 0;
}
TFF_API int tff_gemm_unary(const void* A, const void* W, void* C, int M, int N, int K, int lda, int c_dtype, int kind, void* workspace,
                           size_t workspace_bytes, int w_once, tff_stream_t stream) {
    TFF_REQUIRE(A && W && C, "gemm_unary: null pointer");
    TFF_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K && kind >= 1 && kind <= 4, "gemm_unary: bad sizes M=%d N=%d K=%d lda=%d or kind %d", M, N, K, lda, kind);
    TFF_REQUIRE(((uintptr_t)workspace % 16) == 0, "gemm_unary: the workspace must be 16-byte aligned");
    if (M == 0) return 0;
    return tff_gemm_bf16((const bf16_t*)A, (const bf16_t*)W, C, M, N, K, lda, GemmCall{{{nullptr, glu_act(__builtin_inff(), 1.0f, 0.0f)}, kind, 0, 0}, w_once},
                         c_dtype, 0, (float*)workspace, workspace ? workspace_bytes : 0, 0, (hipStream_t)stream);
}

// Several products of the same sizes in one launch: C[p] = A[p] . W[p]^T, p < planes, A[p] = A + p * a_step, C [planes, M, N] float32; W
// their weights one after the other in fragment order.  Four products of 4,096 x 4,096 of 1,500 rows go three times round the CUs
// instead of four times one that fills three quarters of them, and of one row they are one stream of 134 MB.
// us, one by one / now: 4 x 4,096 x 4,096, 1,500 rows 234 / 181, one row 31 / 25.
TFF_API int tff_gemm_planes_supported(int N, int K) { return N % 128 == 0 && K % 64 == 0; }
TFF_API int tff_gemm_planes(const void* A, size_t a_step, const void* W, float* C, int planes, int M, int N, int K, int lda, int w_once, tff_stream_t stream) {
    TFF_REQUIRE(A && W && C, "gemm_planes: null pointer");
    TFF_REQUIRE(M >= 0 && planes > 0 && N > 0 && K > 0 && lda >= K && (long)planes * N < (1L << 30), "gemm_planes: bad sizes %d x M=%d N=%d K=%d lda=%d",
                planes, M, N, K, lda);
    TFF_REQUIRE(tff_gemm_planes_supported(N, K) && a_step % 8 == 0, "gemm_planes: N=%d in units of 128, K=%d of 64, rows' planes (%zu apart) of 8", N, K, a_step);
    if (M == 0) return 0;
    return tff_gemm_bf16((const bf16_t*)A, (const bf16_t*)W, C, M, planes * N, K, lda, GemmCall{{{nullptr, glu_act(__builtin_inff(), 1.0f, 0.0f)}, 0, N, a_step}, w_once},
                         TFF_F32, 0, nullptr, 0, 0, (hipStream_t)stream);
}
// Their plan's tile, for tests.
TFF_API int tff_gemm_planes_plan(int planes, int M, int N, int K, int* tile_rows, int* tile_cols) {
    TFF_REQUIRE(planes > 0 && M > 0 && N > 0 && K > 0 && (long)planes * N < (1L << 30) && tff_gemm_planes_supported(N, K) && tile_rows && tile_cols,
                "gemm_planes_plan: bad sizes %d x M=%d N=%d K=%d", planes, M, N, K);
    const GemmPlan p = plan_for(M, planes * N, K, false, false, N);
    *tile_rows = p.tile;
    *tile_cols = p.bn;
    return 0;
}

// ------------------------------------------------------------- packing ---
// Row-major [N, K] -> fragment order, with zero padding to 16 rows and 32 k.
__global__ void pack_weight_kernel(const bf16_t* __restrict__ src, bf16_t* __restrict__ dst, int N,
                                   int K, int KB, size_t total_chunks) {
    // one thread per 16-byte chunk of the packed matrix
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= total_chunks) return;
    const int l = (int)(c & 63);
    const size_t frag = c >> 6;
    const int kb = (int)(frag % KB);
    const int nb = (int)(frag / KB);
    const int n = nb * 16 + (l & 15);
    const int k = kb * 32 + (l >> 4) * 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (n < N && k < K) v = *reinterpret_cast<const uint4*>(src + (size_t)n * K + k);   // K % 8 == 0
    *reinterpret_cast<uint4*>(dst + c * 8) = v;
}

TFF_API int tff_pack_weight(const void* src, void* dst, int N, int K, tff_stream_t stream) {
    TFF_REQUIRE(src && dst, "pack_weight: null pointer");
    TFF_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "pack_weight: inner size %d must be a multiple of 8", K);
    const int NB = (N + 15) / 16, KB = (K + 31) / 32;
    const size_t chunks = (size_t)NB * KB * 64;
    const size_t blocks = (chunks + 255) / 256;
    TFF_REQUIRE(blocks < 2147483647ULL, "pack_weight: matrix too large");
    pack_weight_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>((const bf16_t*)src, (bf16_t*)dst, N, K,
                                                                           KB, chunks);
    return tff_check_launch("pack_weight");
}

// Gather of rows out of a matrix in fragment order (the embedding of a model whose
// output head shares the table): out[t, :] = float(E[ids[t], :]).
__global__ void embed_packed_kernel(const bf16_t* __restrict__ table, const int32_t* __restrict__ ids,
                                    float* __restrict__ out, int H, int V, int KB) {
    const int t = blockIdx.x;
    int id = ids[t];
    const bool bad = id < 0 || id >= V;
    if (bad) id = 0;
    const bf16_t* base = table + (size_t)(id / 16) * KB * 512 + (id % 16) * 8;
    float* o = out + (size_t)t * H;
    for (int c = threadIdx.x; c < H / 8; c += blockDim.x) {   // chunk c holds k = 8c .. 8c+7
        const bf16_t* p = base + (size_t)(c / 4) * 512 + (c % 4) * 128;
        union { uint4 u; bf16_t h[8]; } v;
        v.u = *reinterpret_cast<const uint4*>(p);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[c * 8 + e] = bad ? __builtin_nanf("") : (float)v.h[e];
    }
}

TFF_API int tff_embed_packed(const void* table, const int32_t* ids, float* out, int T, int H, int V,
                             tff_stream_t stream) {
    TFF_REQUIRE(table && ids && out, "embed: null pointer");
    TFF_REQUIRE(T >= 0 && H > 0 && V > 0 && H % 8 == 0, "embed: bad sizes T=%d H=%d V=%d", T, H, V);
    if (T == 0) return 0;
    embed_packed_kernel<<<T, 256, 0, (hipStream_t)stream>>>((const bf16_t*)table, ids, out, H, V, (H + 31) / 32);
    return tff_check_launch("embed_packed");
}
