// What the products of four waves a block share: operand types, MFMAs that accumulate in place, copies from global memory
// into LDS by a uniform base, the wait for them by count.
#pragma once
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// s_waitcnt's immediate that waits until at most v copies or loads of the wave are in flight
constexpr int vmcnt_imm(int v) { return (v & 15) | (7 << 4) | (15 << 8) | ((v >> 4) << 14); }
// the same, and until every read of LDS has come back
constexpr int vmcnt_lgkm0_imm(int v) { return (v & 15) | (7 << 4) | ((v >> 4) << 14); }

__device__ __forceinline__ void mfma_acc(floatx4& c, const bf16x8& a, const bf16x8& b) {
    // accumulate in place, in the accumulation registers, as the instruction itself says it: through
    // the builtin the register allocator moves accumulators between the two files around every MFMA
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
// An MFMA and a copy of 16 bytes a lane into LDS at lds_wave_addr + lds_off: M0, which holds the copy's LDS address, is written before the
// MFMA, so that the wait state between that write and the copy is the MFMA, and each of the gaps on its two sides holds one instruction more.
// NT: bytes that nobody asks for again (what that gives: the streaming product's note).
template <bool NT = false>
__device__ __forceinline__ void mfma_acc_copy(floatx4& c, const bf16x8& a, const bf16x8& b, unsigned lds_wave_addr, const unsigned lds_off,
                                              unsigned lane_off, unsigned long long base) {
    if constexpr (NT)
        asm volatile("s_add_u32 m0, %3, %4\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %5, %6 nt"
                     : "+a"(c)
                     : "v"(a), "v"(b), "s"(lds_wave_addr), "i"(lds_off), "v"(lane_off), "s"(base)
                     : "memory", "m0", "scc");
    else
        asm volatile("s_add_u32 m0, %3, %4\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %5, %6"
                     : "+a"(c)
                     : "v"(a), "v"(b), "s"(lds_wave_addr), "i"(lds_off), "v"(lane_off), "s"(base)
                     : "memory", "m0", "scc");
}
// min(x + step, end) and the next place of a ring of END bytes, issued where they stand (the compiler would gather them in one gap)
__device__ __forceinline__ unsigned step_to(unsigned x, const unsigned step, unsigned end) {
    asm volatile("s_add_u32 %0, %0, %1\n\ts_min_u32 %0, %0, %2" : "+s"(x) : "i"(step), "s"(end) : "scc");
    return x;
}
template <unsigned STEP, unsigned END>
__device__ __forceinline__ unsigned ring_next(unsigned x) {
    asm volatile("s_add_u32 %0, %0, %1\n\ts_cmp_eq_u32 %0, %2\n\ts_cselect_b32 %0, 0, %0" : "+s"(x) : "i"(STEP), "i"(END) : "scc");
    return x;
}
template <bool NT = false>
__device__ __forceinline__ void copy16_to_lds_sbase(unsigned long long base, unsigned lane_off, unsigned lds_wave_addr) {
    // the address is a uniform base and a 32-bit offset per lane: walking k is scalar work
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" : : "s"(lds_wave_addr), "v"(lane_off), "s"(base) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_wave_addr), "v"(lane_off), "s"(base) : "memory", "m0");
}

// The lane's index, taken where it is asked for: what the epilogue works out from it is then worked out
// after the main loop, where there are registers for it, instead of before it and kept (or spilled) across.
__device__ __forceinline__ int w4_lane() {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}
