// Device helpers shared by the prefill GEMMs: pair lookup, operand packing and dequantization, the
// LDS swizzle, stage waits and the activation.
#pragma once

#include "brx_internal.h"

namespace brx {

// What the thin-tile GEMM takes from the prefill launcher beside the forward's arguments.
struct ThinArgs {
    const int32_t* order;
    const int32_t* tile_start;
    const int4* tinfo;
    uint16_t* hbuf;
    uint16_t* y_routed;
    uint16_t* y_shared;
    int E_ext, Imax, mt_pad, tile_rows;
};
hipError_t launch_thin(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s);

namespace {

constexpr int kXcd = 8;           // XCDs: block b runs on XCD b % 8

__device__ __forceinline__ int pair_token(const FwdArgs& a, int pair) {
    return pair < a.P ? pair_tok(a, pair) : pair - a.P;
}

__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, bf16x2_t{(__bf16)lo, (__bf16)hi});
}

// native vector (not HIP's uint4 struct, whose copies are memcpys that keep arrays of it in
// scratch memory)
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3_t __attribute__((ext_vector_type(3)));

typedef __attribute__((address_space(3))) void* LDS_PTR;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// swizzle key of A tile row m: 16-byte chunk c of the row sits in slot c ^ a_key(m); rows
// 2t and 2t + 1 share a 256-byte bank row, so keys (m >> 1) & 7 spread 16 consecutive rows
// over 16 distinct bank groups
__device__ __forceinline__ int a_key(int m) { return (m >> 1) & 7; }

// waits for this wave's LDS accesses, then for every wave
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// waits until at most N of this wave's memory loads (copies into LDS and loads into registers)
// are in flight, then for every wave. The wait is the builtin, so the compiler's own wait
// placement knows which loads it covers and adds none for the registers it has made ready;
// the barrier is inline asm with a memory clobber, so no LDS access moves across it.
template <int N>
__device__ __forceinline__ void dma_wait_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
    asm volatile("s_barrier" ::: "memory");
}

// the same wait, and for this wave's LDS reads too: every slot a wave has read is free for new
// copies after the barrier
template <int N>
__device__ __forceinline__ void thin_wait_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | ((N >> 4) << 14));
    asm volatile("s_barrier" ::: "memory");
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// Dequantize piece kk (8 weights, natural K order) of a lane's words `w` into a bf16x8 MFMA
// operand.
//   affine: w = s q + b with one fp32 rounding, then rounded to bf16 (v_cvt_pk_bf16_f32).
//     Each code q is read as the fp16 subnormal q 2^-24 (the code alone in a 16-bit half, exact
//     when widened to fp32: q < 1024) and v_fma_mix_f32 forms fma(q 2^-24, s 2^24, b): the
//     product is exactly s q, so the result is the same fl(s q + b) as fmaf(s, q, b). `s24` is
//     s 2^24 (exact for any scale below 2^104). piece_pair puts codes i and 4 + i in the two
//     halves of one register, so a 4-bit piece costs 7 extractions, 8 fma_mix and 4 packs.
//   MXFP4: the hardware converts two e2m1 codes with the e8m0 scale, exact in bf16.
//   Unquantized bf16 weights are the operand as loaded.
template <int MODE>
__device__ __forceinline__ bf16x8_t dq8(const uint32_t* w, int kk, float s24, float b, float sc) {
    uint32_t o[4];
    if constexpr (kAffine<MODE>) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // codes i (low half) and 4 + i (high half)
            const uint32_t t = piece_pair<kBits<MODE>>(w, kk, i);
            v[i] = __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(t & 0xFFFFu)), s24, b);
            v[4 + i] = __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(t >> 16)), s24, b);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = pk_bf16(v[2 * j], v[2 * j + 1]);
    } else if constexpr (MODE == kModeBf16) {
        // unquantized: the piece is 8 bf16 weights, 4 words in natural K order
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = w[4 * kk + j];
    } else {
        const uint32_t q = w[kk];
        o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 0));
        o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 1));
        o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 2));
        o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 3));
    }
    return __builtin_bit_cast(bf16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
}

// B words a lane holds per stage (half of a row's 64-code stage segment: 32 codes), and the
// loads that bring them in (16-byte loads, plus one 8-byte load for 6 bits; one 8- or 12-byte
// load for 2 and 3 bits; four 16-byte loads for bf16 weights).
template <int MODE>
constexpr int kBW = kBits<MODE>;
template <int MODE>
constexpr int kBLoads = kBits<MODE> == 16 ? 4 : kBits<MODE> >= 6 ? 2 : 1;
// The activation of one output element with the rule fixed at compile time (act_apply's
// arithmetic for that rule, so the same bits).
template <int ACT>
__device__ __forceinline__ float act_fixed(float g, float u, float alpha, float limit) {
    if constexpr (ACT == BRX_ACT_SWIGLU) return silu_mul(g, u);
    else if constexpr (ACT == BRX_ACT_SILU_MLP) return x_sigmoid(g, 1.0f);
    else {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return x_sigmoid(g, alpha) * (u + 1.0f);
    }
}

}  // namespace
}  // namespace brx
