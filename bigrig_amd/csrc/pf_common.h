// Device helpers shared by the prefill GEMMs: pair lookup, operand packing and dequantization, the
// LDS swizzle, stage waits and the activation.
#pragma once

#include "brx_internal.h"

namespace brx {

constexpr int kCus = 256;
constexpr int kDenseRows = 256;   // pairs of the tallest M tile of bf16 experts (k_dense.hip)

// What the thin-tile and bf16 GEMMs take from the prefill launcher beside the forward's arguments.
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
hipError_t launch_dense(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s);   // bf16 weights

namespace {

constexpr int kXcd = 8;           // XCDs: block b runs on XCD b % 8
constexpr int kBM = 128;          // pairs per M tile
constexpr int kBK = 64;           // K step
constexpr int kGemmWaves = 4;
constexpr int kGemmThreads = 64 * kGemmWaves;
constexpr int kNJ = 2;                       // 32-column fragments per wave
constexpr int kWaveN = 32 * kNJ;             // columns per wave
constexpr int kBlockN = kGemmWaves * kWaveN; // columns per block

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

// The 8 affine codes of a chunk into the 4 words of an MFMA operand: c holds them as BITS-bit
// fields (6 bits: codes 0-3 and 4-7 in the low 24 bits of c[0] and c[1]; 8 bits: bytes; fewer: all
// in c[0], whose bits above them are ignored). Every value is fl(s q + b) with one fp32 rounding,
// then rounded to bf16 (v_cvt_pk_bf16_f32): a code field at bit p of a 16-bit half, alone in it and
// below bit 10, reads as the fp16 subnormal q 2^(p - 24), exactly, and meets s 2^(24 - p) in
// v_fma_mix_f32, so the product is exactly s q. `s` is s 2^24 (8 bits: s itself; both exact for any
// scale below 2^104). A 4-bit chunk takes 5 extractions, 8 fma_mix and 4 packs (7 extractions when
// every field was shifted down to bit 0), a 3-bit one 10 (16).
template <int BITS>
__device__ __forceinline__ void dq_affine(const uint32_t* c, float s, float b, uint32_t (&o)[4]) {
    float v[8];
    auto lo = [&](uint32_t t, float sc) __attribute__((always_inline)) {
        return __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(t & 0xFFFFu)), sc, b);
    };
    auto hi = [&](uint32_t t, float sc) __attribute__((always_inline)) {
        return __builtin_fmaf((float)__builtin_bit_cast(_Float16, (uint16_t)(t >> 16)), sc, b);
    };
    if constexpr (BITS == 4) {
        const float s20 = s * 0.0625f;
        const uint32_t u = c[0] >> 8;
        const uint32_t t0 = c[0] & 0x000F000Fu, t1 = c[0] & 0x00F000F0u;
        const uint32_t t2 = u & 0x000F000Fu, t3 = u & 0x00F000F0u;
        v[0] = lo(t0, s); v[4] = hi(t0, s); v[1] = lo(t1, s20); v[5] = hi(t1, s20);
        v[2] = lo(t2, s); v[6] = hi(t2, s); v[3] = lo(t3, s20); v[7] = hi(t3, s20);
    } else if constexpr (BITS == 3) {
        const float s21 = s * 0.125f, s18 = s * 0.015625f;
        const uint32_t r = (c[0] & 0x1FFu) | ((c[0] << 7) & 0x01FF0000u);   // codes 0-2 | 3-5
        const uint32_t t0 = r & 0x00070007u, t1 = r & 0x00380038u, t2 = r & 0x01C001C0u;
        const uint32_t q = c[0] >> 18;
        v[0] = lo(t0, s); v[3] = hi(t0, s); v[1] = lo(t1, s21); v[4] = hi(t1, s21);
        v[2] = lo(t2, s18); v[5] = hi(t2, s18); v[6] = lo(q & 0x7u, s); v[7] = lo(q & 0x38u, s21);
    } else if constexpr (BITS == 2) {
        const float s22 = s * 0.25f, s20 = s * 0.0625f, s18 = s * 0.015625f, s16 = s * 0.00390625f;
        const uint32_t q = c[0] >> 10;
        v[0] = lo(c[0] & 0x3u, s); v[1] = lo(c[0] & 0xCu, s22); v[2] = lo(c[0] & 0x30u, s20);
        v[3] = lo(c[0] & 0xC0u, s18); v[4] = lo(c[0] & 0x300u, s16);
        v[5] = lo(q & 0x3u, s); v[6] = lo(q & 0xCu, s22); v[7] = lo(q & 0x30u, s20);
    } else if constexpr (BITS == 6) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = lo((c[i >> 2] >> (6 * (i & 3))) & 0x3Fu, s);
    } else {
        static_assert(BITS == 8, "affine widths are 2, 3, 4, 6 and 8 bits");
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = __builtin_fmaf((float)((c[i >> 2] >> (8 * (i & 3))) & 0xFFu), s, b);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pk_bf16(v[2 * j], v[2 * j + 1]);
}

// The factor dq_affine's `s` carries.
template <int MODE>
constexpr float kScaleUp = kBits<MODE> == 8 ? 1.0f : 16777216.0f;

// Two e2m1 codes at a time with the e8m0 scale `sc`, exact in bf16 (the hardware's conversion).
__device__ __forceinline__ void dq_fp4(uint32_t q, float sc, uint32_t (&o)[4]) {
    o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 0));
    o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 1));
    o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 2));
    o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q, sc, 3));
}

// Dequantize piece kk (8 weights, natural K order) of a lane's words `w` into a bf16x8 MFMA operand.
template <int MODE>
__device__ __forceinline__ bf16x8_t dq8(const uint32_t* w, int kk, float s, float b) {
    constexpr int B = kBits<MODE>;
    uint32_t o[4];
    if constexpr (kAffine<MODE>) {
        uint32_t c[2];
        if constexpr (B == 8) { c[0] = w[2 * kk]; c[1] = w[2 * kk + 1]; }
        else if constexpr (B == 6) { c[0] = bits_at(w, 48 * kk, 24); c[1] = bits_at(w, 48 * kk + 24, 24); }
        else if constexpr (B == 4) c[0] = w[kk];
        else if constexpr (B == 3) c[0] = bits_at(w, 24 * kk, 24);
        else c[0] = w[kk >> 1] >> (16 * (kk & 1));
        dq_affine<B>(c, s, b, o);
    } else {
        dq_fp4(w[kk], s, o);
    }
    return __builtin_bit_cast(bf16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
}

// B words a lane holds per stage (half of a row's 64-code stage segment: 32 codes), and the
// loads that bring them in (16-byte loads, plus one 8-byte load for 6 bits; one 8- or 12-byte
// load for 2 and 3 bits).
template <int MODE>
constexpr int kBW = kBits<MODE>;
template <int MODE>
constexpr int kBLoads = kBits<MODE> >= 6 ? 2 : 1;
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

// The gate/up epilogue of one activation rule: act(gate + bias, up + bias) (or SiLU(fc1 + bias))
// of every accumulator into the LDS tile T (row stride TS elements), NaN for an absent expert.
// A gated tile's wave holds 32 features: fragment 0 their gate rows, fragment 1 their up rows;
// a two-layer expert's fragment nj holds 32 fc1 features of its own. Element i of a 32 x 32
// fragment is row 8 (i / 4) + 4 kh + i % 4, column l32.
template <int MR, int ACT>
__device__ __forceinline__ void pf_store_h(const FwdArgs& a, const Layout& L, const uint8_t* base, int inter,
                                           bool absent, int nt, const f32x16_t (&acc)[MR][kNJ], uint16_t* T,
                                           int wv, int kh, int l32) {
    const float nan = absent_nan();
    if constexpr (ACT == BRX_ACT_SILU_MLP) {
        constexpr int TS = kBlockN + 8;
#pragma unroll
        for (int nj = 0; nj < kNJ; ++nj) {
            const int fl = nj * 128 + wv * 32 + l32;
            const int f = min(nt * kBlockN + fl, inter - 1);
            const float bg = L.p[0].bias >= 0 ? bf2f(reinterpret_cast<const uint16_t*>(base + L.p[0].bias)[f]) : 0.f;
#pragma unroll
            for (int mi = 0; mi < MR; ++mi) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float h = act_fixed<ACT>(acc[mi][nj][i] + bg, 0.f, a.alpha, a.limit);
                    h = absent ? nan : h;
                    T[(mi * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)) * TS + fl] = __builtin_bit_cast(uint16_t, (__bf16)h);
                }
            }
        }
    } else {
        constexpr int TS = kBlockN / 2 + 8;
        const int fl = wv * (kWaveN / 2) + l32;
        const int f = min(nt * (kBlockN / 2) + fl, inter - 1);
        float bg = 0.f, bu = 0.f;
        if (L.p[0].bias >= 0) {
            bg = bf2f(reinterpret_cast<const uint16_t*>(base + L.p[0].bias)[f]);
            bu = bf2f(reinterpret_cast<const uint16_t*>(base + L.p[1].bias)[f]);
        }
#pragma unroll
        for (int mi = 0; mi < MR; ++mi) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float h = act_fixed<ACT>(acc[mi][0][i] + bg, acc[mi][1][i] + bu, a.alpha, a.limit);
                h = absent ? nan : h;
                T[(mi * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)) * TS + fl] = __builtin_bit_cast(uint16_t, (__bf16)h);
            }
        }
    }
}

// The epilogue of a GEMM tile: MR x kNJ fragments of fp32 accumulators per wave go through LDS
// (`ring`, free once the caller has waited for every copy into it and synchronised) so the
// global stores are 16-byte chunks of contiguous row segments. KIND 0: the activation (one code
// path per rule, chosen once per tile) stored as bf16 h rows at their bucketed positions; KIND 1:
// + bias, each pair's row stored at its (token, k) position (dst_s). An absent expert's h rows
// are NaN.
template <int KIND, int MR>
__device__ __forceinline__ void pf_store(const FwdArgs& a, const Layout& L, const uint8_t* base, bool mlp, int inter,
                                         int slot, int nt, int m0, int rows, const f32x16_t (&acc)[MR][kNJ],
                                         uint8_t* ring, const int32_t* dst_s, uint16_t* __restrict__ hbuf,
                                         int hstride, uint16_t* __restrict__ y_routed,
                                         uint16_t* __restrict__ y_shared) {
    constexpr int MF = MR * 2;
    const int H = a.H;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = lane >> 5, l32 = lane & 31;
    uint16_t* T = reinterpret_cast<uint16_t*>(ring);
    if constexpr (KIND == 0) {
        const bool absent = slot == kAbsentCode;
        if (mlp)
            pf_store_h<MR, BRX_ACT_SILU_MLP>(a, L, base, inter, absent, nt, acc, T, wv, kh, l32);
        else if (a.act == BRX_ACT_SWIGLU_CLAMPED)
            pf_store_h<MR, BRX_ACT_SWIGLU_CLAMPED>(a, L, base, inter, absent, nt, acc, T, wv, kh, l32);
        else
            pf_store_h<MR, BRX_ACT_SWIGLU>(a, L, base, inter, absent, nt, acc, T, wv, kh, l32);
        lds_barrier();
        // a two-layer expert's tile holds kBlockN features, a gated one's kBlockN / 2
        const int fpb = mlp ? kBlockN : kBlockN / 2;
        const int TS = fpb + 8;
        const int CH = fpb / 8;
        for (int c = tid; c < MF * 16 * CH; c += kGemmThreads) {
            const int r = c / CH, f0 = nt * fpb + (c % CH) * 8;
            if (r < rows && f0 < inter)
                *reinterpret_cast<u32x4_t*>(hbuf + (int64_t)(m0 + r) * hstride + f0) =
                    *reinterpret_cast<const u32x4_t*>(T + r * TS + (c % CH) * 8);
        }
    } else {
        constexpr int TS = kBlockN + 8;
        constexpr int CH = kBlockN / 8;
#pragma unroll
        for (int nj = 0; nj < kNJ; ++nj) {
            const int nl = wv * kWaveN + nj * 32 + l32;
            float bd = 0.f;
            if (L.p[2].bias >= 0)
                bd = bf2f(reinterpret_cast<const uint16_t*>(base + L.p[2].bias)[min(nt * kBlockN + nl, H - 1)]);
#pragma unroll
            for (int mi = 0; mi < MR; ++mi) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    T[(mi * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)) * TS + nl] =
                        __builtin_bit_cast(uint16_t, (__bf16)(acc[mi][nj][i] + bd));
            }
        }
        lds_barrier();
        for (int c = tid; c < MF * 16 * CH; c += kGemmThreads) {
            const int r = c / CH, n0 = nt * kBlockN + (c % CH) * 8;
            if (r < rows && n0 < H) {
                const int d = dst_s[r];
                uint16_t* dst = d >= 0 ? y_routed + (int64_t)d * H + n0 : y_shared + (int64_t)(-2 - d) * H + n0;
                *reinterpret_cast<u32x4_t*>(dst) = *reinterpret_cast<const u32x4_t*>(T + r * TS + (c % CH) * 8);
            }
        }
    }
}

}  // namespace
}  // namespace brx
