// Grouped GEMM of thin M tiles (at most 64 of an expert's pairs): batches and short chunks, whose
// experts have few rows each, so the stream of packed weights and its dequantization set the
// time, not the MFMAs.
//
// The contraction is k_pf_gemm's (k_prefill.hip). Its MFMA there is v_mfma_f32_32x32x16_bf16; here
// v_mfma_f32_16x16x32_bf16 does the work of two of those in the same K order, and on gfx950 the
// two give the same bits (the lane groups' 8-element products are added in order either way), so a
// row's value does not depend on which kernel computed it.
//
// One block = 4 waves; a wave owns 16 NC weight rows and up to 64 of the tile's pairs (16 MQ rows,
// MQ chosen by the tile). Against the 256-column blocks of k_pf_gemm this gives a small batch two
// or four times the waves, a tile of at most 16 pairs half the MFMA work, and 3-8 blocks a CU
// (56-108 registers, 26-52 KB of LDS at K 2048) to cover each other's waits. What bounds it: 4-bit
// affine codes the dequantization (about 85 VALU instructions per 1 KB of codes and wave) and, at
// a few blocks per CU, each block's start and end; MXFP4 the weight stream. Layers on one MI355X
// before (k_pf_gemm) and after, whole block: Qwen3 shape, 4-bit, 9 / 32 / 128 tokens 62 / 68 / 105
// -> 47 / 54 / 92 us; gpt-oss shape MXFP4, 32 / 128 / 512 tokens 342 / 478 / 500 -> 270 / 407 / 467
// us (3.64-4.2 TB/s); 256 experts, 8-bit, 301 tokens 250 -> 224 us; bf16, 64 tokens 155 -> 121 us.
//
// Code size matters as much as the loop: every launch starts with a cold instruction cache, and
// the first version (four steps unrolled, the odd stage's code and each activation's epilogue
// written out, 34 KB a kernel against 18) took 111 instead of 94 us for two 9-token layers.
#include <type_traits>

#include "pf_common.h"
#include "stage_addr.h"

namespace brx {
namespace {

constexpr int kTThreads = 64 * kTWaves;
// weight rows per block (16 NC a wave) and floats between rows of the output tile in LDS
template <int NC>
constexpr int kTN = 16 * NC * kTWaves;
template <int NC>
constexpr int kTS = kTN<NC> + 4;

// 64-K stages a step copies and multiplies between two barriers, and steps in the ring. Affine
// codes are bound by their dequantization, and more blocks per CU beat more steps in flight (ring
// of 2 / 3 / 4: 107 / 110 / 125 us for two 32-token layers); MXFP4 streams faster with more (512
// tokens: 532 us with 2, 467 with 3).
template <int MODE>
constexpr int kTSG = kBits<MODE> == 16 ? 1 : 2;
template <int MODE, int MQ>
constexpr int kTNR = kAffine<MODE> ? 2 : MQ == 4 ? 3 : 4;
template <int MODE, int MQ>
constexpr int kTRing = kTNR<MODE, MQ> * kTSG<MODE> * 16 * MQ * 128;

// Bytes of one row of a scale array of K inputs, the bytes between the rows of its table in LDS
// and the table's bytes for `rows` rows (a whole number of 4 KB copies).
struct ThinScales {
    int rowbytes, pitch, bytes;
};
__host__ __device__ inline ThinScales thin_scales(int mode, int K, int gshift, int rows) {
    ThinScales t;
    t.rowbytes = mode == kModeBf16 ? 0 : mode == BRX_QUANT_MXFP4 ? K / 32 : ((K / 64) >> gshift) * 2;
    t.pitch = t.rowbytes % 16 ? t.rowbytes : t.rowbytes + 16;
    t.bytes = t.rowbytes ? (rows * t.pitch + 4095) / 4096 * 4096 : 0;
    return t;
}

// The value of a register pair after the lane halves trade: v0 = (v0 of lanes 0-31, v1 of lanes
// 0-31), v1 = (v0 of lanes 32-63, v1 of lanes 32-63).
__device__ __forceinline__ void swap32(uint32_t& v0, uint32_t& v1) {
    const auto p = __builtin_amdgcn_permlane32_swap(v0, v1, false, false);
    v0 = p[0];
    v1 = p[1];
}

// The same for the 16-lane groups: v0 = (v0 of groups 0 and 2) with v1's of the same two after each,
// v1 = (v0 of groups 1 and 3) with v1's of the same two after each.
__device__ __forceinline__ void swap16(uint32_t& v0, uint32_t& v1) {
    const auto p = __builtin_amdgcn_permlane16_swap(v0, v1, false, false);
    v0 = p[0];
    v1 = p[1];
}

// A lane's codes of one step: chunk (8 codes) j of stage t in c[t][j], as chunk_ops takes them.
template <int MODE>
constexpr int kCW = kBits<MODE> == 16 ? 4 : kBits<MODE> >= 6 ? 2 : 1;   // words a chunk
template <int MODE>
struct Chunks {
    uint32_t c[kTSG<MODE>][2][kCW<MODE>];
};

// The words a lane loads a step: a quarter of its row's 128-code segment (bits words), or, for
// bf16, a chunk of each half of the 64-code stage (chunks 0, 2, 1, 3 of it for lane groups 0 to 3).
template <int MODE>
constexpr int kTW = kBits<MODE> == 16 ? 8 : kBits<MODE>;

// A step's chunks from the quarter q = 2 t + h of the row segment that lane group q loaded: it
// holds chunks 4 h + 2 j + b of stage t, while the MFMA order gives group 2 b + h chunks
// 4 h + 2 j + b of both stages. So the lane halves trade t for b: one v_permlane32_swap a word
// pair. A bf16 lane group holds chunks i and 4 + i of one stage, and groups 2 b and 2 b + 1 trade in
// the same way (v_permlane16_swap): loads of chunks 4 (g & 1) + 2 j + (g >> 1) straight into place
// would read 32 bytes of a row at a time instead of 64.
template <int MODE>
__device__ __forceinline__ void to_chunks(const uint32_t (&w)[kTW<MODE>], Chunks<MODE>& o) {
    constexpr int B = kBits<MODE>;
    if constexpr (B == 16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t a = w[i], b = w[4 + i];
            swap16(a, b);
            o.c[0][0][i] = a;
            o.c[0][1][i] = b;
        }
    } else if constexpr (B == 2) {
        // word j holds chunks b = 0 and 1 in its halves: both lanes of a pair take the word of
        // stage 0's lane and that of stage 1's, and shift their own half down
        const int sh = (threadIdx.x & 32) ? 16 : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t a = w[j], b = w[j];
            swap32(a, b);
            o.c[0][j][0] = a >> sh;
            o.c[1][j][0] = b >> sh;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int i = 0; i < kCW<MODE>; ++i) {
                uint32_t a, b;
                if constexpr (B == 3) {
                    a = bits_at(w, 48 * j, 24);
                    b = bits_at(w, 48 * j + 24, 24);
                } else if constexpr (B == 6) {
                    a = bits_at(w, 96 * j + 24 * i, 24);
                    b = bits_at(w, 96 * j + 48 + 24 * i, 24);
                } else if constexpr (B == 8) {
                    a = w[4 * j + i];
                    b = w[4 * j + 2 + i];
                } else {
                    a = w[2 * j];
                    b = w[2 * j + 1];
                }
                swap32(a, b);
                o.c[0][j][i] = a;
                o.c[1][j][i] = b;
            }
        }
    }
}

// A chunk as an MFMA operand (s: the scale times kScaleUp, or the e8m0 scale).
template <int MODE>
__device__ __forceinline__ bf16x8_t chunk_ops(const uint32_t (&c)[kCW<MODE>], float s, float b) {
    uint32_t o[4];
    if constexpr (kAffine<MODE>) {
        dq_affine<kBits<MODE>>(c, s, b, o);
    } else if constexpr (MODE == kModeBf16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = c[i];
    } else {
        dq_fp4(c[0], s, o);
    }
    return __builtin_bit_cast(bf16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
}

template <int MODE, bool F16, int KIND, int NC, int MQ>
__device__ __forceinline__ void thin_tile(const FwdArgs& a, const int32_t* __restrict__ order,
                                          uint16_t* __restrict__ hbuf, int hstride,
                                          uint16_t* __restrict__ y_routed, uint16_t* __restrict__ y_shared,
                                          uint8_t* smem, int ring_bytes, int32_t* dst_s, int e, int m0, int rows,
                                          int slot, int nt) {
    constexpr int B = kBits<MODE>;
    constexpr int TN = kTN<NC>, TS = kTS<NC>;
    constexpr int SG = kTSG<MODE>, NR = kTNR<MODE, MQ>;
    constexpr int SAst = 16 * MQ * 128;            // A bytes of a stage
    constexpr int SA = SG * SAst;                  // ... of a step
    constexpr int NA = kTAWave<SG, MQ>;            // 1 KB A copies of a wave and step
    constexpr int LPC = B == 16 || B == 6 || B == 8 ? 2 : 1;   // loads per column fragment and step
    constexpr int NV = NA + NC * LPC;
    const bool sh = e >= a.E;
    const int inter = sh ? a.I_sh : a.I;
    const int H = a.H;
    const int K = KIND == 0 ? H : inter;
    const int nst = K / 64;                        // stages
    const int nsteps = (nst + SG - 1) / SG;
    const Layout& L = sh ? a.lay_sh : a.lay;
    const uint8_t* base = sh ? a.shared : code_base(a, clamp_code(a, slot));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const bool mlp = KIND == 0 && a.act == BRX_ACT_SILU_MLP;

    // ---- A rows of this wave's copies: the pair list is read first, the first steps' B is
    // requested under it
    const uint32_t a_bytes = KIND == 0 ? (uint32_t)((int64_t)a.T * H * 2)
                                       : (uint32_t)((int64_t)(m0 + rows) * hstride * 2);
    int pr[NA];
    if constexpr (KIND == 0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int rl = thin_a_row<SG, MQ>(wv, i, lane);
            pr[i] = order[m0 + min(rl, rows - 1)];
        }
    }
    // ---- B: wave wv owns the block's weight rows 16 NC wv + 16 n + l16; lane group g loads quarter
    // g of a row's step segment, so an instruction reads 16 rows x 8 B bytes or more in a row
    auto mat_row = [&](int br) __attribute__((always_inline)) {
        return KIND == 0 ? (mlp ? min(nt * TN + br, inter - 1) : nt * (TN / 2) + (br & (TN / 2 - 1)))
                         : min(nt * TN + br, H - 1);
    };
    const int pj = KIND == 0 ? (mlp || wv < kTWaves / 2 ? 0 : 1) : 2;
    const int br0 = wv * 16 * NC + l16;
    uint32_t vbw[NC];
#pragma unroll
    for (int n = 0; n < NC; ++n)
        vbw[n] = thin_b_lane(B, K, (uint32_t)mat_row(br0 + 16 * n), g);
    const uint32_t wbase = (uint32_t)L.p[pj].w;
    struct BReg {
        uint32_t w[NC][kTW<MODE>];
    };
    // Steps past the last are issued like the others, through a descriptor of no bytes (the range
    // check answers without memory traffic): every wait below then counts the same loads, also
    // the compiler's own for the B registers, which would drain the counter after a guarded load.
    // An odd last stage's step reads on past the row, into the next row or the matrix's scales.
    auto issue_b = [&](int p, BReg& r) __attribute__((always_inline)) {
        const StageSrc src = stage_src(p, nsteps, (uint32_t)L.bytes, wbase + thin_b_step(B, SG, p));
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(base, src.records);
        const uint32_t go = src.soffset;
#pragma unroll
        for (int n = 0; n < NC; ++n) {
            uint32_t* q = r.w[n];
            if constexpr (B == 2) {
                const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rb, vbw[n], go, 0);
                q[0] = v[0]; q[1] = v[1];
            } else if constexpr (B == 3) {
                const u32x3_t v = __builtin_amdgcn_raw_buffer_load_b96(rb, vbw[n], go, 0);
                q[0] = v[0]; q[1] = v[1]; q[2] = v[2];
            } else {
#pragma unroll
                for (int l = 0; l < kTW<MODE> / 4; ++l) {
                    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rb, vbw[n] + (B == 16 ? 64 : 16) * l, go, 0);
                    q[4 * l] = v[0]; q[4 * l + 1] = v[1]; q[4 * l + 2] = v[2]; q[4 * l + 3] = v[3];
                }
                if constexpr (B == 6) {
                    const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rb, vbw[n] + 16, go, 0);
                    q[4] = v[0]; q[5] = v[1];
                }
            }
        }
    };
    BReg bq[NR];
#pragma unroll
    for (int t = 0; t < NR - 1; ++t) issue_b(t, bq[t]);

    // ---- scales (and biases): the block's rows of each array, copied once. Rows of the arrays
    // are contiguous, so a copy instruction reads 1 KB in a row; rows that are a multiple of 16
    // bytes get 16 bytes of padding in LDS, the others keep their odd pitch, so that a stage's
    // reads down the rows spread over the banks.
    const ThinScales ts = thin_scales(MODE, K, kAffine<MODE> ? a.gshift : 0, TN);
    uint8_t* const tbl = smem + ring_bytes;
    if constexpr (kScaled<MODE>) {
        const __amdgpu_buffer_rsrc_t rb_rsrc = make_rsrc(base, (uint32_t)L.bytes);
        const int plo = KIND == 0 ? 0 : 2, phi = KIND == 0 ? (mlp ? 0 : 1) : 2;
        const uint32_t s_lo = (uint32_t)L.p[plo].s, s_hi = (uint32_t)L.p[phi].s;
        const uint32_t b_lo = (uint32_t)L.p[plo].b, b_hi = (uint32_t)L.p[phi].b;
        const bool split = KIND == 0 && !mlp;      // gate rows, then up rows
        const int rb = ts.rowbytes, row0 = nt * (split ? TN / 2 : TN);
        const bool pad = ts.pitch != rb;
#pragma unroll 1
        for (int c = 0; c * 4096 < ts.bytes; ++c) {
            const int q = c * kTThreads + tid;
            int r, in;                              // row of the block, byte in it (image: from row 0)
            if (pad) {
                r = q / (rb / 16 + 1);
                in = min((q - r * (rb / 16 + 1)) * 16, rb - 16);
            } else {
                r = q * 16 >= (TN / 2) * rb ? TN / 2 : 0;
                in = q * 16 - r * rb;
            }
            const bool up = r >= TN / 2;
            const uint32_t vo = (uint32_t)((row0 + (split && up ? r - TN / 2 : r)) * rb + in);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb_rsrc, (LDS_PTR)(tbl + c * 4096 + wv * 1024), 16,
                                                     vo + (up ? s_hi : s_lo), 0, 0, 0);
            if constexpr (kAffine<MODE>)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rb_rsrc, (LDS_PTR)(tbl + ts.bytes + c * 4096 + wv * 1024),
                                                         16, vo + (up ? b_hi : b_lo), 0, 0, 0);
        }
        asm volatile("" ::: "memory");
    }
    uint32_t va[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int rl = thin_a_row<SG, MQ>(wv, i, lane);
        const uint32_t row = KIND == 0 ? (uint32_t)pair_token(a, pr[i]) * (uint32_t)(H * 2)
                                       : (uint32_t)(m0 + min(rl, rows - 1)) * (uint32_t)(hstride * 2);
        // rows past the tile's pairs: from past the buffer's end (zeros, no cache access)
        va[i] = a_lane_offset(rl, rows, row, (lane & 7) ^ a_key(rl), a_bytes);
    }
    if constexpr (KIND == 1) {
        if (tid < 16 * MQ) {
            int d = -1;
            if (tid < rows) {
                const int pair = order[m0 + tid];
                d = pair < a.P ? pair_row(a, pair) : -2 - (pair - a.P);
            }
            dst_s[tid] = d;
        }
    }
    auto issue_a = [&](int p) __attribute__((always_inline)) {
        uint8_t* st = smem + (p % NR) * SA;
        const int q = p * SG + thin_a_stage<SG, MQ>(wv);
        const StageSrc src = stage_src(q, nst, a_bytes, (uint32_t)q * 128u);
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(KIND == 0 ? (const void*)a.x : (const void*)hbuf, src.records);
#pragma unroll
        for (int i = 0; i < NA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR)(st + thin_a_copy<SG, MQ>(wv, i) * 1024), 16, va[i],
                                                     src.soffset, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < NR - 1; ++t) issue_a(t);
    // the first NR - 1 steps land together (their B was requested before the pair list was
    // read), so the counted waits of the loop start at step NR - 1
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)

    f32x4_t acc[MQ][NC];
#pragma unroll
    for (int i = 0; i < MQ; ++i)
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][n][r] = 0.f;

    // the lane's A operand addresses: chunk 4 (g & 1) + 2 j + (g >> 1) of row l16 (+ 16 m) of a stage
    // (rows 16 apart share a swizzle key)
    uint32_t ax[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
        ax[j] = (uint32_t)(l16 * 128 + ((4 * (g & 1) + 2 * j + (g >> 1)) ^ a_key(l16)) * 16);
    const uint8_t* const srow = tbl + br0 * ts.pitch;
    const int gs = kAffine<MODE> ? a.gshift : 0;

    auto step = [&](int p, const BReg& r, int slotp) __attribute__((always_inline)) {
        Chunks<MODE> ch[NC];
#pragma unroll
        for (int n = 0; n < NC; ++n) to_chunks<MODE>(r.w[n], ch[n]);
#pragma unroll
        for (int t = 0; t < SG; ++t) {
            const int s = p * SG + t;
            if (s >= nst) break;      // uniform: an odd last stage, or a step past the end
            float sv[NC], bv[NC];
#pragma unroll
            for (int n = 0; n < NC; ++n) {
                sv[n] = bv[n] = 0.f;
                const uint8_t* sr = srow + 16 * n * ts.pitch;
                if constexpr (kAffine<MODE>) {
                    const uint32_t s16 = *reinterpret_cast<const uint16_t*>(sr + 2 * (s >> gs));
                    const uint32_t b16 = *reinterpret_cast<const uint16_t*>(sr + ts.bytes + 2 * (s >> gs));
                    sv[n] = (F16 ? h2f(s16) : bf2f(s16)) * kScaleUp<MODE>;
                    bv[n] = F16 ? h2f(b16) : bf2f(b16);
                } else if constexpr (kScaled<MODE>) {
                    const uint32_t s16 = *reinterpret_cast<const uint16_t*>(sr + 2 * s);
                    sv[n] = e8m0_f32((s16 >> (8 * (g & 1))) & 0xFFu);
                }
            }
            const uint8_t* As = smem + slotp * SA + t * SAst;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                bf16x8_t af[MQ];
#pragma unroll
                for (int m = 0; m < MQ; ++m) af[m] = *reinterpret_cast<const bf16x8_t*>(As + m * 2048 + ax[j]);
#pragma unroll
                for (int n = 0; n < NC; ++n) {
                    const bf16x8_t bop = chunk_ops<MODE>(ch[n].c[t][j], sv[n], bv[n]);
#pragma unroll
                    for (int m = 0; m < MQ; ++m)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[m], bop, acc[m][n], 0, 0, 0);
                }
            }
        }
    };

    for (int p0 = 0; p0 < nsteps; p0 += NR) {
#pragma unroll
        for (int v = 0; v < NR; ++v) {
            // (the last round's steps past the end only keep the loads' count; a break here would
            // give the loop paths on which the compiler must drain the counter)
            const int p = p0 + v;
            // step p landed in every wave (the NR - 2 steps issued after it may be in flight), and
            // every wave is done reading step p - 1, whose ring slot and registers step p + NR - 1
            // takes
            thin_wait_barrier<(NR - 2) * NV>();
            issue_b(p + NR - 1, bq[(v + NR - 1) % NR]);
            issue_a(p + NR - 1);
            asm volatile("" ::: "memory");
            step(p, bq[v], v);
        }
    }

    // ---- epilogue: the fp32 tile through LDS, so one thread has a gate and its up value and
    // stores 8 consecutive outputs of a row
    thin_wait_barrier<0>();
    float* T = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int m = 0; m < MQ; ++m)
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) T[(m * 16 + 4 * g + i) * TS + br0 + 16 * n] = acc[m][n][i];
    lds_barrier();
    auto load8 = [&](const float* t, int64_t boff, float (&o)[8]) __attribute__((always_inline)) {
        const f32x4_t v0 = *reinterpret_cast<const f32x4_t*>(t), v1 = *reinterpret_cast<const f32x4_t*>(t + 4);
        u32x4_t bw{0u, 0u, 0u, 0u};
        if (boff >= 0) bw = *reinterpret_cast<const u32x4_t*>(base + boff);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t b16 = (j & 1) ? bw[j >> 1] >> 16 : bw[j >> 1] & 0xFFFFu;
            o[j] = (j < 4 ? v0[j & 3] : v1[j & 3]) + bf2f(b16);
        }
    };
    auto store8 = [&](uint16_t* dst, const float (&o)[8]) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4_t*>(dst) =
            u32x4_t{pk_bf16(o[0], o[1]), pk_bf16(o[2], o[3]), pk_bf16(o[4], o[5]), pk_bf16(o[6], o[7])};
    };
    auto bias_at = [&](int p, int row) { return L.p[p].bias >= 0 ? (int64_t)L.p[p].bias + 2 * row : (int64_t)-1; };
    if constexpr (KIND == 0) {
        const bool absent = slot == kAbsentCode;
        const float nan = absent_nan();
        const bool clamped = a.act == BRX_ACT_SWIGLU_CLAMPED;
        const float alpha = clamped ? a.alpha : 1.0f;
        const int CH = mlp ? TN / 8 : TN / 16;    // 8-feature chunks a row
#pragma unroll 1
        for (int c = tid; c < 16 * MQ * CH; c += kTThreads) {
            const int r = c / CH, fl = (c % CH) * 8, f0 = nt * CH * 8 + fl;
            if (r >= rows || f0 >= inter) continue;
            float gv[8], u[8], h[8];
            load8(T + r * TS + fl, bias_at(0, f0), gv);
            load8(T + r * TS + (mlp ? 0 : TN / 2) + fl, mlp ? (int64_t)-1 : bias_at(1, f0), u);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                // act_fixed's arithmetic with the rule picked by selects: one copy of the code
                const float gc = clamped ? fminf(gv[j], a.limit) : gv[j];
                const float uc = mlp ? 1.0f : clamped ? fminf(fmaxf(u[j], -a.limit), a.limit) + 1.0f : u[j];
                h[j] = x_sigmoid(gc, alpha) * uc;
                h[j] = absent ? nan : h[j];
            }
            store8(hbuf + (int64_t)(m0 + r) * hstride + f0, h);
        }
    } else {
#pragma unroll 1
        for (int c = tid; c < 16 * MQ * (TN / 8); c += kTThreads) {
            const int r = c / (TN / 8), nl = (c % (TN / 8)) * 8, n0 = nt * TN + nl;
            if (r >= rows || n0 >= H) continue;
            float o[8];
            load8(T + r * TS + nl, bias_at(2, n0), o);
            const int d = dst_s[r];
            store8(d >= 0 ? y_routed + (int64_t)d * H + n0 : y_shared + (int64_t)(-2 - d) * H + n0, o);
        }
    }
}

template <int MODE, bool F16, int KIND, int NC>
__global__ __launch_bounds__(kTThreads) __attribute__((amdgpu_waves_per_eu(NC == 1 ? 4 : 3)))
void k_thin_gemm(FwdArgs a, const int32_t* __restrict__ order, const int32_t* __restrict__ tile_start,
                 const int4* __restrict__ tinfo, int E_ext, int ntn, uint16_t* __restrict__ hbuf, int hstride,
                 uint16_t* __restrict__ y_routed, uint16_t* __restrict__ y_shared, int ring_bytes) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ int32_t dst_s[KIND == 1 ? 64 : 1];
    prefetch_args(a);
    const int blk = blockIdx.x;
    const int loc = blk / kXcd;
    const int nt = loc % ntn;
    const int mt = (loc / ntn) * kXcd + blk % kXcd;
    const int total = tile_start[E_ext];
    const int4 ti = tinfo[mt];
    if (mt >= total) return;
    const int e = ti.x, m0 = ti.y, rows = ti.z;
    if (KIND == 0) {
        const int inter = e >= a.E ? a.I_sh : a.I;
        if (nt * (a.act == BRX_ACT_SILU_MLP ? kTN<NC> : kTN<NC> / 2) >= inter) return;
    } else {
        if (nt * kTN<NC> >= a.H) return;
    }
#define BRX_TILE(MQ) \
    thin_tile<MODE, F16, KIND, NC, MQ>(a, order, hbuf, hstride, y_routed, y_shared, smem, ring_bytes, dst_s, e, m0, rows, ti.w, nt)
    if (rows <= 16) BRX_TILE(1);
    else if (rows <= 32) BRX_TILE(2);
    else BRX_TILE(4);
#undef BRX_TILE
}

// The ring's bytes and the launch's whole LDS for M tiles of at most `tile_rows`.
template <int MODE>
int thin_ring(int tile_rows) {
    int r = kTRing<MODE, 1>;
    if (tile_rows > 16 && kTRing<MODE, 2> > r) r = kTRing<MODE, 2>;
    if (tile_rows > 32 && kTRing<MODE, 4> > r) r = kTRing<MODE, 4>;
    return r;
}
template <int MODE, int NC>
int thin_lds(const FwdArgs& a, int K, int tile_rows) {
    const int tile = (tile_rows > 32 ? 64 : tile_rows > 16 ? 32 : 16) * kTS<NC> * 4;
    const int all = thin_ring<MODE>(tile_rows) + (kAffine<MODE> ? 2 : 1) * thin_scales(MODE, K, a.gshift, kTN<NC>).bytes;
    return all > tile ? all : tile;
}

template <int MODE, bool F16, int NC>
hipError_t launch_nc(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s) {
    if (phases & 1) {
        const int fpb = a.act == BRX_ACT_SILU_MLP ? kTN<NC> : kTN<NC> / 2;
        const int ntn = (t.Imax + fpb - 1) / fpb;
        hipLaunchKernelGGL((k_thin_gemm<MODE, F16, 0, NC>), dim3(t.mt_pad * ntn), dim3(kTThreads),
                           (thin_lds<MODE, NC>(a, a.H, t.tile_rows)), s, a, t.order, t.tile_start, t.tinfo, t.E_ext, ntn,
                           t.hbuf, t.Imax, t.y_routed, t.y_shared, thin_ring<MODE>(t.tile_rows));
        hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (phases & 2) {
        const int ntn = (a.H + kTN<NC> - 1) / kTN<NC>;
        hipLaunchKernelGGL((k_thin_gemm<MODE, F16, 1, NC>), dim3(t.mt_pad * ntn), dim3(kTThreads),
                           (thin_lds<MODE, NC>(a, t.Imax, t.tile_rows)), s, a, t.order, t.tile_start, t.tinfo, t.E_ext, ntn,
                           t.hbuf, t.Imax, t.y_routed, t.y_shared, thin_ring<MODE>(t.tile_rows));
        return hipGetLastError();
    }
    return hipSuccess;
}

template <int MODE, bool F16>
hipError_t launch_mode(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s) {
    // 64-row blocks while they are what fills the chip: at most that many 128-row blocks if every
    // pair (or every expert) has a tile of its own, and few pairs an expert (two 9-token layers 94
    // against 100 us, 32 tokens 107 / 111, 64 tokens equal); past that 128-row blocks share each A
    // tile among twice the columns (301 tokens of 8-bit experts 239 -> 224 us, 512 tokens of MXFP4
    // 535 -> 467).
    const int tiles = a.P < t.E_ext ? a.P : t.E_ext;
    const bool small = tiles * ((t.Imax + 63) / 64) <= 1600 && a.P <= 4 * t.E_ext;
    return small ? launch_nc<MODE, F16, 1>(a, t, phases, s) : launch_nc<MODE, F16, 2>(a, t, phases, s);
}

}  // namespace

hipError_t launch_thin(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s) {
#define BRX_THIN(M) (a.scale_f16 ? launch_mode<M, true>(a, t, phases, s) : launch_mode<M, false>(a, t, phases, s))
    switch (a.quant_mode) {
        case kModeAffine4: return BRX_THIN(kModeAffine4);
        case kModeAffine3: return BRX_THIN(kModeAffine3);
        case kModeAffine2: return BRX_THIN(kModeAffine2);
        case kModeAffine6: return BRX_THIN(kModeAffine6);
        case kModeAffine8: return BRX_THIN(kModeAffine8);
        case BRX_QUANT_MXFP4: return launch_mode<BRX_QUANT_MXFP4, false>(a, t, phases, s);
        case kModeBf16: return launch_mode<kModeBf16, false>(a, t, phases, s);
        default: return hipErrorInvalidValue;
    }
#undef BRX_THIN
}

}  // namespace brx
