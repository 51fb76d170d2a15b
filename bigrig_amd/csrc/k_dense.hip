// Grouped GEMM of unquantized bf16 experts (chunks; batches and short chunks go to k_thin.hip).
//
// One block = 8 waves, one block a CU; tile = 256, 128, 64 or 32 of an expert's pairs (the tallest a call
// cuts: tile_rows in k_prefill.hip) x 256 weight rows (KIND 0: the gate and up rows of 128 features). Wave (wm, wn) owns 32 MR pairs and 64 weight
// rows, so at MR 4 a 16-K step reads 4 A and 2 B fragments from LDS for 8 v_mfma_f32_32x32x16_bf16
// (96 of the 128 bytes a clock LDS gives at the full MFMA rate). There is nothing to dequantize, so
// both operands are copied straight into LDS by the buffer unit in 64-K stages: whole 128-byte lines
// (32-K stages, half a line at a time, took 389 + 273 us where these take 355 + 253: each line
// crossed from L2 twice). A 64-K stage is summed in the order of the other grouped GEMMs, chunks kk and
// 4 + kk (8 K each) in MFMA kk, so a row has the same bits from this kernel and from k_thin.hip, and
// those its exactly representable quantized weights give; the operands come from LDS, where any
// order costs the same.
//
// Bound (4096 tokens of the Qwen3 shape, gate/up 355 us, of which the MFMAs alone are 117, the copies
// alone 182 and a tile's start, barriers and epilogue 123): the copies, then the start and end of a
// tile, which one block a CU does not hide. Shorter tiles at two blocks a CU hide them but copy twice
// the bytes (128 rows, 32-K stages: 371 + 255 us). The general kernel's 64-row tiles, whose lanes
// loaded their own B operands, took 567 + 306.
#include "pf_common.h"
#include "stage_addr.h"

namespace brx {
namespace {

constexpr int kDThreads = 512;
// M tiles in a row of the list an XCD takes before the next XCD's: the tiles of one expert then share
// its weights in that XCD's L2 (1 / 2 / 4 / 8, 4096 tokens: 657 / 645 / 646 / 659 us a layer)
constexpr int kDRun = 2;
constexpr int kDM = kDenseRows;               // pairs of the tallest tile
constexpr int kDB = kBlockN * 128;            // B bytes of a stage
constexpr int kDTile = kDM * (kBlockN + 8) * 2;   // the widest output tile
template <int MR, int WM>
constexpr int kDStage = 32 * MR * WM * 128 + kDB;
template <int MR>
constexpr int kDNS = MR == 4 ? 2 : 3;         // ring stages
constexpr int kDLds = kDNS<2> * kDStage<2, 2> > kDTile ? kDNS<2> * kDStage<2, 2> : kDTile;
static_assert(kDNS<4> * kDStage<4, 2> <= kDLds, "the ring fits the block's LDS");

// Tile of up to 32 MR WM pairs; with WM 1 the waves of wm 1 only copy.
template <int KIND, int MR, int WM>
__device__ __forceinline__ void dense_tile(const FwdArgs& a, const int32_t* __restrict__ order,
                                           uint16_t* __restrict__ hbuf, int hstride, uint16_t* __restrict__ y_routed,
                                           uint16_t* __restrict__ y_shared, uint8_t* ring, int32_t* dst_s, int e, int m0,
                                           int rows, int slot, int nt) {
    constexpr int NS = kDNS<MR>, STAGE = kDStage<MR, WM>;
    constexpr int TR = 32 * MR * WM;                             // rows of the tile
    constexpr int kWaves = kDThreads / 64;
    constexpr int NAC = TR / 8;                                  // 1 KB A copies a stage, NA of them a wave
    constexpr int NA = (NAC + kWaves - 1) / kWaves;
    constexpr int NB = 4;                                        // B copies of a wave: 32 rows
    constexpr int NV = NA + NB;
    const bool sh = e >= a.E;
    const int inter = sh ? a.I_sh : a.I;
    const int H = a.H;
    const int K = KIND == 0 ? H : inter;
    const int nst = K / 64;
    const Layout& L = sh ? a.lay_sh : a.lay;
    const uint8_t* base = sh ? a.shared : code_base(a, clamp_code(a, slot));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv >> 2, wn = wv & 3;
    const int kh = lane >> 5, l32 = lane & 31;
    const bool mlp = KIND == 0 && a.act == BRX_ACT_SILU_MLP;

    // ---- A: copy i of this wave (past the last copy of a low tile: repeated) fills 8 rows; lane l
    // carries chunk (l % 8) ^ key of row l / 8. Rows past the tile's pairs come from past the
    // buffer's end (zeros, no cache access).
    const uint32_t a_bytes = KIND == 0 ? (uint32_t)((int64_t)a.T * H * 2)
                                       : (uint32_t)((int64_t)(m0 + rows) * hstride * 2);
    auto copy_of = [&](int i) __attribute__((always_inline)) { return min(wv * NA + i, NAC - 1); };
    uint32_t va[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int rl = copy_of(i) * 8 + (lane >> 3), r = min(rl, rows - 1);
        const uint32_t row = KIND == 0 ? (uint32_t)pair_token(a, order[m0 + r]) * (uint32_t)(H * 2)
                                       : (uint32_t)(m0 + r) * (uint32_t)(hstride * 2);
        va[i] = a_lane_offset(rl, rows, row, (lane & 7) ^ a_key(rl), a_bytes);
    }
    // ---- B: LDS row 64 n + 32 j + q is column q of fragment j of the waves wn = n. KIND 0: fragment
    // 0 is 32 gate rows (nt * 128 + 32 n + q), fragment 1 the same features' up rows; a two-layer
    // expert's fragment j holds fc1 rows nt * 256 + 128 j + 32 n + q; KIND 1: rows in order.
    uint32_t vb[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int lr = wv * 32 + i * 8 + (lane >> 3);
        const int c = (lane & 7) ^ a_key(lr);
        const int n = lr >> 6, j = (lr >> 5) & 1, q = lr & 31;
        const int row = KIND == 0 ? (mlp ? min(nt * 256 + 128 * j + 32 * n + q, inter - 1)
                                         : min(nt * 128 + 32 * n + q, inter - 1))
                                  : min(nt * 256 + lr, H - 1);
        const uint32_t w = (uint32_t)(KIND == 1 ? L.p[2].w : (j == 1 && !mlp) ? L.p[1].w : L.p[0].w);
        vb[i] = w + (uint32_t)row * (uint32_t)(K * 2) + c * 16;
    }
    if constexpr (KIND == 1) {
        if (tid < TR) {
            int d = -1;
            if (tid < rows) {
                const int pair = order[m0 + tid];
                d = pair < a.P ? pair_row(a, pair) : -2 - (pair - a.P);
            }
            dst_s[tid] = d;
        }
    }
    // a stage past the last is issued through descriptors of no bytes, so the waits count the same
    // copies throughout
    auto issue = [&](int s, int at) __attribute__((always_inline)) {
        const StageSrc sa = stage_src(s, nst, a_bytes, (uint32_t)s * 128u);
        const StageSrc sb = stage_src(s, nst, (uint32_t)L.bytes, (uint32_t)s * 128u);
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(KIND == 0 ? (const void*)a.x : (const void*)hbuf, sa.records);
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(base, sb.records);
        uint8_t* st = ring + at * STAGE;
#pragma unroll
        for (int i = 0; i < NB; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (LDS_PTR)(st + (wv * NB + i) * 1024), 16, vb[i], sb.soffset, 0, 0);
#pragma unroll
        for (int i = 0; i < NA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (LDS_PTR)(st + kDB + copy_of(i) * 1024), 16, va[i], sa.soffset, 0, 0);
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) issue(s, s);

    f32x16_t acc[MR][kNJ];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int j = 0; j < kNJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // operand addresses of MFMA kk: chunk 4 kh + kk of row l32 (+ 32 m: the same key)
    uint32_t ad[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) ad[kk] = (uint32_t)(l32 * 128 + (((4 * kh + kk) ^ a_key(l32)) << 4));
    const bool active = wm < WM;   // uniform

    int at = 0, next = NS - 1;
    for (int s = 0; s < nst; ++s) {
        // stage s landed in every wave, and stage s - 1's slot is free for stage s + NS - 1
        thin_wait_barrier<(NS - 2) * NV>();
        issue(s + NS - 1, next);
        const uint8_t* Bs = ring + at * STAGE + wn * 8192;
        const uint8_t* As = ring + at * STAGE + kDB + wm * (MR * 4096);
        if (active) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                bf16x8_t af[MR], bf[kNJ];
#pragma unroll
                for (int j = 0; j < kNJ; ++j) bf[j] = *reinterpret_cast<const bf16x8_t*>(Bs + j * 4096 + ad[kk]);
#pragma unroll
                for (int m = 0; m < MR; ++m) af[m] = *reinterpret_cast<const bf16x8_t*>(As + m * 4096 + ad[kk]);
#pragma unroll
                for (int m = 0; m < MR; ++m)
#pragma unroll
                    for (int j = 0; j < kNJ; ++j)
                        acc[m][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[m], bf[j], acc[m][j], 0, 0, 0);
            }
        }
        at = at + 1 == NS ? 0 : at + 1;
        next = next + 1 == NS ? 0 : next + 1;
    }
    thin_wait_barrier<0>();

    // ---- epilogue: the bf16 tile through LDS, then 16-byte stores of row segments. Element i of a
    // fragment is row 8 (i / 4) + 4 kh + i % 4, column l32.
    uint16_t* T = reinterpret_cast<uint16_t*>(ring);
    const bool gated = KIND == 0 && !mlp;
    const int cols = gated ? kBlockN / 2 : kBlockN, TS = cols + 8;
    const int n_all = KIND == 0 ? inter : H;
    auto bias = [&](int p, int row) __attribute__((always_inline)) {
        return L.p[p].bias >= 0 ? bf2f(reinterpret_cast<const uint16_t*>(base + L.p[p].bias)[min(row, n_all - 1)]) : 0.f;
    };
    if (active) {
        const float nan = absent_nan();
        const bool absent = slot == kAbsentCode, clamped = a.act == BRX_ACT_SWIGLU_CLAMPED;
        const float alpha = clamped ? a.alpha : 1.0f;
        // columns of the tile (and their biases) fragment j of this wave fills
        const int c0 = gated ? wn * 32 + l32 : mlp ? wn * 32 + l32 : wn * 64 + l32, c1 = mlp ? c0 + 128 : c0 + 32;
        const float b0 = bias(KIND == 0 ? 0 : 2, nt * cols + c0);
        const float b1 = gated ? bias(1, nt * cols + c0) : bias(KIND == 0 ? 0 : 2, nt * cols + c1);
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                uint16_t* t = T + ((wm * MR + m) * 32 + 8 * (i >> 2) + 4 * kh + (i & 3)) * TS;
                const float v0 = acc[m][0][i] + b0, v1 = acc[m][1][i] + b1;
                if constexpr (KIND == 0) {
                    // act_fixed's arithmetic with the rule picked by selects: one copy of the code
                    if (gated) {
                        const float gc = clamped ? fminf(v0, a.limit) : v0;
                        const float uc = clamped ? fminf(fmaxf(v1, -a.limit), a.limit) + 1.0f : v1;
                        const float h = x_sigmoid(gc, alpha) * uc;
                        t[c0] = __builtin_bit_cast(uint16_t, (__bf16)(absent ? nan : h));
                    } else {
                        t[c0] = __builtin_bit_cast(uint16_t, (__bf16)(absent ? nan : x_sigmoid(v0, 1.0f)));
                        t[c1] = __builtin_bit_cast(uint16_t, (__bf16)(absent ? nan : x_sigmoid(v1, 1.0f)));
                    }
                } else {
                    t[c0] = __builtin_bit_cast(uint16_t, (__bf16)v0);
                    t[c1] = __builtin_bit_cast(uint16_t, (__bf16)v1);
                }
            }
    }
    lds_barrier();
    const int CH = cols / 8;
#pragma unroll 1
    for (int c = tid; c < TR * CH; c += kDThreads) {
        const int r = c / CH, cl = (c % CH) * 8, n0 = nt * cols + cl;
        if (r >= rows || n0 >= n_all) continue;
        uint16_t* dst;
        if constexpr (KIND == 0) {
            dst = hbuf + (int64_t)(m0 + r) * hstride + n0;
        } else {
            const int d = dst_s[r];
            dst = d >= 0 ? y_routed + (int64_t)d * H + n0 : y_shared + (int64_t)(-2 - d) * H + n0;
        }
        *reinterpret_cast<u32x4_t*>(dst) = *reinterpret_cast<const u32x4_t*>(T + r * TS + cl);
    }
}

template <int KIND>
__global__ __launch_bounds__(kDThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_dense_gemm(FwdArgs a, const int32_t* __restrict__ order, const int32_t* __restrict__ tile_start,
                  const int4* __restrict__ tinfo, int E_ext, int ntn, int mt_pad, uint16_t* __restrict__ hbuf,
                  int hstride, uint16_t* __restrict__ y_routed, uint16_t* __restrict__ y_shared) {
    __shared__ __attribute__((aligned(16))) uint8_t ring[kDLds];
    __shared__ int32_t dst_s[KIND == 1 ? kDM : 1];
    prefetch_args(a);
    // an XCD takes every column tile of a run of M tiles before its next run
    const int loc = blockIdx.x / kXcd;
    const int nt = (loc / kDRun) % ntn;
    const int mt = (loc / (kDRun * ntn) * kXcd + blockIdx.x % kXcd) * kDRun + loc % kDRun;
    const int total = tile_start[E_ext];
    const int4 ti = tinfo[min(mt, mt_pad - 1)];
    if (mt >= total) return;
    const int e = ti.x, m0 = ti.y, rows = ti.z;
    if (KIND == 0) {
        const int inter = e >= a.E ? a.I_sh : a.I;
        if (nt * (a.act == BRX_ACT_SILU_MLP ? kBlockN : kBlockN / 2) >= inter) return;
    } else {
        if (nt * kBlockN >= a.H) return;
    }
#define BRX_TILE(MR, WM) \
    dense_tile<KIND, MR, WM>(a, order, hbuf, hstride, y_routed, y_shared, ring, dst_s, e, m0, rows, ti.w, nt)
    if (rows <= 32) BRX_TILE(1, 1);
    else if (rows <= 64) BRX_TILE(1, 2);
    else if (rows <= 128) BRX_TILE(2, 2);
    else BRX_TILE(4, 2);
#undef BRX_TILE
}

}  // namespace

hipError_t launch_dense(const FwdArgs& a, const ThinArgs& t, int phases, hipStream_t s) {
    const int tiles = (t.mt_pad + kXcd * kDRun - 1) / (kXcd * kDRun) * (kXcd * kDRun);
    if (phases & 1) {
        const int fpb = a.act == BRX_ACT_SILU_MLP ? kBlockN : kBlockN / 2;
        const int ntn = (t.Imax + fpb - 1) / fpb;
        hipLaunchKernelGGL(k_dense_gemm<0>, dim3(tiles * ntn), dim3(kDThreads), 0, s, a, t.order, t.tile_start,
                           t.tinfo, t.E_ext, ntn, t.mt_pad, t.hbuf, t.Imax, t.y_routed, t.y_shared);
        hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
    }
    if (phases & 2) {
        const int ntn = (a.H + kBlockN - 1) / kBlockN;
        hipLaunchKernelGGL(k_dense_gemm<1>, dim3(tiles * ntn), dim3(kDThreads), 0, s, a, t.order, t.tile_start,
                           t.tinfo, t.E_ext, ntn, t.mt_pad, t.hbuf, t.Imax, t.y_routed, t.y_shared);
        return hipGetLastError();
    }
    return hipSuccess;
}

}  // namespace brx
