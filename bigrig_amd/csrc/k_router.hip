// Router top-k: logits = x . W_r^T (+ bias), top-k by logit (or by the sigmoid rules'
// selection values), routing weights.
//
// Replaces the MoE block's `gate(x)` + softmax + argpartition + take (+ renorm) that the
// reference restates at bigrig_engine/stream.py:895 and 1436-1439 (rule: adapter.py:75-93).
//
// Reduction order (the contract that makes indices reproducible bit for bit): lane l of a
// wave accumulates the 8-element chunks c = l, l+64, ... with fmaf in element order, then the
// 64 partials are combined by an xor butterfly (offsets 32, 16, ..., 1). Top-k is selected
// on the logits, descending, ties to the lower expert id; softmax is monotonic, so this is the
// top-k of the probabilities except at exact fp32 probability ties, where the order is
// defined here rather than left to argpartition.
#include "brx_internal.h"

namespace brx {
namespace {

constexpr int kRouterThreads = 256;
constexpr int kSmallT = 64;  // up to this many tokens: one wave per (row, 4 tokens) (5 us at 64); above: MFMA tiles (9 us)
constexpr int kWideH = 5120;  // wider rows: see small_call

// ---------------------------------------------------------------- many tokens
// k_router_mfma: a block computes the logits of 16 M tokens x 16 M experts on fp32 MFMAs, in the
// order above. v_mfma_f32_16x16x1_4b_f32 is one fused multiply-add per output and block (measured
// bit for bit equal to fmaf chains, subnormals included), so a lane chain l is 8 of them a chunk;
// the instruction's four blocks are the chains l, l + 16, l + 32 and l + 48 (lane group g of 16
// lanes feeds chain l0 + 16 g). The butterfly is then: (block 0 + block 2) + (block 1 + block 3)
// for offsets 32 and 16, and with l0 = 8 s + i (s < 2, i < 8): s for offset 8, in the wave i, and
// the waves i ^ 4, i ^ 2 and i ^ 1 through LDS for offsets 4, 2 and 1.
//
// Step (s, j) copies chunks 64 j + 8 (s + 2 g) + i of the block's token rows and weight rows, four
// runs of 128 bytes a row (256 of an fp32 row), into one slot of a ring (buffer_load ... lds; chunks
// past the row's end and rows past the last come as zeros, which leave a chain as it is).
//
// Bound: the fp32 MFMA rate, 64 FMA a clock and SIMD (8 us for 2048 tokens x 128 experts x 2048),
// and for few tiles the copies' latency. 16 x 16 tiles (M 1, two blocks a CU) while they are one
// round of the chip; above it their copies bound them (a 16 x 16 tile reads 128 KB for 0.5 M FMA:
// 25 us for 2048 tokens) and 32 x 32 tiles halve the bytes. The kernel this replaces formed the
// same chains with VALU fmaf at a quarter of the MFMA's rate, converting every activation. Before
// and after, 2048 x 128 experts: 128 tokens 13.1 -> 9.1 us, 512 15.1 -> 10.0, 2048 30.1 -> 21.9, 4096
// 61.6 -> 44.5; 301 tokens x 257 rows 25.3 -> 12.2; 512 tokens at 2880 x 128 19.9 -> 14.1.
typedef __attribute__((address_space(3))) void* RT_LDS;
constexpr int kRtThreads = 512;
template <bool WF32, int M>
constexpr int kRtStep = 16 * M * 512 * (WF32 ? 3 : 2);   // bytes: 32 chunks of each row
template <bool WF32>
constexpr int kRtRing = WF32 ? 3 : 4;                     // steps in the ring

template <int N>
__device__ __forceinline__ void rt_wait_barrier() {
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | ((N >> 4) << 14));   // vmcnt(N) lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
}

template <bool WF32, int M>
__global__ __launch_bounds__(kRtThreads) void k_router_mfma(
    const uint16_t* __restrict__ x, const void* __restrict__ w, const float* __restrict__ bias, int T, int H,
    int E, int net, float* __restrict__ logits) {
    constexpr int NR = kRtRing<WF32>;
    constexpr int RT = 16 * M;
    constexpr int XB = RT * 512;                   // x bytes of a step
    constexpr int STEP = kRtStep<WF32, M>;
    constexpr int NX = M, NW = WF32 ? 2 * M : M;   // 1 KB copies of a wave and step: x, weights
    constexpr int NV = NX + NW;
    __shared__ __attribute__((aligned(16))) uint8_t ring[NR * STEP];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // an XCD takes every expert tile of a token tile, so the x rows are read into one L2
    const int loc = blockIdx.x / 8;
    const int t0 = ((loc / net) * 8 + blockIdx.x % 8) * RT, e0 = (loc % net) * RT;
    if (t0 >= T) return;
    const int J = (H + 511) / 512, nsteps = 2 * J;
    const uint32_t xb = (uint32_t)min(T - t0, RT) * H * 2, wb = (uint32_t)min(E - e0, RT) * H * (WF32 ? 4 : 2);
    const uint8_t* xp = reinterpret_cast<const uint8_t*>(x) + (int64_t)t0 * H * 2;
    const uint8_t* wp = reinterpret_cast<const uint8_t*>(w) + (int64_t)e0 * H * (WF32 ? 4 : 2);
    const __amdgpu_buffer_rsrc_t rx =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(xp), (short)0, (int)xb, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(wp), (short)0, (int)wb, 0x00020000);
    // 16-byte slot q of a tile whose rows hold `per` slots a lane group g and chunk (1: bf16, 2:
    // fp32 halves): slot (row r, g', i', half) holds chunk i = i' ^ (r & 7) of group g = g' ^ (r >> 3 &
    // 1), so the 16 rows a read touches fall in distinct banks
    auto slot_of = [&](int q, int per, int& r, int& g, int& i, int& half) __attribute__((always_inline)) {
        half = q % per;
        const int c = q / per;
        r = c >> 5;
        g = ((c >> 3) & 3) ^ ((r >> 3) & 1);
        i = (c & 7) ^ (r & 7);
    };
    // issue the copies of step n = s J + j (a step past the last is all zeros and reads nothing)
    auto issue = [&](int n) __attribute__((always_inline)) {
        uint8_t* st = ring + (n % NR) * STEP;
        const int s = n >= J ? 1 : 0, j = n - s * J;
        const int lim = n < nsteps ? H / 8 : 0;
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            int r, g, i, h;
            slot_of((wv * NX + u) * 64 + lane, 1, r, g, i, h);
            const int c = 64 * j + 8 * (s + 2 * g) + i;
            const uint32_t vo = c < lim ? (uint32_t)(r * H * 2 + c * 16) : xb;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (RT_LDS)(st + (wv * NX + u) * 1024), 16, vo, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < NW; ++u) {
            int r, g, i, h;
            slot_of((wv * NW + u) * 64 + lane, WF32 ? 2 : 1, r, g, i, h);
            const int c = 64 * j + 8 * (s + 2 * g) + i;
            const uint32_t vo = c < lim ? (uint32_t)(WF32 ? r * H * 4 + c * 32 + h * 16 : r * H * 2 + c * 16) : wb;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (RT_LDS)(st + XB + (wv * NW + u) * 1024), 16, vo, 0, 0, 0);
        }
        asm volatile("" ::: "memory");
    };
#pragma unroll
    for (int n = 0; n < NR - 1; ++n) issue(n);
    const int r = lane & 15, g = lane >> 4;
    const int q0 = r * 32 + (g ^ ((r >> 3) & 1)) * 8 + (wv ^ (r & 7));   // this wave's chunk of row r
    auto unpack = [&](uint4 v, float (&f)[8]) __attribute__((always_inline)) {
        const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f[2 * b] = bf2f(q[b] & 0xFFFFu);
            f[2 * b + 1] = __uint_as_float(q[b] & 0xFFFF0000u);
        }
    };
    f32x16_t acc[M][M];
    f32x4_t first[M][M];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int n = 0; n < M; ++n) {
#pragma unroll
            for (int b = 0; b < 16; ++b) acc[m][n][b] = 0.0f;
#pragma unroll
            for (int b = 0; b < 4; ++b) first[m][n][b] = 0.0f;
        }
    // a block's chains of one s, complete: offsets 32 and 16
    auto blocks_sum = [&](const f32x16_t& a, int b) __attribute__((always_inline)) {
        return (a[b] + a[8 + b]) + (a[4 + b] + a[12 + b]);
    };
    for (int n = 0, slot = 0; n < nsteps; ++n) {
        // step n landed in every wave, and step n - 1's slot is free for step n + NR - 1
        rt_wait_barrier<(NR - 2) * NV>();
        issue(n + NR - 1);
        const uint8_t* st = ring + slot * STEP;
        slot = slot + 1 == NR ? 0 : slot + 1;
        float xf[M][8], wf[M][8];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            unpack(*reinterpret_cast<const uint4*>(st + (q0 + m * 512) * 16), xf[m]);
            if constexpr (WF32) {
                const uint8_t* p = st + XB + (q0 + m * 512) * 32;
                const f32x4_t v0 = *reinterpret_cast<const f32x4_t*>(p), v1 = *reinterpret_cast<const f32x4_t*>(p + 16);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    wf[m][b] = v0[b];
                    wf[m][4 + b] = v1[b];
                }
            } else {
                unpack(*reinterpret_cast<const uint4*>(st + XB + (q0 + m * 512) * 16), wf[m]);
            }
        }
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int v = 0; v < M; ++v)
                    acc[m][v] = __builtin_amdgcn_mfma_f32_16x16x1f32(xf[m][b], wf[v][b], acc[m][v], 0, 0, 0);
        if (n == J - 1) {
#pragma unroll
            for (int m = 0; m < M; ++m)
#pragma unroll
                for (int v = 0; v < M; ++v) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) first[m][v][b] = blocks_sum(acc[m][v], b);
#pragma unroll
                    for (int b = 0; b < 16; ++b) acc[m][v][b] = 0.0f;
                }
        }
    }
    // offset 8 in the wave, 4, 2 and 1 across the waves
    rt_wait_barrier<0>();
    float* red = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int v = 0; v < M; ++v)
#pragma unroll
            for (int b = 0; b < 4; ++b)
                red[wv * RT * RT + (16 * m + 4 * g + b) * RT + 16 * v + r] = first[m][v][b] + blocks_sum(acc[m][v], b);
    __syncthreads();
    for (int o = tid; o < RT * RT; o += kRtThreads) {
        const float* p = red + o;
        constexpr int S = RT * RT;
        const float v = ((p[0] + p[4 * S]) + (p[2 * S] + p[6 * S])) + ((p[S] + p[5 * S]) + (p[3 * S] + p[7 * S]));
        const int t = t0 + o / RT, e = e0 + o % RT;
        if (t < T && e < E) logits[(int64_t)t * (E + 1) + e] = bias ? v + bias[e] : v;
    }
}

template <int M>
hipError_t mfma_launch(const brx_layer_desc& d, const void* x, const void* w_router, const float* bias, int T,
                       float* logits, hipStream_t s) {
    const int net = (d.n_experts + 16 * M - 1) / (16 * M), ntt = (T + 16 * M - 1) / (16 * M);
    dim3 grid((ntt + 7) / 8 * 8 * net), block(kRtThreads);
    if (d.router_dtype == BRX_DT_F32)
        hipLaunchKernelGGL((k_router_mfma<true, M>), grid, block, 0, s, (const uint16_t*)x, w_router, bias, T,
                           d.hidden, d.n_experts, net, logits);
    else
        hipLaunchKernelGGL((k_router_mfma<false, M>), grid, block, 0, s, (const uint16_t*)x, w_router, bias, T,
                           d.hidden, d.n_experts, net, logits);
    return hipGetLastError();
}

// ---------------------------------------------------------------- small T
// k_router_logits: one wave per (expert row, tile of TT tokens), WPB waves per block; every
// load of the wave is issued before the first FMA. Same per-lane chain and butterfly as
// k_router_mfma's, so the logits are the same bits.
template <bool WF32, int TT, int WPB>
__global__ __launch_bounds__(WPB * kWave) void k_router_logits(
    const uint16_t* __restrict__ x, const void* __restrict__ w, const float* __restrict__ bias,
    const uint16_t* __restrict__ sgw, int T, int H, int E, float* __restrict__ logits) {
    constexpr int kNJ = 6;                      // chunks per lane per pass (one pass: H <= 3072)
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * WPB + (threadIdx.x >> 6);
    const int rows = E + (sgw ? 1 : 0);
    const int t0 = blockIdx.y * TT;
    const int nt = min(TT, T - t0);
    const int nch = H / 8;
    if (r >= rows) return;
    const bool wf32 = WF32 && r < E;
    float acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = 0.0f;
    // passes of kNJ chunks per lane continue each lane's chain in chunk order; every load of a
    // pass is issued before its first FMA
    for (int jb = 0; jb < nch; jb += kWave * kNJ) {
        uint4 wv[kNJ][2];
        uint4 xv[TT][kNJ];
#pragma unroll
        for (int j = 0; j < kNJ; ++j) {
            const int c = jb + lane + kWave * j;
            if (c < nch) {
                if (wf32) {
                    const uint4* p = reinterpret_cast<const uint4*>(
                        reinterpret_cast<const float*>(w) + (int64_t)r * H + 8 * c);
                    wv[j][0] = p[0];
                    wv[j][1] = p[1];
                } else {
                    const uint16_t* src = r < E ? reinterpret_cast<const uint16_t*>(w) + (int64_t)r * H : sgw;
                    wv[j][0] = *reinterpret_cast<const uint4*>(src + 8 * c);
                }
#pragma unroll
                for (int t = 0; t < TT; ++t)
                    if (t < nt) xv[t][j] = *reinterpret_cast<const uint4*>(x + (int64_t)(t0 + t) * H + 8 * c);
            }
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
#pragma unroll
            for (int j = 0; j < kNJ; ++j) {
                const int c = jb + lane + kWave * j;
                if (c < nch && t < nt) {
                    uint32_t xw[4] = {xv[t][j].x, xv[t][j].y, xv[t][j].z, xv[t][j].w};
                    float wf[8];
                    if (wf32) {
                        wf[0] = __uint_as_float(wv[j][0].x); wf[1] = __uint_as_float(wv[j][0].y);
                        wf[2] = __uint_as_float(wv[j][0].z); wf[3] = __uint_as_float(wv[j][0].w);
                        wf[4] = __uint_as_float(wv[j][1].x); wf[5] = __uint_as_float(wv[j][1].y);
                        wf[6] = __uint_as_float(wv[j][1].z); wf[7] = __uint_as_float(wv[j][1].w);
                    } else {
                        uint32_t ww[4] = {wv[j][0].x, wv[j][0].y, wv[j][0].z, wv[j][0].w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            wf[2 * i] = bf2f(ww[i] & 0xFFFFu);
                            wf[2 * i + 1] = bf2f(ww[i] >> 16);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        acc[t] = fmaf(bf2f(xw[i] & 0xFFFFu), wf[2 * i], acc[t]);
                        acc[t] = fmaf(bf2f(xw[i] >> 16), wf[2 * i + 1], acc[t]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        if (t >= nt) break;   // uniform
        float s = wave_sum_xor(acc[t]);
        if (lane == 0) logits[(int64_t)(t0 + t) * (E + 1) + r] = (r < E && bias) ? s + bias[r] : s;
    }
}

// Top-k of one token's logits row `l` ([E + 1], the last entry the shared-gate logit) and its
// routing weights, by the calling wave.
template <int kPer>
__device__ __forceinline__ void topk_row(const float* __restrict__ l, const uint16_t* __restrict__ x,
                                         const uint16_t* __restrict__ sgw, int t, int H, int E, int k,
                                         const RouteRule& rr, int has_sg, int32_t* __restrict__ out_idx,
                                         float* __restrict__ out_w, float* __restrict__ out_sg) {
    const int lane = threadIdx.x & 63;
    float v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = lane + kWave * i;
        v[i] = e < E ? l[e] : 0.0f;
    }
    // the shared gate's logit, where the logits come without it: the wave's lanes are its chains
    float gate = 0.0f;
    if (sgw) {
        constexpr int kG = 4;                       // chunks a lane has in flight
        for (int c0 = lane; c0 < H / 8; c0 += kWave * kG) {
            uint4 xv[kG], gv[kG];
#pragma unroll
            for (int u = 0; u < kG; ++u) {
                const int c = min(c0 + kWave * u, H / 8 - 1);
                xv[u] = *reinterpret_cast<const uint4*>(x + (int64_t)t * H + 8 * c);
                gv[u] = *reinterpret_cast<const uint4*>(sgw + 8 * c);
            }
#pragma unroll
            for (int u = 0; u < kG; ++u) {
                if (c0 + kWave * u >= H / 8) break;
                const uint32_t xw[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
                const uint32_t gw[4] = {gv[u].x, gv[u].y, gv[u].z, gv[u].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    gate = fmaf(bf2f(xw[i] & 0xFFFFu), bf2f(gw[i] & 0xFFFFu), gate);
                    gate = fmaf(bf2f(xw[i] >> 16), bf2f(gw[i] >> 16), gate);
                }
            }
        }
        gate = wave_sum_xor(gate);
    }
    int my_id;
    float my_v;
    wave_select<kPer>(v, rr, E, k, my_id, my_v);
    const float wt = wave_weight<kPer>(v, rr, E, k, my_id, my_v);
    if (lane < k) {
        out_idx[(int64_t)t * k + lane] = my_id;
        out_w[(int64_t)t * k + lane] = wt;
    }
    if (lane == 0 && has_sg && out_sg) out_sg[t] = 1.0f / (1.0f + expf(-(sgw ? gate : l[E])));
}

// One wave per token over logits [T][E + 1]; with `sgw` given it also forms the shared gate's logit.
template <int kPer>
__global__ __launch_bounds__(kRouterThreads) void k_router_topk(
    const float* __restrict__ logits, const uint16_t* __restrict__ x, const uint16_t* __restrict__ sgw, int T, int H,
    int E, int k, RouteRule rr, int has_sg, int32_t* __restrict__ out_idx, float* __restrict__ out_w,
    float* __restrict__ out_sg) {
    const int t = blockIdx.x * (kRouterThreads / kWave) + (threadIdx.x >> 6);
    if (t >= T) return;
    topk_row<kPer>(logits + (int64_t)t * (E + 1), x, sgw, t, H, E, k, rr, has_sg, out_idx, out_w, out_sg);
}

template <bool WF32>
hipError_t logits_launch(const brx_layer_desc& d, const void* x, const void* w_router, const float* bias,
                         const void* sgw, int T, float* logits, hipStream_t s) {
    constexpr int TT = 4, WPB = 1;
    const int rows = d.n_experts + (sgw ? 1 : 0);
    dim3 grid((rows + WPB - 1) / WPB, (T + TT - 1) / TT);
    hipLaunchKernelGGL((k_router_logits<WF32, TT, WPB>), grid, dim3(WPB * kWave), 0, s,
                       (const uint16_t*)x, w_router, bias, (const uint16_t*)sgw, T, d.hidden,
                       d.n_experts, logits);
    return hipGetLastError();
}

hipError_t topk_launch(const brx_layer_desc& d, int T, int has_sg, const float* logits, const void* x,
                       const void* sgw, const float* bias, int32_t* out_idx, float* out_w, float* out_sg, hipStream_t s) {
    const int E = d.n_experts;
    const RouteRule rr = route_rule(d, bias);
    dim3 grid((T + 3) / 4), block(kRouterThreads);
#define BRX_TOPK(KP) hipLaunchKernelGGL(k_router_topk<KP>, grid, block, 0, s, logits, (const uint16_t*)x, \
                                        (const uint16_t*)sgw, T, d.hidden, E, d.top_k, rr, has_sg, out_idx, out_w, out_sg)
    if (E <= 64) BRX_TOPK(1);
    else if (E <= 128) BRX_TOPK(2);
    else if (E <= 256) BRX_TOPK(4);
    else BRX_TOPK(8);
#undef BRX_TOPK
    return hipGetLastError();
}

// Calls that take one wave per (row, 4 tokens). Above kWideH inputs those of a few tiles do so past
// kSmallT tokens too: a tile's K loop is then longer than the waves take, and this is the kernel those
// calls had before the tiles. Waves / tiles, us, at 6144 inputs (5184 and 8192 move both alike; narrower
// rows had a slower kernel than either before the tiles):
//   to 128 tokens   bf16 8 experts x 100 9.2 / 19.7, 128 x 128 17.1 / 20.1, 256 x 80 20.4 / 20.5; fp32
//                   128 x 100 20.2 / 21.5, 256 x 80 23.4 / 27.1; past the line 256 x 100 28.7 / 27.6
//   to 256          bf16 64 x 256 16.2 / 20.0; fp32 32 x 256 13.9 / 21.3; past 128 x 180 21.9 / 20.4
//   to 512          bf16 16 x 512 14.4 / 20.0; fp32 8 x 512 17.7 / 21.5; past 64 x 512 30.5 / 20.2
//   to 1024         4 x 1024 15.0 / 20.0; past 8 x 1024 20.9 / 20.1
bool small_call(const brx_layer_desc& d, int T) {
    if (T <= kSmallT) return true;
    if (d.hidden <= kWideH) return false;
    const bool f32 = d.router_dtype == BRX_DT_F32;
    const int rows_tokens = T <= 128 ? 20480 : T <= 256 ? (f32 ? 12800 : 16640) : T <= 512 ? (f32 ? 8192 : 16640)
                          : T <= 1024 ? 4096 : 0;
    return (int64_t)d.n_experts * T <= rows_tokens;
}

}  // namespace

size_t router_workspace_bytes(const brx_layer_desc& d, int T) {
    return sizeof(float) * (size_t)T * (d.n_experts + 1);
}

hipError_t launch_router_logits(const brx_layer_desc& d, const void* x, const void* w_router,
                                const float* bias, const void* sgw, int T, float* logits,
                                hipStream_t s) {
    // sigmoid rules keep the logits raw: their bias enters the selection only
    if (d.route_mode >= BRX_ROUTE_SIGMOID_TOPK) bias = nullptr;
    return d.router_dtype == BRX_DT_F32 ? logits_launch<true>(d, x, w_router, bias, sgw, T, logits, s)
                                        : logits_launch<false>(d, x, w_router, bias, sgw, T, logits, s);
}

hipError_t launch_router(const brx_layer_desc& d, const void* x, const void* w_router,
                         const float* bias, const void* sgw, int T, int32_t* out_idx,
                         float* out_w, float* out_sg, float* ws_logits, hipStream_t s) {
    if (T <= 0) return hipSuccess;
    if (small_call(d, T)) {
        hipError_t e = launch_router_logits(d, x, w_router, bias, sgw, T, ws_logits, s);
        if (e != hipSuccess) return e;
        return topk_launch(d, T, sgw ? 1 : 0, ws_logits, nullptr, nullptr, bias, out_idx, out_w, out_sg, s);
    }
    const float* lbias = d.route_mode >= BRX_ROUTE_SIGMOID_TOPK ? nullptr : bias;
    const int64_t tiles16 = (int64_t)((T + 15) / 16) * ((d.n_experts + 15) / 16);
    hipError_t e = tiles16 <= 512 ? mfma_launch<1>(d, x, w_router, lbias, T, ws_logits, s)
                                  : mfma_launch<2>(d, x, w_router, lbias, T, ws_logits, s);
    if (e != hipSuccess) return e;
    return topk_launch(d, T, sgw ? 1 : 0, ws_logits, x, sgw, bias, out_idx, out_w, out_sg, s);
}

}  // namespace brx
