// k_route.hip -- router softmax + top-8 and the prefix-sum expert bucket fill.
#include "moe_internal.hpp"
#include "bucket_fill.hpp"

namespace moe {

// ---------------------------------------------------------------- router top-8
// One 64-lane wave per token.  Replaces shaders/router_topk.comp, whose 256-lane workgroup
// ran two 8-step LDS tree reductions and a serial insertion sort on lane 0
// (router_topk.comp:37-85).  Here each lane keeps E/64 logits in registers; each of the 8
// rounds is one wave max of the order-preserving key (six DPP steps into lane 63) and a
// ballot of the lanes holding it; the lowest index holding it wins, like the shader's strict
// '>' insertion (router_topk.comp:76).  Lane r then stores rank r and its weight, lane 8 the
// shared slot.  E <= 256 (moe_create's limit), so four logits per lane.
__global__ __launch_bounds__(64) void k_router_topk(const float *__restrict__ logits, int M, int E, int renorm,
                                                    uint16_t *__restrict__ ids, float *__restrict__ w) {
    // one wave per workgroup: the dispatcher spreads the tokens over every CU and SIMD
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x;
    if (t >= M) return; // whole wave leaves together
    int id;
    float wt;
    route_wave<4>(logits + (size_t)t * E, E, renorm, lane, id, wt);
    if (lane < SLOTS) {
        ids[(size_t)t * SLOTS + lane] = (uint16_t)id;
        w[(size_t)t * SLOTS + lane] = wt;
    }
}

// The same with four waves per token (route_wg4, the same results): about 2.5 times less
// latency per token, for small M where latency, not throughput, is what a launch costs.
__global__ __launch_bounds__(256) void k_router_topk_wg4(const float *__restrict__ logits, int M, int E, int renorm,
                                                         uint16_t *__restrict__ ids, float *__restrict__ w) {
    __shared__ RouteLds R;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = blockIdx.x;
    int id;
    float wt;
    route_wg4(logits + (size_t)t * E, E, renorm, lane, wv, R, id, wt);
    if (wv == 0 && lane < SLOTS) {
        ids[(size_t)t * SLOTS + lane] = (uint16_t)id;
        w[(size_t)t * SLOTS + lane] = wt;
    }
}

constexpr int ROUTER_WG4_MAX_M = 256;

hipError_t launch_router_topk(const float *logits, int M, int E, int renorm, uint16_t *ids, float *w,
                              hipStream_t st, KernelTimer *T) {
    if (M <= 0) return hipSuccess;
    if (E < TOPK || E > 256) return hipErrorInvalidValue;
    {
        TimedLaunch tl(T, MOE_K_ROUTER_TOPK, st);
        if (M <= ROUTER_WG4_MAX_M)
            hipLaunchKernelGGL(k_router_topk_wg4, dim3((unsigned)M), dim3(256), 0, st, logits, M, E, renorm, ids, w);
        else
            hipLaunchKernelGGL(k_router_topk, dim3((unsigned)M), dim3(64), 0, st, logits, M, E, renorm, ids, w);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- router gate GEMV
// logits[t][e] = sum_k xin[t][k] * Wg[e][k], xin = x or RMSNorm(x); Wg [E][H], rows = experts,
// in the caller's buffer as GGML IQ4_XS (136-byte super-blocks), f32 or f16 (the types a GGUF
// file's ffn_gate_inp comes in: llama.cpp's quantizer keeps that tensor F32 or F16).
// Replaces shaders/router.comp:21-61 (dispatched at src/inference.rs:598-605), whose 64x8 f32
// tiles re-dequantized every weight per tile.  One wave per (expert row, group of TM tokens:
// 1, 2 or 4 by M), four waves per workgroup: lane l owns the 32 weights 32l..32l+31 of the
// row (H = 2048 is one sub-block per lane) and reads them once -- IQ4_XS: decoded into
// biased codebook bytes and one f32 scale; f32: eight 16-byte loads; f16: four, converted
// exactly -- then for each token takes one f32 dot of 32 against x (loaded for all the
// group's tokens before any is used) and a wave sum.  All f32: the weights are exact, so the
// logits differ from an f64 sum by f32 rounding only.
//
// The top-8 follows as a k_router_topk launch.  Measured on MI355X, one launch for both at
// M <= 8 -- the last workgroup of a token group routing it after the others' logits were
// handed over through a device counter -- was slower than two launches in a graph: 8.8 us
// at M = 1 with an agent-scope release / acquire pair (each writes back / invalidates the XCD's
// whole L2), 6.2 us with write-through stores and system-scope loads instead, against 5.6 us.
constexpr int RG_WAVES = 4; // experts per workgroup
constexpr int RG_GEMV_MAX_WAVES = 1024; // waves of the 4-token form (4 per CU); beyond: k_router_gemm

struct RouterGemvArgs {
    const void *wg;
    const float *x;
    int M, E, rmsnorm;
    float *logits;
};

// The lane's 32 weights of row e as f32 (dense types), or its codebook bytes and scale (IQ4_XS).
template <int H, int WT>
__device__ __forceinline__ void router_row_weights(const void *wg, int e, int sl, bool on, uint32_t (&kv)[8],
                                                   float &dl, float (&wf)[32]) {
    if constexpr (WT == MOE_WG_IQ4_XS) {
        constexpr int SBR = H / QK;
        const uint8_t *blk = (const uint8_t *)wg + ((size_t)e * SBR + sl / 8) * SB_BYTES;
        const u32x2 hdr = ldg<u32x2>(blk);
        const int j = sl % 8;
        const u32x2 q01 = ldg<u32x2>(blk + 8 + 16 * j), q23 = ldg<u32x2>(blk + 16 + 16 * j);
        const uint32_t q[4] = {q01.x, q01.y, q23.x, q23.y};
#pragma unroll
        for (int d = 0; d < 4; ++d) kv_biased8(q[d], kv[2 * d], kv[2 * d + 1]);
        dl = on ? sub_scale(hdr, j) : 0.0f;
    } else if constexpr (WT == MOE_WG_F32) {
        load32((const float *)wg + (size_t)e * H + 32 * sl, wf);
        if (!on)
#pragma unroll
            for (int k = 0; k < 32; ++k) wf[k] = 0.0f;
    } else {
        const _Float16 *src = (const _Float16 *)wg + (size_t)e * H + 32 * sl;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 v = ldg<u32x4>(src + 8 * i);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const f16x2 h2 = __builtin_bit_cast(f16x2, (uint32_t)v[d]);
                wf[8 * i + 2 * d] = on ? (float)h2[0] : 0.0f;
                wf[8 * i + 2 * d + 1] = on ? (float)h2[1] : 0.0f;
            }
        }
    }
}

template <int H, int RG_TM, int WT>
__global__ __launch_bounds__(64 * RG_WAVES) void k_router_gemv(RouterGemvArgs a) {
    constexpr int NSB = H / 32;
    static_assert(H % QK == 0 && NSB <= 64, "one sub-block per lane");
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int e = blockIdx.x * RG_WAVES + wv;
    const int t0 = blockIdx.y * RG_TM;
    const int M = a.M, E = a.E;
    if (e < E) { // whole wave
        const bool on = lane < NSB;
        const int sl = on ? lane : 0; // idle lanes (H < 2048) read sub-block 0 and add nothing
        uint32_t kv[8];
        float dl = 0.0f, wf[32];
        router_row_weights<H, WT>(a.wg, e, sl, on, kv, dl, wf);
        float xv[RG_TM][32];
#pragma unroll
        for (int i = 0; i < RG_TM; ++i) {
            const int t = t0 + i < M ? t0 + i : M - 1; // rows past M repeat the last; not stored
            load32(a.x + (size_t)t * H + 32 * sl, xv[i]);
        }
#pragma unroll
        for (int i = 0; i < RG_TM; ++i) {
            float xs = 0.f, ss = 0.f;
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                xs += xv[i][k];
                ss = __builtin_fmaf(xv[i][k], xv[i][k], ss);
            }
            float part;
            if constexpr (WT == MOE_WG_IQ4_XS) {
                part = dl * subblock_dot(kv, xv[i], xs);
            } else {
                part = 0.0f;
#pragma unroll
                for (int k = 0; k < 32; ++k) part = __builtin_fmaf(wf[k], xv[i][k], part);
            }
            const float dot = wave_sum(part);
            float inv = 1.0f;
            if (a.rmsnorm) inv = 1.0f / sqrtf(wave_sum(on ? ss : 0.0f) * (1.0f / (float)H) + 1e-6f);
            if (lane == 0 && t0 + i < M) a.logits[(size_t)(t0 + i) * E + e] = dot * inv;
        }
    }
}

// ---------------------------------------------------------------- router gate product, many tokens
// The same logits as a matrix product on the f32 matrix cores (v_mfma_f32_16x16x4_f32: f32
// operands and sums, the weights exact in f32, so again only f32 rounding).  A workgroup owns
// TILE x TILE logits (tokens x experts) and its NW waves split K, each keeping its partial block
// in registers; x and Wg go straight from memory into MFMA operands, a ring of ND 32-K stages in
// flight (no LDS: the waves share no operand), the partial blocks are summed through LDS, and the
// tokens' RMSNorm factors come from the same x registers.
// K inside a stage: the order is free as long as both operands agree.  Lane (g, i) takes K =
// 16 q + 4 g + j of row i (q < 2, j < 4), so the four lanes of a row read 64 consecutive bytes of
// x per load, and one IQ4_XS qs dword has the lane's 8 weights: low nibbles q = 0, high q = 1.
// Rounding: an MFMA chain covers one stage (32 K); the chains are added in f32 per wave and the
// waves' sums and the RMSNorm factor taken in f64.  Relative 2-norm against f64 (E = 256): 1.2e-7
// (1.34e-7 in the 64 x 64 form) for every gate type, the one-row form 1.34e-7 (IQ4_XS 2.6e-7).
// f16 gate, M = 4096: 947 -> 48 us; the f32 matrix cores alone need 31 us at their measured
// 139 TFLOP/s.  Bound by one wave's chain of f32 MFMAs and conversions per SIMD: with both operands staged
// in LDS instead the 64 x 64 form takes 44.8 us against 46.6, and its error is larger (1.54e-7).
template <int WT>
struct RmW; // a lane's 8 weights of one stage as loaded; off: byte offset of the lane's first one
template <>
struct RmW<MOE_WG_F32> {
    f32x4 v[2];
    static __device__ __forceinline__ uint32_t offset(int H, int e, int g) { return ((uint32_t)e * H + 4 * g) * 4u; }
    __device__ __forceinline__ void load(const uint8_t *wg, int k0, uint32_t off) {
        v[0] = ldg<f32x4>(wg + 4 * k0 + off);
        v[1] = ldg<f32x4>(wg + 4 * k0 + 64 + off);
    }
    __device__ __forceinline__ void get(int, float (&f)[8]) const {
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = v[k / 4][k % 4];
    }
};
template <>
struct RmW<MOE_WG_F16> {
    u32x2 v[2];
    static __device__ __forceinline__ uint32_t offset(int H, int e, int g) { return ((uint32_t)e * H + 4 * g) * 2u; }
    __device__ __forceinline__ void load(const uint8_t *wg, int k0, uint32_t off) {
        v[0] = ldg<u32x2>(wg + 2 * k0 + off);
        v[1] = ldg<u32x2>(wg + 2 * k0 + 32 + off);
    }
    __device__ __forceinline__ void get(int, float (&f)[8]) const {
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = (float)__builtin_bit_cast(f16x2, (uint32_t)v[k / 4][k % 4 / 2])[k % 2];
    }
};
template <>
struct RmW<MOE_WG_IQ4_XS> {
    u32x2 hdr;
    uint32_t q;
    // a row is whole 16-byte pieces (1088 or 272 bytes), so the low bits are the lane's place in
    // its sub-block's 16 qs bytes
    static __device__ __forceinline__ uint32_t offset(int H, int e, int g) {
        return (uint32_t)e * (H / QK * SB_BYTES) + 4u * (uint32_t)g;
    }
    __device__ __forceinline__ void load(const uint8_t *wg, int k0, uint32_t off) {
        const uint8_t *blk = wg + k0 / QK * SB_BYTES;
        hdr = ldg<u32x2>(blk + (off & ~15u));
        q = ldg<uint32_t>(blk + 8 + 16 * (k0 % QK / 32) + off);
    }
    __device__ __forceinline__ void get(int k0, float (&f)[8]) const {
        const float dl = sub_scale(hdr, k0 % QK / 32), off = -128.0f * dl;
        uint32_t b[2];
        kv_biased8(q, b[0], b[1]);
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = __builtin_fmaf(ubyte(b[k / 4], k % 4), dl, off); // (b - 128) dl, exact
    }
};

template <int RB, int NW>
struct RmShape { // RB x RB MFMA blocks of 16 x 16 per wave
    static constexpr int TILE = 16 * RB, THREADS = 64 * NW;
    static constexpr size_t SMEM = ((size_t)NW * TILE * TILE + NW * TILE + TILE) * 4;
};

template <int H, int WT, int RB, int NW, int ND>
__global__ __launch_bounds__(64 * NW, NW / 4) void k_router_gemm(RouterGemvArgs a) {
    using S = RmShape<RB, NW>;
    constexpr int TILE = S::TILE, KW = H / NW, NST = KW / 32, DEPTH = ND < NST ? ND : NST;
    static_assert(KW % 32 == 0 && H % QK == 0 && NST % DEPTH == 0, "whole turns of the ring per wave");
    extern __shared__ float rm_smem[];
    float *red = rm_smem, *s_ss = red + NW * TILE * TILE, *s_inv = s_ss + NW * TILE;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int M = a.M, E = a.E;
    // workgroup w runs on XCD w % 8: the expert tiles of one token tile on one XCD, so its x rows
    // come from memory once
    const int nct = (E + TILE - 1) / TILE, w = (int)blockIdx.x;
    const int rt = 8 * ((w >> 3) / nct) + (w & 7), ct = (w >> 3) % nct;
    const int t0 = rt * TILE, e0 = ct * TILE;
    if (t0 >= M) return;
    // this lane's rows as byte offsets on the wave-uniform x (of the tile) and Wg plus the stage's
    // K (tokens and experts past the end repeat the last)
    const uint8_t *xt = (const uint8_t *)(a.x + (size_t)t0 * H), *wg = (const uint8_t *)a.wg;
    uint32_t xo[RB], wo[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        xo[r] = (uint32_t)(min(16 * r + i, M - 1 - t0) * H + 4 * g) * 4u;
        wo[r] = RmW<WT>::offset(H, min(e0 + 16 * r + i, E - 1), g);
    }
    struct Stage {
        f32x4 x[RB][2];
        RmW<WT> w[RB];
    } st[DEPTH];
    auto issue = [&](Stage &s, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            s.x[r][0] = ldg<f32x4>(xt + 4 * k0 + xo[r]);
            s.x[r][1] = ldg<f32x4>(xt + 4 * k0 + 64 + xo[r]);
            s.w[r].load(wg, k0, wo[r]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x4 tot[RB][RB], ss[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) {
        ss[r] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < RB; ++c) tot[r][c] = f32x4{0, 0, 0, 0};
    }
    auto compute = [&](const Stage &s, int k0) __attribute__((always_inline)) {
        float wf[RB][8];
#pragma unroll
        for (int r = 0; r < RB; ++r) s.w[r].get(k0, wf[r]);
        f32x4 acc[RB][RB];
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int c = 0; c < RB; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.x[r][k / 4][k % 4], wf[c][k],
                                                                     k ? acc[r][c] : f32x4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RB; ++r) {
#pragma unroll
            for (int c = 0; c < RB; ++c) tot[r][c] += acc[r][c];
#pragma unroll
            for (int k = 0; k < 8; ++k) ss[r][k % 4] = __builtin_fmaf(s.x[r][k / 4][k % 4], s.x[r][k / 4][k % 4], ss[r][k % 4]);
        }
    };
    // the loop stays rolled, one turn of the ring an iteration (unrolled over all stages the
    // compiler kept hundreds of operands live and spilled); requests past the last stage re-read it
    const int kw = wv * KW;
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) issue(st[d], kw + 32 * d);
#pragma unroll 1
    for (int k0 = kw; k0 < kw + KW; k0 += 32 * DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            issue(st[(d + DEPTH - 1) % DEPTH], min(k0 + 32 * (d + DEPTH - 1), kw + KW - 32));
            compute(st[d], k0 + 32 * d);
        }
    }
    // partial blocks and sums of squares to LDS (C: row 4 g + n, column i), then each logit summed
#pragma unroll
    for (int r = 0; r < RB; ++r) {
#pragma unroll
        for (int c = 0; c < RB; ++c)
#pragma unroll
            for (int n = 0; n < 4; ++n) red[(wv * TILE + 16 * r + 4 * g + n) * TILE + 16 * c + i] = tot[r][c][n];
        float q = (ss[r][0] + ss[r][1]) + (ss[r][2] + ss[r][3]);
        q += __shfl_xor(q, 16);
        q += __shfl_xor(q, 32);
        if (g == 0) s_ss[wv * TILE + 16 * r + i] = q;
    }
    __syncthreads();
    if (tid < TILE) {
        double q = 0.0;
#pragma unroll
        for (int v = 0; v < NW; ++v) q += (double)s_ss[v * TILE + tid];
        s_inv[tid] = a.rmsnorm ? (float)(1.0 / sqrt(q * (1.0 / H) + 1e-6)) : 1.0f;
    }
    __syncthreads();
    for (int o = tid; o < TILE * TILE; o += S::THREADS) {
        const int r = o / TILE, c = o % TILE;
        double v = 0.0;
#pragma unroll
        for (int p = 0; p < NW; ++p) v += (double)red[p * TILE * TILE + o];
        if (t0 + r < M && e0 + c < E) a.logits[(size_t)(t0 + r) * E + e0 + c] = (float)(v * (double)s_inv[r]);
    }
}

template <int H, int WT, int RB, int NW, int ND>
static void launch_router_gemm_t(const RouterGemvArgs &a, hipStream_t st) {
    using S = RmShape<RB, NW>;
    const int nrt = ((a.M + S::TILE - 1) / S::TILE + 7) / 8 * 8, nct = (a.E + S::TILE - 1) / S::TILE;
    hipLaunchKernelGGL((k_router_gemm<H, WT, RB, NW, ND>), dim3((unsigned)(nrt * nct)), dim3(S::THREADS), S::SMEM, st, a);
}

template <int H, int TM, int WT>
static void launch_router_gemv_t(const RouterGemvArgs &a, hipStream_t st) {
    const dim3 grid((unsigned)((a.E + RG_WAVES - 1) / RG_WAVES), (unsigned)((a.M + TM - 1) / TM));
    hipLaunchKernelGGL((k_router_gemv<H, TM, WT>), grid, dim3(64 * RG_WAVES), 0, st, a);
}

template <int RB, int NW>
static int rm_tiles(const RouterGemvArgs &a) {
    using S = RmShape<RB, NW>;
    return ((a.M + S::TILE - 1) / S::TILE) * ((a.E + S::TILE - 1) / S::TILE);
}

// One row per wave while its waves fit the 1,024 SIMDs (M <= 16 at E = 256, 64 at E = 64), then
// the matrix product with the smallest tile that fills the 256 CUs at most twice.  Measured (us,
// f32 gate, E = 256, graph replays; E = 128, M = 16 / 64: 6.6 / 11.4 by rows, 9.0 / 9.1 by tiles):
//     M                  8     16     64    256    512   1000   2048   4096
//     one row per wave  6.7    6.8   20.8   73     142    276    558   1112
//     16 x 16           8.0    9.2    9.2    9.4  17.3   33.2   65.1    127
//     32 x 32          13.8   15.2   18.2   18.3  18.5   19.1   35.5   68.1
//     64 x 64          41.2   41.5   43.3   43.7  43.7   43.4   43.9   45.8
// A workgroup of the 64 x 64 form takes the same ~41 us whatever M is (its waves' f32 MFMAs over all of
// K), so the smaller tiles win until they need a second round on the CUs.
template <int H, int WT>
static void launch_router_gemv_w(const RouterGemvArgs &a, hipStream_t st) {
    // a wave's tokens past M repeat the last one: at small M fewer tokens per wave
    if (a.M == 1) launch_router_gemv_t<H, 1, WT>(a, st);
    else if (a.M == 2) launch_router_gemv_t<H, 2, WT>(a, st);
    else if (a.E * ((a.M + 3) / 4) <= RG_GEMV_MAX_WAVES) launch_router_gemv_t<H, 4, WT>(a, st);
    else if (rm_tiles<1, 8>(a) <= 512) launch_router_gemm_t<H, WT, 1, 8, 8>(a, st);
    else if (rm_tiles<2, 8>(a) <= 512) launch_router_gemm_t<H, WT, 2, 8, 2>(a, st);
    else launch_router_gemm_t<H, WT, 4, 4, 2>(a, st);
}

template <int H>
static void launch_router_gemv_h(int wtype, const RouterGemvArgs &a, hipStream_t st) {
    if (wtype == MOE_WG_IQ4_XS) launch_router_gemv_w<H, MOE_WG_IQ4_XS>(a, st);
    else if (wtype == MOE_WG_F32) launch_router_gemv_w<H, MOE_WG_F32>(a, st);
    else launch_router_gemv_w<H, MOE_WG_F16>(a, st);
}

hipError_t launch_router_gemv(int H, int wtype, const void *wg, const float *x, int M, int E, int rmsnorm,
                              float *logits, int renorm, uint16_t *ids, float *w, hipStream_t st, KernelTimer *T) {
    if (M <= 0) return hipSuccess;
    if (H != 2048 && H != 512) return hipErrorInvalidValue;
    if (wtype != MOE_WG_IQ4_XS && wtype != MOE_WG_F32 && wtype != MOE_WG_F16) return hipErrorInvalidValue;
    if (E < TOPK || E > 256) return hipErrorInvalidValue;
    RouterGemvArgs a{wg, x, M, E, rmsnorm, logits};
    {
        TimedLaunch tl(T, MOE_K_ROUTER_GEMV, st);
        if (H == 2048) launch_router_gemv_h<2048>(wtype, a, st);
        else launch_router_gemv_h<512>(wtype, a, st);
    }
    hipError_t he = hipGetLastError();
    if (he == hipSuccess && ids) he = launch_router_topk(logits, M, E, renorm, ids, w, st, T);
    return he;
}

// ---------------------------------------------------------------- bucket fill
__global__ __launch_bounds__(BF_THREADS) void k_bucket_fill(BucketArgs a) { bucket_fill_one_wg(a); }
__global__ __launch_bounds__(BF_CHUNK_THREADS) void k_bucket_count(BucketArgs a) { bucket_count_chunk(a, blockIdx.x); }
__global__ __launch_bounds__(BF_THREADS) void k_bucket_scan(BucketArgs a) { bucket_scan_wg(a); }
__global__ __launch_bounds__(BF_CHUNK_THREADS) void k_bucket_scatter(BucketArgs a) { bucket_scatter_chunk(a, blockIdx.x); }

hipError_t launch_bucket_fill(const BucketArgs &a, hipStream_t st, KernelTimer *T) {
    if (a.M < 0) return hipSuccess; // M == 0 still writes all-zero ranges
    TimedLaunch tl(T, MOE_K_BUCKET_FILL, st);
    if (bucket_one_wg(a.M, a.E1)) {
        hipLaunchKernelGGL(k_bucket_fill, dim3(1), dim3(BF_THREADS), bucket_smem_one(a.E1, a.M), st, a);
    } else {
        const dim3 grid((unsigned)((a.M + 63) / 64));
        const size_t smem = bucket_chunk_smem(a.E1);
        hipLaunchKernelGGL(k_bucket_count, grid, dim3(BF_CHUNK_THREADS), smem, st, a);
        hipLaunchKernelGGL(k_bucket_scan, dim3(1), dim3(BF_THREADS), bucket_smem(a.E1, false), st, a);
        hipLaunchKernelGGL(k_bucket_scatter, grid, dim3(BF_CHUNK_THREADS), smem, st, a);
    }
    return hipGetLastError();
}

} // namespace moe
