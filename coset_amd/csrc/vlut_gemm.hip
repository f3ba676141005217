// vlut_gemm.hip -- the vLUT matmul of large batches (whole prompts) on the
// matrix cores, for weights in the decoded formats.
//
// out[t, o] = s_o sum_k a[t, k] x_hat[o, k] with 2 x_hat held as bytes
// (VLUT_DECODED, VLUT_DECODED6).  One workgroup of 8 waves per BT tokens x BR
// rows of the output and K range (the whole K, or K splits whose partials a
// reduce adds); both operands are staged in LDS, 64 K a stage, double-buffered
// with one LDS-only barrier per stage:
//   activations  [token][8 chunks of 16 bytes], chunk c of token t at
//                c ^ ((t >> 1) & 7): 16 lanes reading one chunk of 16
//                consecutive tokens hit 16 distinct 16-byte bank groups;
//   weights      decoded once per workgroup into fp16 / bf16 MFMA operands in
//                fragment order ([row tile][k-quad][lane]), so their stores
//                and reads are linear.
// A wave multiplies 16 TT tokens x 16 RT rows: the weights are the MFMA's
// first operand, so a lane ends with 4 consecutive output rows of one token.
// The loads of stage s + 2 go out while stage s is multiplied and their data is
// stored to LDS in the middle of stage s + 1.
//
// fp32 activations (from 43 tokens): one launch and a reduce, where the planes
// took a split launch, 3B tokens on the deep kernel and a reduce: 197 tokens of
// 768 x 3072 26.6 -> 17.5 us, 48 of 3072 x 768 13.5 -> 10.6, 4096 of 3072 x 768
// 306 -> 86; error against 64 bits (197 of 768 x 3072) 5.8e-8 -> 3.9e-8.  At few
// tokens the time is the latency of the stages (0.9 us each, 64 x 64 tiles) and
// of the reduce.
//
// Bound: at 3072 x 768 x 4096 tokens 38 us on the plan's 128 x 128 tiles, three
// rounds of 256 (the deep kernel, which decodes each weight for 64 tokens, takes
// 104): 464 TFLOP/s in a kernel trace, no LDS bank conflicts, the matrix cores
// busy about a fifth of the time; the rest is the wait for a stage's operands, its
// decode and, last in each round, the stores of 50 MB of fp32 output (10 us).
// The 256 x 256 tiles, forced at 4096 x 4096 x 4096 tokens, reach 1148 TFLOP/s, but
// the plan takes the 256-token tiles up to kOneChainK only.  Decoding at the
// store to LDS costs one decode per BT tokens (128 above kOneChainK), 20 VALU
// operations per 8 weights in bf16.  Waves in
// two groups a phase apart (one loads while the other multiplies) measured the
// same at full load and slower on the smaller shapes; 4 waves of 128 x 128
// do not fit the registers.
#include <algorithm>

#include "vlut_mfma.hpp"

namespace coset {
namespace {

constexpr int kGemmStageK = 64;                       // K per stage: 2 k-quads, 8 chunks of 8 activations
constexpr int kGemmChunks = kGemmStageK / 8;

// all waves' LDS accesses done; global loads and stores stay in flight
__device__ __forceinline__ void gemm_lds_barrier()
{
    __builtin_amdgcn_sched_barrier(0);
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// WT x WR waves (tokens x rows) of TT token tiles x RT row tiles of 16.
// A32: fp32 activations, split at the store to LDS into their three exact bf16
// planes (split3), which share each weight operand; the second and third plane
// (2^-8 and 2^-16 of the first) share an accumulator.  blockIdx.y: K range of `per` stages (partials
// [split][B][rows] of 2 x_hat products; the caller reduces them).
template <bool BF16, bool D6, bool A32, int TT, int RT, int WT, int WR>
__global__ void __launch_bounds__(WT * WR * 64) vlut_gemm_kernel(VlutMatmulArgs p, int tiles_r, int tiles, int per)
{
    static_assert(!A32 || BF16, "fp32 activations run as bf16 planes");
    constexpr int NP = A32 ? 3 : 1;                   // planes
    constexpr int NW = WT * WR;
    constexpr int T = NW * 64;
    constexpr int BT = 16 * TT * WT, BR = 16 * RT * WR;
    constexpr int AL = BT * kGemmChunks / T;          // activation chunks per thread and stage
    constexpr int UW = BR / 16 * 2 / NW;      // (row tile, k-quad) units per wave and stage
    static_assert(AL * T == BT * kGemmChunks && UW * NW == BR / 16 * 2, "whole loads per thread");
    constexpr int kChA = NP * BT * kGemmChunks, kChW = BR / 16 * 2 * 64;   // 16-byte chunks of a stage
    __shared__ uint4 s_lds[2 * (kChA + kChW)];
    uint4 (*s_a)[kChA] = reinterpret_cast<uint4 (*)[kChA]>(s_lds);
    uint4 (*s_w)[kChW] = reinterpret_cast<uint4 (*)[kChW]>(s_lds + 2 * kChA);

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wt = wave / WR, wr = wave % WR;

    // workgroup b runs on XCD b % 8: each XCD takes a run of consecutive
    // tiles (row tiles fastest), which share activation panels in its L2
    const int b = blockIdx.x, x = b & 7, run = tiles >> 3, rem = tiles & 7;
    const int tile = x * run + min(x, rem) + (b >> 3);
    const int64_t t_base = (int64_t)(tile / tiles_r) * BT;
    const int64_t r_base = (int64_t)(tile % tiles_r) * BR;

    const int64_t kb_total = p.K / 8;
    const int64_t kq_total = (kb_total + 3) / 4;
    const int all = (int)((kq_total + 1) / 2), st0 = (int)blockIdx.y * per;
    const int stages = min(per, all - st0);   // >= 1 (the launcher)
    const bool ragged = (kb_total & 7) != 0;
    const int64_t rt_last = (p.rows + 15) / 16 - 1;
    const int bias = D6 ? p.d6_bias : kVlutDecodedBias;
    const _Float16 f16_off = (_Float16)(1024 + bias);
    const float f32_off = (float)bias;

    // activation chunk i of this thread: token (tid + T i) / 8 (clamped to the
    // last token: those outputs are not stored), chunk tid % 8 of the stage
    constexpr int kActBytes = A32 ? 4 : 2;
    const int a_ch = tid & 7;
    const char* a_src[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i)
        a_src[i] = reinterpret_cast<const char*>(p.act) +
                   std::min<int64_t>(t_base + ((tid + T * i) >> 3), p.B - 1) * p.K * kActBytes;
    // weight unit u of this wave: row tile idx / 2 (clamped to the last one),
    // k-quad idx % 2 of the stage
    const uint32_t* w_src[UW];
#pragma unroll
    for (int u = 0; u < UW; ++u) {
        const int idx = wave * UW + u;
        const int64_t rt = std::min<int64_t>(r_base / 16 + (idx >> 1), rt_last);
        w_src[u] = reinterpret_cast<const uint32_t*>(p.words) +
                   vlut_word_index(D6 ? VLUT_DECODED6 : VLUT_DECODED, rt * 16 + r, g + (D6 ? 0 : 4 * (idx & 1)), 0,
                                   kb_total, p.M);
    }

    uint4 av[AL][A32 ? 2 : 1];
    uint32_t wv[UW][D6 ? 3 : 2];
    auto load = [&](int s) {
        const int st = st0 + s;
        const int64_t kb = std::min<int64_t>((int64_t)st * kGemmChunks + a_ch, kb_total - 1);
#pragma unroll
        for (int i = 0; i < AL; ++i)
#pragma unroll
            for (int h = 0; h < (A32 ? 2 : 1); ++h)
                av[i][h] = *reinterpret_cast<const uint4*>(a_src[i] + kb * 8 * kActBytes + 16 * h);
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            if constexpr (D6) {
                // k-quads 2 st, 2 st + 1 of the lane: 12 bytes of its chunk of 8
                const uint32_t* src = w_src[u] + (int64_t)(st >> 2) * 64 * kD6Words + (st & 3) * 3;
                wv[u][0] = src[0];
                wv[u][1] = src[1];
                wv[u][2] = src[2];
            } else {
                const uint2 v = *reinterpret_cast<const uint2*>(w_src[u] + (int64_t)st * 64 * 4);
                wv[u][0] = v.x;
                wv[u][1] = v.y;
            }
        }
    };
    auto store = [&](int s, int buf) {
        const int st = st0 + s;
        if (ragged && st == all - 1 && (int64_t)st * kGemmChunks + a_ch >= kb_total) {
            // past K: zero activations (the weights there are x_hat = 0, but 0 x inf is not)
#pragma unroll
            for (int i = 0; i < AL; ++i)
#pragma unroll
                for (int h = 0; h < (A32 ? 2 : 1); ++h) av[i][h] = make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int t = (tid + T * i) >> 3;
            const int at = t * kGemmChunks + (a_ch ^ ((t >> 1) & 7));
            if constexpr (A32) {
                const uint32_t w[8] = {av[i][0].x, av[i][0].y, av[i][0].z, av[i][0].w,
                                       av[i][1].x, av[i][1].y, av[i][1].z, av[i][1].w};
                uint32_t h[3][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint16_t lo[3], hi[3];
                    split3(__uint_as_float(w[2 * j]), lo[0], lo[1], lo[2]);
                    split3(__uint_as_float(w[2 * j + 1]), hi[0], hi[1], hi[2]);
#pragma unroll
                    for (int q = 0; q < 3; ++q) h[q][j] = (uint32_t)lo[q] | ((uint32_t)hi[q] << 16);
                }
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    s_a[buf][q * BT * kGemmChunks + at] = make_uint4(h[q][0], h[q][1], h[q][2], h[q][3]);
            } else {
                s_a[buf][at] = av[i][0];
            }
        }
#pragma unroll
        for (int u = 0; u < UW; ++u) {
            const int idx = wave * UW + u;
            uint32_t x0, x1;
            if constexpr (D6) {
                uint32_t y0, y1;
                d6_bytes(wv[u][0], wv[u][1], x0, x1);
                d6_bytes(__builtin_amdgcn_alignbit(wv[u][2], wv[u][1], 16), wv[u][2] >> 16, y0, y1);
                x0 = idx & 1 ? y0 : x0;
                x1 = idx & 1 ? y1 : x1;
            } else {
                x0 = wv[u][0];
                x1 = wv[u][1];
            }
            s_w[buf][idx * 64 + lane] = bytes_to_operand<BF16>(x0, x1, f16_off, f32_off);
        }
    };

    // kTwo: sums in two steps -- every 256 K the products' accumulator is added to
    // a total and cleared -- so the error stays that of the deep kernel's short
    // chains (768 x 3072 fp32: 6.1e-8 against 64 bits, 7.8e-8 in one chain).  The
    // 256-token shapes have no registers for it; the plan gives them up to
    // kOneChainK.
    constexpr bool kTwo = A32 || RT * TT <= 8;
    constexpr int NA = A32 ? 2 : 1;
    float4_t acc[RT][NA * TT];   // token tile t; A32: the lower planes at TT + t
    float4_t total[kTwo ? RT : 1][kTwo ? TT : 1];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < NA * TT; ++t) {
            acc[i][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
            if (kTwo && t < TT) total[i][t] = acc[i][t];
        }
    auto read = [&](int buf, int ks, uint4 (&wf)[RT], uint4 (&af)[NP * TT]) {
#pragma unroll
        for (int i = 0; i < RT; ++i) wf[i] = s_w[buf][((wr * RT + i) * 2 + ks) * 64 + lane];
#pragma unroll
        for (int t = 0; t < NP * TT; ++t)
            af[t] = s_a[buf][((t / TT) * BT + (wt * TT + t % TT) * 16 + r) * kGemmChunks + ((4 * ks + g) ^ (r >> 1))];
    };
    auto multiply = [&](const uint4 (&wf)[RT], const uint4 (&af)[NP * TT]) {
#pragma unroll
        for (int t = 0; t < NP * TT; ++t)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                float4_t& c = acc[i][(t >= TT ? TT : 0) + t % TT];
                if (BF16)
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[i]),
                                                                __builtin_bit_cast(bf16x8_t, af[t]), c, 0, 0, 0);
                else
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, wf[i]),
                                                               __builtin_bit_cast(half8_t, af[t]), c, 0, 0, 0);
            }
    };

    load(0);
    store(0, 0);
    load(std::min(1, stages - 1));
    gemm_lds_barrier();
    for (int st = 0; st < stages; ++st) {
        const int buf = st & 1;
        uint4 w0[RT], a0[NP * TT], w1[RT], a1[NP * TT];
        constexpr bool kAhead = NP * RT * TT <= 16;
        read(buf, 0, w0, a0);
        if (kAhead) read(buf, 1, w1, a1);
        multiply(w0, a0);
        if (st + 1 < stages) {
            store(st + 1, buf ^ 1);
            load(std::min(st + 2, stages - 1));
        }
        if (!kAhead) read(buf, 1, w1, a1);
        multiply(w1, a1);
        if (kTwo && (st & 3) == 3) {
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    total[i][t] += acc[i][t];
                    acc[i][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
                }
        }
        gemm_lds_barrier();
    }

    // Epilogue: each wave turns its tile round in LDS of its own (the last
    // barrier has freed the stages), PT token tiles at a time -- lane (g, r)
    // holds rows 16 i + 4 g .. + 3 of token 16 t + r; chunk c = 4 i + g (4
    // rows) of a token's row lies at c ^ (token % CP) -- and reads it back
    // with the chunks of a token in consecutive lanes, so the stores write
    // 64 RT consecutive bytes per token and a lane keeps the same 4 rows'
    // scale and bias throughout.  The loop is not unrolled: straight-line code
    // for every element of the tile is bound by instruction fetch.
    constexpr int CP = RT <= 1 ? 4 : RT == 2 ? 8 : RT <= 4 ? 16 : 32;   // chunks per token, padded
    if constexpr (kTwo) {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                acc[i][t] = total[i][t] + acc[i][t];
                if (A32) acc[i][t] += acc[i][(NA - 1) * TT + t];
            }
    }
    constexpr int kWaveChunks = 2 * (kChA + kChW) / NW;
    constexpr int SW = CP < 16 ? CP - 1 : 15;
    constexpr int kFit = kWaveChunks / (16 * CP);
    constexpr int PT = kFit >= TT ? TT : kFit >= 4 ? 4 : kFit >= 2 ? 2 : 1;
    static_assert(kFit >= 1 && TT % PT == 0, "whole passes");
    float4_t* red = reinterpret_cast<float4_t*>(s_lds) + wave * kWaveChunks;
    const int c = lane & (CP - 1);
    const int64_t o0 = r_base + wr * RT * 16 + 4 * c;
    const bool live = c < 4 * RT && o0 < p.rows;
    // with K splits the partials leave as they are (the reduce halves, scales
    // and adds the bias); otherwise the output
    const bool whole = gridDim.y == 1;
    float* out = whole ? p.out : p.partial + (int64_t)blockIdx.y * p.B * p.rows;
    const float* add = whole ? p.bias : nullptr;
    const float* lsq_alpha = whole ? p.lsq_alpha : nullptr;
    const float half = whole ? 0.5f : 1.f;
    const bool v4 = (p.rows & 3) == 0 && ((uintptr_t)out & 15) == 0;
    float sc[4], bi[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t o = std::min<int64_t>(o0 + e, p.rows - 1);
        sc[e] = whole && p.scale ? (p.scale_mode == 0 ? p.scale[o] : 1.f / p.scale[o]) : 1.f;
        bi[e] = add ? add[o] : 0.f;
    }
#pragma unroll
    for (int t0 = 0; t0 < TT; t0 += PT) {
#pragma unroll
        for (int t = 0; t < PT; ++t)
#pragma unroll
            for (int i = 0; i < RT; ++i) red[(16 * t + r) * CP + ((4 * i + g) ^ (r & SW))] = acc[i][t0 + t];
        // a wave's LDS operations complete in order: no barrier
        __asm__ volatile("" ::: "memory");
        constexpr int kIter = 16 * PT * CP / 64, kStep = 64 / CP;   // tokens per store
        const int64_t tok0 = t_base + (wt * TT + t0) * 16 + lane / CP;
        float* dst = out + tok0 * p.rows + o0;
        const int n = live ? (int)std::min<int64_t>(std::max<int64_t>((p.B - tok0 + kStep - 1) / kStep, 0), kIter) : 0;
        auto value = [&](int k) {
            const int tl = k * kStep + lane / CP;
            return red[tl * CP + (c ^ (tl & SW))];
        };
        if (v4 && !lsq_alpha) {
            // four reads in flight
#pragma unroll 4
            for (int k = 0; k < kIter; ++k) {
                const float4_t v = value(k);
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    y[e] = v[e] * half * sc[e];
                    if (add) y[e] = __fadd_rn(y[e], bi[e]);
                }
                if (k < n)
                    *reinterpret_cast<float4*>(dst + (int64_t)k * kStep * p.rows) = make_float4(y[0], y[1], y[2], y[3]);
            }
        } else {
#pragma unroll 1
            for (int k = 0; k < n; ++k) {
                const float4_t v = value(k);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (o0 + e < p.rows)
                        dst[(int64_t)k * kStep * p.rows + e] =
                            vlut_epilogue_b(v[e] * half * sc[e], bi[e], add, lsq_alpha, p.lsq_qmax);
            }
        }
        __asm__ volatile("" ::: "memory");
    }
}

// Tile shapes (tokens x rows) with the time of one 64-K stage of one workgroup
// and of everything around the stages (launch, first loads, epilogue), both
// in us, measured at 768 and 3072 K with fewer workgroups than CUs.  Two
// workgroups of a smaller shape on one CU take twice the stage time.
struct GemmShape {
    int bt, br;
    double stage_us, fixed_us;
};
// The most K that the 256-token tiles, whose sums are one chain, take: above,
// their error against 64 bits is larger than the deep kernel's (fp16, 1000 K
// 7.7e-8 against 6.7e-8, 128 x 128 tiles 6.5e-8; bf16, 768 K 5.1e-8, 5.0e-8,
// 5.0e-8), though 4096 tokens of 3072 x 768 take 29 us on them and 38 on 128 x
// 128.  Up to it they serve large outputs: 8192 tokens of 8192 x 256 77 us against
// 100 on 128 x 128 tiles, 16384 of 4096 x 128 63 / 85, 8192 of 3072 x 256 32 / 37
constexpr int64_t kOneChainK = 256;
constexpr GemmShape kGemmShapes[] = {{256, 256, 1.51, 8.3}, {256, 192, 1.26, 8.1}, {128, 128, 0.61, 4.1},
                                     {128, 64, 0.43, 3.5}};

constexpr GemmShape kGemmShapes32[] = {{128, 128, 1.98, 4.3}, {64, 128, 1.1, 3.7}, {64, 64, 0.9, 3.3}};

template <bool BF16, bool D6, bool A32>
hipError_t launch(const VlutMatmulArgs& p, int shape, int splits, hipStream_t s)
{
    const GemmShape g = A32 ? kGemmShapes32[shape] : kGemmShapes[shape];
    const int64_t tr = (p.rows + g.br - 1) / g.br, tt = (p.B + g.bt - 1) / g.bt;
    const int64_t all = ((p.K / 8 + 3) / 4 + 1) / 2;   // stages
    const int per = (int)((all + splits - 1) / splits);
    if (tr * tt > 0x7fffffff || splits < 1 || splits > 65535 || (int64_t)per * (splits - 1) >= all)
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)(tr * tt), (unsigned)splits);
    const int n = (int)(tr * tt), r = (int)tr;
#define COSET_GEMM(TT, RT, WT, WR) \
    hipLaunchKernelGGL((vlut_gemm_kernel<BF16, D6, A32, TT, RT, WT, WR>), grid, dim3(WT * WR * 64), 0, s, p, r, n, per)
    if constexpr (A32) {
        switch (shape) {
        case 0: COSET_GEMM(4, 2, 2, 4); break;
        case 1: COSET_GEMM(2, 2, 2, 4); break;
        default: COSET_GEMM(2, 1, 2, 4); break;
        }
    } else {
        switch (shape) {
        case 0: COSET_GEMM(8, 4, 2, 4); break;
        case 1: COSET_GEMM(8, 3, 2, 4); break;
        case 2: COSET_GEMM(4, 2, 2, 4); break;
        default: COSET_GEMM(2, 2, 4, 2); break;
        }
    }
#undef COSET_GEMM
    return hipGetLastError();
}

}  // namespace

// The fastest (shape, splits) of a shape table by its measured costs; splits
// up to max_splits, each of at least two stages; a reduce costs reduce_us (launch
// gap and prologue; 4.5 us fits the 16-bit calls, 3.5 the fp32 ones, whose stages
// are longer) and its traffic at 6 TB/s.
template <int N>
double best_gemm(const GemmShape (&shapes)[N], double reduce_us, int64_t rows, int64_t B, int64_t K, int cus,
                 int64_t max_splits, VlutPlan* best)
{
    const int64_t all = ((K / 8 + 3) / 4 + 1) / 2;
    double best_us = 1e30;
    for (int i = 0; i < N; ++i) {
        const GemmShape& g = shapes[i];
        if (K > kOneChainK && g.bt > 128) continue;
        const int64_t tiles = ((rows + g.br - 1) / g.br) * ((B + g.bt - 1) / g.bt);
        for (int64_t sp = 1; sp <= max_splits && sp <= 64; ++sp) {
            const int64_t per = (all + sp - 1) / sp;
            if (sp > 1 && (per < 2 || per * (sp - 1) >= all)) continue;
            const double us = g.fixed_us + (double)((tiles * sp + cus - 1) / cus) * (double)per * g.stage_us +
                              (sp > 1 ? reduce_us + (double)(sp + 1) * (double)(B * rows) * 4.0 / 6.0e6 : 0.0);
            if (us < best_us) {
                best_us = us;
                *best = {VK_MFMA_GEMM, (int)sp, i};
            }
        }
    }
    return best_us;
}

VlutPlan vlut_gemm_plan(int64_t rows, int64_t B, int64_t K, int cus)
{
    const VlutPlan none{VK_MFMA_DEEP, 0, -1};
    // below two token tiles of the deep kernel its K splits win (64 tokens of
    // 4096 x 4096: 10.8 us against 31)
    if (B <= 2 * kDeepTokens - 1) return none;
    // the deep kernel: 64 x 64 tiles of at most 1024 K, 7.2 us a round of one
    // workgroup per CU (its phases do not overlap), and every XCD reads the
    // activations, which few rows of many tokens wait for (2000 tokens of 512 x 2048
    // 25 us, two rounds; this kernel 18.5).  The reduce of its splits takes 0.8 us
    // where each XCD reads the partials its own workgroups wrote (rows a multiple of
    // 8 groups of 64), else 2.0.  With these costs the choice is within 2.5 % of the
    // faster kernel at all but 8 of 806 measured calls replayed from a graph
    // (256..4096 x 256..4096, 128 to 8192 tokens, bf16 and fp16; the worst 10 % off).
    // A split deep call is charged 1.5 us more against an unsplit one of this kernel:
    // an eager call waits for the host, which takes 14 us for two launches and 9.5
    // for one.  That decides 40 of the calls, by up to 15 % for the slower kernel
    // in a graph and 26 % for the faster one outside (2048 x 1000 x 160: 9.7 / 10.6).
    // bf16, us, deep / this kernel, in a graph: 768 x 3072 x 160 tokens (the splits
    // fill the chip) 11.4 / 12.4, x 512 18.4 / 15.6, x 1024 28.5 / 20.3; 768 x 768 x 160
    // 11.3 / 8.7; 3072 x 768 x 4096 103.9 / 38.1; 4096 x 4096 x 256 34.3 / 22.5, x 4096
    // 557 / 157 on 128 x 128 tiles (120 on 256 x 256, which sum 4096 K in one chain)
    const int64_t kq = (K / 8 + 3) / 4;
    const int64_t groups = ((rows + kDeepRows - 1) / kDeepRows) * ((B + kDeepTokens - 1) / kDeepTokens);
    const int64_t min_splits = (kq + kDeepKqWg - 1) / kDeepKqWg;
    const int64_t splits = std::max(min_splits, std::min<int64_t>(std::max<int64_t>(1, cus / groups), kq));
    const double reduce_us = splits == 1 ? 0.0 : rows % (8 * kDeepRows) == 0 ? 0.8 : 2.0;
    const double reads_us = 8.0 * (double)(B * K) * 2.0 / 33.0e6;
    const double deep_us = 1.3 + 7.2 * (double)((groups * splits + cus - 1) / cus) + reads_us + reduce_us;
    // workspaces are sized for the deep plan's splits
    VlutPlan best;
    const double us = best_gemm(kGemmShapes, 4.5, rows, B, K, cus, splits, &best);
    return us < deep_us + (splits > 1 && best.splits == 1 ? 1.5 : 0.0) ? best : none;
}

VlutPlan vlut_gemm32_plan(int64_t rows, int64_t B, int64_t K, int cus, int64_t max_splits)
{
    VlutPlan best{VK_MFMA_GEMM, 1, 0};
    best_gemm(kGemmShapes32, 3.5, rows, B, K, cus, max_splits, &best);
    return best;
}

hipError_t vlut_launch_gemm(const VlutMatmulArgs& p, const VlutPlan& plan, hipStream_t s)
{
    if (plan.splits > 1 && !p.partial) return hipErrorInvalidValue;
    const bool d6 = p.prepared == VLUT_DECODED6;
    if (p.act_dtype == DT_F32)
        return d6 ? launch<true, true, true>(p, plan.shape, plan.splits, s)
                  : launch<true, false, true>(p, plan.shape, plan.splits, s);
    const bool bf = p.act_dtype == DT_BF16;
    if (d6)
        return bf ? launch<true, true, false>(p, plan.shape, plan.splits, s)
                  : launch<false, true, false>(p, plan.shape, plan.splits, s);
    return bf ? launch<true, false, false>(p, plan.shape, plan.splits, s)
              : launch<false, false, false>(p, plan.shape, plan.splits, s);
}

}  // namespace coset
