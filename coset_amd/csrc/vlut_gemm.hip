// vlut_gemm.hip -- the vLUT matmul of large batches (whole prompts) on the
// matrix cores, for weights in the decoded formats.
//
// out[t, o] = s_o sum_k a[t, k] x_hat[o, k] with 2 x_hat held as bytes
// (VLUT_DECODED, VLUT_DECODED6).  One workgroup of 8 waves per BT tokens x BR
// rows of the output over the whole K; both operands are staged in LDS, 64 K
// a stage, double-buffered with one LDS-only barrier per stage:
//   activations  [token][8 chunks of 16 bytes], chunk c of token t at
//                c ^ ((t >> 1) & 7): 16 lanes reading one chunk of 16
//                consecutive tokens hit 16 distinct 16-byte bank groups;
//   weights      decoded once per workgroup into fp16 / bf16 MFMA operands in
//                fragment order ([row tile][k-quad][lane]), so their stores
//                and reads are linear.
// A wave multiplies 16 TT tokens x 16 RT rows: the weights are the MFMA's
// first operand, so a lane ends with 4 consecutive output rows of one token.  The loads of stage s + 2 go out while stage s is
// multiplied and their data is stored to LDS in the middle of stage s + 1.
//
// Bound: at 4096 x 4096 x 4096 tokens 1148 TFLOP/s (bf16), the matrix cores at
// the clock the chip holds under them; at 3072 x 768 x 4096 tokens 29.3 us, of
// which the 50 MB of fp32 output take 10 (the deep kernel, which decodes each
// weight for 64 tokens, takes 90.5).  Decoding at the store to LDS costs one
// decode per BT tokens, 20 VALU operations per 8 weights in bf16.  Waves in
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
template <bool BF16, bool D6, int TT, int RT, int WT, int WR>
__global__ void __launch_bounds__(WT * WR * 64) vlut_gemm_kernel(VlutMatmulArgs p, int tiles_r, int tiles)
{
    constexpr int NW = WT * WR;
    constexpr int T = NW * 64;
    constexpr int BT = 16 * TT * WT, BR = 16 * RT * WR;
    constexpr int AL = BT * kGemmChunks / T;          // activation chunks per thread and stage
    constexpr int UW = BR / 16 * 2 / NW;      // (row tile, k-quad) units per wave and stage
    static_assert(AL * T == BT * kGemmChunks && UW * NW == BR / 16 * 2, "whole loads per thread");
    __shared__ uint4 s_lds[2 * (BT * kGemmChunks + BR / 16 * 2 * 64)];
    uint4 (*s_a)[BT * kGemmChunks] = reinterpret_cast<uint4 (*)[BT * kGemmChunks]>(s_lds);
    uint4 (*s_w)[BR / 16 * 2 * 64] = reinterpret_cast<uint4 (*)[BR / 16 * 2 * 64]>(s_lds + 2 * BT * kGemmChunks);

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wt = wave / WR, wr = wave % WR;

    // workgroup b runs on XCD b % 8: each XCD takes a run of consecutive
    // tiles (row tiles fastest), which share activation panels in its L2
    const int b = blockIdx.x, x = b & 7, per = tiles >> 3, rem = tiles & 7;
    const int tile = x * per + min(x, rem) + (b >> 3);
    const int64_t t_base = (int64_t)(tile / tiles_r) * BT;
    const int64_t r_base = (int64_t)(tile % tiles_r) * BR;

    const int64_t kb_total = p.K / 8;
    const int64_t kq_total = (kb_total + 3) / 4;
    const int stages = (int)((kq_total + 1) / 2);
    const bool ragged = (kb_total & 7) != 0;
    const int64_t rt_last = (p.rows + 15) / 16 - 1;
    const int bias = D6 ? p.d6_bias : kVlutDecodedBias;
    const _Float16 f16_off = (_Float16)(1024 + bias);
    const float f32_off = (float)bias;

    // activation chunk i of this thread: token (tid + T i) / 8 (clamped to the
    // last token: those outputs are not stored), chunk tid % 8 of the stage
    const uint16_t* act = reinterpret_cast<const uint16_t*>(p.act);
    const int a_ch = tid & 7;
    const uint16_t* a_src[AL];
#pragma unroll
    for (int i = 0; i < AL; ++i)
        a_src[i] = act + std::min<int64_t>(t_base + ((tid + T * i) >> 3), p.B - 1) * p.K;
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

    uint4 av[AL];
    uint32_t wv[UW][D6 ? 3 : 2];
    auto load = [&](int st) {
        const int64_t kb = std::min<int64_t>((int64_t)st * kGemmChunks + a_ch, kb_total - 1);
#pragma unroll
        for (int i = 0; i < AL; ++i) av[i] = *reinterpret_cast<const uint4*>(a_src[i] + kb * 8);
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
    auto store = [&](int st, int buf) {
        if (ragged && st == stages - 1 && (int64_t)st * kGemmChunks + a_ch >= kb_total) {
            // past K: zero activations (the weights there are x_hat = 0, but 0 x inf is not)
#pragma unroll
            for (int i = 0; i < AL; ++i) av[i] = make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int t = (tid + T * i) >> 3;
            s_a[buf][t * kGemmChunks + (a_ch ^ ((t >> 1) & 7))] = av[i];
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

    float4_t acc[RT][TT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[i][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
    auto read = [&](int buf, int ks, uint4 (&wf)[RT], uint4 (&af)[TT]) {
#pragma unroll
        for (int i = 0; i < RT; ++i) wf[i] = s_w[buf][((wr * RT + i) * 2 + ks) * 64 + lane];
#pragma unroll
        for (int t = 0; t < TT; ++t)
            af[t] = s_a[buf][((wt * TT + t) * 16 + r) * kGemmChunks + ((4 * ks + g) ^ (r >> 1))];
    };
    auto multiply = [&](const uint4 (&wf)[RT], const uint4 (&af)[TT]) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                if (BF16)
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[i]),
                                                                        __builtin_bit_cast(bf16x8_t, af[t]), acc[i][t],
                                                                        0, 0, 0);
                else
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, wf[i]),
                                                                       __builtin_bit_cast(half8_t, af[t]), acc[i][t],
                                                                       0, 0, 0);
            }
    };

    load(0);
    store(0, 0);
    load(std::min(1, stages - 1));
    gemm_lds_barrier();
    for (int st = 0; st < stages; ++st) {
        const int buf = st & 1;
        uint4 w0[RT], a0[TT], w1[RT], a1[TT];
        read(buf, 0, w0, a0);
        if (RT * TT <= 16) read(buf, 1, w1, a1);
        multiply(w0, a0);
        if (st + 1 < stages) {
            store(st + 1, buf ^ 1);
            load(std::min(st + 2, stages - 1));
        }
        if (RT * TT > 16) read(buf, 1, w1, a1);
        multiply(w1, a1);
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
    constexpr int kWaveChunks = (2 * BT * kGemmChunks + 2 * BR / 16 * 2 * 64) / NW;
    constexpr int SW = CP < 16 ? CP - 1 : 15;
    constexpr int kFit = kWaveChunks / (16 * CP);
    constexpr int PT = kFit >= TT ? TT : kFit >= 4 ? 4 : kFit >= 2 ? 2 : 1;
    static_assert(kFit >= 1 && TT % PT == 0, "whole passes");
    float4_t* red = reinterpret_cast<float4_t*>(s_lds) + wave * kWaveChunks;
    const int c = lane & (CP - 1);
    const int64_t o0 = r_base + wr * RT * 16 + 4 * c;
    const bool live = c < 4 * RT && o0 < p.rows;
    const bool v4 = (p.rows & 3) == 0 && ((uintptr_t)p.out & 15) == 0;
    float sc[4], bi[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t o = std::min<int64_t>(o0 + e, p.rows - 1);
        sc[e] = p.scale ? (p.scale_mode == 0 ? p.scale[o] : 1.f / p.scale[o]) : 1.f;
        bi[e] = p.bias ? p.bias[o] : 0.f;
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
        float* dst = p.out + tok0 * p.rows + o0;
        const int n = live ? (int)std::min<int64_t>(std::max<int64_t>((p.B - tok0 + kStep - 1) / kStep, 0), kIter) : 0;
        auto value = [&](int k) {
            const int tl = k * kStep + lane / CP;
            return red[tl * CP + (c ^ (tl & SW))];
        };
        if (v4 && !p.lsq_alpha) {
            // four reads in flight
#pragma unroll 4
            for (int k = 0; k < kIter; ++k) {
                const float4_t v = value(k);
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    y[e] = v[e] * 0.5f * sc[e];
                    if (p.bias) y[e] = __fadd_rn(y[e], bi[e]);
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
                            vlut_epilogue_b(v[e] * 0.5f * sc[e], bi[e], p.bias, p.lsq_alpha, p.lsq_qmax);
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
constexpr GemmShape kGemmShapes[] = {{256, 256, 1.51, 8.3}, {256, 192, 1.26, 8.1}, {128, 128, 0.59, 4.1},
                                     {128, 64, 0.42, 3.5}};

template <bool BF16, bool D6>
hipError_t launch(const VlutMatmulArgs& p, int shape, hipStream_t s)
{
    const GemmShape g = kGemmShapes[shape];
    const int64_t tr = (p.rows + g.br - 1) / g.br, tt = (p.B + g.bt - 1) / g.bt;
    if (tr * tt > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(tr * tt));
    const int n = (int)(tr * tt), r = (int)tr;
    switch (shape) {
#define COSET_GEMM(TT, RT, WT, WR) \
    hipLaunchKernelGGL((vlut_gemm_kernel<BF16, D6, TT, RT, WT, WR>), grid, dim3(WT * WR * 64), 0, s, p, r, n)
    case 0: COSET_GEMM(8, 4, 2, 4); break;
    case 1: COSET_GEMM(8, 3, 2, 4); break;
    case 2: COSET_GEMM(4, 2, 2, 4); break;
    default: COSET_GEMM(2, 2, 4, 2); break;
#undef COSET_GEMM
    }
    return hipGetLastError();
}

}  // namespace

int vlut_gemm_shape(int64_t rows, int64_t B, int64_t K, int cus)
{
    // below two token tiles of the deep kernel its K splits win (64 tokens of
    // 4096 x 4096: 10.8 us against 31)
    if (B <= 2 * kDeepTokens - 1) return -1;
    const int64_t kq = (K / 8 + 3) / 4, stages = (kq + 1) / 2;
    int best = -1;
    double best_us = 0.0;
    for (int i = 0; i < (int)(sizeof(kGemmShapes) / sizeof(kGemmShapes[0])); ++i) {
        const GemmShape& g = kGemmShapes[i];
        const int64_t tiles = ((rows + g.br - 1) / g.br) * ((B + g.bt - 1) / g.bt);
        const double us = g.fixed_us + (double)((tiles + cus - 1) / cus) * (double)stages * g.stage_us;
        if (best < 0 || us < best_us) {
            best = i;
            best_us = us;
        }
    }
    // the deep kernel: 64 x 64 tiles of at most 1024 K, 7.2 us a round of one
    // workgroup per CU (its phases do not overlap), 1.5 us for the reduce of
    // its splits.  bf16, us, deep / this kernel: 768 x 3072 x 256 tokens (the
    // splits fill the chip) 12.0 / 23.7, x 1024 28.5 / 24.0; 3072 x 768 x 256
    // 9.3 / 8.8, x 4096 90.5 / 29.3; 4096 x 4096 x 256 34.0 / 31.2, x 4096
    // 557 / 120 (1148 TFLOP/s; a large bf16 product of the library 1235)
    const int64_t groups = ((rows + kDeepRows - 1) / kDeepRows) * ((B + kDeepTokens - 1) / kDeepTokens);
    const int64_t min_splits = (kq + kDeepKqWg - 1) / kDeepKqWg;
    const int64_t splits = std::max(min_splits, std::min<int64_t>(std::max<int64_t>(1, cus / groups), kq));
    const double deep_us = 2.5 + 7.2 * (double)((groups * splits + cus - 1) / cus) + (splits > 1 ? 1.5 : 0.0);
    return best_us < deep_us ? best : -1;
}

hipError_t vlut_launch_gemm(const VlutMatmulArgs& p, int shape, hipStream_t s)
{
    const bool bf = p.act_dtype == DT_BF16;
    if (p.prepared == VLUT_DECODED6) return bf ? launch<true, true>(p, shape, s) : launch<false, true>(p, shape, s);
    return bf ? launch<true, false>(p, shape, s) : launch<false, false>(p, shape, s);
}

}  // namespace coset
