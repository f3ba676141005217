// gemm_wgrad.hip -- dW_q = gy^T x for the shapes gemm_tn.hip's one-round grid
// does not take: many tokens, ragged token counts, wide layers (the QAT
// layer's F.linear, coset/core/layers.py:478, whose autograd runs this
// product in the reference).
//
// C[M, N] = A^T B, A [K, M] and B [K, N] bf16 with the token dimension K
// outermost.  One workgroup of 8 waves per BM x BN outputs and K range (split
// K: fp32 partials that a second kernel adds in split order), 64 tokens a
// stage, double-buffered in LDS with one LDS-only barrier per stage.  A thread
// loads an 8 x 8 block (16 bytes of 8 tokens), turns it round in registers
// (32 v_perm) and stores 8 tokens of each of its 8 columns as one 16-byte MFMA
// operand chunk: [16-column tile][32 tokens][(token / 8 % 4) * 16 + column],
// the column xor-ed with its tile's number so that the 16 lanes of a store
// (8 tiles, 2 columns each) hit 16 distinct bank groups; the operand reads
// are then linear.  B is the MFMA's first operand, so a lane ends with 4
// consecutive columns of one row of C.
//
// Column sums of A (the bias gradient) come from the same LDS operands: one
// more MFMA per operand with a first operand of ones, each K stage's by the
// workgroup of one column tile in turn, so every workgroup adds 1 / tiles_n of
// them; the partials [splits * tiles_n][M] are added in order, compensated.
//
// Bound: the main loop reaches 1.0 PFLOP/s of the 1.24 a large library product
// holds on this chip (LDS operand reads and the turning share the issue slots
// with the MFMAs: taking the loads' 64-bit address arithmetic and a modulo out
// of the loop gave 8 %).  16384 tokens x 768 x 3072 with the column sums: 88 us
// (4 splits of 64 tiles, ~9 of them the reduce), against 149 us for the library's
// product and 14 for coset_colsum; 8192 x 3072 x 3072: 156 against 153 + 14.
// 256 x 256 tiles spill (the turning blocks beside 128 accumulators).
#include <algorithm>

#include "gemm.hpp"
#include "rounding.hpp"

namespace coset {
namespace {

typedef __bf16 bf16x8_gw __attribute__((ext_vector_type(8)));
typedef float f32x4_gw __attribute__((ext_vector_type(4)));

constexpr int kGwWaves = 8;
constexpr int kGwT = kGwWaves * 64;
constexpr int kGwStage = 64;            // tokens per stage

__device__ __forceinline__ void gw_barrier()
{
    __builtin_amdgcn_sched_barrier(0);
    __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

struct GwArgs {
    const uint16_t *A, *B;
    int64_t lda, ldb;
    void* C;            // OUT 0 fp32, 1 bf16 [M, ldc] (one split), 2 fp32 partials [splits][M][N]
    int64_t ldc, M, N, K;
    int tiles_m, tiles_n, splits, stages;   // stages per split
    float* colsum;      // partials [splits * tiles_n][M], or null
};

// TM x TN tiles of 16 x 16 per wave, WM x WN waves
template <int OUT, int TM, int TN, int WM, int WN>
__global__ void __launch_bounds__(kGwT, 2) gemm_wgrad_kernel(GwArgs p)
{

    static_assert(WM * WN == kGwWaves, "waves");
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    static_assert(BM % 64 == 0 && BN % 64 == 0 && BM + BN <= kGwT, "a wave loads blocks of one operand");
    constexpr int kChA = BM * 8, kCh = (BM + BN) * 8;   // 16-byte chunks per stage
    __shared__ uint4 s_lds[2 * kCh];

    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, r = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;

    // workgroup b runs on XCD b % 8; each XCD takes a run of consecutive
    // (split, tile) pairs, the tiles ordered in bands of 4 row tiles so that a
    // run shares operand panels
    const int tiles = p.tiles_m * p.tiles_n, total = tiles * p.splits;
    const int b = blockIdx.x, x = b & 7, per = total >> 3, rem = total & 7;
    const int id = x * per + min(x, rem) + (b >> 3);
    const int split = id / tiles, tile = id % tiles;
    const int band = tile / (4 * p.tiles_n), in_band = tile % (4 * p.tiles_n);
    const int band_m = min(4, p.tiles_m - 4 * band);
    const int tm = 4 * band + in_band % band_m, tn = in_band / band_m;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int64_t st0 = (int64_t)split * p.stages;
    const int64_t st_all = (p.K + kGwStage - 1) / kGwStage;
    const int stages = (int)std::min<int64_t>(p.stages, st_all - st0);   // >= 1 (the plan)

    // this thread's block: operand by wave, columns 8 mo .. + 7 of the tile
    // (clamped to the matrix: those outputs are not stored), tokens 8 ko .. + 7
    const bool is_a = wave < BM / 64, loads = wave < (BM + BN) / 64;
    const int blk = is_a ? tid : tid - BM;
    const int octets = (is_a ? BM : BN) / 8;
    const int mo = blk % octets, ko = (blk / octets) & 7;
    const int64_t ld = is_a ? p.lda : p.ldb;
    const int64_t col = std::min<int64_t>((is_a ? m0 : n0) / 8 + mo, (is_a ? p.M : p.N) / 8 - 1) * 8;
    const uint16_t* src = (is_a ? p.A : p.B) + col;
    const char* base = reinterpret_cast<const char*>(is_a ? p.A : p.B);
    const uint32_t lane_off = (uint32_t)((8 * ko * ld + col) * 2);   // pitches up to 2^24 (the entry point refuses more)
    // chunk of column 8 (mo % 2) + j of tile mo / 2
    uint4* dst = s_lds + (is_a ? 0 : kChA) + ((mo >> 1) * 2 + (ko >> 2)) * 64 + (ko & 3) * 16;
    const int c0 = 8 * (mo & 1), sw = (mo >> 1) & 15;

    // stages st and st + 1 in flight in two register sets
    uint4 va[8], vb[8];
    auto load = [&](int st, uint4 (&v)[8]) {
        if (!loads) return;
        const int64_t k0 = (st0 + st) * kGwStage + 8 * ko;
        if ((st0 + st + 1) * kGwStage <= p.K) {
            // uniform row addresses, one 32-bit offset per lane
            const char* row = base + (st0 + st) * kGwStage * ld * 2;
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const uint4*>(row + j * ld * 2 + lane_off);
        } else {
            // tokens past K: the last one instead, zeroed at the store
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = *reinterpret_cast<const uint4*>(src + std::min<int64_t>(k0 + j, p.K - 1) * ld);
        }
    };
    auto store = [&](int st, int buf, uint4 (&v)[8]) {
        if (!loads) return;
        if ((st0 + st + 1) * kGwStage > p.K) {
            const int64_t k0 = (st0 + st) * kGwStage + 8 * ko;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (k0 + j >= p.K) v[j] = make_uint4(0u, 0u, 0u, 0u);
        }
        uint4* d = dst + buf * kCh;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t sel = j & 1 ? 0x07060302u : 0x05040100u;
            const uint32_t* w = reinterpret_cast<const uint32_t*>(v) + (j >> 1);
            d[(c0 + j) ^ sw] = make_uint4(__builtin_amdgcn_perm(w[4], w[0], sel), __builtin_amdgcn_perm(w[12], w[8], sel),
                                          __builtin_amdgcn_perm(w[20], w[16], sel),
                                          __builtin_amdgcn_perm(w[28], w[24], sel));
        }
    };

    f32x4_gw acc[TN][TM], cs[TM];
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        cs[j] = (f32x4_gw){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < TN; ++i) acc[i][j] = (f32x4_gw){0.f, 0.f, 0.f, 0.f};
    }
    const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    auto read = [&](int buf, int ks, uint4 (&fa)[TM], uint4 (&fb)[TN]) {
#pragma unroll
        for (int i = 0; i < TN; ++i) {
            const int t = wn * TN + i;
            fb[i] = s_lds[buf * kCh + kChA + (t * 2 + ks) * 64 + g * 16 + (r ^ (t & 15))];
        }
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int t = wm * TM + j;
            fa[j] = s_lds[buf * kCh + (t * 2 + ks) * 64 + g * 16 + (r ^ (t & 15))];
        }
    };
    auto multiply = [&](const uint4 (&fa)[TM], const uint4 (&fb)[TN], bool sums) {
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int i = 0; i < TN; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_gw, fb[i]),
                                                                    __builtin_bit_cast(bf16x8_gw, fa[j]), acc[i][j], 0,
                                                                    0, 0);
        if (sums) {
#pragma unroll
            for (int j = 0; j < TM; ++j)
                cs[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_gw, ones),
                                                                __builtin_bit_cast(bf16x8_gw, fa[j]), cs[j], 0, 0, 0);
        }
    };

    const int last = stages - 1;
    load(0, va);
    load(min(1, last), vb);
    store(0, 0, va);
    load(min(2, last), va);
    gw_barrier();
    const bool with_sums = p.colsum && wn == 0;
    int turn = (int)((tn - st0 % p.tiles_n + p.tiles_n) % p.tiles_n);   // stages until this tile's next column sums
    // stage st from buffer st & 1; st + 1 (register set `v`) goes to the other
    // buffer, and st + 3 into the registers that leaves
    auto stage = [&](int st, int buf, uint4 (&v)[8]) {
        const bool sums = with_sums && turn == 0;
        turn = turn == 0 ? p.tiles_n - 1 : turn - 1;
        uint4 fa0[TM], fb0[TN], fa1[TM], fb1[TN];
        read(buf, 0, fa0, fb0);
        if (TM * TN <= 8) read(buf, 1, fa1, fb1);
        multiply(fa0, fb0, sums);
        if (st < last) {
            store(st + 1, buf ^ 1, v);
            load(min(st + 3, last), v);
        }
        if (TM * TN > 8) read(buf, 1, fa1, fb1);
        multiply(fa1, fb1, sums);
        gw_barrier();
    };
    for (int st = 0; st < stages; st += 2) {
        stage(st, 0, vb);
        if (st + 1 < stages) stage(st + 1, 1, va);
    }

    // D[column 4 g + e][row r]: the wave's tile turned round in LDS of its own,
    // PM row tiles at a time (chunk c = 4 columns of a row at c ^ (row % CP))
    constexpr int CP = TN <= 1 ? 4 : TN == 2 ? 8 : 16;
    constexpr int kWaveChunks = 2 * kCh / kGwWaves;
    constexpr int kFit = kWaveChunks / (16 * CP);
    constexpr int PM = kFit >= TM ? TM : (TM % 4 == 0 && kFit >= 4) ? 4 : (TM % 3 == 0 && kFit >= 3) ? 3 : kFit >= 2 ? 2 : 1;
    static_assert(kFit >= 1 && TM % PM == 0, "whole passes");
    f32x4_gw* red = reinterpret_cast<f32x4_gw*>(s_lds) + wave * kWaveChunks;
    const int c = lane & (CP - 1);
    const int64_t nc = n0 + wn * TN * 16 + 4 * c;
    const bool live = c < 4 * TN && nc < p.N;
    float* cf = static_cast<float*>(p.C) + (OUT == 2 ? (int64_t)split * p.M * p.N : 0);
    uint16_t* ch = static_cast<uint16_t*>(p.C);
    const int64_t ldc = OUT == 2 ? p.N : p.ldc;
#pragma unroll
    for (int j0 = 0; j0 < TM; j0 += PM) {
#pragma unroll
        for (int j = 0; j < PM; ++j)
#pragma unroll
            for (int i = 0; i < TN; ++i) red[(16 * j + r) * CP + ((4 * i + g) ^ (r & (CP - 1)))] = acc[i][j0 + j];
        __asm__ volatile("" ::: "memory");   // a wave's LDS operations complete in order
        constexpr int kIter = 16 * PM * CP / 64, kStep = 64 / CP;
        const int64_t row0 = m0 + (wm * TM + j0) * 16 + lane / CP;
#pragma unroll 4
        for (int k = 0; k < kIter; ++k) {
            const int rl = k * kStep + lane / CP;
            const f32x4_gw y = red[rl * CP + (c ^ (rl & (CP - 1)))];
            const int64_t row = row0 + k * kStep;
            if (live && row < p.M) {
                if (OUT == 1)
                    *reinterpret_cast<uint2*>(ch + row * ldc + nc) = make_uint2(pack_bf16(y[0], y[1]), pack_bf16(y[2], y[3]));
                else
                    *reinterpret_cast<float4*>(cf + row * ldc + nc) = make_float4(y[0], y[1], y[2], y[3]);
            }
        }
        __asm__ volatile("" ::: "memory");
    }
    if (p.colsum && wn == 0 && g == 0) {
        float* out = p.colsum + ((int64_t)split * p.tiles_n + tn) * p.M;
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int64_t row = m0 + (wm * TM + j) * 16 + r;
            if (row < p.M) out[row] = cs[j][0];
        }
    }
}

// C = sum over splits of the partials [splits][M][N] in split order (8
// outputs a thread), then colsum = sum over its parts [parts][M] in order.
// splits = 0: C is written already.
template <int OUT>
__global__ void __launch_bounds__(256) gemm_wgrad_reduce_kernel(const float* __restrict__ part, int splits, int64_t M,
                                                                int64_t N, void* __restrict__ C, int64_t ldc,
                                                                const float* __restrict__ cs_part, int cs_parts,
                                                                float* __restrict__ colsum)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t n8 = splits > 0 ? M * N / 8 : 0, pad = (n8 + 255) / 256 * 256;
    if (i >= pad) {
        const int64_t m = i - pad;
        if (!colsum || m >= M) return;
        // compensated: up to splits * tiles_n parts, added in turn
        // 9.8e-8 against 64 bits at 16384 tokens where coset_colsum has 7.0e-8
        float s = 0.f, low = 0.f;
#pragma unroll 16
        for (int k = 0; k < cs_parts; ++k) two_sum(s, low, cs_part[k * M + m]);
        colsum[m] = two_sum_value(s, low);
        return;
    }
    if (i >= n8) return;
    f32x4_gw a = {0.f, 0.f, 0.f, 0.f}, b = a;
    const f32x4_gw* src = reinterpret_cast<const f32x4_gw*>(part) + 2 * i;
    for (int s = 0; s < splits; ++s) {
        a += src[0];
        b += src[1];
        src += M * N / 4;
    }
    const int64_t o = (8 * i / N) * ldc + 8 * i % N;
    if (OUT == 1) {
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(C) + o) =
            make_uint4(pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]),
                       pack_bf16(b[2], b[3]));
    } else {
        f32x4_gw* d = reinterpret_cast<f32x4_gw*>(static_cast<float*>(C) + o);
        d[0] = a;
        d[1] = b;
    }
}

// Tile shapes with the time of one 64-token stage of a workgroup and of
// everything around the stages, us, fitted to 768 x 3072 at 4096 and 16384
// tokens (192) and 768 x 768 (128); a reduce costs 3 us and its traffic at 6 TB/s.
struct GwShape {
    int bm, bn;
    double stage_us, fixed_us;
};
constexpr GwShape kGwShapes[] = {{192, 192, 1.07, 7.6}, {128, 128, 0.66, 7.0}};

}  // namespace

int g_gemm_wgrad = 1;

GemmWgradPlan gemm_wgrad_plan(int64_t M, int64_t N, int64_t K)
{
    GemmWgradPlan best{-1, 0, 0, 0, 0};
    if (M < 8 || N < 8 || K < 1 || M % 8 || N % 8) return best;
    const int64_t st = (K + kGwStage - 1) / kGwStage;
    double best_us = 0.0;
    for (int i = 0; i < (int)(sizeof(kGwShapes) / sizeof(kGwShapes[0])); ++i) {
        if (g_gemm_wgrad >= 2 && g_gemm_wgrad - 2 != i) continue;
        const GwShape& s = kGwShapes[i];
        const int64_t tm = (M + s.bm - 1) / s.bm, tn = (N + s.bn - 1) / s.bn, tiles = tm * tn;
        if (tiles > (1 << 20)) continue;   // the grid stays below 2^31
        for (int64_t sp = 1; sp <= 32 && sp <= st; ++sp) {
            const int64_t per = (st + sp - 1) / sp;
            if ((st + per - 1) / per != sp) continue;   // no empty split
            const double rounds = (double)((tiles * sp + 255) / 256);
            const double us = rounds * (s.fixed_us + (double)per * s.stage_us) +
                              (sp > 1 ? 3.0 + (double)(sp + 1) * (double)(M * N) * 4.0 / 6.0e6 : 0.0);
            if (best.shape < 0 || us < best_us) {
                best_us = us;
                best = {i, (int)tm, (int)tn, (int)sp, (int)per};
            }
        }
    }
    return best;
}

int64_t gemm_wgrad_workspace_floats(const GemmWgradPlan& p, int64_t M, int64_t N)
{
    if (p.shape < 0) return 0;
    return (p.splits > 1 ? (int64_t)p.splits * M * N : 0) + (int64_t)p.splits * p.tiles_n * M;
}

hipError_t gemm_wgrad_bf16(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb, void* C, int64_t ldc,
                           int out_bf16, int64_t M, int64_t N, int64_t K, const GemmWgradPlan& plan, float* workspace,
                           float* colsum, hipStream_t s)
{
    if (plan.shape < 0 || !workspace) return hipErrorInvalidValue;
    const bool split = plan.splits > 1;
    float* cs_part = workspace + (split ? (int64_t)plan.splits * M * N : 0);
    GwArgs p{A, B, lda, ldb, split ? (void*)workspace : C, ldc, M, N, K, plan.tiles_m, plan.tiles_n, plan.splits,
             plan.stages, colsum ? cs_part : nullptr};
    const dim3 grid((unsigned)(plan.tiles_m * plan.tiles_n * plan.splits)), block(kGwT);
#define COSET_GW(TM, TN, WM, WN)                                                                        \
    if (split) hipLaunchKernelGGL((gemm_wgrad_kernel<2, TM, TN, WM, WN>), grid, block, 0, s, p);         \
    else if (out_bf16) hipLaunchKernelGGL((gemm_wgrad_kernel<1, TM, TN, WM, WN>), grid, block, 0, s, p); \
    else hipLaunchKernelGGL((gemm_wgrad_kernel<0, TM, TN, WM, WN>), grid, block, 0, s, p);
    if (plan.shape == 0) {
        COSET_GW(6, 3, 2, 4)
    } else {
        COSET_GW(4, 2, 2, 4)
    }
#undef COSET_GW
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || (!split && !colsum)) return e;
    const int64_t n8 = split ? M * N / 8 : 0;
    const dim3 rgrid((unsigned)((n8 + 255) / 256 + (colsum ? (M + 255) / 256 : 0)));
    if (out_bf16)
        hipLaunchKernelGGL((gemm_wgrad_reduce_kernel<1>), rgrid, dim3(256), 0, s, workspace, split ? plan.splits : 0, M,
                           N, C, ldc, cs_part, plan.splits * plan.tiles_n, colsum);
    else
        hipLaunchKernelGGL((gemm_wgrad_reduce_kernel<0>), rgrid, dim3(256), 0, s, workspace, split ? plan.splits : 0, M,
                           N, C, ldc, cs_part, plan.splits * plan.tiles_n, colsum);
    return hipGetLastError();
}

}  // namespace coset
