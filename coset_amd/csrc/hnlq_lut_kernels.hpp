// hnlq_lut_kernels.hpp -- E8 HNLQ codec for q in {2, 4} with table decode in LDS.
//
// Same contract and bit-exact results as hnlq_codec.hip (the generic path),
// but each decode level is two LDS lookups instead of a projection:
//   2r = 2Gb - q * (2c),  c = coarse[cid_map[idx]]    (tables.hip)
// 2Gb is integer arithmetic on the digits, and the level sum
// x_hat = sum_m q^m r_m (exact in the reference's fp32) is accumulated as
// integers and halved at the end.
//
// Launch: persistent grid, one 1024-thread workgroup per CU.  The q = 4 map
// (65536 x uint16 = 128 KiB) plus the coarse points (<= 8 KiB) fill most of
// the 160 KiB LDS of a gfx950 CU; every workgroup stages them once and then
// walks blocks: the general kernel with a grid stride, the fixed-format one
// in tiles handed out by a per-stream counter (so workgroups that run ahead
// take more tiles), and HBM sees one contiguous read of x and one write of
// the outputs.
//
// Instantiated per q by hnlq_lut_q2.hip and hnlq_lut_q4.hip; dispatch and the
// counter ring are in hnlq_lut.hip.
#pragma once

#include <algorithm>

#include "codec_kernels.hpp"
#include "counters.hpp"
#include "tables.hpp"

namespace coset {

template <int Q>
struct LutShape {
    static constexpr int kCodes = Q * Q * Q * Q * Q * Q * Q * Q;
};

constexpr int kLutThreads = 1024;

// Tile counters of the dynamic schedule: a pair taken from the per-device
// counter ring (counters.hpp) for each launch -- [0] hands out tiles, [1]
// counts finished workgroups, and the workgroup that finishes last puts both
// back to zero and then releases the slot to the host.
constexpr int kTileBlocks = 2;        // blocks per thread in a dynamic tile (1 where float codes are written)
constexpr int64_t kDynamicMinBlocks = 3 << 21;   // the fp32 round trip takes its tiles from a counter from here on
constexpr int64_t kDynamicMinBlocksCodes = 1 << 21;   // the same where float codes are written

// Copies the decode tables to LDS: the map (n_map uint4) and the byte or
// coarse table (n_tab uint64).  Each thread issues all its loads before any
// LDS store (one round trip to L2, not one per element), and each workgroup
// starts at its own offset so the CUs do not all request the same lines at
// once.  blockDim.x == kLutThreads.
template <int PM, int PT>
__device__ __forceinline__ void stage_tables(const uint4* __restrict__ g_map, uint4* s_map, int n_map,
                                             const uint64_t* __restrict__ g_tab, uint64_t* s_tab, int n_tab)
{
    // loads are unconditional (an index past the end reads the last element)
    // so none of them waits behind a branch; only the stores are predicated
    const unsigned salt = blockIdx.x * 2459u;
    const int rm = n_map > 0 ? (int)(salt % (unsigned)n_map) : 0;
    const int rt = n_tab > 0 ? (int)(salt % (unsigned)n_tab) : 0;
    auto at = [](int i, int r, int n) {
        if (i >= n) return n - 1;
        const int j = i + r;
        return j >= n ? j - n : j;
    };
    uint4 m[PM];
    uint64_t t[PT];
#pragma unroll
    for (int k = 0; k < PM; ++k) m[k] = g_map[at(threadIdx.x + k * kLutThreads, rm, n_map)];
    if (n_tab > 0) {
#pragma unroll
        for (int k = 0; k < PT; ++k) t[k] = g_tab[at(threadIdx.x + k * kLutThreads, rt, n_tab)];
    }
#pragma unroll
    for (int k = 0; k < PM; ++k) {
        const int i = threadIdx.x + k * kLutThreads;
        if (i < n_map) s_map[at(i, rm, n_map)] = m[k];
    }
#pragma unroll
    for (int k = 0; k < PT; ++k) {
        const int i = threadIdx.x + k * kLutThreads;
        if (i < n_tab) s_tab[at(i, rt, n_tab)] = t[k];
    }
}

// Block schedules of the persistent kernels.  Each walks blocks 0..n-1
// (n >= 1) of its workgroup's share, calling load(i, in) for a block's input
// into a register set and body(i, in) for the rest, with the next input in
// flight while a body runs.  Loads and stores share one in-order completion
// counter, so the wait before a body leaves the other set's loads and the
// last body's stores in flight only if their number is the same on every
// path into it: the loads are unconditional (past the end they read block
// n - 1), and the first step is peeled so each loop is entered as it is
// re-entered.  A partial last tile recomputes block n - 1 and stores the same
// values to it.  In the grid stride and the whole-tile schedule pro() runs
// once, by every thread of a workgroup that has work, after its first loads
// are issued (the decoder stages its LDS tables there, so the first input
// and the tables arrive together).

// Grid stride (no tile counter): one block ahead.  The loop runs on the
// workgroup's base index, so every lane of a wave takes every step (a lane
// past the end works on block n - 1), which the bodies' wave-wide stores
// assume.
template <typename In, typename Load, typename Body, typename Pro>
__device__ __forceinline__ void schedule_stride(int64_t n, Load& load, Body& body, Pro& pro)
{
    const int64_t last = n - 1;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    auto blk = [&](int64_t b) {
        const int64_t i = b + threadIdx.x;
        return i < n ? i : last;
    };
    int64_t b = (int64_t)blockIdx.x * blockDim.x;
    if (b >= n) return;
    In in0, in1;
    load(blk(b), in0);
    int64_t b1 = b + stride;
    load(blk(b1), in1);
    pro();
    body(blk(b), in0);
    while (b1 < n) {
        const int64_t b2 = b1 + stride;
        load(blk(b2), in0);
        body(blk(b1), in1);
        if (b2 >= n) break;
        b1 = b2 + stride;
        load(blk(b1), in1);
        body(blk(b2), in0);
    }
}

// The counter pair's protocol: a workgroup's first two tiles are its own number
// and that plus the grid (256 workgroups taking both from the counter waited
// for 512 atomics on one address, ~13 ns each, before the last could start);
// thread 0 takes the others with atomicInc (the
// compiler rewrites a uniform-address atomicAdd into a wave reduction that
// waits for its result at once) two tiles ahead and publishes them through
// LDS behind an LDS-only barrier; when a workgroup has seen its last tile it
// counts itself done, and the last one resets the pair and then sets the
// slot's release flag (host memory, system scope): only after that does the
// host hand the pair to another launch.
__device__ __forceinline__ void tiles_done(unsigned* tiles, unsigned* release)
{
    if (threadIdx.x == 0 && atomicAdd(tiles + 1, 1u) == gridDim.x - 1) {
        atomicExch(tiles, 0u);
        atomicExch(tiles + 1, 0u);
        __threadfence_system();
        __hip_atomic_store(release, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Dynamic tiles of KT blocks per thread, blockDim.x apart, with one block
// ahead; one LDS barrier per tile.
template <int KT, typename In, typename Load, typename Body>
__device__ __forceinline__ void schedule_tiles(int64_t n, TileCounters tc, unsigned* s_tile, Load& load, Body& body)
{
    static_assert(KT == 1 || KT == 2, "register sets alternate per block");
    unsigned* tiles = tc.pair;
    const int64_t last = n - 1;
    const int64_t ntiles = (n + KT * (int64_t)blockDim.x - 1) / (KT * (int64_t)blockDim.x);
    auto blk = [&](int64_t t, int j) {
        const int64_t b = (t * KT + j) * blockDim.x + threadIdx.x;
        return b < n ? b : last;
    };
    const int64_t t0 = blockIdx.x;
    int64_t t1 = t0 + gridDim.x;
    In in0, in1;
    // s0 holds the tile's first block; with KT == 1 the next tile's starts in s1, else in s0
    auto tile = [&](int64_t cur, int64_t nxt, In& s0, In& s1, int slot) {
        if constexpr (KT == 2) {
            load(blk(cur, 1), s1);
            body(blk(cur, 0), s0);
        }
        In& now = KT == 2 ? s1 : s0;
        In& ahead = KT == 2 ? s0 : s1;
        unsigned grab = 0;
        if (threadIdx.x == 0) grab = atomicInc(tiles, ~0u);
        load(blk(nxt, 0), ahead);
        body(blk(cur, KT - 1), now);
        if (threadIdx.x == 0) s_tile[slot] = grab;
        lds_barrier();
        return (int64_t)s_tile[slot] + 2 * (int64_t)gridDim.x;
    };
    if (t0 < ntiles) {
        load(blk(t0, 0), in0);
        int64_t t2 = tile(t0, t1, in0, in1, 0);
        if constexpr (KT == 1) {
            while (t1 < ntiles) {
                const int64_t t3 = tile(t1, t2, in1, in0, 1);
                if (t2 >= ntiles) break;
                t1 = t3;
                t2 = tile(t2, t3, in0, in1, 0);
            }
        } else {
            int slot = 1;
            while (t1 < ntiles) {
                const int64_t t3 = tile(t1, t2, in0, in1, slot);
                slot ^= 1;
                t1 = t2;
                t2 = t3;
            }
        }
    }
    tiles_done(tiles, tc.release);
}

// SWAR: each level's 2r comes from three byte tables (tables.hpp) added as
// two 32-bit words, levels are summed with shifts, and the bytes hold
// 2 x_hat + swar_bias; otherwise 2r = 2Gb - q (2c) from the unpacked digits.
template <int Q, int M, int MODE, bool SWAR>
__global__ void __launch_bounds__(kLutThreads) hnlq_lut_kernel(CodecArgs a, const uint16_t* __restrict__ g_map,
                                                            const uint64_t* __restrict__ g_tab,
                                                            int n_coarse, int swar_bias)
{
    constexpr int NC = LutShape<Q>::kCodes;
    __shared__ __align__(16) uint16_t s_map[NC];
    __shared__ uint64_t s_tab[SWAR ? 512 + kMaxCoarse : kMaxCoarse];

    if (MODE != MODE_ENCODE) {
        stage_tables<(NC / 8 + kLutThreads - 1) / kLutThreads,
                     ((SWAR ? 512 : 0) + kMaxCoarse + kLutThreads - 1) / kLutThreads>(
            reinterpret_cast<const uint4*>(g_map), reinterpret_cast<uint4*>(s_map), NC / 8, g_tab, s_tab,
            SWAR ? 512 + n_coarse : n_coarse);
        __syncthreads();
    }
    const float half_bias = 0.5f * (float)swar_bias;

    if (blockIdx.x == 0 && threadIdx.x == 0 && a.step_counter) *a.step_counter += 1;
    const float qf = (float)Q;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.n; i += stride) {
        float scale = 1.f;
        if (a.scale_mode == SCALE_CODEC)
            scale = a.beta;
        else if (a.scale_mode == SCALE_LAYER)
            scale = layer_scale(a, i);

        // Level words are collected in one 64-bit register (M <= 4 words of
        // 16 bits); each level is encoded, then decoded from its digits.
        uint64_t pack = 0;
        float xl[8];
        if (MODE != MODE_DECODE) {
            if (a.x_dtype == DT_BF16) {
                uint4 v = reinterpret_cast<const uint4*>(a.x)[i];
                uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    xl[2 * j] = __uint_as_float(w[j] << 16);
                    xl[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
                }
            } else {
                const float4* p = reinterpret_cast<const float4*>(a.x) + 2 * i;
                float4 u = p[0], v = p[1];
                xl[0] = u.x; xl[1] = u.y; xl[2] = u.z; xl[3] = u.w;
                xl[4] = v.x; xl[5] = v.y; xl[6] = v.z; xl[7] = v.w;
            }
            if (a.scale_mode == SCALE_CODEC) {
                if (a.beta_is_pow2) {
                    if (a.beta_inv != 1.f) {  // x / 1 = x
#pragma unroll
                        for (int j = 0; j < 8; ++j) xl[j] = __fmul_rn(xl[j], a.beta_inv);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) xl[j] = __fdiv_rn(xl[j], scale);
                }
            } else if (a.scale_mode == SCALE_LAYER) {
#pragma unroll
                for (int j = 0; j < 8; ++j) xl[j] = __fmul_rn(xl[j], scale);
            }
            if (a.dither) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    xl[j] = __fadd_rn(xl[j], a.dither[a.dither_stride * i + j]);
            }
        } else {
            const uint16_t* pw = reinterpret_cast<const uint16_t*>(a.packed_in) + (size_t)i * M;
            if (M == 2) {
                pack = *reinterpret_cast<const uint32_t*>(pw);
            } else if (M == 4) {
                pack = *reinterpret_cast<const uint64_t*>(pw);
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) pack |= (uint64_t)pw[m] << (16 * m);
            }
        }

        int acc2[8];  // sum_m q^m * 2 r_m, exact integers
#pragma unroll
        for (int j = 0; j < 8; ++j) acc2[j] = 0;
        uint32_t sw0 = 0u, sw1 = 0u;  // SWAR: bytes 0-3 / 4-7 of sum_m q^m (2 r_m + bias)
        int wq = 1;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            int b[8];
            uint32_t word;
            if (MODE != MODE_DECODE) {
                encode_level<Q>(xl, a.fast_projection, Q, b);
                word = pack_word<Q>(b, Q);
                pack |= (uint64_t)word << (16 * m);
                if (a.codes_f32) {
                    float4* cp = reinterpret_cast<float4*>(a.codes_f32 + ((size_t)i * M + m) * 8);
                    cp[0] = make_float4((float)b[0], (float)b[1], (float)b[2], (float)b[3]);
                    cp[1] = make_float4((float)b[4], (float)b[5], (float)b[6], (float)b[7]);
                }
                if (m + 1 < M) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) xl[j] = div_q<Q>(xl[j], qf);
                }
            } else {
                word = (uint32_t)(pack >> (16 * m)) & (uint32_t)(NC - 1);  // table bounds for any input
                unpack_word<Q>(word, Q, b);
            }
            if (MODE != MODE_ENCODE && SWAR) {
                const uint2 tl = *reinterpret_cast<const uint2*>(&s_tab[256 + (word & 0xffu)]);
                const uint2 tc = *reinterpret_cast<const uint2*>(&s_tab[512 + s_map[word]]);
                uint32_t l0 = tl.x + tc.x, l1 = tl.y + tc.y;
                if (Q != 2) {
                    const uint2 th = *reinterpret_cast<const uint2*>(&s_tab[(word >> 8) & 0xffu]);
                    l0 += th.x;
                    l1 += th.y;
                }
                sw0 += l0 * (uint32_t)wq;  // q^m: a shift, no byte overflows (checked when tables are built)
                sw1 += l1 * (uint32_t)wq;
                wq *= Q;
            } else if (MODE != MODE_ENCODE) {
                int u[8];  // 2 G b
                u[0] = 4 * b[0] - 2 * b[1] + b[7];
#pragma unroll
                for (int j = 1; j < 6; ++j) u[j] = 2 * (b[j] - b[j + 1]) + b[7];
                u[6] = 2 * b[6] + b[7];
                u[7] = b[7];
                uint64_t c = s_tab[s_map[word]];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    int two_c = (int)(int8_t)(uint8_t)(c >> (8 * j));
                    acc2[j] += wq * (u[j] - Q * two_c);
                }
                wq *= Q;
            }
        }
        if (MODE != MODE_DECODE && a.packed) {
            uint16_t* pw = reinterpret_cast<uint16_t*>(a.packed) + (size_t)i * M;
            if (M == 1) {
                pw[0] = (uint16_t)pack;
            } else if (M == 2) {
                *reinterpret_cast<uint32_t*>(pw) = (uint32_t)pack;
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) pw[m] = (uint16_t)(pack >> (16 * m));
            }
        }
        if (MODE == MODE_ENCODE) continue;

        if (!a.out) continue;
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float v;
            if (SWAR) {  // (byte - bias) / 2, exact
                const uint32_t w = j < 4 ? sw0 : sw1;
                v = __fmaf_rn((float)((w >> (8 * (j & 3))) & 0xffu), 0.5f, -half_bias);
            } else {
                v = __fmul_rn((float)acc2[j], 0.5f);  // exact
            }
            if (a.scale_mode == SCALE_CODEC) {
                if (a.beta != 1.f) v = __fmul_rn(v, scale);  // x * 1 = x
            } else if (a.scale_mode == SCALE_LAYER) {
                v = __fdiv_rn(v, scale);
                v = (v != v) ? v : fminf(fmaxf(v, -a.clip), a.clip);  // clamp keeps NaN
            }
            o[j] = v;
        }
        if (a.out_dtype == DT_BF16) {
            uint4 v;
            v.x = f32_to_bf16(o[0]) | ((uint32_t)f32_to_bf16(o[1]) << 16);
            v.y = f32_to_bf16(o[2]) | ((uint32_t)f32_to_bf16(o[3]) << 16);
            v.z = f32_to_bf16(o[4]) | ((uint32_t)f32_to_bf16(o[5]) << 16);
            v.w = f32_to_bf16(o[6]) | ((uint32_t)f32_to_bf16(o[7]) << 16);
            reinterpret_cast<uint4*>(a.out)[i] = v;
        } else {
            float4* p = reinterpret_cast<float4*>(a.out) + 2 * i;
            p[0] = make_float4(o[0], o[1], o[2], o[3]);
            p[1] = make_float4(o[4], o[5], o[6], o[7]);
        }
    }
}

typedef float f32x4_nt __attribute__((ext_vector_type(4)));

// Streaming (non-temporal) stores of the outputs, which nothing reads back
// in the same launch: 2^24-block round trip 203.9 -> 200.3 us on one box
// (non-temporal loads of the input measured slower and are not used).
__device__ __forceinline__ void store_nt(void* p, const float4& v)
{
    __builtin_nontemporal_store(__builtin_bit_cast(f32x4_nt, v), static_cast<f32x4_nt*>(p));
}

__device__ __forceinline__ void store_nt(uint32_t* p, uint32_t v)
{
    __builtin_nontemporal_store(v, p);
}

// Stores one block's 8 decoded floats (32 bytes) through the wave's 1 KiB
// LDS slice st: half the wave at a time writes its blocks' 32 bytes there
// and the whole wave reads them back 16 bytes a lane, so each of the two
// stores writes 32 consecutive blocks (1 KiB) rather than every lane 32
// bytes.  Every lane is active and the lanes of a wave hold consecutive
// blocks clamped to n - 1 (the schedules' contract), so lane q's block is
// min(i_0 + q, n - 1), i_0 being lane 0's.  LDS operations of one wave
// complete in order, so the slice needs no barrier, only compiler fences:
// a lane reads what other lanes wrote, which a single lane's view of
// memory does not show.
__device__ __forceinline__ void store_out_wave(float* out, int64_t n, int64_t i, const float o[8], float4* st)
{
    const int lane = threadIdx.x & 63;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)i);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)i >> 32));
    const int64_t i0 = (int64_t)(((uint64_t)hi << 32) | lo);
    const int64_t room = n - 1 - i0;
    const int lim = room < 63 ? (int)room : 63;
    char* dst = reinterpret_cast<char*>(out + 8 * i0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if ((lane >> 5) == h) {
            st[2 * (lane & 31)] = make_float4(o[0], o[1], o[2], o[3]);
            st[2 * (lane & 31) + 1] = make_float4(o[4], o[5], o[6], o[7]);
        }
        __asm__ volatile("" ::: "memory");
        const float4 v = st[lane];
        __asm__ volatile("" ::: "memory");
        const uint32_t q = min(32 * h + (lane >> 1), lim);
        store_nt(dst + (q * 32u + (lane & 1) * 16u), v);  // 32-bit lane offset
    }
}

// The float code tensor [n, 2, 8] of the two level words of a block (low 16
// bits: level 0), 64 bytes a block, through the wave's 1 KiB LDS slice as
// in store_out_wave: a quarter of the wave at a time writes its blocks'
// codes there and the whole wave reads them back 16 bytes a lane, so each
// of the four stores writes 16 consecutive blocks (1 KiB).  NT: the stores
// are non-temporal (measured faster for the encoder, whose only other output
// is the packed words, and slower beside the decoded-block stores of the
// round trip).
template <int Q, bool NT>
__device__ __forceinline__ void store_codes_wave(float* codes, int64_t n, int64_t i, uint32_t words, uint4* st)
{
    uint32_t e[4][4];  // e[chunk][dword]: chunk c = level c / 2, coordinates 4 (c % 2) ..
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        int b[8];
        unpack_word<Q>((words >> (16 * m)) & 0xffffu, Q, b);
#pragma unroll
        for (int d = 0; d < 8; ++d) e[2 * m + d / 4][d % 4] = __float_as_uint((float)b[d]);
    }
    const int lane = threadIdx.x & 63;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)i);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)i >> 32));
    const int64_t i0 = (int64_t)(((uint64_t)hi << 32) | lo);
    const int64_t room = n - 1 - i0;
    const int lim = room < 63 ? (int)room : 63;
    char* dst = reinterpret_cast<char*>(codes + 16 * i0);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        if ((lane >> 4) == h) {
#pragma unroll
            for (int c = 0; c < 4; ++c) st[4 * (lane & 15) + c] = make_uint4(e[c][0], e[c][1], e[c][2], e[c][3]);
        }
        __asm__ volatile("" ::: "memory");
        const uint4 v = st[lane];
        __asm__ volatile("" ::: "memory");
        const uint32_t q = min(16 * h + (lane >> 2), lim);
        char* p = dst + (q * 64u + (lane & 3) * 16u);  // 32-bit lane offset
        if constexpr (NT)
            store_nt(p, __builtin_bit_cast(float4, v));
        else
            *reinterpret_cast<uint4*>(p) = v;
    }
}

// Same contract for the common cases, with everything the general kernel
// decides per block fixed at compile time: fp32 or bf16 input (XBF) and
// output (OBF), no scale, a codec beta (2^k:
// x / beta == x * 2^-k exactly; others divide, SC_DIV, where the decode
// multiplies either way) or the layer's stored per-row betas (SC), no dither, byte-table decode, the
// encoder's fast projection on; the float code tensor is an optional output
// (CODES).  The loop is
// unrolled twice so the next block's input loads into the other register
// set while the current block is processed.
// One encoder level straight to its word idx(b).  On the fast path each
// digit (the low bits of a row) is funnelled into the top of an accumulator
// as the accumulator shifts right, one v_alignbit per digit.
// CLEAR: condition (5) of e8_fast.hpp (weights hold zeros and tiny values).
template <int Q, bool CLEAR>
__device__ __forceinline__ uint32_t encode_level_word(const float xl[8], bool in_range)
{
    static_assert(Q == 2 || Q == 4, "byte-table formats");
    constexpr int L = Q == 2 ? 1 : 2;
    int c[8];
    const bool ok = fast_rows<CLEAR>(xl, c, in_range);
#pragma unroll
    for (int i = 0; i < 8; ++i) __asm__ volatile("" : "+v"(c[i]));  // rows computed ahead of the fallback
    if (ok) {
        uint32_t acc = 0u;
#pragma unroll
        for (int j = 7; j >= 0; --j) acc = __builtin_amdgcn_alignbit((uint32_t)c[j], acc, L);
        return acc >> (32 - 8 * L);  // digit 0 highest: sum_j b_j Q^(7-j)
    }
    float y[8];
    int b[8];
    project<false, false>(xl, y);
    lattice_digits<Q>(y, Q, b);
    return pack_word<Q>(b, Q);
}

// PROBE (measurement, the round trip only): 0 is the codec; 1 keeps the
// launch, table staging, tile schedule, loads and stores but writes each
// block's input back out and a word folded from its bits, with no lattice
// arithmetic -- the streaming ceiling of this kernel's access pattern; 2 is
// 1 without the table staging.
//
// Per-row betas and bf16 (SC_LAYER, XBF, OBF): storing and loading bf16
// weights.  4193792 blocks of 4096-wide rows, q4 M2, against the general
// kernel: encode to words 54.2 -> 43.8 us, decode to bf16 39.6 -> 15.9 us (5.3 TB/s).  The encoder
// is bound by its VALU work (~360 instructions a block), the decoder by the
// LDS gathers and the conversion; the scale of a block comes in with its
// input, one tile ahead, and dec / beta from one reciprocal (div_by_recip).
enum PlainScale { SC_NONE = 0, SC_POW2 = 1, SC_LAYER = 2, SC_DIV = 3 };

template <int Q, int M, int MODE, int SC, bool CODES, bool PK, bool XBF = false, bool OBF = false, int PROBE = 0>
__global__ void __launch_bounds__(kLutThreads) hnlq_plain_kernel(CodecArgs a, const uint16_t* __restrict__ g_map,
                                                              const uint64_t* __restrict__ g_tab, int n_coarse,
                                                              int swar_bias, TileCounters tc)
{
    constexpr int NC = LutShape<Q>::kCodes;
    __shared__ __align__(16) uint16_t s_map[NC];
    __shared__ uint64_t s_tab[512 + kMaxCoarse];
    // tiles from a counter in the fp32 round trip and where float codes are written: the counter hands out one
    // tile per ~13 ns whatever the tile holds, which the shorter bodies wait
    // for (bf16 decode of 2^24 blocks: 106 us from the counter, 53 with the grid
    // stride; encode 165 / 157), and its hand-back at the end costs 2-4 us
    // (kDynamicMinBlocks: round trip of 2^22 blocks 52.5 / 50.5, of 2^23 98.7 /
    // 107.7, of 2^24 203 / 227).  Float codes are 64 bytes of stores a block, whose
    // speed differs between workgroups (kDynamicMinBlocksCodes, tiles of one block
    // per thread): encode of 2^20 blocks 20.2 / 19.0, of 2^21 34.3 / 37.3, of 2^24
    // 263 / 322; round trip 26.7 / 25.3, 44.9 / 46.8, 368 / 432
    constexpr bool kDynamic = CODES || (MODE == MODE_ROUNDTRIP && !XBF && !OBF);
    __shared__ unsigned s_tile[kDynamic ? 2 : 1];
    __shared__ float4 s_stage[MODE == MODE_ENCODE && !CODES ? 1 : kLutThreads / 64][64];  // store_*_wave
    auto stage = [&]() {
        stage_tables<(NC / 8 + kLutThreads - 1) / kLutThreads, (512 + kMaxCoarse + kLutThreads - 1) / kLutThreads>(
            reinterpret_cast<const uint4*>(g_map), reinterpret_cast<uint4*>(s_map), NC / 8, g_tab, s_tab,
            512 + n_coarse);
    };
    // The decoder stages its tables after the first tile's loads are issued
    // (an LDS-only barrier: the loads stay in flight), 2.5 us sooner per
    // launch at 2^24 blocks; the round trip stages them first (measured
    // faster that way on the same box).
    static_assert(PROBE == 0 || (MODE == MODE_ROUNDTRIP && M == 2 && PK && !CODES && SC == SC_NONE), "probe: C2's outputs");
    if constexpr (MODE == MODE_ROUNDTRIP && PROBE != 2) {
        stage();
        __syncthreads();
    }
    auto pro = [&]() {
        if constexpr (MODE == MODE_DECODE) {
            stage();
            lds_barrier();
        }
    };
    const float half_bias = 0.5f * (float)swar_bias;
    const float4* xs = reinterpret_cast<const float4*>(a.x);
    const int64_t n = a.n;

    struct In {
        float4 u, v;
        uint64_t w;
        float s;
    };
    auto load = [&](int64_t i, In& in) {
        if (SC == SC_LAYER) in.s = a.beta_row[u32div((uint32_t)i, a.row_div)];
        if (MODE != MODE_DECODE && XBF) {
            in.u = xs[i];
        } else if (MODE != MODE_DECODE) {
            in.u = xs[2 * i];
            in.v = xs[2 * i + 1];
        } else {
            const uint16_t* pw = reinterpret_cast<const uint16_t*>(a.packed_in) + (size_t)i * M;
            if (M == 2) {
                in.w = *reinterpret_cast<const uint32_t*>(pw);
            } else if (M == 4) {
                in.w = *reinterpret_cast<const uint64_t*>(pw);
            } else {
                uint64_t w = 0;
#pragma unroll
                for (int m = 0; m < M; ++m) w |= (uint64_t)pw[m] << (16 * m);
                in.w = w;
            }
        }
    };
    auto body = [&](int64_t i, const In& in) {
        if constexpr (PROBE != 0) {
            const uint32_t f = __float_as_uint(in.u.x) ^ __float_as_uint(in.u.y) ^ __float_as_uint(in.u.z) ^
                               __float_as_uint(in.u.w) ^ __float_as_uint(in.v.x) ^ __float_as_uint(in.v.y) ^
                               __float_as_uint(in.v.z) ^ __float_as_uint(in.v.w);
            *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(a.packed) + (size_t)i * 2) = f;
            const float o[8] = {in.u.x, in.u.y, in.u.z, in.u.w, in.v.x, in.v.y, in.v.z, in.v.w};
            store_out_wave(static_cast<float*>(a.out), n, i, o, s_stage[threadIdx.x >> 6]);
            return;
        }
        float xl[8] = {in.u.x, in.u.y, in.u.z, in.u.w, in.v.x, in.v.y, in.v.z, in.v.w};
        if constexpr (XBF) {
            const uint32_t h[4] = {__float_as_uint(in.u.x), __float_as_uint(in.u.y), __float_as_uint(in.u.z),
                                   __float_as_uint(in.u.w)};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                xl[2 * j] = __uint_as_float(h[j] << 16);
                xl[2 * j + 1] = __uint_as_float(h[j] & 0xffff0000u);
            }
        }
        uint64_t pack = MODE == MODE_DECODE ? in.w : 0;
        if (MODE != MODE_DECODE && SC != SC_NONE) {
#pragma unroll
            for (int j = 0; j < 8 && SC != SC_DIV; ++j) xl[j] = __fmul_rn(xl[j], SC == SC_LAYER ? in.s : a.beta_inv);
            if constexpr (SC == SC_DIV) {
                // the launcher's beta lies in [2^-20, 2^20]; with every |x| in
                // [2^-80, 2^80] all of div_by_recip's terms are normal and its
                // two corrections exact; zeros and the rest divide
                float lo = fabsf(xl[0]), hi = lo;
#pragma unroll
                for (int j = 1; j < 8; ++j) {
                    lo = fminf(lo, fabsf(xl[j]));
                    hi = fmaxf(hi, fabsf(xl[j]));
                }
                if (lo >= 0x1p-80f && hi <= 0x1p80f) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) xl[j] = div_by_recip<2>(xl[j], a.beta, a.beta_inv);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) xl[j] = __fdiv_rn(xl[j], a.beta);
                }
            }
        }
        // level m's input is xl * Q^-m exactly, so max |x_m| < 2^21 is
        // max |x_0| < 2^21 Q^m
        float amax = 0.f;
        if (MODE != MODE_DECODE) {
            amax = fabsf(xl[0]);
#pragma unroll
            for (int j = 1; j < 8; ++j) amax = fmaxf(amax, fabsf(xl[j]));
        }
        uint32_t sw0 = 0u, sw1 = 0u;
        float lim = kFastMaxAbs;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            uint32_t word;
            if (MODE != MODE_DECODE) {
                word = encode_level_word<Q, SC == SC_LAYER || XBF>(xl, amax < lim);
                lim *= (float)Q;
                pack |= (uint64_t)word << (16 * m);
                if (CODES && M != 2) {  // the reference's float code tensor [n, M, 8]
                    int b[8];
                    unpack_word<Q>(word, Q, b);
                    float4* cp = reinterpret_cast<float4*>(a.codes_f32 + ((size_t)i * M + m) * 8);
                    cp[0] = make_float4((float)b[0], (float)b[1], (float)b[2], (float)b[3]);
                    cp[1] = make_float4((float)b[4], (float)b[5], (float)b[6], (float)b[7]);
                }
                if (m + 1 < M) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) xl[j] = __fmul_rn(xl[j], 1.0f / (float)Q);  // exact: Q = 2^k
                }
            } else {
                word = (uint32_t)(pack >> (16 * m)) & (uint32_t)(NC - 1);  // table bounds for any input
            }
            if (MODE != MODE_ENCODE) {
                const uint2 tl = *reinterpret_cast<const uint2*>(&s_tab[256 + (word & 0xffu)]);
                const uint2 tc = *reinterpret_cast<const uint2*>(&s_tab[512 + s_map[word]]);
                uint32_t l0 = tl.x + tc.x, l1 = tl.y + tc.y;
                if (Q != 2) {
                    const uint2 th = *reinterpret_cast<const uint2*>(&s_tab[(word >> 8) & 0xffu]);
                    l0 += th.x;
                    l1 += th.y;
                }
                constexpr int L = Q == 2 ? 1 : 2;
                sw0 += l0 << (L * m);  // q^m, no byte overflows (checked when the tables are built)
                sw1 += l1 << (L * m);
            }
        }
        if (MODE != MODE_DECODE && CODES && M == 2)
            store_codes_wave<Q, MODE == MODE_ENCODE>(a.codes_f32, n, i, (uint32_t)pack, reinterpret_cast<uint4*>(s_stage[threadIdx.x >> 6]));
        if (MODE != MODE_DECODE && PK) {
            uint16_t* pw = reinterpret_cast<uint16_t*>(a.packed) + (size_t)i * M;
            if (M == 1) {
                pw[0] = (uint16_t)pack;
            } else if (M == 2) {
                store_nt(reinterpret_cast<uint32_t*>(pw), (uint32_t)pack);
            } else if (M == 4) {
                *reinterpret_cast<uint64_t*>(pw) = pack;
            } else {
#pragma unroll
                for (int m = 0; m < M; ++m) pw[m] = (uint16_t)(pack >> (16 * m));
            }
        }
        if (MODE == MODE_ENCODE) return;
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t w = j < 4 ? sw0 : sw1;
            o[j] = __fmaf_rn((float)((w >> (8 * (j & 3))) & 0xffu), 0.5f, -half_bias);  // (byte - bias) / 2, exact
            if (SC == SC_POW2 || SC == SC_DIV) o[j] = __fmul_rn(o[j], a.beta);
        }
        bool plain_values = true;   // finite, normal quotients (or no division): no NaN to keep
        if constexpr (SC == SC_LAYER) {
            const float ab = fabsf(in.s);
            plain_values = ab >= 0x1p-64f && ab <= 0x1p64f;
            if (plain_values) {
                // half-integers of at most 127 / 2: one correction step (fastdiv.hpp)
                const float y = __fdiv_rn(1.f, in.s);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    o[j] = __builtin_amdgcn_fmed3f(div_by_recip<1>(o[j], in.s, y), -a.clip, a.clip);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float v = __fdiv_rn(o[j], in.s);
                    o[j] = v != v ? v : fminf(fmaxf(v, -a.clip), a.clip);  // clamp keeps NaN
                }
            }
        }
        if constexpr (OBF) {
            typedef float f32x2_t __attribute__((ext_vector_type(2)));
            typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
            uint32_t h[4];
            if (plain_values) {
#pragma unroll
                for (int j = 0; j < 4; ++j)   // round to nearest even in hardware
                    h[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){o[2 * j], o[2 * j + 1]}, bf16x2_t));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) h[j] = f32_to_bf16(o[2 * j]) | ((uint32_t)f32_to_bf16(o[2 * j + 1]) << 16);
            }
            store_nt(reinterpret_cast<uint4*>(a.out) + i,
                     make_float4(__uint_as_float(h[0]), __uint_as_float(h[1]), __uint_as_float(h[2]),
                                 __uint_as_float(h[3])));
            return;
        }
        // staged whole-line stores measured faster for the decoder and the
        // round trip with packed words, direct stores for the round trip
        // without them (A/B on one box, 2^24 blocks: 1.2 and 2.7 us)
        if constexpr (MODE == MODE_DECODE || PK) {
            store_out_wave(static_cast<float*>(a.out), n, i, o, s_stage[threadIdx.x >> 6]);
        } else {
            float4* p = reinterpret_cast<float4*>(a.out) + 2 * i;
            store_nt(p, make_float4(o[0], o[1], o[2], o[3]));
            store_nt(p + 1, make_float4(o[4], o[5], o[6], o[7]));
        }
    };

    // every store of a body is unconditional (see the schedules above)
    if constexpr (kDynamic) {
        if (tc.pair) {
            schedule_tiles<CODES ? 1 : kTileBlocks, In>(n, tc, s_tile, load, body);
            return;
        }
    }
    schedule_stride<In>(n, load, body, pro);
}

namespace {

int cu_count()
{
    static int cached[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (!cached[dev]) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev] = n;
    }
    return cached[dev];
}

// Byte tables hold q^M-weighted sums for q = 2 (M <= 4) and q = 4 (M <= 2);
// the encoder alone needs no tables.
template <int Q, int M, int MODE>
hipError_t launch_plain(const CodecArgs& a, int grid, const uint16_t* map, const uint64_t* sw, int nc, int bias,
                        hipStream_t s)
{
    if constexpr (MODE == MODE_ENCODE || Q == 2 || M <= 2) {
        const bool scaled = a.scale_mode == SCALE_CODEC && a.beta != 1.f;
        const bool layer = a.scale_mode == SCALE_LAYER;
        const bool codes = MODE != MODE_DECODE && a.codes_f32;
        const bool xbf = MODE != MODE_DECODE && a.x_dtype == DT_BF16, obf = MODE != MODE_ENCODE && a.out_dtype == DT_BF16;
        const bool div = a.scale_mode == SCALE_CODEC && !a.beta_is_pow2;
        const bool dynamic = codes || (MODE == MODE_ROUNDTRIP && !xbf && !obf);
        const TileCounters tiles = g_codec_dynamic && dynamic && a.n >= (codes ? kDynamicMinBlocksCodes : kDynamicMinBlocks)
                                       ? take_counters(s)
                                       : TileCounters{nullptr, nullptr, -1};
        // packed words are always written by the encoder, optional in the
        // round trip (e8_quantize asks for the decoded blocks only)
        const bool pk = MODE == MODE_ENCODE || (MODE == MODE_ROUNDTRIP && a.packed);
#define COSET_PLAIN(SC, CO, P, XB, OB) \
    hipLaunchKernelGGL((hnlq_plain_kernel<Q, M, MODE, SC, CO, P, XB, OB>), dim3(grid), dim3(kLutThreads), 0, s, a, map, sw, nc, \
                       bias, tiles)
#define COSET_PLAIN_SC(CO, P, XB, OB)                                                      \
    do {                                                                                   \
        if (layer) COSET_PLAIN(SC_LAYER, CO, P, XB, OB);                                   \
        else if (div && MODE == MODE_ENCODE) COSET_PLAIN(SC_DIV, CO, P, XB, OB);           \
        else if (scaled) COSET_PLAIN(SC_POW2, CO, P, XB, OB);                              \
        else COSET_PLAIN(SC_NONE, CO, P, XB, OB);                                          \
    } while (0)
        if constexpr (MODE == MODE_DECODE) {
            if (obf) COSET_PLAIN_SC(false, false, false, true); else COSET_PLAIN_SC(false, false, false, false);
        } else if constexpr (MODE == MODE_ENCODE) {
            if (codes) {
                if (div) COSET_PLAIN(SC_DIV, true, true, false, false);
                else if (scaled) COSET_PLAIN(SC_POW2, true, true, false, false); else COSET_PLAIN(SC_NONE, true, true, false, false);
            } else if (xbf) {
                COSET_PLAIN_SC(false, true, true, false);
            } else {
                COSET_PLAIN_SC(false, true, false, false);
            }
        } else if (layer) {
            if (xbf) {
                if (obf) COSET_PLAIN(SC_LAYER, false, true, true, true); else COSET_PLAIN(SC_LAYER, false, true, true, false);
            } else {
                if (obf) COSET_PLAIN(SC_LAYER, false, true, false, true); else COSET_PLAIN(SC_LAYER, false, true, false, false);
            }
        } else if (xbf) {
            if (div) COSET_PLAIN(SC_DIV, false, true, true, false);
            else if (scaled) COSET_PLAIN(SC_POW2, false, true, true, false); else COSET_PLAIN(SC_NONE, false, true, true, false);
        } else if (pk) {
            if (div) {
                COSET_PLAIN(SC_DIV, false, true, false, false);
            } else if (scaled) {
                if (codes) COSET_PLAIN(SC_POW2, true, true, false, false); else COSET_PLAIN(SC_POW2, false, true, false, false);
            } else {
                if (codes) COSET_PLAIN(SC_NONE, true, true, false, false); else COSET_PLAIN(SC_NONE, false, true, false, false);
            }
        } else {
            if (scaled) {
                if (codes) COSET_PLAIN(SC_POW2, true, false, false, false); else COSET_PLAIN(SC_POW2, false, false, false, false);
            } else {
                if (codes) COSET_PLAIN(SC_NONE, true, false, false, false); else COSET_PLAIN(SC_NONE, false, false, false, false);
            }
        }
#undef COSET_PLAIN_SC
#undef COSET_PLAIN
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return_counters(tiles);
        return e;
    }
    return hipErrorInvalidValue;
}

template <int Q, int MODE>
hipError_t launch_q(const CodecArgs& a, const DecodeTables* t, hipStream_t s)
{
    int64_t need = (a.n + kLutThreads - 1) / kLutThreads;
    int grid = (int)std::min<int64_t>(need, (int64_t)cu_count());
    const uint16_t* map = t ? t->cid_map : nullptr;
    int nc = t ? t->n_coarse : 0;
    const bool swar = t && a.M <= t->swar_max_m;
    const uint64_t* tab = t ? (swar ? t->swar : t->coarse) : nullptr;
    const int bias = swar ? t->swar_bias[a.M] : 0;
    const bool layer = a.scale_mode == SCALE_LAYER, div = a.scale_mode == SCALE_CODEC && !a.beta_is_pow2;
    const bool plain = lut_plain_supported(a, MODE) && (MODE == MODE_ENCODE || swar);
    if (plain) {
        const uint64_t* sw = t ? t->swar : nullptr;
        CodecArgs b = a;
        if (layer) b.row_div = u32div_of((uint32_t)a.blocks_per_row);
        if (div) b.beta_inv = 1.f / a.beta;   // correctly rounded on the host
        switch (a.M) {
        case 1: return launch_plain<Q, 1, MODE>(b, grid, map, sw, nc, bias, s);
        case 2: return launch_plain<Q, 2, MODE>(b, grid, map, sw, nc, bias, s);
        case 3: return launch_plain<Q, 3, MODE>(b, grid, map, sw, nc, bias, s);
        case 4: return launch_plain<Q, 4, MODE>(b, grid, map, sw, nc, bias, s);
        default: return hipErrorInvalidValue;
        }
    }
#define COSET_LUT(MM, SW) \
    hipLaunchKernelGGL((hnlq_lut_kernel<Q, MM, MODE, SW>), dim3(grid), dim3(kLutThreads), 0, s, a, map, tab, nc, bias)
    switch (a.M) {
    case 1: if (swar) COSET_LUT(1, true); else COSET_LUT(1, false); break;
    case 2: if (swar) COSET_LUT(2, true); else COSET_LUT(2, false); break;
    case 3: if (Q == 2 && swar) COSET_LUT(3, Q == 2); else COSET_LUT(3, false); break;
    case 4: if (Q == 2 && swar) COSET_LUT(4, Q == 2); else COSET_LUT(4, false); break;
    default: return hipErrorInvalidValue;
    }
#undef COSET_LUT
    return hipGetLastError();
}

}  // namespace

// all modes of one q (hnlq_lut_q2.hip, hnlq_lut_q4.hip)
hipError_t launch_lut_q2(const CodecArgs& a, int mode, const DecodeTables* t, hipStream_t s);
hipError_t launch_lut_q4(const CodecArgs& a, int mode, const DecodeTables* t, hipStream_t s);

}  // namespace coset
