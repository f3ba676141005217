// hnlq_lut.hip -- dispatch of the q in {2, 4} table codec
// (hnlq_lut_kernels.hpp) and its per-device counter ring.
#include <atomic>
#include <map>
#include <mutex>
#include <utility>

#include "hnlq_lut_kernels.hpp"

namespace coset {

int g_codec_plain = 1;
int g_codec_dynamic = 1;

static __device__ __align__(256) unsigned g_counter_ring[kCounterRing];

namespace {

// Per-device counter rings: the pairs' device address, the release flags
// (coherent host memory, and their device address) and the host bookkeeping.
constexpr int kRingDevices = 64;
std::mutex g_ring_mu;
unsigned* g_ring_pairs[kRingDevices] = {nullptr};
unsigned* g_ring_release_dev[kRingDevices] = {nullptr};
CounterRing* g_ring[kRingDevices] = {nullptr};

CounterRing* device_ring(int dev)
{
    std::lock_guard<std::mutex> lock(g_ring_mu);
    if (!g_ring[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_counter_ring)) != hipSuccess || !p) {
            (void)hipGetLastError();
            return nullptr;
        }
        // the kernels write the flags with system-scope stores; every slot starts free
        void* h = nullptr;
        if (hipHostMalloc(&h, kCounterSlots * sizeof(uint32_t), hipHostMallocCoherent) != hipSuccess || !h) {
            (void)hipGetLastError();
            return nullptr;
        }
        void* hd = nullptr;
        if (hipHostGetDevicePointer(&hd, h, 0) != hipSuccess || !hd) {
            (void)hipGetLastError();
            (void)hipHostFree(h);
            return nullptr;
        }
        uint32_t* flags = static_cast<uint32_t*>(h);
        for (uint32_t i = 0; i < kCounterSlots; ++i) flags[i] = 1u;
        CounterRing* r = new CounterRing;
        r->release = flags;
        g_ring_pairs[dev] = static_cast<unsigned*>(p);
        g_ring_release_dev[dev] = static_cast<unsigned*>(hd);
        g_ring[dev] = r;
    }
    return g_ring[dev];
}

}  // namespace

// A counter pair of the current device's ring for one launch on stream s
// (counters.hpp), or none (pair null: the static schedule) while s captures a
// graph (a replayed graph keeps the counters it was captured with and may
// run beside later launches), while every slot is held by a launch still in
// flight, or when the ring cannot be set up.
TileCounters take_counters(hipStream_t s)
{
    const TileCounters none{nullptr, nullptr, -1};
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess) {
        (void)hipGetLastError();  // the query's own error, not the launch's
        return none;
    }
    if (cap != hipStreamCaptureStatusNone) return none;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kRingDevices) return none;
    CounterRing* r = device_ring(dev);
    if (!r) return none;
    const int64_t slot = ring_acquire(*r);
    if (slot < 0) return none;
    return TileCounters{g_ring_pairs[dev] + 2 * slot, g_ring_release_dev[dev] + slot, slot};
}

// Hands back the slot of a launch that failed to start (its kernel never
// releases it); call on the device the slot was taken on.
void return_counters(const TileCounters& tc)
{
    if (!tc.pair || tc.slot < 0) return;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kRingDevices) return;
    CounterRing* r = g_ring[dev];
    if (r) ring_release(*r, tc.slot);
}

bool lut_path_supported(const CodecArgs& a, int mode)
{
    if (a.q != 2 && a.q != 4) return false;
    if (a.M < 1 || a.M > 4) return false;
    if (mode == MODE_DECODE && a.codes_in_f32) return false;  // float codes may be off-grid
    // the words of a block move as one load or store of 4 (M = 2) or 8 (M = 4)
    // bytes; a view that starts inside one goes to the generic kernel, which
    // moves each word by itself
    const uintptr_t words = (uintptr_t)(mode == MODE_DECODE ? a.packed_in : a.packed);
    const uintptr_t align = a.M == 2 ? 4 : a.M == 4 ? 8 : 2;
    if (words % align) return false;
    return true;
}

// No scale, a codec beta (other than 2^k: in [2^-20, 2^20] and with words only
// for the encoders) or stored per-row betas (32-bit block numbers, a positive
// clip), no dither, no step counter, the encoder's fast projection on (it is a
// compile-time constant there) and the mode's outputs present (the kernel's
// stores are unconditional; the round trip's packed words are a compile-time
// option).  Float codes and the round trip without words come with fp32 and no
// per-row betas only, an unscaled bf16 round trip writes fp32.  The decode
// also needs byte tables for M (checked with the tables at hand).
bool lut_plain_supported(const CodecArgs& a, int mode)
{
    const bool enc = mode != MODE_DECODE, dec = mode != MODE_ENCODE;
    const bool layer = a.scale_mode == SCALE_LAYER, div = a.scale_mode == SCALE_CODEC && !a.beta_is_pow2;
    const bool xbf = enc && a.x_dtype == DT_BF16, obf = dec && a.out_dtype == DT_BF16;
    if (!g_codec_plain || a.dither || a.step_counter) return false;
    if (enc && (!a.fast_projection || (a.x_dtype != DT_F32 && !xbf))) return false;
    if (dec && (!a.out || (a.out_dtype != DT_F32 && !obf))) return false;
    if (mode == MODE_ENCODE && !a.packed) return false;
    if (dec && !((a.q == 4 && a.M <= 2) || (a.q == 2 && a.M <= 4))) return false;
    if (layer && (a.use_theta || !a.beta_row || a.n > (int64_t)0xffffffffLL || a.blocks_per_row < 1 ||
                  a.blocks_per_row > (int64_t)0xffffffffLL || (dec && !(a.clip > 0.f))))
        return false;
    if (div && enc &&
        (!(a.beta >= 0x1p-20f && a.beta <= 0x1p20f) || (mode == MODE_ROUNDTRIP && (!a.packed || a.codes_f32))))
        return false;
    if (enc && (layer || xbf || obf) && (a.codes_f32 || (mode == MODE_ROUNDTRIP && (!a.packed || (obf && !layer)))))
        return false;
    return true;
}

// From 2^20 blocks on always (below, the general kernel's table staging does
// not pay).  The fixed-format kernel starts earlier: its decode at 2^18 blocks
// (q4 M2 fp32, us, generic / table: 2^17 4.6 / 4.7, 2^18 6.3 / 5.5), its fp32 round
// trip at 2^19 (2^18 8.2 / 7.5 unscaled but 7.6 / 7.7 by rows, 2^19 13.2 / 10.7), float
// codes of two levels at 2^18 (10.9 / 7.9).  The other encoders and round trips
// are bound by their arithmetic, which one workgroup of 1024 threads per CU
// spreads in whole rounds of 2^18 blocks and the generic kernel in small ones:
// they take the table kernel where the last round is full to nine tenths of all
// (encode q4 M2 by rows in bf16: 300000 blocks 7.1 / 8.2, 2^19 9.4 / 9.3, 800000 12.0 /
// 13.4, 10^6 13.8 / 13.7; round trip unscaled in bf16, q4 M1: 600000 blocks 10.6 /
// 12.7), and never where bf16 values come unscaled or by 2^k, whose ties the
// generic encoder resolves faster (2^19 blocks q4 M1 8.8 / 9.7).
bool lut_pays(const CodecArgs& a, int mode)
{
    if (a.n >= (1 << 20)) return true;
    if (!lut_plain_supported(a, mode) || a.n < (mode == MODE_ROUNDTRIP ? 1 << 19 : 1 << 18)) return false;
    const bool layer = a.scale_mode == SCALE_LAYER;
    const bool bf = (mode != MODE_DECODE && a.x_dtype == DT_BF16) || (mode != MODE_ENCODE && a.out_dtype == DT_BF16);
    if (mode == MODE_DECODE) return true;
    if (mode == MODE_ROUNDTRIP && (layer ? a.q == 2 : !bf)) return true;   // by rows at q = 4: the layer kernel
    if (mode == MODE_ENCODE && a.codes_f32 && a.M == 2) return true;
    if (mode == MODE_ENCODE && bf && !layer && (a.scale_mode != SCALE_CODEC || a.beta_is_pow2)) return false;
    const int64_t round = (int64_t)cu_count() * kLutThreads, rounds = (a.n + round - 1) / round;
    return 10 * a.n >= 9 * rounds * round;
}

hipError_t launch_codec_lut(const CodecArgs& a, int mode, hipStream_t s)
{
    const DecodeTables* t = nullptr;
    if (mode != MODE_ENCODE) {
        hipError_t e = get_decode_tables(a.q, 0, &t);
        if (e != hipSuccess) return e;
    }
    return a.q == 4 ? launch_lut_q4(a, mode, t, s) : launch_lut_q2(a, mode, t, s);
}

}  // namespace coset
