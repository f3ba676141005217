// hnlq_lut_q4.hip -- the q = 4 instantiations of the table codec (hnlq_lut_kernels.hpp).
#include "probes.hpp"
#include "hnlq_lut_kernels.hpp"

namespace coset {

hipError_t launch_lut_q4(const CodecArgs& a, int mode, const DecodeTables* t, hipStream_t s)
{
    switch (mode) {
    case MODE_ENCODE: return launch_q<4, MODE_ENCODE>(a, t, s);
    case MODE_DECODE: return launch_q<4, MODE_DECODE>(a, t, s);
    default: return launch_q<4, MODE_ROUNDTRIP>(a, t, s);
    }
}

hipError_t launch_c2_stream_probe(const float* x, int64_t n, uint32_t* packed, float* out, int staged, hipStream_t s)
{
    CodecArgs a{};
    a.x = x;
    a.x_dtype = DT_F32;
    a.n = n;
    a.q = 4;
    a.M = 2;
    a.packed = packed;
    a.out = out;
    a.out_dtype = DT_F32;
    const DecodeTables* t = nullptr;
    hipError_t e = get_decode_tables(4, 0, &t);
    if (e != hipSuccess) return e;
    const int grid = (int)std::min<int64_t>((n + kLutThreads - 1) / kLutThreads, (int64_t)cu_count());
    const TileCounters tiles = g_codec_dynamic ? take_counters(s) : TileCounters{nullptr, nullptr, -1};
    if (staged)
        hipLaunchKernelGGL((hnlq_plain_kernel<4, 2, MODE_ROUNDTRIP, SC_NONE, false, true, false, false, 1>), dim3(grid),
                           dim3(kLutThreads), 0, s, a, t->cid_map, t->swar, t->n_coarse, t->swar_bias[2], tiles);
    else
        hipLaunchKernelGGL((hnlq_plain_kernel<4, 2, MODE_ROUNDTRIP, SC_NONE, false, true, false, false, 2>), dim3(grid),
                           dim3(kLutThreads), 0, s, a, t->cid_map, t->swar, t->n_coarse, t->swar_bias[2], tiles);
    e = hipGetLastError();
    if (e != hipSuccess) return_counters(tiles);
    return e;
}

}  // namespace coset
