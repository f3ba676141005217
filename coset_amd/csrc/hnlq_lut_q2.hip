// hnlq_lut_q2.hip -- the q = 2 instantiations of the table codec (hnlq_lut_kernels.hpp).
#include "hnlq_lut_kernels.hpp"

namespace coset {

hipError_t launch_lut_q2(const CodecArgs& a, int mode, const DecodeTables* t, hipStream_t s)
{
    switch (mode) {
    case MODE_ENCODE: return launch_q<2, MODE_ENCODE>(a, t, s);
    case MODE_DECODE: return launch_q<2, MODE_DECODE>(a, t, s);
    default: return launch_q<2, MODE_ROUNDTRIP>(a, t, s);
    }
}

}  // namespace coset
