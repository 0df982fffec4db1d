// kq_skinny_i4_g128.hip -- the skinny matrix-core kernels of int4 weights in
// quant groups of 128 (kq_skinny_kernel.h).
#include "kq_skinny_kernel.h"

namespace kq {

hipError_t launch_skinny_i4_g128(const skinny::Args& a, const skinny::Plan& pl, bool sb, bool bf,
                               hipStream_t s) {
    if (sb) return bf ? skinny::dispatch<0, 128, true, true>(a, pl, s) : skinny::dispatch<0, 128, true, false>(a, pl, s);
    return bf ? skinny::dispatch<0, 128, false, true>(a, pl, s) : skinny::dispatch<0, 128, false, false>(a, pl, s);
}

}  // namespace kq
