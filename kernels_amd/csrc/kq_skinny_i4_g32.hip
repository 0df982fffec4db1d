// kq_skinny_i4_g32.hip -- the skinny matrix-core kernels of int4 weights in
// quant groups of 32 (kq_skinny_kernel.h).
#include "kq_skinny_kernel.h"

namespace kq {

hipError_t launch_skinny_i4_g32(const skinny::Args& a, const skinny::Plan& pl, bool sb, bool bf,
                               hipStream_t s) {
    if (sb) return bf ? skinny::dispatch<0, 32, true, true>(a, pl, s) : skinny::dispatch<0, 32, true, false>(a, pl, s);
    return bf ? skinny::dispatch<0, 32, false, true>(a, pl, s) : skinny::dispatch<0, 32, false, false>(a, pl, s);
}

}  // namespace kq
