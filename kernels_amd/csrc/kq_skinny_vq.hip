// kq_skinny_vq.hip -- the skinny matrix-core kernels of codebook weights
// (kq_skinny_kernel.h). gm: the kernel's scale form (32, 64, 128 or 0).
#include "kq_skinny_kernel.h"

namespace kq {

namespace {
// The lookups address the codebooks from LDS address 0, where the dynamic area
// starts only while the kernel has no static LDS.
template <int GM, int T, bool X8>
bool from_zero() {
    static const bool ok = [] {
        hipFuncAttributes at{};
        return hipFuncGetAttributes(&at, reinterpret_cast<const void*>(
                                             skinny::skinny_k<1, GM, false, false, T, X8>)) == hipSuccess &&
               at.sharedSizeBytes == 0;
    }();
    return ok;
}
template <int GM>
bool all_from_zero() {
    bool ok = from_zero<GM, 1, false>() && from_zero<GM, 1, true>() && from_zero<GM, 2, false>() &&
              from_zero<GM, 2, true>();
    if constexpr (GM != 32) ok = ok && from_zero<GM, 4, false>() && from_zero<GM, 4, true>();
    return ok;
}
}  // namespace

bool skinny_vq_usable(int gm) {
    switch (gm) {
        case 0: return all_from_zero<0>();
        case 32: return all_from_zero<32>();
        case 64: return all_from_zero<64>();
        default: return all_from_zero<128>();
    }
}

hipError_t launch_skinny_vq_gm(const skinny::Args& a, const skinny::Plan& pl, int gm, hipStream_t s) {
    switch (gm) {
        case 0: return skinny::dispatch<1, 0, false, false>(a, pl, s);
        case 32: return skinny::dispatch<1, 32, false, false>(a, pl, s);
        case 64: return skinny::dispatch<1, 64, false, false>(a, pl, s);
        default: return skinny::dispatch<1, 128, false, false>(a, pl, s);
    }
}

}  // namespace kq
