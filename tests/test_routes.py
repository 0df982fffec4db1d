"""Which kernels a call runs, on the CPU: the planners' choices need no GPU (256
compute units are assumed without one). The functions are libkq's own C++ ones,
declared in kernels_amd/csrc/kq_internal.h."""
import ctypes as C

import pytest

from kernels_amd import kq


def vq_takes_skinny(*args):
    f = kq.lib()["_ZN2kq15vq_takes_skinnyEjjjjj"]
    f.restype = C.c_bool
    return f(*(C.c_uint32(a) for a in args))


# Codebook blocks whose tiles divide badly would leave the skinny kernels 5-32
# workgroups (measured up to 39 times slower than the passes): the passes take
# them at every token count. Blocks of a power of 2, or one codebook: skinny.
@pytest.mark.parametrize("M,K,rpc,skinny", [
    (11008, 4096, 1376, False), (18944, 3584, 592, False), (5120, 5120, 1264, False),
    (28672, 8192, 1072, False), (28672, 8192, 4112, False), (8373, 3904, 6928, False),
    (14336, 4096, 256, True), (4096, 14336, 4096, True), (4096, 4096, 512, True),
])
def test_vq_route_follows_the_plans_duration(M, K, rpc, skinny):
    for sg in (32, K):
        for batch in (3, 5, 8, 16):
            assert vq_takes_skinny(M, K, rpc, sg, batch) == skinny, (sg, batch)
