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


# Standalone gate/up: the streaming (2 tokens) or per-tile kernel where the
# partitioned kernel's plan and staging of every token's x cost more than it
# saves (measured 1.1 to 1.56 times as long on the False rows).
@pytest.mark.parametrize("hidden,inter,ne,tk,batch,part", [
    (704, 2304, 82, 1, 12, False), (2048, 512, 12, 2, 2, False), (1024, 1024, 8, 1, 2, False),
    (576, 3584, 43, 2, 8, False), (640, 1600, 45, 2, 8, False), (1024, 1024, 72, 4, 16, False),
    (2880, 2880, 128, 4, 1, False), (2880, 2880, 128, 4, 3, True), (2880, 2880, 128, 4, 16, True),
    (3072, 512, 8, 8, 16, True),
])
def test_standalone_gate_up_route(hidden, inter, ne, tk, batch, part):
    d = kq.MoEDesc(hidden=hidden, inter=inter, n_experts=ne, top_k=tk, blob=1 << 25)
    f = kq.lib()["_ZN2kq22moe_gate_up_partitionsERK11kq_moe_descj"]
    f.restype = C.c_bool
    assert f(C.byref(d), C.c_uint32(batch)) == part
