"""Which kernels a call runs, on the CPU: the planners' choices need no GPU."""
import pytest

from kernels_amd import kq
from tests._util import REFUSED, SKINNY, int4_route, moe_gate_up_partitions, vq_takes_skinny

VALU, MFMA = kq.PATH_VALU, kq.PATH_MFMA


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


# AUTO's choice where the skinny kernels were slower than the path they had
# replaced (measured by 6% to 44%), and where they are the faster one.
@pytest.mark.parametrize("M,K,G,batch,inter,want", [
    (8192, 28672, 32, 2, True, VALU), (13824, 5120, 32, 2, True, VALU),
    (23570, 18784, 32, 3, True, VALU), (6912, 1792, 32, 3, True, VALU),
    (18816, 2048, 64, 16, False, MFMA), (20138, 2688, 64, 13, False, MFMA),
    (18598, 2944, 64, 13, True, MFMA), (14336, 4096, 64, 16, False, MFMA),
    (24570, 640, 64, 15, True, MFMA),
    (7089, 6144, 64, 11, True, MFMA), (14336, 4096, 64, 8, True, MFMA),
    (28672, 8192, 64, 8, True, MFMA), (28672, 8192, 128, 16, False, MFMA),
    (4096, 4096, 64, 8, True, SKINNY), (1024, 4096, 64, 8, True, SKINNY),
    (4096, 14336, 64, 8, True, SKINNY), (8192, 28672, 128, 16, False, SKINNY),
    (4096, 24448, 64, 8, True, SKINNY), (18205, 3456, 64, 7, False, SKINNY),
    (20361, 1024, 64, 11, False, SKINNY), (5003, 2848, 32, 4, True, SKINNY), (2880, 5024, 32, 4, True, SKINNY),
    (4096, 4096, 64, 1, True, VALU), (1024, 4096, 64, 2, True, VALU),
])
def test_int4_auto_route(M, K, G, batch, inter, want):
    assert int4_route(M, K, G, batch, inter) == want


# Separate 128-wide groups with an odd number of spans: the skinny kernels where
# the matrix cores are asked for or chosen, int4_mfma where K is too short for them
# or its launch shape is given.
def test_int4_odd_spans_route():
    for batch in (1, 5, 16):
        assert int4_route(300, 128, 128, batch, False, MFMA) == MFMA
        assert int4_route(300, 1152, 128, batch, False, MFMA) == SKINNY
        for forced in ((1, 12), (3, 24), (9, 12), (3, 42)):
            assert int4_route(300, 1152, 128, batch, False, MFMA, forced=forced) == MFMA
        assert int4_route(300, 1152, 128, batch, False, MFMA, forced=(2, 12)) == REFUSED
        assert int4_route(300, 1152, 128, batch, False, MFMA, meta8=False) == REFUSED
    assert int4_route(640, 13440, 128, 5, False) == SKINNY
    assert int4_route(300, 128, 128, 16, False) == MFMA


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
    assert moe_gate_up_partitions(d, batch) == part
