"""Config 2: the batched skinny int4 GEMM at its own shapes, W 28672 x 8192
(70B-class FFN up) and 8192 x 28672 (down), group 64, X fp16 [B][K] ~ N(0, 1),
for B in {1, 2, 3, 4, 8, 16}, on the vector path, the matrix-core path and AUTO,
each against the fp64 oracle through the C ABI.

The batch-B oracle is the batch-1 oracle applied per row of X (no reference
kernel takes a batch), so the fp64 result at B = 16 is computed once per
shape and its first B rows are the expected output at B.

Bar: |got - ref| <= 1e-2 + 1e-3 |ref| (fp16 y, fp32 accumulation) and the
reference harness's max|d| / max|ref| < 2e-3 (int4-gemv/src/main.mm:475-479).
"""
import numpy as np
import pytest
import torch

import oracle
from kernels_amd import gen, kq
from tests._util import (SKINNY as SKINNY_PATH, SkinnyPlan, assert_close, dev, inf_rel, int4_route, to_f64,
                         vq_skinny_plan, vq_takes_skinny)

pytestmark = pytest.mark.gpu

SHAPES = [(28672, 8192), (8192, 28672)]
BATCHES = [1, 2, 3, 4, 8, 16]
PATHS = {"valu": kq.PATH_VALU, "mfma": kq.PATH_MFMA, "auto": kq.PATH_AUTO}


@pytest.fixture(scope="module", params=SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def problem(request, gpu):
    M, K = request.param
    p = gen.int4_problem(M, K, 64, batch=16, seed=M // 7 + K)
    ref = oracle.int4_gemv(p["W"], p["SB"], None, p["X"], M, K, 64, 1)  # [16][M]
    bufs = dict(W=dev(p["W"], gpu), SB=dev(p["SB"], gpu), X=dev(p["X"], gpu))
    yield M, K, bufs, ref
    del bufs
    torch.cuda.empty_cache()


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("batch", BATCHES)
def test_config2_skinny(problem, batch, path):
    M, K, b, ref = problem
    Y = torch.full((batch, M), float("nan"), dtype=torch.float16, device=b["W"].device)
    kq.int4_gemv(b["W"], b["SB"], b["X"][:batch], Y, kq.GemvParams(M, K, 64), batch=batch,
                 path=PATHS[path])
    torch.cuda.synchronize()
    got = to_f64(Y)
    what = f"{M}x{K} batch {batch} path {path}"
    assert_close(got, ref[:batch], what=what)
    assert inf_rel(got, ref[:batch]) < 2e-3, what


# The skinny kernels' edges in one round, against the oracle: K = one pair of spans,
# a last pair that overlaps, partial tiles and last workgroups, one K part and
# many, both x forms (8 / 9 tokens), every layout. Where they run (AUTO takes another
# path for some of these), 1e-5 of the largest value: float32 sums of products that
# carry 64 + q measure about 1e-6. Elsewhere 2e-3 + 1e-4 |y|: products that carry up to
# 1024 + q are 1.3e-5 of y's size (up to ~30) off, five times that at the worst of
# 1e5 values.
SKINNY = [(1, 256, 64), (17, 288, 32), (300, 608, 32), (4097, 320, 64), (9000, 256, 128),
          (5003, 2848, 32), (2880, 5056, 64), (6144, 1152, 128)]


@pytest.mark.parametrize("layout,sb", [("sb", kq.F16), ("sb", kq.BF16), ("split", kq.F16), ("split", kq.BF16)])
@pytest.mark.parametrize("M,K,G", SKINNY)
def test_skinny_edges(gpu, M, K, G, layout, sb):
    for batch in (5, 8, 9, 16):
        p = gen.int4_problem(M, K, G, batch=batch, seed=M + K + batch)
        if sb == kq.BF16:
            f = lambda a: gen.bf16_bits(a.view(np.float16).astype(np.float32))  # noqa: E731
            p = dict(p, S=f(p["S"]), B=f(p["B"]), SB=f(p["SB"]))
        S, B = (p["SB"], None) if layout == "sb" else (p["S"], p["B"])
        y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
        kq.int4_gemv(dev(p["W"], gpu), dev(S, gpu), dev(p["X"], gpu), y, kq.GemvParams(M, K, G),
                     B=None if B is None else dev(B, gpu), batch=batch, sb_dtype=sb)
        torch.cuda.synchronize()
        ref = oracle.int4_gemv(p["W"], S, B, p["X"], M, K, G, layout == "sb",
                               oracle.BF16 if sb == kq.BF16 else oracle.F16)
        assert_close(to_f64(y), ref, atol=2e-3, rtol=1e-4, what=f"{M}x{K} g{G} {layout} b{batch}")
        if int4_route(M, K, G, batch, layout == "sb") == SKINNY_PATH:
            assert inf_rel(to_f64(y), ref) < 1e-5, f"{M}x{K} g{G} {layout} b{batch}"


# Plans that AUTO takes beyond those edges, (T tiles a wave, K parts > 1, rounds > 1,
# J > 4 pairs a part: a second window of scales) by layout and x form: one wave's
# tiles and windows, the K-part sums over rounds in both buffers, rounds without K
# parts. The plan is asserted, so that a change of the planner cannot empty the test.
PLANS = [  # M, K, G, layout, batch, (T, P > 1, rounds > 1, J > 4)
    (64, 9472, 32, "split", 9, (1, True, False, True)), (76, 8832, 32, "sb", 9, (1, True, False, True)),
    (813, 10240, 32, "sb", 8, (1, True, False, True)), (65, 11648, 64, "split", 8, (1, True, False, True)),
    (66, 8576, 64, "split", 9, (1, True, False, True)), (112, 11648, 64, "sb", 8, (1, True, False, True)),
    (65, 9344, 64, "sb", 9, (1, True, False, True)), (66, 11648, 128, "split", 8, (1, True, False, True)),
    (66, 8448, 128, "split", 9, (1, True, False, True)), (101, 11648, 128, "sb", 8, (1, True, False, True)),
    (68, 8320, 128, "sb", 9, (1, True, False, True)),
    (8267, 4128, 32, "split", 9, (2, True, False, True)), (4326, 8224, 32, "sb", 5, (2, True, False, True)),
    (4128, 8704, 64, "split", 5, (2, True, False, True)), (8314, 4160, 64, "split", 9, (2, True, False, True)),
    (4105, 8256, 64, "sb", 5, (2, True, False, True)), (4364, 8576, 128, "split", 5, (2, True, False, True)),
    (8659, 1088, 64, "sb", 9, (4, True, False, False)), (8209, 1152, 128, "split", 9, (4, True, False, False)),
    (8351, 1152, 128, "sb", 9, (4, True, False, False)), (65547, 256, 64, "sb", 8, (4, False, False, False)),
    (65636, 256, 64, "split", 8, (4, False, False, False)), (65538, 256, 128, "split", 8, (4, False, False, False)),
    (34268, 800, 32, "split", 9, (2, True, True, False)), (16837, 1568, 32, "sb", 9, (2, True, True, False)),
    (33669, 832, 64, "split", 9, (2, True, True, False)), (65706, 288, 32, "sb", 2, (2, True, True, False)),
    (65725, 320, 64, "sb", 2, (2, True, True, False)), (65557, 384, 128, "sb", 2, (2, True, True, False)),
    (66000, 256, 32, "sb", 5, (2, False, True, False)), (66000, 256, 32, "split", 9, (2, False, True, False)),
    (132000, 256, 64, "split", 5, (2, False, True, False)), (132000, 256, 128, "sb", 9, (2, False, True, False)),
]


@pytest.mark.parametrize("M,K,G,layout,batch,want", PLANS)
def test_skinny_plans(gpu, M, K, G, layout, batch, want):
    pl = SkinnyPlan()
    assert int4_route(M, K, G, batch, layout == "sb", plan=pl) == SKINNY_PATH
    assert (pl.T, pl.P > 1, pl.rounds > 1, pl.J > 4) == want
    p = gen.int4_problem(M, K, G, batch=batch, seed=M + K + batch)
    S, B = (p["SB"], None) if layout == "sb" else (p["S"], p["B"])
    y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
    kq.int4_gemv(dev(p["W"], gpu), dev(S, gpu), dev(p["X"], gpu), y, kq.GemvParams(M, K, G),
                 B=None if B is None else dev(B, gpu), batch=batch)
    torch.cuda.synchronize()
    ref = oracle.int4_gemv(p["W"], S, B, p["X"], M, K, G, layout == "sb", oracle.F16)
    assert inf_rel(to_f64(y), ref) < 1e-5


# Separate scales and biases at any multiple of 2 bytes (the skinny kernels load
# them as words), codebook scales too.
@pytest.mark.parametrize("M,K,G", [(300, 608, 32), (4097, 320, 64), (2880, 5056, 64), (6144, 1152, 128)])
@pytest.mark.parametrize("batch", [8, 16])
def test_skinny_scales_at_2_mod_4(gpu, M, K, G, batch):
    p = gen.int4_problem(M, K, G, batch=batch, seed=M + K)

    def odd(a):  # the same values, two bytes on
        t = torch.zeros(a.size + 1, dtype=torch.int16, device=gpu)
        t[1:] = dev(a, gpu).view(-1)
        assert t[1:].data_ptr() % 4 == 2
        return t[1:]
    if G != 32 or batch > 8:
        assert int4_route(M, K, G, batch, False, meta8=False) == SKINNY_PATH
    y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
    kq.int4_gemv(dev(p["W"], gpu), odd(p["S"]), dev(p["X"], gpu), y, kq.GemvParams(M, K, G), B=odd(p["B"]),
                 batch=batch)
    torch.cuda.synchronize()
    ref = oracle.int4_gemv(p["W"], p["S"], p["B"], p["X"], M, K, G, False, oracle.F16)
    assert inf_rel(to_f64(y), ref) < (1e-5 if G != 32 or batch > 8 else 1e-4)
    q = gen.vq_problem(M, K, rows_per_cb=M, scale_group=32, batch=batch, seed=M)
    assert vq_takes_skinny(M, K, M, 32, batch)
    kq.vq_gemv(dev(q["IDX"], gpu), dev(q["C"], gpu), odd(q["S"]), dev(q["X"], gpu), y, kq.VQParams(M, K, M, 32),
               batch=batch)
    torch.cuda.synchronize()
    ref = oracle.vq_gemv(q["IDX"], q["C"], q["S"], q["X"], M, K, M, 32)
    assert inf_rel(to_f64(y), ref) < 2e-6


# The same for codebook weights, by scale form (a group of 32, 64, 128 or more, a
# scale per row).
VQ_PLANS = [  # M, K, rows_per_cb, scale_group, batch, (T, P > 1, rounds > 1, J > 4)
    (65, 10240, 256, 10240, 5, (1, True, False, True)), (67, 8704, 256, 8704, 9, (1, True, False, True)),
    (64, 10240, 2048, 32, 5, (1, True, False, True)), (64, 8704, 4096, 32, 9, (1, True, False, True)),
    (64, 10240, 512, 64, 5, (1, True, False, True)), (64, 8704, 512, 64, 9, (1, True, False, True)),
    (70, 10240, 2048, 512, 5, (1, True, False, True)), (64, 8704, 256, 512, 9, (1, True, False, True)),
    (65608, 512, 2048, 512, 2, (4, False, False, False)), (8336, 1536, 2048, 1536, 9, (4, True, False, False)),
    (65711, 512, 512, 64, 2, (4, False, False, False)), (8439, 1536, 4096, 64, 9, (4, True, False, False)),
    (66937, 512, 2048, 128, 2, (4, False, False, False)), (8194, 1536, 4096, 512, 9, (4, True, False, False)),
    (66237, 512, 66237, 512, 2, (2, True, True, False)), (70220, 512, 70220, 32, 2, (2, True, True, False)),
    (32998, 1024, 32998, 32, 9, (2, True, True, False)), (66138, 512, 4096, 32, 2, (2, False, True, False)),
    (65949, 512, 512, 32, 9, (2, False, True, False)),
]


@pytest.mark.parametrize("M,K,rpc,sg,batch,want", VQ_PLANS)
def test_skinny_vq_plans(gpu, M, K, rpc, sg, batch, want):
    assert vq_takes_skinny(M, K, rpc, sg, batch)
    pl = vq_skinny_plan(M, K, rpc, sg, batch)
    assert (pl.T, pl.P > 1, pl.rounds > 1, pl.J > 4) == want
    p = gen.vq_problem(M, K, rows_per_cb=rpc, scale_group=sg, batch=batch, seed=M + K + batch)
    y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
    kq.vq_gemv(dev(p["IDX"], gpu), dev(p["C"], gpu), dev(p["S"], gpu), dev(p["X"], gpu), y,
               kq.VQParams(M, K, rpc, sg), batch=batch)
    torch.cuda.synchronize()
    ref = oracle.vq_gemv(p["IDX"], p["C"], p["S"], p["X"], M, K, rpc, sg)
    assert inf_rel(to_f64(y), ref) < 2e-6  # float32 sums: about 1e-7


# The edges for codebook weights: codebooks that end inside a tile or are smaller
# than a workgroup's share (the passes), shares widened to divide one, scale groups
# of every form.
SKINNY_VQ = [(1, 256, 1, 256), (300, 288, 256, 288), (4100, 512, 256, 32), (700, 608, 16, 608),
             (5000, 1024, 256, 64), (3000, 2048, 7, 2048), (9000, 256, 256, 128),
             (2000, 5120, 2000, 512), (2900, 1088, 256, 32)]


@pytest.mark.parametrize("M,K,rpc,sg", SKINNY_VQ)
def test_skinny_vq_edges(gpu, M, K, rpc, sg):
    for batch in (3, 5, 8, 9, 16):
        p = gen.vq_problem(M, K, rows_per_cb=rpc, scale_group=sg, batch=batch, seed=M + K + batch)
        y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
        kq.vq_gemv(dev(p["IDX"], gpu), dev(p["C"], gpu), dev(p["S"], gpu), dev(p["X"], gpu), y,
                   kq.VQParams(M, K, rpc, sg), batch=batch)
        torch.cuda.synchronize()
        ref = oracle.vq_gemv(p["IDX"], p["C"], p["S"], p["X"], M, K, rpc, sg)
        assert_close(to_f64(y), ref, atol=2e-5, rtol=1e-6, what=f"vq {M}x{K} cb{rpc} sg{sg} b{batch}")


# Separate scales of 128-wide groups with an odd number of spans, which
# int4_mfma does not take: the matrix-core path asked for by name, and a K that
# the vector path's LDS does not hold. 1e-5 of the largest value: float32 sums of
# products that carry 64 + q measure about 1e-6.
@pytest.mark.parametrize("M,K,path", [(300, 1152, kq.PATH_MFMA), (17, 131200, kq.PATH_AUTO)])
def test_odd_spans_split_g128(gpu, M, K, path):
    for batch in (1, 5, 16):
        p = gen.int4_problem(M, K, 128, batch=batch, seed=K + batch)
        y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
        kq.int4_gemv(dev(p["W"], gpu), dev(p["S"], gpu), dev(p["X"], gpu), y, kq.GemvParams(M, K, 128),
                     B=dev(p["B"], gpu), batch=batch, path=path)
        torch.cuda.synchronize()
        ref = oracle.int4_gemv(p["W"], p["S"], p["B"], p["X"], M, K, 128, False, oracle.F16)
        assert inf_rel(to_f64(y), ref) < 1e-5, f"{M}x{K} b{batch}"


# The same in int4_mfma, wherever a K part has an odd number of spans: K too short
# for the skinny kernels, the launch shape given (P, 10 T + ring depth), and an even
# number of spans cut into odd parts, by a given P or the planner's (512 and 2048 at
# few rows). The last row's last scale, and its bias, are the last two bytes of
# their arrays. 5e-5 of the largest value: sums of products that carry 64 and 1024 +
# q are up to 1.4e-5 off.
@pytest.mark.parametrize("M,K,parts,unroll", [(300, 128, 0, 0), (17, 128, 1, 42), (300, 1152, 1, 12), (257, 1152, 9, 12),
                                              (300, 1152, 3, 24), (4097, 1152, 3, 42), (2, 512, 0, 0),
                                              (300, 2048, 0, 0), (17, 1536, 4, 12), (17, 1536, 4, 24),
                                              (300, 256, 2, 42), (100, 14336, 16, 12)])
def test_odd_spans_split_g128_int4_mfma(gpu, M, K, parts, unroll):
    for batch in (1, 5, 16):
        p = gen.int4_problem(M, K, 128, batch=batch, seed=K + batch + parts)
        y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
        kq.int4_gemv(dev(p["W"], gpu), dev(p["S"], gpu), dev(p["X"], gpu), y, kq.GemvParams(M, K, 128),
                     B=dev(p["B"], gpu), batch=batch, path=kq.PATH_MFMA, rows=parts, unroll=unroll)
        torch.cuda.synchronize()
        ref = oracle.int4_gemv(p["W"], p["S"], p["B"], p["X"], M, K, 128, False, oracle.F16)
        assert inf_rel(to_f64(y), ref) < 5e-5, f"{M}x{K} P{parts} T,D {unroll} b{batch}"
        assert inf_rel(to_f64(y)[:, -1:], ref[:, -1:]) < 5e-4, "the last row"


# Codebook blocks of an odd tile count: the skinny kernels with a workgroup a
# block, or the passes, whichever the route gives.
@pytest.mark.parametrize("M,K,rpc,sg", [(5120, 512, 1264, 512), (2768, 1056, 592, 32), (4128, 288, 1376, 288)])
def test_vq_uneven_codebook_blocks(gpu, M, K, rpc, sg):
    for batch in (3, 8, 16):
        p = gen.vq_problem(M, K, rows_per_cb=rpc, scale_group=sg, batch=batch, seed=M + K + batch)
        y = torch.full((batch, M), float("nan"), dtype=torch.float32, device=gpu)
        kq.vq_gemv(dev(p["IDX"], gpu), dev(p["C"], gpu), dev(p["S"], gpu), dev(p["X"], gpu), y,
                   kq.VQParams(M, K, rpc, sg), batch=batch)
        torch.cuda.synchronize()
        ref = oracle.vq_gemv(p["IDX"], p["C"], p["S"], p["X"], M, K, rpc, sg)
        assert_close(to_f64(y), ref, atol=2e-5, rtol=1e-6, what=f"vq {M}x{K} cb{rpc} sg{sg} b{batch}")
