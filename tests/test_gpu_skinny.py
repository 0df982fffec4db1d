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
from tests._util import assert_close, dev, inf_rel, to_f64

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


# The skinny kernels' edges, against the vector path's oracle: K = one pair of
# spans, a last pair that overlaps, several rounds, partial tiles and last
# workgroups, one K part and many, both x forms (8 / 9 tokens), every layout.
# 2e-3 + 1e-4 |y|: float32 sums of products that carry up to 1024 + q are 1.3e-5
# of y's size (up to ~30) off, five times that at the worst of 1e5 values; the
# small shapes that another path takes included.
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


# The same for codebook weights: codebooks that end inside a tile or are
# smaller than a workgroup's share (the passes), shares widened to divide one,
# scale groups of every form.
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


# The same in int4_mfma: K too short for the skinny kernels, and its launch shape
# given (P, 10 T + ring depth; none divides its spans evenly into windows). The last
# row's last scale, and its bias, are the last two bytes of their arrays. 5e-5 of
# the largest value: sums of products that carry 64 and 1024 + q are up to 1.4e-5 off.
@pytest.mark.parametrize("M,K,parts,unroll", [(300, 128, 0, 0), (17, 128, 1, 42), (300, 1152, 1, 12), (257, 1152, 9, 12),
                                              (300, 1152, 3, 24), (4097, 1152, 3, 42)])
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
