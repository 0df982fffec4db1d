"""Shared helpers for the tests (device upload, tolerance checks, the planners'
choices)."""
import ctypes as C

import numpy as np

# Tolerance for fp16/fp32 outputs with fp32 accumulation, read as allclose:
# |got - ref| <= ATOL + RTOL * |ref|  (max-abs 1e-2, rel 1e-3).
ATOL = 1e-2
RTOL = 1e-3


def dev(arr, device):
    """numpy array -> torch tensor on `device` with the same bytes.
    uint32 -> int32, uint16 -> int16 storage (kernels see raw bits)."""
    import torch
    a = np.ascontiguousarray(arr)
    view = {np.dtype(np.uint32): np.int32, np.dtype(np.uint16): np.int16,
            np.dtype(np.uint8): np.uint8}.get(a.dtype)
    if view is not None:
        a = a.view(view)
    return torch.from_numpy(a).to(device)


def host_bits(t, dtype):
    """torch tensor -> numpy array reinterpreted as `dtype`."""
    import torch
    a = t.detach().cpu()
    if a.dtype in (torch.float16, torch.bfloat16):
        a = a.view(torch.int16)
    return a.numpy().view(dtype)


def to_f64(t):
    import torch
    return t.detach().to(torch.float64).cpu().numpy()


def assert_close(got, ref, atol=ATOL, rtol=RTOL, what=""):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    assert got.shape == ref.shape, (got.shape, ref.shape)
    assert np.all(np.isfinite(got)), f"{what}: non-finite output"
    err = np.abs(got - ref)
    bad = err > atol + rtol * np.abs(ref)
    if bad.any():
        i = np.flatnonzero(bad.ravel())[:5]
        raise AssertionError(
            f"{what}: {bad.sum()} of {bad.size} outside atol={atol} rtol={rtol}; "
            f"first at {i.tolist()}: got {got.ravel()[i].tolist()} ref {ref.ravel()[i].tolist()}; "
            f"max abs err {err.max():.3e}")


def inf_rel(got, ref):
    """The reference harness's metric: max|got-ref| / max|ref|
    (int4-gemv/src/main.mm:470-476)."""
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    return float(np.max(np.abs(got - ref)) / max(1e-30, np.max(np.abs(ref))))


def tie_weights(M, K, seed):
    """Weights [M][K] float32 (for one scale per row: every row's is 1) whose
    pairs crowd 144 places with coordinates halfway between two fp16 values, or
    one float32 step above: cluster means lie a fraction of a step above the
    tie, where rounding through float32 goes the other way."""
    rng = np.random.default_rng(seed)
    tie = (0.5 + (4 * np.arange(12) * 40 + 1) * 2.0**-12).astype(np.float32)
    W = rng.choice(tie, (M, K)).astype(np.float32)
    W += (rng.random((M, K)) < 0.3).astype(np.float32) * np.float32(2.0**-24)
    W[:, :2] = 1.0
    return W


# ---- which kernels a call runs, and how: libkq's own C++ functions, declared in
# kernels_amd/csrc/kq_internal.h (256 compute units are assumed without a GPU)
class SkinnyPlan(C.Structure):
    """kq::skinny::Plan: T tiles a wave, P K parts x Q row lanes, J pairs of spans
    a part, rounds a workgroup."""
    _fields_ = ([(n, C.c_uint32) for n in ("T", "P", "Q", "J", "NP", "rounds", "tiles_wg", "nwg")] +
                [(n, C.c_size_t) for n in ("part_lds", "x_lds")])


SKINNY, REFUSED = 4, 0  # int4_route beside kq.PATH_VALU, _MFMA and _SCALAR


def _internal(name, restype):
    from kernels_amd import kq
    f = kq.lib()[name]
    f.restype = restype
    return f


def int4_route(M, K, G, batch, inter, path=0, meta8=True, forced=None, plan=None):
    """The path of an int4 call; a SkinnyPlan given as plan is filled for SKINNY."""
    f = _internal("_ZN2kq10int4_routeEjjjjbbiPNS_6skinny4PlanEPKNS_7Int4CfgE", C.c_int)
    return f(*(C.c_uint32(a) for a in (M, K, G, batch)), C.c_bool(inter), C.c_bool(meta8), C.c_int(path),
             C.byref(plan) if plan else None, (C.c_int * 2)(*forced) if forced else None)


def vq_takes_skinny(M, K, rpc, sg, batch):
    f = _internal("_ZN2kq15vq_takes_skinnyEjjjjj", C.c_bool)
    return f(*(C.c_uint32(a) for a in (M, K, rpc, sg, batch)))


def vq_skinny_plan(M, K, rpc, sg, batch):
    f = _internal("_ZN2kq14vq_skinny_planEjjjjjRNS_6skinny4PlanE", C.c_bool)
    p = SkinnyPlan()
    assert f(*(C.c_uint32(a) for a in (M, K, rpc, sg, batch)), C.byref(p))
    return p


def moe_gate_up_partitions(d, batch):
    f = _internal("_ZN2kq22moe_gate_up_partitionsERK11kq_moe_descj", C.c_bool)
    return f(C.byref(d), C.c_uint32(batch))
