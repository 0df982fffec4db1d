"""The work a decode loop gives this library, as cases to be timed and compared.

Kinds of case (the "kind" of the dict):

  int4      the int4 group-affine projections of one or more transformer
            layers, 1 to 16 tokens (kq.int4_gemv)
  vq        the same with codebook (VQ) weights (kq.vq_gemv)
  quantize  a dense matrix into the VQ format (kq.vq_quantize), the offline
            step before `vq`
  moe       mixture-of-experts blocks in the gpt-oss expert-blob layout,
            1 to 16 tokens (kq.moe_block, or its three passes one by one)

A stack of layers has its own weights per layer, as a model has: one layer of
a served model never finds its weights in a cache, because all the others were
read since. Where a case is marked "graph" the calls of one pass are captured
once in `prepare` and replayed, which is how a serving loop runs the launches
of a decode step; the others are plain calls.
"""
import math

import torch

from kernels_amd import kq

DEV = "cuda"

LLAMA_8B = "4096x4096+1024x4096+1024x4096+4096x4096+14336x4096+14336x4096+4096x14336"
MLP_8B = "14336x4096+14336x4096+4096x14336"
MLP_70B = "28672x8192+8192x28672"


def _int4(name, mats, layers, batch, G=64, meta="f16", split=False, out="f16", graph=True):
    return {"name": name, "kind": "int4", "mats": mats, "layers": layers, "batch": batch, "G": G,
            "meta": meta, "split": split, "out": out, "graph": graph}


def _vq(name, mats, layers, batch, cb_rows, scale_group, out="f16", graph=True):
    """cb_rows 0: one codebook per matrix; scale_group 0: one scale per row."""
    return {"name": name, "kind": "vq", "mats": mats, "layers": layers, "batch": batch,
            "cb_rows": cb_rows, "scale_group": scale_group, "out": out, "graph": graph}


def _quantize(name, M, K, cb_rows, scale_group, dtype, iters=25, sample=200_000):
    return {"name": name, "kind": "quantize", "M": M, "K": K, "cb_rows": cb_rows,
            "scale_group": scale_group, "dtype": dtype, "iters": iters, "sample": sample}


def _moe(name, layers, batch, hidden=2880, inter=2880, experts=128, top_k=4, x="f16", out="f32",
         form="block", graph=True):
    return {"name": name, "kind": "moe", "layers": layers, "batch": batch, "hidden": hidden,
            "inter": inter, "experts": experts, "top_k": top_k, "x": x, "out": out, "form": form,
            "graph": graph}


def listed():
    return [
        # the smallest call: one key/value projection of Llama-3-8B, one token
        _int4("int4_kv_proj_b1", "1024x4096", 1, 1, graph=False),
        # one token through all linear layers of Llama-3-8B: the decode step
        _int4("int4_llama8b_step_b1", LLAMA_8B, 32, 1),
        # the same layers for 8 sequences at once (8 of the 32 layers)
        _int4("int4_llama8b_layers_b8", LLAMA_8B, 8, 8),
        # the wide MLP projections of a 70B model at the largest batch, scales
        # and biases in arrays of their own (bf16), float32 results
        _int4("int4_mlp70b_b16", MLP_70B, 1, 16, G=128, meta="bf16", split=True, out="f32",
              graph=False),
        # sizes that fit no tile: odd rows, a K that is no multiple of 64
        _int4("int4_ragged_b4", "5003x2848+2880x5024", 1, 4, G=32, graph=False),
        # VQ MLP of Llama-3-8B, one token, a codebook per 256 rows and a scale
        # per row
        _vq("vq_mlp8b_b1", MLP_8B, 4, 1, 256, 0),
        # VQ MLP at 8 tokens in the reference's format (one codebook per
        # matrix, a scale per 32 weights), float32 results
        _vq("vq_mlp8b_ref_b8", MLP_8B, 4, 8, 0, 32, out="f32"),
        # quantising one MLP matrix of Llama-3-8B from its bf16 checkpoint
        _quantize("vq_quantize_rowscale", 14336, 4096, 256, 0, "bf16"),
        # and into the reference's format from float32
        _quantize("vq_quantize_ref", 4096, 14336, 0, 32, "f32"),
        # gpt-oss-120b MoE blocks, one token
        _moe("moe_gptoss_b1", 8, 1),
        # 8 tokens, the float32 residual stream as input
        _moe("moe_gptoss_b8", 4, 8, x="f32"),
        # the largest batch through the three separate passes (as a caller that
        # streams experts in between does), fp16 results
        _moe("moe_gptoss_calls_b16", 3, 16, out="f16", form="calls", graph=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _stack(rng, M, K, bits):
    """Layers of a drawn matrix: enough to be more than a cache holds, within reason."""
    return max(1, min(_log_int(rng, 1, 8), int(400e6 / (M * K * bits / 8))))


def draw(rng):
    kind = rng.choice(["int4", "int4", "int4", "vq", "vq", "quantize", "moe", "moe"])
    if kind == "int4":
        G = rng.choice([32, 64, 64, 128])
        M, K = _log_int(rng, 256, 28672), max(1, _log_int(rng, 512, 28672) // G) * G
        c = _int4("", "%dx%d" % (M, K), _stack(rng, M, K, 4), _log_int(rng, 1, 16), G,
                  rng.choice(["f16", "bf16"]), rng.random() < 0.4, rng.choice(["f16", "f32"]),
                  rng.random() < 0.6)
    elif kind == "vq":
        sg = rng.choice([0, 0, 32, 32, 128])
        step = sg or 32
        M, K = _log_int(rng, 256, 28672), max(1, _log_int(rng, 512, 28672) // step) * step
        c = _vq("", "%dx%d" % (M, K), _stack(rng, M, K, 4), _log_int(rng, 1, 16),
                rng.choice([0, 256, 256]), sg, rng.choice(["f16", "f32"]), rng.random() < 0.6)
    elif kind == "quantize":
        sg = rng.choice([0, 32, 64])
        step = sg or 32
        M = _log_int(rng, 256, 14336)
        K = max(1, min(_log_int(rng, 512, 14336), 14336 * 4096 // M) // step) * step
        c = _quantize("", M, K, rng.choice([0, 256]), sg, rng.choice(["f32", "f16", "bf16"]),
                      rng.randint(5, 25), _log_int(rng, 20_000, 200_000))
    else:
        hidden, inter = (64 * _log_int(rng, 8, 64) for _ in range(2))
        experts = _log_int(rng, 8, 128)
        c = _moe("", rng.randint(1, 3), _log_int(rng, 1, 16), hidden, inter, experts,
                 min(experts, rng.choice([1, 2, 4, 4, 8])), rng.choice(["f16", "f32"]),
                 rng.choice(["f16", "f32"]), rng.choice(["block", "block", "calls"]),
                 rng.random() < 0.6)
    del c["name"]
    return c


# ---------------------------------------------------------------------------

_FLOAT = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_KQ_META = {"f16": kq.F16, "bf16": kq.BF16}


def _mats(case):
    return [tuple(int(v) for v in m.split("x")) for m in case["mats"].split("+")]


def _words(n, g):
    """n random 32-bit words."""
    return torch.randint(-2**31, 2**31, (n,), dtype=torch.int32, device=DEV, generator=g)


def _normal(shape, g, mean=0.0, std=1.0, dtype=torch.float32):
    t = torch.empty(shape, dtype=torch.float32, device=DEV)
    return t.normal_(mean, std, generator=g).to(dtype)


def _affine(shape, g, dtype):
    """Scales and biases as min/max quantisation of N(0, 0.02) weights in
    groups gives them: the bias is the minimum, the scale a 15th of the span."""
    return _normal(shape, g, 0.0064, 0.001).abs_().to(dtype), _normal(shape, g, -0.048, 0.004, dtype)


def _x(batch, K, g, dtype=torch.float16):
    return _normal((batch, K), g, dtype=dtype)


def _prepare_int4(case, g):
    G, batch, dtype = case["G"], case["batch"], _FLOAT[case["out"]]
    layers = []
    for _ in range(case["layers"]):
        x = {K: _x(batch, K, g) for K in sorted({K for _, K in _mats(case)})}
        calls, total = [], sum(M for M, _ in _mats(case))
        y, at = torch.zeros(batch * total, dtype=dtype, device=DEV), 0
        for M, K in _mats(case):
            S, B = _affine((M, K // G), g, _FLOAT[case["meta"]])
            if not case["split"]:
                S, B = torch.stack([S, B], -1).contiguous(), None
            calls.append((_words(M * K // 8, g).view(M, K // 8), S, B, x[K],
                          y[at:at + batch * M].view(batch, M), kq.GemvParams(M, K, G)))
            at += batch * M
        layers.append((calls, y))

    def go():
        for calls, _ in layers:
            for W, S, B, x, y, P in calls:
                kq.int4_gemv(W, S, x, y, P, B=B, batch=batch, sb_dtype=_KQ_META[case["meta"]])

    return {"layers": layers, "go": go, "out": [y for _, y in layers]}


def _cb_rows(case, M):
    return case["cb_rows"] or M


def _prepare_vq(case, g):
    batch, dtype = case["batch"], _FLOAT[case["out"]]
    layers = []
    for _ in range(case["layers"]):
        x = {K: _x(batch, K, g) for K in sorted({K for _, K in _mats(case)})}
        calls, total = [], sum(M for M, _ in _mats(case))
        y, at = torch.zeros(batch * total, dtype=dtype, device=DEV), 0
        for M, K in _mats(case):
            R, sg = _cb_rows(case, M), case["scale_group"] or K
            idx = _words(M * K // 8, g).view(torch.uint8).view(M, K // 2)
            # codewords of abs-max-normalised weights: within +-1, the scale is
            # the largest weight of its group
            C = _normal((-(-M // R), 256, 2), g, 0.0, 0.35).clamp_(-1, 1).half()
            S = _normal((M, K // sg), g, 0.06, 0.01).abs_().half()
            calls.append((idx, C, S, x[K], y[at:at + batch * M].view(batch, M),
                          kq.VQParams(M, K, R, sg)))
            at += batch * M
        layers.append((calls, y))

    def go():
        for calls, _ in layers:
            for idx, C, S, x, y, P in calls:
                kq.vq_gemv(idx, C, S, x, y, P, batch=batch)

    return {"layers": layers, "go": go, "out": [y for _, y in layers]}


def _prepare_quantize(case, g):
    M, K = case["M"], case["K"]
    R, sg = _cb_rows(case, M), case["scale_group"] or K
    W = _normal((M, K), g, 0.0, 0.02, _FLOAT[case["dtype"]])
    idx = torch.zeros((M, K // 2), dtype=torch.uint8, device=DEV)
    C = torch.zeros((-(-M // R), 256, 2), dtype=torch.float16, device=DEV)
    S = torch.zeros((M, K // sg), dtype=torch.float16, device=DEV)
    n = kq.vq_quantize_workspace_size(M, K, R, sg, case["sample"])
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)

    def go():
        kq.vq_quantize(W, idx, C, S, M, K, R, sg, ws, n, iters=case["iters"],
                       sample=case["sample"], seed=5)

    return {"W": W, "go": go, "out": [idx, C, S]}


def _moe_desc(case):
    """The gpt-oss blob: gate, up, down, each W, scales, biases, output bias."""
    d = kq.moe_default_desc()
    h, i = case["hidden"], case["inter"]
    w, s, b = h * i // 2, h * i // 64 * 2, -(-max(h, i) * 2 // 16) * 16
    d.hidden, d.inter, d.n_experts, d.top_k = h, i, case["experts"], case["top_k"]
    d.sub_w, d.sub_s, d.sub_b, d.sub_bi = 0, w, w + s, w + 2 * s
    d.off_gate, d.off_up, d.off_down = 0, w + 2 * s + b, 2 * (w + 2 * s + b)
    d.blob = -(-3 * (w + 2 * s + b) // 4096) * 4096
    return d


def _proj(pool, d, off, rows, cols):
    """(W words, S, B, output bias) of one projection of every expert, as views of the pool."""
    def view(sub, n, dtype, *shape):
        return pool[:, off + sub:off + sub + n].view(dtype).view(pool.shape[0], *shape)
    n = rows * cols // 64 * 2
    return (view(d.sub_w, rows * cols // 2, torch.int32, rows, cols // 8),
            view(d.sub_s, n, torch.bfloat16, rows, cols // 64),
            view(d.sub_b, n, torch.bfloat16, rows, cols // 64),
            view(d.sub_bi, rows * 2, torch.bfloat16, rows))


def _projs(pool, d):
    return [_proj(pool, d, o, r, c) for o, r, c in ((d.off_gate, d.inter, d.hidden),
                                                    (d.off_up, d.inter, d.hidden),
                                                    (d.off_down, d.hidden, d.inter))]


def _prepare_moe(case, g):
    d, batch, E, k = _moe_desc(case), case["batch"], case["experts"], case["top_k"]
    n = kq.moe_workspace_size(d, batch)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    kq.moe_workspace_init(ws, n)
    layers = []
    for _ in range(case["layers"]):
        pool = _words(E * d.blob // 4, g).view(torch.uint8).view(E, d.blob)
        for _, S, B, bias in _projs(pool, d):
            s, b = _affine(S.shape, g, torch.bfloat16)
            S.copy_(s)
            B.copy_(b)
            bias.copy_(_normal(bias.shape, g, 0.0, 0.02))
        R = _normal((E, d.hidden), g, 0.0, 0.02, torch.float16)
        x = _x(batch, d.hidden, g, _FLOAT[case["x"]])
        xh = torch.zeros((batch, d.hidden), dtype=torch.float16, device=DEV) if case["x"] == "f32" else None
        out = {"idx": torch.zeros((batch, k), dtype=torch.int32, device=DEV),
               "wgt": torch.zeros((batch, k), dtype=torch.float32, device=DEV),
               "h": torch.zeros((batch, k, d.inter), dtype=torch.float16, device=DEV),
               "y": torch.zeros((batch, d.hidden), dtype=_FLOAT[case["out"]], device=DEV)}
        layers.append((pool, R, x, xh, out))

    def block():
        for pool, R, x, xh, o in layers:
            kq.moe_block(pool, d, R, x, o["idx"], o["wgt"], o["h"], o["y"], ws, n, batch=batch, xh=xh)

    def calls():
        for pool, R, x, xh, o in layers:
            kq.moe_router_topk(R, x, o["idx"], o["wgt"], d, ws, n, batch=batch, xh=xh)
            kq.moe_gate_up_swiglu(pool, d, o["idx"], x if xh is None else xh, o["h"], ws, n, batch=batch)
            kq.moe_down_combine(pool, d, o["idx"], o["wgt"], o["h"], o["y"], ws, n, batch=batch)

    return {"layers": layers, "ws": ws, "d": d, "go": block if case["form"] == "block" else calls,
            "out": [o for *_, o in layers]}


_PREPARE = {"int4": _prepare_int4, "vq": _prepare_vq, "quantize": _prepare_quantize,
            "moe": _prepare_moe}


def _inputs(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return _PREPARE[case["kind"]](case, g)


def prepare(case, seed):
    state = _inputs(case, seed)
    if case.get("graph"):
        state["go"]()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["go"]()
        state["graph"] = graph
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        state["go"]()
    return state["out"]


# ---------------------------------------------------------------------------

def _size(dtype):
    return 4 if dtype == "f32" else 2


def _distinct(case):
    """Experts that some token chose, on average over random routings."""
    E = case["experts"]
    return E * (1.0 - (1.0 - case["top_k"] / E) ** case["batch"])


def work(case):
    if case["kind"] == "quantize":
        M, K = case["M"], case["K"]
        R, sg = _cb_rows(case, M), case["scale_group"] or K
        blocks = -(-M // R)
        points = sum(min(case["sample"], min(R, M - b * R) * K // 2) for b in range(blocks))
        # W, the indices, scales and codebooks; per assigned pair one score and
        # (in an iteration) the two sums
        return {"bytes": M * K * _size(case["dtype"]) + M * K / 2 + M * (K // sg) * 2 + blocks * 1024,
                "flops": case["iters"] * points * 6.0 + M * K / 2 * 4.0}
    batch, L = case["batch"], case["layers"]
    if case["kind"] == "moe":
        h, i, k = case["hidden"], case["inter"], case["top_k"]
        expert = 3 * (h * i // 2 + h * i // 64 * 4) + 2 * (2 * i + h)
        act = batch * (h * _size(case["x"]) + k * (8 + 4 * i) + h * _size(case["out"]))
        return {"bytes": L * (_distinct(case) * expert + case["experts"] * h * 2 + act),
                "flops": L * batch * (k * 6.0 * h * i + 2.0 * case["experts"] * h)}
    got = {"bytes": 0, "flops": 0}
    for M, K in _mats(case):
        if case["kind"] == "int4":
            weights = M * K // 2 + M * (K // case["G"]) * 4
        else:
            weights = M * K // 2 + M * (K // (case["scale_group"] or K)) * 2 + -(-M // _cb_rows(case, M)) * 1024
        got["bytes"] += L * (weights + batch * (M * _size(case["out"]) + K * 2))
        got["flops"] += L * 2.0 * M * K * batch
    return got


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"  # bytes, and a function of the arguments
    if case["kind"] == "moe":
        # h is fp16 whatever y is: a rounding of h that falls the other way
        # moves y too
        return {"rel": 1e-3, "max": 1e-2, "differ": 0.0}
    if case["out"] == "f16":
        return {"rel": 1e-3, "max": 1e-2}  # one rounding to fp16
    # 32-bit sums; int4 subtracts the 1024 and 64 that its nibbles carry (two
    # paths of it differ by up to 1.6e-5, each is up to 1.4e-5 off 64 bits)
    return {"rel": 6e-5, "max": 3e-4} if case["kind"] == "int4" else {"rel": 1e-6, "max": 1e-5}


def _rows64(W, S, B, G, r0, r1):
    """Rows r0..r1 of an int4 matrix in 64 bits."""
    w = W[r0:r1]
    q = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], -1).view(r1 - r0, -1, G).double()
    return (q * S[r0:r1, :, None].double() + B[r0:r1, :, None].double()).view(r1 - r0, -1)


def _int4_64(W, S, B, G, x):
    M, K = W.shape[0], W.shape[1] * 8
    step = max(1, 2**26 // K)
    return torch.cat([x.double() @ _rows64(W, S, B, G, r, min(M, r + step)).t().contiguous()
                      for r in range(0, M, step)], 1)


def _vq_64(idx, C, S, P, x):
    out, step = [], max(1, 2**26 // P.K)
    for r in range(0, P.M, step):
        rows = torch.arange(r, min(P.M, r + step), device=DEV)
        w = C.double()[(rows // P.rows_per_cb)[:, None], idx[r:r + len(rows)].long()]
        w = w.reshape(len(rows), -1, P.scale_group) * S[r:r + len(rows), :, None].double()
        out.append(x.double() @ w.view(len(rows), P.K).t().contiguous())
    return torch.cat(out, 1)


def _moe_64(case, d, pool, R, x):
    batch, k = case["batch"], case["top_k"]
    top = torch.topk(x.double() @ R.double().t().contiguous(), k)
    idx, wgt = top.indices, torch.softmax(top.values, 1)
    xh = x.half()
    (gW, gS, gB, gb), (uW, uS, uB, ub), (dW, dS, dB, db) = _projs(pool, d)
    h = torch.zeros((batch, k, d.inter), dtype=torch.float64, device=DEV)
    y = torch.zeros((batch, d.hidden), dtype=torch.float64, device=DEV)
    for e in torch.unique(idx).tolist():
        t, s = (idx == e).nonzero(as_tuple=True)
        gate = _int4_64(gW[e], gS[e], gB[e], 64, xh[t]) + gb[e].double()
        up = _int4_64(uW[e], uS[e], uB[e], 64, xh[t]) + ub[e].double()
        gate = gate.clamp(max=7.0)
        he = gate * torch.sigmoid(1.702 * gate) * (up.clamp(-7.0, 7.0) + 1.0)
        h[t, s] = he
        y.index_add_(0, t, wgt[t, s][:, None] * (_int4_64(dW[e], dS[e], dB[e], 64, he) + db[e].double()))
    return {"idx": idx.int(), "wgt": wgt, "h": h, "y": y}


def exact(case, seed):
    state = _inputs(case, seed)
    if case["kind"] == "quantize":
        # the scales; k-means is a run of discrete choices with no 64-bit value
        W, sg = state["W"], case["scale_group"] or case["K"]
        step = max(1, 2**25 // case["K"])
        S = [W[r:r + step].double().abs().view(-1, case["K"] // sg, sg).amax(2)
             for r in range(0, case["M"], step)]
        return [None, None, torch.cat(S)]
    if case["kind"] == "moe":
        return [_moe_64(case, state["d"], pool, R, x) for pool, R, x, _, _ in state["layers"]]
    got = []
    for calls, _ in state["layers"]:
        if case["kind"] == "int4":
            ys = [_int4_64(W, *((S, B) if B is not None else (S[..., 0], S[..., 1])), P.G, x)
                  for W, S, B, x, _, P in calls]
        else:
            ys = [_vq_64(idx, C, S, P, x) for idx, C, S, x, _, P in calls]
        got.append(torch.cat([y.reshape(-1) for y in ys]))
    return got
