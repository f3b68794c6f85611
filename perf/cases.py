"""Performance cases: the calls a training or serving program makes through mi_gemm.

A case is a dict of plain values; `kind` says which path it takes:

* ``linear``     Y = X W (+ b), and with ``train`` also dX = dY W^T and dW = X^T dY;
* ``layer``      the forward of one decoder layer around its attention core (norm, QKV
                 projection, output projection + residual, norm, SiLU-gated up projections, down
                 projection + residual); ``graph``: captured once in a HIP graph and replayed,
                 as a decode loop does;
* ``block``      the 15 matrix products of a decoder block's training step (forward, dW, dX of
                 QKV, output, gate, up and down) in the engine's order; ``accumulate``: weight
                 gradients zeroed at the step's start and accumulated into, else overwritten;
* ``attention``  fused GQA attention, bf16: forward, and with ``train`` the backward;
* ``attention_f32``  attention as the fp32 engine runs it: batched products with the scores
                 held in memory, forward and backward;
* ``lm_head``    output projection, softmax cross-entropy and both gradients; ``chunk`` > 0: in
                 vocabulary chunks by one call, 0: as separate calls on a whole logits matrix;
* ``norm``       RMSNorm forward, and its backward with the residual gradient and dw.

Weights are stored [in, out] (the engine's layout) unless ``w_layout`` says otherwise.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "large-language-model_amd"))
import mi_gemm as mi  # noqa: E402

BF16, F32 = "bf16", "f32"
SMALL = {"D": 768, "QKV": 2304, "H": 2048}    # GPT-small block, 12 heads of 64
LARGE = {"D": 2048, "QKV": 3072, "H": 5632}   # 1.6B block, 16 query / 4 KV heads of 128


def listed():
    return [
        # the smallest call: one fp32 linear layer with bias on 512 tokens
        {"name": "linear_f32_m512", "kind": "linear", "M": 512, "K": 768, "N": 768, "dtype": F32,
         "bias": True, "train": False},
        # token generation for 8 sequences: one layer of the 1.6B model, replayed from a graph
        {"name": "layer_decode_m8", "kind": "layer", "M": 8, **LARGE, "dtype": BF16, "graph": True},
        # prompt processing / evaluation: the same layer on two sequences of 1024 tokens
        {"name": "layer_prefill_m2048", "kind": "layer", "M": 2048, **LARGE, "dtype": BF16,
         "graph": False},
        # fp32 training of the GPT-small block, 4 x 512 tokens
        {"name": "block_f32_m2048", "kind": "block", "M": 2048, **SMALL, "dtype": F32,
         "accumulate": False},
        # bf16 training of the 1.6B block, 8 x 1024 tokens (the benchmark's shape)
        {"name": "block_bf16_m8192", "kind": "block", "M": 8192, **LARGE, "dtype": BF16,
         "accumulate": True},
        # the same block on a last, short batch of 1000 tokens
        {"name": "block_bf16_m1000", "kind": "block", "M": 1000, **LARGE, "dtype": BF16,
         "accumulate": False},
        # bf16 attention of the 1.6B block in training
        {"name": "attention_gqa_t1024", "kind": "attention", "B": 8, "nH": 16, "nKV": 4, "T": 1024,
         "d": 128, "causal": True, "train": True},
        # bf16 attention with 12 heads of 64 on sequences that end at an odd length
        {"name": "attention_mha64_t509", "kind": "attention", "B": 4, "nH": 12, "nKV": 12, "T": 509,
         "d": 64, "causal": True, "train": True},
        # fp32 attention of the GPT-small block in training
        {"name": "attention_f32_t512", "kind": "attention_f32", "B": 4, "nH": 12, "nKV": 12,
         "T": 512, "d": 64},
        # the head and loss of the 1.6B model with the whole logits matrix (the largest case)
        {"name": "lm_head_m8192", "kind": "lm_head", "rows": 8192, "hidden": 2048, "vocab": 32000,
         "chunk": 0, "w_layout": 1, "dtype": BF16},
        # the memory-lean head on 2048 tokens, vocabulary with one added token
        {"name": "lm_head_chunked_v32001", "kind": "lm_head", "rows": 2048, "hidden": 2048,
         "vocab": 32001, "chunk": 8192, "w_layout": 1, "dtype": BF16},
        # the norm in front of a projection, forward and backward, bf16
        {"name": "norm_m8192_d2048", "kind": "norm", "rows": 8192, "dims": 2048, "dtype": BF16},
    ]


# ---- drawn cases -------------------------------------------------------------------------

def _log(rng, lo, hi, step=1):
    """An integer in [lo, hi], spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def _size(rng, lo, hi):
    """As _log: whole multiples of 64 or 8 (layer widths) more often than odd sizes."""
    return _log(rng, lo, hi, rng.choice((64, 64, 8, 1)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "layer", "layer", "block", "block", "attention",
                       "attention", "attention_f32", "lm_head", "lm_head", "norm"))
    if kind == "linear":
        return {"kind": kind, "M": _log(rng, 1, 8192), "K": _size(rng, 128, 4096),
                "N": _size(rng, 128, 4096), "dtype": rng.choice((BF16, F32)),
                "bias": rng.random() < 0.5, "train": rng.random() < 0.5}
    if kind in ("layer", "block"):
        dtype = rng.choice((BF16, BF16, F32))
        dims = dict(SMALL) if dtype == F32 else dict(rng.choice((SMALL, LARGE)))
        if rng.random() < 0.4:  # another width, in whole heads of 64
            D = _log(rng, 256, 1024 if dtype == F32 else 3072, 64)
            dims = {"D": D, "QKV": D + 128 * rng.randint(1, max(1, D // 128)), "H": _log(rng, D, 3 * D, 8)}
        if kind == "block":
            top = 2048 if dtype == F32 else min(8192, int(8192 * (2048 / dims["D"]) ** 2))
            return {"kind": kind, "M": _log(rng, 64, top), **dims, "dtype": dtype,
                    "accumulate": rng.random() < 0.5}
        graph = rng.random() < 0.5
        M = _log(rng, 1, 64) if graph else _log(rng, 64, 2048 if dtype == F32 else 8192)
        return {"kind": kind, "M": M, **dims, "dtype": dtype, "graph": graph}
    if kind == "attention":
        nH, nKV = rng.choice(((12, 12), (16, 4), (16, 16), (8, 1), (32, 8)))
        T = _log(rng, 32, 4096)
        most = max(1, min(16, (8 * 16 * 1024 * 1024) // (nH * T * T)))
        return {"kind": kind, "B": _log(rng, 1, most), "nH": nH, "nKV": nKV, "T": T,
                "d": rng.choice((64, 128, 128, 96)), "causal": rng.random() < 0.8,
                "train": rng.random() < 0.6}
    if kind == "attention_f32":
        nH, nKV = rng.choice(((12, 12), (16, 4), (8, 8)))
        T = _log(rng, 32, 1024)
        most = max(1, min(8, (16 * 1024 * 1024) // (nH * T * T)))
        return {"kind": kind, "B": _log(rng, 1, most), "nH": nH, "nKV": nKV, "T": T,
                "d": rng.choice((64, 128))}
    if kind == "lm_head":
        dtype = rng.choice((BF16, BF16, F32))
        return {"kind": kind, "rows": _log(rng, 16, 1024 if dtype == F32 else 4096),
                "hidden": _log(rng, 256, 1024 if dtype == F32 else 2048, 64),
                "vocab": _size(rng, 1000, 32000),
                "chunk": rng.choice((0, 4096, 8192)) if dtype == BF16 else 0,
                "w_layout": rng.randint(0, 1), "dtype": dtype}
    return {"kind": kind, "rows": _log(rng, 8, 16384), "dims": _size(rng, 256, 8192),
            "dtype": rng.choice((BF16, F32))}


# ---- inputs ------------------------------------------------------------------------------

class _Inputs:
    """Seeded normal tensors on the GPU."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dt = torch.bfloat16 if dtype == BF16 else torch.float32

    def n(self, *shape, std=1.0, mean=0.0, dtype=None):
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return t.mul_(std).add_(mean).to(dtype or self.dt)

    def empty(self, *shape, dtype=None):
        return torch.empty(shape, device="cuda", dtype=dtype or self.dt)

    def ids(self, n, top):
        return torch.randint(0, top, (n,), generator=self.g, device="cuda", dtype=torch.int32)


def _dt(dtype):
    return mi.MI_BF16 if dtype == BF16 else mi.MI_F32


def _workspace(dtype, *gemms):
    """One split-K workspace for all the given (transA, transB, M, N, K, C is fp32)."""
    need = max(mi.workspace_size(ta, tb, M, N, K, _dt(dtype), mi.MI_F32 if f32 else _dt(dtype))
               for ta, tb, M, N, K, f32 in gemms)
    return torch.empty((need + 3) // 4, dtype=torch.float32, device="cuda") if need else None


def _block_projections(c):
    return (("qkv", c["D"], c["QKV"]), ("o", c["D"], c["D"]), ("gate", c["D"], c["H"]),
            ("up", c["D"], c["H"]), ("down", c["H"], c["D"]))


def _tensors(c, seed):
    """The input tensors of a case (shared by prepare and exact)."""
    r = _Inputs(seed, c.get("dtype", F32 if c["kind"] == "attention_f32" else BF16))
    k, t = c["kind"], {}
    if k == "linear":
        t["X"], t["W"] = r.n(c["M"], c["K"]), r.n(c["K"], c["N"], std=0.02)
        t["b"] = r.n(c["N"], std=0.02) if c["bias"] else None
        t["dY"] = r.n(c["M"], c["N"], std=1e-2) if c["train"] else None
    elif k == "layer":
        M, D, H = c["M"], c["D"], c["H"]
        t["x"], t["attn"] = r.n(M, D), r.n(M, D, std=0.5)
        t["n1"], t["n2"] = r.n(D, std=0.1, mean=1.0), r.n(D, std=0.1, mean=1.0)
        t["Wqkv"], t["Wo"] = r.n(D, c["QKV"], std=0.02), r.n(D, D, std=0.02)
        t["Wg"], t["Wu"], t["Wd"] = r.n(D, H, std=0.02), r.n(D, H, std=0.02), r.n(H, D, std=0.02)
    elif k == "block":
        for n, i, o in _block_projections(c):
            t["W_" + n] = r.n(i, o, std=0.02)
            t["dY_" + n] = r.n(c["M"], o, std=1e-2)
            if n != "up":
                t["X_" + n] = r.n(c["M"], i)
        t["X_up"] = t["X_gate"]  # gate and up read the same activations
    elif k in ("attention", "attention_f32"):
        B, T, d = c["B"], c["T"], c["d"]
        t["Q"] = r.n(B, c["nH"], T, d)
        t["K"], t["V"] = r.n(B, c["nKV"], T, d), r.n(B, c["nKV"], T, d)
        if k == "attention_f32" or c["train"]:
            t["dO"] = r.n(B, T, c["nH"] * d, std=1e-2)
    elif k == "lm_head":
        t["X"] = r.n(c["rows"], c["hidden"])
        shape = (c["hidden"], c["vocab"]) if c["w_layout"] == 0 else (c["vocab"], c["hidden"])
        t["W"] = r.n(*shape, std=0.02)
        t["y"] = r.ids(c["rows"], c["vocab"])
    else:
        t["x"], t["dy"] = r.n(c["rows"], c["dims"]), r.n(c["rows"], c["dims"], std=1e-2)
        t["res"], t["w"] = r.n(c["rows"], c["dims"], std=1e-2), r.n(c["dims"], std=0.1, mean=1.0)
    return r, t


def prepare(case, seed):
    c = dict(case)
    r, t = _tensors(c, seed)
    s = {"c": c, **t}
    k = c["kind"]
    if k == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        s["Y"] = r.empty(M, N)
        gemms = [(0, 0, M, N, K, False)]
        if c["train"]:
            s["dX"], s["dW"] = r.empty(M, K), r.empty(K, N, dtype=torch.float32)
            gemms += [(0, 1, M, K, N, False), (1, 0, K, N, M, True)]
        s["ws"] = _workspace(c["dtype"], *gemms)
    elif k == "layer":
        M, D, Q, H = c["M"], c["D"], c["QKV"], c["H"]
        s["y"], s["h"], s["z"], s["out"] = (r.empty(M, D) for _ in range(4))
        s["qkv"], s["act"] = r.empty(M, Q), r.empty(M, H)
        s["ws"] = _workspace(c["dtype"], (0, 0, M, Q, D, False), (0, 0, M, D, D, False), (0, 0, M, D, H, False))
        if c["graph"]:
            _layer(s)  # the library's kernels are loaded before the capture
            torch.cuda.synchronize()
            s["replay"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["replay"]):
                _layer(s)
    elif k == "block":
        gemms = []
        for n, i, o in _block_projections(c):
            s["Y_" + n], s["dX_" + n] = r.empty(c["M"], o), r.empty(c["M"], i)
            s["dW_" + n] = r.empty(i, o, dtype=torch.float32)
            gemms += [(0, 0, c["M"], o, i, False), (0, 1, c["M"], i, o, False), (1, 0, i, o, c["M"], True)]
        s["ws"] = _workspace(c["dtype"], *gemms)
    elif k == "attention":
        B, nH, T = c["B"], c["nH"], c["T"]
        s["O"], s["lse"] = r.empty(B, T, nH * c["d"]), r.empty(B, nH, T, dtype=torch.float32)
        if c["train"]:
            n = int(mi.load_library().mi_flash_attn_bwd_workspace_size(B, nH, T))
            s["ws"] = r.empty(n // 2) if n else None
    elif k == "lm_head":
        M, H, V = c["rows"], c["hidden"], c["vocab"]
        s["dX"], s["dW"] = r.empty(M, H), r.empty(*s["W"].shape, dtype=torch.float32)
        s["row_loss"], s["loss"] = r.empty(M, dtype=torch.float32), r.empty(1, dtype=torch.float32)
        if c["chunk"]:
            s["ws"] = r.empty(mi.lm_head_xent_workspace_size(M, H, V, c["chunk"]), dtype=torch.uint8)
        else:
            s["logits"] = r.empty(M, V)
            l1 = c["w_layout"]
            s["ws"] = _workspace(c["dtype"], (0, l1, M, V, H, False), (0, 1 - l1, M, H, V, False),
                                 (1, 0, V, H, M, True) if l1 else (1, 0, H, V, M, True))
    elif k == "norm":
        s["out"], s["dx"] = r.empty(c["rows"], c["dims"]), r.empty(c["rows"], c["dims"])
        s["rstd"], s["dw"] = r.empty(c["rows"], dtype=torch.float32), r.empty(c["dims"], dtype=torch.float32)
    return s


# ---- one pass ----------------------------------------------------------------------------

def _layer(s):
    c, ws = s["c"], s["ws"]
    M, D, Q, H = c["M"], c["D"], c["QKV"], c["H"]
    mi.rms_norm_forward(s["x"], s["n1"], out=s["y"], sync=False)
    mi.gemm(s["y"], s["Wqkv"], s["qkv"], M, Q, D, workspace=ws, sync=False)
    mi.gemm(s["attn"], s["Wo"], s["h"], M, D, D, residual=s["x"], workspace=ws, sync=False)
    mi.rms_norm_forward(s["h"], s["n2"], out=s["z"], sync=False)
    mi.gemm(s["z"], s["Wg"], s["act"], M, H, D, B2=s["Wu"], workspace=ws, sync=False)
    mi.gemm(s["act"], s["Wd"], s["out"], M, D, H, residual=s["h"], workspace=ws, sync=False)


def run(s):
    c = s["c"]
    k = c["kind"]
    if k == "linear":
        M, K, N, ws = c["M"], c["K"], c["N"], s["ws"]
        mi.gemm(s["X"], s["W"], s["Y"], M, N, K, bias=s["b"], workspace=ws, sync=False)
        if not c["train"]:
            return {"Y": s["Y"]}
        mi.gemm(s["X"], s["dY"], s["dW"], K, N, M, transA=True, workspace=ws, sync=False)
        mi.gemm(s["dY"], s["W"], s["dX"], M, K, N, transB=True, workspace=ws, sync=False)
        return {"Y": s["Y"], "dX": s["dX"], "dW": s["dW"]}
    if k == "layer":
        if c["graph"]:
            s["replay"].replay()
        else:
            _layer(s)
        return {n: s[n] for n in ("qkv", "h", "act", "out")}
    if k == "block":
        M, ws = c["M"], s["ws"]
        names = _block_projections(c)
        beta = 1.0 if c["accumulate"] else 0.0
        if c["accumulate"]:
            for n, _, _ in names:
                s["dW_" + n].zero_()
        for n, i, o in names:
            mi.gemm(s["X_" + n], s["W_" + n], s["Y_" + n], M, o, i, workspace=ws, sync=False)

        def dw(n, i, o):
            mi.gemm(s["X_" + n], s["dY_" + n], s["dW_" + n], i, o, M, transA=True, beta=beta,
                    workspace=ws, sync=False)

        def dx(n, i, o):
            mi.gemm(s["dY_" + n], s["W_" + n], s["dX_" + n], M, i, o, transB=True, workspace=ws,
                    sync=False)

        qkv, o, gate, up, down = names
        dw(*down), dx(*down), dw(*gate), dw(*up), dx(*gate), dx(*up)
        dw(*o), dx(*o), dw(*qkv), dx(*qkv)
        return {p + n: s[p + n] for n, _, _ in names for p in ("Y_", "dX_", "dW_")}
    if k == "attention":
        O = mi.flash_attn_fwd(s["Q"], s["K"], s["V"], O=s["O"], lse=s["lse"], causal=c["causal"],
                              sync=False)
        if not c["train"]:
            return {"O": O}
        dQ, dK, dV = mi.flash_attn_bwd(s["Q"], s["K"], s["V"], O, s["dO"], s["lse"],
                                       causal=c["causal"], sync=False, workspace=s["ws"])
        return {"O": O, "lse": s["lse"], "dQ": dQ, "dK": dK, "dV": dV}
    if k == "attention_f32":
        mi.begin_scope()  # one wait at the end of the step, as the engine's scopes do
        O, P = mi.attention_forward(s["Q"], s["K"], s["V"])
        dQ, dK, dV = mi.attention_backward(s["Q"], s["K"], s["V"], s["dO"], P)
        mi.end_scope()
        return {"O": O, "dQ": dQ, "dK": dK, "dV": dV}
    if k == "lm_head":
        M, H, V, l1, ws = c["rows"], c["hidden"], c["vocab"], c["w_layout"], s["ws"]
        X, W, dX, dW = s["X"], s["W"], s["dX"], s["dW"]
        if c["chunk"]:
            mi.lm_head_xent(X, W, s["y"], w_layout=l1, chunk=c["chunk"], dX=dX, dW=dW,
                            row_loss=s["row_loss"], loss=s["loss"], workspace=ws, sync=False)
            return {"loss": s["loss"], "row_loss": s["row_loss"], "dX": dX, "dW": dW}
        L = s["logits"]
        mi.gemm(X, W, L, M, V, H, transB=bool(l1), workspace=ws, sync=False)
        mi.cross_entropy(L, s["y"], grad="inplace", row_loss=s["row_loss"], loss=s["loss"], sync=False)
        mi.gemm(L, W, dX, M, H, V, transB=not l1, workspace=ws, sync=False)
        if l1:
            mi.gemm(L, X, dW, V, H, M, transA=True, workspace=ws, sync=False)
        else:
            mi.gemm(X, L, dW, H, V, M, transA=True, workspace=ws, sync=False)
        return {"loss": s["loss"], "row_loss": s["row_loss"], "dlogits": L, "dX": dX, "dW": dW}
    mi.rms_norm_forward(s["x"], s["w"], out=s["out"], rstd=s["rstd"], sync=False)
    mi.rms_norm_backward(s["dy"], s["x"], s["w"], residual_grad=s["res"], dx=s["dx"], dw=s["dw"],
                         sync=False)
    return {"y": s["out"], "rstd": s["rstd"], "dx": s["dx"], "dw": s["dw"]}


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    c = case
    e = 2 if c.get("dtype", F32 if c["kind"] == "attention_f32" else BF16) == BF16 else 4
    k = c["kind"]
    if k == "linear":
        M, K, N = c["M"], c["K"], c["N"]
        b, f = e * (M * K + K * N + M * N + (N if c["bias"] else 0)), 2 * M * N * K
        if c["train"]:
            b, f = b + e * (M * N + M * K) + 4 * K * N, 3 * f
    elif k == "layer":
        M, D, Q, H = c["M"], c["D"], c["QKV"], c["H"]
        b = e * (D * Q + D * D + 3 * D * H + 2 * D + M * (4 * D + Q + H))
        f = 2 * M * (D * Q + D * D + 3 * D * H)
    elif k == "block":
        M, w = c["M"], sum(i * o for _, i, o in _block_projections(c))
        acts = M * (sum(i + 2 * o + i for _, i, o in _block_projections(c)) - c["D"])
        b, f = e * (acts + w) + 4 * w, 6 * M * w
    elif k in ("attention", "attention_f32"):
        B, T, nH, nKV, d = c["B"], c["T"], c["nH"], c["nKV"], c["d"]
        causal = c.get("causal", True)
        train = c.get("train", True)
        f = 2 * B * nH * d * (T * (T + 1) // 2 if causal else T * T) * (6 if train else 2)
        b = e * B * T * d * (2 * nH + 2 * nKV + (2 * nH + 2 * nKV if train else 0))
        if train and k == "attention":
            b += 4 * B * nH * T
    elif k == "lm_head":
        M, H, V = c["rows"], c["hidden"], c["vocab"]
        b, f = e * (2 * M * H + H * V) + 4 * (H * V + 2 * M), 6 * M * H * V
        if not c["chunk"]:
            b += e * M * V  # the logits' gradient is an output
    else:
        R, D = c["rows"], c["dims"]
        b, f = e * (5 * R * D + D) + 4 * (R + D), 14 * R * D
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the largest error against 64 bits that the listed and 40 drawn cases showed:
    fp32 8.1e-7 (largest single value 8.3e-6); bf16 one rounding of the outputs, 1.7e-3 (3.9e-3), or
    the roundings that a layer (3.8e-3, 5.9e-2), the attention's P and dS (2.6e-3, 0.11) and the
    head's logits (3.3e-3, 2.3e-2) add up."""
    k = case["kind"]
    if k == "attention":
        return {"rel": 0.01, "max": 0.45}
    if k == "attention_f32" or case["dtype"] == F32:
        return {"rel": 3.5e-6, "max": 3.5e-5}
    return {"layer": {"rel": 0.015, "max": 0.24},
            "lm_head": {"rel": 0.013, "max": 0.1}}.get(k, {"rel": 0.007, "max": 0.016})


# ---- the same in 64 bits ---------------------------------------------------------------------

def _attention_exact(Q, K, V, dO, causal):
    B, nH, T, d = Q.shape
    g = nH // K.shape[1]
    Kx, Vx = K.repeat_interleave(g, 1), V.repeat_interleave(g, 1)
    S = torch.matmul(Q, Kx.transpose(2, 3).contiguous()) / math.sqrt(d)
    if causal:
        S.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=S.device).triu_(1), -math.inf)
    lse = torch.logsumexp(S, -1)
    P = S.sub_(lse.unsqueeze(-1)).exp_()
    O = torch.matmul(P, Vx)
    bthd = lambda x: x.permute(0, 2, 1, 3).reshape(B, T, nH * d)  # noqa: E731
    if dO is None:
        return bthd(O), lse, None, None, None
    G = dO.reshape(B, T, nH, d).permute(0, 2, 1, 3).contiguous()
    fold = lambda x: x.reshape(B, nH // g, g, T, d).sum(2)  # noqa: E731
    dV = fold(torch.matmul(P.transpose(2, 3).contiguous(), G))
    dS = torch.matmul(G, Vx.transpose(2, 3).contiguous())
    dS.sub_((G * O).sum(-1, keepdim=True)).mul_(P).div_(math.sqrt(d))
    dQ = torch.matmul(dS, Kx)
    dK = fold(torch.matmul(dS.transpose(2, 3).contiguous(), Q))
    return bthd(O), lse, dQ, dK, dV


def exact(case, seed):
    c = case
    _, t = _tensors(c, seed)
    t = {n: (x.double() if x is not None and x.is_floating_point() else x) for n, x in t.items()}
    k = c["kind"]
    if k == "linear":
        Y = t["X"] @ t["W"] + (t["b"] if c["bias"] else 0)
        return {"Y": Y, "dX": t["dY"] @ t["W"].T, "dW": t["X"].T @ t["dY"]} if c["train"] else {"Y": Y}

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w

    if k == "layer":
        qkv = norm(t["x"], t["n1"]) @ t["Wqkv"]
        h = t["attn"] @ t["Wo"] + t["x"]
        z = norm(h, t["n2"])
        act = torch.nn.functional.silu(z @ t["Wg"]) * (z @ t["Wu"])
        return {"qkv": qkv, "h": h, "act": act, "out": act @ t["Wd"] + h}
    if k == "block":
        out = {}
        for n, _, _ in _block_projections(c):
            X, W, dY = t["X_" + n], t["W_" + n], t["dY_" + n]
            out.update({"Y_" + n: X @ W, "dX_" + n: dY @ W.T, "dW_" + n: X.T @ dY})
        return out
    if k in ("attention", "attention_f32"):
        O, lse, dQ, dK, dV = _attention_exact(t["Q"], t["K"], t["V"], t.get("dO"), c.get("causal", True))
        if k == "attention_f32":
            return {"O": O, "dQ": dQ, "dK": dK, "dV": dV}
        return {"O": O, "lse": lse, "dQ": dQ, "dK": dK, "dV": dV} if c["train"] else {"O": O}
    if k == "lm_head":
        X, W, y = t["X"], t["W"], t["y"].long()
        W = W if c["w_layout"] == 0 else W.T
        L = X @ W
        row = torch.logsumexp(L, -1) - L.gather(1, y[:, None])[:, 0]
        G = torch.softmax(L, -1)
        G[torch.arange(len(y), device=G.device), y] -= 1
        G /= len(y)
        dW = X.T @ G
        out = {"loss": row.mean().reshape(1), "row_loss": row, "dX": G @ W.T,
               "dW": dW if c["w_layout"] == 0 else dW.T.contiguous()}
        return out if c["chunk"] else {"dlogits": G, **out}
    x, dy, w = t["x"], t["dy"], t["w"]
    rstd = 1 / torch.sqrt((x * x).mean(-1) + 1e-5)
    xh = x * rstd[:, None]
    dx = (dy * w - xh * (dy * w * xh).mean(-1, keepdim=True)) * rstd[:, None] + t["res"]
    return {"y": xh * w, "rstd": rstd, "dx": dx, "dw": (dy * xh).sum(0)}
