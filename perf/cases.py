"""Performance cases of the MI355X backend: the work its users have it do, timed
one call (or one forward + backward) at a time.

Most cases go through the C ABI (include/aar_hip.h, libaar_hip.so), the entry
points a C++ core binds, on tensors that torch holds on the GPU; the last kind
runs a whole model through the aargrad Python package.  Every case draws fp32
inputs of the scale the path meets in training: activations and gradients of
unit scale, weights of 1/sqrt(fan-in).
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "aar-vlm_amd"
if str(PKG) not in sys.path:
    sys.path.insert(0, str(PKG))

import aargrad as ag  # noqa: E402
from aargrad import nn  # noqa: E402

NN, NT, TN = 0, 1, 2
OPS = {"nn": NN, "nt": NT, "tn": TN}
UNSUPPORTED = -3  # AAR_EUNSUPPORTED: the caller runs the separate passes
DEV = "cuda"


# ------------------------------------------------------------------ C ABI

def _load():
    lib = ctypes.CDLL(str(PKG / "aargrad" / "libaar_hip.so"))
    vp, i64, sz, i32, f32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_size_t, ctypes.c_int, ctypes.c_float
    sig = {
        "aar_gemm_f32": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_workspace_bytes": (sz, [i32, i64, i64, i64]),
        "aar_gemm_f32_bias": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_bias_relu": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_bias_relu_bits": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_bias_add": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_mask_bits_colsum": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_colsum_a": (i32, [i32, i64, i64, i64, vp, vp, vp, vp, vp, sz, vp]),
        "aar_gemm_f32_colsum_a_workspace_bytes": (sz, [i32, i64, i64, i64]),
        "aar_colsum_f32": (i32, [vp, vp, i64, i64, vp, sz, vp]),
        "aar_colsum_workspace_bytes": (sz, [i64, i64]),
        "aar_relu_bwd_f32": (i32, [vp, vp, vp, i64, vp]),
        "aar_softmax_fwd_f32": (i32, [vp, vp, i64, i64, vp]),
        "aar_softmax_bwd_f32": (i32, [vp, vp, vp, i64, i64, vp]),
        "aar_layernorm_fwd_f32": (i32, [vp, vp, vp, vp, vp, vp, i64, i64, f32, vp]),
        "aar_layernorm_bwd_f32": (i32, [vp] * 8 + [i64, i64, vp, sz, vp]),
        "aar_layernorm_bwd_workspace_bytes": (sz, [i64, i64]),
        "aar_cross_entropy_fwd_f32": (i32, [vp, vp, vp, i64, i64, i64, vp, vp, sz, vp]),
        "aar_cross_entropy_bwd_f32": (i32, [vp, vp, vp, vp, i64, i64, i64, vp, sz, vp]),
        "aar_cross_entropy_workspace_bytes": (sz, [i64]),
        "aar_flash_fwd_strided_f32": (i32, [vp] * 5 + [i64] * 4 + [vp, i32, f32, vp, sz, vp]),
        "aar_flash_fwd_workspace_bytes": (sz, [i64, i64, i64, i32]),
        "aar_flash_bwd_strided_f32": (i32, [vp] * 9 + [i64] * 4 + [vp, i32, f32, vp, sz, vp]),
        "aar_flash_bwd_fast_workspace_bytes": (sz, [i64, i64, i64, i32]),
    }
    for name, (res, args) in sig.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = res, args
    return lib


_L = _load()


def _ok(rc):
    if rc != 0:
        raise RuntimeError("aar status %d" % rc)


def _p(t):
    return t.data_ptr()


def _new(*shape):
    return torch.empty(shape, dtype=torch.float32, device=DEV)


def _scratch(nbytes):
    """Workspace a program keeps beside its plan (256 bytes when none is needed)."""
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=DEV)


def _rand(gen, *shape, scale=1.0):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).mul_(scale)


def _generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    return gen


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # a single small product: launch latency and how few workgroups there are
        {"name": "matmul_256", "kind": "matmul", "op": "nn", "M": 256, "N": 256, "K": 256},
        # a mid-size square product, about one workgroup per CU
        {"name": "matmul_1024", "kind": "matmul", "op": "nt", "M": 1024, "N": 1024, "K": 1024},
        # the headline product
        {"name": "matmul_4096", "kind": "matmul", "op": "nn", "M": 4096, "N": 4096, "K": 4096},
        # the GPT's qkv projection with a bias at batch 64 x 256 tokens, forward and backward
        {"name": "linear_qkv", "kind": "linear", "rows": 16384, "inp": 384, "out": 1152},
        # a linear layer with extents that are no multiple of 4 (unaligned rows)
        {"name": "linear_odd", "kind": "linear", "rows": 5001, "inp": 771, "out": 1025},
        # the GPT's MLP (linear, relu, linear, residual) at the same batch, forward and backward
        {"name": "mlp_gpt", "kind": "mlp", "rows": 16384, "d": 384, "hidden": 1536},
        # the vocabulary head with its cross entropy, forward and backward
        {"name": "head_loss", "kind": "head", "rows": 16384, "d": 384, "vocab": 65},
        # the GPT's attention over the packed projection, forward and backward
        {"name": "attention_t256", "kind": "attention", "B": 64, "H": 6, "T": 256, "d": 64, "causal": True},
        # long-context attention, forward and backward (the largest case)
        {"name": "attention_t4096", "kind": "attention", "B": 8, "H": 12, "T": 4096, "d": 64, "causal": True},
        # ragged, non-causal attention of a small head count and another head size
        {"name": "attention_ragged", "kind": "attention", "B": 4, "H": 5, "T": 777, "d": 40, "causal": False},
        # layer normalisation over the GPT's width, forward and backward, larger than the caches
        {"name": "layernorm_384", "kind": "layernorm", "rows": 65536, "cols": 384},
        # a whole model's logits, batch 4 x 256 tokens, through aargrad, read back by the caller
        {"name": "gpt_logits", "kind": "gpt", "layers": 6, "d": 384, "heads": 6, "T": 256, "B": 4, "vocab": 65},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """A size spread over the logarithm: half the time a multiple of 64, else
    a multiple of 4, else any."""
    n = _log_int(rng, lo, hi)
    form = rng.random()
    step = 64 if form < 0.5 else 4 if form < 0.75 else 1
    return max(min(step, hi), n // step * step)


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "linear", "linear", "mlp", "head", "attention", "attention", "layernorm",
                       "softmax", "gpt"])
    most = 2.0 * 4096 ** 3
    while True:
        if kind == "matmul":
            c = {"kind": kind, "op": rng.choice(list(OPS)), "M": _extent(rng, 64, 16384), "N": _extent(rng, 64, 16384),
                 "K": _extent(rng, 64, 16384)}
        elif kind == "linear":
            c = {"kind": kind, "rows": _extent(rng, 64, 32768), "inp": _extent(rng, 64, 4096),
                 "out": _extent(rng, 64, 4096)}
        elif kind == "mlp":
            d = _extent(rng, 64, 1024)
            c = {"kind": kind, "rows": _extent(rng, 64, 32768), "d": d, "hidden": 4 * d}
        elif kind == "head":
            c = {"kind": kind, "rows": _extent(rng, 256, 32768), "d": _extent(rng, 64, 1024),
                 "vocab": _log_int(rng, 40, 2048)}
        elif kind == "attention":
            c = {"kind": kind, "B": _log_int(rng, 1, 64), "H": rng.randint(1, 12), "T": _extent(rng, 32, 4096),
                 "d": rng.choice([32, 64, 64, 64, 128, 40, 96, 30]), "causal": rng.random() < 0.7}
        elif kind in ("layernorm", "softmax"):
            c = {"kind": kind, "rows": _extent(rng, 64, 131072), "cols": _extent(rng, 64, 8192)}
        else:
            heads = rng.choice([2, 4, 6, 8])
            c = {"kind": kind, "layers": rng.randint(1, 6), "d": heads * rng.choice([32, 64]), "heads": heads,
                 "T": _extent(rng, 32, 256), "B": rng.randint(1, 8), "vocab": rng.randint(40, 128)}
        w = work(c)
        if w["flops"] <= most and w["bytes"] <= 1.0e9:
            return c


# ------------------------------------------------------------------ inputs

def _inputs(case, seed):
    g = _generator(seed)
    k = case["kind"]
    if k == "matmul":
        M, N, K, op = case["M"], case["N"], case["K"], OPS[case["op"]]
        a = _rand(g, *((K, M) if op == TN else (M, K)), scale=K ** -0.5)
        b = _rand(g, *((N, K) if op == NT else (K, N)))
        return {"a": a, "b": b}
    if k == "linear":
        rows, inp, out = case["rows"], case["inp"], case["out"]
        return {"x": _rand(g, rows, inp), "w": _rand(g, out, inp, scale=inp ** -0.5), "b": _rand(g, out, scale=0.1),
                "gy": _rand(g, rows, out, scale=1e-2)}
    if k == "mlp":
        rows, d, h = case["rows"], case["d"], case["hidden"]
        s = {"x": _rand(g, rows, d), "r": _rand(g, rows, d), "w1": _rand(g, h, d, scale=d ** -0.5),
             "b1": _rand(g, h, scale=0.1), "w2": _rand(g, d, h, scale=h ** -0.5), "b2": _rand(g, d, scale=0.1),
             "gy": _rand(g, rows, d, scale=1e-2)}
        # the hidden activations an earlier forward saved for the backward
        # pass: their signs decide which gradients pass, so they are inputs
        # here, rounded from 64 bits
        s["saved_h"] = torch.relu(s["x"].double() @ s["w1"].double().t() + s["b1"].double()).float()
        return s
    if k == "head":
        rows, d, v = case["rows"], case["d"], case["vocab"]
        return {"x": _rand(g, rows, d), "w": _rand(g, v, d, scale=d ** -0.5),
                "t": torch.randint(0, v, (rows,), generator=g, device=DEV, dtype=torch.int64),
                "one": torch.ones(1, device=DEV)}
    if k == "attention":
        B, H, T, d = case["B"], case["H"], case["T"], case["d"]
        return {"qkv": _rand(g, B, T, 3, H, d), "do": _rand(g, B, T, H, d)}
    if k == "layernorm":
        rows, cols = case["rows"], case["cols"]
        return {"x": _rand(g, rows, cols).add_(0.3), "w": 1.0 + _rand(g, cols, scale=0.1), "b": _rand(g, cols, scale=0.1),
                "gy": _rand(g, rows, cols)}
    if k == "softmax":
        rows, cols = case["rows"], case["cols"]
        return {"x": _rand(g, rows, cols, scale=3.0), "gy": _rand(g, rows, cols)}
    raise ValueError(k)


def _mask_bits(h):
    """relu's mask as the ABI packs it: word [r / 32][c] holds rows r % 32."""
    rows, cols = h.shape
    blocks = (rows + 31) // 32
    m = torch.zeros(blocks * 32, cols, dtype=torch.int64, device=h.device)
    m[:rows] = (h > 0).long()
    shift = torch.arange(32, device=h.device, dtype=torch.int64).view(1, 32, 1)
    words = (m.view(blocks, 32, cols) << shift).sum(1)
    return torch.where(words >= 2 ** 31, words - 2 ** 32, words).to(torch.int32).contiguous()


class _Block(nn.Module):
    """Pre-norm transformer block with a ReLU MLP."""

    def __init__(self, d, heads, rng):
        super().__init__()
        self.ln1 = nn.LayerNorm(d)
        self.attn = nn.MultiHeadAttention(d, heads, causal=True, bias=False, rng=rng)
        self.ln2 = nn.LayerNorm(d)
        self.mlp = nn.Sequential(nn.Linear(d, 4 * d, bias=True, rng=rng), nn.ReLU(),
                                 nn.Linear(4 * d, d, bias=True, rng=rng))

    def forward(self, x):
        x = ag.add(x, self.attn(self.ln1(x)))
        return ag.add(x, self.mlp(self.ln2(x)))


class _Gpt(nn.Module):
    """Decoder-only character GPT: token + position embeddings, blocks, final norm, head."""

    def __init__(self, c, rng):
        super().__init__()
        self.tok = nn.Embedding(c["vocab"], c["d"], rng=rng)
        self.pos = nn.Embedding(c["T"], c["d"], rng=rng)
        self.blocks = nn.Sequential(*[_Block(c["d"], c["heads"], rng) for _ in range(c["layers"])])
        self.norm = nn.LayerNorm(c["d"])
        self.head = nn.Linear(c["d"], c["vocab"], rng=rng)

    def forward(self, ids, pos):
        x = ag.add(self.tok(ids), self.pos(pos))
        return self.head(self.norm(self.blocks(x)))


def _gpt_arrays(case, seed):
    rng = np.random.default_rng(seed)
    model = _Gpt(case, rng)
    ids = rng.integers(0, case["vocab"], size=(case["B"], case["T"]), dtype=np.int64)
    pos = np.tile(np.arange(case["T"], dtype=np.int64), (case["B"], 1))
    return model, ids, pos


def _attention_strides(B, H, T, d):
    """Element strides (sb, sh, st) of q, k, v in the packed projection and of o in [B, T, H, d]."""
    packed, merged = [T * 3 * H * d, d, 3 * H * d], [T * H * d, d, H * d]
    return packed, merged


def prepare(case, seed):
    """Inputs on the GPU, outputs and workspaces a program allocates once."""
    k = case["kind"]
    if k == "gpt":
        model, ids, pos = _gpt_arrays(case, seed)
        model.to(ag.Device.CUDA)
        model.eval()
        return {"case": case, "model": model, "ids": ag.from_numpy(ids).to(ag.Device.CUDA),
                "pos": ag.from_numpy(pos).to(ag.Device.CUDA)}
    s = _inputs(case, seed)
    s["case"] = case
    if k == "matmul":
        M, N, K, op = case["M"], case["N"], case["K"], OPS[case["op"]]
        s["c"] = _new(M, N)
        s["ws"] = _scratch(_L.aar_gemm_f32_workspace_bytes(op, M, N, K))
    elif k == "linear":
        rows, inp, out = case["rows"], case["inp"], case["out"]
        s.update(y=_new(rows, out), dx=_new(rows, inp), dw=_new(out, inp), db=_new(out))
        s["ws"] = _scratch(_linear_workspace(rows, inp, out))
    elif k == "mlp":
        rows, d, h = case["rows"], case["d"], case["hidden"]
        s["bits"] = _mask_bits(s["saved_h"])
        s.update(h=_new(rows, h), h_bits=torch.empty_like(s["bits"]), y=_new(rows, d), dh=_new(rows, h),
                 dx=_new(rows, d), dw1=_new(h, d), db1=_new(h), dw2=_new(d, h), db2=_new(d))
        s["ws"] = _scratch(max(_linear_workspace(rows, d, h), _linear_workspace(rows, h, d)))
    elif k == "head":
        rows, d, v = case["rows"], case["d"], case["vocab"]
        s.update(logits=_new(rows, v), loss=_new(1), dlogits=_new(rows, v), dx=_new(rows, d), dw=_new(v, d))
        s["ws"] = _scratch(max(_linear_workspace(rows, d, v), _L.aar_cross_entropy_workspace_bytes(rows)))
    elif k == "attention":
        B, H, T, d = case["B"], case["H"], case["T"], case["d"]
        s.update(o=_new(B, T, H, d), lse=_new(B, H, T), dqkv=_new(B, T, 3, H, d))
        packed, merged = _attention_strides(B, H, T, d)
        s["fwd_strides"] = (ctypes.c_int64 * 12)(*(packed * 3 + merged))
        s["bwd_strides"] = (ctypes.c_int64 * 24)(*(packed * 3 + merged * 2 + packed * 3))
        c = int(case["causal"])
        s["fwd_bytes"] = _L.aar_flash_fwd_workspace_bytes(B * H, T, d, c)
        s["bwd_bytes"] = _L.aar_flash_bwd_fast_workspace_bytes(B * H, T, d, c)
        s["ws"] = _scratch(max(s["fwd_bytes"], s["bwd_bytes"]))
    elif k == "layernorm":
        rows, cols = case["rows"], case["cols"]
        s.update(y=_new(rows, cols), mean=_new(rows), rstd=_new(rows), dx=_new(rows, cols), dw=_new(cols),
                 db=_new(cols))
        s["ws"] = _scratch(_L.aar_layernorm_bwd_workspace_bytes(rows, cols))
    else:
        rows, cols = case["rows"], case["cols"]
        s.update(y=_new(rows, cols), dx=_new(rows, cols))
    return s


def _linear_workspace(rows, inp, out):
    return max(_L.aar_gemm_f32_workspace_bytes(NT, rows, out, inp), _L.aar_gemm_f32_workspace_bytes(NN, rows, inp, out),
               _L.aar_gemm_f32_workspace_bytes(TN, out, inp, rows),
               _L.aar_gemm_f32_colsum_a_workspace_bytes(TN, out, inp, rows), _L.aar_colsum_workspace_bytes(rows, out))


# ------------------------------------------------------------------ one pass

def _weight_grads(gy, x, dw, db, rows, inp, out, ws):
    """dW = gy^T x and db = column sums of gy, in one pass where the library has one."""
    nb = ws.numel()
    rc = _L.aar_gemm_f32_colsum_a(TN, out, inp, rows, _p(gy), _p(x), _p(dw), _p(db), _p(ws), nb, None)
    if rc == UNSUPPORTED:
        _ok(_L.aar_gemm_f32(TN, out, inp, rows, _p(gy), _p(x), _p(dw), _p(ws), nb, None))
        rc = _L.aar_colsum_f32(_p(gy), _p(db), rows, out, _p(ws), nb, None)
    _ok(rc)


def run(state):
    s, c = state, state["case"]
    k = c["kind"]
    if k == "gpt":
        return ag.to_numpy(s["model"](s["ids"], s["pos"]).to(ag.Device.CPU))
    ws = s.get("ws")
    nb = ws.numel() if ws is not None else 0
    if k == "matmul":
        _ok(_L.aar_gemm_f32(OPS[c["op"]], c["M"], c["N"], c["K"], _p(s["a"]), _p(s["b"]), _p(s["c"]), _p(ws), nb, None))
        return s["c"]
    if k == "linear":
        rows, inp, out = c["rows"], c["inp"], c["out"]
        _ok(_L.aar_gemm_f32_bias(NT, rows, out, inp, _p(s["x"]), _p(s["w"]), _p(s["b"]), _p(s["y"]), _p(ws), nb, None))
        _ok(_L.aar_gemm_f32(NN, rows, inp, out, _p(s["gy"]), _p(s["w"]), _p(s["dx"]), _p(ws), nb, None))
        _weight_grads(s["gy"], s["x"], s["dw"], s["db"], rows, inp, out, ws)
        return {n: s[n] for n in ("y", "dx", "dw", "db")}
    if k == "mlp":
        rows, d, h = c["rows"], c["d"], c["hidden"]
        rc = _L.aar_gemm_f32_bias_relu_bits(NT, rows, h, d, _p(s["x"]), _p(s["w1"]), _p(s["b1"]), _p(s["h"]),
                                            _p(s["h_bits"]), _p(ws), nb, None)
        if rc == UNSUPPORTED:
            rc = _L.aar_gemm_f32_bias_relu(NT, rows, h, d, _p(s["x"]), _p(s["w1"]), _p(s["b1"]), _p(s["h"]), _p(ws),
                                           nb, None)
        _ok(rc)
        _ok(_L.aar_gemm_f32_bias_add(NT, rows, d, h, _p(s["h"]), _p(s["w2"]), _p(s["b2"]), _p(s["r"]), _p(s["y"]),
                                     _p(ws), nb, None))
        rc = _L.aar_gemm_f32_mask_bits_colsum(NN, rows, h, d, _p(s["gy"]), _p(s["w2"]), _p(s["bits"]), _p(s["dh"]),
                                              None, _p(ws), nb, None)
        if rc == UNSUPPORTED:
            _ok(_L.aar_gemm_f32(NN, rows, h, d, _p(s["gy"]), _p(s["w2"]), _p(s["dh"]), _p(ws), nb, None))
            rc = _L.aar_relu_bwd_f32(_p(s["dh"]), _p(s["saved_h"]), _p(s["dh"]), rows * h, None)
        _ok(rc)
        _weight_grads(s["gy"], s["saved_h"], s["dw2"], s["db2"], rows, h, d, ws)
        _weight_grads(s["dh"], s["x"], s["dw1"], s["db1"], rows, d, h, ws)
        _ok(_L.aar_gemm_f32(NN, rows, d, h, _p(s["dh"]), _p(s["w1"]), _p(s["dx"]), _p(ws), nb, None))
        return {n: s[n] for n in ("h", "y", "dx", "dw1", "db1", "dw2", "db2")}
    if k == "head":
        rows, d, v = c["rows"], c["d"], c["vocab"]
        _ok(_L.aar_gemm_f32(NT, rows, v, d, _p(s["x"]), _p(s["w"]), _p(s["logits"]), _p(ws), nb, None))
        _ok(_L.aar_cross_entropy_fwd_f32(_p(s["logits"]), _p(s["t"]), _p(s["loss"]), rows, v, -100, None, _p(ws), nb,
                                         None))
        _ok(_L.aar_cross_entropy_bwd_f32(_p(s["one"]), _p(s["logits"]), _p(s["t"]), _p(s["dlogits"]), rows, v, -100,
                                         _p(ws), nb, None))
        _ok(_L.aar_gemm_f32(NN, rows, d, v, _p(s["dlogits"]), _p(s["w"]), _p(s["dx"]), _p(ws), nb, None))
        _ok(_L.aar_gemm_f32(TN, v, d, rows, _p(s["dlogits"]), _p(s["x"]), _p(s["dw"]), _p(ws), nb, None))
        return {n: s[n] for n in ("logits", "loss", "dlogits", "dx", "dw")}
    if k == "attention":
        B, H, T, d, causal = c["B"], c["H"], c["T"], c["d"], int(c["causal"])
        q, g, step = _p(s["qkv"]), _p(s["dqkv"]), 4 * H * d
        scale = 1.0 / math.sqrt(d)
        _ok(_L.aar_flash_fwd_strided_f32(q, q + step, q + 2 * step, _p(s["o"]), _p(s["lse"]), B, H, T, d,
                                         s["fwd_strides"], causal, scale, _p(ws), s["fwd_bytes"], None))
        _ok(_L.aar_flash_bwd_strided_f32(q, q + step, q + 2 * step, _p(s["o"]), _p(s["lse"]), _p(s["do"]), g, g + step,
                                         g + 2 * step, B, H, T, d, s["bwd_strides"], causal, scale, _p(ws),
                                         s["bwd_bytes"], None))
        return {n: s[n] for n in ("o", "lse", "dqkv")}
    rows, cols = c["rows"], c["cols"]
    if k == "layernorm":
        _ok(_L.aar_layernorm_fwd_f32(_p(s["x"]), _p(s["w"]), _p(s["b"]), _p(s["y"]), _p(s["mean"]), _p(s["rstd"]), rows,
                                     cols, 1e-5, None))
        _ok(_L.aar_layernorm_bwd_f32(_p(s["gy"]), _p(s["x"]), _p(s["w"]), _p(s["mean"]), _p(s["rstd"]), _p(s["dx"]),
                                     _p(s["dw"]), _p(s["db"]), rows, cols, _p(ws), nb, None))
        return {n: s[n] for n in ("y", "dx", "dw", "db")}
    _ok(_L.aar_softmax_fwd_f32(_p(s["x"]), _p(s["y"]), rows, cols, None))
    _ok(_L.aar_softmax_bwd_f32(_p(s["gy"]), _p(s["y"]), _p(s["dx"]), rows, cols, None))
    return {n: s[n] for n in ("y", "dx")}


# ------------------------------------------------------------------ what a pass needs

def work(case):
    """Bytes (each input read once, each output written once) and FLOPs of one pass."""
    c, k = case, case["kind"]
    if k == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 4.0 * (M * K + K * N + M * N), "flops": 2.0 * M * N * K}
    if k == "linear":
        r, i, o = c["rows"], c["inp"], c["out"]
        return {"bytes": 4.0 * (2 * r * i + 2 * r * o + 2 * i * o + 2 * o), "flops": 6.0 * r * i * o}
    if k == "mlp":
        r, d, h = c["rows"], c["d"], c["hidden"]
        return {"bytes": 4.0 * (5 * r * d + 2 * r * h + 4 * d * h), "flops": 12.0 * r * d * h}
    if k == "head":
        r, d, v = c["rows"], c["d"], c["vocab"]
        return {"bytes": 4.0 * (2 * r * d + 2 * r * v + 2 * v * d) + 8.0 * r, "flops": 6.0 * r * d * v}
    if k == "attention":
        n = float(c["B"] * c["H"] * c["T"])
        pairs = n * c["T"] * (0.5 if c["causal"] else 1.0)
        return {"bytes": 4.0 * (8 * n * c["d"] + n), "flops": 14.0 * pairs * c["d"]}
    if k == "layernorm":
        return {"bytes": 4.0 * (4 * c["rows"] * c["cols"] + 2 * c["rows"]), "flops": 18.0 * c["rows"] * c["cols"]}
    if k == "softmax":
        return {"bytes": 4.0 * 4 * c["rows"] * c["cols"], "flops": 9.0 * c["rows"] * c["cols"]}
    n, d = float(c["B"] * c["T"]), c["d"]
    params = c["layers"] * 12.0 * d * d + 2.0 * c["vocab"] * d + c["T"] * d
    return {"bytes": 4.0 * (params + n * c["vocab"]) + 16.0 * n,
            "flops": n * (c["layers"] * (24.0 * d * d + 2.0 * c["T"] * d) + 2.0 * c["vocab"] * d)}


def tolerance(case):
    """About four times the distance between two correct fp32 orders of the sums."""
    k = case["kind"]
    if k in ("softmax", "layernorm"):
        return {"rel": 2e-6, "max": 2e-5}
    if k == "matmul":
        return {"rel": 4e-8 * math.sqrt(case["K"]) + 1e-6, "max": 1e-5 + 2e-7 * math.sqrt(case["K"])}
    if k in ("linear", "mlp"):
        r = max(case["rows"], case.get("hidden", 0), case.get("out", 0), case.get("inp", 0))
        return {"rel": 4e-8 * math.sqrt(r) + 1e-6, "max": 1e-5 + 4e-7 * math.sqrt(r)}
    if k == "head":
        return {"rel": 6e-6, "max": 1e-4}
    if k == "attention":
        return {"rel": 6e-6, "max": 2e-4}
    return {"rel": 2e-5, "max": 2e-4}


# ------------------------------------------------------------------ in 64 bits

def exact(case, seed):
    k = case["kind"]
    if k == "gpt":
        return _exact_gpt(case, seed)
    s = {n: t.double() if t.is_floating_point() else t for n, t in _inputs(case, seed).items()}
    if k == "matmul":
        op = OPS[case["op"]]
        a = s["a"].t() if op == TN else s["a"]
        return a @ (s["b"].t() if op == NT else s["b"])
    if k == "linear":
        return {"y": s["x"] @ s["w"].t() + s["b"], "dx": s["gy"] @ s["w"], "dw": s["gy"].t() @ s["x"], "db": s["gy"].sum(0)}
    if k == "mlp":
        h = torch.relu(s["x"] @ s["w1"].t() + s["b1"])
        dh = (s["gy"] @ s["w2"]) * (s["saved_h"] > 0)
        return {"h": h, "y": h @ s["w2"].t() + s["b2"] + s["r"], "dx": dh @ s["w1"], "dw1": dh.t() @ s["x"],
                "db1": dh.sum(0), "dw2": s["gy"].t() @ s["saved_h"], "db2": s["gy"].sum(0)}
    if k == "head":
        rows = case["rows"]
        logits = s["x"] @ s["w"].t()
        lp = torch.log_softmax(logits, -1)
        at = torch.arange(rows, device=DEV)
        dl = lp.exp()
        dl[at, s["t"]] -= 1.0
        dl /= rows
        return {"logits": logits, "loss": -lp[at, s["t"]].mean().reshape(1), "dlogits": dl, "dx": dl @ s["w"],
                "dw": dl.t() @ s["x"]}
    if k == "attention":
        return _exact_attention(case, s["qkv"], s["do"])
    if k == "layernorm":
        x, gy, cols = s["x"], s["gy"], case["cols"]
        mean = x.mean(-1, keepdim=True)
        rstd = ((x - mean).square().mean(-1, keepdim=True) + 1e-5).rsqrt()
        xh, gw = (x - mean) * rstd, gy * s["w"]
        dx = rstd * (gw - gw.mean(-1, keepdim=True) - xh * (gw * xh).sum(-1, keepdim=True) / cols)
        return {"y": xh * s["w"] + s["b"], "dx": dx, "dw": (gy * xh).sum(0), "db": gy.sum(0)}
    y = torch.softmax(s["x"], -1)
    return {"y": y, "dx": y * (s["gy"] - (s["gy"] * y).sum(-1, keepdim=True))}


def _exact_attention(case, qkv, do):
    B, H, T, d = case["B"], case["H"], case["T"], case["d"]
    scale = 1.0 / math.sqrt(d)
    o = torch.empty(B, T, H, d, dtype=torch.float64, device=DEV)
    lse = torch.empty(B, H, T, dtype=torch.float64, device=DEV)
    g = torch.empty(B, T, 3, H, d, dtype=torch.float64, device=DEV)
    hide = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1) if case["causal"] else None
    for b in range(B):
        for h in range(H):
            q, k, v, gy = (t.contiguous() for t in (qkv[b, :, 0, h], qkv[b, :, 1, h], qkv[b, :, 2, h], do[b, :, h]))
            sc = (q @ k.t()) * scale
            if hide is not None:
                sc.masked_fill_(hide, -math.inf)
            l = torch.logsumexp(sc, -1)
            p = torch.exp(sc - l[:, None])
            out = p @ v
            ds = p * (gy @ v.t() - (gy * out).sum(-1, keepdim=True)) * scale
            o[b, :, h], lse[b, h] = out, l
            g[b, :, 0, h], g[b, :, 1, h], g[b, :, 2, h] = ds @ k, ds.t() @ q, p.t() @ gy
    return {"o": o, "lse": lse, "dqkv": g}


def _exact_gpt(case, seed):
    model, ids, pos = _gpt_arrays(case, seed)

    def w(p):
        return torch.from_numpy(ag.to_numpy(p.tensor)).to(DEV).double()

    def norm(x, m):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w(m.weight), w(m.bias), m.eps)

    B, T, d, H = case["B"], case["T"], case["d"], case["heads"]
    x = w(model.tok.weight)[torch.from_numpy(ids).to(DEV)] + w(model.pos.weight)[torch.from_numpy(pos).to(DEV)]
    hide = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
    for blk in model.blocks._modules.values():
        qkv = (norm(x, blk.ln1) @ w(blk.attn.qkv_proj.weight).t()).view(B, T, 3, H, d // H)
        q, k, v = (qkv[:, :, i].transpose(1, 2).contiguous() for i in range(3))
        sc = (q @ k.transpose(2, 3).contiguous()) / math.sqrt(d // H)
        a = torch.softmax(sc.masked_fill(hide, -math.inf), -1) @ v
        x = x + a.transpose(1, 2).reshape(B, T, d) @ w(blk.attn.out_proj.weight).t()
        up, down = blk.mlp.layer_0, blk.mlp.layer_2
        h = torch.relu(norm(x, blk.ln2) @ w(up.weight).t() + w(up.bias))
        x = x + h @ w(down.weight).t() + w(down.bias)
    return (norm(x, model.norm) @ w(model.head.weight).t()).cpu().numpy()
