"""The work that users of this framework have it do, as cases that can be timed and checked.

listed() names the fixed cases, draw() gives more of the same ranges, and each
case is run through the package's public entry points: the kernel API of
mi355x_pjrt.kernels, a StableHLO module compiled and executed through the
PJRT plugin, and the GPT-2 training step.  exact() is the same computation in
plain torch in 64 bits.
"""

from __future__ import annotations

import math
import os
import sys
import weakref

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (_ROOT, os.path.join(_ROOT, "mccl-jax_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from mi355x_pjrt import gpt2, modules, pjrt  # noqa: E402
from mi355x_pjrt import kernels as K  # noqa: E402

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEV = "cuda"


def listed():
    return [
        # The headline: a causal prompt of a long-context model, one attention call.
        {"name": "attention_long", "kind": "prefill", "batch": 4, "heads": 16, "seq": 8192, "dim": 128, "causal": True},
        # The shortest length of the published sweep: a small prompt, where the chip is not full.
        {"name": "attention_short", "kind": "prefill", "batch": 4, "heads": 16, "seq": 512, "dim": 128, "causal": True},
        # One new token of eight running sequences against their key / value caches.
        {"name": "attention_decode", "kind": "decode", "batch": 8, "heads": 16, "queries": 1, "keys": 4096, "dim": 128},
        # One layer's attention in GPT-2-small training: forward with its row statistics, then backward,
        # on the fused QKV projection's layout.
        {"name": "attention_train", "kind": "attention_train", "batch": 8, "heads": 12, "seq": 1024, "dim": 64},
        # One layer's MLP in GPT-2-small training: forward and every gradient.
        {"name": "mlp_train", "kind": "mlp_train", "tokens": 8192, "d": 768, "ff": 3072},
        # The MLP of a model of width 4096 for one token of each of 16 sequences: the weights are the traffic.
        {"name": "mlp_decode", "kind": "mlp_decode", "tokens": 16, "d": 4096, "ff": 16384},
        # A jitted fp32 two-layer MLP through the plugin: compile once, execute per batch.
        {"name": "mlp_jit_f32", "kind": "mlp_jit", "batch": 256, "d": 1024, "ff": 4096},
        # The vocabulary head of GPT-2-small training: logits, loss, and the gradients of both operands.
        {"name": "head_train", "kind": "head_train", "tokens": 8192, "d": 768, "vocab": 50257},
        # A pre-LayerNorm block's residual add and norm in training, forward and backward.
        {"name": "norm_train", "kind": "norm_train", "rows": 8192, "cols": 768, "dtype": "bf16"},
        # Greedy decoding: the next token of 32 sequences from rows of 50257 logits (rows that start unaligned).
        {"name": "rows_argmax", "kind": "rows", "op": "argmax", "rows": 32, "cols": 50257, "dtype": "bf16"},
        # Token embeddings of 32 sequences of 2048: the lookup, and its gradient back into the table.
        {"name": "embedding_train", "kind": "embedding", "ids": 65536, "vocab": 50257, "d": 768},
        # A whole GPT-2-small training step (forward, backward, Adam), replayed as the captured graph.
        {"name": "train_step", "kind": "step", "layers": 12, "d": 768, "heads": 12, "seq": 1024, "batch": 8,
         "vocab": 50257},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_mult(rng, lo, hi, m):
    return max(lo, _log(rng, lo, hi) // m * m)


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "decode", "attention_train", "mlp_train", "mlp_decode", "mlp_jit",
                       "head_train", "norm_train", "rows", "rows", "embedding", "step"])
    if kind == "prefill":
        seq = _log(rng, 64, 8192)
        pairs = max(1, min(128, _log(rng, 4, 128), int(64 * 8192 ** 2 / seq ** 2)))
        heads = rng.choice([h for h in (1, 4, 8, 12, 16) if h <= pairs])
        return {"kind": kind, "batch": max(1, pairs // heads), "heads": heads, "seq": seq, "dim": rng.choice([64, 128]),
                "causal": pairs > 64 or rng.random() < 0.75}
    if kind == "decode":
        keys = _log(rng, 64, 16384)
        return {"kind": kind, "batch": max(1, min(_log(rng, 1, 32), 131072 // keys)), "heads": rng.choice([8, 12, 16]),
                "queries": rng.choice([1, 1, 1, 2, 4, 7]), "keys": keys, "dim": rng.choice([64, 128])}
    if kind == "attention_train":
        seq = _log(rng, 128, 4096)
        heads, dim = rng.choice([(12, 64), (16, 64), (8, 128), (16, 128)])
        return {"kind": kind, "batch": max(1, min(8, _log(rng, 1, 16384) // seq)), "heads": heads, "seq": seq,
                "dim": dim}
    if kind == "mlp_train":
        d = _log_mult(rng, 256, 2048, 64)
        return {"kind": kind, "tokens": _log(rng, 256, 8192), "d": d, "ff": 4 * d}
    if kind == "mlp_decode":
        d = _log_mult(rng, 512, 4096, 64)
        return {"kind": kind, "tokens": _log(rng, 1, 64), "d": d, "ff": 4 * d}
    if kind == "mlp_jit":
        d = _log_mult(rng, 128, 1024, 32)
        return {"kind": kind, "batch": _log(rng, 1, 1024), "d": d, "ff": 4 * d}
    if kind == "head_train":
        return {"kind": kind, "tokens": _log(rng, 512, 8192), "d": _log_mult(rng, 256, 768, 64),
                "vocab": _log(rng, 8000, 50257)}
    if kind == "norm_train":
        return {"kind": kind, "rows": _log(rng, 64, 32768), "cols": _log_mult(rng, 128, 2048, 4),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "rows":
        rows = _log(rng, 1, 65536)
        return {"kind": kind, "op": rng.choice(["argmax", "layernorm", "gelu", "softmax", "sum"]), "rows": rows,
                "cols": min(_log(rng, 64, 50257), max(64, 8192 * 16384 // rows)),
                "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "embedding":
        return {"kind": kind, "ids": _log(rng, 64, 65536), "vocab": _log(rng, 1000, 50257),
                "d": _log_mult(rng, 128, 1024, 8)}
    heads = rng.choice([2, 4, 8, 12])
    return {"kind": "step", "layers": rng.randint(1, 4), "d": 64 * heads, "heads": heads,
            "seq": _log_mult(rng, 128, 1024, 8), "batch": rng.randint(1, 8), "vocab": _log(rng, 2000, 50257)}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype=BF16, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device=DEV) * std + mean).to(dtype)


def _ints(g, shape, high):
    return torch.randint(high, shape, generator=g, device=DEV, dtype=torch.int32)


def _dtype(case):
    return BF16 if case["dtype"] == "bf16" else F32


def _client():
    """The process's one PJRT client, as a program that registers the plugin has."""
    if not hasattr(_client, "c"):
        _client.c = pjrt.Plugin().client()
    return _client.c


class _Module:
    """A compiled module and its resident arguments."""

    def __init__(self, text, arrays):
        self.exe = _client().compile(text)
        self.args = [_client().put(a) for a in arrays]
        self.shapes = self.exe.output_shapes()
        for r in (self.exe, *self.args):
            weakref.finalize(self, r.destroy)


class _Result:
    """An output buffer of a module that torch can read where it is (fp32)."""

    def __init__(self, buffer, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (buffer.device_pointer, False),
                                         "version": 2, "strides": None}
        weakref.finalize(self, buffer.destroy)


def _inputs(case, seed):
    """The tensors of one pass, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("prefill", "decode"):
        # q, k and v as the published benchmark draws them; the caches hold room beyond the keys in use
        B, H, D = case["batch"], case["heads"], case["dim"]
        std = 1 / math.sqrt(D) if kind == "prefill" else 1.0
        if kind == "prefill":
            return {n: _normal(g, (B, H, case["seq"], D), std=std) for n in "qkv"}
        room = (case["keys"] + 255) // 256 * 256
        s = {"q": _normal(g, (B, H, case["queries"], D))}
        for n in "kv":
            s[n] = _normal(g, (B, H, room, D))[:, :, :case["keys"]]
        return s
    if kind == "attention_train":
        B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
        qkv = _normal(g, (B, S, 3, H, D)).permute(2, 0, 3, 1, 4)  # views into one projection's output
        return {"q": qkv[0], "k": qkv[1], "v": qkv[2], "do": _normal(g, (B, S, H, D), std=0.1).transpose(1, 2)}
    if kind in ("mlp_train", "mlp_decode"):
        T, d, f = case["tokens"], case["d"], case["ff"]
        s = {"x": _normal(g, (T, d)), "w1": _normal(g, (d, f), std=1 / math.sqrt(d)), "b1": _normal(g, (f,), std=0.1),
             "w2": _normal(g, (f, d), std=1 / math.sqrt(f)), "b2": _normal(g, (d,), std=0.1)}
        if kind == "mlp_train":
            s["dy"] = _normal(g, (T, d), std=0.1)
        return s
    if kind == "mlp_jit":
        m, d, f = case["batch"], case["d"], case["ff"]
        return {n: _normal(g, shape, F32, std=0.02) for n, shape in
                (("x", (m, d)), ("w1", (d, f)), ("b1", (f,)), ("w2", (f, d)), ("b2", (d,)))}
    if kind == "head_train":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        return {"h": _normal(g, (T, d)), "wte": _normal(g, (V, d), std=0.02), "labels": _ints(g, (T,), V)}
    if kind == "norm_train":
        R, C, dt = case["rows"], case["cols"], _dtype(case)
        s = {n: _normal(g, (R, C), dt) for n in ("a", "b")}
        s.update(bias=_normal(g, (C,), dt, 0.1) if dt == BF16 else None, gamma=_normal(g, (C,), dt, 0.1, 1.0),
                 beta=_normal(g, (C,), dt, 0.1), dy=_normal(g, (R, C), dt, 0.1), dres=_normal(g, (R, C), dt, 0.1))
        return s
    if kind == "rows":
        dt, C = _dtype(case), case["cols"]
        s = {"x": _normal(g, (case["rows"], C), dt)}
        if case["op"] == "layernorm":
            s.update(gamma=_normal(g, (C,), dt, 0.1, 1.0), beta=_normal(g, (C,), dt, 0.1))
        return s
    if kind == "embedding":
        n, V, d = case["ids"], case["vocab"], case["d"]
        return {"table": _normal(g, (V, d), std=0.02), "grad": _normal(g, (V, d), F32, 0.01), "ids": _ints(g, (n,), V),
                "updates": _normal(g, (n, d), F32, 0.01)}
    raise ValueError(kind)


def _prepare_step(case, seed):
    cfg = gpt2.GPT2Config(n_layer=case["layers"], d_model=case["d"], n_head=case["heads"], seq=case["seq"],
                          batch=case["batch"], vocab=case["vocab"])
    g, params = _gen(seed), {}
    for name, shape in cfg.param_shapes():
        leaf = name.split(".")[-1]
        if leaf.endswith("_g"):
            p = torch.ones(shape, device=DEV)
        elif leaf.startswith("b_") or leaf.endswith("_b"):
            p = torch.zeros(shape, device=DEV)
        else:
            p = _normal(g, shape, F32, 0.02)
        params[name] = p.cpu().numpy()
    step = gpt2.GPT2TrainStep(cfg, params=params, stream=torch.cuda.Stream())
    step.set_batch(_ints(g, (cfg.tokens,), cfg.vocab), _ints(g, (cfg.tokens,), cfg.vocab))
    torch.cuda.synchronize()
    step.step()  # the eager step that capture() asks for
    step.stream.synchronize()
    step.capture()
    return {"step": step}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        s = _prepare_step(case, seed)
    elif kind == "mlp_jit":
        m, d, f = case["batch"], case["d"], case["ff"]
        s = {"module": _Module(modules.mlp(m, d, f, d), [t.cpu().numpy() for t in _inputs(case, seed).values()])}
    else:
        s = _inputs(case, seed)
    if kind == "head_train":
        # logits in rows padded to 16 bytes, as the training step keeps them
        V = case["vocab"]
        s["logits"] = torch.zeros(case["tokens"], (V + 7) // 8 * 8, dtype=BF16, device=DEV)[:, :V]
    s["case"] = case
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "prefill":
        return K.sdpa_fwd(s["q"], s["k"], s["v"], 1 / math.sqrt(case["dim"]), causal=case["causal"])
    if kind == "decode":
        return K.sdpa_fwd(s["q"], s["k"], s["v"], 1 / math.sqrt(case["dim"]), causal=False)
    if kind == "attention_train":
        q, scale = s["q"], 1 / math.sqrt(case["dim"])
        o = torch.empty_like(s["do"])
        lse = torch.empty(q.shape[:3], dtype=F32, device=DEV)
        K.sdpa_fwd(q, s["k"], s["v"], scale, causal=True, out=o, lse=lse)
        dq, dk, dv = K.sdpa_bwd(q, s["k"], s["v"], o, s["do"], lse, scale, causal=True)
        return {"o": o, "dq": dq, "dk": dk, "dv": dv}
    if kind == "mlp_train":
        x, w1, w2, dy = s["x"], s["w1"], s["w2"], s["dy"]
        pre, act = K.gemm_bias_gelu(x, w1, s["b1"])
        y = K.gemm(act, w2, bias=s["b2"])
        dw2 = K.gemm_splitk(act.t(), dy, 4)
        db2 = K.col_sum(dy)
        dact = K.gemm(dy, w2.t())
        dpre, db1 = K.gelu_tanh_bwd_colsum(pre, dact, out=dact)
        dw1 = K.gemm_splitk(x.t(), dpre, 4)
        dx = K.gemm(dpre, w1.t())
        return {"y": y, "dx": dx, "dw1": dw1, "db1": db1, "dw2": dw2, "db2": db2}
    if kind == "mlp_decode":
        return K.gemm(K.gelu_tanh(K.gemm(s["x"], s["w1"], bias=s["b1"])), s["w2"], bias=s["b2"])
    if kind == "mlp_jit":
        m = s["module"]
        outs = m.exe.execute(m.args, wait=False)
        return [torch.as_tensor(_Result(b, shape), device=DEV) for b, shape in zip(outs, m.shapes)]
    if kind == "head_train":
        logits, wte, T = s["logits"], s["wte"], case["tokens"]
        K.gemm(s["h"], wte.t(), out=logits)
        loss, dlogits = K.softmax_xent(logits, s["labels"], 1 / T, dlogits=logits)
        dh = K.gemm_splitk(dlogits, wte, 8, out_dtype=BF16)
        dwte = K.gemm(dlogits.t(), s["h"], out_dtype=F32)
        return {"loss": loss, "dlogits": dlogits, "dh": dh, "dwte": dwte}
    if kind == "norm_train":
        x, y = K.add_layernorm(s["a"], s["b"], s["bias"], s["gamma"], s["beta"])
        dx, dgamma, dbeta, dbias = K.layernorm_bwd(x, s["gamma"], s["dy"], dres=s["dres"], want_colsum=True)
        return {"x": x, "y": y, "dx": dx, "dgamma": dgamma, "dbeta": dbeta, "dbias": dbias}
    if kind == "rows":
        x, op = s["x"], case["op"]
        if op == "argmax":
            index, value = K.row_argmax(x)
            return {"index": index, "value": value}
        if op == "layernorm":
            return K.layernorm(x, s["gamma"], s["beta"])
        if op == "gelu":
            return K.gelu_tanh(x)
        return K.softmax_rows(x) if op == "softmax" else K.row_reduce(x, "sum")
    if kind == "embedding":
        return {"rows": K.gather_rows(s["table"], s["ids"]),
                "grad": K.scatter_add_rows(s["grad"], s["ids"], s["updates"])}
    step = s["step"]
    loss = step.replay()
    return {"loss": loss, "param": step.param, **_gradients(step)}


def _gradients(step):
    """The step's gradients by parameter name, a layer parameter's of all layers as one view."""
    (first, _), layers = step.offsets["h0.ln1_g"], step.cfg.n_layer
    pitch = (step.offsets["lnf_g"][0] - first) // layers
    grads = {n: step.view(step.grad, n) for n in ("wte", "wpe", "lnf_g", "lnf_b")}
    for name, (offset, shape) in step.offsets.items():
        if name.startswith("h0."):
            grads[name[3:]] = step.grad.as_strided((layers, math.prod(shape)), (pitch, 1), offset)
    return grads


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("prefill", "attention_train"):
        B, H, S, D = case["batch"], case["heads"], case["seq"], case["dim"]
        pairs = S * (S + 1) / 2 if case.get("causal", True) else S * S  # the (query, key) pairs that are seen
        product, tensor = 2 * B * H * pairs * D, 2 * B * H * S * D
        if kind == "prefill":
            return {"flops": 2 * product, "bytes": 4 * tensor}
        return {"flops": 7 * product, "bytes": 8 * tensor}
    if kind == "decode":
        B, H, Q, S, D = (case[n] for n in ("batch", "heads", "queries", "keys", "dim"))
        return {"flops": 4 * B * H * Q * S * D, "bytes": 4 * B * H * (Q + S) * D}
    if kind in ("mlp_train", "mlp_decode"):
        T, d, f = case["tokens"], case["d"], case["ff"]
        if kind == "mlp_decode":
            return {"flops": 4 * T * d * f, "bytes": 2 * (2 * d * f + d + f + 2 * T * d)}
        return {"flops": 12 * T * d * f, "bytes": 2 * 4 * T * d + (4 + 8) * d * f + 6 * (d + f)}
    if kind == "mlp_jit":
        m, d, f = case["batch"], case["d"], case["ff"]
        return {"flops": 4 * m * d * f, "bytes": 4 * (2 * d * f + d + f + 2 * m * d)}
    if kind == "head_train":
        T, d, V = case["tokens"], case["d"], case["vocab"]
        # the logits' gradient is written; logits and exponentials need not be
        return {"flops": 6 * T * d * V, "bytes": 2 * T * V + 4 * T * d + 6 * V * d + 8 * T}
    if kind == "norm_train":
        R, C, e = case["rows"], case["cols"], 2 if case["dtype"] == "bf16" else 4
        return {"flops": 20 * R * C, "bytes": 7 * R * C * e + 3 * C * e + 12 * C}
    if kind == "rows":
        R, C, e = case["rows"], case["cols"], 2 if case["dtype"] == "bf16" else 4
        out = {"argmax": R * (4 + e), "sum": 4 * R}.get(case["op"], R * C * e)
        return {"flops": 4 * R * C, "bytes": R * C * e + out}
    if kind == "embedding":
        n, V, d = case["ids"], case["vocab"], case["d"]
        used = min(n, V) * 2 * d  # rows of the table that are looked up, once each
        return {"flops": n * d, "bytes": 2 * 4 * n + used + n * d * (2 + 4) + 8 * V * d}
    cfg = gpt2.GPT2Config(n_layer=case["layers"], d_model=case["d"], n_head=case["heads"], seq=case["seq"],
                          batch=case["batch"], vocab=case["vocab"])
    n = sum(math.prod(shape) for _, shape in cfg.param_shapes())
    return {"flops": cfg.flops_per_step(), "bytes": 30 * n}  # weights and Adam state read and written, the gradient


def tolerance(case):
    kind = case["kind"]
    if kind == "embedding" or (kind == "rows" and case["op"] == "argmax"):
        return "exact"  # copies, whole numbers, and sums whose order the entry point fixes
    if kind == "mlp_jit" or (kind == "rows" and case["op"] == "sum"):
        return {"rel": 1e-5}
    if kind in ("rows", "norm_train") and case["dtype"] == "f32":
        return {"rel": 1e-5}
    if kind == "step":
        return {"rel": 3e-2, "max": 0.6}  # roundings to bf16 travel through all layers
    return {"rel": 8e-3}  # results, or values they are computed from, rounded to bf16


# ---------------------------------------------------------------- the same in 64 bits
def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _gelu64_grad(x):
    c = math.sqrt(2 / math.pi)
    t = torch.tanh(c * (x + 0.044715 * x ** 3))
    return 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * c * (1 + 3 * 0.044715 * x * x)


def _attention64(s, case, causal):
    """o (and, with a cotangent, the three gradients) head by head."""
    q, scale = s["q"], 1 / math.sqrt(case["dim"])
    outs = {"o": torch.empty(q.shape, dtype=F64, device=DEV)}
    if "do" in s:
        outs.update({n: torch.empty(q.shape, dtype=F64, device=DEV) for n in ("dq", "dk", "dv")})
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            qh, kh, vh = (s[n][b, h].double() for n in "qkv")
            p = (qh @ kh.t()) * scale
            if causal:
                p.masked_fill_(torch.ones_like(p, dtype=torch.bool).triu_(1), -math.inf)
            p = torch.softmax(p, -1)
            outs["o"][b, h] = p @ vh
            if "do" in s:
                do = s["do"][b, h].double()
                dp = do @ vh.t()
                ds = p * (dp - (dp * p).sum(-1, keepdim=True)) * scale
                outs["dq"][b, h], outs["dk"][b, h], outs["dv"][b, h] = ds @ kh, ds.t() @ qh, p.t() @ do
    return outs


def _layernorm64(x, gamma, beta, eps=1e-5):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], gamma, beta, eps)


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        return None
    s = _inputs(case, seed)
    if kind in ("prefill", "decode"):
        return _attention64(s, case, case.get("causal", False))["o"]
    if kind == "attention_train":
        return _attention64(s, case, True)
    d = {n: t.double() if t is not None and t.is_floating_point() else t for n, t in s.items()}
    if kind == "mlp_train":
        pre = d["x"] @ d["w1"] + d["b1"]
        act = _gelu64(pre)
        dpre = (d["dy"] @ d["w2"].t()) * _gelu64_grad(pre)
        return {"y": act @ d["w2"] + d["b2"], "dx": dpre @ d["w1"].t(), "dw1": d["x"].t() @ dpre, "db1": dpre.sum(0),
                "dw2": act.t() @ d["dy"], "db2": d["dy"].sum(0)}
    if kind == "mlp_decode":
        return _gelu64(d["x"] @ d["w1"] + d["b1"]) @ d["w2"] + d["b2"]
    if kind == "mlp_jit":
        return [torch.relu(d["x"] @ d["w1"] + d["b1"]) @ d["w2"] + d["b2"]]
    if kind == "head_train":
        h, wte, labels = d["h"], d["wte"], d["labels"].long()[:, None]
        x = h @ wte.t()
        lse = torch.logsumexp(x, -1, keepdim=True)
        loss = (lse - x.gather(1, labels))[:, 0]
        x.sub_(lse).exp_().scatter_add_(1, labels, torch.full_like(lse, -1.0)).div_(case["tokens"])
        return {"loss": loss, "dlogits": x, "dh": x @ wte, "dwte": x.t() @ h}
    if kind == "norm_train":
        x = d["a"] + d["b"] + (0 if d["bias"] is None else d["bias"])
        mean, var = x.mean(-1, keepdim=True), x.var(-1, unbiased=False, keepdim=True)
        rstd = torch.rsqrt(var + 1e-5)
        xh, g = (x - mean) * rstd, d["dy"] * d["gamma"]
        dx = rstd * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True)) + d["dres"]
        return {"x": x, "y": xh * d["gamma"] + d["beta"], "dx": dx, "dgamma": (d["dy"] * xh).sum(0),
                "dbeta": d["dy"].sum(0), "dbias": dx.sum(0)}
    if kind == "rows":
        x, op = d["x"], case["op"]
        if op == "argmax":
            value = x.amax(-1, keepdim=True)
            return {"index": (x == value).to(torch.uint8).argmax(-1).int(), "value": value[:, 0]}
        if op == "layernorm":
            return _layernorm64(x, d["gamma"], d["beta"])
        if op == "gelu":
            return _gelu64(x)
        return torch.softmax(x, -1) if op == "softmax" else x.sum(-1)
    ids = d["ids"].long()
    return {"rows": d["table"][ids], "grad": d["grad"].index_add(0, ids, d["updates"])}
