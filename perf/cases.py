"""Performance cases: the work a user of the HIP realizer has it do.

Every case is one pass through the public bridge (``HipRealizerBridge``) or the
walker, on operands that are already resident, and leaves its results resident.
Outputs are torch views of the result handles' device memory; a state releases
the handles of its last pass at its next one.
"""
from __future__ import annotations

import math
from typing import Any, Dict, List, Optional, Tuple

import numpy as np
import torch

from browsergrad_amd.bridge import HipRealizerBridge
from browsergrad_amd.jit import GpuBufferTable, Session, autocast
from browsergrad_amd.jit.configs import gpt2_block
from browsergrad_amd.jit.realize import prepare as prepare_graph
from browsergrad_amd.jit.realize import walk

ITEM = {"float32": 4, "float16": 2, "bfloat16": 2}
TORCH = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
VIEW = {"float32": "<f4", "float16": "<f2", "bfloat16": "<i2"}
ACT = {"none": 0, "relu": 1, "gelu": 2}
ADAMW = dict(lr=6e-4, beta1=0.9, beta2=0.95, eps=1e-8, weight_decay=0.1, step=10)
EPS = 1e-5


def listed() -> List[Dict[str, Any]]:
    return [
        # A small classifier (784 -> 128 -> 10) on one batch: latency and launches.
        {"name": "mlp_f32", "op": "mlp", "batch": 64, "din": 784, "hidden": 128, "dout": 10},
        # An elementwise chain with a row sum at a size that streams from HBM.
        {"name": "fused_rowsum_f32", "op": "fused", "rows": 4096, "cols": 4096, "dtype": "float32"},
        # A large layer under float16 autocast, weight already laid out as [N][K].
        {"name": "linear_f16", "op": "linear", "m": 4096, "n": 4096, "k": 4096, "dtype": "float16",
         "out": "float16", "trans_b": True, "act": "none", "residual": False},
        # An MLP layer in bfloat16 on a ragged number of rows (prompts packed without padding).
        {"name": "linear_bf16_gelu", "op": "linear", "m": 2047, "n": 3072, "k": 768, "dtype": "bfloat16",
         "out": "bfloat16", "trans_b": True, "act": "gelu", "residual": False},
        # The bridge's own product: float32 x @ w with w as [K][N].
        {"name": "matmul_f32", "op": "linear", "m": 4096, "n": 4096, "k": 4096, "dtype": "float32",
         "out": "float32", "trans_b": False, "act": "none", "residual": False},
        # Causal self attention of a long batch (prefill, training forward).
        {"name": "attention_f16", "op": "attention", "b": 8, "h": 16, "sq": 2048, "sk": 2048, "d": 64,
         "causal": True, "dtype": "float16"},
        # One new token for each sequence against its cached keys (decode).
        {"name": "attention_decode_f16", "op": "attention", "b": 8, "h": 12, "sq": 1, "sk": 1024, "d": 64,
         "causal": False, "dtype": "float16"},
        # Attention in the bridge's own dtype at a length that no tile divides.
        {"name": "attention_f32", "op": "attention", "b": 4, "h": 12, "sq": 1000, "sk": 1000, "d": 64,
         "causal": True, "dtype": "float32"},
        # One GPT-2 block under float16 autocast through the walker: a whole call.
        {"name": "gpt2_block_f16", "op": "block", "b": 8, "s": 1024, "heads": 12},
        # LayerNorm in training: forward and its three gradients.
        {"name": "layernorm_train", "op": "layernorm", "rows": 8192, "cols": 768},
        # AdamW over the largest tensor of GPT-2 small (the 50257 x 768 embedding).
        {"name": "adamw_embedding", "op": "adamw", "n": 50257 * 768},
        # A 3x3 ResNet layer in training: forward and the three gradients.
        {"name": "conv2d_train", "op": "conv", "n": 32, "c": 128, "o": 128, "hw": 28, "k": 3, "stride": 1, "pad": 1},
    ]


def _log(rng: Any, lo: float, hi: float) -> int:
    """A whole number between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: Any) -> Dict[str, Any]:
    op = rng.choice(["mlp", "fused", "linear16", "linear32", "attention16", "attention32", "decode", "block",
                     "layernorm", "adamw", "conv"])
    if op == "mlp":
        return {"op": "mlp", "batch": _log(rng, 1, 512), "din": _log(rng, 16, 2048), "hidden": _log(rng, 16, 1024),
                "dout": _log(rng, 2, 256)}
    if op == "fused":
        cols = _log(rng, 64, 65536)
        return {"op": "fused", "rows": _log(rng, 16, max(16, 2 ** 24 // cols)), "cols": cols,
                "dtype": rng.choice(["float32", "float16", "bfloat16"])}
    if op in ("linear16", "linear32"):
        wide = op == "linear32"
        n, k = (rng.choice([768, 1024, 2304, 3072, 4096, _log(rng, 64, 4096)]) for _ in range(2))
        dtype = "float32" if wide else rng.choice(["float16", "bfloat16"])
        return {"op": "linear", "m": _log(rng, 1, 4096), "n": n, "k": k, "dtype": dtype,
                "out": dtype if wide else rng.choice([dtype, "float32"]), "trans_b": rng.choice([True, False]) if wide
                else True, "act": rng.choice(["none", "relu"] if wide else ["none", "relu", "gelu"]),
                "residual": False if not wide else rng.choice([True, False])}
    if op in ("attention16", "attention32"):
        s = _log(rng, 16, 2048)
        heads = _log(rng, 1, max(1, min(128, (128 if op == "attention16" else 48) * 2 ** 21 // (s * s))))
        b = rng.choice([x for x in (1, 2, 4, 8) if x <= heads])
        causal = rng.choice([True, False])
        return {"op": "attention", "b": b, "h": max(1, heads // b), "sq": s, "sk": s if causal else _log(rng, 16, 2048),
                "d": rng.choice([64, 64, 32]), "causal": causal,
                "dtype": "float32" if op == "attention32" else rng.choice(["float16", "bfloat16"])}
    if op == "decode":
        return {"op": "attention", "b": _log(rng, 1, 64), "h": rng.choice([12, 16]), "sq": rng.choice([1, 1, 1, 2, 4]),
                "sk": _log(rng, 16, 4096), "d": 64, "causal": False,
                "dtype": rng.choice(["float16", "float16", "bfloat16", "float32"])}
    if op == "block":
        return {"op": "block", "b": rng.choice([1, 2, 4, 8]), "s": _log(rng, 16, 1024), "heads": rng.choice([6, 8, 12])}
    if op == "layernorm":
        cols = rng.choice([256, 768, 1024, 2048, 4096, _log(rng, 64, 8192)])
        return {"op": "layernorm", "rows": _log(rng, 8, 2 ** 23 // cols), "cols": cols}
    if op == "adamw":
        return {"op": "adamw", "n": _log(rng, 768, 50257 * 768)}
    hw = rng.choice([7, 14, 28, 56, _log(rng, 7, 64)])
    c, o = (rng.choice([32, 64, 128, 256, _log(rng, 3, 256)]) for _ in range(2))
    k = rng.choice([3, 3, 3, 1, 5])
    top = int(32 * 128 * 128 * 28 * 28 * 9 / (c * o * hw * hw * k * k))
    return {"op": "conv", "n": _log(rng, 1, max(1, min(64, top))), "c": c, "o": o, "hw": hw, "k": k,
            "stride": rng.choice([1, 1, 2]), "pad": k // 2}


# ---------------------------------------------------------------------------- inputs

def _tensors(case: Dict[str, Any], seed: int) -> Dict[str, torch.Tensor]:
    """The case's operands, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)

    def normal(*shape: int, std: float = 1.0, mean: float = 0.0, dtype: str = "float32") -> torch.Tensor:
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=g)
        return t.to(TORCH[dtype])

    def uniform(*shape: int, lim: float = 1.0, dtype: str = "float32") -> torch.Tensor:
        t = torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(-lim, lim, generator=g)
        return t.to(TORCH[dtype])

    op = case["op"]
    if op == "mlp":
        l1, l2 = case["din"] ** -0.5, case["hidden"] ** -0.5
        return {"x": normal(case["batch"], case["din"]), "w1": uniform(case["hidden"], case["din"], lim=l1),
                "b1": uniform(case["hidden"], lim=l1), "w2": uniform(case["dout"], case["hidden"], lim=l2),
                "b2": uniform(case["dout"], lim=l2)}
    if op == "fused":
        return {n: normal(case["rows"], case["cols"], dtype=case["dtype"]) for n in "abc"}
    if op == "linear":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        t = {"a": normal(m, k, dtype=dt), "b": uniform(*((n, k) if case["trans_b"] else (k, n)), lim=k ** -0.5, dtype=dt),
             "bias": uniform(n, lim=k ** -0.5)}
        if case["residual"]:
            t["residual"] = normal(m, n)
        return t
    if op == "attention":
        b, h, d, dt = case["b"], case["h"], case["d"], case["dtype"]
        return {"q": normal(b, h, case["sq"], d, dtype=dt), "k": normal(b, h, case["sk"], d, dtype=dt),
                "v": normal(b, h, case["sk"], d, dtype=dt)}
    if op == "block":
        e = case["heads"] * 64
        t = {"x": normal(case["b"], case["s"], e)}
        for name, o, i in (("qkv", 3 * e, e), ("o", e, e), ("up", 4 * e, e), ("down", e, 4 * e)):
            t["w_" + name] = normal(o, i, std=0.02)
            t["b_" + name] = normal(o, std=0.02)
        for name in ("ln1", "ln2"):
            t[name + "_w"] = normal(e, std=0.1, mean=1.0)
            t[name + "_b"] = normal(e, std=0.02)
        return t
    if op == "layernorm":
        r, c = case["rows"], case["cols"]
        return {"x": normal(r, c, mean=0.1), "dy": normal(r, c, std=0.1), "w": normal(c, std=0.1, mean=1.0),
                "b": normal(c, std=0.02)}
    if op == "adamw":
        n = case["n"]
        return {"p": normal(n, std=0.02), "g": normal(n, std=1e-3), "m": normal(n, std=1e-3),
                "v": normal(n, std=1e-3).square_()}
    n, c, o, hw, k = (case[x] for x in ("n", "c", "o", "hw", "k"))
    out = _conv_out(case)
    return {"x": normal(n, c, hw, hw), "w": normal(o, c, k, k, std=(c * k * k) ** -0.5), "b": normal(o, std=0.1),
            "dy": normal(n, o, out, out)}


def _conv_out(case: Dict[str, Any]) -> int:
    return (case["hw"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1


# ---------------------------------------------------------------------------- the pass

_BRIDGE: Optional[HipRealizerBridge] = None


def _bridge() -> HipRealizerBridge:
    """The program's one bridge (one context: one device and stream)."""
    global _BRIDGE
    if _BRIDGE is None:
        _BRIDGE = HipRealizerBridge(device=0)
    return _BRIDGE


class _Memory:
    """A result handle's device memory, for torch.as_tensor."""

    def __init__(self, ptr: int, shape: Tuple[int, ...], dtype: str) -> None:
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": VIEW[dtype], "version": 2}


class State:
    """What a user's program holds: operand handles, a prepared graph, and the last pass's results."""

    def __init__(self, case: Dict[str, Any], seed: int) -> None:
        self.case = case
        self.br = _bridge()
        self.h: Dict[str, int] = {}
        self.results: List[int] = []
        self.views: Dict[Tuple, torch.Tensor] = {}
        self.graph: Any = None
        t = _tensors(case, seed)
        if case["op"] == "block":
            self._prepare_block({k: v.cpu().numpy() for k, v in t.items()})
            return
        for name, x in t.items():
            host = x.view(torch.int16) if x.dtype == torch.bfloat16 else x
            self.h[name] = self.br.upload(host.cpu().numpy(), tuple(x.shape), str(x.dtype).split(".")[1])

    def _prepare_block(self, t: Dict[str, np.ndarray]) -> None:
        s = Session()
        leaf = {k: s.from_numpy(v, k) for k, v in t.items()}
        with autocast("float16"):
            y = gpt2_block(leaf["x"], leaf, self.case["heads"])
        self.buffers = s.buffers
        self.graph = prepare_graph(y.uop, s.buffers)
        self.gbt = GpuBufferTable(self.br)
        self.shape = tuple(y.uop.shape)

    def hold(self, *results: Tuple[int, Tuple[int, ...], str]) -> Any:
        """Keeps these results, gives the last pass's back and returns tensors of the new ones."""
        for h in self.results:
            self.br.release(h)
        self.results = [r[0] for r in results]
        out = []
        for h, shape, dtype in results:
            key = (self.br.device_ptr(h), shape, dtype)
            v = self.views.get(key)
            if v is None:
                if len(self.views) >= 32:
                    self.views.clear()
                v = torch.as_tensor(_Memory(*key), device="cuda")
                v = self.views[key] = v.view(torch.bfloat16) if dtype == "bfloat16" else v
            out.append(v)
        return out[0] if len(out) == 1 else out

    def __del__(self) -> None:
        try:
            for h in [*self.results, *self.h.values()]:
                self.br.release(h)
            if self.graph is not None:
                self.gbt.release_all()
        except Exception:  # the interpreter is shutting down
            pass


def prepare(case: Dict[str, Any], seed: int) -> State:
    return State(case, seed)


FUSED_OPS = [("MUL", -1, -2, 0), ("ADD", 0, -3, 0), ("IMM", 0, 0, 0), ("CMP_GT", 1, 2, 0), ("WHERE", 3, 1, 2),
             ("NEG", -1, 0, 0), ("MUL", 5, -1, 0), ("EXP", 6, 0, 0), ("MUL", 4, 7, 0)]


def run(s: State) -> Any:
    c, br, h = s.case, s.br, s.h
    op = c["op"]
    if op == "mlp":
        b, i, m, o = c["batch"], c["din"], c["hidden"], c["dout"]
        h1 = br.matmul_ex(h["x"], h["w1"], m=b, n=m, k=i, trans_b=True, bias=h["b1"], act=ACT["relu"])
        y = br.matmul_ex(h1, h["w2"], m=b, n=o, k=m, trans_b=True, bias=h["b2"])
        br.release(h1)
        return s.hold((y, (b, o), "float32"))
    if op == "fused":
        # sum over each row of relu(a * b + c) * exp(-a * a)
        y = br.fused_ex([h["a"], h["b"], h["c"]], FUSED_OPS, (c["rows"], c["cols"]), "float32", imms=[0.0], reduce=1)
        return s.hold((y, (c["rows"],), "float32"))
    if op == "linear":
        y = br.matmul_ex(h["a"], h["b"], m=c["m"], n=c["n"], k=c["k"], trans_b=c["trans_b"], in_dtype=c["dtype"],
                         out_dtype=c["out"], bias=h["bias"], act=ACT[c["act"]], residual=h.get("residual"))
        return s.hold((y, (c["m"], c["n"]), c["out"]))
    if op == "attention":
        y = br.attention_ex(h["q"], h["k"], h["v"], batch=c["b"], heads=c["h"], sq=c["sq"], sk=c["sk"], d=c["d"],
                            scale=c["d"] ** -0.5, causal=c["causal"], in_dtype=c["dtype"], out_dtype=c["dtype"])
        return s.hold((y, (c["b"], c["h"], c["sq"], c["d"]), c["dtype"]))
    if op == "block":
        return s.hold((walk(s.graph, s.buffers, s.gbt, materialize=False), s.shape, "float32"))
    if op == "layernorm":
        r, n = c["rows"], c["cols"]
        y = br.layer_norm(h["x"], h["w"], h["b"], r, n, EPS)
        dx = br.layer_norm_backward_input(h["dy"], h["x"], h["w"], r, n, EPS)
        dw = br.layer_norm_backward_weight(h["dy"], h["x"], r, n, EPS)
        db = br.layer_norm_backward_bias(h["dy"], r, n)
        return s.hold((y, (r, n), "float32"), (dx, (r, n), "float32"), (dw, (n,), "float32"), (db, (n,), "float32"))
    if op == "adamw":
        n = c["n"]
        m = br.optimizer_update("ADAMW_UPDATE_M", [h["m"], h["g"]], n, **ADAMW)
        v = br.optimizer_update("ADAMW_UPDATE_V", [h["v"], h["g"]], n, **ADAMW)
        p = br.optimizer_update("ADAMW_UPDATE_PARAM", [h["p"], h["g"], m, v], n, **ADAMW)
        return s.hold((p, (n,), "float32"), (m, (n,), "float32"), (v, (n,), "float32"))
    n, ci, o, hw, k, st, out = c["n"], c["c"], c["o"], c["hw"], c["k"], c["stride"], _conv_out(c)
    geo = dict(n=n, c_in=ci, c_out=o, in_size=(hw, hw), out_size=(out, out), k=(k, k), stride=(st, st),
               pad=(c["pad"], c["pad"]), dilation=(1, 1))
    y = br.conv_ex("forward", h["x"], h["w"], h["b"], **geo)
    dx = br.conv_ex("backward_input", h["dy"], h["w"], **geo)
    dw = br.conv_ex("backward_weight", h["dy"], h["x"], **geo)
    db = br.conv_ex("backward_bias", h["dy"], **geo)
    return s.hold((y, (n, o, out, out), "float32"), (dx, (n, ci, hw, hw), "float32"), (dw, (o, ci, k, k), "float32"),
                  (db, (o,), "float32"))


# ---------------------------------------------------------------------------- what a pass cannot do without

def _pairs(c: Dict[str, Any]) -> int:
    return c["sq"] * (c["sq"] + 1) // 2 if c["causal"] else c["sq"] * c["sk"]


def work(c: Dict[str, Any]) -> Dict[str, float]:
    op = c["op"]
    if op == "mlp":
        b, i, h, o = c["batch"], c["din"], c["hidden"], c["dout"]
        return {"bytes": 4 * (b * i + h * i + h + o * h + o + b * o), "flops": 2 * b * (i * h + h * o)}
    if op == "fused":
        return {"bytes": 3 * ITEM[c["dtype"]] * c["rows"] * c["cols"] + 4 * c["rows"], "flops": 8 * c["rows"] * c["cols"]}
    if op == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": ITEM[c["dtype"]] * (m * k + n * k) + 4 * n + ITEM[c["out"]] * m * n
                + (4 * m * n if c["residual"] else 0), "flops": 2 * m * n * k}
    if op == "attention":
        return {"bytes": ITEM[c["dtype"]] * c["b"] * c["h"] * c["d"] * 2 * (c["sq"] + c["sk"]),
                "flops": 4 * c["b"] * c["h"] * c["d"] * _pairs(c)}
    if op == "block":
        e, t = c["heads"] * 64, c["b"] * c["s"]
        # x in and y out in float32, the weights once as the float16 the products read
        return {"bytes": 2 * 4 * t * e + 2 * 12 * e * e, "flops": 24 * t * e * e + 2 * c["b"] * e * c["s"] * (c["s"] + 1)}
    if op == "layernorm":
        return {"bytes": 4 * (4 * c["rows"] * c["cols"] + 4 * c["cols"]), "flops": 25 * c["rows"] * c["cols"]}
    if op == "adamw":
        return {"bytes": 28 * c["n"], "flops": 15 * c["n"]}
    out = _conv_out(c)
    x, y, w = c["n"] * c["c"] * c["hw"] ** 2, c["n"] * c["o"] * out ** 2, c["o"] * c["c"] * c["k"] ** 2
    return {"bytes": 4 * (2 * x + 2 * y + 2 * w + 2 * c["o"]), "flops": 3 * 2 * y * c["c"] * c["k"] ** 2}


def tolerance(c: Dict[str, Any]) -> Any:
    """About four times what the 64-bit result differs by (a sum of K 32-bit terms grows with K)."""
    op = c["op"]
    if op == "linear" and c["dtype"] != "float32":
        # the result's own rounding; sums and activation are 32-bit
        return {"rel": {"float16": 1e-3, "bfloat16": 8e-3, "float32": 1e-5}[c["out"]]}
    if op == "attention" and c["dtype"] != "float32":
        # probabilities and result are rounded to 16 bits
        return {"rel": 1.5e-3 if c["dtype"] == "float16" else 1e-2}
    if op == "block":
        return {"rel": 1e-3}  # float16 operands in every layer, a float32 residual stream
    # one 32-bit sum of up to 4096 terms or up to 200704 in slices (linear, conv), short or none otherwise
    return {"rel": 1e-5 if op in ("linear", "conv") else 2e-6}


def exact(c: Dict[str, Any], seed: int) -> Any:
    t = {k: v.double() for k, v in _tensors(c, seed).items()}
    op = c["op"]
    if op == "mlp":
        return torch.relu(t["x"] @ t["w1"].T + t["b1"]) @ t["w2"].T + t["b2"]
    if op == "fused":
        return (torch.relu(t["a"] * t["b"] + t["c"]) * torch.exp(-t["a"] * t["a"])).sum(-1)
    if op == "linear":
        y = t["a"] @ (t["b"].T if c["trans_b"] else t["b"]) + t["bias"]
        y = torch.relu(y) if c["act"] == "relu" else _gelu(y) if c["act"] == "gelu" else y
        return y + t["residual"] if c["residual"] else y
    if op == "attention":
        return _attention(t["q"], t["k"], t["v"], c["causal"])
    if op == "block":
        return _block(t, c["heads"])
    if op == "layernorm":
        mean, var = t["x"].mean(-1, keepdim=True), t["x"].var(-1, unbiased=False, keepdim=True)
        inv = torch.rsqrt(var + EPS)
        xh = (t["x"] - mean) * inv
        g = t["dy"] * t["w"]
        dx = inv * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
        return [xh * t["w"] + t["b"], dx, (t["dy"] * xh).sum(0), t["dy"].sum(0)]
    if op == "adamw":
        a = ADAMW
        m = a["beta1"] * t["m"] + (1 - a["beta1"]) * t["g"]
        v = a["beta2"] * t["v"] + (1 - a["beta2"]) * t["g"].square()
        mh, vh = m / (1 - a["beta1"] ** a["step"]), v / (1 - a["beta2"] ** a["step"])
        p = t["p"] - a["lr"] * mh / (vh.sqrt() + a["eps"]) - a["lr"] * a["weight_decay"] * t["p"]
        return [p, m, v]
    # A convolution as one product for each tap.
    st, out = c["stride"], _conv_out(c)
    span = (out - 1) * st + 1
    pad = torch.nn.functional.pad(t["x"], [c["pad"]] * 4)
    dpad = torch.zeros_like(pad)
    y = torch.zeros((c["n"], c["o"], out, out), dtype=torch.float64, device=pad.device)
    dw = torch.zeros_like(t["w"])
    dy2 = t["dy"].permute(1, 0, 2, 3).reshape(c["o"], -1)
    for kh in range(c["k"]):
        for kw in range(c["k"]):
            part = pad[:, :, kh:kh + span:st, kw:kw + span:st].permute(1, 0, 2, 3).reshape(c["c"], -1)
            tap = t["w"][:, :, kh, kw]
            y += (tap @ part).reshape(c["o"], c["n"], out, out).permute(1, 0, 2, 3)
            dw[:, :, kh, kw] = dy2 @ part.T
            dpad[:, :, kh:kh + span:st, kw:kw + span:st] += (tap.T @ dy2).reshape(c["c"], c["n"], out, out).permute(
                1, 0, 2, 3)
    p, hw = c["pad"], c["hw"]
    return [y + t["b"][None, :, None, None], dpad[:, :, p:p + hw, p:p + hw], dw, t["dy"].sum((0, 2, 3))]


def _gelu(x: torch.Tensor) -> torch.Tensor:
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: bool) -> torch.Tensor:
    out = torch.empty_like(q)
    for i in range(q.shape[0]):
        for j in range(q.shape[1]):
            s = (q[i, j] @ k[i, j].T) * q.shape[-1] ** -0.5
            if causal:
                s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
            out[i, j] = torch.softmax(s, -1) @ v[i, j]
    return out


def _block(t: Dict[str, torch.Tensor], heads: int) -> torch.Tensor:
    x = t["x"]
    b, s, e = x.shape

    def norm(h: torch.Tensor, n: str) -> torch.Tensor:
        return torch.nn.functional.layer_norm(h, (e,), t[n + "_w"], t[n + "_b"], EPS)

    def linear(h: torch.Tensor, n: str) -> torch.Tensor:
        return (h.reshape(b * s, -1) @ t["w_" + n].T + t["b_" + n]).reshape(b, s, -1)

    q, k, v = (z.reshape(b, s, heads, e // heads).permute(0, 2, 1, 3) for z in linear(norm(x, "ln1"), "qkv").split(e, -1))
    h = x + linear(_attention(q, k, v, True).permute(0, 2, 1, 3).reshape(b, s, e), "o")
    return h + linear(_gelu(linear(norm(h, "ln2"), "up")), "down")
