"""What the framework is timed on: calls of its public entry points over the
sizes, data types and options its users run.

``listed()`` names twelve cases, ``draw(rng)`` makes one more of the same
ranges. A case is a dict of plain values with a ``kind``:

- ``matmul``    ``matmul`` of bf16 or f32 operands, any transpose, optionally an f32 result or an activation
- ``linear``    a cached ``linear`` layer with bias and activation: prefill (many rows) and decode (few rows)
- ``prepacked`` ``matmul_prepacked_b`` of activations and a weight packed once
- ``backward``  the gradients of a linear layer: two ``matmul`` and a ``column_sum``
- ``splitk``    ``bmm`` of few tiles and a long contraction
- ``attention`` ``bmm``, ``softmax`` and ``bmm`` of one attention block
- ``rows``      ``softmax``, ``rms_norm`` and ``group_norm`` of one ``[m, n]`` tensor
- ``softmax``   ``softmax`` alone, of few long rows (a vocabulary)
- ``reduce``    ``row_sum``, ``column_sum``, ``row_dot``, ``matvec`` and ``relu`` of one ``[m, n]`` tensor
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "helion-mlir-xsmm_amd"))

import helion_mlir_utils as U  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
ACTIVATIONS = {"none": None, "relu": F.relu, "silu": F.silu, "gelu": F.gelu}


def listed() -> list[dict]:
    return [
        # The smallest call: an f32 product of 512 x 512, bound by its launches.
        {"name": "matmul_f32_512", "kind": "matmul", "dtype": "f32", "m": 512, "n": 512, "k": 512,
         "trans_a": False, "trans_b": False, "out": "f32", "act": "none"},
        # The square bf16 GEMM that the framework quotes.
        {"name": "matmul_bf16_4096", "kind": "matmul", "dtype": "bf16", "m": 4096, "n": 4096, "k": 4096,
         "trans_a": False, "trans_b": False, "out": "bf16", "act": "none"},
        # Extents that no tile divides, rows that keep no 16-byte alignment.
        {"name": "matmul_bf16_ragged", "kind": "matmul", "dtype": "bf16", "m": 1500, "n": 2001, "k": 1100,
         "trans_a": False, "trans_b": False, "out": "bf16", "act": "none"},
        # Prefill of a gated MLP's projection: the largest call.
        {"name": "linear_prefill_8192", "kind": "linear", "dtype": "bf16", "rows": 8192, "n": 11008, "k": 4096,
         "act": "silu"},
        # Decode through the same layer: 32 sequences, one token each.
        {"name": "linear_decode_32", "kind": "linear", "dtype": "bf16", "rows": 32, "n": 11008, "k": 4096,
         "act": "silu"},
        # The layer with its weight packed once, a ragged batch of 100 rows.
        {"name": "prepacked_100", "kind": "prepacked", "rows": 100, "n": 11008, "k": 4096, "layout": "vnni_panels",
         "panel": 64, "act": "none"},
        # Backward of a 4096 x 4096 layer over 3000 tokens.
        {"name": "backward_3000", "kind": "backward", "dtype": "bf16", "rows": 3000, "n": 4096, "k": 4096},
        # Sixteen 256 x 256 products contracted over 65536.
        {"name": "splitk_bmm_f32", "kind": "splitk", "dtype": "f32", "batch": 16, "m": 256, "n": 256, "k": 65536},
        # One attention block: 48 heads of 500 tokens, 64 channels.
        {"name": "attention_500", "kind": "attention", "batch": 48, "seq_q": 500, "seq_k": 500, "d": 64},
        # The normalizations of 32768 tokens of 4096 channels.
        {"name": "rows_bf16_32768", "kind": "rows", "dtype": "bf16", "m": 32768, "n": 4096, "groups": 32},
        # Probabilities over a large vocabulary for a batch of tokens.
        {"name": "softmax_f32_vocab", "kind": "softmax", "dtype": "f32", "m": 512, "n": 50001},
        # Reductions and an activation of one layer's output.
        {"name": "reduce_bf16_4096", "kind": "reduce", "dtype": "bf16", "m": 4096, "n": 4096},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    """An integer of [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _extent(rng: random.Random, lo: int, hi: int) -> int:
    """An extent of [lo, hi]: as often a multiple of 64 (where one fits), a
    multiple of 8 or any integer."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 8, 1))
    return v if v < step else v // step * step


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("matmul", "matmul", "linear", "linear", "prepacked", "backward", "splitk", "attention",
                       "rows", "rows", "softmax", "reduce"))
    if kind == "matmul":
        dtype = rng.choice(("bf16", "bf16", "f32"))
        return {"kind": kind, "dtype": dtype, "m": _extent(rng, 64, 4096), "n": _extent(rng, 64, 4096),
                "k": _extent(rng, 64, 4096), "trans_a": rng.random() < 0.25, "trans_b": rng.random() < 0.5,
                "out": rng.choice((dtype, dtype, "f32")), "act": rng.choice(("none", "none", "relu", "silu", "gelu"))}
    if kind == "linear":
        rows = _log(rng, 1, 64) if rng.random() < 0.5 else _log(rng, 65, 8192)
        return {"kind": kind, "dtype": rng.choice(("bf16", "bf16", "bf16", "f32")) if rows <= 1024 else "bf16",
                "rows": rows, "n": _extent(rng, 512, 11008), "k": _extent(rng, 512, 4096),
                "act": rng.choice(("none", "relu", "silu", "gelu"))}
    if kind == "prepacked":
        layout = rng.choice(("vnni_panels", "vnni_panels", "blocked", "blocked_vnni", "panels"))
        panel = rng.choice((32, 64, 128, 256)) if layout in ("vnni_panels", "panels") else 32
        return {"kind": kind, "rows": _log(rng, 1, 2048), "n": _log(rng, 512, 11008) // 256 * 256,
                "k": _log(rng, 512, 4096) // 32 * 32, "layout": layout, "panel": panel,
                "act": rng.choice(("none", "relu", "silu"))}
    if kind == "backward":
        return {"kind": kind, "dtype": "bf16", "rows": _extent(rng, 64, 4096), "n": _extent(rng, 256, 4096),
                "k": _extent(rng, 256, 4096)}
    if kind == "splitk":
        dtype = rng.choice(("f32", "bf16"))
        batch = _log(rng, 1, 16)
        return {"kind": kind, "dtype": dtype, "batch": batch, "m": _extent(rng, 32, 256), "n": _extent(rng, 32, 256),
                "k": _extent(rng, 2048, 65536)}
    if kind == "attention":
        seq = _extent(rng, 32, 1024)
        return {"kind": kind, "batch": _log(rng, 1, 64), "seq_q": seq,
                "seq_k": seq if rng.random() < 0.7 else _extent(rng, 32, 1024), "d": rng.choice((64, 80, 96, 128))}
    if kind == "rows":
        dtype = rng.choice(("bf16", "f32"))
        n = _extent(rng, 64, 16384)
        groups = rng.choice([g for g in (1, 1, 8, 32) if n % g == 0])
        return {"kind": kind, "dtype": dtype, "m": _log(rng, 16, max(16, min(65536, (1 << 26) // n))), "n": n,
                "groups": groups}
    if kind == "softmax":
        n = _extent(rng, 8192, 131072)
        return {"kind": kind, "dtype": rng.choice(("bf16", "f32")), "m": _log(rng, 1, (1 << 26) // n), "n": n}
    n = _extent(rng, 64, 32768)
    return {"kind": "reduce", "dtype": rng.choice(("bf16", "f32")), "m": _log(rng, 16, min(65536, (1 << 26) // n)),
            "n": n}


# -- inputs ------------------------------------------------------------------
# Values have the distributions the entry points meet: U[-1, 1] operands of
# plain products, unit-normal activations, weights and gradients of the scale
# that keeps a layer's output near one, norm inputs of standard deviation 2.


class _Inputs:
    def __init__(self, seed: int) -> None:
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(self, *shape: int, dtype: str) -> torch.Tensor:
        t = torch.rand(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return t.mul_(2.0).sub_(1.0).to(DTYPES[dtype])

    def normal(self, *shape: int, std: float = 1.0, dtype: str) -> torch.Tensor:
        t = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return t.mul_(std).to(DTYPES[dtype])


def _tensors(case: dict, seed: int) -> dict:
    """The case's plain input tensors, from the seed alone."""
    make, kind = _Inputs(seed), case["kind"]
    if kind == "matmul":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        return {"a": make.uniform(*((k, m) if case["trans_a"] else (m, k)), dtype=dt),
                "b": make.uniform(*((n, k) if case["trans_b"] else (k, n)), dtype=dt)}
    if kind in ("linear", "prepacked"):
        n, k, dt = case["n"], case["k"], case.get("dtype", "bf16")
        std = 1.28 / math.sqrt(k)
        return {"x": make.normal(case["rows"], k, dtype=dt), "w": make.normal(n, k, std=std, dtype=dt),
                "b": make.normal(n, std=0.02, dtype=dt)}
    if kind == "backward":
        r, n, k, dt = case["rows"], case["n"], case["k"], case["dtype"]
        return {"x": make.normal(r, k, dtype=dt), "w": make.normal(n, k, std=1.28 / math.sqrt(k), dtype=dt),
                "dy": make.normal(r, n, std=0.1, dtype=dt)}
    if kind == "splitk":
        s, m, n, k, dt = case["batch"], case["m"], case["n"], case["k"], case["dtype"]
        return {"a": make.uniform(s, m, k, dtype=dt), "b": make.uniform(s, k, n, dtype=dt)}
    if kind == "attention":
        s, q, k, d = case["batch"], case["seq_q"], case["seq_k"], case["d"]
        return {"q": make.normal(s, q, d, std=1.0 / math.sqrt(d), dtype="bf16"),
                "k": make.normal(s, k, d, dtype="bf16"), "v": make.normal(s, k, d, dtype="bf16")}
    m, n, dt = case["m"], case["n"], case["dtype"]
    t = {"x": make.normal(m, n, std=2.0, dtype=dt)}
    if kind == "rows":
        t["weight"] = make.uniform(n, dtype="f32").mul_(0.5).add_(1.0).to(DTYPES[dt])
        t["scale"] = make.uniform(n, dtype="f32").mul_(0.5).add_(1.0)
        t["shift"] = make.normal(n, std=0.1, dtype="f32")
    if kind == "reduce":
        t["v"] = make.uniform(n, dtype="f32")
        t["col"] = make.uniform(n, 1, dtype=dt)
    return t


def prepare(case: dict, seed: int) -> dict:
    state = {"case": case, **_tensors(case, seed)}
    if case["kind"] == "linear":
        layer = torch.nn.utils.skip_init(torch.nn.Linear, case["k"], case["n"], device="cuda",
                                         dtype=DTYPES[case["dtype"]])
        with torch.no_grad():
            layer.weight.copy_(state.pop("w"))
            layer.bias.copy_(state.pop("b"))
        state["layer"], state["cache"] = layer, None
    elif case["kind"] == "prepacked":
        w, layout = state.pop("w"), case["layout"]
        if layout == "vnni_panels":
            state["packed"] = U.pack_b_vnni_t(w, case["panel"])
        elif layout == "panels":
            state["packed"] = U.pack_b_panels(w.t().contiguous(), case["panel"])
        elif layout == "blocked":
            state["packed"] = U.pack_b_blocked_t(w)
        else:
            state["packed"] = U.pack_b_blocked_vnni_t(w)
    return state


def _epilogue(case: dict) -> dict:
    act = ACTIVATIONS[case["act"]]
    return {} if act is None else {"epilogue": act}


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "matmul":
        return U.matmul(state["a"], state["b"], trans_a=case["trans_a"], trans_b=case["trans_b"],
                        out_dtype=DTYPES[case["out"]], **_epilogue(case))
    if kind == "linear":
        y, state["cache"] = U.linear(state["x"], state["layer"], cache=state["cache"], **_epilogue(case))
        return y
    if kind == "prepacked":
        return U.matmul_prepacked_b(state["x"], state["packed"], case["n"], state["b"], **_epilogue(case))
    if kind == "backward":
        return {"dx": U.matmul(state["dy"], state["w"]), "dw": U.matmul(state["dy"], state["x"], trans_a=True),
                "db": U.column_sum(state["dy"])}
    if kind == "splitk":
        return U.bmm(state["a"], state["b"])
    if kind == "attention":
        q, k, v = state["q"], state["k"], state["v"]
        s, rows, keys = case["batch"], case["seq_q"], case["seq_k"]
        p = U.softmax(U.bmm(q, k.transpose(1, 2)).view(s * rows, keys)).view(s, rows, keys)
        return {"p": p, "out": U.bmm(p, v)}
    if kind == "softmax":
        return U.softmax(state["x"])
    x = state["x"]
    if kind == "rows":
        return {"softmax": U.softmax(x), "rms_norm": U.rms_norm(x, state["weight"]),
                "group_norm": U.group_norm(x, case["groups"], state["scale"], state["shift"], 1e-5)}
    return {"row_sum": U.row_sum(x), "column_sum": U.column_sum(x), "row_dot": U.row_dot(x, state["v"]),
            "matvec": U.matvec(x, state["col"]), "relu": U.relu(x)}


# -- what a pass cannot do without -----------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    size = {"bf16": 2, "f32": 4}
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m + n) * k * size[case["dtype"]] + m * n * size[case["out"]], "flops": 2 * m * n * k}
    if kind in ("linear", "prepacked"):
        r, n, k, e = case["rows"], case["n"], case["k"], size[case.get("dtype", "bf16")]
        return {"bytes": (r * k + n * k + n + r * n) * e, "flops": 2 * r * n * k}
    if kind == "backward":
        r, n, k, e = case["rows"], case["n"], case["k"], size[case["dtype"]]
        # dx reads dy and w, dw reads dy and x, db reads dy.
        return {"bytes": (3 * r * n + 2 * n * k + 2 * r * k) * e + 4 * n, "flops": 4 * r * n * k}
    if kind == "splitk":
        s, m, n, k, e = case["batch"], case["m"], case["n"], case["k"], size[case["dtype"]]
        return {"bytes": s * ((m + n) * k + m * n) * e, "flops": 2 * s * m * n * k}
    if kind == "attention":
        s, q, k, d = case["batch"], case["seq_q"], case["seq_k"], case["d"]
        # Three calls: scores written and read, probabilities written and read.
        return {"bytes": s * (2 * q * d + 2 * k * d + 4 * q * k) * 2, "flops": 4 * s * q * k * d}
    m, n, e = case["m"], case["n"], size[case["dtype"]]
    if kind == "rows":
        return {"bytes": 6 * m * n * e + n * (e + 8), "flops": 20 * m * n}
    if kind == "softmax":
        return {"bytes": 2 * m * n * e, "flops": 5 * m * n}
    # Five calls, each reading x.
    return {"bytes": 6 * m * n * e + 3 * m * e + n * (8 + e), "flops": 7 * m * n}


def tolerance(case: dict):
    """Four times the error against 64 bits that the kernels show: one
    rounding to bf16 of each output (1.7e-3), the two more roundings inside
    an attention block, and 32-bit sums."""
    kind = case["kind"]
    if kind == "attention":
        return {"rel": 1.6e-2}
    if kind in ("linear", "prepacked", "backward"):
        return {"rel": 7e-3 if case.get("dtype", "bf16") == "bf16" else 1e-5}
    if kind == "matmul":
        return {"rel": 7e-3 if case["out"] == "bf16" else 1e-5}
    return {"rel": 7e-3 if case["dtype"] == "bf16" else 1e-5}


# -- the same in 64 bits ------------------------------------------------------------


def _act64(case: dict, y: torch.Tensor) -> torch.Tensor:
    act = ACTIVATIONS[case["act"]]
    return y if act is None else act(y)


def exact(case: dict, seed: int):
    t = {name: v.double() for name, v in _tensors(case, seed).items()}
    kind = case["kind"]
    if kind == "matmul":
        a = t["a"].t() if case["trans_a"] else t["a"]
        b = t["b"].t() if case["trans_b"] else t["b"]
        return _act64(case, a @ b)
    if kind in ("linear", "prepacked"):
        return _act64(case, t["x"] @ t["w"].t() + t["b"])
    if kind == "backward":
        return {"dx": t["dy"] @ t["w"], "dw": t["dy"].t() @ t["x"], "db": t["dy"].sum(0)}
    if kind == "splitk":
        return torch.stack([a @ b for a, b in zip(t["a"], t["b"])])
    if kind == "attention":
        p, out = [], []
        for q, k, v in zip(t["q"], t["k"], t["v"]):
            p.append(torch.softmax(q @ k.t(), -1))
            out.append(p[-1] @ v)
        return {"p": torch.stack(p), "out": torch.stack(out)}
    x = t["x"]
    if kind == "softmax":
        return torch.softmax(x, -1)
    if kind == "rows":
        rms = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * t["weight"]
        return {"softmax": torch.softmax(x, -1), "rms_norm": rms,
                "group_norm": F.group_norm(x, case["groups"], t["scale"], t["shift"], 1e-5)}
    return {"row_sum": x.sum(1, keepdim=True), "column_sum": x.sum(0), "row_dot": x @ t["v"][:, None],
            "matvec": x @ t["col"], "relu": torch.relu(x)}
