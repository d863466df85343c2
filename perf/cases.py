# SPDX-License-Identifier: BSD-3-Clause
"""The calls whose speed this backend is judged by, with inputs, required
work, float64 results and tolerances.

Every case is a graph built with the operator DSL, compiled by the HIP backend
under its default schedule (what a user who tunes nothing gets) into a payload
that queues its kernels and returns, as bench.py compiles it: a program that
runs payloads back to back waits once at the end.  Operands live in HBM.

Kinds of case:
  matmul      one matmul node: fp32, bf16 (fp32 result) or fp64; B may be
              stored transposed (tensor layout [1, 0])
  mlp         matmul -> relu -> matmul
  conv        pad2d -> conv2d (-> bias_add) (-> relu), NHWC x RSCF
  pad_matmul  pad -> matmul -> unpad, the graphs of tests/test_padding_graphs.py
"""

from __future__ import annotations

import ctypes
from typing import Any

import torch

import xtc_amd.graphs.xtc.op as O
from xtc_amd.backends.hip import Backend
from xtc_amd.runtimes.hip.device import HipDevice

_TORCH = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float64": torch.float64}
_BYTES = {"float32": 4, "bfloat16": 2, "float64": 8}


def _matmul(name: str, dtype: str, m: int, n: int, k: int, trans_b: bool = False) -> dict[str, Any]:
    return {"name": name, "kind": "matmul", "dtype": dtype, "m": m, "n": n, "k": k, "trans_b": trans_b}


def _conv(name: str, dtype: str, nb: int, h: int, w: int, c: int, f: int, r: int, stride: int, bias: bool,
          relu: bool) -> dict[str, Any]:
    return {"name": name, "kind": "conv", "dtype": dtype, "nb": nb, "h": h, "w": w, "c": c, "f": f, "r": r,
            "stride": stride, "pad": r // 2, "bias": bias, "relu": relu}


def listed() -> list[dict[str, Any]]:
    return [
        # the plumbing workload C1 and the default size of the explorer: launch-bound
        _matmul("matmul_f32_512", "float32", 512, 512, 512),
        # a user's own sizes, no multiple of anything: no row is 16-byte aligned
        _matmul("matmul_f32_odd", "float32", 509, 1021, 777),
        # the headline workload C3a: the largest call
        _matmul("matmul_bf16_8192", "bfloat16", 8192, 8192, 8192),
        # C3b: one decode step of 16 sequences through a square projection, streams the weights
        _matmul("matmul_bf16_decode", "bfloat16", 16, 8192, 8192),
        # Gemma27B_QKV of the named layers: the projection of a 256-token prefill
        _matmul("matmul_bf16_prefill", "bfloat16", 256, 8192, 4608),
        # Gemma27B_QK with its weights stored [out][in], as most checkpoints keep them
        _matmul("matmul_bf16_bt", "bfloat16", 256, 4608, 8192, True),
        # double precision: scientific codes and float64 graphs
        _matmul("matmul_f64_1024", "float64", 1024, 1024, 1024),
        # C5: two-layer MLP in fp32, relu between
        {"name": "mlp_f32", "kind": "mlp", "dtype": "float32", "m": 2048, "k": 1024, "h": 4096, "n": 1024},
        # C4: the middle of a ResNet, batch 8
        _conv("conv_f32_56x56", "float32", 8, 56, 56, 64, 64, 3, 1, False, True),
        # the stem of a ResNet: 3 channels, 7x7 stride 2, bias and relu
        _conv("conv_f32_stem", "float32", 4, 224, 224, 3, 64, 7, 2, True, True),
        # Yolo9000_08 in bf16: inference of a detector, batch 1
        _conv("conv_bf16_68x68", "bfloat16", 1, 68, 68, 128, 256, 3, 1, False, False),
        # the padding graphs: odd operands brought to whole vectors by pad, the result cropped back
        {"name": "pad_matmul_f32", "kind": "pad_matmul", "dtype": "float32", "m": 1000, "n": 1100, "k": 1196, "pad": 2},
    ]


def _log(rng: Any, lo: int, hi: int) -> int:
    return int(round(lo * (hi / lo) ** rng.random()))


def _up(x: int, step: int) -> int:
    return max(step, (x + step // 2) // step * step)


def draw(rng: Any) -> dict[str, Any]:
    while True:
        case = _draw(rng)
        cost = work(case)["flops"]
        odd = case["kind"] == "matmul" and case["dtype"] == "float32" and (case["k"] % 4 or case["n"] % 4)
        top = 1e9 if odd else {"float32": 4e10, "bfloat16": 4e11, "float64": 1e10}[case["dtype"]]
        if 1e6 <= cost <= top:
            del case["name"]
            return case


def _draw(rng: Any) -> dict[str, Any]:
    kind = rng.choice(("f32", "f32", "odd", "bf16", "bf16", "decode", "bt", "f64", "mlp", "conv_f32", "conv_f32",
                       "conv_bf16", "pad_matmul"))
    if kind == "f32":
        # whole vectors of 4, from every class of row count
        step = rng.choice((4, 16, 128))
        return _matmul("", "float32", _log(rng, 32, 4096), _up(_log(rng, 64, 8192), step), _up(_log(rng, 64, 8192), step))
    if kind == "odd":
        return _matmul("", "float32", _log(rng, 17, 1500), _log(rng, 17, 1500), _log(rng, 17, 1500))
    if kind == "bf16":
        step = rng.choice((8, 64, 256))
        return _matmul("", "bfloat16", _up(_log(rng, 32, 8192), rng.choice((1, 128))), _up(_log(rng, 128, 8192), step),
                       _up(_log(rng, 128, 8192), step))
    if kind == "decode":
        return _matmul("", "bfloat16", rng.randint(1, 16), _up(_log(rng, 1024, 8192), 128), _up(_log(rng, 1024, 8192), 512))
    if kind == "bt":
        return _matmul("", "bfloat16", _up(_log(rng, 64, 2048), rng.choice((1, 128))), _up(_log(rng, 256, 8192), 64),
                       _up(_log(rng, 256, 8192), 64), True)
    if kind == "f64":
        return _matmul("", "float64", _log(rng, 64, 2048), _up(_log(rng, 64, 2048), 2), _up(_log(rng, 64, 2048), 2))
    if kind == "mlp":
        return {"name": "", "kind": "mlp", "dtype": "float32", "m": _up(_log(rng, 128, 2048), 32),
                "k": _up(_log(rng, 256, 2048), 64), "h": _up(_log(rng, 512, 4096), 64), "n": _up(_log(rng, 256, 2048), 64)}
    if kind == "pad_matmul":
        p = rng.choice((1, 2, 3))
        q = 2 * p  # pads on both sides: the padded sizes are whole vectors
        return {"name": "", "kind": "pad_matmul", "dtype": "float32", "m": _log(rng, 100, 1500),
                "n": _up(_log(rng, 100, 1500), 4) + 8 - q, "k": _up(_log(rng, 100, 1500), 4) + 8 - q, "pad": p}
    dtype = "bfloat16" if kind == "conv_bf16" else "float32"
    size = _log(rng, 7, 112)
    c = rng.choice((3, 16, 32, 48, 64, 96, 128, 192, 256, 384, 512))
    f = rng.choice((16, 32, 48, 64, 96, 128, 192, 256, 384, 512))
    r = rng.choice((1, 3, 3, 3, 5, 7)) if c < 128 else rng.choice((1, 3, 3))
    return _conv("", dtype, rng.choice((1, 1, 2, 4, 8)), size, size + rng.choice((0, 0, 1, 3)), c, f, r,
                 rng.choice((1, 1, 2)), rng.random() < 0.3, rng.random() < 0.7)


def _conv_out(case: dict[str, Any]) -> tuple[int, int]:
    p, r, s = case["pad"], case["r"], case["stride"]
    return (case["h"] + 2 * p - r) // s + 1, (case["w"] + 2 * p - r) // s + 1


def _graph(case: dict[str, Any]) -> Any:
    kind, dt = case["kind"], case["dtype"]
    out = {"out_dtype": "float32"} if dt == "bfloat16" else {}
    if kind == "matmul":
        a = O.tensor((case["m"], case["k"]), dt, name="A")
        layout = {"layout": [1, 0]} if case["trans_b"] else {}
        b = O.tensor((case["k"], case["n"]), dt, name="B", **layout)
        with O.graph(name="matmul") as gb:
            O.matmul(a, b, name="C", **out)
    elif kind == "mlp":
        x = O.tensor((case["m"], case["k"]), dt, name="X")
        w1 = O.tensor((case["k"], case["h"]), dt, name="W1")
        w2 = O.tensor((case["h"], case["n"]), dt, name="W2")
        with O.graph(name="mlp") as gb:
            O.matmul(O.relu(O.matmul(x, w1, name="fc1"), name="act"), w2, name="fc2")
    elif kind == "pad_matmul":
        a = O.tensor((case["m"], case["k"]), dt, name="A")
        b = O.tensor((case["k"], case["n"]), dt, name="B")
        with O.graph(name="pad_matmul_unpad") as gb:
            pa = O.pad(a, padding=case["pad"], name="A_pad")
            pb = O.pad(b, padding=case["pad"], name="B_pad")
            O.unpad(O.matmul(pa, pb, name="matmul_padded"), padding=case["pad"], name="C")
    else:
        x = O.tensor((case["nb"], case["h"], case["w"], case["c"]), dt, name="I")
        w = O.tensor((case["r"], case["r"], case["c"], case["f"]), dt, name="W")
        bias = O.tensor((case["f"],), "float32", name="bias") if case["bias"] else None
        with O.graph(name="conv") as gb:
            t = O.pad2d(x, padding=case["pad"], axes=(1, 2), name="pad") if case["pad"] else x
            t = O.conv2d(t, w, stride=(case["stride"], case["stride"]), name="conv", **out)
            if bias is not None:
                t = O.bias_add(t, bias, name="add")
            if case["relu"]:
                O.relu(t, name="relu")
    return gb.graph


def _inputs(case: dict[str, Any], seed: int) -> list[torch.Tensor]:
    """The graph's inputs in HBM: uniform [-1, 1) operands; MLP weights normal
    with deviation 0.02; conv images uniform [0, 1) (what a relu or an image
    decoder leaves) with He-initialised weights."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dt = _TORCH[case["dtype"]]

    def uniform(*shape: int, lo: float = -1.0) -> torch.Tensor:
        base = torch.float64 if dt == torch.float64 else torch.float32
        return torch.empty(shape, device="cuda", dtype=base).uniform_(lo, 1.0, generator=gen).to(dt)

    def normal(std: float, *shape: int, dtype: torch.dtype = dt) -> torch.Tensor:
        return torch.empty(shape, device="cuda", dtype=torch.float32).normal_(0.0, std, generator=gen).to(dtype)

    if case["kind"] == "matmul":
        b = (case["n"], case["k"]) if case["trans_b"] else (case["k"], case["n"])
        return [uniform(case["m"], case["k"]), uniform(*b)]
    if case["kind"] == "pad_matmul":
        return [uniform(case["m"], case["k"]), uniform(case["k"], case["n"])]
    if case["kind"] == "mlp":
        return [uniform(case["m"], case["k"]), normal(0.02, case["k"], case["h"]), normal(0.02, case["h"], case["n"])]
    taps = case["r"] * case["r"] * case["c"]
    ins = [uniform(case["nb"], case["h"], case["w"], case["c"], lo=0.0),
           normal((2.0 / taps) ** 0.5, case["r"], case["r"], case["c"], case["f"])]
    if case["bias"]:
        ins.append(normal(0.1, case["f"], dtype=torch.float32))
    return ins


def _out_shape(case: dict[str, Any]) -> tuple[int, ...]:
    if case["kind"] == "conv":
        return (case["nb"], *_conv_out(case), case["f"])
    return (case["m"], case["n"])


def prepare(case: dict[str, Any], seed: int) -> dict[str, Any]:
    backend = Backend(_graph(case))
    module = backend.get_compiler(synchronize=False, schedule_policy="strict").compile(backend.get_scheduler().schedule())
    device = HipDevice()
    device.init_device()
    device.load_module(module)
    call = device.get_module_function(module, module.payload_name)
    call.restype = None
    ins = _inputs(case, seed)
    out = torch.empty(_out_shape(case), device="cuda", dtype=torch.float64 if case["dtype"] == "float64" else torch.float32)
    args = [ctypes.c_void_p(t.data_ptr()) for t in (*ins, out)]
    return {"module": module, "call": call, "args": args, "ins": ins, "out": out}


def run(state: dict[str, Any]) -> torch.Tensor:
    state["call"](*state["args"])
    return state["out"]


def exact(case: dict[str, Any], seed: int) -> torch.Tensor:
    ins = [t.double() for t in _inputs(case, seed)]
    if case["kind"] == "matmul":
        return ins[0] @ (ins[1].t().contiguous() if case["trans_b"] else ins[1])
    if case["kind"] == "pad_matmul":
        # the padded border of k adds zero products and the cropped border of m and n is dropped
        return ins[0] @ ins[1]
    if case["kind"] == "mlp":
        return (ins[0] @ ins[1]).relu() @ ins[2]
    p, r, s = case["pad"], case["r"], case["stride"]
    oh, ow = _conv_out(case)
    x = torch.nn.functional.pad(ins[0], (0, 0, p, p, p, p))
    out = torch.zeros(case["nb"] * oh * ow, case["f"], device="cuda", dtype=torch.float64)
    for i in range(r):
        for j in range(r):
            tap = x[:, i : i + (oh - 1) * s + 1 : s, j : j + (ow - 1) * s + 1 : s, :]
            out += tap.reshape(-1, case["c"]).contiguous() @ ins[1][i, j]
    out = out.reshape(case["nb"], oh, ow, case["f"])
    if case["bias"]:
        out = out + ins[2]
    return out.relu() if case["relu"] else out


def work(case: dict[str, Any]) -> dict[str, float]:
    size = _BYTES[case["dtype"]]
    out = 8 if case["dtype"] == "float64" else 4
    if case["kind"] in ("matmul", "pad_matmul"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": float((m * k + k * n) * size + m * n * out), "flops": 2.0 * m * n * k}
    if case["kind"] == "mlp":
        m, k, h, n = case["m"], case["k"], case["h"], case["n"]
        return {"bytes": float((m * k + k * h + h * n + m * n) * size), "flops": 2.0 * m * h * (k + n)}
    oh, ow = _conv_out(case)
    taps = case["r"] * case["r"] * case["c"]
    read = case["nb"] * case["h"] * case["w"] * case["c"] + taps * case["f"]
    pixels = case["nb"] * oh * ow
    return {"bytes": float(read * size + pixels * case["f"] * out), "flops": 2.0 * pixels * case["f"] * taps}


def tolerance(case: dict[str, Any]) -> Any:
    """Sums of fp32 products (bf16 products are exact in fp32) in another
    order; fp64 likewise at its own precision.  About four times the error
    against float64 at the longest sums drawn (K = 8192, fp32: 1.6e-6 in the
    norm, 1.5e-5 of the root mean square at the worst element; the fp64 case:
    1.2e-15)."""
    if case["dtype"] == "float64":
        return {"rel": 1e-14, "max": 1e-13}
    return {"rel": 6e-6, "max": 8e-5}
