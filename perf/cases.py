"""What this framework is timed on: its public entry points over the sizes that programs call them with.

Five kinds of pass:

* "linear":  `feather_ops(out_dtype).Linear.forward` on a layer loaded from an e5m2 checkpoint: what a model runs for
             every quantized layer (any row count, fp16 or bf16 activations, with or without a bias);
* "mm":      `scaled_mm_hip_any_m`, the GEMM entry itself, for programs that call it directly (e5m2 or e4m3fn weights);
* "lora":    `Linear.forward` with unmerged LoRA patches attached to the layer;
* "load":    `make_feather_quantized_weight` on a checkpoint weight (fp16, bf16, fp32, or e5m2 to be laid out);
* "merge":   `Linear.convert_weight` and `Linear.set_weight`: the weight back in 16 bits, and a patched one quantized.

Rows M are tokens: 1 or 2 for a conditioning vector, tens to hundreds for text, thousands for image and video latents.
N and K are layer widths; K is a multiple of 16 (most are multiples of 64), N of 16.
"""

import importlib
import importlib.util
import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

_PKG = "featherops_amd"
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32,
           "e5m2": torch.float8_e5m2, "e4m3": torch.float8_e4m3fn}


def _module(name):
    """A module of the plugin package (its folder's name is not a Python identifier)."""
    if _PKG not in sys.modules:
        folder = Path(__file__).resolve().parents[1] / "comfyui-featherops_amd"
        spec = importlib.util.spec_from_file_location(_PKG, folder / "__init__.py",
                                                      submodule_search_locations=[str(folder)])
        package = importlib.util.module_from_spec(spec)
        sys.modules[_PKG] = package
        spec.loader.exec_module(package)
    return importlib.import_module(f"{_PKG}.{name}")


def listed():
    return [
        # one conditioning vector through a modulation layer: the smallest call, latency and launches count
        {"name": "linear_vector", "kind": "linear", "M": 1, "N": 12288, "K": 3072, "x": "bf16", "out": "bf16",
         "bias": True},
        # a few rows against a square weight: the weight stream
        {"name": "mm_few_rows", "kind": "mm", "M": 16, "N": 4096, "K": 4096, "x": "fp16", "w": "e5m2", "out": "fp16",
         "bias": True},
        # one text prompt through a wide text-encoder layer
        {"name": "linear_prompt", "kind": "linear", "M": 154, "N": 10240, "K": 4096, "x": "bf16", "out": "bf16",
         "bias": False},
        # the text stream of a joint transformer block: the down projection
        {"name": "linear_text", "kind": "linear", "M": 512, "N": 3072, "K": 12288, "x": "bf16", "out": "bf16",
         "bias": True},
        # a small latent image, e4m3fn weights, no bias
        {"name": "mm_small_image_e4m3", "kind": "mm", "M": 1024, "N": 3072, "K": 3072, "x": "fp16", "w": "e4m3",
         "out": "fp16", "bias": False},
        # sizes that are multiples of 16 and of no tile, an odd row count
        {"name": "mm_ragged", "kind": "mm", "M": 1003, "N": 2320, "K": 3216, "x": "fp16", "w": "e5m2", "out": "fp16",
         "bias": True},
        # an image's tokens through the up projection
        {"name": "linear_image", "kind": "linear", "M": 4096, "N": 12288, "K": 3072, "x": "bf16", "out": "bf16",
         "bias": True},
        # a video's tokens: the largest call
        {"name": "mm_video", "kind": "mm", "M": 32768, "N": 13824, "K": 5120, "x": "fp16", "w": "e5m2", "out": "fp16",
         "bias": True},
        # a prompt's tokens (an odd number) through a layer with two LoRA patches
        {"name": "lora_text", "kind": "lora", "M": 333, "N": 3072, "K": 3072, "x": "bf16", "out": "bf16", "bias": True,
         "rank": 16, "patches": 2},
        # an image's and a prompt's tokens together, one patch of the usual large rank
        {"name": "lora_image", "kind": "lora", "M": 4608, "N": 3072, "K": 3072, "x": "bf16", "out": "bf16",
         "bias": True, "rank": 64, "patches": 1},
        # loading a 16-bit checkpoint: one wide weight of a video model
        {"name": "load_bf16", "kind": "load", "N": 13824, "K": 5120, "w": "bf16"},
        # merging a patch into a square weight: back to 16 bits, and quantized again
        {"name": "merge_fp16", "kind": "merge", "N": 5120, "K": 5120, "w": "fp16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64, sometimes only of 16."""
    step = 16 if rng.random() < 0.25 else 64
    return max(step, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mm", "mm", "lora", "lora", "load", "merge"])
    if kind == "load":
        return {"kind": kind, "N": _width(rng, 1024, 13824), "K": _width(rng, 1024, 5120),
                "w": rng.choice(["fp16", "bf16", "fp32", "e5m2"])}
    if kind == "merge":
        return {"kind": kind, "N": _width(rng, 1024, 13824), "K": _width(rng, 1024, 5120),
                "w": rng.choice(["fp16", "bf16"])}
    # the weight holds at least a million elements and at most the largest listed one's 71 million
    N, K = _width(rng, 1024, 13824), _width(rng, 1024, 12288)
    while N * K > 13824 * 5120:
        N, K = _width(rng, 1024, 13824), _width(rng, 1024, 12288)
    case = {"kind": kind, "M": _log_int(rng, 1, 8192), "N": N, "K": K}
    if kind == "mm":
        case.update(x=rng.choice(["fp16", "bf16"]), w=rng.choice(["e5m2", "e5m2", "e4m3"]))
    else:
        case.update(x=rng.choice(["bf16", "bf16", "fp16"]))
    case.update(out=rng.choice(["bf16", "fp16"]) if kind == "mm" else case["x"], bias=rng.random() < 0.7)
    if kind == "lora":
        case.update(rank=rng.choice([8, 16, 32, 64, 128]), patches=rng.choice([1, 1, 2]))
    return case


def _inputs(case, seed):
    """Plain tensors on the GPU, from the seed alone: unit-variance activations (a layer's input after a norm), weights
    and factors of a trained layer's size."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)

    def normal(*shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=gen, device=dev) * std).to(dtype)

    N, K = case["N"], case["K"]
    t = {}
    w = normal(N, K, std=K ** -0.5)
    if case["kind"] == "load" and case["w"] != "e5m2":
        t["w"] = w.to(_DTYPES[case["w"]])
        return t
    fp8 = torch.float8_e4m3fn if case.get("w") == "e4m3" else torch.float8_e5m2
    t["scale"] = w.abs().amax() / torch.finfo(fp8).max
    t["codes"] = (w / t["scale"]).to(fp8)
    if case["kind"] == "load":
        return t
    if case["kind"] == "merge":
        t["patched"] = (w + normal(N, K, std=0.1 * K ** -0.5)).to(_DTYPES[case["w"]])
        return t
    t["x"] = normal(case["M"], K, dtype=_DTYPES[case["x"]])
    t["bias"] = normal(N, std=0.1, dtype=_DTYPES[case["out"]]) if case["bias"] else None
    if case["kind"] == "lora":
        R = case["rank"]
        t["patches"] = [(0.8 + 0.1 * i, normal(N, R, std=0.05, dtype=torch.bfloat16),
                         normal(R, K, std=K ** -0.5, dtype=torch.bfloat16), 0.5 * R)
                        for i in range(case["patches"])]
    return t


def _layer(case, t, out_dtype):
    """The layer as a program has it after loading a checkpoint with this weight."""
    ops = _module("comfy_feather.ops").feather_ops(out_dtype=out_dtype)
    with torch.device("meta"):
        layer = ops.Linear(case["K"], case["N"], bias=t.get("bias") is not None)
    state = {"weight": t["codes"], "weight_scale": t["scale"]}
    if t.get("bias") is not None:
        state["bias"] = t["bias"]
    layer.load_state_dict(state)
    return layer


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mm":
        return {"fn": _module("kernel.hip.hip_kernel").scaled_mm_hip_any_m, "x": t["x"],
                "w": _module("comfy_feather.quant").prepack_transpose(t["codes"]), "scale": t["scale"],
                "bias": t["bias"], "out": _DTYPES[case["out"]], "kind": kind}
    if kind == "load":
        return {"fn": _module("comfy_feather.quant").make_feather_quantized_weight, "kind": kind,
                "w": t["w"] if "w" in t else t["codes"], "scale": t.get("scale")}
    layer = _layer(case, t, _DTYPES[case["w"] if kind == "merge" else case["out"]])
    if kind == "merge":
        return {"layer": layer, "patched": t["patched"], "kind": kind}
    if kind == "lora":
        # the patch objects that a ComfyUI model patcher attaches to a layer
        entries = [(strength, SimpleNamespace(weights=(up, down, alpha, None)), 1.0, None, None)
                   for strength, up, down, alpha in t["patches"]]
        layer.weight_function = [SimpleNamespace(patches={"w": entries}, key="w")]
    return {"layer": layer, "x": t["x"], "kind": kind}


def run(state):
    kind = state["kind"]
    if kind == "mm":
        return state["fn"](state["x"], state["w"], state["scale"], state["bias"], state["out"])
    if kind == "load":
        q = state["fn"](state["w"], state["scale"], torch.bfloat16)
        return [q._qdata.view(torch.uint8), q._params.scale]
    if kind == "merge":
        layer = state["layer"]
        plain = layer.convert_weight(layer.weight)
        q = layer.set_weight(state["patched"], return_weight=True)
        return [plain, q._qdata.view(torch.uint8), q._params.scale]
    with torch.inference_mode():
        return state["layer"](state["x"])


def work(case):
    N, K = case["N"], case["K"]
    if case["kind"] == "load":
        return {"bytes": N * K * (_DTYPES[case["w"]].itemsize + 1), "flops": 2 * N * K}
    if case["kind"] == "merge":  # codes -> 16 bits, 16 bits -> codes
        return {"bytes": 2 * N * K * 3, "flops": 4 * N * K}
    M = case["M"]
    nbytes = 2 * M * K + N * K + 2 * M * N + (2 * N if case["bias"] else 0)
    flops = 2 * M * N * K
    if case["kind"] == "lora":
        R = case["rank"] * case["patches"]
        nbytes += 2 * R * (N + K)
        flops += 2 * M * R * (N + K)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] in ("load", "merge"):
        return "exact"
    # about four times the distance from exact() (2-norm): bf16 results 1.7e-3 to 2.4e-3 off, fp16 ones 2.2e-4 to 3.5e-4
    return {"rel": 1e-2 if case["out"] == "bf16" else 1.4e-3}


def exact(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "load":
        # an e5m2 checkpoint's scale is handed on; a 16- or 32-bit one's is its largest magnitude over e5m2's
        scale = t["scale"].double() if "w" not in t else t["w"].double().abs().amax() / 57344.0
        return [None, scale]
    if case["kind"] == "merge":
        scale = t["patched"].double().abs().amax() / 57344.0
        if case["w"] == "fp16":  # quantizing in fp16 keeps the reciprocal finite
            scale = scale.clamp(min=1.0 / 65504.0)
        return [t["codes"].double() * t["scale"].double(), None, scale]
    x = t["x"].double()
    y = (x @ t["codes"].double().t()) * t["scale"].double()
    if t["bias"] is not None:
        y += t["bias"].double()
    for strength, up, down, alpha in t.get("patches", ()):
        y += (x @ down.double().t()) @ up.double().t() * (strength * alpha / down.shape[0])
    return y
