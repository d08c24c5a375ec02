"""What a program that uses this package has it do, as cases that can be timed.

Four kinds, each through the public names such a program calls:

  predict    SamPredictor.set_torch_image on one camera image, the interactive use: uint8 pixels whose
             long side is 1024, normalised, padded to the square, encoded, the embedding kept
  encode     sam.image_encoder(batch) without autograd, the offline use: normalised bf16 squares
  attention  flash_4._attention_rel_h_rel_w, the operator with the caller's own bias factors
  linear     one swapped Linear (Int8DynamicLinear, or its 2:4-sparse form) called as a module

A program loads its weights once and then sees new images, so `prepare` keeps the encoder of a
(model, linears) pair between calls and makes the images from the seed; operators and Linears get
all their tensors from the seed.
"""

import math
import os
import sys
from collections import OrderedDict

import torch

sys.path.insert(0, os.path.abspath("segment-anything-fast_amd"))

import samfast_amd  # noqa: E402
from samfast_amd import sparse  # noqa: E402
from samfast_amd.flash_4 import _attention_rel_h_rel_w  # noqa: E402

# width, blocks, heads; every fourth part of the depth ends in a global block
_MODELS = {"vit_b": (768, 12, 12), "vit_l": (1024, 24, 16), "vit_h": (1280, 32, 16)}
_TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # an annotation tool that embeds the picture a person has just opened: the smallest encoder,
        # int8 linears, a landscape photo; launches and gaps between them count
        dict(name="predict_vit_b_int8", kind="predict", model="vit_b", linears="int8", height=683, width=1024),
        # the registry's default model with nothing swapped, a portrait photo
        dict(name="predict_vit_h_bf16", kind="predict", model="vit_h", linears="bf16", height=1024, width=767),
        # a small odd batch of the middle model in plain bf16: too long for a recorded graph
        dict(name="encode_vit_l_bf16_5", kind="encode", model="vit_l", linears="bf16", images=5),
        # the benchmark's configuration
        dict(name="encode_vit_h_int8_16", kind="encode", model="vit_h", linears="int8", images=16),
        # int8 with 2:4-sparse MLP weights over a full batch: the largest
        dict(name="encode_vit_h_sparse_32", kind="encode", model="vit_h", linears="sparse", images=32),
        # the operator alone on one image's global block, batch 1, head_dim 64
        dict(name="attention_grid_b1_h12_d64", kind="attention", batch=1, heads=12, rows=64, cols=64, dim=64, type="bf16"),
        # the same on a batch, head_dim 80, in fp16, the operator's other type
        dict(name="attention_grid_b8_h16_d80", kind="attention", batch=8, heads=16, rows=64, cols=64, dim=80, type="fp16"),
        # the 25 windows of one image
        dict(name="attention_windows_25_d64", kind="attention", batch=25, heads=12, rows=14, cols=14, dim=64, type="bf16"),
        # a Linear over a handful of tokens (prompts): the smallest call
        dict(name="linear_7x256x2048", kind="linear", weight="int8", rows=7, inputs=256, outputs=2048),
        # one image's tokens through the smallest model's first MLP layer
        dict(name="linear_4096x768x3072", kind="linear", weight="int8", rows=4096, inputs=768, outputs=3072),
        # a batch of 16 images through the largest model's qkv
        dict(name="linear_65536x1280x3840", kind="linear", weight="int8", rows=65536, inputs=1280, outputs=3840),
        # the sparse form on a row count that is no multiple of anything
        dict(name="linear_sparse_5003x5120x1280", kind="linear", weight="sparse", rows=5003, inputs=5120, outputs=1280),
    ]


def _log_uniform(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("predict", "encode", "attention", "attention", "linear", "linear"))
    if kind == "predict":
        short = rng.randint(256, 1024)
        height, width = rng.choice(((short, 1024), (1024, short)))
        return dict(kind=kind, model=rng.choice(tuple(_MODELS)), linears=rng.choice(("int8", "bf16")), height=height, width=width)
    if kind == "encode":
        return dict(kind=kind, model=rng.choice(tuple(_MODELS)), linears=rng.choice(("int8", "bf16", "sparse")), images=_log_uniform(rng, 1, 16))
    if kind == "attention":
        dim, heads, dtype = rng.choice((64, 80)), rng.randint(8, 16), rng.choice(("bf16", "fp16"))
        if rng.random() < 0.5:  # global blocks: a grid 64 tokens wide, square or not (an even number of rows)
            rows = rng.choice((64, 2 * rng.randint(2, 32)))
            return dict(kind=kind, batch=_log_uniform(rng, 1, 16), heads=heads, rows=rows, cols=64, dim=dim, type=dtype)
        rows, cols = rng.choice(((14, 14), (rng.randint(5, 14), rng.randint(5, 14))))
        return dict(kind=kind, batch=_log_uniform(rng, 1, 400), heads=heads, rows=rows, cols=cols, dim=dim, type=dtype)
    rows = _log_uniform(rng, 1, 65536)
    width = rng.choice(tuple(_MODELS.values()))[0]
    inputs, outputs = rng.choice(((width, 3 * width), (width, width), (width, 4 * width), (4 * width, width),
                                  (128 * rng.randint(2, 20), 8 * rng.randint(16, 320))))
    return dict(kind=kind, weight=rng.choice(("int8", "int8", "sparse")), rows=rows, inputs=inputs, outputs=outputs)


_encoders = OrderedDict()  # (model, linears) -> Sam, the last few


def _sam(model, linears):
    """The model as a program loads it, with one fixed set of weights (Linear weights 0.02 wide, unit norms)."""
    key = (model, linears)
    if key in _encoders:
        _encoders.move_to_end(key)
        return _encoders[key]
    while len(_encoders) > 3:
        _encoders.popitem(last=False)
    with torch.device("cuda"):
        sam = samfast_amd.sam_model_fast_registry[model]()
    gen = torch.Generator(device="cuda").manual_seed(7)
    with torch.no_grad():
        for name, p in sam.image_encoder.named_parameters():
            if ".norm" in name or ".neck.1." in name or ".neck.3." in name:
                p.fill_(1.0 if name.endswith("weight") else 0.0)
            else:
                p.normal_(0.0, 0.02, generator=gen)
        if linears == "sparse":
            samfast_amd.apply_sparse(sam.image_encoder, sparse.mlp_only)
        if linears != "bf16":
            samfast_amd.apply_dynamic_quant(sam.image_encoder)
    _encoders[key] = sam
    return sam


def _normal(gen, shape, std, dtype):
    return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] in ("predict", "encode"):
        sam = _sam(case["model"], case["linears"])
        if case["kind"] == "predict":
            size = (case["height"], case["width"])
            image = torch.randint(0, 256, (1, 3) + size, generator=gen, device="cuda", dtype=torch.uint8)
            return ("predict", samfast_amd.SamPredictor(sam), image, size)
        pixels = torch.rand((case["images"], 3, 1024, 1024), generator=gen, device="cuda") * 255.0
        return ("encode", sam.image_encoder, ((pixels - sam.pixel_mean) / sam.pixel_std).to(torch.bfloat16))
    if case["kind"] == "attention":
        # q, k, v and both bias factors ~ N(0, 0.5), the recipe of the operator's own test
        dtype, rows, cols = _TYPES[case["type"]], case["rows"], case["cols"]
        lead = (case["batch"], case["heads"], rows * cols)
        q, k, v = (_normal(gen, lead + (case["dim"],), 0.5, dtype) for _ in range(3))
        rel_h = _normal(gen, lead + (rows, 1), 0.5, dtype)
        rel_w = _normal(gen, lead + (1, cols), 0.5, dtype)
        return ("attention", q, k, v, rel_h, rel_w)
    # activations ~ N(0, 1) with 0.1 % of the rows 20 times as large, weights ~ N(0, 0.02)
    linear = torch.nn.Linear(case["inputs"], case["outputs"], device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        linear.weight.normal_(0.0, 0.02, generator=gen)
        linear.bias.normal_(0.0, 0.02, generator=gen)
    x = torch.randn((case["rows"], case["inputs"]), generator=gen, device="cuda")
    x *= 1.0 + 19.0 * (torch.rand((case["rows"], 1), generator=gen, device="cuda") < 1e-3)
    make = samfast_amd.Int8Sparse24Linear if case["weight"] == "sparse" else samfast_amd.Int8DynamicLinear
    return ("linear", make.from_float(linear), x.to(torch.bfloat16))


@torch.no_grad()
def run(state):
    kind = state[0]
    if kind == "predict":
        _, predictor, image, size = state
        predictor.set_torch_image(image, size)
        return predictor.get_image_embedding()
    if kind == "attention":
        return _attention_rel_h_rel_w(*state[1:])
    return state[1](state[2])  # an encoder, or a Linear


def work(case):
    if case["kind"] == "attention":
        tokens, slices = case["rows"] * case["cols"], case["batch"] * case["heads"]
        values = tokens * (4 * case["dim"] + case["rows"] + case["cols"])
        return {"bytes": 2 * slices * values, "flops": 4 * slices * tokens * tokens * case["dim"]}
    if case["kind"] == "linear":
        m, k, n = case["rows"], case["inputs"], case["outputs"]
        kept = 1 if case["weight"] == "int8" else 2  # of every four weights, all or two are multiplied
        stored = n * k if case["weight"] == "int8" else n * k * 9 // 16
        return {"bytes": 2 * m * (k + n) + stored + 8 * n, "flops": 2 * m * n * k // kept}
    c, blocks, heads = _MODELS[case["model"]]
    images = case.get("images", 1)
    tokens = 64 * 64
    mlp_kept = 2 if case["linears"] == "sparse" else 1
    linears = 2 * tokens * c * c * (4 + 8 / mlp_kept)
    attention = 4 * c * (4 * tokens * tokens + (blocks - 4) * 25 * 196 * 196)
    ends = 2 * tokens * c * 768 + 2 * tokens * (c * 256 + 9 * 256 * 256)
    weight_bytes = {"bf16": 24, "int8": 12, "sparse": 4 + 8 * 9 / 16}[case["linears"]]
    image_bytes = 3 * case["height"] * case["width"] if case["kind"] == "predict" else images * 3 * 1024 * 1024 * 2
    weights = blocks * c * c * weight_bytes + 2 * (768 * c + tokens * c + 256 * c + 9 * 256 * 256)
    return {"bytes": image_bytes + weights + images * 2 * tokens * 256, "flops": images * (blocks * linears + attention + ends)}


def tolerance(case):
    if case["kind"] == "linear":
        return {"rel": 5e-3}  # the sum is exact in int32, the result is rounded to bf16
    if case["kind"] == "attention":
        return {"rel": 1e-2 if case["type"] == "bf16" else 2e-3}  # probabilities and result in the half type
    # dozens of blocks of bf16 activations, each rounding free to move an int8 code by one
    return {"rel": 2e-2}
