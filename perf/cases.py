"""Timed cases of the DINOv3 ViT-S+/16 forward pass, through its public calls.

A program uses the model in three ways, the `call` of a case:
  "graph"  device tensors in and out, `forward_noalloc` captured once into a
           HIP graph and replayed for each new batch (a serving loop);
  "eager"  the same call queued directly on the current stream (a PyTorch
           program that runs the encoder between its own operations);
  "host"   `forward` on float32 host arrays, any number of images, cut into
           chunks of the model's max_batch (offline feature extraction).
`plan` is the launch plan the call runs: "folded" (the default, LayerNorm
folded into the matrix products) or "separate" (LayerNorm and split-K kernels
of their own, `set_layernorm_fusion(False)` and `set_splitk(1)`).

Every case returns the whole float32 [images, tokens, 384] output.
"""
import atexit
import json
import math
import os
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "dinov3-loom_amd"))

HIDDEN, HEADS, HEAD_DIM, LAYERS, FF, PREFIX = 384, 6, 64, 12, 1536, 5
SCRATCH_BYTES = 64 << 20  # what forward_noalloc may use
HOST_BATCH = 64           # the largest resident batch
LARGEST_FLOPS = 1.9e12    # no drawn case costs more than the largest listed one


def _case(name, call, image_size, images, plan="folded"):
    return {"name": name, "call": call, "image_size": image_size, "images": images, "plan": plan}


def listed():
    return [
        # One image: interactive latency (a query image, a camera frame).
        _case("graph_224_b1", "graph", 224, 1),
        _case("eager_224_b1", "eager", 224, 1),
        _case("host_224_b1", "host", 224, 1),
        # A small, odd batch: requests gathered by a server over a few ms.
        _case("graph_224_b5", "graph", 224, 5),
        # An ordinary batch inside a PyTorch program.
        _case("eager_224_b16", "eager", 224, 16),
        # The largest 224x224 batch the allocation-free call takes.
        _case("graph_224_b43", "graph", 224, 43),
        # Dense features at 512x512 (1029 tokens): one image, and a batch.
        _case("graph_512_b1", "graph", 512, 1),
        _case("graph_512_b8", "graph", 512, 8),
        # Sizes without a shape of their own: 384x384 (581 tokens, a ragged
        # row count) and the largest image (4101 tokens).
        _case("graph_384_b3", "graph", 384, 3),
        _case("graph_1024_b2", "graph", 1024, 2),
        # The plan with LayerNorm and split-K kernels of their own.
        _case("graph_224_b8_separate", "graph", 224, 8, "separate"),
        # Feature extraction from host memory: two full chunks and a ragged one.
        _case("host_224_b150", "host", 224, 150),
    ]


def _tokens(case):
    return (case["image_size"] // 16) ** 2 + PREFIX


def _scratch(image_size, images, plan):
    """Bytes of scratch forward_noalloc lays out for a batch."""
    t = (image_size // 16) ** 2 + PREFIX
    rows = images * t
    frag_rows = (rows + 31) // 32 * 32
    heads = images * HEADS * ((t + 127) // 128 * 128) * HEAD_DIM * 2
    sizes = [frag_rows * HIDDEN * 2] * 2 + [heads] * 3 + [frag_rows * FF * 2]
    sizes += [frag_rows * HIDDEN * 2, 4 * rows * HIDDEN * 4] if plan == "separate" else [rows * 48]
    return sum((s + 255) // 256 * 256 for s in sizes)


def _flops(image_size, images):
    t = (image_size // 16) ** 2 + PREFIX
    gemm = 2 * t * HIDDEN * (3 * HIDDEN + HIDDEN + 3 * FF)
    attention = 4 * t * t * HIDDEN
    embed = 2 * (t - PREFIX) * 768 * HIDDEN
    return float(images * (embed + LAYERS * (gemm + attention)))


def _host_batch(image_size):
    """Resident batch of a host model: the pixels of 64 images of 224x224."""
    return max(1, min(HOST_BATCH, HOST_BATCH * 224 * 224 // image_size ** 2))


def draw(rng):
    call = rng.choice(["graph", "graph", "graph", "eager", "host"])
    plan = "separate" if rng.random() < 0.15 else "folded"
    # Image sides from 64 to 1024 in steps of 16, spread over their logarithm.
    size = max(64, min(1024, 16 * round(64 * 16 ** rng.random() / 16)))
    if call == "host":
        most = max(1, 5 * _host_batch(size) // 2)
    else:
        most = 1
        while most < 64 and _scratch(size, most + 1, plan) <= SCRATCH_BYTES - (1 << 20):
            most += 1
    while most > 1 and _flops(size, most) > LARGEST_FLOPS:
        most -= 1
    images = max(1, min(most, int(round(math.exp(rng.uniform(0, math.log(most + 0.49)))))))
    return {"call": call, "image_size": size, "images": images, "plan": plan}


# ---------------------------------------------------------------------------
# Weights: one seeded checkpoint per process, written as a program would find
# it on disk (HF names, float32). Matrices hold float16 values, so that the
# loader's narrowing is exact. Query and key weights are wide enough for
# peaked attention, layer scales and LayerNorm affines are not trivial.

_tensors = None
_file = None


def _weights():
    global _tensors
    if _tensors is not None:
        return _tensors
    gen = torch.Generator().manual_seed(20240917)

    def normal(shape, std, mean=0.0):
        return torch.randn(shape, generator=gen) * std + mean

    def matrix(shape, std):
        return normal(shape, std).clamp_(-2 * std, 2 * std).half().float()

    w = {
        "embeddings.patch_embeddings.weight": matrix((HIDDEN, 3, 16, 16), 0.02),
        "embeddings.patch_embeddings.bias": normal((HIDDEN,), 0.02),
        "embeddings.cls_token": matrix((1, 1, HIDDEN), 0.02),
        "embeddings.register_tokens": matrix((1, 4, HIDDEN), 0.02),
        "embeddings.mask_token": torch.zeros(1, 1, HIDDEN),
    }
    for i in range(LAYERS):
        p = f"layer.{i}."
        for n in ("norm1", "norm2"):
            w[p + n + ".weight"] = normal((HIDDEN,), 0.1, 1.0)
            w[p + n + ".bias"] = normal((HIDDEN,), 0.1)
        for n, std in (("q", 0.06), ("k", 0.06), ("v", 0.02), ("o", 0.02)):
            w[p + f"attention.{n}_proj.weight"] = matrix((HIDDEN, HIDDEN), std)
            if n != "k":
                w[p + f"attention.{n}_proj.bias"] = normal((HIDDEN,), 0.02)
        for n in ("gate", "up"):
            w[p + f"mlp.{n}_proj.weight"] = matrix((FF, HIDDEN), 0.02)
            w[p + f"mlp.{n}_proj.bias"] = normal((FF,), 0.02)
        w[p + "mlp.down_proj.weight"] = matrix((HIDDEN, FF), 0.02)
        w[p + "mlp.down_proj.bias"] = normal((HIDDEN,), 0.02)
        for n in ("layer_scale1", "layer_scale2"):
            w[p + n + ".lambda1"] = normal((HIDDEN,), 0.2, 0.8)
    w["norm.weight"] = normal((HIDDEN,), 0.1, 1.0)
    w["norm.bias"] = normal((HIDDEN,), 0.1)
    _tensors = w
    return w


def _weight_file():
    global _file
    if _file is None:
        folder = tempfile.mkdtemp(prefix="dinov3-cases-")
        atexit.register(shutil.rmtree, folder, ignore_errors=True)
        header, at, parts = {}, 0, []
        for name, t in _weights().items():
            raw = t.contiguous().numpy().tobytes()
            header[name] = {"dtype": "F32", "shape": list(t.shape), "data_offsets": [at, at + len(raw)]}
            at += len(raw)
            parts.append(raw)
        text = json.dumps(header).encode()
        text += b" " * (-len(text) % 8)
        path = os.path.join(folder, "model.safetensors")
        with open(path, "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for raw in parts:
                f.write(raw)
        _file = path
    return _file


_models = {}


def _model(case):
    """The loaded model a program keeps for its images' size and its plan."""
    import dinov3_hrx as d

    size = case["image_size"]
    batch = _host_batch(size) if case["call"] == "host" else 1
    key = (size, batch, case["plan"])
    if key not in _models:
        m = d.DINOv3.load(_weight_file(), d.Options(0, batch, size))
        if case["plan"] == "separate":
            m.set_layernorm_fusion(False)
            m.set_splitk(1)
        _models[key] = m
    return _models[key]


def _pixels(case, seed):
    """ImageNet-normalised pixels: zero mean, unit variance."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = case["image_size"]
    return torch.randn((case["images"], 3, s, s), generator=gen, device="cuda")


def prepare(case, seed):
    state = {"model": _model(case), "images": case["images"], "call": case["call"]}
    pixels = _pixels(case, seed)
    if case["call"] == "host":
        state["pixels"] = pixels.cpu().numpy()
        return state
    state["pixels"] = pixels
    state["out"] = torch.empty((case["images"], _tokens(case), HIDDEN), device="cuda")
    if case["call"] == "graph":
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            _queue(state)
        state["graph"] = graph
    return state


def _queue(state):
    state["model"].forward_noalloc(state["pixels"].data_ptr(), state["images"], state["out"].data_ptr(),
                                   torch.cuda.current_stream().cuda_stream)


def run(state):
    if state["call"] == "host":
        return state["model"].forward(state["pixels"])
    if state["call"] == "graph":
        state["graph"].replay()
    else:
        _queue(state)
    return state["out"]


def work(case):
    """Pixels and weights read once, tokens written once; the products of the model."""
    s = case["image_size"]
    matrices = 2 * (HIDDEN * 768 + LAYERS * (4 * HIDDEN * HIDDEN + 3 * HIDDEN * FF))
    pixels = case["images"] * 3 * s * s * 4
    out = case["images"] * _tokens(case) * HIDDEN * 4
    return {"bytes": float(matrices + pixels + out), "flops": _flops(s, case["images"])}


def tolerance(case):
    # float16 weights, activations and softmax weights with float32 sums over
    # twelve layers: measured against exact(), rel 1.07e-3 to 1.29e-3 and the
    # largest single difference 6.5e-3 to 1.0e-2 over sizes, batches and plans.
    return {"rel": 5e-3, "max": 4e-2}


def exact(case, seed):
    """The same forward in float64, from the same float32 pixels and weights."""
    w = {k: v.to("cuda", torch.float64) for k, v in _weights().items()}
    pixels = _pixels(case, seed)
    grid = case["image_size"] // 16
    t = _tokens(case)
    pos = (2 * (torch.arange(grid, dtype=torch.float64, device="cuda") + 0.5) / grid - 1) * 2 * math.pi
    freq = 100.0 ** (-torch.arange(16, dtype=torch.float64, device="cuda") / 16)
    ang_y = (pos[:, None] * freq)[:, None, :].expand(grid, grid, 16)
    ang_x = (pos[:, None] * freq)[None, :, :].expand(grid, grid, 16)
    angle = torch.cat([ang_y, ang_x, ang_y, ang_x], -1).reshape(grid * grid, 64)
    cos = torch.cat([torch.ones(PREFIX, 64, dtype=torch.float64, device="cuda"), angle.cos()])
    sin = torch.cat([torch.zeros(PREFIX, 64, dtype=torch.float64, device="cuda"), angle.sin()])

    def norm(x, name):
        mean = x.mean(-1, keepdim=True)
        var = (x - mean).square().mean(-1, keepdim=True)
        return (x - mean) / torch.sqrt(var + 1e-5) * w[name + ".weight"] + w[name + ".bias"]

    def linear(x, name):
        y = x @ w[name + ".weight"].t().contiguous()
        return y + w[name + ".bias"] if name + ".bias" in w else y

    def rope(x):  # [t, 64]
        turned = torch.cat([-x[:, 32:], x[:, :32]], -1)
        return x * cos + turned * sin

    out = torch.empty((case["images"], t, HIDDEN), dtype=torch.float64, device="cuda")
    for first in range(0, case["images"], 16):
        px = pixels[first:first + 16].double()
        n = px.shape[0]
        patches = px.reshape(n, 3, grid, 16, grid, 16).permute(0, 2, 4, 1, 3, 5).reshape(n * grid * grid, 768)
        kernel = w["embeddings.patch_embeddings.weight"].reshape(HIDDEN, 768).t().contiguous()
        embed = (patches.contiguous() @ kernel + w["embeddings.patch_embeddings.bias"]).reshape(n, grid * grid, HIDDEN)
        prefix = torch.cat([w["embeddings.cls_token"], w["embeddings.register_tokens"]], 1).expand(n, -1, -1)
        x = torch.cat([prefix, embed], 1).reshape(n * t, HIDDEN)
        for i in range(LAYERS):
            p = f"layer.{i}."
            h = norm(x, p + "norm1")
            q, k, v = (linear(h, p + f"attention.{c}_proj") for c in "qkv")
            a = torch.empty_like(x)
            for img in range(n):
                r = slice(img * t, (img + 1) * t)
                for head in range(HEADS):
                    c = slice(head * HEAD_DIM, (head + 1) * HEAD_DIM)
                    score = rope(q[r, c]) @ rope(k[r, c]).t().contiguous() / 8
                    a[r, c] = torch.softmax(score, -1) @ v[r, c].contiguous()
            x = x + w[p + "layer_scale1.lambda1"] * linear(a, p + "attention.o_proj")
            h = norm(x, p + "norm2")
            gate, up = linear(h, p + "mlp.gate_proj"), linear(h, p + "mlp.up_proj")
            y = linear(gate * torch.sigmoid(gate) * up, p + "mlp.down_proj")
            x = x + w[p + "layer_scale2.lambda1"] * y
        out[first:first + n] = norm(x, "norm").reshape(n, t, HIDDEN)
    return out
