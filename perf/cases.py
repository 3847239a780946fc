"""The work this package is measured on: whole models through `model(images)`, and the packed-query operators as the
reference's layers call them, forward and backward.

Three kinds of case:

  model      one inference forward of DeiT+DGE or PVT+DGE over a batch of images: what a classification service, an
             offline scoring job or (without a classifier) a detector's backbone runs;
  operators  the `vtpack.layers` operators of one encoder layer on their own - index->patch, compress, attention of the
             packed queries, scatter back - as a program that keeps the reference's own layer files calls them;
  train      the same operators with gradients: the sparse training branch (per-sample products around a softmax).
"""
import math

import torch

from vtpack_amd import engine, layers
from vtpack_amd.layers.sparse_ops import sparse_attention_train
from vtpack_amd.models import dge as zoo
from vtpack_amd.synthetic import IMAGENET_MEAN, IMAGENET_STD, set_synthetic_router

REGION = 4                       # tokens along the edge of a region; splits 4, 2, 1
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

DEIT = {  # width: (factory, channels, heads)
    "tiny": ("deit_dge_s124_tiny_patch16_256", 192, 3),
    "small": ("deit_dge_s124_small_patch16_256", 384, 6),
    "base": ("deit_dge_s124_base_patch16_256", 768, 12),
}
PVT = {   # size: (factory, depths)
    "tiny": ("pvt_dge_s124_tiny_256", (2, 2, 2, 2)),
    "small": ("pvt_dge_s124_small_256", (3, 4, 6, 3)),
}
PVT_DIMS, PVT_MLP, PVT_SR = (64, 128, 320, 512), (8, 8, 4, 4), (8, 4, 2, 1)


def _model(name, family, size, dtype, img, batch, classes=1000):
    return {"name": name, "kind": "model", "family": family, "size": size, "dtype": dtype, "img": img, "batch": batch,
            "classes": classes}


def _ops(name, kind, dtype, batch, grid, heads, sr, extra):
    return {"name": name, "kind": kind, "dtype": dtype, "batch": batch, "grid": grid, "heads": heads, "sr": sr,
            "extra": extra}


def listed():
    return [
        # one picture at a time, as an interactive service sees it: latency, launches and host work
        _model("deit_small_bf16_256_b1", "deit", "small", "bf16", 256, 1),
        # a server's small dynamic batch, odd in number
        _model("deit_small_bf16_256_b13", "deit", "small", "bf16", 256, 13),
        # the headline configuration: offline throughput at 256 px
        _model("deit_small_bf16_256_b256", "deit", "small", "bf16", 256, 256),
        # high resolution: 1025 tokens, long key/value sequences
        _model("deit_small_bf16_512_b64", "deit", "small", "bf16", 512, 64),
        # the published small checkpoint in its own data type, evaluation batch
        _model("deit_tiny_f32_256_b128", "deit", "tiny", "f32", 256, 128),
        # the widest model, the last batch of an evaluation (50000 mod 99)
        _model("deit_base_bf16_256_b5", "deit", "base", "bf16", 256, 5),
        _model("deit_base_bf16_256_b99", "deit", "base", "bf16", 256, 99),
        # the pyramid model: four widths, spatially reduced keys and values
        _model("pvt_small_bf16_256_b256", "pvt", "small", "bf16", 256, 256),
        # its feature maps for a dense-prediction head, full precision, few pictures of a larger size
        _model("pvt_tiny_f32_384_b6_maps", "pvt", "tiny", "f32", 384, 6, 0),
        # the operators under the reference's own layer files, evaluation
        _ops("operators_f32_c384_b64", "operators", "f32", 64, 16, 6, 1, 1),
        # sparse training of one layer: an ordinary per-GPU batch of the small model, and one of the tiny model
        _ops("train_f32_c192_b64", "train", "f32", 64, 16, 3, 1, 1),
        _ops("train_bf16_c384_b128", "train", "bf16", 128, 16, 6, 1, 1),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["model", "model", "model", "model", "operators", "train"])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "model":
        family = rng.choice(["deit", "deit", "pvt"])
        size = rng.choice(["tiny", "small", "base"] if family == "deit" else ["tiny", "small"])
        img = 64 * rng.randint(2, 8) if family == "deit" else 128 * rng.randint(1, 4)
        case = _model("", family, size, dtype, img, 1, rng.choice([1000, 1000, 100, 0]) if family == "pvt" else 1000)
        # as many pictures as keep the pass below the largest listed one: 1.6 TFLOP in bf16, an eighth of it in fp32
        one = _model_flops(case)
        top = int((1.5e12 if dtype == "bf16" else 1.9e11) / one)
        case["batch"] = _log_int(rng, 1, max(1, min(256, top)))
    else:
        heads = rng.choice([1, 2, 3, 5, 6, 8, 12])
        grid = REGION * rng.randint(2, 8)
        sr = rng.choice([1, 1, 1, 2])
        extra = rng.choice([0, 1, 1, 2]) if sr == 1 else 0
        case = _ops("", kind, dtype, 1, grid, heads, sr, extra)
        top = int(128 * 257 * 6 * 64 / ((grid * grid + extra) * heads * 64))
        if kind == "train":     # scores of every query and key are kept: bound them as well
            top = min(top, int(128 * 113 * 257 * 6 / (_queries(case) * _keys(case) * heads)))
        case["batch"] = _log_int(rng, 2, max(2, min(256, top)))
    del case["name"]
    return case


# ------------------------------------------------------------------ work
def _queries(case):
    """Expected packed queries of a sample: 7 a region (1, 4 and 16 alike) behind the extra tokens."""
    return case["extra"] + 7 * (case["grid"] // REGION) ** 2


def _keys(case):
    return (case["grid"] // case["sr"]) ** 2 + case["extra"]


def _block_flops(tokens, keys, queries, c, mlp, sr):
    f = 2 * queries * c * c * 2 + 4 * keys * c * c + 4 * queries * keys * c + 4 * queries * c * c * mlp
    return f + (2 * tokens * c * c * (sr * sr) / (sr * sr) if sr > 1 else 0)


def _model_flops(case):
    b, img, classes = case["batch"], case["img"], case["classes"]
    if case["family"] == "deit":
        c, grid = DEIT[case["size"]][1], img // 16
        tokens = grid * grid + 1
        f = 12 * _block_flops(tokens, tokens, 1 + 7 * (grid // REGION) ** 2, c, 4, 1) + 2 * grid * grid * c * 768
        return b * (f + 2 * c * classes)
    f, cin, k = 0.0, 3, 4
    for i, c in enumerate(PVT_DIMS):
        grid = img // 4 // 2 ** i
        extra = 1 if i == 3 else 0
        tokens, keys = grid * grid + extra, (grid // PVT_SR[i]) ** 2 + extra
        f += 2 * grid * grid * c * cin * k * k
        f += PVT[case["size"]][1][i] * _block_flops(tokens, keys, extra + 7 * (grid // REGION) ** 2, c, PVT_MLP[i],
                                                    PVT_SR[i])
        cin, k = c, 2
    return b * (f + 2 * PVT_DIMS[3] * classes)


def _model_params(case):
    img, classes = case["img"], case["classes"]
    if case["family"] == "deit":
        c = DEIT[case["size"]][1]
        return 12 * 12 * c * c + 768 * c + (img // 16) ** 2 * c + c * classes
    n, cin, k = 0, 3, 4
    for i, c in enumerate(PVT_DIMS):
        per = 4 * c * c + 2 * PVT_MLP[i] * c * c + (c * c * PVT_SR[i] ** 2 if PVT_SR[i] > 1 else 0)
        n += PVT[case["size"]][1][i] * per + cin * c * k * k + (img // 4 // 2 ** i) ** 2 * c
        cin, k = c, 2
    return n + PVT_DIMS[3] * classes


def work(case):
    e = 2 if case["dtype"] == "bf16" else 4
    b = case["batch"]
    if case["kind"] == "model":
        out = b * case["classes"]
        if case["family"] == "pvt" and case["classes"] == 0:
            out = b * sum(c * (case["img"] // 4 // 2 ** i) ** 2 for i, c in enumerate(PVT_DIMS))
        return {"bytes": e * (_model_params(case) + 3 * b * case["img"] ** 2 + out), "flops": _model_flops(case)}
    c = 64 * case["heads"]
    x = b * (case["grid"] ** 2 + case["extra"]) * c
    kv = 2 * b * _keys(case) * c
    rows = b * _queries(case)
    ints = 8 * b * (case["grid"] // REGION) ** 2 + 32 * rows
    product = 2.0 * rows * _keys(case) * c
    if case["kind"] == "operators":
        return {"bytes": e * (2 * x + kv) + ints, "flops": 2 * product}
    # forward: tokens, keys and values in, tokens out; backward: the output's gradient in, theirs out
    return {"bytes": e * (2 * x + kv) + e * (2 * x + kv) + ints, "flops": 6 * product}


# ------------------------------------------------------------------ tolerance
def tolerance(case):
    """About four times what was measured over the listed cases: models against the same weights run as the modules'
    own composition (library GEMMs, LayerNorm apart: other roundings and orders of the sums), 1.2e-2 to 1.5e-2 of the
    logits in bf16 and up to 1.1e-6 in fp32 (maps: 9.9e-7); operators against float64, 3.7e-7 in fp32 and 4.9e-3 in
    bf16 (gradients; the forward results 6e-8 and 2.4e-3).  A tie of a router that falls the other way in fp32 (two
    logits within about 1e-6, some 0.01 to 0.04 of all seeds at 24576 decisions) would move one picture's logits by
    3e-3: no allowance is made for it."""
    if case["kind"] == "model":
        return {"rel": 5e-2} if case["dtype"] == "bf16" else {"rel": 1e-5}
    return {"rel": 2e-2} if case["dtype"] == "bf16" else {"rel": 2e-6}


# ------------------------------------------------------------------ inputs
def _images(gen, batch, size, dtype, device):
    """Pictures in [0, 1] with large shapes and fine texture, normalised per channel: regions of one picture differ,
    and pictures differ from each other, so the query counts of a batch are ragged."""
    low = torch.rand((batch, 3, 6, 6), generator=gen, device=device)
    amount = torch.rand((batch, 1, 6, 6), generator=gen, device=device)
    up = dict(size=(size, size), mode="bilinear", align_corners=False)
    img = torch.nn.functional.interpolate(low, **up)
    tex = torch.nn.functional.interpolate(amount, **up)
    img = img + tex * (torch.rand((batch, 3, size, size), generator=gen, device=device) - 0.5)
    mean = torch.tensor(IMAGENET_MEAN, device=device).view(1, 3, 1, 1)
    std = torch.tensor(IMAGENET_STD, device=device).view(1, 3, 1, 1)
    return ((img.clamp_(0, 1) - mean) / std).to(dtype)


def prepare(case, seed):
    device = torch.device("cuda:0")
    dtype = DTYPES[case["dtype"]]
    gen = torch.Generator(device).manual_seed(seed)
    if case["kind"] == "model":
        torch.manual_seed(seed)
        factory = DEIT[case["size"]][0] if case["family"] == "deit" else PVT[case["size"]][0]
        with torch.device(device):
            model = getattr(zoo, factory)(img_size=case["img"], num_classes=case["classes"])
        set_synthetic_router(model, seed)      # a mixed gate: an untrained router always takes the finest split
        model = engine.prepare(model.eval().to(dtype))
        return {"model": model, "images": _images(gen, case["batch"], case["img"], dtype, device)}
    b, grid, heads, extra = case["batch"], case["grid"], case["heads"], case["extra"]
    regions = grid // REGION

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=device).to(dtype)

    # every sample with a mix of granularities of its own, from nearly all coarse to nearly all fine
    lean = torch.randn((b, 1, 3), generator=gen, device=device)
    noise = torch.rand((b, regions * regions, 3), generator=gen, device=device).clamp_(1e-6, 1 - 1e-6)
    indices = (lean - (-noise.log()).log()).argmax(dim=-1).reshape(b, regions, regions)
    indices[1] = indices[0]              # the first two samples differ in one region: ragged whatever is drawn
    indices[0, 0, 0], indices[1, 0, 0] = 0, 2
    train = case["kind"] == "train"
    state = {"indices": indices, "splits": torch.tensor([4, 2, 1], device=device), "grid": grid, "extra": extra,
             "heads": heads, "train": train,
             "x": normal(b, grid * grid + extra, 64 * heads).requires_grad_(train),
             "k": normal(heads, b, _keys(case), 64).requires_grad_(train),
             "v": normal(heads, b, _keys(case), 64).requires_grad_(train)}
    if train:
        state["grad"] = normal(b, grid * grid + extra, 64 * heads)
    return state


def run(state):
    if "model" in state:
        with torch.no_grad():
            return state["model"](state["images"])
    x, k, v, grid, extra, heads = (state[n] for n in ("x", "k", "v", "grid", "extra", "heads"))
    patches, lengths = layers.grained_sample_index_to_patch(state["indices"], state["splits"], REGION, extra)
    comp = layers.grained_sample_compress(x, patches, grid, grid, extra)
    q = comp.reshape(-1, heads, 64).transpose(0, 1)
    if not state["train"]:
        o = layers.batched_sparse_attention(q, k, v, lengths, 0.125)
        o = o.transpose(0, 1).reshape(-1, 64 * heads)
        out = layers.grained_sample_decompress(o - comp, patches, x, grid, grid, extra, True)
        return {"out": out, "lengths": lengths}
    o = sparse_attention_train(q, k, v, lengths, 0.125)
    out = layers.grained_sample_decompress(o - comp, patches, x, grid, grid, extra, True)
    gx, gk, gv = torch.autograd.grad(out, (x, k, v), state["grad"])
    return {"out": out.detach(), "grad_x": gx, "grad_k": gk, "grad_v": gv}
