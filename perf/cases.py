"""The work a user of this framework has it do, as cases that can be prepared, run and timed.

Five kinds of call, all through public entry points:

* ``op``     the whole sparse global attention path on post-norm q, k, v and a gate (``sparse_global_attention``)
* ``layer``  the attention layer of the decoder, inference (``SparseFlashAttentionRope`` under ``no_grad``)
* ``grad``   the two attention operators with their gradients (``flash_attn_topk_func``, ``topk_blocksparse_attention``)
* ``train``  the layer's forward and backward as a training step runs it (gradients of the input and of every weight)
* ``model``  the whole multi-view forward (``Pi3SparseLike``): images in, point maps, confidences and poses out

Sizes follow the benchmark's frames (37 x 28 patches and 5 register tokens in row order with 64-token blocks; 36 x 28
patches in 4 x 4-tile order with 16-token blocks and the 32 best blocks, the layer's own setting), 16 heads of 64.
"""
from __future__ import annotations

import math
from functools import partial

import torch
import torch.nn.functional as F
from torch import nn

from speed3r_amd import flash_attn_topk_func, pool_mean, sparse_global_attention, topk_blocksparse_attention, workloads
from speed3r_amd.layers import RoPE2D, SparseFlashAttentionRope
from speed3r_amd.model import Pi3SparseLike
from speed3r_amd.model.token_order import tile_major

HEADS, HEAD_DIM = 16, 64
DIM = HEADS * HEAD_DIM
DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(kind, frames, gh, gw, reg, block, topk, dtype, batch=1, **more):
    return dict(kind=kind, frames=frames, gh=gh, gw=gw, reg=reg, block=block, topk=topk, dtype=dtype, batch=batch, **more)


def listed():
    row, tile = (37, 28, 5), (36, 28, 0)   # patch grid and register tokens of the two token layouts
    cases = {
        # two views, the smallest reconstruction there is: one layer call as a drop-in user writes it (positions, no bound)
        "layer_2_views": _case("layer", 2, *tile, 16, 32, "bf16", bound=False),
        # a short clip in the layer's own setting (4 x 4-tile blocks, the 32 best)
        "layer_32_frames_block16": _case("layer", 32, *tile, 16, 32, "bf16", bound=True),
        # the global layer of a 100-frame sequence, called as the model calls it
        "layer_100_frames": _case("layer", 100, *row, 64, 16, "bf16", bound=True),
        # half precision on other frames: an odd grid, a ragged last block, fewer blocks per query
        "layer_33_frames_fp16": _case("layer", 33, 33, 23, 5, 64, 8, "fp16", bound=False),
        # full precision on a few views (checking, and hosts without mixed precision)
        "op_8_frames_fp32": _case("op", 8, *row, 64, 16, "fp32"),
        # the operator path on a video: a clip, a long clip, a whole recording
        "op_64_frames": _case("op", 64, *row, 64, 16, "bf16"),
        "op_256_frames": _case("op", 256, *row, 64, 16, "bf16"),
        "op_1000_frames": _case("op", 1000, *row, 64, 16, "bf16"),
        # the long clip at the finer setting
        "op_256_frames_block16": _case("op", 256, *row, 16, 32, "bf16"),
        # both operators with gradients on the long clip
        "grad_256_frames": _case("grad", 256, *row, 64, 16, "bf16"),
        # one layer of a training step: two sequences of 12 frames, fp32 weights under autocast
        "train_2x12_frames_block16": _case("train", 12, *tile, 16, 32, "bf16", batch=2, autocast=True),
        # images to point maps for eight views
        "model_8_views": _case("model", 8, *tile, 16, 32, "bf16"),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choices(("op", "layer", "grad", "train", "model"), weights=(4, 4, 2, 2, 1))[0]
    fine = kind == "model" or rng.random() < 0.4       # 16-token blocks in tile order, else 64-token blocks in row order
    if fine:
        gh, gw, reg, block, topk = 4 * rng.randint(5, 9), 4 * rng.randint(5, 9), 0, 16, rng.choice((16, 32, 32))
    else:
        gh, gw, reg, block, topk = rng.randint(20, 37), rng.randint(20, 37), rng.choice((0, 5)), 64, rng.choice((8, 16, 16, 32))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16"))
    most = {"op": 266496 if fine else 1041000, "layer": 104100, "grad": 100000 if fine else 266496, "train": 50000, "model": 8100}[kind]
    if kind == "op" and rng.random() < 0.15:           # full precision: a few views
        dtype, most = "fp32", 8328
    if kind == "op" and topk == 32 and not fine:
        most = 520500
    batch = rng.choice((1, 1, 2)) if kind in ("layer", "train") else 1
    per = (gh * gw + reg) * batch
    least = {"op": 1041, "layer": 1041, "grad": 8000, "train": 4000, "model": 2000}[kind]
    frames = max(1, min(most // per, round(_log_uniform(rng, least, most) / per)))
    more = {"layer": {"bound": rng.random() < 0.5}, "train": {"autocast": rng.random() < 0.5}}.get(kind, {})
    return _case(kind, frames, gh, gw, reg, block, topk, dtype if kind != "model" else "bf16", batch, **more)


# ---- inputs ------------------------------------------------------------------------------------------------------

def _positions(case):
    """(y, x) of every token of the sequence, ``[B, N, 2]``: register tokens at (0, 0) and patches from 1, or patches
    from 0 in 4 x 4-tile order."""
    gh, gw, reg = case["gh"], case["gw"], case["reg"]
    yy, xx = torch.meshgrid(torch.arange(gh, device=DEV), torch.arange(gw, device=DEV), indexing="ij")
    pos = torch.stack((yy, xx), dim=-1).reshape(gh * gw, 2)
    if case["block"] == 16 and reg == 0:
        pos = tile_major(pos[None], gh, gw, 4)[0]
    if reg:
        pos = torch.cat((pos.new_zeros((reg, 2)), pos + 1))
    return pos.repeat(case["frames"], 1)[None].repeat(case["batch"], 1, 1)


def _tokens(case, pos, gen):
    """Normalised decoder tokens ``[B, N, DIM]`` in fp32: what a frame shares, what varies smoothly over its patches and
    over the sequence, and what is the token's own."""
    b, n = pos.shape[:2]
    per = n // case["frames"]
    randn = partial(torch.randn, generator=gen, device=DEV)
    frame = (randn((b, case["frames"], 8)) @ randn((8, DIM)) / 8 ** 0.5).repeat_interleave(per, dim=1)
    wave = pos.float() @ (randn((2, 24)) * 0.05) + randn((b, case["frames"], 24)).repeat_interleave(per, dim=1) * 0.5
    smooth = wave.sin() @ (randn((24, DIM)) / 12 ** 0.5)
    return F.layer_norm(0.6 * frame + 0.8 * smooth + 0.5 * randn((b, n, DIM)), (DIM,))


def _layer(case, dtype):
    layer = SparseFlashAttentionRope(DIM, num_heads=HEADS, qkv_bias=True, qk_norm=True, norm_layer=partial(nn.LayerNorm, eps=1e-6),
                                     rope=RoPE2D(freq=100.0), block_size=math.isqrt(case["block"]), topk=case["topk"])
    with torch.no_grad():
        nn.init.normal_(layer.gate[0].weight, std=0.02)   # a trained gate depends on the token
    return layer.to(dtype)


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    dtype, kind = DTYPES[case["dtype"]], case["kind"]
    state = {"case": case}
    if kind in ("op", "grad"):
        qkv = workloads.make_qkv_on_device(case["frames"], dtype, seed, True, DEV, HEADS, HEAD_DIM, case["gh"] * case["gw"] + case["reg"])
        state["qkv"] = qkv
        if kind == "op":
            state["gate"] = torch.sigmoid(torch.randn((1, HEADS, qkv[0].shape[2], 2), generator=gen, device=DEV)).to(dtype)
            return state
        with torch.no_grad():
            state["pooled"] = [pool_mean(t, case["block"]).requires_grad_() for t in qkv]
        state["qkv"] = [t.requires_grad_() for t in qkv]
        state["douts"] = [torch.randn(t.shape, generator=gen, device=DEV).to(dtype) for t in (state["pooled"][0], qkv[0])]
        return state
    torch.manual_seed(seed)
    with torch.device(DEV):
        if kind == "model":
            gh, gw = case["gh"], case["gw"]
            state["model"] = Pi3SparseLike(grid=(gh, gw), num_register=0, token_order="tile", block_tokens=case["block"],
                                           topk=case["topk"]).to(dtype).eval()
            smooth = torch.rand((case["frames"], 3, 16, 16), generator=gen, device=DEV)
            imgs = F.interpolate(smooth, size=(14 * gh, 14 * gw), mode="bilinear", align_corners=False)
            state["imgs"] = (0.9 * imgs + 0.1 * torch.rand(imgs.shape, generator=gen, device=DEV))[None]
            return state
        # mixed-precision training keeps fp32 weights and inputs, everything else runs in one type
        master = torch.float32 if case.get("autocast") else dtype
        layer = _layer(case, master)
    pos = _positions(case)
    x = _tokens(case, pos, gen).to(master)
    state.update(layer=layer, x=x, pos=pos, n_pos=max(case["gh"], case["gw"]) + 1 if case.get("bound") else None)
    if kind == "train":
        layer.train()
        x.requires_grad_()
        state["dout"] = torch.randn(x.shape, generator=gen, device=DEV).to(dtype)
        state["wrt"] = [x, *layer.parameters()]
    else:
        layer.eval()
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "op":
        with torch.no_grad():
            return sparse_global_attention(*state["qkv"], state["gate"], case["block"], case["topk"])
    if kind == "layer":
        with torch.no_grad():
            return state["layer"](state["x"], xpos=state["pos"], n_pos=state["n_pos"])
    if kind == "grad":
        q, k, v = state["qkv"]
        o_c, idx = flash_attn_topk_func(*state["pooled"], case["topk"])
        o = topk_blocksparse_attention(q, k, v, idx, case["block"])
        return o_c, o, *torch.autograd.grad((o_c, o), (*state["pooled"], q, k, v), state["douts"])
    if kind == "train":
        with torch.autocast("cuda", dtype=DTYPES[case["dtype"]], enabled=case["autocast"]):
            out = state["layer"](state["x"], xpos=state["pos"])
        return out.detach(), *torch.autograd.grad(out, state["wrt"], state["dout"])
    with torch.no_grad():
        return state["model"](state["imgs"])


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def work(case):
    es = DTYPES[case["dtype"]].itemsize
    per = case["gh"] * case["gw"] + case["reg"]
    n, b, block = case["frames"] * per, case["batch"], case["block"]
    nc = -(-n // block)
    seen = min(case["topk"] * block, n)
    attn = 4.0 * DIM * b * (n * seen + nc * nc)
    tokens = float(b * n * DIM * es)
    gates = 2.0 * n * HEADS * es
    kind = case["kind"]
    if kind == "op":
        return {"bytes": 4 * tokens + gates, "flops": attn}
    if kind == "grad":                                   # five products of the backward beside the two of the forward
        return {"bytes": (8 + 8 / block) * tokens, "flops": 3.5 * attn}
    weights = (4 * DIM + 2 * HEADS) * DIM
    gemm = 2.0 * b * n * weights
    if kind == "layer":
        return {"bytes": 2 * tokens + weights * es + 16.0 * b * n, "flops": gemm + attn}
    if kind == "train":
        wes = 4 if case["autocast"] else es
        return {"bytes": (2 * wes / es + 2) * tokens + 2.0 * weights * wes, "flops": 3 * gemm + 3.5 * attn}
    # model: 24 encoder blocks (class and 4 register tokens more per frame), 18 + 18 decoder blocks, 15 head blocks
    block_weights = 12 * DIM * DIM
    enc, dec = case["frames"] * (per + 5), n
    flops = 2.0 * block_weights * (24 * enc + 51 * dec) + 4.0 * DIM * (24 * enc * (per + 5) + 33 * dec * per) + 18 * attn
    flops += 2.0 * dec * DIM * (588 + 3 * 2 * DIM + 2.5 * DIM + 784)
    params = 75 * block_weights + DIM * (588 + 3 * 2 * DIM + 2.5 * DIM + 784)
    pixels = float(case["frames"] * per * 196)
    return {"bytes": params * es + pixels * 4 * (3 + 3 + 3 + 1), "flops": flops}


# relative 2-norm and largest errors of each kind against the same path in 64 bits on the same block choice (model: with
# its norms and pooling summed in another order), times four and rounded; at most 0.03.  The gradients of the operators
# carry the most: a row of dS sums to zero, so that most of dQ cancels for keys that share a component.
TOLERANCE = {
    ("op", "fp32"): {"rel": 2e-6, "max": 2e-5},       # measured 3.5e-7, 2.1e-6
    ("op", "bf16"): {"rel": 1e-2, "max": 5e-2},       # 2.7e-3, 1.1e-2
    ("op", "fp16"): {"rel": 1e-3, "max": 4e-3},       # 2.1e-4, 7.0e-4
    ("layer", "bf16"): {"rel": 1.6e-2, "max": 1e-1},  # 4.4e-3, 2.2e-2
    ("layer", "fp16"): {"rel": 2e-3, "max": 1.2e-2},  # 5.6e-4, 3.0e-3
    ("grad", "bf16"): {"rel": 3e-2, "max": 0.99},     # 4.6e-2, 6.9e-1 (64-token blocks), 2.8e-1, 4.5 (16-token blocks)
    ("grad", "fp16"): {"rel": 2.5e-2, "max": 4e-1},   # 6.2e-3, 8.9e-2
    ("train", "bf16"): {"rel": 3e-2, "max": 2.5e-1},  # 1.2e-2, 6.5e-2
    ("train", "fp16"): {"rel": 6e-3, "max": 4e-2},    # 1.7e-3, 1.0e-2
    ("model", "bf16"): {"rel": 2.8e-2, "max": 1.4e-1},  # 7.2e-3, 3.4e-2
}


def tolerance(case):
    return TOLERANCE[case["kind"], case["dtype"]]
