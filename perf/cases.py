"""The work this engine is used for, as cases that can be timed and compared.

A case is one call of a public entry point on inputs made from a seed:

* ``operator``: ``flash_attn_bsa_3d`` without gradients, what ``Attention._process_attn`` of the reference calls per
  layer and sampling step (longcat_video/modules/attention.py:58-67);
* ``train``: the same call with inputs that require a gradient, and its backward;
* ``module``: the attention sub-chain of a DiT block around the operator, plain (``attention_block_forward``), or the
  adaLN branch of a block (``dit_self_attention_branch``) with a conditioning split that keeps its k / v cache, or
  continuing from such a cache, with or without LoRA side branches on the two projections.

Grids, head counts, chunks and densities are those of the repository's benchmark (480p, 720p and long-video layers of 32
heads x 128, 4x4x4 chunks), of the operator's defaults (4x4x8 chunks, sparsity 0.875), of the plumbing configuration
(fp32, 256 tokens) and of what lies around them: a head-parallel share of a layer, previews, ragged grids.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "longcat-video_amd")      # the tree under the working folder, not this file's
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

from longcat_video_amd.block_sparse_attention.bsa_interface import flash_attn_bsa_3d      # noqa: E402
from longcat_video_amd.modules.attention import Attention, attention_block_forward, dit_self_attention_branch      # noqa: E402
from longcat_video_amd.modules.lora import LoRABranch      # noqa: E402

D = 128
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(name=None, path="operator", dtype="bf16", batch=1, heads=32, T=24, H=30, W=52, chunk_t=4, chunk_h=4, chunk_w=4,
          sparsity=0.9375, cdf=0.0, coherent=False, token_major=False, route="plain", cond=0, lora_rank=0):
    """cdf 0: the top-k rule alone.  coherent: queries and keys vary smoothly over the grid, as over real video, so that
    neighbouring query blocks select largely the same blocks; otherwise selections are random.  token_major: q, k, v are
    views of one [B, N, 3, heads, D] projection.  route, cond (latent frames) and lora_rank belong to modules."""
    c = dict(path=path, dtype=dtype, batch=batch, heads=heads, T=T, H=H, W=W, chunk_t=chunk_t, chunk_h=chunk_h, chunk_w=chunk_w,
             sparsity=sparsity, cdf=cdf, coherent=coherent, token_major=token_major, route=route, cond=cond, lora_rank=lora_rank)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest configuration of the engine: the fp32 plumbing check of a fresh installation, latency alone
        _case("plumbing_fp32", dtype="fp32", heads=4, T=4, H=8, W=8, sparsity=0.5),
        # a short low-resolution preview, two prompts at once, q / k / v as the projection leaves them: ragged in every axis
        _case("preview_bf16", batch=2, heads=8, T=7, H=15, W=26, sparsity=0.875, coherent=True, token_major=True),
        # the base resolution: one 480p layer of the benchmark
        _case("layer_480p_bf16", sparsity=0.9375, coherent=True),
        # one GPU's share of a 720p layer whose 32 heads are spread over eight GPUs
        _case("share_720p_bf16", heads=4, H=45, W=80),
        # the benchmark's headline layer: 720p, random selections
        _case("layer_720p_bf16", H=45, W=80),
        # the operator's default arguments (chunks of 4x4x8, an eighth of the blocks), fp16, a ragged grid
        _case("defaults_fp16", dtype="fp16", heads=16, T=13, H=30, W=53, chunk_w=8, sparsity=0.875),
        # selection by the share of the pooled softmax, never fewer than the top-k rule keeps: lists of unequal length
        _case("cdf_480p_bf16", heads=16, T=20, sparsity=0.9375, cdf=0.5, coherent=True),
        # fine-tuning at 480p: forward and backward of one layer
        _case("train_480p_bf16", path="train"),
        # fine-tuning on short, small clips in fp16: a ragged grid, few work items
        _case("train_clip_fp16", path="train", dtype="fp16", heads=6, T=9, H=17, W=30, sparsity=0.75),
        # the attention sub-chain of a DiT block at 720p: norm, projections, rotation, operator, residual
        _case("block_720p_bf16", path="module", H=45, W=80),
        # long video, first segment: the adaLN branch with conditioning frames of its own, keeping k and v for the next
        # segments, and the LoRA side branches of the distilled model
        _case("block_cond_lora_480p_bf16", path="module", T=21, route="cond", cond=4, lora_rank=128),
        # long video, next segment: the new frames attend to the cached keys and values and to their own
        _case("block_cached_480p_bf16", path="module", T=16, route="cached", cond=5),
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Grids from a few frames of thumbnails to 720p, 1 to 32 heads, the three paths and the options in use."""
    dearest = max(_cost(c) for c in listed())
    while True:
        path = rng.choice(("operator", "operator", "operator", "train", "module"))
        c = _case(path=path, batch=rng.choice((1, 1, 1, 2)), heads=_log_int(rng, 1, 32), T=rng.randint(2, 28),
                  H=_log_int(rng, 6, 48), W=_log_int(rng, 8, 84), chunk_w=rng.choice((4, 4, 4, 8)),
                  sparsity=rng.choice((0.5, 0.75, 0.875, 0.875, 0.9375, 0.9375)), coherent=rng.random() < 0.5,
                  token_major=rng.random() < 0.4)
        if path != "module":
            c["dtype"] = rng.choice(("bf16", "bf16", "bf16", "fp16"))
            if path == "operator" and rng.random() < 0.15:
                c["dtype"], c["token_major"] = "fp32", False
            elif rng.random() < 0.2:
                c["cdf"] = rng.choice((0.25, 0.5, 0.75))
        else:
            c["token_major"], c["coherent"] = False, False
            c["route"] = rng.choice(("plain", "cond", "cached"))
            if c["route"] != "plain":
                c["cond"] = rng.randint(1, 6)
                c["lora_rank"] = rng.choice((0, 0, 64, 128))
            c["heads"] = max(2, c["heads"])
            if c["route"] == "cond" and c["T"] <= c["cond"]:
                continue
        nq, nk = _blocks(c)
        if min(int((1 - c["sparsity"]) * n) for n in nk) < 1 or max(nk) > 4096:
            continue
        if c["dtype"] == "fp32" and c["batch"] * c["heads"] * c["T"] * c["H"] * c["W"] > 100_000:      # a cross-check's sizes
            continue
        # a row of the CDF rule may keep every block
        most = dict(c, sparsity=0.0) if c["cdf"] else c
        if _cost(most) <= dearest:
            return c


# ------------------------------------------------------------------------------------------------ what a pass has to do
def _calls(c):
    """(query frames, key frames) of every operator call of the case"""
    if c["route"] == "cond":
        return [(c["cond"], c["cond"]), (c["T"] - c["cond"], c["T"])]
    if c["route"] == "cached":
        return [(c["T"], c["T"] + c["cond"])]
    return [(c["T"], c["T"])]


def _blocks(c):
    n = lambda t: math.ceil(t / c["chunk_t"]) * math.ceil(c["H"] / c["chunk_h"]) * math.ceil(c["W"] / c["chunk_w"])      # noqa: E731
    return [n(q) for q, _ in _calls(c)], [n(k) for _, k in _calls(c)]


def _attention_flops(c):
    """One product of the attention over the selected pairs of real tokens (2 D a pair), all heads and operator calls.
    With the CDF rule: over the pairs that the top-k rule would keep, which the rule never goes below."""
    total, plane = 0.0, c["H"] * c["W"]
    for (tq, tk), nk in zip(_calls(c), _blocks(c)[1]):
        share = int((1 - c["sparsity"]) * nk) / nk
        total += 2.0 * D * (tq * plane) * (tk * plane) * share
    return total * c["batch"] * c["heads"]


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    dim = case["heads"] * D
    rows = case["batch"] * case["T"] * case["H"] * case["W"]
    one = rows * dim * es                                   # a tensor of the size of q
    product = _attention_flops(case)
    if case["path"] == "operator":
        return {"bytes": 4.0 * one, "flops": 2 * product}
    if case["path"] == "train":                             # q, k, v, dO in; o, dq, dk, dv out; 2 products and 5
        return {"bytes": 8.0 * one, "flops": 7 * product}
    weights = 4.0 * dim * dim * es
    flops = 2 * product + 8.0 * rows * dim * dim
    moved = 2.0 * one + weights
    if case["lora_rank"]:                                   # down and up on qkv (three slices of the rank axis) and proj
        flops += 2.0 * rows * case["lora_rank"] * dim * 8
        moved += 8.0 * case["lora_rank"] * dim * es
    cached = case["batch"] * case["cond"] * case["H"] * case["W"] * dim * es
    if case["route"] == "cond":
        moved += 2.0 * one                                  # the k and v cache of every frame
    elif case["route"] == "cached":
        moved += 2.0 * cached
    return {"bytes": moved, "flops": flops}


def _cost(c):
    w = work(c)
    return max(w["flops"] / 1e15, w["bytes"] / 6e12) * (16 if c["dtype"] == "fp32" else 1)


def tolerance(case):
    """About four times the distance (2-norm, largest) to the same path in fp64 from the same selection, as measured on the
    smaller cases: fp32 6.5e-7 and 3.4e-6; fp16 4.2e-4 and 3.4e-3; bf16 2.4e-3 and 0.010 forward, 3.5e-3 and 0.021 for the
    gradients.  Modules round their projections to bf16 as well."""
    if case["dtype"] == "fp32":
        return {"rel": 3e-6, "max": 3e-5}
    if case["dtype"] == "fp16":
        return {"rel": 1.7e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------------------------------------ inputs
def _rms(x):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)


def _qkv(c, g):
    """q and k RMS-normalised per head like the model's, v and their noise from N(0, 1)."""
    B, Hn, T, H, W, dt = c["batch"], c["heads"], c["T"], c["H"], c["W"], DTYPES[c["dtype"]]
    S = T * H * W
    pos = None
    if c["coherent"]:
        axes = [torch.arange(n, device="cuda", dtype=torch.float32) / 4 for n in (T, H, W)]
        pos = torch.stack([a.reshape(-1) for a in torch.meshgrid(*axes, indexing="ij")], 1)
    if c["token_major"]:
        q, k, v = torch.empty(B, S, 3, Hn, D, dtype=dt, device="cuda").permute(2, 0, 3, 1, 4).unbind(0)
    else:
        q, k, v = (torch.empty(B, Hn, S, D, dtype=dt, device="cuda") for _ in range(3))
    draw_ = lambda *s: torch.randn(*s, generator=g, device="cuda")      # noqa: E731
    for b in range(B):
        for h in range(Hn):
            field = 0.0
            if pos is not None:      # a field of random low spatial frequencies that queries and keys share
                phase = torch.rand(1, D, generator=g, device="cuda") * (2 * math.pi)
                field = torch.cos(pos @ (draw_(3, D) * 0.3) + phase) * math.sqrt(2)
            q[b, h] = _rms(draw_(S, D) + field)
            k[b, h] = _rms(draw_(S, D) + field)
            v[b, h] = draw_(S, D)
    return q, k, v


def _bsa_args(c):
    chunk = [c["chunk_t"], c["chunk_h"], c["chunk_w"]]
    return dict(sparsity=c["sparsity"], cdf_threshold=c["cdf"] or None, chunk_3d_shape_q=chunk, chunk_3d_shape_k=chunk)


def _module(c, g):
    dim, shape = c["heads"] * D, (c["T"], c["H"], c["W"])
    N = c["T"] * c["H"] * c["W"]
    new = lambda *s: torch.randn(*s, generator=g, device="cuda")      # noqa: E731
    with torch.device("cuda"):
        attn = Attention(dim, c["heads"], enable_bsa=True, bsa_params=_bsa_args(c)).to(torch.bfloat16)
    with torch.no_grad():
        for layer in (attn.qkv, attn.proj):
            for row in range(0, layer.weight.shape[0], dim):
                layer.weight[row:row + dim] = new(dim, dim) * dim ** -0.5
            layer.bias.copy_(new(layer.bias.shape[0]) * 0.02)
        for norm in (attn.q_norm, attn.k_norm):
            norm.weight.copy_(1 + 0.1 * new(D))
    if c["lora_rank"]:
        r = c["lora_rank"]
        bf = lambda *s: new(*s).mul_(s[-1] ** -0.5).bfloat16()      # noqa: E731
        attn.qkv_loras.append(LoRABranch(bf(3 * r, dim), [bf(dim, r) for _ in range(3)], 0.5))
        attn.proj_loras.append(LoRABranch(bf(r, dim), [bf(dim, r)], 0.5))
    s = {"attn": attn, "shape": shape, "x": torch.empty(c["batch"], N, dim, dtype=torch.bfloat16, device="cuda")}
    for b in range(c["batch"]):
        s["x"][b] = new(N, dim)
    if c["route"] == "plain":
        s["pre_norm"] = (1 + 0.1 * new(dim)).bfloat16()
    else:
        s["shift"], s["scale"], s["gate"] = (new(c["batch"], c["T"], 1, dim) * 0.3 for _ in range(3))
    if c["route"] == "cached":
        cache = (c["batch"], c["heads"], c["cond"] * c["H"] * c["W"], D)
        s["cache"] = (_rms(new(*cache)).bfloat16(), new(*cache).bfloat16())
    return s


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["path"] == "module":
        return dict(_module(case, g), case=case)
    q, k, v = _qkv(case, g)
    s = {"case": case, "q": q, "k": k, "v": v, "shape": (case["T"], case["H"], case["W"]), "args": _bsa_args(case)}
    if case["path"] == "train":
        s["q"], s["k"], s["v"] = (t.requires_grad_() for t in (q, k, v))
        s["do"] = torch.randn(q.shape, generator=g, device="cuda", dtype=torch.float32).to(q.dtype)
    return s


def run(state):
    c = state["case"]
    if c["path"] == "module":
        if c["route"] == "plain":
            return attention_block_forward(state["x"], state["pre_norm"], state["attn"], state["shape"])
        mod = (state["x"], state["shift"], state["scale"], state["gate"], state["attn"], state["shape"])
        if c["route"] == "cond":
            return dit_self_attention_branch(*mod, num_cond_latents=c["cond"], return_kv=True)
        return dit_self_attention_branch(*mod, num_cond_latents=c["cond"], kv_cache=state["cache"])
    o = flash_attn_bsa_3d(state["q"], state["k"], state["v"], state["shape"], state["shape"], **state["args"])
    if c["path"] == "train":
        return (o.detach(),) + torch.autograd.grad(o, (state["q"], state["k"], state["v"]), state["do"])
    return o
