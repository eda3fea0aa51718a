"""Workloads of the token-correction path, each through the entry points that a server program calls.

Five kinds of work, over the backbones, image sizes, batches, keep ratios and options of this repository's
configurations:

  correct  a correction pass over `depth` blocks (DINOv3ClassifierExecutor.correct_forward), either as the
           replay of a recorded pass (capture_correct_forward: how a latency-bound server runs it) or eager;
  crops    the batched correction of several crops with a score threshold and a fixed width
           (server.multicrop.correct_crops_batched): how a segmentation request is corrected;
  approx   the approximate pass that fills the K/V and residual caches and the server score
           (DINOv3ClassifierExecutor.approx_forward);
  score    the importance of a new frame's patches and the candidates it leaves (pixel residual RMS, pruning);
  nvfp4    an activation quantized to NVFP4 and back, as a client of the packed format does.

Weights, tokens and caches are random with the magnitudes the path meets: linears N(0, 0.02), tokens
N(0, 1), LayerScale 0.1 .. 0.5, keys and values as such linears give them, heavy-tailed patch scores.
"""

from __future__ import annotations

import math

import torch

from appcorr_amd import _lib
from appcorr_amd import kernels as K
from appcorr_amd.dinov3.backbone import dinov3_backbone
from appcorr_amd.server.dinov3_classifier import DINOv3ClassifierExecutor, make_group_plan
from appcorr_amd.server.multicrop import CropItem, correct_crops_batched
from appcorr_amd.server.protocol import ExperimentConfig

PRE = 5  # cls + 4 storage tokens
PATCH = 16

# embed dim, heads, MLP hidden size, SwiGLU, blocks of the whole model
MODELS = {
    "vits16": (384, 6, 1536, False, 12),
    "vitb16": (768, 12, 3072, False, 12),
    "vitl16": (1024, 16, 4096, False, 24),
    "vit7b16": (4096, 32, 8192, True, 40),
}
# Largest input magnitude each low-precision linear was calibrated for.
CALIBRATED = {"attn.qkv": 6.0, "attn.proj": 2.0, "mlp.w1": 6.0, "mlp.w2": 6.0, "mlp.w3": 16.0}


def listed():
    return [
        # A client's new frames: which patches of 16 images changed, and which stay candidates.
        {"name": "score_512_b16", "kind": "score", "batch": 16, "gh": 32, "gw": 32},
        # One small image, whole model, recorded: the latency of a single interactive request.
        correct("vits16_224_b1_pass", "vits16", 12, 1, 14, 14, 0.5, graph=True),
        # A few images of an odd shape (368 x 528), whole model, layer-mean server score plus the mobile hint.
        correct("vitb16_368x528_b3_pass", "vitb16", 12, 3, 23, 33, 0.5, server="patch_attn_prob_layermean",
                fusion="add", graph=True),
        # The benchmark's pass: ViT-L, 512 px, 16 images, the top quarter, whole model, recorded.
        correct("vitl16_512_b16_pass", "vitl16", 24, 16, 32, 32, 0.25, graph=True),
        # The default server score (one per layer, so one plan per layer) fused with the mobile hint; 4 blocks.
        correct("vitl16_512_b16_layer_plans", "vitl16", 4, 16, 32, 32, 0.25, server="cls_attn_prob",
                fusion="geo_mean", graph=True),
        # The largest model at 1024 px, keep 10 %, bf16, and the same with FP8 linears.
        correct("vit7b16_1024_b4_bf16", "vit7b16", 2, 4, 64, 64, 0.1),
        correct("vit7b16_1024_b4_fp8", "vit7b16", 2, 4, 64, 64, 0.1, precision="fp8"),
        # A segmentation request: two crops of 896 px, threshold selection at a fixed width, NVFP4 linears.
        crops("vit7b16_896_crops_fp4", "vit7b16", 1, 2, 56, 56, 0.5, "fp4"),
        # The approximate pass at its default score, and at the score of every query.
        approx("vitl16_512_b16_approx", "vitl16", 2, 16, 32, 32, "cls_attn_prob"),
        approx("vitl16_512_b16_approx_patch", "vitl16", 1, 16, 32, 32, "patch_attn_prob_layermean"),
        # The largest approximate pass: every token of four 1024 px images through a ViT-7B block.
        approx("vit7b16_1024_b4_approx", "vit7b16", 1, 4, 64, 64, "cls_attn_prob"),
        # Activations of the ViT-L MLP packed to NVFP4 and back.
        {"name": "nvfp4_16464x4096", "kind": "nvfp4", "rows": 16464, "cols": 4096},
    ]


def correct(name, backbone, depth, batch, gh, gw, keep, server="none", fusion="add", precision="bf16", graph=False):
    return {"name": name, "kind": "correct", "backbone": backbone, "depth": depth, "batch": batch, "gh": gh, "gw": gw,
            "keep": keep, "server": server, "fusion": fusion, "precision": precision, "graph": graph}


def crops(name, backbone, depth, batch, gh, gw, keep, precision):
    return {"name": name, "kind": "crops", "backbone": backbone, "depth": depth, "batch": batch, "gh": gh, "gw": gw,
            "keep": keep, "precision": precision}


def approx(name, backbone, depth, batch, gh, gw, server):
    return {"name": name, "kind": "approx", "backbone": backbone, "depth": depth, "batch": batch, "gh": gh, "gw": gw,
            "server": server}


def draw(rng):
    limit = max(_cost(c) for c in listed())
    while True:
        case = _draw_any(rng)
        if _cost(case) <= limit:
            del case["name"]
            return case


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 250)


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def _depth(rng, most, precision):
    """Blocks of a low-depth pass. NVFP4 steps are so coarse that one last-bit difference of an activation
    moves whole codes, which after two blocks is no longer the quantizer's own error: one block."""
    return 1 if precision == "fp4" else rng.randint(1, most)


def _draw_any(rng):
    kind = rng.choice(["correct", "correct", "correct", "correct", "approx", "approx", "crops", "score", "nvfp4"])
    if kind == "nvfp4":
        return {"name": "", "kind": "nvfp4", "rows": _log_int(rng, 100, 20000), "cols": 64 * _log_int(rng, 6, 128)}
    gh, gw = rng.randint(14, 64), rng.randint(14, 64)  # 224 .. 1024 px a side
    batch = _log_int(rng, 1, 16)
    if kind == "score":
        return {"name": "", "kind": "score", "batch": batch, "gh": gh, "gw": gw}
    backbone = rng.choice(["vits16", "vitb16", "vitl16", "vitl16", "vit7b16", "vit7b16"])
    if kind == "crops":
        backbone = rng.choice(["vitl16", "vit7b16"])
        gh = gw = rng.randint(24, 56)
        precision = rng.choice(["bf16", "fp4", "fp8"]) if backbone == "vit7b16" else "bf16"
        return crops("", backbone, _depth(rng, 2, precision), rng.randint(2, 4), gh, gw,
                     round(rng.uniform(0.2, 0.6), 3), precision)
    if kind == "approx":
        return approx("", backbone, rng.randint(1, 2), batch, gh, gw, rng.choice(
            ["cls_attn_prob", "cls_attn_prob", "patch_attn_prob_layermean", "patch_pseudo_attn_prob"]))
    precision = rng.choice(["bf16", "fp4", "fp8"]) if backbone == "vit7b16" else "bf16"
    server = rng.choice(["none", "none", "patch_attn_prob_layermean", "cls_attn_prob"])
    depth = _depth(rng, 2, precision) if backbone == "vit7b16" else rng.randint(2, 12)
    keep = rng.choice([0.1, 0.25, 0.5, 0.55, round(rng.uniform(0.03, 0.7), 3), round(rng.uniform(0.03, 0.7), 3)])
    return correct("", backbone, depth, batch, gh, gw, keep, server, rng.choice(["add", "geo_mean"]), precision,
                   graph=backbone != "vit7b16")


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without
# ------------------------------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "nvfp4":
        m, k = case["rows"], case["cols"]
        packed = m * k // 2 + m * k // 16
        return {"bytes": 2 * m * k + packed + packed + 2 * m * k, "flops": 0}
    P = case["gh"] * case["gw"]
    if kind == "score":
        return {"bytes": case["batch"] * (2 * P * PATCH * PATCH * 3 + P * 5), "flops": 0}
    B, L, N = case["batch"], case["depth"], PRE + P
    C, H, hid, swiglu, _ = MODELS[case["backbone"]]
    weights = 4 * C * C + (3 if swiglu else 2) * C * hid
    T = N if kind == "approx" else PRE + int(P * case["keep"])
    M = B * T
    flops = L * (2.0 * M * weights + 4.0 * B * T * N * C)
    size = {"fp8": 1, "fp4": 0.5625}.get(case.get("precision"), 2)
    nbytes = 4.0 * B * N * C + L * weights * size
    if kind == "approx":
        nbytes += L * B * N * (2 * C + C) * 2  # K, V and the residual sum, written
        if case["server"].startswith("patch_attn"):
            flops += L * 2.0 * B * N * N * C  # the probability of every (query, key)
    else:  # K and V read, their selected rows and the residual sum's written, the other rows' read
        nbytes += L * (B * N * 2 * C + M * 2 * C + B * N * C) * 2
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------------


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _gen(seed):
    return torch.Generator(device=_dev()).manual_seed(int(seed))


def _normal(gen, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=gen, device=gen.device).mul_(std).add_(mean).to(torch.bfloat16)


def _uniform(gen, shape, lo, hi, dtype=torch.bfloat16):
    return torch.rand(shape, generator=gen, device=gen.device).mul_(hi - lo).add_(lo).to(dtype)


def _block_weights(case, gen):
    """The blocks' parameters by the names of their state dict."""
    C, _, hid, swiglu, _ = MODELS[case["backbone"]]
    w = {}
    for i in range(case["depth"]):
        p = f"blocks.{i}."
        for n in ("norm1", "norm2"):
            w[p + n + ".weight"] = _uniform(gen, (C,), 0.8, 1.2)
            w[p + n + ".bias"] = _normal(gen, (C,), 0.05)
        for n in ("ls1", "ls2"):
            w[p + n + ".gamma"] = _uniform(gen, (C,), 0.1, 0.5)
        shapes = {"attn.qkv": (3 * C, C), "attn.proj": (C, C)}
        shapes.update({"mlp.w1": (hid, C), "mlp.w2": (hid, C), "mlp.w3": (C, hid)} if swiglu
                      else {"mlp.fc1": (hid, C), "mlp.fc2": (C, hid)})
        for n, s in shapes.items():
            w[p + n + ".weight"] = _normal(gen, s, 0.02)
            w[p + n + ".bias"] = _normal(gen, (s[0],), 0.02)
        if swiglu:  # the largest model has no qkv bias
            del w[p + "attn.qkv.bias"]
        else:
            mask = torch.ones(3 * C, device=gen.device, dtype=torch.bfloat16)
            mask[C:2 * C] = 0.0
            w[p + "attn.qkv.bias_mask"] = mask
    return w


def _tokens(case, gen):
    C = MODELS[case["backbone"]][0]
    return _normal(gen, (case["batch"], PRE + case["gh"] * case["gw"], C))


def _caches(case, gen, layers):
    """What an approximate pass left: K, V and the residual sum of every block, and its server score (a
    probability per key: positive, heavy-tailed, bf16 precision)."""
    C, H, _, _, _ = MODELS[case["backbone"]]
    B, N = case["batch"], PRE + case["gh"] * case["gw"]
    out = {}
    for i in range(layers):
        out[f"layer{i}_kv"] = _normal(gen, (B, N, 2, H, C // H), 0.02 * math.sqrt(C))
        out[f"layer{i}_blocks_out_sum"] = _normal(gen, (B, N, C), 0.3)
        s = torch.rand((B, N), generator=gen, device=gen.device).clamp_(1e-6, 1.0).log_().neg_().div_(N)
        out[f"layer{i}_server_pscore"] = s.to(torch.bfloat16).float()
    return out


def _hint(case, gen):
    """The mobile side's residual energy of each patch, normalised over the image."""
    e = torch.rand((case["batch"], case["gh"] * case["gw"]), generator=gen, device=gen.device).clamp_(1e-6, 1.0)
    e = e.log_().square_()
    return e / e.sum(dim=1, keepdim=True)


def _correct_inputs(case, seed):
    gen = _gen(seed)
    return _block_weights(case, gen), _tokens(case, gen), _caches(case, gen, case["depth"]), _hint(case, gen)


def _threshold(case, hint):
    """A score that about `keep` of the candidates reach, and a width that holds every image's kept ones."""
    thres = float(torch.quantile(hint.flatten()[:1 << 20], 1.0 - case["keep"]))
    most = int((hint >= thres).sum(dim=1).max())
    return thres, min(hint.shape[1], 32 * -(-most // 32))


def _executor(case, weights):
    """An executor around the case's blocks, configured as the server configures it."""
    dev = _dev()
    model = dinov3_backbone(case["backbone"], depth=case["depth"], device=dev, seed=None).eval()
    missing, unexpected = model.load_state_dict(weights, strict=False)
    if unexpected or any(m.startswith("blocks.") for m in missing):
        raise RuntimeError(f"block parameters do not match: {missing} {unexpected}")
    options = {"method": "partial_token"}
    if case["kind"] == "correct":
        options.update(token_keep_ratio=case["keep"], mobile_pscore="residual_energy", mobile_pscore_weight=1.0,
                       server_pscore=case["server"] if case["server"] != "none" else "cls_attn_prob",
                       server_pscore_weight=0.0 if case["server"] == "none" else 1.0,
                       pscore_fusion=case["fusion"] if case["server"] != "none" else "add")
    elif case["kind"] == "approx":
        options.update(server_pscore=case["server"], server_pscore_weight=1.0)
    config = ExperimentConfig(model_name=f"dinov3_classifier_{case['backbone']}", batch_size=case["batch"],
                              image_shape=(case["gh"] * PATCH, case["gw"] * PATCH, 3), backbone=case["backbone"],
                              correct_precision=case.get("precision", "bf16"), appcorr_kwargs=options)
    ex = DINOv3ClassifierExecutor(dev)
    ex.model = model
    ex.configure_dinov3_approx_precision(model, config)
    ex.configure_dinov3_correct_precision(model, config)
    if config.correct_precision != "bf16":  # the activation scales an earlier calibration found
        for blk in ex._dinov3_correct_precision.lowp_blocks:
            for name, mod in blk.named_modules():
                if name in CALIBRATED:
                    mod.amax.fill_(CALIBRATED[name])
                    mod.freeze_activation_scale()
    return ex, config, model.rope_embed(H=case["gh"], W=case["gw"])


def _candidates(case):
    N = PRE + case["gh"] * case["gw"]
    return torch.arange(N, device=_dev()).unsqueeze(0).expand(case["batch"], -1).contiguous()


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "score":
        prev, curr = _frames(case, _gen(seed))
        P = case["gh"] * case["gw"]
        spatial = torch.arange(P, device=_dev()).unsqueeze(0).expand(case["batch"], -1).contiguous()
        return {"case": case, "prev": prev, "curr": curr, "spatial": spatial}
    if kind == "nvfp4":
        x, ts = _activation(case, _gen(seed))
        return {"case": case, "x": x, "ts": ts}
    if kind == "approx":
        gen = _gen(seed)
        ex, config, rope = _executor(case, _block_weights(case, gen))
        ctx = {"input_tokens": _tokens(case, gen), "rope_sincos": rope}
        return {"case": case, "ex": ex, "config": config, "ctx": ctx, "params": {"layers": (0, case["depth"])}}
    weights, x, caches, hint = _correct_inputs(case, seed)
    ex, config, rope = _executor(case, weights)
    if kind == "crops":
        thres, cap = _threshold(case, hint)
        dind = _candidates(case)
        return {"case": case, "ex": ex, "x": x, "caches": caches, "hint": hint, "rope": rope, "dind": dind,
                "options": {"appcorr_method": "partial_token", "token_keep_thres": thres, "token_keep_cap": cap,
                            "mobile_pscore": "residual_energy", "mobile_pscore_weight": 1.0,
                            "server_pscore": "cls_attn_prob", "server_pscore_weight": 0.0, "num_pretokens": PRE}}
    ctx = {"input_tokens": x, "rope_sincos": rope, "mobile_pscore_hint_map": hint, "cache_feature": caches,
           "group_plans": {1: make_group_plan(_candidates(case), PRE)}}
    st = {"case": case, "ex": ex, "config": config, "ctx": ctx, "caches": dict(caches),
          "params": {"layers": (0, case["depth"]), "group_id": 1}}
    if case["graph"]:
        st["replay"] = ex.capture_correct_forward(st["params"], ctx, config)
    return st


def _frames(case, gen):
    """The previous decoded frames and the new ones: most patches move by a few levels, some by many."""
    B, gh, gw = case["batch"], case["gh"], case["gw"]
    prev = torch.randint(0, 256, (B, gh * PATCH, gw * PATCH, 3), generator=gen, device=gen.device, dtype=torch.int16)
    amp = torch.rand((B, gh, 1, gw, 1, 1), generator=gen, device=gen.device).pow_(3).mul_(60.0)
    step = torch.randn((B, gh, PATCH, gw, PATCH, 3), generator=gen, device=gen.device) * amp
    curr = (prev.float() + step.view(prev.shape)).round_().clamp_(0, 255)
    return prev.to(torch.uint8), curr.to(torch.uint8)


def _activation(case, gen):
    """N(0, 1) with one value in a hundred fifty times as large, and its per-tensor scale."""
    m, k = case["rows"], case["cols"]
    x = torch.randn((m, k), generator=gen, device=gen.device)
    x = torch.where(torch.rand((m, k), generator=gen, device=gen.device) < 0.01, x * 50.0, x).to(torch.bfloat16)
    return x, x.abs().max().float() / (448.0 * 6.0)


PRUNE_RMS, PRUNE_MIN = 8.0, 16


@torch.no_grad()
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "score":
        rms = K.patch_residual_score(st["curr"], st["prev"], (PATCH, PATCH), _lib.IMPORTANCE_RMS)
        pk = K.residual_prune_keep(rms, st["spatial"], PRUNE_RMS, PRUNE_MIN)
        return {"rms": rms, "keep": pk.keep, "count": pk.kept_count, "kept": pk.kept_mass, "full": pk.full_mass}
    if kind == "nvfp4":
        q, s = K.quantize_nvfp4_swizzled(st["x"], st["ts"])
        return {"codes": q, "scales": s.view(torch.uint8), "values": K.dequantize_nvfp4(q, s, st["ts"])}
    if kind == "approx":
        ctx = dict(st["ctx"])  # a request's own context: its caches are new tensors
        st["ex"].approx_forward(st["params"], ctx, st["config"])
        c = ctx["cache_feature"]
        keys = [f"layer{i}_{n}" for i in range(case["depth"]) for n in ("kv", "blocks_out_sum", "server_pscore")]
        return {"x": ctx["current_feature"], **{k: c[k] for k in keys}}
    if kind == "crops":
        items = []
        for b in range(case["batch"]):
            cache = {k: v[b:b + 1] for k, v in st["caches"].items()}
            items.append(CropItem(input_tokens=st["x"][b:b + 1], dindice=st["dind"][b:b + 1], num_pre=PRE, cache=cache,
                                  rope=st["rope"], mobile_pscore_hint=st["hint"][b:b + 1]))
        st["ex"].begin_dinov3_correct_event()
        xs = correct_crops_batched(st["ex"].run_dinov3_correct_block, items, 0, case["depth"], **st["options"])
        return {"x": list(xs), "caches": [{k: it.cache[k] for k in _updated(case)} for it in items]}
    ctx = st["ctx"]
    if case["graph"]:
        st["replay"]()
    else:
        ctx["cache_feature"] = dict(st["caches"])  # the tensors of this request's caches, no plan yet
        st["ex"].correct_forward(st["params"], ctx, st["config"])
    return {"x": ctx["current_feature"], **{k: ctx["cache_feature"][k] for k in _updated(case)}}


def _updated(case):
    """The caches a correction returns beside the tokens: those of the first and of the last block."""
    return [f"layer{i}_{n}" for i in sorted({0, case["depth"] - 1}) for n in ("kv", "blocks_out_sum")]


# ------------------------------------------------------------------------------------------------
# The same in 64 bits
# ------------------------------------------------------------------------------------------------


def tolerance(case):
    """About four times what the path is off the 64-bit values of exact(): bf16 0.002 .. 0.008, FP8 0.03
    (codes 1/16 apart that flip with the last bit of an activation), NVFP4 0.08 (codes 1/4 .. 1/2 apart)."""
    kind = case["kind"]
    if kind == "nvfp4":
        return "exact"
    if kind == "score":
        return {"rel": 5e-7, "differ": 0.0}
    return {"rel": {"fp4": 0.3, "fp8": 0.12}.get(case.get("precision"), 0.03)}


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "score":
        return _exact_score(case, seed)
    if kind == "nvfp4":
        x, ts = _activation(case, _gen(seed))
        return {"codes": None, "scales": None, "values": _nvfp4(x, ts) * ts.double()}
    return _exact_approx(case, seed) if kind == "approx" else _exact_correct(case, seed)


def _exact_score(case, seed):
    prev, curr = _frames(case, _gen(seed))
    B, gh, gw = case["batch"], case["gh"], case["gw"]
    d = (curr.double() - prev.double()).view(B, gh, PATCH, gw, PATCH * 3)
    rms = d.square().mean(dim=(2, 4)).sqrt().view(B, gh * gw)
    keep = rms >= PRUNE_RMS
    keep.scatter_(1, rms.topk(min(PRUNE_MIN, gh * gw), dim=1).indices, True)
    return {"rms": rms, "keep": None, "count": None, "kept": (rms * keep).sum(dim=1), "full": rms.sum(dim=1)}


def _e4m3(v):
    return v.float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double()


def _nvfp4(x, ts):
    """e2m1 codes times their e4m3 block scales, without the tensor scale."""
    m, k = x.shape
    b = x.float().view(m, k // 16, 16)
    amax = b.abs().amax(dim=2, keepdim=True)
    s = (amax.double() / 6.0).float()
    s = _e4m3((s.double() / ts.double()).float().clamp(min=1.5258789e-05)).float()
    q = (b.double() / (ts.float() * s).double()).float()
    a = q.abs()
    up = [a > 0.25, a >= 0.75, a > 1.25, a >= 1.75]  # 0.5 a step up to 2, ties to the even code
    v = sum(u.to(torch.float32) for u in up) * 0.5
    v = v + (a > 2.5).float() + (a >= 3.5).float() + (a > 5.0).float() * 2.0
    return (v.copysign(q) * s).view(m, k).double()


def _linear(case, w, block, name, x, like=None):
    """One linear of a block on its route; a low-precision route quantizes the bf16 activation. `like`: the
    linear whose activation scale the quantizer takes (w2 shares w1's operand)."""
    weight, bias = w[f"blocks.{block}.{name}.weight"], w.get(f"blocks.{block}.{name}.bias")
    mask = w.get(f"blocks.{block}.{name}.bias_mask")
    bias = None if bias is None else (bias.double() if mask is None else bias.double() * mask.double())
    route = case.get("precision", "bf16")
    amax = torch.tensor(CALIBRATED.get(name, 0.0), device=x.device)
    if route == "bf16":
        y = x @ weight.double().T
    elif route == "fp8" or name == "attn.proj":
        ws = weight.abs().max().float() / 448.0
        wq = _e4m3((weight / ws.to(torch.bfloat16)).float())
        sa = amax / 448.0
        xq = _e4m3(x.to(torch.bfloat16).float() * (1.0 / sa).to(torch.bfloat16).float())
        y = (xq @ wq.T) * (sa * ws).double()
    else:
        ws = weight.abs().max().float() / (448.0 * 6.0)
        sa = torch.tensor(CALIBRATED[like or name], device=x.device) / (448.0 * 6.0)
        scale = (amax / (448.0 * 6.0) * ws).to(torch.bfloat16).double()
        y = (_nvfp4(x.to(torch.bfloat16), sa) @ _nvfp4(weight, ws).T) * scale
    return y if bias is None else y + bias


def _norm(w, block, name, x):
    p = f"blocks.{block}.{name}."
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w[p + "weight"].double(), w[p + "bias"].double(), 1e-5)


def _rope_tables(case):
    C, H, _, _, _ = MODELS[case["backbone"]]
    q = C // H // 4
    dev = _dev()
    periods = (100.0 ** (2 * torch.arange(q, device=dev, dtype=torch.float32) / (2 * q))).to(torch.bfloat16).double()
    ch = (torch.arange(case["gh"], device=dev, dtype=torch.float64) + 0.5) / case["gh"]
    cw = (torch.arange(case["gw"], device=dev, dtype=torch.float64) + 0.5) / case["gw"]
    at = torch.stack(torch.meshgrid(ch, cw, indexing="ij"), dim=-1).flatten(0, 1) * 2.0 - 1.0
    angle = (2 * math.pi * at[:, :, None] / periods).flatten(1, 2).tile(2)
    return angle.sin(), angle.cos()


def _rotate(v, sin, cos, token):
    """v [B, T, H, D] at the tokens [B, T]; the first PRE tokens of an image are not patches."""
    half = v.shape[-1] // 2
    patch = (token >= PRE)[:, :, None, None]
    at = (token - PRE).clamp_min(0)
    r = v * cos[at][:, :, None] + torch.cat([-v[..., half:], v[..., :half]], dim=-1) * sin[at][:, :, None]
    return torch.where(patch, r, v)


def _attention(q, k, v, each=None):
    """q [B, T, H, D], k / v [B, N, H, D] -> [B, T, H, D]; each(b, h, p): sees every head's [T, N] weights."""
    out = torch.empty_like(q)
    scale = q.shape[-1] ** -0.5
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            p = torch.softmax((q[b, :, h] @ k[b, :, h].T) * scale, dim=-1)
            out[b, :, h] = p @ v[b, :, h]
            if each is not None:
                each(b, h, p)
    return out


def _mlp(case, w, i, x):
    if not MODELS[case["backbone"]][3]:
        return _linear(case, w, i, "mlp.fc2", torch.nn.functional.gelu(_linear(case, w, i, "mlp.fc1", x)))
    gate = torch.nn.functional.silu(_linear(case, w, i, "mlp.w1", x))
    return _linear(case, w, i, "mlp.w3", gate * _linear(case, w, i, "mlp.w2", x, like="mlp.w1"))


def _exact_approx(case, seed):
    gen = _gen(seed)
    w = _block_weights(case, gen)
    x = _tokens(case, gen).double()
    B, N, C = x.shape
    H = MODELS[case["backbone"]][1]
    sin, cos = _rope_tables(case)
    token = _candidates(case)
    out = {}
    for i in range(case["depth"]):
        qkv = _linear(case, w, i, "attn.qkv", _norm(w, i, "norm1", x)).view(B, N, 3, H, C // H)
        q, k, v = _rotate(qkv[:, :, 0], sin, cos, token), _rotate(qkv[:, :, 1], sin, cos, token), qkv[:, :, 2]
        score = torch.zeros((B, N), device=x.device, dtype=torch.float64)

        def each(b, h, p):
            if case["server"].startswith("cls"):
                score[b] += p[0] / H
            elif case["server"].startswith("patch_attn"):
                score[b] += p.mean(dim=0) / H

        attn = _attention(q, k, v, each)
        if case["server"].startswith("patch_pseudo"):
            qp = q[:, PRE:]
            mean = qp.mean(dim=1)
            target = qp.norm(dim=-1).mean(dim=1, keepdim=False)
            mean = mean * (target / mean.norm(dim=-1).clamp_min(2.0 ** -7))[..., None]
            s = (k * mean[:, None]).sum(dim=-1) * (C // H) ** -0.5  # [B, N, H]
            score = torch.softmax(s, dim=1).mean(dim=2)
        inc = w[f"blocks.{i}.ls1.gamma"].double() * _linear(case, w, i, "attn.proj", attn.view(B, N, C))
        xa = x + inc
        mlp = w[f"blocks.{i}.ls2.gamma"].double() * _mlp(case, w, i, _norm(w, i, "norm2", xa))
        out.update({f"layer{i}_kv": torch.stack([k, v], dim=2), f"layer{i}_blocks_out_sum": inc + mlp,
                    f"layer{i}_server_pscore": score})
        x = xa + mlp
    return {"x": x, **out}


def _selected(case, hint, caches, layer):
    """The selected tokens of every image [B, T], by the fp32 scores that the plan compares."""
    if case["kind"] == "crops":
        thres, cap = _threshold(case, hint)
        keep = hint >= thres
        rows = []
        for b in range(hint.shape[0]):
            at = keep[b].nonzero().flatten()
            last = at[-1:] if at.numel() else at.new_zeros(1)
            rows.append(torch.cat([at, last.expand(cap - at.numel())]))
        pick = torch.stack(rows)
    else:
        s = hint
        if case["server"] != "none":
            if case["server"].endswith("_layermean"):
                server = torch.stack([caches[f"layer{i}_server_pscore"] for i in range(case["depth"])]).mean(dim=0)
            else:
                server = caches[f"layer{layer}_server_pscore"]
            s = server[:, PRE:] + hint if case["fusion"] == "add" else (server[:, PRE:] * hint).clamp_min(0).sqrt()
        k = int(s.shape[1] * case["keep"])
        pick = torch.sort(s, dim=1, descending=True, stable=True).indices[:, :k].sort(dim=1).values
    pre = torch.arange(PRE, device=hint.device).expand(hint.shape[0], -1)
    return torch.cat([pre, pick + PRE], dim=1)


def _exact_correct(case, seed):
    w, x, caches, hint = _correct_inputs(case, seed)
    x = x.double()
    B, N, C = x.shape
    H = MODELS[case["backbone"]][1]
    sin, cos = _rope_tables(case)
    img = torch.arange(B, device=x.device)[:, None]
    out = {}
    for i in range(case["depth"]):
        token = _selected(case, hint, caches, i)
        T = token.shape[1]
        xs = x[img, token]
        qkv = _linear(case, w, i, "attn.qkv", _norm(w, i, "norm1", xs).view(-1, C)).view(B, T, 3, H, C // H)
        kv = caches[f"layer{i}_kv"].double()
        kv[img, token] = torch.stack([_rotate(qkv[:, :, 1], sin, cos, token), qkv[:, :, 2]], dim=2)
        attn = _attention(_rotate(qkv[:, :, 0], sin, cos, token), kv[:, :, 0], kv[:, :, 1]).view(-1, C)
        inc = w[f"blocks.{i}.ls1.gamma"].double() * _linear(case, w, i, "attn.proj", attn).view(B, T, C)
        mlp = _mlp(case, w, i, _norm(w, i, "norm2", xs + inc).view(-1, C)).view(B, T, C)
        inc = inc + w[f"blocks.{i}.ls2.gamma"].double() * mlp
        bos = caches[f"layer{i}_blocks_out_sum"].double()
        bos[img, token] = inc
        x = x + bos
        out.update({f"layer{i}_kv": kv, f"layer{i}_blocks_out_sum": bos})
    if case["kind"] == "crops":
        return {"x": [x[b:b + 1] for b in range(B)],
                "caches": [{k: out[k][b:b + 1] for k in _updated(case)} for b in range(B)]}
    return {"x": x, **{k: out[k] for k in _updated(case)}}
