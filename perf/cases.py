"""The calls whose time counts: Pi0's decoder loop, prefix encoder, vision tower and whole
forward, through the entry points a program uses.

  decoder   Pi0DecoderEngine.forward against a prefix K/V cache
  encoder   Pi0EncoderEngine.forward (one request), or pipeline.transformer_encoder over the
            op table for several requests at once, call by call
  vision    pipeline.vision_encoder over the op table, recorded once as the engines record it
  forward   Pi0Inference.forward

The widths are the model's only ones (decoder 1024 / 4096, encoder 2048 / 16384, vision
1152 / 4304, 8 query heads and 1 KV head of 256); what varies in use is the number of
requests, camera views, prompt tokens and actions, and the depth of a stack.
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "flash-vla_amd"))

from flash_vla_amd import Pi0DecoderEngine, Pi0EncoderEngine, Pi0Inference, op_table, pipeline
from flash_vla_amd.arena import ScratchPool
from flash_vla_amd.backends.hip import use_pool
from flash_vla_amd.buffers import allocate_encoder_buffers
from flash_vla_amd.spec import decoder_weight_shapes, weight_shapes

DEV = "cuda"
HEADS, HD = 8, 256
VOCAB = 257152          # the prompt embedding table's rows


def listed() -> list[dict]:
    return [
        # the smallest call: one Euler step of a ten-action chunk with one camera, one layer
        # (bisection, a bring-up check): launches and latency
        _decoder("decoder small", batch=1, prefix=267, chunk=10, steps=1, layers=1),
        # a robot's control step: one request, three cameras, the whole denoising loop
        _decoder("decoder loop", batch=1, prefix=768, chunk=50, steps=10, layers=18),
        # the same with four cameras and a long instruction; 63 actions + state = 64 rows
        _decoder("decoder long prompt", batch=1, prefix=1221, chunk=63, steps=2, layers=6),
        # a server denoising four requests at once, each with its own 48-token prompt
        _decoder("decoder batch 4", batch=4, prefix=816, chunk=50, steps=10, layers=18),
        # the prefix of one camera and a short instruction
        _encoder("encoder one view", batch=1, tokens=269, layers=3, recorded=True),
        # the prefix of three cameras, full depth
        _encoder("encoder prefix", batch=1, tokens=768, layers=18, recorded=True),
        # the same with a 48-token instruction
        _encoder("encoder prompt 48", batch=1, tokens=816, layers=3, recorded=True),
        # four such prefixes at once, written call by call against the op table
        _encoder("encoder batch 4", batch=4, tokens=816, layers=2, recorded=False),
        # the vision tower of one robot, full depth
        _vision("vision 3 views", batch=1, views=3, layers=27),
        # ... and of four at once
        _vision("vision batch 4", batch=4, views=3, layers=3),
        # the whole model: one request without a prompt, and four with 48-token prompts
        _forward("forward", batch=1, views=3, prompt=0, chunk=50, steps=10),
        _forward("forward batch 4", batch=4, views=3, prompt=48, chunk=50, steps=10),
    ]


def _decoder(name, **kw):
    return {"name": name, "path": "decoder", **kw}


def _encoder(name, **kw):
    return {"name": name, "path": "encoder", **kw}


def _vision(name, **kw):
    return {"name": name, "path": "vision", **kw}


def _forward(name, **kw):
    return {"name": name, "path": "forward", **kw}


def _span(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _prompt(rng: random.Random) -> int:
    return rng.choice([0, _span(rng, 3, 200), _span(rng, 3, 200)])


def draw(rng: random.Random) -> dict:
    """Any depth and size of the listed stacks: 1 to 8 requests, 1, 3 or 4 views, prompts of
    0 to 200 tokens, chunks of 5 to 63 actions."""
    case = _any(rng)
    while any(case.items() <= c.items() for c in listed()):
        case = _any(rng)
    return case


def _any(rng: random.Random) -> dict:
    path = rng.choice(["decoder", "decoder", "encoder", "encoder", "vision"])
    batch = rng.choice([1, 1, _span(rng, 2, 8)])
    views = rng.choice([1, 3, 3, 4])
    tokens = views * 256 + _prompt(rng)
    if path == "decoder":
        chunk = _span(rng, 5, 63)
        return {"path": path, "batch": batch, "prefix": tokens, "chunk": chunk,
                "steps": rng.randint(1, 4), "layers": rng.randint(1, 6)}
    if path == "encoder":
        return {"path": path, "batch": batch, "tokens": tokens, "layers": rng.randint(2, 4),
                "recorded": batch == 1}
    return {"path": path, "batch": batch, "views": views, "layers": rng.randint(1, 12)}


# ---- inputs -----------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, *shape, std=1.0):
    return (torch.randn(*shape, generator=gen, device=DEV) * std).to(torch.bfloat16)


def _weights(shapes: dict, gen) -> dict:
    """N(0, 0.02) matrices and biases; LayerNorm scales around 1; the Euler out-projection
    with its dt = -0.1 folded in, as a converted checkpoint has it."""
    out = {}
    for name, shape in shapes.items():
        if name.endswith("norm_w"):
            out[name] = (1 + 0.1 * torch.randn(shape, generator=gen, device=DEV)).to(torch.bfloat16)
        else:
            std = 0.1 * 0.03 if name.startswith("decoder_action_fused_out") else 0.02
            out[name] = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
            for part in (out[name] if len(shape) == 3 else [out[name]]):   # a layer at a time
                part.copy_(torch.randn(part.shape, generator=gen, device=DEV) * std)
    return out


def _depth(shapes: dict, layers: int) -> dict:
    return {k: (layers, *s[1:]) if len(s) > 1 and s[0] in (18, 27) else s
            for k, s in shapes.items()}


def _inputs(case: dict, seed: int) -> tuple[dict, dict]:
    """(weights, inputs) of a case, from the seed alone."""
    gen = _gen(seed)
    path, B = case["path"], case["batch"]
    if path == "decoder":
        w = _weights(decoder_weight_shapes(case["layers"]), gen)
        lead = () if B == 1 else (B,)
        kv = (*lead, case["layers"], case["prefix"], HD)
        x = {"k": _randn(gen, *kv), "v": _randn(gen, *kv), "state": _randn(gen, B, 32),
             "noise": _randn(gen, B, case["chunk"], 32)}
    elif path == "encoder":
        shapes = {k: s for k, s in weight_shapes(0).items() if k in Pi0EncoderEngine.WEIGHTS}
        w = _weights(_depth(shapes, case["layers"]), gen)
        x = {"x": _randn(gen, B * case["tokens"], 2048)}
    elif path == "vision":
        shapes = {k: s for k, s in weight_shapes(0).items()
                  if k.startswith("vision") and "final" not in k}
        w = _weights(_depth(shapes, case["layers"]), gen)
        x = {"images": _images(gen, B * case["views"])}
    else:
        w = _weights(weight_shapes(0), gen)
        x = {"images": _images(gen, B * case["views"]), "state": _randn(gen, B, 32),
             "noise": _randn(gen, B, case["chunk"], 32)}
        if case["prompt"]:
            w["embed_tokens"] = _randn(gen, VOCAB, 2048, std=0.02)
            x["ids"] = torch.randint(0, VOCAB, (B, case["prompt"]), generator=gen, device=DEV,
                                     dtype=torch.int32)
    return w, x


def _images(gen, n: int):
    return (torch.rand(n, 224, 224, 3, generator=gen, device=DEV) * 2 - 1).to(torch.bfloat16)


# ---- what a program has in hand, and its call -------------------------------------------
def _record(call) -> torch.cuda.CUDAGraph:
    """Run `call` twice (packs its weights, fills its scratch pool), then record it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
        call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    return graph


def prepare(case: dict, seed: int) -> dict:
    w, x = _inputs(case, seed)
    path, B = case["path"], case["batch"]
    state = {"case": case, "in": x, "keep": w}
    if path == "decoder":
        state["engine"] = eng = Pi0DecoderEngine(
            w, encoder_seq_len=case["prefix"], chunk_size=case["chunk"], steps=case["steps"],
            layers=case["layers"], batch=B)
        eng.load_prefix(x["k"], x["v"])
    elif path == "forward":
        if case["prompt"]:
            w.pop("language_embeds", None)
        state["engine"] = Pi0Inference(w, num_views=case["views"], chunk_size=case["chunk"],
                                       steps=case["steps"], batch=B,
                                       prompt_tokens=case["prompt"])
        state["keep"] = None                       # the engine holds its own copy
    elif path == "encoder" and case["recorded"]:
        state["engine"] = Pi0EncoderEngine(w, encoder_seq_len=case["tokens"], copy_weights=False)
    else:
        state["ops"], state["pool"] = op_table(), ScratchPool()
        if path == "encoder":
            state["buffers"] = allocate_encoder_buffers(case["tokens"], DEV, batch=B,
                                                        layers=case["layers"])
            for _ in range(2):                     # packs the weights, fills the pool
                run(state)
        else:
            n = B * case["views"]
            state["buffers"] = {
                "observation_images_normalized": x["images"].clone(),
                "vision_x": _zeros(n, 256, 1152), "vision_x_norm": _zeros(n, 256, 1152),
                "vision_QKV": _zeros(n, 256, 3 * 1152), "vision_hidden": _zeros(n, 256, 4304)}
            state["graph"] = _record(lambda: _vision_call(state))
    return state


def _zeros(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16, device=DEV)


def _vision_call(state):
    with use_pool(state["pool"]):
        pipeline.vision_encoder(state["ops"], state["keep"], state["buffers"],
                                state["case"]["views"])


def run(state: dict):
    case, x = state["case"], state["in"]
    path, B = case["path"], case["batch"]
    if path == "decoder":
        eng = state["engine"]
        actions = eng.forward(x["state"], x["noise"])
        if case["layers"] == 18:                   # the whole loop: its result is the chunk
            return {"actions": actions}
        rows = slice(case["prefix"], None)
        return {"actions": actions, "k": eng.buffers["encoder_K"][..., rows, :],
                "v": eng.buffers["encoder_V"][..., rows, :]}
    if path == "forward":
        eng = state["engine"]
        actions = eng.forward(x["images"], x["state"], x["noise"], x.get("ids"))
        rows = slice(0, eng.encoder_seq_len)
        return {"actions": actions, "k": eng.buffers["encoder_K"][..., rows, :],
                "v": eng.buffers["encoder_V"][..., rows, :]}
    if path == "encoder":
        if case["recorded"]:
            k, v = state["engine"].forward(x["x"])
        else:
            b = state["buffers"]
            b["encoder_x"].copy_(x["x"])
            with use_pool(state["pool"]):
                pipeline.transformer_encoder(state["ops"], state["keep"], b, case["tokens"],
                                             project=False)
            k, v = b["encoder_K"], b["encoder_V"]
        return {"k": k, "v": v}
    state["buffers"]["observation_images_normalized"].copy_(x["images"])
    state["graph"].replay()
    return {"x": state["buffers"]["vision_x"]}


# ---- what a pass cannot do without ------------------------------------------------------
def work(case: dict) -> dict:
    """Weights and inputs read once, outputs written once -- except that the Euler steps run
    one after another and a full decoder's 623 MB of layer weights outgrow every cache, so
    each step reads them (and the prefix K/V) again."""
    path, B = case["path"], case["batch"]
    if path == "decoder":
        return _decoder_work(B, case["prefix"], case["chunk"], case["steps"], case["layers"])
    if path == "encoder":
        return _encoder_work(B, case["tokens"], case["layers"])
    if path == "vision":
        return _vision_work(B * case["views"], case["layers"])
    tokens = case["views"] * 256 + case["prompt"]
    parts = [_vision_work(B * case["views"], 27), _encoder_work(B, tokens, 18),
             _decoder_work(B, tokens, case["chunk"], case["steps"], 18)]
    M = B * case["views"] * 256
    parts.append({"bytes": 2 * 1152 * 2048, "flops": 2 * M * 1152 * 2048})
    return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}


def _decoder_work(B, prefix, chunk, steps, layers):
    M, keys = B * (chunk + 1), prefix + chunk + 1
    gemm = 1024 * 2560 + 2048 * 1024 + 3 * 1024 * 4096
    layer_bytes = 2 * gemm + 2 * 2 * B * HD * (prefix + 2 * (chunk + 1))
    layer_flops = 2 * M * gemm + 4 * M * HEADS * keys * HD
    small = 32 * 1024 + 1024 * 1024 + 1024 * 32
    return {"bytes": steps * (layers * layer_bytes + 2 * small) + 2 * 2 * B * chunk * 32,
            "flops": steps * (layers * layer_flops + 2 * B * chunk * small)}


def _encoder_work(B, tokens, layers):
    M = B * tokens
    qkv, rest = 2048 * 2560, 2048 * 2048 + 3 * 2048 * 16384
    return {"bytes": 2 * (layers * qkv + (layers - 1) * rest) + 2 * M * 2048
            + 2 * 2 * layers * M * HD,
            "flops": 2 * M * (layers * qkv + (layers - 1) * rest)
            + (layers - 1) * 4 * M * HEADS * tokens * HD}


def _vision_work(images, layers):
    M = images * 256
    gemm = 1152 * (3 * 1152 + 1152 + 2 * 4304)
    return {"bytes": 2 * (layers * gemm + 588 * 1152) + 2 * images * 224 * 224 * 3
            + 2 * M * 1152,
            "flops": 2 * M * (layers * gemm + 588 * 1152) + layers * 4 * M * 256 * 1152}


def tolerance(case: dict) -> dict:
    """bf16 activations between the calls of a layer, about 2e-3 a rounding, and a difference
    travels through all layers and steps that follow. Measured between two orders of the
    residual GEMMs' sums: encoder 1.9e-3 after 3 layers and 1.05e-2 after 18, decoder rows
    1e-2 after 12 layer passes and the chunk 1.3e-2 after 180."""
    if case["path"] == "forward":
        return {"rel": 0.03}
    if case["path"] == "decoder":
        return {"rel": min(0.03, 0.006 + 0.002 * case["steps"] * case["layers"])}
    return {"rel": min(0.03, 0.006 + 0.0015 * case["layers"])}


# ---- the same in 64 bits, plain torch ---------------------------------------------------
def exact(case: dict, seed: int):
    w, x = _inputs(case, seed)
    path, B = case["path"], case["batch"]
    x = {k: v if v.dtype == torch.int32 else v.double() for k, v in x.items()}
    if path == "decoder":
        outs = []
        for b in range(B):
            k, v = (x[n] if B == 1 else x[n][b] for n in ("k", "v"))
            outs.append(_decoder64(w, x["state"][b], x["noise"][b], k, v, case["steps"]))
        out = _join(outs, B)
        return {"actions": out["actions"]} if case["layers"] == 18 else out
    if path == "encoder":
        outs = [_encoder64(w, xb) for xb in x["x"].reshape(B, case["tokens"], 2048)]
        return {n: torch.stack([o[i] for o in outs]) if B > 1 else outs[0][i]
                for i, n in enumerate("kv")}
    if path == "vision":
        return {"x": _vision64(w, x["images"]).reshape(-1, 256, 1152)}
    outs = []
    for b in range(B):
        n = case["views"]
        vx = _vision64(w, x["images"][b * n:(b + 1) * n])
        px = _layer_norm(vx, w["vision_final_norm_w"], w["vision_final_norm_b"])
        px = px @ w["encoder_multi_modal_projector_w"].double() + \
            w["encoder_multi_modal_projector_b"].double()
        if case["prompt"]:
            emb = w["embed_tokens"][x["ids"][b].long()].double() * 2048 ** 0.5
            px = torch.cat([px, emb])
        K, V = _encoder64(w, px)
        out = _decoder64(w, x["state"][b], x["noise"][b], K, V, case["steps"])
        out["k"], out["v"] = K, V
        outs.append(out)
    return _join(outs, B)


def _join(outs: list, B: int) -> dict:
    return {"actions": torch.cat([o["actions"] for o in outs]),
            **{n: torch.stack([o[n] for o in outs]) if B > 1 else outs[0][n] for n in "kv"}}


def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _layer_norm(x, w, b):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w.double(), b.double(), 1e-5)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _rope(x, first):
    """Adjacent-pair rotation of [rows, n * 256] by the bf16 cos / sin table of the model."""
    rows = x.shape[0]
    freq = 10000.0 ** (-torch.arange(0, HD, 2, device=DEV, dtype=torch.float64) / HD)
    angle = torch.arange(first, first + rows, device=DEV, dtype=torch.float64)[:, None] * freq
    cos, sin = (t.bfloat16().double()[:, None] for t in (angle.cos(), angle.sin()))
    p = x.reshape(rows, -1, HD // 2, 2)
    a, b = p[..., 0], p[..., 1]
    return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).reshape(x.shape)


def _attend(q, k, v, state_keys=None):
    """One KV head, flat (token * heads + head) rows; the first token sees `state_keys` keys."""
    s = q @ k.t() / 16.0
    if state_keys is not None:
        s[:HEADS, state_keys:] = float("-inf")
    return torch.softmax(s, -1) @ v


def _qkv64(x, w, first):
    y = _rms(x) @ w.double()
    q, k, v = y.split([HEADS * HD, HD, HD], 1)
    return _rope(q, first).reshape(-1, HD), _rope(k, first), v


def _gemma64(x, o, w, pre, i):
    x = x + o.reshape(x.shape[0], -1) @ w[pre + "_attn_o_w"][i].double()
    r = _rms(x)
    h = _gelu(r @ w[pre + "_ffn_gate_w"][i].double()) * (r @ w[pre + "_ffn_up_w"][i].double())
    return x + h @ w[pre + "_ffn_down_w"][i].double()


def _encoder64(w, x):
    K, V = [], []
    n = w["encoder_attn_qkv_w"].shape[0]
    for i in range(n):
        q, k, v = _qkv64(x, w["encoder_attn_qkv_w"][i], 0)
        K.append(k)
        V.append(v)
        if i < n - 1:
            x = _gemma64(x, _attend(q, k, v), w, "encoder", i)
    return torch.stack(K), torch.stack(V)


def _decoder64(w, state, noise, K, V, steps):
    prefix = K.shape[1]
    W = {n: t.double() for n, t in w.items() if n.startswith("decoder_") and t.dim() < 3}
    s = state @ W["decoder_state_in_proj_w"] + W["decoder_state_in_proj_b"]
    for step in range(steps):
        h = torch.nn.functional.silu(noise @ W["decoder_action_fused_in_proj_w"]
                                     + W["decoder_action_fused_time_biases"][step % 10])
        x = torch.cat([s[None], h @ W["decoder_action_mlp_w"] + W["decoder_action_mlp_b"]])
        dk, dv = [], []
        for i in range(w["decoder_attn_qkv_w"].shape[0]):
            q, k, v = _qkv64(x, w["decoder_attn_qkv_w"][i], prefix)
            dk.append(k)
            dv.append(v)
            o = _attend(q, torch.cat([K[i].double(), k]), torch.cat([V[i].double(), v]), prefix + 1)
            x = _gemma64(x, o, w, "decoder", i)
        noise = noise + _rms(x[1:]) @ W["decoder_action_fused_out_proj_w"] \
            + W["decoder_action_fused_out_proj_b"]
    return {"actions": noise, "k": torch.stack(dk), "v": torch.stack(dv)}


def _vision64(w, images):
    n = images.shape[0]
    p = images.reshape(n, 16, 14, 16, 14, 3).permute(0, 1, 3, 2, 4, 5).reshape(n, 256, 588)
    x = p @ w["vision_patch_embedding_w"].double().reshape(588, 1152) \
        + w["vision_patch_embedding_b"].double() + w["vision_position_embedding"].double()
    x = x.reshape(n * 256, 1152)
    for i in range(w["vision_attn_qkv_w"].shape[0]):
        W = {k[7:]: t[i].double() for k, t in w.items()
             if k.startswith(("vision_attn", "vision_ffn", "vision_pre"))}
        r = _layer_norm(x, W["pre_attn_norm_w"], W["pre_attn_norm_b"])
        y = (r @ W["attn_qkv_w"] + W["attn_qkv_b"]).reshape(n, 256, 3, 16, 72)
        q, k, v = y.permute(2, 0, 3, 1, 4).reshape(3, n * 16, 256, 72)
        o = torch.softmax(q @ k.transpose(1, 2) / math.sqrt(72), -1) @ v
        o = o.reshape(n, 16, 256, 72).transpose(1, 2).reshape(n * 256, 1152)
        x = x + o @ W["attn_o_w"] + W["attn_o_b"]
        r = _layer_norm(x, W["pre_ffn_norm_w"], W["pre_ffn_norm_b"])
        x = x + _gelu(r @ W["ffn_up_w"] + W["ffn_up_b"]) @ W["ffn_down_w"] + W["ffn_down_b"]
    return x
