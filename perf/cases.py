"""What this framework is timed on: the work its users have it do, through its public modules.

    PyramidSparseAttention      the attention of a video diffusion transformer under a preset of attention_config.yaml
                                (sparse steps, and the dense warm-up steps that open every sampling run)
    PSAAttention                the plug-in module: inference with its default settings, and fine-tuning (forward + backward)
    PyramidAdaptiveBlockSparseAttnTrain   the causal module of a vision-language decoder with grouped-query attention

A case is a dict of plain values.  Sequence lengths come from the video grids of the presets, from the benchmark's workloads
and from the tests; the drawn cases spread over the ranges between them.
"""
import math
import os
import sys

import torch

# (the working folder is the root of the tree that is measured)
sys.path.insert(0, os.path.join(os.getcwd(), "pyramid-sparse-attention_amd"))

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# Level quotas used below.  DEFAULT: PSAConfig's own; BOUND90: the Wan2.1 1.3B threshold preset scaled to the benchmark's
# about 90 % sparsity, BOUND85 to the training workload's about 85 %, BOUND80 to the small layer's and the decoder's about 80 %.
WAN = {1: (0.0, 0.5), 2: (0.5, 0.6), 4: (0.6, 0.7), 8: (0.7, 0.8), 0: (0.8, 1.0)}


def _scaled(tau):
    return {lv: (lo * tau if lv else 0.8 * tau, hi * tau if lv else 1.0) for lv, (lo, hi) in WAN.items()}


RATIOS = {
    "default": {1: (0.0, 0.1), 2: (0.1, 0.15), 4: (0.15, 0.15), 8: (0.15, 0.35), 0: (0.35, 1.0)},
    "bound90": _scaled(0.42),
    "bound85": _scaled(0.55),
    "bound80": _scaled(0.62),
}

# The presets a sampling run is started with, as (heads, head dim, text tokens, pixels / frames per latent token, about
# the density its map ends at).  Where a preset fixes quotas the density follows from them; where it bounds the
# attention mass the figure is what the synthetic fields of prepare() give.
PRESETS = {
    "Wan2.1_1.3b/psa_balanced": dict(heads=12, dim=128, text=0, step=(16, 16, 4), density=0.25),
    "Wan2.1_1.3b/psa_topk": dict(heads=12, dim=128, text=0, step=(16, 16, 4), density=0.1),
    "Wan2.1_14b/psa_balanced": dict(heads=40, dim=128, text=0, step=(16, 16, 4), density=0.2),
    "Wan2.2_5B/psa_balanced": dict(heads=24, dim=128, text=0, step=(32, 32, 4), density=0.25),
    "Wan2.2_A14B/psa_balanced": dict(heads=40, dim=128, text=0, step=(16, 16, 4), density=0.2),
    "CogVideo1.5_5b/psa_balanced": dict(heads=48, dim=64, text=226, step=(16, 16, 8), density=0.15),
    "CogVideo_5b/psa_balanced": dict(heads=48, dim=64, text=226, step=(16, 16, 4), density=0.15),
    "CogVideo_5b/psa_4steps": dict(heads=48, dim=64, text=226, step=(16, 16, 4), density=0.16),
}


def listed():
    return [
        # The smallest call: the plug-in module with its default settings on a short ragged sequence; launches and host work.
        dict(name="plug-in short", kind="plug", B=1, H=8, L=1000, D=64, block_n=64, ratios="default", mode="topk", dtype="bf16"),
        # A small fp32 layer (the benchmark's small workload): every stage computes in fp32.
        dict(name="plug-in fp32", kind="plug", B=1, H=2, L=4096, D=64, block_m=64, block_n=64, tile_n=16, ratios="bound80",
             mode="thresholdbound", dtype="fp32"),
        # The plug-in module with its default settings at an ordinary size, half precision, ragged length.
        dict(name="plug-in fp16", kind="plug", B=2, H=16, L=8200, D=128, block_n=64, ratios="default", mode="topk", dtype="fp16"),
        # Wan2.1 1.3B at 832 x 480, 81 frames: a sparse step under the preset with the similarity cap and the token re-ordering.
        dict(name="video 128-token blocks", kind="video", preset="Wan2.1_1.3b/psa_balanced", B=1, H=12, width=52, height=30, depth=21,
             D=128, dtype="bf16"),
        # The same model under its fixed-quota preset with 32-token kv-blocks.
        dict(name="video 32-token blocks", kind="video", preset="Wan2.1_1.3b/psa_topk", B=1, H=12, width=52, height=30, depth=21,
             D=128, dtype="bf16"),
        # The dense warm-up steps (15 of 50 under that model's presets).
        dict(name="video warm-up step", kind="dense", preset="Wan2.1_1.3b/psa_balanced", B=1, H=12, width=52, height=30, depth=21,
             D=128, dtype="bf16"),
        # CogVideoX-5B, guidance batch of 2, 720 x 480, 49 frames, joint text + video tokens, head dim 64, the 4-step preset.
        dict(name="video and text head dim 64", kind="video", preset="CogVideo_5b/psa_4steps", B=2, H=48, width=45, height=30, depth=13,
             D=64, dtype="bf16"),
        # CogVideoX1.5-5B at 1360 x 768, 81 frames: the longest sequence, 32-token kv-blocks, head dim 64.
        dict(name="long video head dim 64", kind="video", preset="CogVideo1.5_5b/psa_balanced", B=1, H=48, width=85, height=48, depth=11,
             D=64, dtype="bf16"),
        # One fine-tuning step of the attention layer at the Wan2.1 1.3B shape (the benchmark's training workload).
        dict(name="training", kind="train", B=1, H=12, L=32760, D=128, ratios="bound85", mode="thresholdbound", dtype="bf16"),
        # The same for a head-dim-64 model and a shorter clip, fixed quotas (tuning for the 4-step preset).
        dict(name="training head dim 64", kind="train", B=1, H=48, L=8776, D=64, ratios="default", mode="topk", dtype="bf16"),
        # Prefill of a vision-language decoder (28 query heads on 4 kv heads), 1024 text tokens before a long video.
        dict(name="causal prefill", kind="causal", B=1, H=28, Hkv=4, L=32768, D=128, text=1024, stride=8, ratios="bound80",
             mode="energybound", dtype="bf16"),
        # Prefill of the same decoder on one picture: a short ragged prompt.
        dict(name="causal prefill short", kind="causal", B=1, H=28, Hkv=4, L=2345, D=128, text=512, stride=8, ratios="bound80",
             mode="energybound", dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["plug", "plug", "fp32", "video", "video", "video", "dense", "train", "train", "causal", "causal"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "fp32":
        block = rng.choice([64, 64, 128])
        return dict(kind="plug", B=1, H=rng.choice([1, 2, 4, 8]), L=_log(rng, 700, 6000), D=64, block_m=block, block_n=64, tile_n=16,
                    ratios=rng.choice(["bound80", "bound90"]), mode="thresholdbound", dtype="fp32")
    if kind == "plug":
        mode = rng.choice(["topk", "topk", "thresholdbound"])
        return dict(kind="plug", B=rng.choice([1, 1, 2]), H=rng.choice([8, 12, 16, 24]), L=_log(rng, 900, 20000), D=rng.choice([64, 128]),
                    block_n=rng.choice([32, 64, 64, 128]), ratios="default" if mode == "topk" else "bound90", mode=mode, dtype=dtype)
    if kind in ("video", "dense"):
        preset = rng.choice(sorted(PRESETS))
        p = PRESETS[preset]
        tokens = _log(rng, 3000, 32760 if kind == "dense" else 45000)
        depth = rng.randint(5, 21)
        width = max(8, int(round(math.sqrt(tokens / depth * 1.7))))
        return dict(kind=kind, preset=preset, B=rng.choice([1, 2]), H=p["heads"], width=width, height=max(6, tokens // (depth * width)),
                    depth=depth, D=p["dim"], dtype=dtype)
    if kind == "train":
        mode = rng.choice(["topk", "thresholdbound"])
        return dict(kind="train", B=rng.choice([1, 1, 2]), H=rng.choice([8, 12, 16, 24, 48]), L=_log(rng, 2000, 32760), D=rng.choice([64, 128]),
                    ratios="default" if mode == "topk" else "bound85", mode=mode, dtype=dtype)
    mode = rng.choice(["topk", "energybound"])
    heads, kv = rng.choice([(28, 4), (28, 4), (16, 2), (12, 12)])
    return dict(kind="causal", B=1, H=heads, Hkv=kv, L=_log(rng, 1500, 32768), D=128, text=rng.choice([0, 512, 1024]),
                stride=rng.choice([8, 8, 16]), ratios="default" if mode == "topk" else "bound80", mode=mode, dtype="bf16")


def _price(case):
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / (20e12 if case["dtype"] == "fp32" else 1e15))


def draw(rng):
    """One more case of the same ranges; no dearer than the largest listed one."""
    most = max(_price(c) for c in listed())
    while True:
        case = _draw(rng)
        if _price(case) <= most:
            return case


# ---- inputs ---------------------------------------------------------------------------------------------------------------
def _grid_of(case):
    """(tokens of the video grid as (t, y, x), text tokens before it, text tokens behind it, sequence length)."""
    if case["kind"] in ("video", "dense"):
        p = PRESETS[case["preset"]]
        grid = (case["depth"], case["height"], case["width"])
        before, behind = (0, p["text"]) if case["preset"].startswith("CogVideo_5b") else (p["text"], 0)
        return grid, before, behind, grid[0] * grid[1] * grid[2] + p["text"]
    L, text = case["L"], case.get("text", 0)
    text = min(text, L // 2)
    side = max(4, min(52, int(round((L - text) ** 0.4))))
    high = max(4, side * 3 // 5)
    return (-(-(L - text) // (side * high)), high, side), text, 0, L


def _field(gen, grid, before, behind, L, B, H, D):
    """Rows the path meets: every channel a few slow waves over (t, y, x) and noise, text rows N(0, 1); fp32 [B, L, H, D]."""
    dev, waves = "cuda", 8
    T, Y, X = grid
    tt, yy, xx = torch.meshgrid(torch.arange(T, device=dev) / T, torch.arange(Y, device=dev) / Y, torch.arange(X, device=dev) / X,
                                indexing="ij")
    pos = torch.stack([tt, yy, xx], -1).reshape(-1, 3)[:L - before - behind]
    f = torch.rand(waves, 3, generator=gen, device=dev) * 3.0
    amp = torch.randn(waves, H * D, generator=gen, device=dev) / math.sqrt(waves)
    phi = torch.rand(waves, H * D, generator=gen, device=dev) * (2 * math.pi)
    arg = (pos @ f.t()) * (2 * math.pi)
    # sin(a + p) = sin a cos p + cos a sin p
    x = torch.cat([torch.sin(arg), torch.cos(arg)], 1) @ torch.cat([amp * torch.cos(phi), amp * torch.sin(phi)], 0)
    out = torch.randn(B, L, H * D, generator=gen, device=dev)
    out[:, before:L - behind].mul_(0.3).add_(x)
    return out.view(B, L, H, D)


def _qkv(case, gen):
    grid, before, behind, L = _grid_of(case)
    B, H, Hkv, D = case["B"], case["H"], case.get("Hkv", case["H"]), case["D"]
    q, k, v = (_field(gen, grid, before, behind, L, B, h, D) for h in (H, Hkv, Hkv))
    # logits of standard deviation 3
    n = min(L, 1024)
    at = torch.randperm(L, generator=gen, device="cuda")[:n]
    to = torch.randperm(L, generator=gen, device="cuda")[:n]
    s = torch.bmm(q[0, at].transpose(0, 1).contiguous(), k[0, to].repeat_interleave(H // Hkv, 1).permute(1, 2, 0).contiguous())
    c = (3.0 / (s.std() / math.sqrt(D))).sqrt()
    dt = DTYPES[case["dtype"]]
    # the attention processors hand over [B, H, L, D] views of [B, L, H, D] projections; the fp32 layer has plain tensors
    q, k, v = ((t * f).to(dt).transpose(1, 2) for t, f in ((q, c), (k, c), (v, 1.0)))
    return tuple(t.contiguous() for t in (q, k, v)) if case["dtype"] == "fp32" else (q, k, v)


def _ratios(case):
    return dict(RATIOS[case["ratios"]])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = _qkv(case, gen)
    state = dict(case=case, q=q, k=k, v=v, seed=seed)
    kind = case["kind"]
    if kind in ("video", "dense"):
        from psa_hip import AttentionConfig, PyramidSparseAttention
        from psa_hip.config_loader import AttentionConfigLoader

        model, preset = case["preset"].split("/")
        shape = [n * s for n, s in zip((case["width"], case["height"], case["depth"]), PRESETS[case["preset"]]["step"])]
        params = AttentionConfigLoader().get_attention_config(model, preset, shape)["params"]
        # (no log file; every step is a sparse one, or every step a warm-up one)
        params.update(enable_logging=False, warmup_steps=0 if kind == "video" else 50)
        state["module"] = PyramidSparseAttention(AttentionConfig(**params), inference_num=50, layer_num=30)
    elif kind in ("plug", "train"):
        from psa_hip import PSAAttention, PSAConfig

        cfg = dict(block_m=case.get("block_m", 128), block_n=case.get("block_n", 128), tile_n=case.get("tile_n", 32),
                   mask_ratios=_ratios(case), mask_mode=case["mode"])
        if kind == "train":
            cfg["attn_impl"] = "old_mask_type"  # the mask format that has a backward
            state["dout"] = (torch.randn(q.shape, generator=gen, device="cuda") * 0.02).to(q.dtype)
            for t in (q, k, v):
                t.requires_grad_(True)
        state["module"] = PSAAttention(PSAConfig(**cfg))
    else:
        from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

        cfg = AttentionConfig(text_length=case["text"], mask_ratios=_ratios(case), mask_mode=case["mode"], xattn_stride=case["stride"])
        state["module"] = PyramidAdaptiveBlockSparseAttnTrain(cfg, layer_idx=0)
    return state


def _fixed_draw(state):
    """The in-block offsets the block estimate samples: drawn on the device for every pass as the module does by itself, here
    with the state's seed so that a pass can be repeated."""
    from psa_hip import ops

    m, q, k = state["module"], state["q"], state["k"]
    bm, bn = m.config.block_m, m.config.block_n
    m.sample_offsets = ops.draw_sample_offsets(q.shape[0], q.shape[1], k.shape[1], bm, bm // 4, bn, bn // 4, q.device, seed=state["seed"])


def run(state):
    kind, m, q, k, v = state["case"]["kind"], state["module"], state["q"], state["k"], state["v"]
    if kind == "train":
        _fixed_draw(state)
        out = m(q, k, v)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
        return out, dq, dk, dv
    with torch.no_grad():
        if kind == "causal":
            return m(q, k, v, layer_idx=0)
        if kind == "plug":
            _fixed_draw(state)
            return m(q, k, v)
        if kind == "video":
            _fixed_draw(state)
        return m(q, k, v, 0)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
# Share of the dense products that the map keeps: of the quotas themselves, or (thresholds) what the synthetic fields give.
_DENSITY = {"default": 0.15, "bound90": 0.1, "bound85": 0.135, "bound80": 0.2}


def _density(case, L):
    if case["kind"] == "dense":
        return 1.0
    if case["kind"] == "video":
        return PRESETS[case["preset"]]["density"]
    d = _DENSITY[case["ratios"]]
    if case["kind"] == "causal":
        # the text's rows and columns, the diagonal and the first column are kept at full resolution
        n = -(-L // 128)
        rest = n - min(n, -(-case["text"] // 128))
        full = min(1.0, 1.0 - (rest / n) ** 2 + 4.0 * rest / (n * (n + 1)))
        d = full + (1.0 - full) * d
    return d


def work(case):
    L = _grid_of(case)[3]
    B, H, Hkv, D, kind = case["B"], case["H"], case.get("Hkv", case["H"]), case["D"], case["kind"]
    size = 4 if case["dtype"] == "fp32" else 2
    nbytes = B * L * D * size * (2 * H + 2 * Hkv)  # q, k, v read, the output written
    dense = 4.0 * B * H * L * L * D * (0.5 if kind == "causal" else 1.0)
    flops = dense * _density(case, L)
    if kind == "train":
        flops *= 3.5  # dQ, dK, dV: five products where the forward has two
        nbytes += B * L * D * size * 4 * H  # the output's gradient read, dq, dk, dv written
    if kind == "causal":
        flops += dense / 2 / case["stride"]  # every stride-th antidiagonal of the logits
    elif kind != "dense":
        flops += dense / 32  # a quarter of the queries against a quarter of the keys
    return {"bytes": float(nbytes), "flops": flops}


def tolerance(case):
    """About four times what was measured.  Against the same attention in 32 / 64 bits (same level map): outputs 2.0e-3 in
    bf16, 2.5e-4 in fp16, 6e-7 in fp32, gradients 4.4e-3 in bf16 and 4.6e-4 in fp16.  Block scores changed by 3e-6, as by
    sums in another order, turn over a few levels in a million: up to 1.3e-3 of the output as a whole, and single values by
    half to once the output's root mean square."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 5e-3}
    if case["kind"] == "dense":
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3, "max": 5e-2}
    bf16, half = (1.6e-2, 5e-3) if case["kind"] == "train" else (8e-3, 5e-3)
    return {"rel": bf16 if case["dtype"] == "bf16" else half, "max": 0.99}
