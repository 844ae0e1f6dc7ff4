"""Helpers shared by the GPU parity tests."""
import numpy as np
import torch

import psa_oracle as O


def dev():
    return torch.device("cuda:0")


def rnd(*shape, seed=0, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def random_map(B, H, Mq, Nk, seed, p=(0.35, 0.2, 0.15, 0.15, 0.15), ensure_row=True):
    rng = np.random.default_rng(seed)
    m = rng.choice([0, 1, 2, 4, 8], size=(B, H, Mq, Nk), p=p).astype(np.int32)
    if ensure_row:
        m[..., 0] = np.where(m.sum(-1) == 0, 1, m[..., 0])
    return m


def attn_errors(out_gpu, ref):
    d = (out_gpu.float().cpu() - ref.float()).abs()
    return float(d.max()), float(d.mean())


# tolerance of the task statement for bf16 attention outputs
MAX_ABS, MEAN_ABS = 2e-2, 2e-3


def xattn_tile(heads, Lq, Lk, block, stride, chunk, causal):
    """Output tile of the antidiagonal contraction's launch (csrc/psa_xattn.hip, xattn_small; rows that do not overlap) and how many of
    them the busiest workgroup takes: ("large" | "small", tiles)."""
    up = lambda n, m: -(-n // m) * m
    Mr, Nr = up(Lq, chunk) // stride, up(Lk, chunk) // stride
    rows = min(-(-Lq // block) * (block // stride), Mr)

    def tiles(edge):
        per_row = lambda tm: min(-(-Nr // edge), ((tm + 1) * edge - 1 + Nr - Mr) // edge + 1) if causal else -(-Nr // edge)
        return heads * sum(per_row(tm) for tm in range(-(-rows // edge)))

    large, small = tiles(256), tiles(128)
    if (small + 256) * 3 < -(-large // 256) * 2560:
        return "small", 1
    return "large", -(-(-(-large // 8)) // 32)  # 8 XCDs, 32 workgroups each


def fp32_kernel(D, B, Hq, L, bm, far=False):
    """Kernel of the fp32 forward that a call runs (csrc/psa_f32.hip, launch_f32) and its rows per workgroup; far: rows of K or V beyond 32-bit
    offsets."""
    rows16 = B * Hq * -(-L // bm) * (bm // 16)
    full_rounds = 2048 <= rows16 <= 4096 and (rows16 - 1) % 2048 >= 1840
    wins = L > 2048 or not full_rounds if D == 64 else rows16 < 1024 or (rows16 <= 1728 and 4096 <= L <= 20480)
    if wins and not far:
        return "direct", 32 if D == 64 and rows16 > 1280 else 16
    return "tiles", 32 if rows16 < 2048 else 64
