"""Sizes of the one-call layers' workspaces (host functions of the library, no GPU): the estimate's scratch, dead once the map exists,
and the buffers of the stages behind it share their bytes."""
import pytest

SLACK = 16 * 256  # alignment of the parts


@pytest.mark.parametrize("elem,B,Hq,Hkv,L,D,bm,bn,walk", [
    (2, 1, 48, 48, 45106, 64, 128, 32, 1),
    (2, 1, 12, 12, 32760, 128, 128, 128, 1),
    (2, 2, 8, 2, 1000, 64, 128, 64, 0),
    (2, 1, 1, 1, 150000, 64, 128, 32, 1),  # wider than the fused kernel's map: with a buffer of scores
    (4, 1, 2, 2, 4096, 64, 64, 64, 0),
])
@pytest.mark.parametrize("indexed", [0, 1])
def test_layer_stages_share_their_scratch(elem, B, Hq, Hkv, L, D, bm, bn, walk, indexed):
    from psa_hip._lib import lib

    Mq, Nk = -(-L // bm), -(-L // bn)
    pools = 2 * elem * lib.psa_pool_elems(B, Hkv, L, D, bn)
    ordered = 2 * elem * B * Hkv * L * D if indexed else 0
    est = lib.psa_estimate_workspace_bytes(B, Hq, L, L, bm, bn, bm // 4, bn // 4) + (4 * B * Hq * Mq * Nk if Nk > 4096 else 0)
    behind = lib.psa_walk_bytes(B, Hq, Hkv, L, D, bm, bn) if walk and elem == 2 else lib.psa_fwd_workspace_bytes(B, Hq, L, bm)
    need = ordered + (pools + max(est, behind) if indexed else max(est, pools + behind))
    got = lib.psa_layer_workspace_bytes(elem, B, Hq, Hkv, L, D, bm, bn, indexed, walk)
    assert need <= got <= need + SLACK


@pytest.mark.parametrize("B,Hq,Hkv,L,D,block,stride", [(1, 28, 4, 32768, 128, 128, 8), (2, 2, 2, 129, 64, 128, 16)])
def test_causal_layer_stages_share_their_scratch(B, Hq, Hkv, L, D, block, stride):
    from psa_hip._lib import lib

    S = -(-L // block)
    est = lib.psa_estimate_xattn_workspace_bytes(B, Hq, L, L, block, stride, 4096) + 4 * B * Hq * S * S
    behind = 4 * lib.psa_pool_elems(B, Hkv, L, D, block) + lib.psa_walk_bytes(B, Hq, Hkv, L, D, block, block)
    need = B * Hq * S * S + 4 * B * Hkv * S + max(est, behind)
    got = lib.psa_causal_layer_workspace_bytes(B, Hq, Hkv, L, D, block, stride, 4096)
    assert need <= got <= need + SLACK


@pytest.mark.parametrize("dtype,shape,listed", [
    ("bfloat16", (1, 48, 48, 45106, 64, 128, 32), True),
    ("bfloat16", (2, 48, 48, 45106, 64, 128, 64), True),
    ("bfloat16", (1, 40, 40, 262144, 128, 128, 64), False),  # 6.7 GB of list
    ("float16", (1, 40, 40, 262144, 128, 128, 128), True),   # 128-key blocks have always been listed
    ("bfloat16", (1, 8, 8, 1000, 64, 128, 64), False),       # few rows
    ("float32", (1, 48, 48, 45106, 64, 128, 32), False),
    ("bfloat16", (1, 48, 48, 45106, 64, 64, 32), False),     # 64-row q-blocks
])
def test_tile_lists_are_bounded(dtype, shape, listed):
    import torch
    from psa_hip import ops
    from psa_hip._lib import lib

    n = ops._walk_bytes(getattr(torch, dtype), *shape)
    assert n == (lib.psa_walk_bytes(*shape) if listed else 0)
    assert (n > 0) == listed and (shape[-1] == 128 or n <= 1 << 30)
