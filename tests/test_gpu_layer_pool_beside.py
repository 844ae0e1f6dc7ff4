"""Layers whose pooling pass is part of the launch of the estimate's contraction, with the estimate's scratch in the output: the bits of the
same layer with an output that cannot take the scratch (rows apart, misaligned, one of the inputs), and of the pooled pass of its own."""
import ctypes

import pytest
import torch

from gpu_util import dev, rnd

pytestmark = pytest.mark.gpu
RATIOS = {1: (0.0, 0.1), 2: (0.1, 0.15), 4: (0.15, 0.15), 8: (0.15, 0.35), 0: (0.35, 1.0)}


@pytest.mark.parametrize(
    "B,Hq,Hkv,L,D,bm,bn,dtype",
    [
        (1, 8, 8, 1000, 64, 128, 64, torch.bfloat16),
        (2, 4, 2, 1029, 128, 64, 128, torch.float16),   # kv heads shared, 32-key groups
        (1, 3, 3, 700, 64, 128, 32, torch.bfloat16),    # 8-key groups
        (1, 1, 1, 131, 128, 128, 64, torch.bfloat16),   # scratch above the output
        (1, 1, 1, 9000, 64, 128, 64, torch.bfloat16),   # four shares of the keys
        (1, 2, 1, 4096, 64, 64, 64, torch.float32),
        (1, 3, 3, 555, 128, 64, 32, torch.float32),
        (2, 8, 8, 4096, 128, 128, 128, torch.bfloat16), # K and V at 32 MiB
        (2, 8, 8, 4097, 128, 128, 128, torch.bfloat16), # and just above
    ],
)
@pytest.mark.parametrize("capped", [False, True])
def test_scratch_in_the_output(B, Hq, Hkv, L, D, bm, bn, dtype, capped):
    from psa_hip import ops
    from psa_hip._lib import check, lib

    if capped and (Hq != Hkv or dtype == torch.float32):
        pytest.skip("takes the separate operators")
    q, k, v = (rnd(B, h, L, D, seed=L + i).to(dtype).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    off_q, off_k = ops.draw_sample_offsets(B, Hq, Hkv, bm, bm // 4, bn, bn // 4, dev(), seed=L)
    items, m, _ = ops._items(RATIOS, "topk")
    lv, hi = ops._level_items(items)
    Mq, Nk = -(-L // bm), -(-L // bn)
    sizes = (q.element_size(), B, Hq, Hkv, L, D, bm, bn, 0, 1)
    n_ws, n_extra = lib.psa_layer_workspace_bytes(*sizes), lib.psa_layer_extra_bytes(*sizes)

    def layer(query, out):
        ws = torch.full((n_ws + n_extra,), 255, dtype=torch.uint8, device=dev())
        mp = torch.empty(B, Hq, Mq, Nk, dtype=torch.int8, device=dev())
        cap = torch.empty(B, Hkv, Nk, dtype=torch.int32, device=dev()) if capped else None
        thr = (ctypes.c_float * 3)(-0.1, 0.0, 0.1) if capped else None
        at = ws.data_ptr()
        check(lib.psa_layer_fwd_extra(ops._t4(query), ops._t4(k), ops._t4(v), None, off_q.data_ptr(), off_k.data_ptr(), thr, ops._ptr(cap), at,
                                      at + n_ws, mp.data_ptr(), ops._t4(out), B, Hq, Hkv, L, D, bm, bn, D ** -0.5, m, len(items), lv, hi, 1, 0, 0.06,
                                      1, ops._stream(query)), "psa_layer_fwd")
        torch.cuda.synchronize()
        return mp, out

    mp, out = layer(q, torch.empty_like(q))
    spaced = torch.full((B, Hq, L, 2 * D), 7, dtype=dtype, device=dev())
    shifted = torch.full((q.numel() + 8,), 7, dtype=dtype, device=dev())
    inplace = q.clone()
    for query, other in ((q, spaced[..., :D]), (q, shifted[8:].view_as(q)), (inplace, inplace)):
        mp2, out2 = layer(query, other)
        assert torch.equal(mp, mp2) and torch.equal(out, out2)
    assert (spaced[..., D:] == 7).all() and (shifted[:8] == 7).all()
    ref = ops.estimate_sampled_map(q, k, off_q, off_k, bm, bn, bm // 4, bn // 4, RATIOS, 0, "topk", compute_tile=bn, map_dtype=torch.int8)
    if capped:
        ref = ops.map_min_cap(ref, ops.k_similarity(k, bn, -0.1, 0.0, 0.1))
    kp, vp = ops.pool_kv(k, v, bn)
    assert torch.equal(mp, ref)
    assert torch.equal(out, ops.sparse_attention_fwd(q, k, v, ref, bm, bn, D ** -0.5, pools=(kp, vp)))


@pytest.mark.parametrize("H,L,D,bn", [(4, 700, 64, 64), (3, 1029, 128, 128), (2, 333, 64, 32), (3, 700, 128, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_cap_of_keys_that_are_not_finite(H, L, D, bn, dtype):
    """A kv-block with a NaN or infinite key, or with keys whose squared norms are above the largest float, has no mean cosine and takes no
    pooling (cap 1; the thresholds are below all cosines, so every other block has 8): in the contraction's launch as in psa_ksim."""
    from psa_hip import ops

    q, k, v = (rnd(1, H, L, D, seed=L + i).to(dtype).to(dev()) for i in range(3))
    expected = torch.full((1, H, -(-L // bn)), 8, dtype=torch.int32)
    for b, x in enumerate((float("nan"), float("inf"), float("-inf"), 3e19)):
        if not torch.isfinite(torch.tensor(x)) or dtype == torch.bfloat16:
            at = b * bn + 8 * b  # (the first or the last of 8 tokens, which pairs of every distance meet; all of them)
            k[:, b % H, slice(at, at + 8) if x == 3e19 else at + 7 * (b & 1), b] = x
            expected[:, b % H, b] = 1
    k[:, H - 1, L - 1, D - 1] = float("nan")  # (and the pad rows behind it)
    expected[:, H - 1, -1] = 1
    thr = (-2.0, -2.0, -2.0)
    off_q, off_k = ops.draw_sample_offsets(1, H, H, 128, 32, bn, bn // 4, dev(), seed=L)
    _, mp, cap = ops._layer_one_call(q, k, v, off_q, off_k, RATIOS, "topk", 128, bn, bn, D ** -0.5, 0, None, thr)
    assert torch.equal(ops.k_similarity(k, bn, *thr).cpu(), expected)
    assert torch.equal(cap.cpu(), expected)
    ref = ops.estimate_sampled_map(q, k, off_q, off_k, 128, bn, 32, bn // 4, RATIOS, 0, "topk", compute_tile=bn, map_dtype=torch.int8)
    assert torch.equal(mp, ops.map_min_cap(ref, cap))
