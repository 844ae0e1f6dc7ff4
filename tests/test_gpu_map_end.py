"""Level maps that end in their own kernel: similarity cap, map and tile list against the separate operators, bit for bit, at the edges
of blocks, of workgroups of the pooling pass and of the sorts' ranges; NaN and constant scores among them."""
import pytest
import torch

from gpu_util import dev, rnd

pytestmark = pytest.mark.gpu
RATIOS = {1: (0.0, 0.1), 2: (0.1, 0.2), 4: (0.2, 0.3), 8: (0.3, 0.5), 0: (0.5, 1.0)}


@pytest.mark.parametrize("B,Hq,Hkv,L,D,bn,mode,dtype", [
    (1, 9, 9, 129, 64, 128, "topk", torch.bfloat16),
    (2, 4, 2, 1000, 128, 128, "thresholdbound", torch.float16),
    (1, 33, 33, 4097, 64, 64, "topk", torch.bfloat16),            # 64-key blocks are listed above 1024 rows
    (1, 14, 14, 9601, 128, 32, "topk", torch.bfloat16),           # rows of 301 blocks: quotas without a sorted row
    (1, 14, 14, 9601, 64, 32, "thresholdbound", torch.bfloat16),  # ... sorted by the network
])
@pytest.mark.parametrize("indexed,capped,flat", [(False, False, False), (True, True, False), (False, True, True)])
def test_map_and_list_in_one_launch(B, Hq, Hkv, L, D, bn, mode, dtype, indexed, capped, flat):
    from psa_hip import ops

    q, k, v = (rnd(B, h, L, D, seed=L + i).to(dtype).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    if flat:
        k.zero_()  # every score the same
        k[:, 0, L // 3, 0] = float("nan")
    off_q, off_k = ops.draw_sample_offsets(B, Hq, Hkv, 128, 32, bn, bn // 4, dev(), seed=L)
    index = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None
    Mq, Nk = -(-L // 128), -(-L // bn)
    cap = None
    if capped:
        cap = torch.tensor([1, 2, 4, 8], dtype=torch.int32)[torch.randint(0, 4, (B, Hq, Nk), generator=torch.Generator().manual_seed(1))].to(dev())
    both = ops._map_and_walk(q, k, off_q, off_k, RATIOS, mode, 128, bn, 16, D ** -0.5, 40, index, cap)
    assert both is not None
    ref = ops.estimate_sampled_map(q, k, off_q, off_k, 128, bn, 32, bn // 4, RATIOS, 40, mode, compute_tile=16, map_dtype=torch.int8, q_index=index)
    if capped:
        ref = ops.map_min_cap(ref, cap)
    assert torch.equal(both[0], ref)
    v = torch.nan_to_num(v)
    pools = ops.pool_kv(torch.nan_to_num(k), v, bn)
    args = (q, torch.nan_to_num(k), v, ref, 128, bn)
    assert torch.equal(ops.sparse_attention_fwd(*args, pools=pools, _walk=both[1]), ops.sparse_attention_fwd(*args, pools=pools))


@pytest.mark.parametrize("H,L,D,bn", [(1, 1, 128, 128), (3, 1025, 128, 128), (2, 777, 128, 32), (5, 2000, 64, 128), (3, 300, 64, 32)])
@pytest.mark.parametrize("indexed", [False, True])
def test_cap_of_the_pooling_pass(monkeypatch, H, L, D, bn, indexed):
    """The layer in one call forms the cap beside the pooled rows, the separate operators in a pass of its own."""
    from psa_hip import ops

    q, k, v = (rnd(1, H, L, D, seed=L + i).to(dev()) for i in range(3))
    for i in range(1, min(L, 600), 2):
        k[:, :, i] = k[:, :, i - 1]  # neighbours alike: caps of every level
    off_q, off_k = ops.draw_sample_offsets(1, H, H, 128, 32, bn, bn // 4, dev(), seed=L)
    index = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None

    def layer():
        return ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, "topk", 128, bn, 16, token_index=index, return_map=True, return_cap=True,
                                 sim_thresholds=(0.3, 0.1, 0.0))

    one = layer()
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: None)
    for a, b in zip(one, layer()):
        assert torch.equal(a, b)


@pytest.mark.parametrize("Hq,Hkv,L,D,stride,mode", [
    (28, 4, 2345, 128, 8, "energybound"),   # small tiles: pooling beside the contraction
    (8, 8, 12001, 128, 8, "topk"),          # large tiles: pooling before it
    (2, 1, 33000, 64, 16, "energybound"),   # 258 blocks: rows on both sides of the sorts' switch
    (1, 1, 100, 128, 4, "topk"),
])
@pytest.mark.parametrize("nan", [False, True])
def test_causal_map_in_one_launch(Hq, Hkv, L, D, stride, mode, nan):
    from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

    q, k, v = (rnd(1, h, L, D, seed=L + i).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    if nan:
        q[:, :, L // 2, 3] = float("nan")
        q[:, :, L // 3, 3] = -float("nan")
        k[:, :, L - 1, 1] = float("inf")
    m = PyramidAdaptiveBlockSparseAttnTrain(AttentionConfig(text_length=128, mask_mode=mode, xattn_stride=stride, sim_2x_threshold=-0.1,
                                                            sim_4x_threshold=0.0, sim_8x_threshold=0.05), layer_idx=0)
    a = m(q, k, v, layer_idx=0)
    plain = m.sparse_attention_fn
    m.sparse_attention_fn = lambda *x: plain(*x)  # a function of the caller's own: the separate operators
    b = m(q, k, v, layer_idx=0)
    assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


def test_causal_rows_too_wide_for_one_launch():
    """5800 blocks per row: scores, levels and sorting scratch of a row do not fit LDS together; the layer's second buffer changes nothing."""
    import ctypes

    from psa_hip import _lib, ops
    from psa_hip._lib import check, lib

    B, H, D, block, stride = 1, 1, 64, 64, 8
    L = 5800 * block - 3
    chunk = 128 * stride
    q, k, v = (rnd(B, H, L, D, seed=i).to(dev()) for i in range(3))
    items = list(RATIOS.items())
    lv, hi = ops._level_items(items)
    lo = (ctypes.c_double * len(items))(*[float(i[1][0]) for i in items])
    shape = (B, H, H, L, D, block, stride, chunk)
    ws = torch.empty(lib.psa_causal_layer_workspace_bytes(*shape), dtype=torch.uint8, device=dev())
    extra = torch.empty(lib.psa_causal_layer_extra_bytes(*shape), dtype=torch.uint8, device=dev())
    outs = []
    for second in (None, extra.data_ptr()):
        out = torch.empty_like(q)
        check(lib.psa_causal_layer_fwd_extra(ops._t4(q), ops._t4(k), ops._t4(v), (ctypes.c_float * 3)(0.9, 0.9, 0.9), ws.data_ptr(), second,
                                             ops._t4(out), *shape, D ** -0.5, _lib.PSA_MODE_TOPK, len(items), lv, lo, hi, 0, 1, ops._stream(q)),
              "psa_causal_layer_fwd")
        outs.append(out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("mode,Nk", [("thresholdbound", 5300), ("topk", 5300)])
def test_wide_maps_need_no_scores(mode, Nk):
    """A map that is only stored keeps its levels out of LDS: rows of 5300 sorted scores fit beside their sorting scratch
    (8 * 8192 + 12 * 5300 + 4 * 5300 = 150336 bytes of 153600), without the buffer of scores."""
    from psa_hip import ops
    from psa_hip._lib import check, lib

    B, H, D, bm, bn = 1, 1, 64, 128, 32
    L = Nk * bn - 5
    q, k = (rnd(B, H, L, D, seed=i).to(dev()) for i in range(2))
    off_q, off_k = ops.draw_sample_offsets(B, H, H, bm, bm // 4, bn, bn // 4, dev(), seed=3)
    items, m, div = ops._items(RATIOS, mode)
    lv, hi = ops._level_items(items)
    Mq = -(-L // bm)
    ws = torch.empty(lib.psa_estimate_workspace_bytes(B, H, L, L, bm, bn, bm // 4, bn // 4), dtype=torch.uint8, device=dev())
    maps = []
    for scores in (None, torch.empty(B, H, Mq, Nk, dtype=torch.float32, device=dev())):
        mp = torch.zeros(B, H, Mq, Nk, dtype=torch.int32, device=dev())
        check(lib.psa_estimate_sampled_map(ops._t4(q), ops._t4(k), off_q.data_ptr(), off_k.data_ptr(), ops._ptr(scores), ws.data_ptr(), B, H, H, L, L, D,
                                           bm, bn, bm // 4, bn // 4, D ** -0.5, Mq, Nk, mp.data_ptr(), 4, m, len(items), lv, hi, 1, 0, 0.06,
                                           ops._stream(q)), "psa_estimate_sampled_map")
        maps.append(mp)
    ref = ops.level_map(scores, RATIOS, 0, mode, blocksize=bn, compute_tile=bn, map_dtype=torch.int32)
    assert torch.equal(maps[0], ref) and torch.equal(maps[1], ref)
