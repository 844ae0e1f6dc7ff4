"""The layers as one library call (ops.psa_layer_fwd, ops.causal_layer_fwd) against the separate operators: same bits, on either
side of the sizes where the tiles are listed, with and without token index and similarity cap, and on a stream of the caller's."""
import pytest
import torch

from gpu_util import dev, rnd

pytestmark = pytest.mark.gpu
RATIOS = {1: (0.0, 0.1), 2: (0.1, 0.15), 4: (0.15, 0.15), 8: (0.15, 0.35), 0: (0.35, 1.0)}


@pytest.mark.parametrize(
    "B,Hq,Hkv,L,D,bm,bn,mode,dtype",
    [
        (1, 8, 8, 1000, 64, 128, 64, "topk", torch.bfloat16),
        (2, 4, 2, 513, 128, 128, 128, "thresholdbound", torch.float16),   # GQA, 128-key blocks: listed tiles
        (1, 38, 38, 3400, 64, 128, 32, "topk", torch.bfloat16),           # more rows than _WALK_MIN_ROWS
        (1, 2, 2, 1024, 64, 64, 64, "thresholdbound", torch.float32),
        (1, 1, 1, 1, 128, 128, 64, "topk", torch.bfloat16),
    ],
)
@pytest.mark.parametrize("strided,indexed,capped", [(False, False, False), (True, False, True), (True, True, False), (False, True, True)])
def test_one_call_equals_separate_operators(monkeypatch, B, Hq, Hkv, L, D, bm, bn, mode, dtype, strided, indexed, capped):
    from psa_hip import ops

    if capped and (Hq != Hkv or dtype == torch.float32):
        pytest.skip("takes the separate operators")

    q, k, v = (rnd(B, h, L, D, seed=L + i).to(dtype).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    if strided:
        q, k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    off_q, off_k = ops.draw_sample_offsets(B, Hq, Hkv, bm, bm // 4, bn, bn // 4, dev(), seed=L)

    index = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None

    def layer():
        return ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, mode, bm, bn, 16, return_map=True, return_cap=True, text_length=70,
                                 token_index=index, sim_thresholds=(-0.1, 0.0, 0.1) if capped else None)

    calls = []
    real = ops._layer_one_call
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: calls.append(real(*a)) or calls[-1])
    out, mp, cap = layer()
    assert calls and calls[0] is not None and (cap is not None) == capped
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        on_stream = layer()
    s.synchronize()
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: None)
    ref = layer()
    torch.cuda.synchronize()
    for a, b in ((out, ref[0]), (mp, ref[1]), (on_stream[0], ref[0])):
        assert torch.equal(a, b)
    assert not capped or torch.equal(cap, ref[2])


@pytest.mark.parametrize("Hq,Hkv,L,D,stride,mode,text", [(28, 4, 2345, 128, 8, "energybound", 512), (2, 2, 129, 64, 16, "topk", 0), (6, 3, 4200, 64, 4, "topk", 30)])
@pytest.mark.parametrize("causal", [True, False])
def test_causal_one_call_equals_separate_operators(Hq, Hkv, L, D, stride, mode, text, causal):
    from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

    q, k, v = (rnd(2, h, L, D, seed=L + i).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    cfg = AttentionConfig(text_length=text, mask_mode=mode, xattn_stride=stride, causal_main=causal, sim_2x_threshold=-0.1, sim_4x_threshold=0.0,
                          sim_8x_threshold=0.05)
    m = PyramidAdaptiveBlockSparseAttnTrain(cfg, layer_idx=0)
    a = m(q, k, v, layer_idx=0)
    plain = m.sparse_attention_fn
    m.sparse_attention_fn = lambda *x: plain(*x)  # a function of the caller's own: the separate operators
    b = m(q, k, v, layer_idx=0)
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_one_call_refuses_what_the_operators_refuse():
    from psa_hip import ops

    q, k, v = (rnd(1, 2, 256, 64, seed=i).to(dev()) for i in range(3))
    off_q, off_k = ops.draw_sample_offsets(1, 2, 2, 128, 32, 64, 16, dev(), seed=1)
    go = lambda **kw: ops.psa_layer_fwd(*[kw.get(n, x) for n, x in (("q", q), ("k", k), ("v", v), ("off_q", off_q), ("off_k", off_k))],
                                        kw.get("ratios", RATIOS), kw.get("mode", "topk"), 128, 64, kw.get("tile_n", 32))
    for kw in (dict(mode="topk_newtype"), dict(mode="other"), dict(ratios=None), dict(off_q=off_q[:, :1]), dict(off_k=off_k.long()),
               dict(k=k[:, :, :128]), dict(v=v[:, :1]), dict(tile_n=128), dict(q=q[0])):
        with pytest.raises((ValueError, RuntimeError)):
            go(**kw)


@pytest.mark.parametrize("causal", [False, True])
def test_large_layers_hand_their_scratch_back_first(monkeypatch, causal):
    """Above the workspace limit the separate operators run: same bits, and the output is not taken beside the estimate's scratch."""
    from psa_hip import _lib, ops
    from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

    H, L, D = 8, 16000, 64
    q, k, v = (rnd(1, H, L, D, seed=i).to(dev()) for i in range(3))
    if causal:
        m = PyramidAdaptiveBlockSparseAttnTrain(AttentionConfig(text_length=70, xattn_stride=4), layer_idx=0)
        layer = lambda: m(q, k, v, layer_idx=0)
    else:
        off_q, off_k = ops.draw_sample_offsets(1, H, H, 128, 32, 32, 8, dev(), seed=1)
        layer = lambda: ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, "topk", 128, 32, 16)

    def run(limit):
        monkeypatch.setattr(ops, "_ONE_CALL_MAX_BYTES", limit)
        layer()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        out = layer()
        torch.cuda.synchronize()
        return out, torch.cuda.max_memory_allocated() - before

    (a, one), (b, separate) = run(1 << 30), run(1 << 20)
    assert torch.equal(a, b)
    if not causal:  # (K below _SIDE_STREAM_MIN_BYTES, a layer that is one call; the estimate's stage is the larger one)
        est = _lib.lib.psa_estimate_workspace_bytes(1, H, L, L, 128, 32, 32, 8)
        assert one >= est + q.numel() * 2 > separate


def test_causal_one_call_leaves_dual_tensors_to_the_autograd_function(monkeypatch):
    """Forward-mode differentiation has no rule here: it is refused.  An open level alone changes nothing."""
    from torch.autograd import forward_ad

    from psa_hip import ops
    from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

    q, k, v = (rnd(1, 2, 300, 64, seed=i).to(dev()) for i in range(3))
    m = PyramidAdaptiveBlockSparseAttnTrain(AttentionConfig(text_length=0), layer_idx=0)
    with torch.no_grad():
        a = m(q, k, v, layer_idx=0)
        calls = []
        one_call = ops.causal_layer_fwd
        monkeypatch.setattr(ops, "causal_layer_fwd", lambda *x: calls.append(1) or one_call(*x))
        with forward_ad.dual_level():
            b = m(q, k, v, layer_idx=0)
            assert calls
            with pytest.raises(RuntimeError):
                m(q, k, forward_ad.make_dual(v, torch.ones_like(v)), layer_idx=0)
            assert len(calls) == 1
    assert torch.equal(a, b)


def test_layer_runs_on_the_current_stream_without_the_raw_handle(monkeypatch):
    """The public way to the stream's handle, for a torch without the shorter call: the layer follows work that the caller's stream
    still has to do, as with it."""
    from psa_hip import ops

    q, k, v = (rnd(1, 2, 1000, 64, seed=i).to(dev()) for i in range(3))
    off_q, off_k = ops.draw_sample_offsets(1, 2, 2, 128, 32, 64, 16, dev(), seed=1)
    outs = []
    for raw in (ops._raw_stream, None):
        monkeypatch.setattr(ops, "_raw_stream", raw)
        s = torch.cuda.Stream()
        assert ops._stream(q) == torch.cuda.current_stream().cuda_stream
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            assert ops._stream(q) == s.cuda_stream
            x = q
            for _ in range(50):
                x = x * 1.0
            outs.append(ops.psa_layer_fwd(x, k, v, off_q, off_k, RATIOS, "topk", 128, 64, 16))
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])


def _peak(layer):
    """What a call holds at most beside what was there before it."""
    layer()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = layer()
    torch.cuda.synchronize()
    return out, torch.cuda.max_memory_allocated() - before


@pytest.mark.parametrize("H,L,D,bn", [
    (12, 20000, 64, 32),    # scratch of the estimate above the output: the list waits for it to go
    (12, 20000, 128, 128),  # below: the map's kernel writes the list
])
@pytest.mark.parametrize("indexed", [False, True])
def test_a_list_from_the_map_kernel_takes_no_more_memory(monkeypatch, H, L, D, bn, indexed):
    """The separate operators with map and list from one launch hold no more at once than with a launch each; same bits."""
    from psa_hip import _lib, ops

    q, k, v = (rnd(1, H, L, D, seed=i).to(dev()) for i in range(3))
    off_q, off_k = ops.draw_sample_offsets(1, H, H, 128, 32, bn, bn // 4, dev(), seed=1)
    index = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: None)
    real, calls = ops._map_and_walk, []

    def run(fused):
        monkeypatch.setattr(ops, "_map_and_walk", (lambda *a: calls.append(1) or real(*a)) if fused else lambda *a: None)
        return _peak(lambda: ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, "topk", 128, bn, 16, token_index=index))

    (a, one), (b, plain) = run(True), run(False)
    slack = 4 << 20  # (torch leaves up to 1 MiB at the end of a large block)
    assert ops._walk_bytes(q.dtype, 1, H, H, L, D, 128, bn) > 2 * slack
    assert torch.equal(a, b) and one <= plain + slack
    est = _lib.lib.psa_estimate_workspace_bytes(1, H, L, L, 128, bn, 32, bn // 4)
    assert bool(calls) == (est <= q.numel() * 2) == (bn == 128)


@pytest.mark.parametrize("L,bn,dtype,capped", [
    (1000, 64, torch.bfloat16, False),    # few rows of 64-key blocks: neither cap nor list
    (1000, 64, torch.float32, False),
    (1000, 128, torch.float16, False),    # a list, no cap
    (1000, 64, torch.bfloat16, True),     # a cap: pools beside the estimate's scratch
])
def test_layers_take_no_memory_that_serves_nothing(L, bn, dtype, capped):
    from psa_hip import _lib, ops

    H, D, up = 8, 64, lambda n: -(-n // 512) * 512  # (granularity of torch's allocations)
    q, k, v = (rnd(1, H, L, D, seed=i).to(dtype).to(dev()) for i in range(3))
    off_q, off_k = ops.draw_sample_offsets(1, H, H, 128, 32, bn, bn // 4, dev(), seed=1)
    _, peak = _peak(lambda: ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, "topk", 128, bn, 16, sim_thresholds=(0.9, 0.9, 0.9) if capped else None))
    shape, Mq, Nk = (1, H, H, L, D, 128, bn), -(-L // 128), -(-L // bn)
    walk = ops._walk_bytes(dtype, *shape)
    assert (walk > 0) == (bn == 128)
    need = _lib.lib.psa_layer_workspace_bytes(q.element_size(), *shape, 0, int(walk > 0)) + -(-walk // 256) * 256
    if capped:
        need += 2 * (-(-2 * _lib.lib.psa_pool_elems(1, H, L, D, bn) // 256) * 256)
    assert peak <= up(need) + up(H * Mq * Nk) + up(H * L * D * q.element_size()) + (up(H * Nk * 4) if capped else 0)


@pytest.mark.parametrize("Hq,Hkv,L,D,bn,mode,indexed,capped", [
    (8, 8, 1000, 64, 64, "topk", False, False),
    (4, 2, 513, 128, 128, "thresholdbound", False, False),   # listed
    (4, 4, 1537, 128, 128, "topk", False, True),             # ... with the cap, pooling behind the map
    (4, 4, 1537, 128, 128, "topk", True, True),              # ... formed by the pooling pass of the ordered rows, applied by the map's kernel
    (38, 38, 3400, 64, 32, "topk", True, False),             # listed 32-key blocks
    (38, 38, 3400, 64, 32, "thresholdbound", False, True),
])
def test_one_call_without_its_second_buffer(monkeypatch, Hq, Hkv, L, D, bn, mode, indexed, capped):
    """Between the limits for one buffer and for two the stages behind the map overlay the estimate's scratch, and list, cap and pooling
    come from launches of their own where the map's kernel and the pooling pass have no place for them."""
    from psa_hip import ops

    q, k, v = (rnd(1, h, L, D, seed=L + i).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    off_q, off_k = ops.draw_sample_offsets(1, Hq, Hkv, 128, 32, bn, bn // 4, dev(), seed=L)
    index = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None

    def layer():
        return ops.psa_layer_fwd(q, k, v, off_q, off_k, RATIOS, mode, 128, bn, 16, return_map=True, return_cap=True, text_length=70,
                                 token_index=index, sim_thresholds=(0.3, 0.1, 0.0) if capped else None)

    shape = (1, Hq, Hkv, L, D, 128, bn)
    walk = int(ops._walk_bytes(q.dtype, *shape) > 0)
    n_ws = ops.lib.psa_layer_workspace_bytes(2, *shape, int(indexed), walk)
    seconds, call = [], ops.lib.psa_layer_fwd_extra
    monkeypatch.setattr(ops.lib, "psa_layer_fwd_extra", lambda *a: seconds.append(a[9]) or call(*a))
    with_it = layer()
    monkeypatch.setattr(ops, "_ONE_CALL_MAX_BYTES", n_ws)
    without = layer()
    assert len(seconds) == 2 and (seconds[0] is not None) == bool(walk or (capped and not indexed)) and seconds[1] is None
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: None)
    ref = layer()
    for got in (with_it, without):
        for a, b in zip(got, ref):
            assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.parametrize("Hq,Hkv,L,D,stride,mode", [(28, 4, 2345, 128, 8, "energybound"), (8, 8, 12001, 128, 8, "topk"), (2, 2, 129, 64, 16, "topk")])
def test_causal_one_call_without_its_second_buffer(monkeypatch, Hq, Hkv, L, D, stride, mode):
    from psa_hip import ops
    from psa_hip.PSA_casual import AttentionConfig, PyramidAdaptiveBlockSparseAttnTrain

    q, k, v = (rnd(1, h, L, D, seed=L + i).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    m = PyramidAdaptiveBlockSparseAttnTrain(AttentionConfig(text_length=130, mask_mode=mode, xattn_stride=stride, sim_2x_threshold=-0.1,
                                                            sim_4x_threshold=0.0, sim_8x_threshold=0.05), layer_idx=0)
    sizes, size = [], ops.lib.psa_causal_layer_workspace_bytes
    monkeypatch.setattr(ops.lib, "psa_causal_layer_workspace_bytes", lambda *a: sizes.append(size(*a)) or sizes[-1])
    seconds, call = [], ops.lib.psa_causal_layer_fwd_extra
    monkeypatch.setattr(ops.lib, "psa_causal_layer_fwd_extra", lambda *a: seconds.append(a[5]) or call(*a))
    a = m(q, k, v, layer_idx=0)
    monkeypatch.setattr(ops, "_ONE_CALL_MAX_BYTES", sizes[0])
    b = m(q, k, v, layer_idx=0)
    assert len(seconds) == 2 and seconds[0] is not None and seconds[1] is None
    plain = m.sparse_attention_fn
    m.sparse_attention_fn = lambda *x: plain(*x)  # a function of the caller's own: the separate operators
    c = m(q, k, v, layer_idx=0)
    assert torch.equal(a, c) and torch.equal(b, c)
