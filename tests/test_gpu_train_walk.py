"""PSAAttention with gradients: the level map and its tile list from one launch of the estimate's reduction (ops.estimate_walk) against
build_mask + the attention function, which the module takes where either is the caller's own: same outputs and gradients, bit for bit."""
import functools

import pytest
import torch

from gpu_util import dev, rnd

pytestmark = pytest.mark.gpu
RATIOS = {1: (0.0, 0.2), 2: (0.2, 0.3), 4: (0.3, 0.4), 8: (0.4, 0.6), 0: (0.6, 1.0)}


def _step(m, q, k, v, do):
    out = m(q, k, v)
    return (out,) + torch.autograd.grad(out, (q, k, v), do)


@pytest.mark.parametrize("B,Hq,Hkv,L,D", [(1, 8, 8, 1000, 64), (2, 4, 2, 513, 128), (1, 1, 1, 1, 64), (1, 2, 2, 128, 128), (1, 12, 12, 4300, 128)])
@pytest.mark.parametrize("mode", ["topk", "thresholdbound"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("strided", [False, True])
def test_same_bits(monkeypatch, B, Hq, Hkv, L, D, mode, dtype, strided):
    from psa_hip import PSAAttention, PSAConfig, ops

    q, k, v = (rnd(B, h, L, D, seed=L + i).to(dtype).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv)))
    if strided:
        q, k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    q, k, v = (x.requires_grad_(True) for x in (q, k, v))
    do = rnd(B, Hq, L, D, seed=L + 9).to(dtype).to(dev())
    m = PSAAttention(PSAConfig(block_m=128, block_n=128, mask_ratios=RATIOS, mask_mode=mode, attn_impl="old_mask_type"))
    m.sample_offsets = ops.draw_sample_offsets(B, Hq, Hkv, 128, 32, 128, 32, dev(), seed=L)
    calls, real = [], ops._map_and_walk
    monkeypatch.setattr(ops, "_map_and_walk", lambda *a: calls.append(real(*a)) or calls[-1])
    got = _step(m, q, k, v, do)
    assert calls and (calls[0] is None) == (dtype == torch.float32)  # (fp32 layers have no list)
    plain = m.sparse_attention_fn
    m.sparse_attention_fn = lambda *a: plain(*a)
    ref = _step(m, q, k, v, do)
    assert len(calls) == 1
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_a_mask_of_the_callers_own_is_used():
    from psa_hip import PSAAttention, PSAConfig, ops

    class Dense(PSAAttention):
        def build_mask(self, q, k, v):
            n = -(-q.shape[2] // 128)
            return torch.ones(q.shape[0], q.shape[1], n, n, dtype=torch.int32, device=q.device)

    q, k, v = (rnd(1, 2, 700, 64, seed=i).to(dev()).requires_grad_(True) for i in range(3))
    m = Dense(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))
    out = m(q, k, v)
    assert torch.equal(out, ops.sparse_attention_fwd(q.detach(), k.detach(), v.detach(), m.build_mask(q, k, v), 128, 128, return_lse=True)[0])


def test_a_mask_set_on_the_class_is_used(monkeypatch):
    from psa_hip import PSAAttention, PSAConfig, ops

    def dense(self, q, k, v):
        n = -(-q.shape[2] // 128)
        return torch.ones(q.shape[0], q.shape[1], n, n, dtype=torch.int32, device=q.device)

    q, k, v = (rnd(1, 2, 700, 64, seed=i).to(dev()).requires_grad_(True) for i in range(3))
    m = PSAAttention(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))
    monkeypatch.setattr(PSAAttention, "build_mask", dense)
    out = m(q, k, v)
    assert torch.equal(out, ops.sparse_attention_fwd(q.detach(), k.detach(), v.detach(), dense(m, q, k, v), 128, 128, return_lse=True)[0])


def test_a_wrapped_attention_function_is_called():
    from psa_hip import PSAAttention, PSAConfig

    q, k, v = (rnd(1, 2, 300, 64, seed=i).to(dev()).requires_grad_(True) for i in range(3))
    m = PSAAttention(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))
    plain, masks = m.sparse_attention_fn, []

    @functools.wraps(plain)
    def wrapper(q, k, v, mask, sm_scale):
        masks.append(mask)
        return plain(q, k, v, mask, sm_scale)

    m.sparse_attention_fn = wrapper
    m(q, k, v)
    assert len(masks) == 1 and masks[0].shape == (1, 2, 3, 3)


def test_a_function_of_other_blocks_than_the_map():
    """60 tokens are one block of 64 or of 128: the map of a configuration changed later fits, and the function's own block sizes count."""
    from psa_hip import PSAAttention, PSAConfig, ops

    q, k, v = (rnd(1, 2, 60, 64, seed=i).to(dev()).requires_grad_(True) for i in range(3))
    m = PSAAttention(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))
    m.config.block_m = m.config.block_n = 64
    m.sample_offsets = ops.draw_sample_offsets(1, 2, 2, 64, 16, 64, 16, dev(), seed=1)
    assert torch.equal(m(q, k, v), m.sparse_attention_fn(q, k, v, m.build_mask(q, k, v)))


def test_errors_stay():
    from psa_hip import PSAAttention, PSAConfig

    q, k, v = (rnd(1, 2, 300, 64, seed=i).to(dev()).requires_grad_(True) for i in range(3))
    for kw in (dict(mask_mode="other"), dict(mask_ratios=None), dict(tile_n=256)):
        cfg = PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type")
        for n, x in kw.items():
            setattr(cfg, n, x)
        with pytest.raises((ValueError, RuntimeError)):
            m = PSAAttention(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))
            m.config = cfg
            m(q, k, v)
    with pytest.raises(RuntimeError):
        PSAAttention(PSAConfig(block_m=128, block_n=128, attn_impl="old_mask_type"))(q.detach().cpu().requires_grad_(True), k, v)
