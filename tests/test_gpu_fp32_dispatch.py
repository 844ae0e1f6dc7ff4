"""The kernel of the fp32 forward that a launch runs (gpu_util.fp32_kernel: blocks of 16 query rows in the launch, head dim and length): rows straight into
registers, 16 or 32 per workgroup, or tiles through LDS, 32 or 64 rows per workgroup; against float64 on the same map and pooled rows.  Tolerance of the
fp32 path: 2e-5 absolute for values of order 1."""
import pytest
import torch

from gpu_util import dev, fp32_kernel, random_map
from test_gpu_fp32_direct import _check as check
from test_gpu_fp32_split import _rand, _reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H,L,bm,bn,causal,kernel", [
    (64, 80, 250, 64, 32, False, ("direct", 16)),     # 1280 blocks of 16 rows
    (64, 81, 250, 128, 128, False, ("direct", 32)),   # 1296
    (64, 107, 177, 64, 64, True, ("direct", 32)),     # 1284, a last block of 17 rows
    (64, 511, 50, 64, 64, False, ("direct", 32)),     # 2044
    (64, 512, 50, 64, 32, True, ("tiles", 64)),       # 2048: a full round
    (64, 513, 50, 64, 64, False, ("direct", 32)),     # 2052
    (64, 324, 130, 64, 64, False, ("direct", 32)),    # 3888
    (64, 325, 130, 64, 128, True, ("tiles", 64)),     # 3900: nearly two rounds
    (64, 1024, 50, 64, 64, False, ("tiles", 64)),     # 4096
    (64, 1025, 50, 64, 64, False, ("direct", 32)),    # 4100
    (64, 16, 2048, 64, 64, False, ("tiles", 64)),     # the longest rows of that kind
    (64, 8, 4096, 64, 64, False, ("direct", 32)),
    (128, 85, 180, 64, 64, False, ("direct", 16)),    # 1020
    (128, 128, 120, 64, 32, True, ("tiles", 32)),     # 1024
    (128, 255, 120, 64, 128, False, ("tiles", 32)),   # 2040
    (128, 256, 120, 128, 64, False, ("tiles", 64)),   # 2048
    (128, 6, 4096, 128, 128, False, ("direct", 16)),  # 1536 of rows long enough
    (128, 6, 4095, 128, 128, False, ("tiles", 32)),
    (128, 6, 4600, 128, 64, True, ("direct", 16)),    # 1728
    (128, 7, 4097, 64, 64, False, ("tiles", 32)),     # 1820
    (128, 256, 180, 64, 64, False, ("tiles", 64)),    # 3072
    (128, 257, 180, 64, 32, True, ("tiles", 64)),     # 3084
    (128, 400, 100, 128, 64, False, ("tiles", 64)),   # 3200, one block per head
    (64, 1, 5, 64, 64, False, ("direct", 16)),        # fewer rows than a block
])
def test_borders(D, H, L, bm, bn, causal, kernel):
    assert fp32_kernel(D, 1, H, L, bm) == kernel
    q, k, v = _rand(H, L, D, seed=L + H)
    Mq, Nk = -(-L // bm), -(-L // bn)
    m = torch.from_numpy(random_map(1, H, Mq, Nk, L, p=(0.15, 0.25, 0.2, 0.2, 0.2), ensure_row=False)).to(torch.int8).to(dev())
    check(q, k, v, m, bm, bn, causal)


@pytest.mark.parametrize("H,kernels", [
    (2, {64: ("direct", 16), 128: ("direct", 16)}),
    (100, {64: ("direct", 16), 128: ("tiles", 32)}),
    (176, {64: ("direct", 32), 128: ("tiles", 64)}),
])
@pytest.mark.parametrize("L,bm,bn,causal", [(131, 64, 64, False), (192, 64, 32, True), (145, 64, 128, True), (144, 64, 32, False)])
@pytest.mark.parametrize("D", [64, 128])
def test_fwd_splits(H, kernels, L, bm, bn, causal, D):
    from psa_hip import ops

    Mq, Nk = -(-L // bm), -(-L // bn)
    assert fp32_kernel(D, 1, H, L, bm) == kernels[D]
    q, k, v = _rand(H, L, D, seed=L + H)
    m = torch.from_numpy(random_map(1, H, Mq, Nk, L, p=(0.15, 0.25, 0.2, 0.2, 0.2), ensure_row=False)).to(torch.int8).to(dev())
    o, lse, pools = ops.sparse_attention_fwd(q, k, v, m, bm, bn, causal=causal, return_lse=True)
    ro, rl = _reference(q, k, v, m, pools, bm, bn, causal)
    assert float((o.double() - ro).abs().max()) <= 2e-5
    empty = rl == float("-inf")
    assert torch.equal(lse == float("-inf"), empty)
    assert float((lse.double() - rl).masked_fill(empty, 0.0).abs().max()) <= 2e-5


@pytest.mark.parametrize("H,D", [(2, 64), (120, 64), (341, 64), (2, 128), (100, 128), (171, 128)])  # every kernel
def test_infinite_values_stay_in_their_channel(H, D):
    """An infinite value gives its channel an infinity; slots without a key (a sequence of 131 tokens, lists that end inside a tile) none."""
    from psa_hip import ops

    q, k, v = _rand(H, 131, D, seed=9)
    v[:, :, 130, 3] = float("inf")
    m = torch.ones(1, H, 3, 3, dtype=torch.int8, device=dev())
    m[:, :, 1, 2] = 0
    o = ops.sparse_attention_fwd(q, k, v, m, 64, 64)
    assert torch.isinf(o[:, :, :64, 3]).all() and torch.isinf(o[:, :, 128:, 3]).all()
    o[..., 3] = 0
    assert torch.isfinite(o).all() and torch.isfinite(ops.sparse_attention_fwd(q, k, v, m, 64, 64)[:, :, 64:128]).all()


@pytest.mark.parametrize("L,bn", [(131, 64), (4099, 32), (192, 128)])  # partly filled tiles (192: an empty one)
@pytest.mark.parametrize("H", [4, 100, 171])  # 16, 32 and 64 rows per workgroup (head dim 64: 16, 16 and 32), as long as L is short
@pytest.mark.parametrize("lv", [1, 2, 8])
@pytest.mark.parametrize("D", [64, 128])
def test_infinite_value_stays_infinite(H, L, bn, lv, D):
    """Every query sees the last key, whose value is +inf in one channel: that channel is +inf for every query (weights of
    order 1 / L times inf; the empty slots of the last tile add nothing) and the others are finite."""
    from psa_hip import ops

    H = min(H, 4 * 4099 // L)
    q, k, v = _rand(H, L, D, seed=L)
    v[:, :, L - 1, 5] = float("inf")
    m = torch.full((1, H, -(-L // 64), -(-L // bn)), lv, dtype=torch.int8, device=dev())
    o = ops.sparse_attention_fwd(q, k, v, m, 64, bn)
    assert bool((o[..., 5] == float("inf")).all())
    assert bool(torch.isfinite(o[..., [c for c in range(D) if c != 5]]).all())


@pytest.mark.parametrize("D,Hq,Hkv,kernel", [(64, 20, 5, ("direct", 16)), (64, 64, 16, ("direct", 32)), (64, 170, 34, ("tiles", 64)), (128, 20, 5, ("direct", 16)),
                                             (128, 64, 16, ("tiles", 32)), (128, 88, 2, ("tiles", 64))])
@pytest.mark.parametrize("indexed", [False, True])
def test_batches_shared_heads_and_index(D, Hq, Hkv, kernel, indexed):
    """Two batches, query heads that share kv heads, and queries read and written through a token index."""
    from psa_hip import ops

    B, L, bm, bn = 2, 177, 64, 64
    assert fp32_kernel(D, B, Hq, L, bm) == kernel
    g = torch.Generator().manual_seed(Hq + D)
    q, k, v = (torch.randn(B, h, L, D, generator=g).to(dev()) for h in (Hq, Hkv, Hkv))
    m = torch.from_numpy(random_map(B, Hq, 3, 3, Hq, p=(0.15, 0.25, 0.2, 0.2, 0.2), ensure_row=False)).to(torch.int8).to(dev())
    index = torch.randperm(L, generator=g).to(torch.int32).to(dev()) if indexed else None
    o, lse, _ = ops.sparse_attention_fwd(q, k, v, m, bm, bn, return_lse=True, q_index=index)
    at = torch.arange(L, device=dev()) if index is None else index.long()
    kx, vx = (t.repeat_interleave(Hq // Hkv, 1).contiguous() for t in (k, v))
    ro, rl = _reference(q[:, :, at], kx, vx, m, ops.pool_kv(kx, vx, bn), bm, bn, False)
    assert float((o[:, :, at].double() - ro).abs().max()) <= 2e-5
    empty = rl == float("-inf")
    assert torch.equal(lse[:, :, at] == float("-inf"), empty)
    assert float((lse[:, :, at].double() - rl).masked_fill(empty, 0.0).abs().max()) <= 2e-5
