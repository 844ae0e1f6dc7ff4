"""The fp32 forward's kernels at the borders of their dispatch: blocks of 16 query rows up to 1280 of them, of 32 above (head dim 64), tiles through
LDS above 3072 (head dim 128) and for rows too far apart for 32-bit offsets; against float64 on the same map and pooled rows.  Tolerance of the
fp32 path: 2e-5 absolute for values of order 1."""
import pytest
import torch

from gpu_util import dev, random_map
from test_gpu_fp32_split import _rand, _reference

pytestmark = pytest.mark.gpu


def _check(q, k, v, m, bm, bn, causal):
    from psa_hip import ops

    o, lse, pools = ops.sparse_attention_fwd(q, k, v, m, bm, bn, causal=causal, return_lse=True)
    ro, rl = _reference(q, k, v, m, pools, bm, bn, causal)
    assert float((o.double() - ro).abs().max()) <= 2e-5
    empty = rl == float("-inf")
    assert torch.equal(lse == float("-inf"), empty)
    assert float((lse.double() - rl).masked_fill(empty, 0.0).abs().max()) <= 2e-5


@pytest.mark.parametrize("D,H,L,bm,bn,causal", [
    (64, 80, 250, 64, 32, False),    # 1280 blocks of 16 rows
    (64, 81, 250, 128, 128, False),  # 1296
    (64, 107, 177, 64, 64, True),    # 1284, a last block of 17 rows
    (128, 256, 180, 64, 64, False),  # 3072
    (128, 257, 180, 64, 32, True),   # 3084
    (128, 400, 100, 128, 64, False), # 3200, one block per head
    (64, 1, 5, 64, 64, False),       # fewer rows than a block
])
def test_borders(D, H, L, bm, bn, causal):
    q, k, v = _rand(H, L, D, seed=L + H)
    Mq, Nk = -(-L // bm), -(-L // bn)
    m = torch.from_numpy(random_map(1, H, Mq, Nk, L, p=(0.15, 0.25, 0.2, 0.2, 0.2), ensure_row=False)).to(torch.int8).to(dev())
    _check(q, k, v, m, bm, bn, causal)


@pytest.mark.parametrize("stride", [1 << 12, (1 << 22) - 8, 1 << 22])
@pytest.mark.parametrize("D", [64, 128])
def test_rows_far_apart(D, stride):
    """K and V rows up to 16 MiB apart; 127 of them end just below, 131 just above offsets of 2^31 bytes."""
    for L in (127, 131):
        q, k, v = _rand(1, L, D, seed=L)
        wide = torch.empty(2 * D + (L - 1) * stride, device=dev())
        k2, v2 = (wide.as_strided((1, 1, L, D), (0, 0, stride, 1), at) for at in (0, D))
        k2.copy_(k)
        v2.copy_(v)
        m = torch.from_numpy(random_map(1, 1, -(-L // 64), -(-L // 32), L, p=(0.0, 0.6, 0.2, 0.1, 0.1))).to(torch.int8).to(dev())
        _check(q, k2, v2, m, 64, 32, False)
        del wide, k2, v2
        torch.cuda.empty_cache()  # (2 GiB)


@pytest.mark.parametrize("H,D", [(2, 64), (120, 64), (2, 128)])
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
