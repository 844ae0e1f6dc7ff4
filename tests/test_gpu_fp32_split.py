"""The fp32 forward at its three splits of a q-block (16, 32 and 64 rows per workgroup: picked by the number of rows in the
launch) and the fp32 contraction at its key shares, against float64 on the same map and pooled rows.  Tolerance of the fp32
path (test_gpu_dtypes): 2e-5 absolute for values of order 1."""
import pytest
import torch

from gpu_util import dev, random_map

pytestmark = pytest.mark.gpu


def _rand(H, L, D, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(1, H, L, D, generator=g).to(dev()) for _ in range(3)]


def _reference(q, k, v, m, pools, bm, bn, causal):
    """(out, lse) in float64: every retained (q-block, kv-block) pair at its level's pooled rows, bias ln(level)."""
    from psa_hip import ops

    B, H, L, D = q.shape
    kl, vl = (ops.pool_levels(p, B, H, L, D, bn) for p in pools)
    rows = m.repeat_interleave(bm, 2)[:, :, :L]
    s, vals = [], []
    for lv in (1, 2, 4, 8):
        kk, vv = (k, v) if lv == 1 else (kl[lv], vl[lv])
        z = torch.matmul(q.double(), kk.double().transpose(-1, -2).contiguous()) * D ** -0.5 + torch.log(torch.tensor(float(lv), dtype=torch.float64))
        keep = rows.repeat_interleave(bn // lv, 3)[..., :kk.shape[2]] == lv
        if causal:
            last = (torch.arange(kk.shape[2], device=q.device) + 1) * lv - 1
            keep = keep & (last[None, :] <= torch.arange(L, device=q.device)[:, None])
        s.append(z.masked_fill(~keep, float("-inf")))
        vals.append(vv.double())
    s, vals = torch.cat(s, -1), torch.cat(vals, 2)
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse.masked_fill(lse == float("-inf"), 0.0)[..., None])
    return torch.matmul(p, vals), lse


@pytest.mark.parametrize("H,rows_per_wg", [(2, 16), (100, 32), (176, 64)])
@pytest.mark.parametrize("L,bm,bn,causal", [(131, 64, 64, False), (192, 64, 32, True), (145, 64, 128, True), (144, 64, 32, False)])
@pytest.mark.parametrize("D", [64, 128])
def test_fwd_splits(H, rows_per_wg, L, bm, bn, causal, D):
    from psa_hip import ops

    Mq, Nk = -(-L // bm), -(-L // bn)
    units = H * Mq * bm // 64
    assert rows_per_wg == (64 if units >= 512 else 32 if 2 * units >= 512 else 16)
    q, k, v = _rand(H, L, D, seed=L + H)
    m = torch.from_numpy(random_map(1, H, Mq, Nk, L, p=(0.15, 0.25, 0.2, 0.2, 0.2), ensure_row=False)).to(torch.int8).to(dev())
    o, lse, pools = ops.sparse_attention_fwd(q, k, v, m, bm, bn, causal=causal, return_lse=True)
    ro, rl = _reference(q, k, v, m, pools, bm, bn, causal)
    assert float((o.double() - ro).abs().max()) <= 2e-5
    empty = rl == float("-inf")
    assert torch.equal(lse == float("-inf"), empty)
    assert float((lse.double() - rl).masked_fill(empty, 0.0).abs().max()) <= 2e-5


@pytest.mark.parametrize("H,L", [(1, 4096), (2, 600), (24, 1500), (3, 64)])  # 4 shares; 1 share; several heads; one step
@pytest.mark.parametrize("block_n,D", [(32, 64), (64, 64), (128, 64), (64, 128)])  # 8, 16 and 32 keys per group
def test_contraction_shares(H, L, block_n, D):
    from psa_hip import ops

    L = -(-L // block_n) * block_n
    Mq, Nk, kn = -(-L // 64), L // block_n, block_n // 4
    q, k, _ = _rand(H, L, D, seed=L)
    off_q, off_k = ops.draw_sample_offsets(1, H, H, 64, 16, block_n, kn, dev(), seed=L)
    got = ops.estimate_sampled(q, k, off_q, off_k, 64, block_n, 16, kn)
    at_q = (torch.arange(Mq, device=dev())[:, None] * 64 + off_q.view(H, 1, 16)).clamp(max=L - 1).reshape(1, H, -1, 1).expand(-1, -1, -1, D)
    at_k = (torch.arange(Nk, device=dev())[:, None] * block_n + off_k.view(H, 1, kn)).reshape(1, H, -1, 1).expand(-1, -1, -1, D)
    z = torch.matmul(q.double().gather(2, at_q), k.double().gather(2, at_k).transpose(-1, -2).contiguous()) * D ** -0.5
    # (the contraction works on whole 64-key steps: the keys that fill the last one repeat the last sampled key)
    fill = (-z.shape[-1]) % 64
    z = torch.cat([z, z[..., -1:].expand(*z.shape[:-1], fill)], -1)
    r = z.view(1, H, Mq * 16, -1, kn).amax(-1)
    p = torch.exp(r - r.amax(-1, keepdim=True)).view(1, H, Mq, 16, -1).amax(3)
    ref = (p / p.sum(-1, keepdim=True))[..., :Nk]
    assert float((got.double() - ref).abs().max()) <= 2e-6


@pytest.mark.parametrize("L,bn", [(131, 64), (4099, 32), (192, 128)])  # partly filled tiles (192: an empty one); 16 and 32 rows per workgroup
@pytest.mark.parametrize("lv", [1, 2, 8])
@pytest.mark.parametrize("D", [64, 128])
def test_infinite_value_stays_infinite(L, bn, lv, D):
    """Every query sees the last key, whose value is +inf in one channel: that channel is +inf for every query (weights of
    order 1 / L times inf; the empty slots of the last tile add nothing) and the others are finite."""
    from psa_hip import ops

    q, k, v = _rand(4, L, D, seed=L)
    v[:, :, L - 1, 5] = float("inf")
    m = torch.full((1, 4, -(-L // 64), -(-L // bn)), lv, dtype=torch.int8, device=dev())
    o = ops.sparse_attention_fwd(q, k, v, m, 64, bn)
    assert bool((o[..., 5] == float("inf")).all())
    assert bool(torch.isfinite(o[..., [c for c in range(D) if c != 5]]).all())
