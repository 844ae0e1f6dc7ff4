"""Level maps by quotas without a sorted row, and the density figures of a map, at the sizes where their kernels' branches change."""
import numpy as np
import pytest
import torch

import psa_oracle as O
from gpu_util import dev

pytestmark = pytest.mark.gpu

QUOTAS = {1: (0.0, 0.1), 2: (0.1, 0.15), 4: (0.15, 0.15), 8: (0.15, 0.35), 0: (0.35, 1.0)}
ALL_LEVELS = {1: (0.0, 0.05), 2: (0.05, 0.15), 4: (0.15, 0.25), 8: (0.25, 1.0)}  # the last cut is the end of the row


@pytest.mark.parametrize("Nk,bn,tn", [(256, 128, 32), (257, 128, 32), (320, 64, 32), (1023, 32, 32), (1410, 32, 32), (5000, 32, 16)])
@pytest.mark.parametrize("map_dtype", [torch.int8, torch.int32])
def test_quota_levels_bit_exact(Nk, bn, tn, map_dtype):
    from psa_hip import ops

    rng = np.random.default_rng(Nk)
    s = (rng.random((1, 2, 8, Nk), dtype=np.float32) ** 8).astype(np.float32)
    s[0, 0, 0, Nk // 4: Nk // 4 + 70] = s[0, 0, 0, 0]      # a few more equal scores than a candidate list holds
    s[0, 0, 1, : Nk // 8] = 0.5                            # a cut inside equal scores at the top of the row
    s[0, 0, 2] = 1.0 / Nk                                  # all equal: the column decides
    s[0, 0, 3] = np.exp2(-rng.random(Nk).astype(np.float32) * 120)  # spread beyond the histogram's octaves
    s[0, 0, 4] = 0.0
    s[0, 0, 5] = 1.0 + rng.integers(0, 3, Nk).astype(np.float32) * np.float32(2.0 ** -23)  # neighbouring floats
    for ratios, text in ((QUOTAS, 0), (ALL_LEVELS, 226)):
        ref = O.level_map(s, ratios, text, "topk", blocksize=bn, compute_tile=tn)
        got = ops.level_map(torch.from_numpy(s).to(dev()), ratios, text, "topk", blocksize=bn, compute_tile=tn, map_dtype=map_dtype)
        assert np.array_equal(got.cpu().numpy().astype(np.int32), ref)


@pytest.mark.parametrize("B,H,Mq,Nk", [(1, 1, 1, 1), (1, 3, 5, 7), (2, 5, 65, 129), (1, 2, 300, 1410)])
@pytest.mark.parametrize("causal", [False, True])
def test_density_stats(B, H, Mq, Nk, causal):
    from psa_hip import ops

    rng = np.random.default_rng(Nk)
    m = rng.choice([0, 1, 2, 4, 8], size=(B, H, Mq, Nk), p=(0.4, 0.2, 0.15, 0.15, 0.1)).astype(np.int32)
    m[0, 0, 0, 0] = 3  # not a level: counts nothing
    w = np.select([m == 1, m == 2, m == 4, m == 8], [1.0, 0.5, 0.25, 0.125], 0.0)
    seen = np.tril(np.ones((Mq, Nk))) if causal else np.ones((Mq, Nk))
    ref = (w * seen).sum((2, 3)) / seen.sum()
    for dt in (torch.int8, torch.int32):
        d, sparsity, per_head = ops.density_stats(torch.from_numpy(m).to(dt).to(dev()), causal=causal)
        # every figure is one rounding of an exact count (the means: one more per addition)
        np.testing.assert_allclose(d[:-1].cpu().numpy().reshape(B, H), ref, rtol=1e-6, atol=1e-9)
        np.testing.assert_allclose(float(d[-1]), ref.mean(), rtol=1e-6, atol=1e-9)
        np.testing.assert_allclose(float(sparsity), 1 - ref.mean(), rtol=1e-6)
        np.testing.assert_allclose(per_head.cpu().numpy(), ref.mean(0), rtol=1e-6, atol=1e-9)


def _normal_scores(rows, Nk, deviation, seed):
    """What the block estimate gives for independent normal logits: per key group the best of 8, per q-block the best of 32 rows."""
    g = torch.Generator(device=dev()).manual_seed(seed)
    z = torch.randn(rows, 32, Nk, generator=g, device=dev())
    for _ in range(7):
        z = torch.maximum(z, torch.randn(z.shape, generator=g, device=dev()))
    z = z * deviation
    s = torch.exp(z - z.amax(-1, keepdim=True)).amax(1)
    return (s / s.sum(-1, keepdim=True)).view(1, 1, rows, Nk).contiguous()


@pytest.mark.parametrize("Nk", [257, 1024, 2048, 6144])
@pytest.mark.parametrize("deviation", [0.01, 0.25, 0.5, 1.0])
def test_quota_levels_of_flat_rows(Nk, deviation):
    """Hundreds of keys in the histogram bin of a cut."""
    from psa_hip import ops

    s = _normal_scores(6, Nk, deviation, Nk)
    s[0, 0, 1] = torch.where(torch.arange(Nk, device=dev()) % 3 == 0, s[0, 0, 1, 0], s[0, 0, 1])  # a third of the row ties
    s[0, 0, 2, : Nk // 2] = 0.0
    ref = O.level_map(s.cpu().numpy(), QUOTAS, 0, "topk", blocksize=32, compute_tile=32)
    got = ops.level_map(s, QUOTAS, 0, "topk", blocksize=32, compute_tile=32, map_dtype=torch.int32)
    assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("Nk", [512, 1024, 2048])
def test_flat_rows_cost_about_what_peaked_rows_cost(Nk):
    """Time of flat rows against rows whose bins hold a few keys each, of one kernel on one card.  Each of the three cuts adds a
    descent of about six barriers to a kernel of a dozen: a factor of up to two, measured 1.7 to 2.0.  A search through all bits
    of the key took 8 to 16 times as long, a full sort of the row 2 to 7 times."""
    from psa_hip import ops

    def us(s):
        go = lambda: ops.level_map(s, QUOTAS, 0, "topk", blocksize=32, compute_tile=32, map_dtype=torch.int8)
        go()
        times = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                go()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    flat, peaked = (_normal_scores(64, Nk, d, 1).expand(1, 48, 64, Nk).contiguous() for d in (0.25, 3.0))
    assert us(flat) < 5.0 * us(peaked)
