"""128-key slots of the dK/dV walk that are worked on by two workgroups of 64 keys (launches that the chip holds in about one round, lists of a
quarter of the q-blocks and more): against the oracle at the edges of the rule and of the last block, and a head in a launch on one side of the
rule against the same head on the other: the same bits."""
import numpy as np
import pytest
import torch

from gpu_util import dev, random_map, rnd
from test_gpu_bwd import run_bwd

pytestmark = pytest.mark.gpu


def _halve(D, B, Hq, Hkv, L, bm):
    """Shortest list of a halved slot (psa_bwd.hip, halved_slots); 0: none."""
    slots, lists = B * Hkv * -(-L // 128), Hq // Hkv * -(-L // bm)
    if slots <= 8 or lists < (16 if D == 128 else 32) or slots > min(24 * lists, 768 if D == 128 else 1024):
        return 0
    return lists // 4


def _popular(B, H, Mq, Nk, seed, columns):
    """A sparse map whose `columns` every q-block keeps at level 1."""
    m = random_map(B, H, Mq, Nk, seed, p=(0.7, 0.02, 0.1, 0.1, 0.08))
    m[..., columns] = 1
    return m


def _lengths(m, n_rep, causal):
    """[B, Hkv, Nk] list lengths of the 128-key slots."""
    on = m == 1
    if causal:
        on = on & (np.arange(m.shape[3])[None, :] <= np.arange(m.shape[2])[:, None])
    B, H, Mq, Nk = on.shape
    return on.reshape(B, H // n_rep, n_rep * Mq, Nk).sum(2)


@pytest.mark.parametrize("B,Hq,Hkv,L,bm,D,causal", [
    (1, 4, 2, 1024, 128, 128, False),   # lists of 16, 16 slots
    (1, 3, 3, 1900, 128, 128, False),   # lists of 15: whole
    (1, 8, 4, 2048, 128, 64, True),     # lists of 32
    (1, 9, 9, 3968, 128, 64, False),    # lists of 31: whole
    (1, 2, 2, 2048 + 40, 128, 128, False),   # the last token in the first half, the second one without keys; pad rows
    (1, 2, 2, 2048 + 64, 128, 128, True),    # the first half full
    (1, 2, 2, 2048 + 65, 128, 128, False),   # one token in the second half
    (1, 1, 1, 4096 + 127, 128, 64, True),
    (2, 4, 2, 1111, 64, 64, False),     # 64-row q-blocks, two query heads and two batches
    (1, 6, 2, 1300, 64, 128, False),
])
def test_halved_slots(B, Hq, Hkv, L, bm, D, causal):
    Mq, Nk = -(-L // bm), -(-L // 128)
    m = _popular(B, Hq, Mq, Nk, L, [0, Nk // 2, Nk - 1])
    if causal:
        m[..., np.arange(Mq), np.arange(Mq)] = 1
    halve = _halve(D, B, Hq, Hkv, L, bm)
    whole = L in (1900, 3968)
    assert halve == 0 if whole else (_lengths(m, Hq // Hkv, causal) >= halve).any() and (_lengths(m, Hq // Hkv, causal) < halve).any()
    run_bwd(B, Hq, Hkv, L, D, bm, 128, causal, seed=L + D, lmap=m)


@pytest.mark.parametrize("B,Hq,Hkv,L,bm,causal,columns", [
    (1, 25, 25, 4200, 128, False, [0, 9, 32]),        # 825 slots
    (1, 24, 24, 4201, 128, False, [0, 9, 32]),        # 792, issued in octaves: halved at head dim 64
    (1, 13, 13, 10624, 128, False, [2, 50, 82]),      # 1079
    (1, 120, 60, 1000, 128, False, [0, 7]),           # 480 slots, lists of 16; one head alone: 8 slots
    (1, 16, 4, 33000, 128, False, [0, 100, 256, 257]),  # more than 256 kv-blocks
    (2, 52, 26, 2500, 64, False, [1, 19]),            # 1040, 64-row q-blocks
    (1, 40, 40, 4300, 128, True, [0, 5, 33]),
])
@pytest.mark.parametrize("D", [64, 128])
def test_a_head_has_its_bits_on_either_side(B, Hq, Hkv, L, bm, causal, columns, D):
    from psa_hip import ops

    n, Mq, Nk = Hq // Hkv, -(-L // bm), -(-L // 128)
    q, do = (rnd(B, Hq, L, D, seed=L + i, scale=x).to(dev()) for i, x in ((0, 1.0), (3, 0.5)))
    k, v = (rnd(B, Hkv, L, D, seed=L + i).to(dev()) for i in (1, 2))
    m = _popular(B, Hq, Mq, Nk, L, columns)
    if causal:
        m[..., np.arange(Mq), np.arange(Mq)] = 1
    if L != 1000 and (L, D) != (4201, 64):  # one side whole, the other one with halved slots
        assert _halve(D, B, Hq, Hkv, L, bm) == 0
        least = _halve(D, B, n, 1, L, bm)
        assert least > 0 and (_lengths(m, n, causal) >= least).any()
    m = torch.from_numpy(m).to(dev())

    def grads(h0, h1):
        a, d, lm = (t[:, h0 * n:h1 * n].contiguous() for t in (q, do, m))
        b, c = (t[:, h0:h1].contiguous() for t in (k, v))
        out, lse, pools = ops.sparse_attention_fwd(a, b, c, lm, bm, 128, causal=causal, return_lse=True)
        return ops.sparse_attention_bwd(a, b, c, lm, out, d, lse, bm, 128, causal=causal, pools=pools)

    whole = grads(0, Hkv)
    for h in (0, 1, Hkv - 1):
        for name, w, g in zip("qkv", whole, grads(h, h + 1)):
            assert torch.equal(w[:, h * n:(h + 1) * n] if name == "q" else w[:, h:h + 1], g), (h, "d" + name)
