"""The 128-key slots of the dK/dV walk that are cut into parts (lists of more than one and a half times the unit, which is 1.7 times the
head's mean list or 4 q-blocks): against the oracle, and a head in a launch of its own against the same head among others."""
import numpy as np
import pytest
import torch

from gpu_util import dev, random_map, rnd
from test_gpu_bwd import run_bwd

pytestmark = pytest.mark.gpu


def _popular(B, H, Mq, Nk, seed, columns):
    """A sparse map whose `columns` every q-block keeps at level 1 (the last one may be the ragged block with the pad rows)."""
    m = random_map(B, H, Mq, Nk, seed, p=(0.7, 0.02, 0.1, 0.1, 0.08))
    m[..., columns] = 1
    return m


@pytest.mark.parametrize("B,Hq,Hkv,L,bm", [
    (1, 2, 2, 4096, 128),      # lists of 32
    (1, 1, 1, 4300, 128),      # a ragged last block among them: pad rows
    (2, 8, 2, 1000, 128),      # four query heads: lists of 32
    (1, 2, 1, 1500, 64),       # 64-row q-blocks
    (1, 8, 1, 1300, 128),      # lists of 88, several parts
    (1, 2, 1, 1024, 128),      # lists of 16: cut at head dim 128
    (1, 1, 1, 1900, 128),      # lists of 15: not cut
])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_cut_slots(B, Hq, Hkv, L, bm, D, causal):
    if causal and bm != 128:
        pytest.skip("causal maps are square")
    Mq, Nk = -(-L // bm), -(-L // 128)
    lmap = _popular(B, Hq, Mq, Nk, L, [0, Nk - 1])
    if causal:
        lmap[..., np.arange(Mq), np.arange(Mq)] = 1
    run_bwd(B, Hq, Hkv, L, D, bm, 128, causal, seed=L + D, lmap=lmap)


@pytest.mark.parametrize("D", [64, 128])
def test_every_slot_long(D):
    """All lists equally long: nothing is cut, whatever their length.  And one long list among empty ones."""
    run_bwd(1, 2, 2, 4200, D, 128, 128, False, seed=1, lmap=np.ones((1, 2, 33, 33), np.int32))
    m = np.zeros((1, 2, 33, 33), np.int32)
    m[0, 0, :, 4] = 1
    m[0, 1, :, 32] = 1
    run_bwd(1, 2, 2, 4200, D, 128, 128, False, seed=2, lmap=m)


@pytest.mark.parametrize("D", [64, 128])
def test_a_head_has_its_bits_in_any_launch(D):
    from psa_hip import ops

    H, L = 6, 128 * 32 + 40
    n = -(-L // 128)
    q, k, v = (rnd(1, H, L, D, seed=i).to(dev()) for i in range(3))
    do = rnd(1, H, L, D, seed=3, scale=0.5).to(dev())
    m = torch.from_numpy(_popular(1, H, n, n, 5, [3, 11, n - 1])).to(dev())

    def grads(h):
        a, b, c, d, lm = (t[:, h].contiguous() for t in (q, k, v, do, m))
        out, lse, pools = ops.sparse_attention_fwd(a, b, c, lm, 128, 128, return_lse=True)
        return ops.sparse_attention_bwd(a, b, c, lm, out, d, lse, 128, 128, pools=pools)

    whole = grads(slice(0, H))
    for h in (0, H - 1):
        for w, g in zip(whole, grads(slice(h, h + 1))):
            assert torch.equal(w[:, h], g[:, 0])
