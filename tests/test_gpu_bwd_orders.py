"""Issue orders of the backward walks: the row costs and the column costs come from one launch, the sorts of up to three lists
from another; launches with few rows or few kv-blocks leave lists out.  Gradients never depend on the order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (rows of the dQ walk, kv-blocks of the dK/dV walk): rows sorted from 257 on, kv-block slots from 9 on
@pytest.mark.parametrize(
    "B,Hq,Hkv,L,bm,bn",
    [
        (1, 2, 2, 512, 64, 128),  # 16 rows, 8 kv-blocks: no list
        (1, 2, 2, 1111, 128, 128),  # 18 rows, 18 kv-blocks: the two slot lists only
        (1, 66, 2, 500, 128, 128),  # 264 rows, 8 kv-blocks: rows only
        (1, 66, 2, 500, 128, 64),  # 264 rows, 16 kv-blocks of 64: rows and the one slot list
        (1, 33, 11, 1000, 128, 128),  # 264 rows, 88 kv-blocks: all three
    ],
)
@pytest.mark.parametrize("causal", [False, True])
def test_lists_present_and_absent(B, Hq, Hkv, L, bm, bn, causal):
    if causal and bm != bn:
        pytest.skip("causal maps are square")
    from test_gpu_bwd import run_bwd

    run_bwd(B, Hq, Hkv, L, 64, bm, bn, causal, seed=L + Hq + bn)


@pytest.mark.parametrize("D,L,H", [(64, 4201, 24), (64, 4096, 24), (64, 4200, 25), (128, 10624, 10)])
def test_slots_in_classes(D, L, H):
    """More than 768 kv-blocks with heads of up to 5.5 MiB are issued in classes of similar length, head by head: the gradients
    of each head have the bits that the head has in a launch of its own (exact order, no slot twice or left out).  24 heads of
    4096 (768 blocks) are the last on the other side."""
    from gpu_util import dev, random_map, rnd
    from psa_hip import ops

    q, k, v = (rnd(1, H, L, D, seed=L + i).to(dev()) for i in range(3))
    do = rnd(1, H, L, D, seed=L + 3, scale=0.5).to(dev())
    n = -(-L // 128)
    m = torch.from_numpy(random_map(1, H, n, n, L)).to(dev())

    def grads(h):
        a, b, c, d, lm = (t[:, h] for t in (q, k, v, do, m.contiguous()))
        out, lse, pools = ops.sparse_attention_fwd(a, b, c, lm.contiguous(), 128, 128, return_lse=True)
        return ops.sparse_attention_bwd(a, b, c, lm.contiguous(), out, d, lse.contiguous(), 128, 128, pools=pools)

    whole = grads(slice(0, H))
    for h in (0, 1, H // 2, H - 1):
        for w, g in zip(whole, grads(slice(h, h + 1))):
            assert torch.equal(w[:, h], g[:, 0])
