"""The antidiagonal estimate on its two output tiles: a launch of many heads takes 256 x 256 tiles, the same heads a few at a time
128 x 128 tiles.  The contraction and the reduction of a (row, key block) run in the same order on either, so the scores are the
same bits.  (test_gpu_causal compares the estimate with the oracle.)"""
import pytest
import torch

from gpu_util import dev, rnd, xattn_tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,stride,chunk,D,causal", [
    (60, 4096, 8, 4096, 128, True),    # no edge
    (60, 4000, 8, 4096, 64, True),     # the last tiles reach past the sequence
    (64, 2050, 4, 2048, 64, False),    # two tokens in the last chunk
    (90, 129, 16, 2048, 128, False),   # one partly used tile row
])
def test_tiles_give_the_same_bits(H, L, stride, chunk, D, causal):
    from psa_hip import ops

    kind = lambda heads: xattn_tile(heads, L, L, 128, stride, chunk, causal)[0]
    group = 2
    assert kind(group) == "small"
    if L > 129:
        assert kind(H) == "large"
    q, k = (rnd(1, H, L, D, seed=L + i).to(dev()) for i in range(2))
    whole = ops.estimate_xattn(q, k, 128, stride, causal, chunk)
    for h in range(0, H, 14):
        part = ops.estimate_xattn(q[:, h:h + group], k[:, h:h + group], 128, stride, causal, chunk)
        assert torch.equal(whole[:, h:h + group], part)
