"""Maps counted in shares (psa_density_stats) against one workgroup per map (psa_density): the same bits from one share to more shares than lanes
add up at once, below and above 256 maps."""
import pytest
import torch

from gpu_util import dev, random_map
from test_gpu_density import density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Mq,Nk", [(1, 12, 256, 1024), (2, 48, 140, 556), (1, 257, 33, 65), (2, 128, 16, 64), (1, 1, 2000, 2001), (1, 5, 300, 300)])
@pytest.mark.parametrize("causal", [False, True])
def test_shares(B, H, Mq, Nk, causal):
    from psa_hip import ops

    m = torch.from_numpy(random_map(B, H, Mq, Nk, Nk)).to(torch.int8).to(dev())
    ref = density(m, causal)
    d, sparsity, per_head = ops.density_stats(m, causal=causal)
    assert torch.equal(d, ref) and torch.equal(sparsity, 1.0 - ref[-1])
    rows = ref[:-1].view(B, H)
    mean = rows[0].clone()
    for b in range(1, B):
        mean += rows[b]
    assert torch.equal(per_head.flatten(), mean / B)
