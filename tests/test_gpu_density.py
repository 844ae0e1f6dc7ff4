"""The density entry points of the C ABI: psa_density (no workspace: one workgroup per map) at its own range, and against
psa_density_stats."""
import numpy as np
import pytest
import torch

from gpu_util import dev

pytestmark = pytest.mark.gpu


def density(m, causal):
    """The densities of m's maps and their mean, by psa_density."""
    from psa_hip import _lib

    B, H, Mq, Nk = m.shape
    out = torch.full((B * H + 1,), float("nan"), dtype=torch.float32, device=m.device)
    _lib.check(_lib.lib.psa_density(m.data_ptr(), m.element_size(), B * H, Mq, Nk, int(causal), out.data_ptr(),
                                    torch.cuda.current_stream().cuda_stream))
    return out


@pytest.mark.parametrize("B,H,Mq,Nk", [(1, 1, 1, 1), (1, 3, 5, 7), (2, 5, 65, 129), (3, 100, 4, 9), (1, 2, 300, 1410), (1, 1, 256, 1024)])
@pytest.mark.parametrize("causal", [False, True])
def test_density_without_workspace(B, H, Mq, Nk, causal):
    from psa_hip import ops

    rng = np.random.default_rng(Nk)
    m = rng.choice([0, 1, 2, 4, 8], size=(B, H, Mq, Nk), p=(0.4, 0.2, 0.15, 0.15, 0.1)).astype(np.int32)
    w = np.select([m == 1, m == 2, m == 4, m == 8], [1.0, 0.5, 0.25, 0.125], 0.0)
    seen = np.tril(np.ones((Mq, Nk))) if causal else np.ones((Mq, Nk))
    ref = ((w * seen).sum((2, 3)) / seen.sum()).reshape(-1)
    for dt in (torch.int8, torch.int32):
        t = torch.from_numpy(m).to(dt).to(dev())
        d = density(t, causal)
        # one rounding of an exact count; the mean: one more of a sum in float64
        np.testing.assert_allclose(d.cpu().numpy(), np.append(ref, ref.mean()), rtol=1e-6, atol=1e-9)
        assert torch.equal(d, ops.density(t, causal=causal))


def test_density_of_a_map_whose_count_exceeds_32_bits():
    """2^28 entries of level 1 are 2^31 eighths; both entry points."""
    from psa_hip import ops

    m = torch.ones(1, 1, 1 << 14, 1 << 14, dtype=torch.int8, device=dev())
    assert density(m, False).tolist() == [1.0, 1.0]
    assert ops.density(m).tolist() == [1.0, 1.0]
