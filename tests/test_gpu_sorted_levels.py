"""Level maps by attention mass, whose rows are sorted: the lengths at which the sort changes (ranking by counting up to 128 scores, bins
beyond, a bitonic network where a bin holds more than 128) against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import psa_oracle as O
from gpu_util import dev

pytestmark = pytest.mark.gpu

MASS = {1: (0.0, 0.3), 2: (0.3, 0.45), 4: (0.45, 0.6), 8: (0.6, 0.8), 0: (0.8, 1.0)}


def _rows(Nk):
    rng = np.random.default_rng(Nk)
    s = (rng.random((1, 1, 10, Nk), dtype=np.float32) ** 8).astype(np.float32)
    s[0, 0, 1] = 1.0 / Nk                                               # all equal: the column decides, one bin
    s[0, 0, 2] = np.exp2(-rng.random(Nk).astype(np.float32) * 140)      # the whole range of a float
    s[0, 0, 3, Nk // 2:] = 0.0                                          # half of the row in the last bin
    s[0, 0, 4] = 1.0 + rng.integers(0, 3, Nk).astype(np.float32) * np.float32(2.0 ** -23)  # neighbouring floats
    s[0, 0, 5, :129] = 0.5                                              # a bin of one more than the limit (or the whole row)
    s[0, 0, 6, :128] = 0.5                                              # a bin at the limit
    s[0, 0, 7] = np.where(rng.random(Nk) < 0.5, np.float32(0.0), np.float32(-0.0))
    s[0, 0, 7, -1] = 1.0
    s[0, 0, 8] = rng.standard_normal(Nk).astype(np.float32) * 1e-3 + 1.0  # flat
    s[0, 0, 9] = np.sort(s[0, 0, 9])                                    # worst last
    return s


@pytest.mark.parametrize("Nk", [1, 64, 127, 128, 129, 255, 256, 257, 511, 513, 1023, 1024, 1025, 2050, 6144])
def test_mass_levels_bit_exact(Nk):
    from psa_hip import ops

    s = _rows(Nk)
    for text in (0, 100):
        ref = O.level_map(s, MASS, text, "thresholdbound", blocksize=64, compute_tile=16)
        got = ops.level_map(torch.from_numpy(s).to(dev()), MASS, text, "thresholdbound", blocksize=64, compute_tile=16, map_dtype=torch.int32)
        assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("S", [2, 128, 129, 200, 300])
@pytest.mark.parametrize("mode", ["energybound", "topk"])
def test_causal_levels_bit_exact(S, mode):
    from psa_hip import ops

    rng = np.random.default_rng(S)
    s = np.tril(rng.random((1, 2, S, S), dtype=np.float32) ** 6).astype(np.float32)
    s /= s.sum(-1, keepdims=True)
    for causal in (False, True):
        ref = O.level_map_qwen(s, MASS, 70, mode, block_size=128, causal=causal)
        got = ops.level_map_qwen(torch.from_numpy(s).to(dev()), MASS, 70, mode, block_size=128, causal=causal)
        assert np.array_equal(got.cpu().numpy(), ref)
