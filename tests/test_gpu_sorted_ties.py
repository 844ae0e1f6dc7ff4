"""Level maps by attention mass whose rows hold scores tied for the worst place: placed in column order apart from a bin of 33 on, whatever the length of the
row (test_gpu_sorted_levels.py has the lengths and the other rows); against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import psa_oracle as O
from gpu_util import dev
from test_gpu_sorted_levels import MASS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nk", [64, 128, 129, 255, 256, 257, 511, 1023, 1024, 2050, 6144])
def test_ties_for_the_worst_place(Nk):
    from psa_hip import ops

    rng = np.random.default_rng(Nk)
    s = (rng.random((1, 1, 5, Nk), dtype=np.float32) ** 8).astype(np.float32)
    s[0, 0, 0] = np.where(rng.random(Nk) < 0.4, np.float32(0.0), s[0, 0, 0])        # in every wave's columns
    s[0, 0, 1] = np.where(rng.random(Nk) < 0.3, s[0, 0, 1].min(), s[0, 0, 1])       # above zero, others in their bin
    s[0, 0, 2] = np.where(rng.random(Nk) < 0.5, np.float32(0.5), s[0, 0, 2])        # ties that are not the worst ...
    s[0, 0, 2, ::3] = 0.0                                                           # ... beside ties that are
    s[0, 0, 3, :33] = s[0, 0, 3].min()                                              # in the first columns only, just enough of them
    s[0, 0, 4, -32:] = s[0, 0, 4].min()                                             # in the last ones, just too few
    for text in (0, 100):
        ref = O.level_map(s, MASS, text, "thresholdbound", blocksize=64, compute_tile=16)
        got = ops.level_map(torch.from_numpy(s).to(dev()), MASS, text, "thresholdbound", blocksize=64, compute_tile=16, map_dtype=torch.int32)
        assert np.array_equal(got.cpu().numpy(), ref)
