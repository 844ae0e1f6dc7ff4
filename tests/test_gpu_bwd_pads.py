"""Gradients that land on replicate-pad rows belong to the last real token: its row of dK and dV by itself, for every kind of remainder
(whole pooled rows of pads, pooled rows shared with real tokens, none), with the level-0 slots that add them (128-key blocks) and the
un-pooling pass that does (64 and 32).  The bound is the one of the whole gradients (bf16 products and probabilities: about 4e-3)."""
import numpy as np
import pytest
import torch

import psa_oracle as O
from gpu_util import random_map, rnd
from test_gpu_bwd import REL_L2, rel_l2, run_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bn,left", [(128, n) for n in (1, 2, 7, 8, 63, 64, 65, 120, 127, 128)] + [(64, 1), (64, 37), (64, 64), (32, 5), (32, 31)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_last_token(bn, left, D, causal):
    if causal and bn != 128:
        pytest.skip("causal maps are square")
    L = 2 * 128 + left
    n = -(-L // bn)
    lmap = random_map(1, 2, 3, n, left)
    lmap[:, :, :, -1] = np.array([8, 2, 4])[None, None, :]  # the last block pooled by every q-block, once at each level
    if causal:
        lmap[..., np.arange(3), np.arange(3)] = 1
        lmap[0, 1, 2, 2] = 2  # (pooled on the diagonal)
    _, dk, dv, _, _ = run_bwd(1, 2, 1, L, D, 128, bn, causal, seed=left, lmap=lmap)
    q, k, v = rnd(1, 2, L, D, seed=left), rnd(1, 1, L, D, seed=left + 1), rnd(1, 1, L, D, seed=left + 2)
    _, rk, rv = O.psa_backward_dense(q, k, v, lmap, rnd(1, 2, L, D, seed=left + 3, scale=0.5), 128, bn, causal=causal)
    for got, ref in ((dk, rk), (dv, rv)):
        if float(ref[..., -1, :].abs().max()) > 0:
            assert rel_l2(got[..., -1, :], ref[..., -1, :]) <= REL_L2
        assert torch.isfinite(got.float()).all()
