"""The antidiagonal contraction at the edges of its tiles, stages and key blocks, on either output tile, against the oracle in 64 bits.

Tolerance: a logit is a sum of at most 1024 products of N(0, 1) numbers in fp32.  Its rounding is about sqrt(1024) * 2^-24 of the sum of
their magnitudes (650), 1.2e-3, times log2(e) / (sqrt(D) * stride) <= 0.05 (D = 64, stride 4: 512 products), so below 3e-5 in the exponent and of a
score; 1e-4 is taken."""
import numpy as np
import pytest
import torch

import psa_oracle as O
from gpu_util import dev, rnd, xattn_tile

pytestmark = pytest.mark.gpu


def _check(q, k, block, stride, chunk, causal, heads=None):
    from psa_hip import ops

    got = ops.estimate_xattn(q, k, block_size=block, stride=stride, causal=causal, chunk_size=chunk).cpu()
    rep = q.shape[1] // k.shape[1]
    for h in heads or range(q.shape[1]):
        ref = O.estimate_xattn(q[:, h:h + 1].cpu().double(), k[:, h // rep:h // rep + 1].cpu().double(), block_size=block, stride=stride,
                               causal=causal, chunk_size=chunk, dtype=torch.float64)
        np.testing.assert_allclose(got[:, h:h + 1].numpy(), ref.numpy(), rtol=1e-4, atol=1e-9)


@pytest.mark.parametrize("Hq,Hkv,Lq,Lk,D,block,stride,chunk,causal,tile", [
    (64, 64, 4096, 4096, 64, 64, 8, 1024, True, ("large", 1)),     # key blocks of 8 strided keys
    (60, 30, 3999, 3999, 128, 128, 8, 1024, True, ("large", 1)),   # ... of 16, the last group of tokens partly past the sequence
    (28, 28, 2050, 2050, 64, 128, 4, 512, False, ("large", 1)),    # ... of 32; half a tile past the padded rows
    (64, 64, 2050, 2050, 64, 128, 4, 512, False, ("small", 1)),
    (64, 64, 1024, 4096, 64, 128, 4, 512, True, ("large", 1)),     # queries at the end of longer keys
    (64, 32, 2050, 2050, 128, 128, 4, 2048, False, ("large", 3)),  # one tile after the other, whole chunks of padding
    (170, 85, 3999, 3999, 64, 64, 8, 1024, True, ("large", 2)),    # ... masked and unmasked ones
    (2, 1, 129, 129, 128, 128, 16, 2048, True, ("small", 1)),
    (3, 3, 1025, 1025, 64, 64, 8, 1024, False, ("small", 1)),
    (1, 1, 1, 1, 64, 128, 4, 512, True, ("small", 1)),
    (2, 2, 500, 500, 64, 32, 1, 128, True, ("small", 1)),          # a single stage
    (2, 2, 515, 515, 128, 32, 1, 128, False, ("small", 1)),        # two
    (64, 64, 1100, 1100, 64, 32, 1, 128, True, ("small", 1)),
    (34, 34, 1100, 1100, 64, 32, 1, 128, True, ("large", 2)),      # a single stage (a second one of zeros) per tile, one tile after the other
])
def test_edges(Hq, Hkv, Lq, Lk, D, block, stride, chunk, causal, tile):
    assert xattn_tile(Hq, Lq, Lk, block, stride, chunk, causal) == tile
    q, k = rnd(1, Hq, Lq, D, seed=Lq).to(dev()), rnd(1, Hkv, Lk, D, seed=Lk + 1).to(dev())
    _check(q, k, block, stride, chunk, causal, heads=(0, Hq // 2, Hq - 1))


@pytest.mark.parametrize("step", [0, 8, 56])
@pytest.mark.parametrize("which", ["q", "k", "both"])
def test_rows_that_overlap(step, which):
    """Row strides below the head dim: what lies behind the last row is not outside the tensor's memory."""
    H, L, D = 2, 300, 64
    def tensor(overlap, seed):
        if not overlap:
            return rnd(1, H, L, D, seed=seed).to(dev())
        flat = rnd(1, 1, H, (L + 64) * max(step, 8) + D, seed=seed).to(dev())
        return flat.as_strided((1, H, L, D), (flat.numel(), flat.shape[3], step, 1))
    _check(tensor(which != "k", 1), tensor(which != "q", 2), 128, 8, 1024, True)


def test_stride_of_a_single_row():
    q = rnd(1, 2, 1, 64, seed=1).to(dev()).as_strided((1, 2, 1, 64), (128, 64, 0, 1))
    _check(q, q, 128, 8, 1024, True)


def test_layouts():
    """[B, L, H, D] projections, a slice of a wider one, and heads far apart."""
    x = rnd(2, 700, 3, 256, seed=5).to(dev())
    q, k = x[..., :128].transpose(1, 2), x[..., 128:].transpose(1, 2)
    from psa_hip import ops

    a = ops.estimate_xattn(q, k, 128, 8, True, 1024)
    assert torch.equal(a, ops.estimate_xattn(q.contiguous(), k.contiguous(), 128, 8, True, 1024))
    _check(q[1:], k[1:], 128, 8, 1024, True)
