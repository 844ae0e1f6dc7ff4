"""The draw of the sampling offsets against its own definition on the host: the positions of the largest of `block` 64-bit keys, in decreasing
order, for full, short and single-token blocks."""
import pytest
import torch

from gpu_util import dev

pytestmark = pytest.mark.gpu
M = (1 << 64) - 1


def _mix(x):
    x = (x + 0x9E3779B97F4A7C15) & M
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) & M
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) & M
    return x ^ (x >> 31)


@pytest.mark.parametrize("block_m,keep_m,block_n,keep_n", [(128, 32, 64, 16), (128, 128, 128, 1), (100, 33, 33, 33), (1, 1, 31, 8), (97, 97, 96, 5)])
def test_offsets_are_the_positions_of_the_largest_keys(block_m, keep_m, block_n, keep_n):
    from psa_hip import ops

    seed = 987654321
    got = ops.draw_sample_offsets(2, 3, 1, block_m, keep_m, block_n, keep_n, dev(), seed=seed)
    for off, tag, block, keep in zip(got, (0x71717171, 0x6B6B6B6B), (block_m, block_n), (keep_m, keep_n)):
        off = off.flatten(0, 1).cpu()
        for bh in range(off.shape[0]):
            keys = [_mix((_mix(seed ^ tag) + (bh << 20) + i) & M) & ~0xFF | i for i in range(block)]
            assert off[bh].tolist() == sorted(range(block), key=lambda i: -keys[i])[:keep]
            assert off.dtype == torch.int32
