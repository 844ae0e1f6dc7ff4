"""Issue orders of the backward walks: the row costs and the column costs come from one launch, the sorts of up to three lists
from another; launches with few rows or few kv-blocks leave lists out.  Gradients never depend on the order."""
import pytest

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
