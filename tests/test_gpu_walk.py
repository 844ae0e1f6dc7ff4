"""The record walks of the forward kernels (64- / 32-key blocks with their fine tiles, rows of any stride, dense rows without
a map) against the walk that compacts the map row inside the kernel: the tiles come in the same order, so outputs and lse
must be the same bits.  The in-kernel walk is the one that is compared with the oracle at the shapes without records."""
import pytest
import torch

from gpu_util import dev, random_map, rnd

pytestmark = pytest.mark.gpu
BM = 128


def _inputs(B, Hq, Hkv, L, D, seed, strided, dtype=torch.bfloat16):
    t = [rnd(B, h, L, D, seed=seed + i).to(dtype).to(dev()) for i, h in enumerate((Hq, Hkv, Hkv))]
    return [x.transpose(1, 2).contiguous().transpose(1, 2) for x in t] if strided else t


def _same(a, b):
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1].nan_to_num(neginf=-1e30), b[1].nan_to_num(neginf=-1e30))


@pytest.mark.parametrize(
    "Hq,Hkv,L,causal,indexed,p",
    [
        (4, 4, 128 * 70, False, False, (0.35, 0.2, 0.15, 0.15, 0.15)),
        (4, 4, 128 * 66 + 5, False, False, (0.2, 0.2, 0.2, 0.2, 0.2)),   # ragged end, partly filled tiles of every level
        (5, 5, 128 * 60 + 33, False, True, (0.5, 0.05, 0.1, 0.1, 0.25)),  # through a token index
        (6, 2, 128 * 50 + 97, True, False, (0.2, 0.2, 0.2, 0.2, 0.2)),   # causal: fine tiles on the diagonal
        (3, 3, 128 * 90, False, False, (0.0, 0.0, 0.0, 0.5, 0.5)),       # fine tiles only
        (3, 1, 128 * 90 + 64, True, False, (0.0, 1.0, 0.0, 0.0, 0.0)),   # most records a row can have
        (280, 280, 70, False, False, (0.0, 0.0, 0.0, 0.1, 0.9)),         # rows of a few blocks
        (280, 280, 128, True, False, (0.9, 0.0, 0.0, 0.05, 0.05)),       # empty rows
    ],
)
@pytest.mark.parametrize("block_n", [128, 64, 32])
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("D", [128, 64])
def test_record_walk_equals_map_walk(monkeypatch, Hq, Hkv, L, causal, indexed, p, block_n, strided, D):
    from psa_hip import ops

    monkeypatch.setattr(ops, "_WALK_MIN_ROWS", 0)
    q, k, v = _inputs(1, Hq, Hkv, L, D, L, strided, torch.float16 if L % 2 else torch.bfloat16)
    Mq, Nk = -(-L // BM), -(-L // block_n)
    lmap = torch.from_numpy(random_map(1, Hq, Mq, Nk, L + 7, p=p, ensure_row=False)).to(torch.int8).to(dev())
    qi = torch.randperm(L, generator=torch.Generator().manual_seed(L)).to(torch.int32).to(dev()) if indexed else None
    kw = dict(causal=causal, return_lse=True, q_index=qi)
    a = ops.sparse_attention_fwd(q, k, v, lmap, BM, block_n, schedule=False, **kw)
    b = ops.sparse_attention_fwd(q, k, v, lmap, BM, block_n, **kw)
    torch.cuda.synchronize()
    _same(a, b)


@pytest.mark.parametrize("H,Hkv,L,causal,block_n", [(2, 2, 1024, False, 128), (3, 3, 1000, False, 64), (2, 1, 1030, True, 128), (2, 2, 66, True, 32),
                                                    (3, 3, 65, False, 128), (2, 2, 961, True, 64)])
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("D", [128, 64])
def test_dense_walk_equals_map_of_ones(H, Hkv, L, causal, block_n, strided, D):
    from psa_hip import ops

    q, k, v = _inputs(2, H, Hkv, L, D, L, strided)
    ones = torch.ones(2, H, -(-L // BM), -(-L // block_n), dtype=torch.int8, device=dev())
    a = ops.sparse_attention_fwd(q, k, v, ones, BM, block_n, causal=causal, return_lse=True, schedule=False)
    b = ops.sparse_attention_fwd(q, k, v, None, BM, block_n, causal=causal, return_lse=True)
    torch.cuda.synchronize()
    _same(a, b)


@pytest.mark.parametrize("block_n,listed", [(32, False), (64, False), (128, True)])
def test_lists_have_a_byte_limit(monkeypatch, block_n, listed):
    """Above the limit a map of 32- / 64-key blocks is walked in the kernel, by the operator and by the layer in one call: same bits,
    and no memory for a list.  (128-key blocks: always listed.)"""
    from psa_hip import ops

    H, L, D = 80, 1800, 64
    q, k, v = _inputs(1, H, H, L, D, L, False)
    lmap = torch.from_numpy(random_map(1, H, -(-L // BM), -(-L // block_n), L)).to(torch.int8).to(dev())
    ratios = {1: (0.0, 0.1), 2: (0.1, 0.15), 4: (0.15, 0.2), 8: (0.2, 0.35), 0: (0.35, 1.0)}
    off_q, off_k = ops.draw_sample_offsets(1, H, H, BM, 32, block_n, block_n // 4, dev(), seed=1)
    idx = torch.randperm(L, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(dev())
    shape = (1, H, H, L, D, BM, block_n)
    calls = []
    one_call = ops._layer_one_call
    monkeypatch.setattr(ops, "_layer_one_call", lambda *a: calls.append(one_call(*a)) or calls[-1])

    def run():
        fwd = lambda: ops.sparse_attention_fwd(q, k, v, lmap, BM, block_n, return_lse=True)
        fwd()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        a = fwd()[:2]
        torch.cuda.synchronize()
        peak = torch.cuda.max_memory_allocated() - before
        return a, ops.psa_layer_fwd(q, k, v, off_q, off_k, ratios, "topk", BM, block_n, 16, token_index=idx), peak

    (a, la, peak_a), n = run(), ops._walk_bytes(q.dtype, *shape)
    assert n > 0
    monkeypatch.setattr(ops, "_WALK_MAX_BYTES", n - 1)
    assert (ops._walk_bytes(q.dtype, *shape) == n) == listed
    b, lb, peak_b = run()
    _same(a, b)
    assert torch.equal(la, lb)
    assert all(c is not None for c in calls)
    assert listed or peak_b < peak_a - n // 2
