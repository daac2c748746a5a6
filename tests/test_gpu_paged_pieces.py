"""The paged attention's choice of pieces from the lengths (few sequences: pieces of 64 to 512 keys) and the combine launch that
folds them, at lengths around the edges of pieces and of the fold's groups of slots."""
import math

import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ctxs", [[63], [64], [129], [300], [511], [1100], [2049], [16000], [1100, 1], [40, 3000, 700], [600] * 4, [300] * 8, [900] * 16])
@pytest.mark.parametrize("wide", [0, 5])
def test_pieces(dev, ctxs, wide):
    import mdx
    g = torch.Generator().manual_seed(sum(ctxs) + wide)
    hq, hkv, d, page = 4, 2, 128, 256
    counts = [-(-c // page) for c in ctxs]
    pool = sum(counts) + 2
    q = torch.randn(len(ctxs), 32, hq, d, generator=g).bfloat16()
    kc, vc = (torch.randn(pool, page, hkv, d, generator=g).bfloat16() for _ in range(2))
    bt = torch.full((len(ctxs), max(counts) + wide), -1, dtype=torch.int32)
    order, at = torch.randperm(pool, generator=g).int(), 0
    for b, n in enumerate(counts):
        bt[b, :n] = order[at:at + n]
        at += n
    lens = torch.tensor(ctxs, dtype=torch.int32)
    o = mdx.flash_attn_with_kvcache(q.to(dev), kc.to(dev), vc.to(dev), cache_seqlens=lens.to(dev), block_table=bt.to(dev), softmax_scale=1 / math.sqrt(d))
    ref = oracle.paged_block_attn(q, kc, vc, bt, lens, 1 / math.sqrt(d))
    assert (o.float().cpu() - ref).abs().max().item() < 2e-2


@pytest.mark.parametrize("ctxs", [[1030], [1400], [2048], [1, 3500], [3500, 200], [3584, 3584]])
def test_pieces_folded_twelve_at_a_time(dev, ctxs):
    """Tables wide enough for 8 to 14 pieces of a sequence: fewer, as many and more than the fold asks for at once."""
    test_pieces(dev, ctxs, 0)
