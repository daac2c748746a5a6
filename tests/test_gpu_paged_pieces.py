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


@pytest.mark.parametrize("ctxs,page,hq,hkv", [
    ([700, 64, 65, 63, 1], 32, 4, 2),                       # pages smaller than a tile of 64 keys
    ([700, 300, 96], 96, 4, 2),                             # not a power of two
    ([700, 64, 127, 128, 129], 64, 4, 2),                   # a tile per page
    ([1000, 511, 200], 128, 2, 2), ([900, 511, 200], 64, 2, 2),      # one head per workgroup: tiles of 128 keys, as long as a page and longer
    ([5000] * 2 + [300] * 30, 64, 16, 8),                   # pieces of more pages than a wavefront has lanes
    ([2600] * 16, 256, 16, 8), ([2200] * 16, 256, 16, 8),   # most resident workgroups used: one lookup per pass after the first tiles; with a merging last workgroup
])
def test_tiles_and_pages(dev, ctxs, page, hq, hkv):
    """A tile's keys looked up by page: rows behind the context hold NaN, and one page in the middle of every longer context has an id that does not
    exist, so that its keys are left out."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(sum(ctxs) + page)
    d, scale = 128, 128 ** -0.5
    counts = [-(-c // page) for c in ctxs]
    pool = sum(counts) + 2
    q = torch.randn(len(ctxs), 32, hq, d, generator=g, device=dev).bfloat16()
    kc, vc = (torch.randn(pool, page, hkv, d, generator=g, device=dev).bfloat16() for _ in range(2))
    bt = torch.full((len(ctxs), max(counts)), -1, dtype=torch.int32)
    order, at = torch.randperm(pool, generator=g, device=dev).int().cpu(), 0
    for b, n in enumerate(counts):
        bt[b, :n] = order[at:at + n]
        at += n
        kc[bt[b, n - 1], ctxs[b] - (n - 1) * page:] = float("nan")
        vc[bt[b, n - 1], ctxs[b] - (n - 1) * page:] = float("nan")
    holes = [n // 2 if n > 2 else None for n in counts]
    want = torch.empty(len(ctxs), 32, hq, d)
    for b, n in enumerate(counts):
        rows = [r for r in range(n) if r != holes[b]]
        k, v = (x[bt[b, rows].long().to(dev)].float().flatten(0, 1)[:ctxs[b] - (n - len(rows)) * page].repeat_interleave(hq // hkv, 1) for x in (kc, vc))
        p = torch.softmax(torch.bmm(q[b].float().transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) * scale, -1)
        want[b] = torch.bmm(p, v.transpose(0, 1).contiguous()).transpose(0, 1).cpu()
        if holes[b] is not None:
            bt[b, holes[b]] = -1 if b % 2 else pool + 3
    lens = torch.tensor(ctxs, dtype=torch.int32, device=dev)
    o = mdx.flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, block_table=bt.to(dev), softmax_scale=scale)
    assert (o.float().cpu() - want).abs().max().item() < 2e-2


@pytest.mark.parametrize("bs,hq,hkv,dtype", [(1, 16, 8, torch.bfloat16), (2, 16, 8, torch.bfloat16), (8, 16, 8, torch.bfloat16), (9, 16, 8, torch.bfloat16),
                                             (3, 3, 1, torch.bfloat16), (4, 4, 2, torch.float16), (6, 64, 32, torch.bfloat16), (2, 4, 2, torch.float32)])
def test_reading_ahead_changes_nothing(dev, bs, hq, hkv, dtype):
    """Rows of a pass with readers behind the attention's workgroups and, beyond the rule or for other types, without: the same bits as the
    call that reads nothing, eagerly and from a graph, for weights of any size and layout."""
    import mdx
    from mdx import ops
    g = torch.Generator().manual_seed(bs * hq)
    d, page, ctx = 128, 256, 900
    pool = bs * 4
    q = torch.randn(bs, 32, hq, d, generator=g).to(dtype).to(dev)
    kc, vc = (torch.randn(pool, page, hkv, d, generator=g).to(dtype).to(dev) for _ in range(2))
    bt = torch.randperm(pool, generator=g).int().view(bs, 4).to(dev)
    lens = torch.tensor([ctx - 37 * b for b in range(bs)], dtype=torch.int32, device=dev)
    want = mdx.flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, block_table=bt, softmax_scale=d ** -0.5)
    w = torch.zeros(24 << 20, dtype=torch.bfloat16, device=dev)
    for a, b in ((w[:8], w[:3]), (w[:1 << 20], w), (w, w), (w[1:9], w[:1 << 20].view(1024, 1024).t()), (w[:0], w[:8200])):
        assert torch.equal(ops.flash_attn_with_kvcache_read_ahead(q, kc, vc, lens, bt, d ** -0.5, a, b), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.flash_attn_with_kvcache_read_ahead(q, kc, vc, lens, bt, d ** -0.5, w[:1 << 22], w)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


@pytest.mark.parametrize("bs,pages", [(1, 14), (1, 15), (2, 15), (2, 32)])
def test_reading_ahead_in_wide_tables(dev, bs, pages):
    """Tables on both sides of what leaves each reader of 32 rows a CU (16 heads on 8: 14 pages do, 15 do not), and 64 rows, which do not ask: the same bits."""
    import mdx
    from mdx import ops
    g = torch.Generator().manual_seed(pages)
    q = torch.randn(bs, 32, 16, 128, generator=g).bfloat16().to(dev)
    kc, vc = (torch.randn(pages, 256, 8, 128, generator=g).bfloat16().to(dev) for _ in range(2))
    bt = torch.stack([torch.randperm(pages, generator=g).int() for _ in range(bs)]).to(dev)
    lens = torch.tensor([pages * 256, 1088][:bs], dtype=torch.int32, device=dev)
    w = torch.zeros(24 << 20, dtype=torch.bfloat16, device=dev)
    want = mdx.flash_attn_with_kvcache(q, kc, vc, cache_seqlens=lens, block_table=bt, softmax_scale=128 ** -0.5)
    assert torch.equal(ops.flash_attn_with_kvcache_read_ahead(q, kc, vc, lens, bt, 128 ** -0.5, w[:4 << 20], w), want)


def _spread(n, lo, hi):
    return [lo + (hi - lo) * ((7 * b) % n) // max(1, n - 1) for b in range(n)]


@pytest.mark.parametrize("ctxs,hq,hkv,dtype", [
    (_spread(24, 90, 1500), 16, 8, torch.bfloat16),                        # a pair per CU: cut by shares
    ([0, 0] + _spread(22, 1, 2100), 16, 8, torch.float16),                 # absent sequences among them
    ([4000] + [60] * 23, 16, 8, torch.bfloat16),                           # one far above the rest: as many pieces as there is room for
    ([640] * 24, 16, 8, torch.bfloat16),                                   # whole, all of one length
    ([0, 1100, 0] + [1030 + 3 * b for b in range(29)], 16, 8, torch.bfloat16),   # whole, a pair per CU: sequences taken as they come, absent ones too
    ([1030 + 3 * b for b in range(63)] + [0], 16, 8, torch.float16),       # the most pairs that are resident at once
    ([1030 + 3 * b for b in range(63)] + [0], 18, 9, torch.bfloat16),      # more than that: whole, the longest first
    (_spread(64, 30, 1290), 10, 5, torch.bfloat16),                        # more pairs than CUs
    (_spread(64, 30, 1290), 3, 1, torch.bfloat16),                         # one head per workgroup
    (_spread(8, 700, 2560), 12, 6, torch.bfloat16),                        # few sequences, 10 pages: five and six pieces merged by the last
    (_spread(8, 700, 2561), 12, 6, torch.bfloat16),                        # 11 pages: the combine launch
    (_spread(8, 65, 129), 12, 6, torch.float16),
])
def test_pieces_merged_by_the_last_to_arrive(dev, ctxs, hq, hkv, dtype):
    """One launch whose last split of a pair merges them: the oracle's result and the bits of attention + combine, whichever split is the last, on
    counters that every launch leaves zero; from a graph too, replayed between eager calls on other counters."""
    import mdx
    g = torch.Generator().manual_seed(sum(ctxs) + hq)
    d, page = 128, 256
    counts = [-(-c // page) for c in ctxs]
    pool = sum(counts) + 2
    q = torch.randn(len(ctxs), 32, hq, d, generator=g).to(dtype)
    kc, vc = (torch.randn(pool, page, hkv, d, generator=g).to(dtype) for _ in range(2))
    bt = torch.full((len(ctxs), max(counts)), -1, dtype=torch.int32)
    order, at = torch.randperm(pool, generator=g).int(), 0
    for b, n in enumerate(counts):
        bt[b, :n] = order[at:at + n]
        at += n
    lens = torch.tensor(ctxs, dtype=torch.int32)
    args = (q.to(dev), kc.to(dev), vc.to(dev))
    kw = dict(cache_seqlens=lens.to(dev), block_table=bt.to(dev), softmax_scale=1 / math.sqrt(d))
    two = mdx.flash_attn_with_kvcache(*args, **kw, counters=False)
    assert (two.float().cpu() - oracle.paged_block_attn(q, kc, vc, bt, lens, 1 / math.sqrt(d))).abs().max().item() < 2e-2
    own, other = (torch.zeros(64 * 64, device=dev) for _ in range(2))
    for _ in range(4):
        assert torch.equal(mdx.flash_attn_with_kvcache(*args, **kw, counters=own), two)
        assert own.abs().sum().item() == 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = mdx.flash_attn_with_kvcache(*args, **kw, counters=own)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(mdx.flash_attn_with_kvcache(*args, **kw, counters=other), two)
        torch.cuda.synchronize()
        assert torch.equal(got, two) and own.abs().sum().item() == 0


def _paged_args(dev, ctxs, hq, hkv, seed):
    g = torch.Generator().manual_seed(seed)
    d, page = 128, 256
    counts = [-(-c // page) for c in ctxs]
    q = torch.randn(len(ctxs), 32, hq, d, generator=g).bfloat16().to(dev)
    kc, vc = (torch.randn(sum(counts), page, hkv, d, generator=g).bfloat16().to(dev) for _ in range(2))
    bt, at = torch.full((len(ctxs), max(counts)), -1, dtype=torch.int32), 0
    for b, n in enumerate(counts):
        bt[b, :n] = torch.arange(at, at + n)
        at += n
    return (q, kc, vc), dict(cache_seqlens=torch.tensor(ctxs, dtype=torch.int32, device=dev), block_table=bt.to(dev), softmax_scale=d ** -0.5)


def test_eager_and_captured_calls_count_in_buffers_of_their_own(dev):
    """A graph may be replayed beside eager calls on the stream that it was captured on, so neither uses the other's arrival counters.  Counters that don't begin at
    zero merge nothing: with the other kind's set to a half, each call gives the right result and leaves them alone."""
    import mdx
    from mdx.ops import _host
    many, few = _paged_args(dev, _spread(24, 90, 1500), 16, 8, 1), _paged_args(dev, _spread(16, 300, 1280), 16, 8, 2)   # cut by shares; pieces merged where counters are at hand
    call = lambda case: mdx.flash_attn_with_kvcache(*case[0], **case[1])                               # noqa: E731
    want = [mdx.flash_attn_with_kvcache(*case[0], **case[1], counters=False) for case in (many, few)]
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        assert torch.equal(call(many), want[0]) and torch.equal(call(few), want[1])
        eager, captured = _host().kept_counters(many[0][0])
        torch.cuda.synchronize()
        assert eager.data_ptr() + 4 * eager.numel() <= captured.data_ptr() or captured.data_ptr() + 4 * captured.numel() <= eager.data_ptr()
        assert not eager.any() and not captured.any()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = [call(many), call(few)]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        captured.fill_(0.5)
        assert torch.equal(call(many), want[0]) and torch.equal(call(few), want[1])
        assert not eager.any() and (captured == 0.5).all()
        captured.zero_()
        eager.fill_(0.5)
    torch.cuda.synchronize()
    for _ in range(3):                       # on the current stream, another than the graph was captured on
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want)) and not captured.any() and (eager == 0.5).all()
    eager.zero_()
    torch.cuda.synchronize()


def test_counters_of_the_context_reach_the_attention(dev):
    """mdx.Attention in decode mode counts in the buffer that set_context was given, eagerly and from a graph, not in the kept ones."""
    import mdx
    from mdx.ops import _host
    (q, kc, vc), kw = _paged_args(dev, _spread(24, 90, 1500), 16, 8, 3)
    want = mdx.flash_attn_with_kvcache(q, kc, vc, **kw).flatten(2)
    attn = mdx.Attention(16, 128, 128 ** -0.5, 8)
    attn.k_cache, attn.v_cache = kc, vc
    slots = torch.full((24, 32), -1, dtype=torch.int32, device=dev)                      # (stores nothing)
    own = torch.zeros(64 * 64, device=dev)
    kept = _host().kept_counters(q)
    new = torch.zeros_like(q[:, :, :8])

    def call(counters):
        mdx.set_context(False, slot_mapping=slots, context_lens=kw["cache_seqlens"], block_tables=kw["block_table"], counters=counters)
        try:
            return attn(q, new, new)
        finally:
            mdx.reset_context()
    kept[0].fill_(0.5)                                                                   # (merges nothing)
    got = call(own)
    assert torch.equal(got, want) and not own.any()
    kept[0].zero_()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call(own)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(call(None), want) and torch.equal(call(False), want)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and not own.any()
    with pytest.raises(AssertionError):
        call(own.double())
    assert mdx.get_context().counters is None
