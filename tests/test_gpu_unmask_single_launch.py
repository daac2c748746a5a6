"""GPU parity: the unmask step whose vocabulary pass selects by itself, against the call of two launches, which the other tests hold against the
oracle.  Both compute the same sums in the same order: equal bit for bit.  Every case runs twice on the same arrival counters, which a call has to leave at zero."""
import pytest
import torch

pytestmark = pytest.mark.gpu
MASK_ID = 151669


def _data(bs, S, V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    logits = (torch.randn(bs, S, V, generator=g) * 3).to(dtype)
    logits.view(-1, V)[::3, V // 2] += 20                                 # some positions above the threshold
    tokens = torch.randint(0, 1000, (bs, S), generator=g)
    tokens[torch.rand(bs, S, generator=g) < 0.7] = MASK_ID
    tokens[0] = MASK_ID
    return logits, tokens, 0.5 + torch.rand(bs, generator=g)


def _two_launches(logits, tokens, temps, seed, offset, threshold, k):
    import mdx
    L, dev = mdx.lib(), logits.device
    bs, S, V = logits.shape
    x0, p = torch.empty(bs, S, dtype=torch.int64, device=dev), torch.empty(bs, S, device=dev)
    transfer, count = torch.empty(bs, S, dtype=torch.bool, device=dev), torch.empty(bs, dtype=torch.int32, device=dev)
    n = L.mdx_confidence_argmax_workspace_bytes(bs * S, V)
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device=dev)
    dtype = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[logits.dtype]
    rest = (tokens.data_ptr(), MASK_ID, threshold, k, x0.data_ptr(), p.data_ptr(), transfer.data_ptr(), count.data_ptr(), bs, S, V, ws.data_ptr(), n,
            torch.cuda.current_stream().cuda_stream)
    if seed is None:
        rc = L.mdx_unmask_step(logits.data_ptr(), V, dtype, temps.data_ptr(), None, 0, *rest)
    else:
        rc = L.mdx_unmask_step_gumbel(logits.data_ptr(), V, dtype, temps.data_ptr(), seed, offset, None, None, *rest)
    assert rc == 0, L.mdx_last_error()
    return x0, p, transfer, count


# one split per row and several (1024 rows are the limit), blocks of one position, of a whole wavefront's and beyond one (two launches), rows
# of less than a 16-byte chunk, splits that every lane of the merge takes one, none or two of
@pytest.mark.parametrize("bs, S, V", [(1, 1, 7), (1, 32, 151936), (3, 32, 40000), (2, 64, 100003), (33, 32, 5000), (2, 65, 20000), (40, 3, 50000)])
@pytest.mark.parametrize("seed", [None, 5])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_step_equals_two_launches(dev, bs, S, V, seed, dtype):
    import mdx
    for call in range(2):
        logits, tokens, temps = _data(bs, S, V, dtype, 100 * call + S)
        logits, temps = logits.to(dev), temps.to(dev)
        one, two = tokens.to(dev), tokens.to(dev)
        x0, p, transfer, count = mdx.unmask_step(logits, one, MASK_ID, 0.9, 2, temperatures=temps, seed=seed, offset=3)
        ex0, ep, et, ec = _two_launches(logits, two, temps, seed, 3, 0.9, 2)
        torch.cuda.synchronize()
        assert torch.equal(x0, ex0) and torch.equal(p, ep)
        assert torch.equal(transfer, et) and torch.equal(count, ec) and torch.equal(one, two)


# rows of masked positions only, on both sides of the row count from which the sampler takes one launch; a sequence without any
@pytest.mark.parametrize("bs, unmasked", [(2, None), (7, None), (7, 3), (12, 0)])
@pytest.mark.parametrize("seed", [None, 9])
def test_sampler_equals_step(dev, bs, unmasked, seed):
    import mdx
    from mdx.engine import SamplingParams, Sequence
    S, V = 32, 30000
    sampler = mdx.Sampler(k=2, seed=seed)
    for call in range(2):
        logits, tokens, temps = _data(bs, S, V, torch.bfloat16, 7 + call)
        if unmasked is not None:
            tokens[unmasked] = 11
        logits, temps = logits.to(dev), temps.to(dev)
        seqs = [Sequence([1, 2, 3], SamplingParams(), S, MASK_ID) for _ in range(bs)]
        for s, row in zip(seqs, tokens):
            s.current_denoising_block = row.clone()
            s.current_denoise_step = 5
        committed = sampler(logits, temps, seqs)
        want = tokens.to(dev)
        _, _, transfer, count = mdx.unmask_step(logits, want, MASK_ID, seqs[0].sampling_params.dynamic_threshold, 2, temperatures=temps, seed=seed, offset=call)
        assert committed == int(count.sum())
        assert torch.equal(torch.stack([s.current_denoising_block for s in seqs]), want.cpu())
        assert torch.equal(torch.stack([s.current_step_map for s in seqs]) == 5, transfer.cpu())


def test_captured_step_keeps_no_counters(dev):
    """A graph may be replayed beside other work: a captured step makes its two launches, and its replays equal the eager step."""
    import mdx
    logits, tokens, temps = _data(3, 32, 40000, torch.bfloat16, 3)
    logits, temps, start = logits.to(dev), temps.to(dev), tokens.to(dev)
    want = start.clone()
    eager = mdx.unmask_step(logits, want, MASK_ID, 0.9, 2, temperatures=temps)
    block = start.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        mdx.unmask_step(logits, block, MASK_ID, 0.9, 2, temperatures=temps)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = mdx.unmask_step(logits, block, MASK_ID, 0.9, 2, temperatures=temps)
    for _ in range(3):
        block.copy_(start)
        graph.replay()
        mdx.unmask_step(logits, start.clone(), MASK_ID, 0.9, 2, temperatures=temps)
        torch.cuda.synchronize()
        assert torch.equal(block, want)
        for a, b in zip(out, eager):
            assert torch.equal(a, b)


# counters that a call is given are used whatever mdx.unmask_step would choose: many arrivals at one, many rows, and what lies between
@pytest.mark.parametrize("bs, S, V", [(1, 32, 151936), (1, 64, 151936), (3, 48, 151936), (80, 32, 1000), (70, 32, 5000), (4, 64, 151936)])
@pytest.mark.parametrize("seed", [None, 5])
def test_given_counters_are_used(dev, bs, S, V, seed):
    import mdx
    L = mdx.lib()
    counters = torch.zeros(L.mdx_unmask_step_counter_bytes(bs, S) // 4, dtype=torch.int32, device=dev)
    for call in range(2):
        logits, tokens, temps = _data(bs, S, V, torch.bfloat16, 50 * call + bs)
        logits, temps = logits.to(dev), temps.to(dev)
        one, two = tokens.to(dev), tokens.to(dev)
        x0, p = torch.empty(bs, S, dtype=torch.int64, device=dev), torch.empty(bs, S, device=dev)
        transfer, count = torch.empty(bs, S, dtype=torch.bool, device=dev), torch.empty(bs, dtype=torch.int32, device=dev)
        n = L.mdx_confidence_argmax_workspace_bytes(bs * S, V)
        ws = torch.empty(max(n, 16), dtype=torch.uint8, device=dev)
        rc = L.mdx_unmask_step_single_launch(logits.data_ptr(), V, 0, temps.data_ptr(), None, 0, int(seed is not None), seed or 0, 3, None, one.data_ptr(), MASK_ID, 0.9, 2,
                                             x0.data_ptr(), p.data_ptr(), transfer.data_ptr(), count.data_ptr(), bs, S, V, ws.data_ptr(), n,
                                             counters.data_ptr(), counters.nbytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, L.mdx_last_error()
        ex0, ep, et, ec = _two_launches(logits, two, temps, seed, 3, 0.9, 2)
        torch.cuda.synchronize()
        assert torch.equal(x0, ex0) and torch.equal(p, ep) and torch.equal(transfer, et) and torch.equal(count, ec) and torch.equal(one, two)
        assert not bool(counters.any())
