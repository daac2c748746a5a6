"""The work that users of this framework have it do, as cases that can be timed.

Five kinds of use, all at the shapes of the language model that the engine serves (16 query heads, 8 KV heads of 128
columns, blocks of 32 positions, pages of 256 tokens, a vocabulary of 151 936, 28 layers of width 2048):

  prefill   mdx.Attention in its prefill mode: one layer stores the K/V rows of packed prompts and attends over them
  decode    mdx.Attention in its decode mode: one layer stores the block's K/V rows and attends over the paged cache
  unmask    the denoising step on logits: mdx.unmask_step (plain, sampled, or behind the top-k / top-p filter) and
            mdx.Sampler, which takes its blocks from the host and returns them there as the engine's runner has it
  head      mdx.lm_head_confidence: vocabulary projection and confidence without logits in memory
  generate  mdx.engine.BlockDiffusionEngine: requests in, finished token blocks out (prefill, decode, unmask, page
            allocation and scheduling together), with the decode passes captured as graphs

Prompt lengths and context lengths of a case are spread evenly between "shortest" and "longest", the same for every seed:
only the values change with the seed.
"""
import math
import os
import random
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "mineru-diffusion_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import mdx  # noqa: E402
from mdx.engine import BlockDiffusionEngine, Decoder, DecoderConfig, SamplingParams, Sequence  # noqa: E402

HQ, HKV, D, BLOCK, PAGE = 16, 8, 128, 32, 256
VOCAB, HIDDEN, INTERMEDIATE, LAYERS, MASK_ID = 151936, 2048, 6144, 28, 151669
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
QKV = (HQ + 2 * HKV) * D


# ----------------------------------------------------------------------------- the cases
def listed():
    return [
        # a single short prompt (a line of text, a formula): the prefill call is a handful of launches
        {"name": "prefill, one short prompt", "kind": "prefill", "dtype": "f16", "seqs": 1, "shortest": 77, "longest": 77},
        # a few document pages admitted together: about 1024 vision tokens and a short instruction each
        {"name": "prefill, six pages", "kind": "prefill", "dtype": "bf16", "seqs": 6, "shortest": 900, "longest": 1500},
        # benchmark config 3: long, ragged packed prompts
        {"name": "prefill, config 3", "kind": "prefill", "dtype": "bf16", "seqs": 8, "shortest": 1024, "longest": 8192},
        # benchmark config 1: one block over a prefix of 1024 tokens, fp32
        {"name": "decode, config 1 fp32", "kind": "decode", "dtype": "f32", "seqs": 1, "shortest": 1024, "longest": 1024},
        # one user, one page being read: what a block costs in latency
        {"name": "decode, one sequence", "kind": "decode", "dtype": "bf16", "seqs": 1, "shortest": 1337, "longest": 1337},
        # benchmark config 2: a batch of ragged contexts
        {"name": "decode, config 2", "kind": "decode", "dtype": "bf16", "seqs": 16, "shortest": 512, "longest": 4096},
        # benchmark config 4: the denoising step of a full batch
        {"name": "unmask, config 4", "kind": "unmask", "call": "step", "dtype": "bf16", "seqs": 32, "temperature": 1.0,
         "sampled": False, "top_k": 0, "top_p": 1.0, "k": 4},
        # the runner's sampler call with the reference's own sampling (Gumbel noise), a few sequences
        {"name": "unmask, sampler, three", "kind": "unmask", "call": "sampler", "dtype": "bf16", "seqs": 3, "temperature": 0.8,
         "sampled": True, "top_k": 0, "top_p": 1.0, "k": 1},
        # the HF variant's generate loop: top-k and top-p filters in front of a sampled step
        {"name": "unmask, filtered", "kind": "unmask", "call": "step", "dtype": "bf16", "seqs": 12, "temperature": 0.7,
         "sampled": True, "top_k": 50, "top_p": 0.9, "k": 4},
        # the head of a decode pass in which about half of the positions of a batch of 32 are still masked
        {"name": "head, 500 rows", "kind": "head", "rows": 500, "temperature": 1.0},
        # one request through the engine: every pass is a few dozen rows deep
        {"name": "generate, one request", "kind": "generate", "requests": 1, "prefix": 1024, "prompt": 64, "new": 128, "k": 4},
        # benchmark config 5, shortened to 128 of its 2048 generated tokens: a full batch through the engine
        {"name": "generate, config 5", "kind": "generate", "requests": 32, "prefix": 1024, "prompt": 64, "new": 128, "k": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "decode", "decode", "unmask", "unmask", "head", "generate"])
    if kind == "prefill":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        seqs = _log(rng, 1, 16)
        most = min(8192, (4096 if dtype == "f32" else 32768) // seqs)     # fp32 prompts are small ones, for checking
        longest = _log(rng, 40, most)
        return {"kind": kind, "dtype": dtype, "seqs": seqs, "shortest": _log(rng, max(8, longest // 8), longest), "longest": longest}
    if kind == "decode":
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        seqs = _log(rng, 1, 8 if dtype == "f32" else 64)
        longest = _log(rng, 100, min(16384, 150000 // seqs))
        return {"kind": kind, "dtype": dtype, "seqs": seqs, "shortest": _log(rng, max(32, longest // 8), longest), "longest": longest}
    if kind == "unmask":
        call = rng.choice(["step", "step", "sampler"])
        filtered = call == "step" and rng.random() < 0.4
        return {"kind": kind, "call": call, "dtype": rng.choice(["bf16", "bf16", "f16"]), "seqs": _log(rng, 1, 24 if call == "sampler" else 32),
                "temperature": round(rng.choice([1.0, rng.uniform(0.5, 1.5)]), 2), "sampled": rng.random() < 0.5,
                "top_k": rng.choice([0, 20, 50, 400]) if filtered else 0, "top_p": rng.choice([0.8, 0.9, 0.95]) if filtered else 1.0,
                "k": 1 if call == "sampler" else rng.choice([1, 2, 4])}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 4, 1024), "temperature": round(rng.choice([1.0, rng.uniform(0.5, 1.5)]), 2)}
    return {"kind": kind, "requests": _log(rng, 1, 16), "prefix": rng.choice([0, _log(rng, 64, 1024)]), "prompt": _log(rng, 16, 512),
            "new": BLOCK * rng.randint(1, 4), "k": rng.choice([2, 4, 8])}


def _lengths(case):
    """One length from each of the equal parts of the range, in mixed order."""
    n, lo, hi = case["seqs"], case["shortest"], case["longest"]
    rng = random.Random("%d %d %d" % (n, lo, hi))
    lens = [lo + int((i + rng.random()) / n * (hi + 1 - lo)) for i in range(n)]
    rng.shuffle(lens)
    return lens


# ----------------------------------------------------------------------------- inputs
def _tables(counts, spare, gen):
    """Page tables over a pool of randomly ordered pages, as a server that has run for a while has them."""
    pool = sum(counts) + spare
    order = torch.randperm(pool, generator=gen).tolist()
    tables, at = [], 0
    for n in counts:
        tables.append(order[at:at + n])
        at += n
    return tables, pool


def _slots(table, lo, hi):
    return [table[t // PAGE] * PAGE + t % PAGE for t in range(lo, hi)]


def _qkv(tokens, dtype, gen):
    """q, k as the rotary embedding leaves them, v a view of the fused projection's output."""
    fused = torch.randn(tokens, QKV, generator=gen, device="cuda", dtype=torch.float32).to(dtype)
    q = fused[:, :HQ * D].reshape(tokens, HQ, D).contiguous()
    k = fused[:, HQ * D:(HQ + HKV) * D].reshape(tokens, HKV, D).contiguous()
    return q, k, fused[:, (HQ + HKV) * D:].view(tokens, HKV, D)


def _prepare_prefill(case, gen, host):
    lens = [n + BLOCK for n in _lengths(case)]            # the prompt and the block to be denoised, which is not stored
    dtype = DTYPES[case["dtype"]]
    tables, pool = _tables([-(-n // PAGE) for n in lens], 8, host)
    slots, cu = [], [0]
    for n, table in zip(lens, tables):
        slots += _slots(table, 0, n - BLOCK) + [-1] * BLOCK
        cu.append(cu[-1] + n)
    attn = mdx.Attention(HQ, D, D ** -0.5, HKV)
    attn.k_cache = torch.zeros(pool, PAGE, HKV, D, dtype=dtype, device="cuda")
    attn.v_cache = torch.zeros_like(attn.k_cache)
    q, k, v = _qkv(cu[-1], dtype, gen)
    cu = torch.tensor(cu, dtype=torch.int32, device="cuda")
    return {"attn": attn, "q": q, "k": k, "v": v,
            "context": (True, cu, cu, max(lens), max(lens), torch.tensor(slots, dtype=torch.int32, device="cuda"), None, None, BLOCK)}


def _prepare_decode(case, gen, host):
    prefix, dtype = _lengths(case), DTYPES[case["dtype"]]
    tables, pool = _tables([-(-(n + BLOCK) // PAGE) for n in prefix], 8, host)
    width = max(len(t) for t in tables)
    attn = mdx.Attention(HQ, D, D ** -0.5, HKV)
    attn.k_cache = torch.empty(pool, PAGE, HKV, D, dtype=dtype, device="cuda").normal_(generator=gen)
    attn.v_cache = torch.empty_like(attn.k_cache).normal_(generator=gen)
    q, k, v = _qkv(len(prefix) * BLOCK, dtype, gen)
    shape = (len(prefix), BLOCK)
    slots = [_slots(t, n, n + BLOCK) for t, n in zip(tables, prefix)]
    table = [t + [-1] * (width - len(t)) for t in tables]
    i32 = dict(dtype=torch.int32, device="cuda")
    return {"attn": attn, "q": q.view(*shape, HQ, D), "k": k.view(*shape, HKV, D), "v": v.unflatten(0, shape),
            "context": (False, None, None, 0, 0, torch.tensor(slots, **i32), torch.tensor([n + BLOCK for n in prefix], **i32),
                        torch.tensor(table, **i32), BLOCK)}


def _prepare_unmask(case, gen, host):
    n, dtype = case["seqs"], DTYPES[case["dtype"]]
    logits = torch.empty(n, BLOCK, VOCAB, dtype=dtype, device="cuda")
    for row in logits:
        row.copy_(torch.randn(BLOCK, VOCAB, generator=gen, device="cuda") * 3)
    # the model is sure of some positions: one token of every third row stands clear of the rest
    sure = logits.view(-1, VOCAB)[::3]
    sure.scatter_(1, torch.randint(0, VOCAB, (sure.shape[0], 1), generator=gen, device="cuda"),
                  (20 + 4 * torch.rand(sure.shape[0], 1, generator=gen, device="cuda")).to(dtype))
    tokens = torch.randint(0, 1000, (n, BLOCK), generator=host)
    for row in tokens:                                    # between half and all of a block is still masked
        left = int(torch.randint(BLOCK // 2, BLOCK + 1, (1,), generator=host))
        row[torch.randperm(BLOCK, generator=host)[:left]] = MASK_ID
    seed = int(torch.randint(0, 1 << 30, (1,), generator=host))
    temps = torch.full((n, 1), case["temperature"], device="cuda")
    state = {"case": case, "logits": logits, "temps": temps}
    if case["call"] == "sampler":
        params = SamplingParams(temperature=case["temperature"])
        state["seqs"] = [Sequence([1, 2, 3], params, BLOCK, MASK_ID) for _ in range(n)]
        state["blocks"] = list(tokens)
        state["sampler"] = mdx.Sampler(k=case["k"], seed=seed if case["sampled"] else None)
    else:
        state["tokens"] = tokens.cuda()
        state["options"] = dict(top_k=case["top_k"], top_p=case["top_p"], seed=seed if case["sampled"] else None, offset=7)
    return state


def _prepare_head(case, gen, host):
    weight = torch.empty(VOCAB, HIDDEN, dtype=torch.bfloat16, device="cuda").normal_(0.0, 0.02, generator=gen)
    x = torch.randn(case["rows"], HIDDEN, generator=gen, device="cuda")
    # every third row points at a token, as the hidden state of a position that the model is sure of does
    sure = x[::3]
    sure += 25 * weight[torch.randint(0, VOCAB, (sure.shape[0],), generator=gen, device="cuda")].float()
    x = x * torch.rsqrt(x.square().mean(1, keepdim=True))
    return {"x": x.to(torch.bfloat16), "weight": weight, "temps": torch.full((case["rows"],), case["temperature"], device="cuda")}


def _prepare_generate(case, gen, host):
    weights, pages = torch.randint(0, 1 << 30, (2,), generator=host).tolist()
    with torch.device("cuda"):
        model = Decoder(DecoderConfig(), "cuda", seed=weights)
    # Random weights predict by a hair's breadth.  A trained model mostly does not, and only then does every correct
    # way of summing commit the same tokens: the head finds the token after the one that the embedding put in, and
    # the embeddings are large enough to be found behind 28 layers.
    model.lm_head.data.copy_(model.embed_tokens.data.roll(1, 0))
    model.embed_tokens.data.mul_(400)
    new, length = case["new"], case["prefix"] + case["prompt"]
    engine = BlockDiffusionEngine(model, num_pages=case["requests"] * (-(-(length + new) // PAGE) + 1), decode_graphs=True,
                                  shuffle_pages_seed=pages, max_model_len=2048)
    # no position is sure enough for the threshold, so k are committed in every pass
    params = SamplingParams(max_new_tokens=new, ignore_eos=True, transfer_count=case["k"], dynamic_threshold=1.0)
    requests = []
    for _ in range(case["requests"]):
        ids = [0] * case["prefix"] + torch.randint(0, 151000, (case["prompt"],), generator=host).tolist()
        vision = torch.empty(case["prefix"], HIDDEN, dtype=torch.bfloat16, device="cuda").normal_(0.0, 8.0, generator=gen) if case["prefix"] else None
        requests.append((ids, vision))
    return {"engine": engine, "params": params, "requests": requests}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    make = {"prefill": _prepare_prefill, "decode": _prepare_decode, "unmask": _prepare_unmask, "head": _prepare_head,
            "generate": _prepare_generate}[case["kind"]]
    return dict(make(case, gen, host), kind=case["kind"])


# ----------------------------------------------------------------------------- one pass
def run(state):
    kind = state["kind"]
    if kind in ("prefill", "decode"):
        attn = state["attn"]
        mdx.set_context(*state["context"])
        return {"o": attn(state["q"], state["k"], state["v"]), "k_cache": attn.k_cache, "v_cache": attn.v_cache}
    if kind == "unmask":
        if state["case"]["call"] == "sampler":
            for seq, block in zip(state["seqs"], state["blocks"]):
                seq.current_denoising_block = block
            count = state["sampler"](state["logits"], state["temps"], state["seqs"])
            return {"count": count, "blocks": [s.current_denoising_block for s in state["seqs"]],
                    "step_maps": [s.current_step_map for s in state["seqs"]]}
        tokens = state["tokens"].clone()                  # the step commits in place
        x0, x0_p, transfer, count = mdx.unmask_step(state["logits"], tokens, MASK_ID, 0.9, state["case"]["k"], temperatures=state["temps"],
                                                    **state["options"])
        return {"x0": x0, "x0_p": x0_p, "transfer": transfer, "count": count, "tokens": tokens}
    if kind == "head":
        x0, x0_p = mdx.lm_head_confidence(state["x"], state["weight"], state["temps"])
        return {"x0": x0, "x0_p": x0_p}
    engine = state["engine"]
    seqs = [engine.add_request(ids, state["params"], prefix_embeds=vision) for ids, vision in state["requests"]]
    engine.generate()
    return {"tokens": torch.tensor([s.completion_token_ids for s in seqs]), "kv_cache": engine.kv_cache}


# ----------------------------------------------------------------------------- what a pass cannot do without
def _visible_pairs(n):
    """(query, key) pairs of a sequence of n tokens whose blocks are aligned to its end."""
    first = n % BLOCK or BLOCK
    pairs, end = first * first, first
    while end < n:
        end += BLOCK
        pairs += BLOCK * end
    return pairs


def _attention_work(kind, lens, size):
    """Bytes and operations of one attention layer: `lens` holds the tokens of each prompt with its block (prefill) or of
    each context with its block (decode)."""
    if kind == "prefill":
        tokens = sum(lens)
        stored = tokens - BLOCK * len(lens)
        return (tokens * (QKV + HQ * D) + 2 * stored * HKV * D) * size, 4 * D * HQ * sum(_visible_pairs(n) for n in lens)
    rows = BLOCK * len(lens)
    return (rows * (2 * HQ + 2 * HKV) * D + 2 * sum(lens) * HKV * D) * size, 4 * D * HQ * BLOCK * sum(lens)


def work(case):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        size = 4 if case["dtype"] == "f32" else 2
        by, fl = _attention_work(kind, [n + BLOCK for n in _lengths(case)], size)
        return {"bytes": by, "flops": fl}
    if kind == "unmask":
        logits = case["seqs"] * BLOCK * VOCAB
        return {"bytes": 2 * logits + case["seqs"] * BLOCK * 29, "flops": 4 * logits}
    if kind == "head":
        return {"bytes": 2 * (VOCAB + case["rows"]) * HIDDEN + 12 * case["rows"], "flops": 2 * case["rows"] * VOCAB * HIDDEN}
    n, length, blocks = case["requests"], case["prefix"] + case["prompt"], case["new"] // BLOCK
    layer = HIDDEN * (QKV + HQ * D + 3 * INTERMEDIATE)
    steps = BLOCK // case["k"]
    # the prefill pass is the first denoising pass of the first block; its head sees every position of the block
    by, fl = _attention_work("prefill", [length + BLOCK] * n, 2)
    by, fl = LAYERS * (by + 2 * layer), LAYERS * (fl + 2 * n * (length + BLOCK) * layer)
    by, fl = by + 2 * VOCAB * HIDDEN, fl + 2 * n * BLOCK * VOCAB * HIDDEN
    for b in range(blocks):
        for step in range(1 if b == 0 else 0, steps + 1):
            a_by, a_fl = _attention_work("decode", [length + (b + 1) * BLOCK] * n, 2)
            by, fl = by + LAYERS * (a_by + 2 * layer), fl + LAYERS * (a_fl + 2 * n * BLOCK * layer)
            rows = n * (BLOCK - step * case["k"])         # positions that are still masked; none in the pass that stores the block
            if rows:
                by, fl = by + 2 * VOCAB * HIDDEN, fl + 2 * rows * VOCAB * HIDDEN
    return {"bytes": by, "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind in ("prefill", "decode"):
        # outputs and probabilities of 16 bits; fp32 tensors are summed and rounded in fp32
        return {"rel": 1e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 1e-2, "max": 0.1}
    if kind == "unmask":
        # confidences are fp32 sums over the vocabulary; a decision on a rounding boundary may fall either way
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.002}
    if kind == "head":
        # a logit on a rounding boundary lands on either of two bf16 values
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    # K and V rows of every layer, through activations of 16 bits
    return {"rel": 2e-2, "max": 0.5}
