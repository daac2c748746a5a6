"""The two layers that own the hot path, as the engine defines them."""
from __future__ import annotations

import torch
from torch import nn

from .context import get_context
from .ops import _host


class Attention(nn.Module):
    """nanovllm/layers/sdar_attention.py:19-57: store the step's K/V into the paged cache,
    then staircase attention over the packed prompt (prefill) or non-causal attention of
    the current block over the cache (decode).  Inputs arrive through the global Context."""

    def __init__(self, num_heads, head_dim, scale, num_kv_heads):
        super().__init__()
        self.num_heads = num_heads
        self.head_dim = head_dim
        self.scale = scale
        self.num_kv_heads = num_kv_heads
        self.k_cache = self.v_cache = torch.tensor([])

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor):
        context = get_context()
        if context.is_prefill:
            # the prefill attention reads k / v, not the cache: the store rides in its launch where the rows allow it
            return _host().attention_prefill(q, k, v, self.k_cache, self.v_cache, context.slot_mapping, context.cu_seqlens_q,
                                             context.cu_seqlens_k, context.block_size, context.max_seqlen_k, self.scale)
        return _host().attention_decode(q, k, v, self.k_cache, self.v_cache, context.slot_mapping, context.context_lens,
                                        context.block_tables, self.scale, context.counters)


class Sampler(nn.Module):
    """nanovllm/layers/sampler.py:6-61.  The device does the whole step (confidence, argmax,
    selection); only the [bs, S] results cross to the host to update the Sequence objects.

    `k` is the number of positions committed when fewer than k exceed the threshold
    (1 = the engine's rule, sampler.py:44-50).  The Gumbel term of sampler.py:15-18 comes from `seed`
    (drawn inside the kernel by a counter-based generator; every call takes the next offset, so a seed
    reproduces a run) or from `noise_fn(logits) -> fp32 noise`; neither = plain argmax."""

    def __init__(self, k: int = 1, noise_fn=None, seed: int | None = None):
        super().__init__()
        assert noise_fn is None or seed is None, "either a noise function or a seed"
        self.k = k
        self.noise_fn = noise_fn
        self.seed = seed
        self.calls = 0                                      # the generator offset of the next call

    def _noise_args(self, logits):
        if self.seed is not None:
            self.calls += 1
            return dict(seed=self.seed, offset=self.calls - 1)
        return dict(noise=self.noise_fn(logits) if self.noise_fn is not None else None)

    def prepare(self, logits: torch.Tensor, temperatures: torch.Tensor):
        from .ops import confidence_argmax
        return confidence_argmax(logits, temperatures, **self._noise_args(logits))

    def forward(self, logits: torch.Tensor, temperatures: torch.Tensor, seqs) -> int:
        strategy = seqs[0].sampling_params.denoising_strategy
        if strategy != 'low_confidence_dynamic':
            raise NotImplementedError(f"Denoising strategy {strategy} not implemented")
        noise = self._noise_args(logits)
        blocks, committed = _host().sampler_step(
            logits, temperatures, [seq.current_denoising_block for seq in seqs], [seq.current_step_map for seq in seqs],
            [seq.current_denoise_step for seq in seqs], seqs[0].mask_token_id, seqs[0].sampling_params.dynamic_threshold, self.k,
            noise.get("noise"), noise.get("seed"), noise.get("offset", 0), None, None)
        for seq, block in zip(seqs, blocks):
            seq.current_denoising_block = block
            seq.current_denoise_step += 1
        return committed
