"""The reference's hot-path functions, same signatures, running in libmdx.so.

Tensors must live on the GPU; every kernel is enqueued on torch's current
stream, allocates nothing itself (outputs and workspaces come from torch's
caching allocator, so the calls are safe under graph capture) and never
synchronises.  Argument checks, allocation and the C calls are done by the native host
module (csrc/host_ops.cpp); the functions here name the arguments and say what they mean.
"""
from __future__ import annotations

import torch

from . import _lib
from ._lib import MdxError, check

_native = None


def _host():
    """The native host module, loaded on the first call of an op."""
    global _native
    if _native is None:
        _native = _lib.host()
    return _native


# --------------------------------------------------------------------------- store_kvcache
def store_kvcache(key: torch.Tensor, value: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
                  slot_mapping: torch.Tensor) -> None:
    """nanovllm/layers/attention.py:33-40: key/value [N, Hkv, d] (row stride free, rows dense),
    caches [pages, page, Hkv, d], slot_mapping [N] int32 with -1 = skip.  In place."""
    _host().store_kvcache(key, value, k_cache, v_cache, slot_mapping)


def store_kvcache_maybe4d(k, v, k_cache, v_cache, slot_mapping) -> None:
    """nanovllm/layers/sdar_attention.py:11-16: [b, s, h, d] inputs are flattened to [(b s), h, d]."""
    _host().store_kvcache_maybe4d(k, v, k_cache, v_cache, slot_mapping)


def qk_norm_rope_store(qkv: torch.Tensor, q_weight: torch.Tensor, k_weight: torch.Tensor, eps: float,
                       cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                       num_q_heads: int, num_kv_heads: int, head_dim: int,
                       k_cache: torch.Tensor | None = None, v_cache: torch.Tensor | None = None,
                       slot_mapping: torch.Tensor | None = None, want_k: bool = True):
    """One launch for nanovllm/models/sdar.py:79-83 plus the cache store: qkv [..., (Hq+2Hkv)*d]
    -> (q [..., Hq, d], k [..., Hkv, d] or None, v view [..., Hkv, d]); rotated k and raw v are
    written to the caches at slot_mapping when caches are given.  cos/sin: fp32 [max_pos, d/2]."""
    return _host().qk_norm_rope_store(qkv, q_weight, k_weight, eps, cos, sin, positions, num_q_heads, num_kv_heads, head_dim,
                                      k_cache, v_cache, slot_mapping, want_k)


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, residual: torch.Tensor | None = None):
    """RMSNorm.forward (nanovllm/layers/layernorm.py:43-51): returns the normed x, or with a
    residual the pair (normed x + residual, x + residual), in one launch."""
    return _host().rms_norm(x, weight, eps, residual)


def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
    """SiluAndMul.forward (nanovllm/layers/activation.py:13-16): x [..., 2I] -> silu(x[..., :I]) * x[..., I:]."""
    return _host().silu_and_mul(x)


# --------------------------------------------------------------------------- linear layers
# Partial sums ([splits, ..., n] fp32) are the product's sums over slices of K, which rms_norm_partials and
# qk_norm_rope_store_partials add up on their way.  None where the library's product is the better one (many rows) or the
# shape is not covered.
def linear(x: torch.Tensor, weight: torch.Tensor, partials: bool = False) -> torch.Tensor | None:
    """x . weight^T (nanovllm/layers/linear.py) for up to 1536 rows (wide layers: up to 52 GFLOP): bf16 [..., n], or with
    `partials` what is the faster of that and partial sums (one dimension more than x).  Without, a layer of long K and few
    columns is slower than the library's (2048 x 6144: 25 us against 17 at 32 rows, 54 against 45 at 1536)."""
    return _host().linear(x, weight, partials)


def linear_gated(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor | None:
    """silu_and_mul(x . weight^T) in one launch, beyond 8192 rows where weight has 2048 rows or more and twice as many as columns (nanovllm/models/sdar.py:105-111)."""
    return _host().linear_gated(x, weight)


def linear_qk_norm_rope_store(x, weight, q_weight, k_weight, eps, cos, sin, positions, num_q_heads, num_kv_heads, head_dim,
                              k_cache=None, v_cache=None, slot_mapping=None, want_kv: bool = True):
    """qk_norm_rope_store(x . weight^T, ...) for 384 to 1536 rows and heads of 128 columns in one launch (nanovllm/models/sdar.py:73-83
    and the cache store): (q, k, v), k and v None unless wanted.  None where two launches are the faster."""
    return _host().linear_qk_norm_rope_store(x, weight, q_weight, k_weight, eps, cos, sin, positions, num_q_heads, num_kv_heads, head_dim,
                                             k_cache, v_cache, slot_mapping, want_kv)


def linear_partials(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor | None:
    """The partial sums of up to 128 rows, also where there is one slice only."""
    return _host().linear_partials(x, weight)


def linear_silu(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor | None:
    """linear_gated for up to 64 rows (weight rows a multiple of 48, k of 512)."""
    return _host().linear_silu(x, weight)


def rms_norm_partials(partials: torch.Tensor, weight: torch.Tensor, eps: float, residual: torch.Tensor):
    """rms_norm(x, weight, eps, residual) with x given as partial sums."""
    return _host().rms_norm_partials(partials, weight, eps, residual)


def qk_norm_rope_store_partials(partials, q_weight, k_weight, eps, cos, sin, positions, num_q_heads, num_kv_heads, head_dim,
                                k_cache, v_cache, slot_mapping) -> torch.Tensor:
    """The decode form of qk_norm_rope_store with qkv given as partial sums: returns q; k and v go to the caches."""
    return _host().qk_norm_rope_store_partials(partials, q_weight, k_weight, eps, cos, sin, positions, num_q_heads, num_kv_heads, head_dim,
                                               k_cache, v_cache, slot_mapping)


# --------------------------------------------------------------------------- staircase prefill
def sparse_attn_varlen(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cu_seqlens_q: torch.Tensor,
                       cu_seqlens_k: torch.Tensor, staircase_size: int = 4, *, max_seqlen: int | None = None,
                       softmax_scale: float | None = None) -> torch.Tensor:
    """block_prefill_attention_v2.py:168-202: q [N, Hq, d], k/v [N, Hkv, d] packed over
    sequences, cu_seqlens int32 [B+1], blocks of `staircase_size` right-aligned; returns o like q.
    max_seqlen (keyword, not in the reference) sizes the grid and must be >= the longest sequence:
    rows beyond it are not computed, and the lengths live on the device, so this call cannot check
    it.  None (the default) takes the total token count, which is always enough; the engine passes
    the value it computed on the host while building cu_seqlens (Context.max_seqlen_k)."""
    return _host().sparse_attn_varlen(q, k, v, cu_seqlens_q, cu_seqlens_k, staircase_size, max_seqlen, softmax_scale)


sparse_attn_varlen_v2 = sparse_attn_varlen


# --------------------------------------------------------------------------- paged decode
def flash_attn_with_kvcache(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, *,
                            cache_seqlens: torch.Tensor, block_table: torch.Tensor,
                            softmax_scale: float | None = None, causal: bool = False,
                            counters: torch.Tensor | None | bool = None) -> torch.Tensor:
    """The subset of flash_attn.flash_attn_with_kvcache used at sdar_attention.py:50-55:
    q [bs, Sq, Hq, d], caches [pages, page, Hkv, d], block_table [bs, max_pages] int32,
    cache_seqlens [bs] int32, non-causal.  Returns o like q.

    counters (keyword, not in the reference): None = single launch, where that pays, with this module's arrival
    counters (per device and stream, one buffer for eager calls and one for captured ones, which only launches that need them
    take); a zeroed fp32 tensor of the caller's = the same with those; False = attention launch + combine launch."""
    if causal:
        raise MdxError("flash_attn_with_kvcache: only causal=False (block-diffusion decode) is implemented")
    return _host().flash_attn_with_kvcache(q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale, counters)


def flash_attn_with_kvcache_read_ahead(q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale, next_weight, then_weight,
                                       counters: torch.Tensor | None | bool = None) -> torch.Tensor:
    """flash_attn_with_kvcache in a decode pass, whose launch also reads the weights of the two products behind it where it leaves the
    chip idle (up to 256 rows): the same result; the products find them in the device's cache."""
    return _host().flash_attn_with_kvcache_read_ahead(q, k_cache, v_cache, cache_seqlens, block_table, softmax_scale, next_weight, then_weight, counters)


# --------------------------------------------------------------------------- unmask step
def gumbel_noise(rows: int, vocab: int, seed: int, offset: int = 0, device=None,
                 offset_dev: torch.Tensor | None = None, row_ids: torch.Tensor | None = None) -> torch.Tensor:
    """The [rows, vocab] fp32 noise tensor that `seed` / `offset` stand for in confidence_argmax and
    unmask_step: passing it as `noise` gives the same result as passing the two integers."""
    out = torch.empty((rows, vocab), dtype=torch.float32, device=device if device is not None else "cuda")
    if not out.is_cuda:
        raise MdxError("mdx ops run on the GPU only: got a tensor on " + str(out.device))
    if offset_dev is not None:
        assert offset_dev.dtype == torch.int64 and offset_dev.numel() == 1 and offset_dev.is_cuda
    if row_ids is not None:
        assert row_ids.dtype == torch.int64 and row_ids.numel() == rows and row_ids.is_contiguous() and row_ids.is_cuda
    rc = _lib.lib().mdx_gumbel_noise(out.data_ptr(), out.stride(0) if rows else vocab, rows, vocab, int(seed) & (2 ** 64 - 1),
                                     int(offset) & (2 ** 64 - 1), None if offset_dev is None else offset_dev.data_ptr(),
                                     None if row_ids is None else row_ids.data_ptr(),
                                     torch.cuda.current_stream(out.device).cuda_stream)
    check(rc, "gumbel_noise")
    return out


def confidence_argmax(logits: torch.Tensor, temperatures: torch.Tensor | None = None,
                      noise: torch.Tensor | None = None, seed: int | None = None, offset: int = 0,
                      offset_dev: torch.Tensor | None = None, row_ids: torch.Tensor | None = None):
    """Sampler.prepare (nanovllm/layers/sampler.py:11-22):
    logits [bs, S, V], temperatures [bs] or [bs, 1] fp32 -> (x0 int64 [bs, S], x0_p fp32 [bs, S]).
    The Gumbel noise that the reference adds to logits/T before the argmax is either an explicit tensor
    `noise` ([bs, S, V] fp32), or drawn inside the kernel from (`seed`, `offset`): a counter-based
    generator, so the same integers give the same tokens (give every step another offset; `offset_dev`,
    a one-element int64 device tensor, is added to it at run time; `row_ids` [rows] int64 names the
    generator row of each logits row when rows were compacted).  Neither = plain argmax."""
    return _host().confidence_argmax(logits, temperatures, noise, seed, offset, offset_dev, row_ids)


def lm_head_confidence(x: torch.Tensor, weight: torch.Tensor, temperatures: torch.Tensor | None = None,
                       rows_per_temp: int | None = None, row_ids: torch.Tensor | None = None):
    """ParallelLMHead.forward's F.linear(x, weight) (nanovllm/layers/embed_head.py:61-67) followed by
    Sampler.prepare without noise (layers/sampler.py:11-22), in one pass that never writes the logits:
    x [..., hidden] bf16, weight [vocab, hidden] bf16 -> (x0 int64 [...], x0_p fp32 [...]) = argmax and softmax
    confidence of bf16(x . weight^T) / T.  temperatures [n] fp32: row r uses entry (row_ids[r] if given else r)
    // rows_per_temp (default rows / n), so that compacted rows keep the temperature of their sequence."""
    return _host().lm_head_confidence(x, weight, temperatures, rows_per_temp, row_ids)


def filter_logits(logits: torch.Tensor, top_k: int = 0, top_p: float = 1.0,
                  temperatures: torch.Tensor | None = None, out: torch.Tensor | None = None) -> torch.Tensor:
    """top_k_logits then top_p_logits of the HF variant (modeling_mineru_diffusion.py:585-600, in the
    order of :608-611) on bf16 / fp16 logits [..., V]: a copy (or `out`, which may be `logits`) with
    every element below the row's cut-off set to -inf.  Feed the result to confidence_argmax /
    unmask_step; their `noise` input (Gumbel) then samples from the filtered distribution.  top_k = 0
    and top_p >= 1 switch the respective filter off.  temperatures as for confidence_argmax (they
    enter the top-p probabilities only)."""
    return _host().filter_logits(logits, top_k, top_p, temperatures, out)


def num_transfer_tokens(block_length: int, steps: int) -> list[int]:
    """get_num_transfer_tokens (modeling_mineru_diffusion.py:617-623): how many positions each denoising step of a
    block commits at least -- block_length split over the steps, the remainder given to the first steps.  The k of
    unmask_step / select_transfer for step i is entry min(i, steps - 1) (modeling_mineru_diffusion.py:712)."""
    base, rem = divmod(int(block_length), int(steps))
    return [base + (1 if i < rem else 0) for i in range(int(steps))]


def select_transfer(x0: torch.Tensor, x0_p: torch.Tensor, tokens: torch.Tensor, mask_token_id: int,
                    threshold: float, k: int = 1):
    """Device form of the selection loop (sampler.py:32-54, modeling_mineru_diffusion.py:518-532).
    tokens [bs, S] int64 is updated in place; returns (transfer bool [bs, S], count int32 [bs])."""
    return _host().select_transfer(x0, x0_p, tokens, mask_token_id, threshold, k)


def unmask_step(logits: torch.Tensor, tokens: torch.Tensor, mask_token_id: int, threshold: float, k: int = 1,
                temperatures: torch.Tensor | None = None, noise: torch.Tensor | None = None,
                top_k: int = 0, top_p: float = 1.0, seed: int | None = None, offset: int = 0,
                offset_dev: torch.Tensor | None = None):
    """One whole unmask step on the device: logits [bs, S, V], tokens [bs, S] int64 (in place).
    Returns (x0, x0_p, transfer, count).  top_k / top_p (off by default, as in
    modeling_mineru_diffusion.py:602,633-634) put filter_logits in front of the step; `noise` or
    (`seed`, `offset`, `offset_dev`) as for confidence_argmax."""
    return _host().unmask_step(logits, tokens, mask_token_id, threshold, k, temperatures, top_k, top_p,
                               noise, seed, offset, offset_dev, None)