"""The C ABI without a GPU: the library loads, exports every symbol include/mdx.h declares,
and refuses bad arguments before launching anything."""
import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def L():
    import mdx
    if not mdx.library_path().exists():
        from importlib import import_module
        import sys
        sys.path.insert(0, str(ROOT))
        import_module("__graft_entry__").build()
    return mdx.lib()


def _declared():
    text = (ROOT / "include" / "mdx.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mdx_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree(L):
    from mdx import _lib
    names = _declared()
    assert names, "no declarations found in include/mdx.h"
    assert sorted(_lib.SIGNATURES) == names
    for n in names:
        assert hasattr(L, n), f"libmdx.so does not export {n}"


def test_version_matches_header(L):
    text = (ROOT / "include" / "mdx.h").read_text()
    assert L.mdx_version() == int(re.search(r"#define MDX_VERSION (\d+)", text).group(1))


def test_workspace_queries_are_pure_host_arithmetic(L):
    assert L.mdx_confidence_argmax_workspace_bytes(1024, 151936) == 0 or \
        L.mdx_confidence_argmax_workspace_bytes(1024, 151936) % 24 == 0
    few = L.mdx_confidence_argmax_workspace_bytes(32, 151936)
    assert few > 0 and few % (32 * 24) == 0            # small batches split rows over workgroups
    ws = L.mdx_paged_block_attn_workspace_bytes(16, 32, 16, 8, 128, 17, 256)
    assert ws > 16 and (ws - 16) % (16 * 16 * 32 * 130 * 4) == 0      # partial slots + the split-size word
    assert L.mdx_paged_block_attn_workspace_bytes(0, 32, 16, 8, 128, 17, 256) == 0


def test_bad_arguments_are_refused_without_a_launch(L):
    null = None
    one = ctypes.c_void_p(16)     # never dereferenced: every call below must fail validation first
    assert L.mdx_store_kvcache(null, null, 0, 0, null, null, null, 5, 1024, 2, 10, null) == -1
    assert b"null" in L.mdx_last_error()
    assert L.mdx_store_kvcache(one, one, 0, 0, one, one, one, 5, 1024, 3, 10, null) == -2
    assert L.mdx_store_kvcache(null, null, 0, 0, null, null, null, 0, 1024, 2, 10, null) == 0   # empty: no-op
    sa = lambda **kw: L.mdx_staircase_attn_varlen(                                            # noqa: E731
        one, one, one, one, 2048, 128, 1024, 128, 1024, 128, 2048, 128, one, one, 1, 100, 100,
        kw.get("hq", 16), kw.get("hkv", 8), kw.get("d", 128), kw.get("S", 32), kw.get("scale", 0.1), kw.get("dtype", 0), null)
    assert sa(d=260) == -2 and b"head_dim" in L.mdx_last_error()    # up to 256 columns (above 128: the fp32-arithmetic kernel)
    assert sa(d=70) == -2 and b"head_dim" in L.mdx_last_error()     # multiples of 4 only
    assert sa(S=48) == -1 and b"staircase_size" in L.mdx_last_error()
    assert sa(hq=12) == -1
    assert sa(dtype=3) == -2 and b"dtype" in L.mdx_last_error()     # bf16, fp16 and fp32 are the element types
    assert sa(scale=-1.0) == -1
    st = lambda hkv, d: L.mdx_staircase_attn_store(                                              # noqa: E731
        one, one, one, one, 2048, 128, 1024, d, 1024, d, 2048, 128, one, one, 1, 100, 100, 16, hkv, d, 32, 0.1, 0, one, one, one, 10, null)
    assert st(0, 128) == -1 and st(8, 0) == -2                      # no KV heads, no columns: an error, not a division
    pa = lambda **kw: L.mdx_paged_block_attn(                                                  # noqa: E731
        one, one, one, one, 65536, 2048, 128, 65536, 2048, 128, 262144, 1024, 128, one, 17, one,
        4, kw.get("sq", 32), 16, 8, kw.get("d", 128), 17, kw.get("page", 256), 100, 0.1, 0, kw.get("ws", null), kw.get("ws_bytes", 0), null)
    assert pa(sq=129) == -2 and b"queries per sequence" in L.mdx_last_error()    # up to four tiles of 32 queries
    assert pa(page=100) == -2
    assert pa(d=260) == -2 and b"head_dim" in L.mdx_last_error()    # up to 256 columns (above 128: the fp32-arithmetic kernel)
    assert pa(d=42) == -2                                           # multiples of 4 only
    assert L.mdx_paged_block_attn_workspace_bytes(16, 32, 16, 8, 256, 17, 256) == 0     # that kernel never splits a sequence
    assert pa() == -3 and b"workspace" in L.mdx_last_error()
    assert L.mdx_select_transfer(one, one, one, 7, 0.9, -1, one, one, 2, 32, null) == -1      # k < 0
    assert L.mdx_select_transfer(one, one, one, 7, 0.9, 1, one, one, 2, 2000, null) == -2      # block too long
    assert L.mdx_confidence_argmax(one, 10, 0, null, 1, null, 0, one, one, 4, 20, null, 0, null) == -2   # stride < vocab
    fl = lambda **kw: L.mdx_filter_logits(one, kw.get("stride", 100), kw.get("dtype", 0), null, 1,           # noqa: E731
                                          kw.get("k", 5), kw.get("p", 0.9), one, 100, kw.get("rows", 4), 100, null)
    assert fl(dtype=2) == -2 and b"16-bit" in L.mdx_last_error()      # fp32 logits: the cut-off is found by counting 16-bit values
    assert fl(k=-1) == -1 and fl(p=-0.5) == -1 and fl(p=float("nan")) == -1
    assert fl(stride=50) == -2
    assert fl(rows=0) == 0
    # the single-launch paged call: with about a pair per CU (32 sequences x 8 head groups) it needs the counters
    big = ctypes.c_void_p(1 << 20)
    ws32 = L.mdx_paged_block_attn_workspace_bytes(32, 32, 16, 8, 128, 17, 256)
    sl = lambda counters, nbytes: L.mdx_paged_block_attn_single_launch(                          # noqa: E731
        one, one, one, one, 65536, 2048, 128, 65536, 2048, 128, 262144, 1024, 128, one, 17, one,
        32, 32, 16, 8, 128, 17, 256, 100, 0.1, 0, big, ws32, counters, nbytes, null)
    # one counter per (sequence, head group, query tile), sized for the longest block (four tiles of 32 queries)
    assert ws32 > 0 and L.mdx_paged_block_attn_counter_bytes(32, 16, 8) == 32 * 8 * 4 * 4
    assert sl(null, 0) == -3 and b"counters" in L.mdx_last_error()
    assert sl(one, 32 * 8 * 4 - 4) == -3
    assert sl(ctypes.c_void_p(18), 4096) == -3 and b"aligned" in L.mdx_last_error()


def test_fused_head_and_calibration_arguments_are_validated(L):
    null = None
    one = ctypes.c_void_p(16)
    ws = L.mdx_lm_head_confidence_workspace_bytes(1024, 151936)
    assert ws == 1024 * 1188 * 16 and L.mdx_lm_head_confidence_workspace_bytes(0, 151936) == 0     # one record per row and 128-entry slice
    big = ctypes.c_void_p(1 << 20)
    head = lambda **kw: L.mdx_lm_head_confidence(                                                   # noqa: E731
        kw.get("x", one), kw.get("xs", 2048), one, 2048, null, 1, null, one, one, kw.get("rows", 1024), 151936, kw.get("hidden", 2048),
        kw.get("ws", big), kw.get("ws_bytes", ws), null)
    assert head(x=null) == -1 and b"null" in L.mdx_last_error()
    assert head(hidden=2000) == -2 and b"hidden" in L.mdx_last_error()
    assert head(xs=2047) == -2
    assert head(ws_bytes=ws - 16) == -3 and b"workspace" in L.mdx_last_error()
    assert head(rows=0) == 0
    assert L.mdx_calib_mfma_loop(7, one, one, 4, 8, null) == -1
    assert L.mdx_calib_mfma_loop(32, null, one, 4, 8, null) == -1
    assert L.mdx_calib_mfma_loop_flops(32, 256, 8) == 256 * 4 * 8 * 8 * 32 * 32 * 16 * 2
    assert L.mdx_calib_mfma_loop_flops(16, 256, 3) == 256 * 4 * 8 * 16 * 16 * 16 * 32 * 2              # iterations rounded up to 8


def test_calls_that_join_two_steps_refuse_what_either_does(L):
    """mdx_staircase_attn_store and mdx_unmask_step_filtered."""
    null, one, big = None, ctypes.c_void_p(16), ctypes.c_void_p(1 << 20)
    st = lambda **kw: L.mdx_staircase_attn_store(                                                # noqa: E731
        kw.get("q", one), one, one, one, 2048, 128, kw.get("kst", 1024), kw.get("ksh", 128), 1024, kw.get("vsh", 128), 2048, 128, one, one, kw.get("batch", 1),
        kw.get("longest", 100), 100, kw.get("hq", 16), kw.get("hkv", 8), kw.get("d", 128), kw.get("S", 32), kw.get("scale", 0.1), kw.get("dtype", 0),
        kw.get("kc", one), one, kw.get("slots", one), kw.get("num_slots", 10), null)
    assert st(ksh=64) == -2 and b"dense" in L.mdx_last_error() and st(vsh=256) == -2
    assert st(q=null) == -1 and st(batch=-1) == -1 and st(longest=-1) == -1 and st(hq=12) == -1 and st(S=48) == -1 and st(scale=0.0) == -1
    assert st(dtype=7) == -2
    # the store's own refusals come before the attention's launch (which would end in a launch error here)
    assert st(kc=null) == -1 and st(slots=null) == -1 and st(num_slots=-1) == -1 and st(kst=-1024) == -2
    fs = lambda **kw: L.mdx_unmask_step_filtered(                                                # noqa: E731
        kw.get("logits", one), kw.get("stride", 1000), kw.get("dtype", 0), null, kw.get("top_k", 50), kw.get("top_p", 0.9), kw.get("noise", null),
        kw.get("noise_stride", 0), kw.get("seeded", 0), 1, 2, null, kw.get("tokens", one), 7, 0.9, kw.get("k", 1), kw.get("x0", one), one, one,
        kw.get("count", one), kw.get("bs", 4), kw.get("S", 32), kw.get("vocab", 1000), kw.get("ws", big), kw.get("ws_bytes", 1 << 30), null)
    for bad in ("logits", "tokens", "x0", "count"):
        assert fs(**{bad: null}) == -1 and b"null" in L.mdx_last_error()
    assert fs(noise=one, noise_stride=1000, seeded=1) == -1 and b"seed" in L.mdx_last_error()
    assert fs(noise=one, noise_stride=999) == -1
    assert fs(k=-1) == -1 and fs(bs=-1) == -1 and fs(S=1025) == -2 and fs(stride=999) == -2 and fs(dtype=2) == -2 and fs(vocab=0) == -1
    assert fs(top_k=-1) == -1 and fs(top_p=-0.1) == -1 and fs(top_p=float("nan")) == -1
    assert fs(bs=0) == 0 and fs(S=0) == 0
    for top_k in (50, 0):                                                                        # candidate lists; row cut-offs
        need = L.mdx_unmask_step_filtered_workspace_bytes(4 * 32, 1000, top_k)
        assert need > 0
        assert fs(top_k=top_k, ws=null) == -3 and fs(top_k=top_k, ws_bytes=need - 1) == -3 and b"workspace" in L.mdx_last_error()
        assert fs(top_k=top_k, ws=ctypes.c_void_p((1 << 20) + 8), ws_bytes=need) == -3
    assert L.mdx_unmask_step_filtered_workspace_bytes(0, 1000, 50) == 0 and L.mdx_unmask_step_filtered_workspace_bytes(4, 0, 50) == 0


def test_decode_linear_arguments_are_validated(L):
    """The products of few rows and the two calls that take their partial sums."""
    null, one, odd = None, ctypes.c_void_p(16), ctypes.c_void_p(24)
    assert L.mdx_decode_linear_splits(32, 2048, 2048) > 0 and 2048 // 256 % L.mdx_decode_linear_splits(32, 2048, 2048) == 0
    for rows, n, k in ((0, 64, 256), (129, 64, 256), (-1, 64, 256), (4, 72, 256), (4, 0, 256), (4, -64, 256), (4, 64, 320), (4, 64, 0), (4, 1 << 30, 256)):
        assert L.mdx_decode_linear_splits(rows, n, k) == 0
    for n, k in ((1 << 28, 256), (64, 1 << 28), (64, (1 << 30) - 256), ((1 << 30) - 64, 256)):
        assert L.mdx_decode_linear_splits(4, n, k) > 0 and k // 256 % L.mdx_decode_linear_splits(4, n, k) == 0
    pl = lambda **kw: L.mdx_decode_linear_partials(kw.get("x", one), kw.get("xs", 256), kw.get("w", one), kw.get("ws", 256), kw.get("p", one),    # noqa: E731
                                                   kw.get("rows", 4), 64, 256, null)
    sl = lambda **kw: L.mdx_decode_linear_silu(kw.get("x", one), kw.get("xs", 512), kw.get("w", one), kw.get("ws", 512), kw.get("y", one),        # noqa: E731
                                               kw.get("ys", 24), kw.get("rows", 4), kw.get("n", 24), 512, null)
    for call in (pl, sl):
        assert call(x=null) == -1 and call(w=null) == -1 and b"null" in L.mdx_last_error()
        assert call(x=odd) == -2 and call(w=odd) == -2 and call(xs=100) == -2 and call(ws=515) == -2 and call(xs=516) == -2
        assert call(rows=129) == -2
    assert pl(p=null) == -1 and pl(p=odd) == -2
    assert sl(y=null) == -1 and sl(y=odd) == -2 and sl(ys=20) == -2 and sl(ys=26) == -2 and sl(rows=65) == -2 and sl(n=32) == -2
    for rows, n, k in ((0, 24, 512), (65, 24, 512), (4, 16, 512), (4, 24, 256), (4, 0, 512), (4, 24, 0), (4, 3 << 28, 512), (4, 24, 1 << 30)):
        assert L.mdx_decode_linear_silu_supported(rows, n, k) == 0
    assert L.mdx_decode_linear_silu_supported(4, 3 << 27, 512) == 1 and L.mdx_decode_linear_silu_supported(4, 24, 1 << 28) == 1
    rn = lambda **kw: L.mdx_add_rms_norm_partials(kw.get("p", one), kw.get("splits", 2), kw.get("res", one), kw.get("rs", 64), kw.get("res_out", one), 64,  # noqa: E731
                                                  one, kw.get("eps", 1e-6), kw.get("out", one), 64, kw.get("rows", 4), kw.get("hidden", 64), kw.get("dtype", 0), null)
    assert rn(p=null) == -1 and rn(out=null) == -1 and rn(res=null) == -1 and rn(splits=0) == -1 and rn(rs=56) == -1 and rn(eps=-1.0) == -1
    assert rn(p=odd) == -2 and rn(hidden=60) == -2 and rn(dtype=2) == -2 and rn(rows=0) == 0
    qk = lambda **kw: L.mdx_qk_norm_rope_store_partials(kw.get("p", one), kw.get("splits", 2), one, one, 1e-6, one, one, 64, kw.get("pos", one), one, 256,  # noqa: E731
                                                        kw.get("kc", one), one, kw.get("slots", one), 10, kw.get("n", 4), kw.get("hq", 2), kw.get("hkv", 1),
                                                        kw.get("d", 128), kw.get("dtype", 0), null)
    assert qk(p=null) == -1 and qk(pos=null) == -1 and qk(kc=null) == -1 and qk(slots=null) == -1 and qk(splits=0) == -1 and qk(hq=0) == -1 and qk(hkv=0) == -1
    assert qk(p=odd) == -2 and qk(d=64) == -2 and qk(dtype=1) == -2 and qk(n=0) == 0


def test_ops_fail_loudly_off_gpu():
    import torch
    import mdx
    x = torch.zeros(4, 8, 128, dtype=torch.bfloat16)
    with pytest.raises(mdx.MdxError):
        mdx.store_kvcache(x, x, torch.zeros(1, 256, 8, 128, dtype=torch.bfloat16),
                          torch.zeros(1, 256, 8, 128, dtype=torch.bfloat16), torch.zeros(4, dtype=torch.int32))
    with pytest.raises(mdx.MdxError):
        mdx.sparse_attn_varlen(x, x, x, torch.tensor([0, 4], dtype=torch.int32), torch.tensor([0, 4], dtype=torch.int32), 32)


def test_context_mirror():
    import mdx
    mdx.set_context(True, max_seqlen_q=5, block_size=32)
    assert mdx.get_context().is_prefill and mdx.get_context().max_seqlen_q == 5
    mdx.reset_context()
    assert not mdx.get_context().is_prefill and mdx.get_context().slot_mapping is None


def test_generated_kernel_core_is_current():
    """staircase_pair_core.inc, its fp16 twin and lm_head_core.inc are the committed outputs of their generators: regenerate and compare."""
    import subprocess
    import sys
    from pathlib import Path
    csrc = Path(__file__).resolve().parents[1] / "mineru-diffusion_amd" / "csrc"
    out = subprocess.run([sys.executable, str(csrc / "gen_staircase_pair_core.py")], capture_output=True, text=True, check=True)
    assert out.stdout == (csrc / "staircase_pair_core.inc").read_text()
    out = subprocess.run([sys.executable, str(csrc / "gen_staircase_pair_core.py"), "f16"], capture_output=True, text=True, check=True)
    assert out.stdout == (csrc / "staircase_pair_core_f16.inc").read_text()
    # the core of the fused vocabulary projection
    out = subprocess.run([sys.executable, str(csrc / "gen_lm_head_core.py")], capture_output=True, text=True, check=True)
    assert out.stdout == (csrc / "lm_head_core.inc").read_text()


def test_read_ahead_arguments_are_validated(L):
    """What an attention launch is asked to read ahead: whole 16-byte pieces that exist; all other arguments as in the plain call."""
    one, null = ctypes.c_void_p(256), ctypes.c_void_p(0)
    ra = lambda **kw: L.mdx_paged_block_attn_read_ahead(                                       # noqa: E731
        one, one, one, one, 65536, 2048, 128, 65536, 2048, 128, 262144, 1024, 128, one, 17, one,
        kw.get("bs", 4), kw.get("sq", 32), 16, 8, 128, 17, 256, 100, 0.1, 0, null, 0, kw.get("counters", null), 0,
        kw.get("a", one), kw.get("na", 256), kw.get("b", one), kw.get("nb", 256), null)
    assert ra(na=-16) == -1 and ra(nb=8) == -1 and ra(a=null) == -1 and ra(b=ctypes.c_void_p(264)) == -1 and b"16 bytes" in L.mdx_last_error()
    assert ra(bs=-1) == -1 and ra(sq=129) == -2 and ra(bs=0) == 0
    assert ra() == -3 and ra(a=null, na=0, b=null, nb=0) == -3 and b"workspace" in L.mdx_last_error()


def test_linear_arguments_are_validated(L):
    null, one, odd = None, ctypes.c_void_p(16), ctypes.c_void_p(24)
    for rows, n, k in ((0, 64, 256), (-1, 64, 256), (1537, 64, 256), (4, 68, 256), (4, 0, 256), (4, -64, 256), (4, 64, 320), (4, 64, 128), (4, 1 << 28, 256)):
        assert L.mdx_linear_splits(rows, n, k) == -1
    assert L.mdx_linear_splits(32, 2048, 6144) > 1 and L.mdx_linear_splits(1024, 4096, 2048) == 0
    # wide layers: beyond 52 GFLOP only those whose K is long beside n
    assert L.mdx_linear_splits(512, 7168, 5120) >= 0 and L.mdx_linear_splits(1280, 7168, 5120) == -1 and L.mdx_linear_splits(1024, 8192, 8192) == -1
    assert L.mdx_linear_splits(1536, 2048, 6144) >= 0 and L.mdx_linear_splits(1024, 5120, 17408) >= 0
    assert L.mdx_linear_silu_supported(8192, 64, 256) == 1 and L.mdx_linear_silu_supported(8193, 64, 256) == 0 and L.mdx_linear_silu_supported(4, 60, 256) == 0
    li = lambda f: lambda **kw: f(kw.get("x", one), kw.get("xs", 256), kw.get("w", one), kw.get("ws", 256), kw.get("y", one), kw.get("ys", 64),    # noqa: E731
                                  kw.get("rows", 4), kw.get("n", 64), kw.get("k", 256), null)
    for call in (li(L.mdx_linear), li(L.mdx_linear_silu)):
        assert call(x=null) == -1 and call(w=null) == -1 and call(y=null) == -1 and b"null" in L.mdx_last_error()
        assert call(x=odd) == -2 and call(w=odd) == -2 and call(y=odd) == -2 and call(xs=100) == -2 and call(ws=264 - 1) == -2 and call(xs=248) == -2
        assert call(xs=1 << 28) == -2 and call(ys=60) == -2 and call(ys=66) == -2 and call(rows=0) == -2 and call(n=68) == -2 and call(k=192) == -2
    pl = lambda **kw: L.mdx_linear_partials(kw.get("x", one), 6144, one, 6144, kw.get("p", one), kw.get("rows", 32), 2048, 6144, null)             # noqa: E731
    assert pl(x=null) == -1 and pl(p=null) == -1 and pl(p=odd) == -2 and pl(rows=1537) == -2

    hd = lambda **kw: L.mdx_linear_qk_norm_rope_store(kw.get("x", one), kw.get("xs", 256), one, 256, kw.get("qw", one), one, 1e-6, one, one, 8, kw.get("pos", one),   # noqa: E731
                                                      kw.get("q", one), kw.get("qs", 256), null, 0, null, 0, kw.get("kc", null), kw.get("vc", null), kw.get("slots", null), 0,
                                                      kw.get("rows", 400), 2, 1, kw.get("d", 128), 256, null)
    # one launch where its tiles of a head cost no more than the product's own and a second launch: the model's heads at all rows, others by their rounds
    hs = L.mdx_linear_qk_norm_rope_store_supported
    assert all(hs(rows, 16, 8, 128, 2048) == 1 for rows in range(384, 1537)) and hs(383, 16, 8, 128, 2048) == 0 and hs(1537, 16, 8, 128, 2048) == 0
    assert hs(512, 64, 8, 128, 8192) == 1 and hs(1536, 64, 8, 128, 8192) == 0 and hs(768, 32, 8, 128, 2560) == 1 and hs(1024, 32, 8, 128, 2560) == 0
    assert hs(384, 16, 2, 128, 2048) == 0 and hs(512, 16, 2, 128, 2048) == 1
    assert hd(x=null) == -1 and hd(qw=null) == -1 and hd(pos=null) == -1 and hd(q=null) == -1 and hd(kc=one) == -1 and hd(kc=one, vc=one) == -1
    assert hd(rows=383) == -2 and hd(rows=1537) == -2 and hd(d=64) == -2 and hd(q=odd) == -2 and hd(qs=260) == -2 and hd(qw=odd) == -2 and hd(xs=248) == -2
