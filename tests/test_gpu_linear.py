"""The linear layers (rounded, as partial sums, with the SiLU-and-multiply) against fp32 products on the host of the same bf16
values: sizes that take each tile of the plan in each form, with ragged last rows and columns, the fewest steps of K and many,
one slice of K and several."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 8, 256), (31, 72, 384), (64, 136, 2048), (129, 520, 768), (520, 2056, 384), (333, 2048, 6144), (600, 4104, 512), (130, 16392, 256),
         (1000, 4104, 512), (1120, 4104, 512), (1100, 2056, 3072), (260, 16648, 256), (1030, 12304, 256)]


def _xw(dev, rows, n, k):
    g = torch.Generator().manual_seed(rows + n + k)
    x, w = torch.randn(rows, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) * 0.05).bfloat16()
    return x.float() @ w.float().T, x.to(dev), w.to(dev)


def _close(got, ref, rel):
    return (got.float().cpu() - ref).norm() < rel * ref.norm()


@pytest.mark.parametrize("rows,n,k", SIZES)
def test_linear(dev, rows, n, k):
    """fp32 sums in another order: 2e-6 of the norm for up to 6144 terms; rounding to bf16 (8 bits) adds at most 2^-8 of each value."""
    from mdx import ops
    ref, x, w = _xw(dev, rows, n, k)
    y = ops.linear(x, w)
    assert y.dtype == torch.bfloat16 and y.shape == ref.shape and _close(y, ref, 2.0 ** -8)
    either = ops.linear(x, w, True)
    assert torch.equal(either, y) if either.dim() == 2 else _close(either.sum(0), ref, 2e-6)
    padded = torch.zeros(rows, k + 8, dtype=torch.bfloat16, device=dev)                  # rows that are not contiguous
    padded[:, :k] = x
    assert torch.equal(ops.linear(padded[:, :k], w), y)


@pytest.mark.parametrize("rows,n,k", SIZES)
def test_linear_gated(dev, rows, n, k):
    import mdx
    from mdx import ops
    ref, x, w = _xw(dev, rows, 2 * n, k)
    y = ops.linear_gated(x, w)
    # the same roundings on both sides; a gate or up value on a rounding boundary may fall either way: 2^-7 of it, for few of them
    want = mdx.silu_and_mul(ref.bfloat16().to(dev)).float().cpu()
    assert y.shape == want.shape and _close(y, want, 3e-3)


def test_linear_says_what_it_does_not_cover(dev):
    from mdx import ops
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)                     # noqa: E731
    for x, w in ((z(1537, 256), z(64, 256)), (z(4, 256), z(68, 256)), (z(4, 128), z(64, 128)), (z(4, 320), z(64, 320)), (z(4, 256).float(), z(64, 256).float()),
                 (z(0, 256), z(64, 256)), (z(5, 257)[:, 1:], z(64, 256))):
        assert ops.linear(x, w) is None and ops.linear(x, w, True) is None
    assert ops.linear_gated(z(8193, 256), z(64, 256)) is None and ops.linear_gated(z(4, 256), z(72, 256)) is None
    assert ops.linear(z(2, 3, 256), z(64, 256)).shape == (2, 3, 64) and ops.linear_gated(z(2, 3, 256), z(64, 256)).shape == (2, 3, 32)


@pytest.mark.parametrize("rows,n,k", [(40, 72, 384), (333, 2056, 512), (1100, 4104, 256)])
def test_rows_of_w_in_a_wider_matrix(dev, rows, n, k):
    """W with rows further apart than k, rounded, as partial sums, with the SiLU (whose second half of W begins n such rows on) and with the
    head rows: the results for dense rows, bit for bit."""
    from mdx import ops
    _, x, w = _xw(dev, rows, 2 * n, k)
    wide = torch.full((2 * n, k + 24), float("nan"), dtype=torch.bfloat16, device=dev)
    wide[:, :k] = w
    w2 = wide[:, :k]
    for partials in (False, True):
        assert torch.equal(ops.linear(x, w2[:n], partials), ops.linear(x, w[:n], partials))
    assert torch.equal(ops.linear_gated(x, w2), ops.linear_gated(x, w))
    if rows >= 384:
        one, pos = torch.ones(128, dtype=torch.bfloat16, device=dev), torch.arange(rows, device=dev)
        table = torch.rand(rows, 64, device=dev)
        heads = lambda w: ops.linear_qk_norm_rope_store(x, w[:4096], one, one, 1e-6, table, table, pos, 16, 8, 128)      # noqa: E731
        assert all(torch.equal(a, b) for a, b in zip(heads(w2), heads(w)))


@pytest.mark.parametrize("rows,n,k", [(1537, 520, 256), (3000, 2056, 384), (9000, 1032, 256)])
def test_rows_beyond_what_the_dispatch_takes(dev, rows, n, k):
    """The C entries take more rows than pay, and results in wider matrices, whose other columns stay as they are."""
    import mdx
    ref, x, w = _xw(dev, rows, 2 * n, k)
    L, stream = mdx._lib.lib(), torch.cuda.current_stream().cuda_stream
    for call, want, rel in ((L.mdx_linear, ref[:, :n], 2.0 ** -8), (L.mdx_linear_silu, mdx.silu_and_mul(ref.bfloat16().to(dev)).float().cpu(), 3e-3)):
        y = torch.full((rows, n + 12), 7.0, dtype=torch.bfloat16, device=dev)
        assert call(x.data_ptr(), k, w.data_ptr(), k, y.data_ptr(), n + 12, rows, n, k, stream) == 0
        torch.cuda.synchronize()
        assert _close(y[:, :n], want, rel) and bool((y[:, n:] == 7.0).all())


@pytest.mark.parametrize("rows,n,k", [(20, 72, 384), (130, 136, 2048), (520, 4104, 384), (1100, 4104, 256)])
def test_values_that_are_not_finite(dev, rows, n, k):
    """NaN and infinities in a row of x or of W reach that row's or column's results and no others, in every form."""
    import mdx
    from mdx import ops
    inf, nan = float("inf"), float("nan")
    _, x, w = _xw(dev, rows, 2 * n, k)
    x[3, 5], x[rows - 1, k - 1], x[4, 7] = nan, inf, -inf
    w[6, 9], w[n - 1, 0], w[n + 8, 3] = inf, nan, nan
    ref = x.float().cpu() @ w.float().cpu().T

    def same(got, want, rel):
        got, plain = got.float().cpu(), want.isfinite()
        return torch.equal(got.isnan(), want.isnan()) and torch.equal(got[~plain & ~want.isnan()], want[~plain & ~want.isnan()]) and _close(got[plain], want[plain], rel)

    first = ref[:, :n].contiguous()
    assert same(ops.linear(x, w[:n]), first.bfloat16().float(), 2.0 ** -8)
    either = ops.linear(x, w[:n], True)
    assert either.dim() == 2 or same(either.sum(0), first, 2e-6)
    assert same(ops.linear_gated(x, w), mdx.silu_and_mul(ref.bfloat16().to(dev)).float().cpu(), 3e-3)


def test_rows_far_apart(dev):
    """Rows 2^28 elements and more apart: computed by the two calls for few rows, left to the library by the others."""
    import mdx
    from mdx import ops
    far = (1 << 28) + 8
    buffer = torch.empty(63 * far + 2048, dtype=torch.bfloat16, device=dev)               # 32 GB, of which the rows below are written

    def apart(t, offset):
        view = buffer.as_strided(t.shape, (far, 1), offset)
        view.copy_(t)
        return view

    for rows, n, k in ((3, 64, 256), (33, 64, 768), (64, 64, 512)):
        ref, x, w = _xw(dev, rows, n, k)
        for a, b in ((apart(x, 0), w), (x, apart(w, 1024)), (apart(x, 0), apart(w, 1024))):
            p = ops.linear_partials(a, b)
            assert p.shape == (mdx._lib.lib().mdx_decode_linear_splits(rows, n, k), rows, n) and _close(p.sum(0), ref, 2e-6)
            assert ops.linear(a, b) is None and ops.linear(a, b, True) is None and ops.linear_gated(a, b) is None
    for rows, n in ((3, 24), (40, 24)):
        ref, x, w = _xw(dev, rows, 2 * n, 512)
        want = mdx.silu_and_mul(ref.bfloat16().to(dev)).float().cpu()
        for a, b in ((apart(x, 0), w), (x, apart(w, 1024)), (apart(x, 0), apart(w, 1024))):
            y = ops.linear_silu(a, b)
            assert y.shape == want.shape and _close(y, want, 3e-3)
    del buffer
    torch.cuda.empty_cache()


@pytest.mark.parametrize("rows,hq,hkv,k", [(384, 16, 8, 384), (385, 2, 1, 256), (513, 4, 2, 512), (1000, 16, 8, 256), (1100, 16, 8, 256), (1536, 6, 3, 256)])
@pytest.mark.parametrize("caches", [True, False])
def test_linear_qk_norm_rope_store(dev, rows, hq, hkv, k, caches):
    """Each of the tiles with head rows finished in the epilogue against qk_norm_rope_store on the rounded product: last row tiles of
    few rows, positions beyond the table, slots that are skipped or out of range, with and without caches and k / v."""
    import mdx
    from mdx import ops
    d, n = 128, (hq + 2 * hkv) * 128
    _, x, w = _xw(dev, rows, n, k)
    g = torch.Generator().manual_seed(rows)
    qw, kw = torch.randn(d, generator=g).bfloat16().to(dev), torch.randn(d, generator=g).bfloat16().to(dev)
    cos, sin = torch.rand(2000, d // 2, generator=g).to(dev), torch.rand(2000, d // 2, generator=g).to(dev)
    pos = torch.randint(0, 2000, (rows,), generator=g)
    pos[::17], pos[5] = 2000, -1
    slots = torch.randperm(2048, generator=g)[:rows].int()
    slots[::7], slots[3] = -1, 4096
    pos, slots = pos.to(dev), slots.to(dev)
    store = lambda: (torch.zeros(8, 256, hkv, d, dtype=torch.bfloat16, device=dev), torch.zeros(8, 256, hkv, d, dtype=torch.bfloat16, device=dev), slots)   # noqa: E731
    one, two = store(), store()
    q, kk, v = ops.linear_qk_norm_rope_store(x, w, qw, kw, 1e-6, cos, sin, pos, hq, hkv, d, *(one if caches else (None,) * 3), want_kv=True)
    q2, k2, v2 = mdx.qk_norm_rope_store(ops.linear(x, w), qw, kw, 1e-6, cos, sin, pos, hq, hkv, d, *(two if caches else (None,) * 3))
    pairs = [(q, q2), (kk, k2), (v, v2)] + list(zip(one[:2], two[:2])) * caches
    for a, b in pairs:                        # the same roundings; the two products' orders of summation may round apart
        assert a.shape == b.shape and (a.float() - b.float()).norm() < 3e-3 * b.float().norm()
    if caches:
        assert all(torch.equal(a == 0, b == 0) for a, b in zip(one[:2], two[:2]))
    q3, none, nothing = ops.linear_qk_norm_rope_store(x, w, qw, kw, 1e-6, cos, sin, pos, hq, hkv, d, *(one if caches else (None,) * 3), want_kv=False)
    assert none is None and nothing is None and torch.equal(q3, q)


def test_linear_qk_norm_rope_store_says_what_it_does_not_cover(dev):
    from mdx import ops
    z = lambda *s, dtype=torch.bfloat16: torch.zeros(*s, dtype=dtype, device=dev)                # noqa: E731
    call = lambda x, w, hq, hkv, d: ops.linear_qk_norm_rope_store(x, w, z(d), z(d), 1e-6, z(8, d // 2, dtype=torch.float32), z(8, d // 2, dtype=torch.float32),   # noqa: E731
                                                                  z(x.shape[0], dtype=torch.int64), hq, hkv, d)
    assert call(z(383, 256), z(512, 256), 2, 1, 128) is None and call(z(1537, 256), z(512, 256), 2, 1, 128) is None
    assert call(z(400, 256), z(256, 256), 2, 1, 64) is None and call(z(400, 320), z(512, 320), 2, 1, 128) is None
    assert call(z(400, 264)[:, 1:257], z(512, 256), 2, 1, 128) is None and call(z(400, 256), z(512, 256), 2, 1, 128) is not None


@pytest.mark.parametrize("rows", [1, 16, 32, 33, 64, 65])
def test_layer_of_few_rows_rounds_where_the_reference_does(dev, rows):
    """Behind the attention a decoder layer rounds the normed sum, and again behind the norm's weight (layernorm.py:28-41), however few rows there are.  Small
    integers and rows of an identity matrix as weights: every product is exact in any order, so that what comes out is the oracle's but for a reciprocal
    root or a SiLU on a rounding boundary (below 3 % of the values, one step; with one rounding for both, nearly half of them differ)."""
    import oracle
    from mdx.engine import DecoderConfig, DecoderLayer
    h = 512
    c = DecoderConfig(hidden_size=h, num_heads=4, num_kv_heads=2, intermediate_size=h)
    layer = DecoderLayer(c).to(dev, torch.bfloat16)
    g = torch.Generator().manual_seed(rows)
    o, w = (torch.randint(-2, 3, s, generator=g).bfloat16() for s in ((rows, h), (h, h)))
    x, nw = (torch.randn(rows, h, generator=g) * 9).bfloat16(), (1 + 0.3 * torch.randn(h, generator=g)).bfloat16()
    eye = torch.eye(h).bfloat16()
    with torch.no_grad():
        layer.o_proj.copy_(w)
        layer.gate_up_proj.copy_(torch.cat((eye, eye.roll(7, 0))))
        layer.down_proj.copy_(eye)
        layer.post_attention_layernorm.copy_(nw)
        layer._attend_fused = lambda *_: o.to(dev)
        y, residual = layer(None, x.to(dev), None, None, None)
    y = (y.sum(0) if y.dim() == 3 else y).bfloat16().cpu()
    normed, s = oracle.add_rms_norm((o.float() @ w.float().T).bfloat16(), x, nw, c.rms_norm_eps)
    want = oracle.silu_and_mul(torch.cat((normed, normed.roll(7, 1)), 1))
    assert torch.equal(residual.cpu(), s)
    assert (y == want).float().mean() > 0.97
    assert (y.float() - want.float()).norm() < 2.0 ** -9 * want.float().norm()
