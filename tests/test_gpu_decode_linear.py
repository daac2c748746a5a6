"""The linear layers of a decode pass (partial sums, SiLU form) and the two kernels that add partial sums up, against fp32
products on the host of the same bf16 values."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _xw(dev, rows, n, k, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * 0.05).bfloat16()
    return x, w, x.to(dev), w.to(dev)


@pytest.mark.parametrize("rows", [1, 15, 32, 33, 64, 65, 100, 128])
@pytest.mark.parametrize("n,k", [(64, 256), (192, 768), (2048, 512), (2112, 6144), (16448, 256)])
def test_linear_partials(dev, rows, n, k):
    """Edges of the row tiles, one and several slices of K, one and several steps of a slice, more tiles than CUs."""
    from mdx import ops
    x, w, dx, dw = _xw(dev, rows, n, k, rows + n)
    p = ops.linear_partials(dx, dw)
    assert p.dtype == torch.float32 and p.shape[1:] == (rows, n)
    ref = x.float() @ w.float().T
    assert (p.sum(0).cpu() - ref).norm() < 2e-6 * ref.norm() + 1e-6
    padded = torch.zeros(rows, k + 8, dtype=torch.bfloat16, device=dev)              # rows of x that are not contiguous
    padded[:, :k] = dx
    assert torch.equal(ops.linear_partials(padded[:, :k], dw), p)


def test_linear_partials_and_silu_say_what_they_do_not_cover(dev):
    from mdx import ops
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device=dev)                 # noqa: E731
    assert ops.linear_partials(z(129, 256), z(64, 256)) is None and ops.linear_partials(z(4, 256), z(72, 256)) is None
    assert ops.linear_partials(z(4, 320), z(64, 320)) is None and ops.linear_partials(z(4, 256).float(), z(64, 256).float()) is None
    assert ops.linear_silu(z(65, 512), z(48, 512)) is None and ops.linear_silu(z(4, 256), z(48, 256)) is None


@pytest.mark.parametrize("x_at,x_pad,w_at,w_pad", [(1, 0, 0, 0), (0, 3, 0, 0), (0, 0, 1, 0), (0, 0, 0, 4), (0, -256, 0, 0)])
def test_linear_leaves_rows_that_are_not_aligned_to_the_library(dev, x_at, x_pad, w_at, w_pad):
    """A view off a 16-byte boundary, rows whose stride is no multiple of 8 elements, and rows that overlap: None, not an error."""
    from mdx import ops
    k = 512
    rows = lambda n, at, pad: torch.zeros(n * (k + 8) + 8, dtype=torch.bfloat16, device=dev).as_strided((n, k), (k + pad, 1), at)    # noqa: E731
    assert ops.linear_partials(rows(4, x_at, x_pad), rows(64, w_at, w_pad)) is None
    assert ops.linear_silu(rows(4, x_at, x_pad), rows(48, w_at, w_pad)) is None
    assert ops.linear_partials(rows(4, 8, 8), rows(64, 8, 8)) is not None and ops.linear_silu(rows(4, 8, 8), rows(48, 8, 8)) is not None


@pytest.mark.parametrize("rows", [1, 16, 31, 32, 33, 64])
@pytest.mark.parametrize("inter,k", [(24, 512), (72, 1536), (6144, 2048)])
def test_linear_silu(dev, rows, inter, k):
    import mdx
    from mdx import ops
    x, w, dx, dw = _xw(dev, rows, 2 * inter, k, rows + inter)
    y = ops.linear_silu(dx, dw)
    ref = mdx.silu_and_mul((x.float() @ w.float().T).bfloat16().to(dev))
    assert y.shape == ref.shape and (y.float() - ref.float()).norm() < 3e-3 * ref.float().norm()


@pytest.mark.parametrize("splits", [1, 3, 4, 8, 11])
def test_partials_are_taken_in_like_the_sum(dev, splits):
    """rms_norm and qk_norm_rope_store on partial sums against the same calls on their bf16 sum."""
    import mdx
    from mdx import ops
    g = torch.Generator().manual_seed(splits)
    rows, hq, hkv, d = 40, 4, 2, 128
    for hidden in (2048, 2056):
        p = torch.randn(splits, rows, hidden, generator=g).to(dev)
        total = p[0].clone()
        for s in range(1, splits):
            total += p[s]
        w, res = torch.randn(hidden, generator=g).bfloat16().to(dev), torch.randn(rows, hidden, generator=g).bfloat16().to(dev)
        for a, b in zip(ops.rms_norm_partials(p, w, 1e-6, res), mdx.rms_norm(total.bfloat16(), w, 1e-6, res)):
            assert (a.float() - b.float()).norm() < 2e-3 * b.float().norm()          # the orders of summation may round apart
    width = (hq + 2 * hkv) * d
    p = torch.randn(splits, rows, width, generator=g).to(dev)
    qw, kw = torch.randn(d, generator=g).bfloat16().to(dev), torch.randn(d, generator=g).bfloat16().to(dev)
    cos, sin = torch.rand(64, d // 2, generator=g).to(dev), torch.rand(64, d // 2, generator=g).to(dev)
    pos, slots = torch.arange(rows, device=dev), torch.randperm(64, generator=g)[:rows].int().to(dev)
    caches = [torch.zeros(1, 64, hkv, d, dtype=torch.bfloat16, device=dev) for _ in range(4)]
    q = ops.qk_norm_rope_store_partials(p, qw, kw, 1e-6, cos, sin, pos, hq, hkv, d, caches[0], caches[1], slots)
    q2, _, _ = mdx.qk_norm_rope_store(p.sum(0).bfloat16(), qw, kw, 1e-6, cos, sin, pos, hq, hkv, d, caches[2], caches[3], slots)
    for a, b in ((q, q2), (caches[0], caches[2]), (caches[1], caches[3])):
        assert (a.float() - b.float()).norm() < 3e-3 * b.float().norm()
