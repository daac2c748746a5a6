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
