"""The tiles of the linear layers and the vocabulary head at the fewest steps of K and at their edges in rows and columns, on small integers: sums are
exact in any order, so results are those of an fp32 product rounded once, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _integers(rows, n, k):
    g = torch.Generator().manual_seed(rows * 7 + n + k)
    return (torch.randint(-2, 3, (rows, k), generator=g).bfloat16(), torch.randint(-2, 3, (n, k), generator=g).bfloat16())


@pytest.mark.parametrize("k", [256, 384, 640, 6144])
@pytest.mark.parametrize("rows,n", [(33, 72), (129, 264), (192, 2056), (257, 4104), (577, 2056), (1025, 4104), (1120, 6152), (1536, 8200), (2049, 6152), (4100, 6152), (1000, 2048), (1280, 2048)])
def test_products_at_few_steps(dev, rows, n, k):
    import mdx
    x, w = _integers(rows, n, k)
    want = (x.to(dev).float() @ w.to(dev).float().T).bfloat16()
    L, stream = mdx._lib.lib(), torch.cuda.current_stream().cuda_stream
    x, w = x.to(dev), w.to(dev)
    y = torch.full((rows, n + 4), 7.0, dtype=torch.bfloat16, device=dev)
    assert L.mdx_linear(x.data_ptr(), k, w.data_ptr(), k, y.data_ptr(), n + 4, rows, n, k, stream) == 0
    assert torch.equal(y[:, :n], want) and bool((y[:, n:] == 7.0).all())
    half = n // 2 // 8 * 8
    act = torch.full((rows, half + 4), 7.0, dtype=torch.bfloat16, device=dev)
    assert L.mdx_linear_silu(x.data_ptr(), k, w.data_ptr(), k, act.data_ptr(), half + 4, rows, half, k, stream) == 0
    # the gates are whole numbers, of which both kernels make the same bf16 (test_silu_of_every_gate), and the product with the other half is rounded once
    assert torch.equal(act[:, :half], mdx.silu_and_mul(want[:, :2 * half].contiguous())) and bool((act[:, half:] == 7.0).all())
    splits = L.mdx_linear_splits(rows, n, k)
    if splits > 0:
        parts = torch.full((splits, rows, n), 7.0, device=dev)
        assert L.mdx_linear_partials(x.data_ptr(), k, w.data_ptr(), k, parts.data_ptr(), rows, n, k, stream) == 0
        assert torch.equal(parts.sum(0).bfloat16(), want)


# slices of four and five steps, six and more: both depths of the two smallest tiles, at their edges in rows
@pytest.mark.parametrize("rows,n,k", [(1, 64, 256), (32, 72, 256), (33, 1024, 256), (64, 520, 256), (128, 512, 512), (17, 1024, 640), (32, 2048, 2048), (64, 1032, 1024), (65, 512, 1280),
                                      (160, 512, 384), (48, 1024, 3072)])
def test_products_of_the_small_tiles(dev, rows, n, k):
    test_products_at_few_steps(dev, rows, n, k)


@pytest.mark.parametrize("rows,n,k,taken", [(8193, 1024, 512, True), (8400, 2056, 640, True), (8193, 1016, 512, False), (8193, 1024, 1152, False)])
def test_gated_product_of_many_rows(dev, rows, n, k, taken):
    """Beyond 8192 rows the gated product is taken where W's halves are no narrower than 1024 and K: the two steps' result."""
    import mdx
    x, w = _integers(rows, 2 * n, k)
    x, w = x.to(dev), w.to(dev)
    y = mdx.ops.linear_gated(x, w)
    assert (y is not None) == taken
    if taken:
        assert torch.equal(y, mdx.silu_and_mul((x.float() @ w.float().T).bfloat16()))


def test_silu_of_every_gate(dev):
    """Every bf16 value, times powers of two, as the gate of the product's own SiLU and of the kernel that divides: the same bits."""
    import mdx
    k, n = 256, 16
    gates = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = torch.zeros(65536, k, dtype=torch.bfloat16)
    x[:, 0], x[:, 1] = gates, 1.0
    w = torch.zeros(2 * n, k, dtype=torch.bfloat16)
    w[:n, 0] = 2.0 ** (torch.arange(n) - 8.0)
    w[n:, 1] = 1.0 + torch.arange(n) / 16
    x, w = x.to(dev), w.to(dev)
    L, stream = mdx._lib.lib(), torch.cuda.current_stream().cuda_stream
    product = torch.empty(65536, 2 * n, dtype=torch.bfloat16, device=dev)
    y = torch.empty(65536, n, dtype=torch.bfloat16, device=dev)
    assert L.mdx_linear(x.data_ptr(), k, w.data_ptr(), k, product.data_ptr(), 2 * n, 65536, 2 * n, k, stream) == 0
    assert L.mdx_linear_silu(x.data_ptr(), k, w.data_ptr(), k, y.data_ptr(), n, 65536, n, k, stream) == 0
    want = mdx.silu_and_mul(product)
    assert torch.equal(y.isnan(), want.isnan())
    assert torch.equal(y.nan_to_num(nan=7.0).view(torch.int16), want.nan_to_num(nan=7.0).view(torch.int16))


@pytest.mark.parametrize("rows,vocab,hidden", [(1, 100, 2048), (17, 1000, 1024), (33, 70001, 256), (64, 129, 512), (65, 70001, 256), (100, 40001, 1024), (128, 257, 384), (32, 40001, 2048), (31, 70001, 1024), (20, 33000, 2048), (129, 511, 256), (192, 30000, 256), (193, 30001, 384), (256, 70000, 256), (384, 40003, 256), (385, 769, 512), (512, 70001, 256)])
def test_head_at_few_steps(dev, rows, vocab, hidden):
    import mdx
    x, w = _integers(rows, vocab, hidden)
    x, w = x.to(dev), w.to(dev)
    x0, p = mdx.lm_head_confidence(x, w)
    logits = (x.float() @ w.float().T).bfloat16()
    tx0, tp = mdx.confidence_argmax(logits.unsqueeze(0))
    assert torch.equal(x0, tx0.view(-1))
    # two sums of the same fp32 terms: 2^-24 per addition and of each exponent's argument
    assert torch.allclose(p, tp.view(-1), rtol=3e-5, atol=0)


# up to 32 rows and rows of 512 and 1024 columns that the workgroups stream past x: from five tiles of 128 entries per CU on (131 072 entries and more), an odd number of
# tiles in a workgroup's turn, a last tile of one entry; and both sides of that line, of 32 rows and of the widths
@pytest.mark.parametrize("rows,vocab,hidden", [(1, 131073, 512), (17, 151936, 512), (32, 163841, 512), (16, 131073, 1024), (32, 151936, 1024), (31, 200001, 1024),
                                               (32, 131072, 512), (33, 131073, 512), (5, 131073, 1536), (32, 300, 2048), (9, 131073, 2048)])
def test_head_of_few_rows_at_other_widths(dev, rows, vocab, hidden):
    import mdx
    x, w = _integers(rows, vocab, hidden)
    w[vocab // 2] = w[vocab - 1] = w[3]                    # equal rows: equal logits wherever they stand
    x[0] = w[3]                                            # and of row 0 the largest: the first of them is taken
    x, w = x.to(dev), w.to(dev)
    x0, p = mdx.lm_head_confidence(x, w)
    logits = (x.float() @ w.float().T).bfloat16()
    tx0, tp = mdx.confidence_argmax(logits.unsqueeze(0))
    assert int(x0[0]) == 3 and torch.equal(x0, tx0.view(-1))
    assert torch.allclose(p, tp.view(-1), rtol=3e-5, atol=0)


# the tiles of 65 to 128 rows: two steps in LDS (a round of tiles of 128 entries and one more, widths of two whole steps of the pipeline and up to the limit), twice as wide
# where that halves the rounds, four steps otherwise; one and two row tiles of the others
@pytest.mark.parametrize("rows,vocab,hidden", [(65, 70001, 256), (128, 70001, 384), (100, 131073, 1152), (128, 131073, 1280), (65, 32769, 256), (128, 50001, 512), (77, 65536, 2048),
                                               (100, 32768, 256), (128, 511, 1024)])
def test_head_tiles_of_up_to_128_rows(dev, rows, vocab, hidden):
    test_head_at_few_steps(dev, rows, vocab, hidden)


# vocabularies that tiles of 256 entries leave CUs empty with: 128 x 256 and 192 x 192, at their edges in rows, and both sides of a full round
@pytest.mark.parametrize("rows,vocab,hidden", [(129, 32000, 256), (192, 32000, 2048), (256, 16001, 384), (300, 16000, 512), (150, 48000, 256), (192, 48129, 1024), (250, 65536, 256),
                                               (193, 257, 640), (500, 8000, 256)])
def test_head_tiles_of_small_vocabularies(dev, rows, vocab, hidden):
    test_head_at_few_steps(dev, rows, vocab, hidden)
