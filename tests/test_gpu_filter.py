"""GPU parity: top-k / top-p logit filtering through the C ABI vs the oracle.

The kept set is compared exactly.  The top-p cut-off compares a cumulative probability with p; the
kernel sums it in fp32, the oracle in fp64, so a row is only compared when no cumulative probability
of its distinct values lies within 2e-5 of p (almost every row: the tests assert how many)."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _f64(t):
    return t.detach().cpu().to(torch.float64).numpy()


def _decided_rows(x, keep_k, p, T):
    """Rows of x (fp64 [rows, V]; keep_k = what top-k left) whose top-p cut-off does not hinge on rounding."""
    ok = np.ones(x.shape[0], dtype=bool)
    if p >= 1.0:
        return ok
    for r in range(x.shape[0]):
        v = x[r][keep_k[r]] / T[r]
        if v.size == 0 or not np.isfinite(v.max()):       # nothing finite in the row: no softmax, left alone
            continue
        vals, counts = np.unique(v, return_counts=True)
        mass = counts * np.exp(vals - vals[-1])
        cum = np.cumsum(mass[::-1]) / mass.sum()
        ok[r] = np.abs(cum - p).min() > 2e-5
    return ok


def _check(dev, logits, k, p, temps=None, out=None, min_decided=0.9):
    import mdx
    rows = logits.reshape(-1, logits.shape[-1]).shape[0]
    got = mdx.filter_logits(logits.to(dev) if out is None else out, top_k=k, top_p=p,
                            temperatures=None if temps is None else temps.to(dev), out=out)
    torch.cuda.synchronize()
    x = _f64(logits).reshape(rows, -1)
    T = np.ones(rows) if temps is None else np.repeat(temps.numpy().astype(np.float64), rows // temps.numel())
    want = oracle.filter_logits(x, top_k=k, top_p=p, temperatures=T)
    g = _f64(got).reshape(rows, -1)
    decided = _decided_rows(x, np.isfinite(oracle.filter_logits(x, top_k=k)), p, T)
    assert decided.mean() >= min_decided, f"only {decided.mean():.2f} of the rows are clear of a rounding boundary"
    assert np.array_equal(g[decided], want[decided])            # -inf where dropped, the same bits elsewhere
    return got, decided


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [1, 9, 257, 4096 + 5, 151936])
@pytest.mark.parametrize("k,p", [(50, 1.0), (0, 0.9), (20, 0.8), (1, 1.0), (0, 0.0), (0, 0.2)])
def test_filter_shapes(dev, dtype, V, k, p):
    g = torch.Generator().manual_seed(V + k)
    logits = (torch.randn(3, 4, V, generator=g) * 3).to(dtype)
    _check(dev, logits, k, p)


def test_filter_temperatures_per_sequence(dev):
    g = torch.Generator().manual_seed(2)
    logits = (torch.randn(4, 8, 30011, generator=g) * 2.5).bfloat16()
    temps = torch.tensor([0.5, 1.0, 1.7, 0.9])
    _, decided = _check(dev, logits, 0, 0.85, temps)
    _check(dev, logits, 100, 0.6, temps)
    # colder sequences keep fewer elements
    import mdx
    kept = torch.isfinite(mdx.filter_logits(logits.to(dev), top_p=0.85, temperatures=temps.to(dev)).float()).sum(-1).float().mean(-1).cpu()
    assert kept[0] < kept[1] < kept[2]


def test_filter_in_place_unaligned_rows_and_existing_minus_inf(dev):
    """Rows that start off a 16-byte boundary, input and output aligned differently, out == logits, and
    rows that already hold -inf (kept at -inf; an all -inf row is left alone)."""
    import mdx
    g = torch.Generator().manual_seed(5)
    V, stride = 3001, 3003
    buf = (torch.randn(10, stride, generator=g) * 3).bfloat16()
    buf[2, :V:3] = float("-inf")
    buf[7, :] = float("-inf")
    logits = buf[:, :V]                                           # row stride 3003: every row starts elsewhere mod 16
    x = _f64(logits)
    want = oracle.filter_logits(x, top_k=64, top_p=0.95)
    decided = _decided_rows(x, np.isfinite(oracle.filter_logits(x, top_k=64)), 0.95, np.ones(10))
    assert decided.sum() >= 9
    d = buf.to(dev)
    out_other = torch.empty(10, V + 1, dtype=torch.bfloat16, device=dev)[:, 1:]     # another alignment than the input's
    got = mdx.filter_logits(d[:, :V], top_k=64, top_p=0.95, out=out_other)
    torch.cuda.synchronize()
    assert np.array_equal(_f64(got)[decided], want[decided])
    got2 = mdx.filter_logits(d[:, :V], top_k=64, top_p=0.95, out=d[:, :V])         # in place
    torch.cuda.synchronize()
    assert got2.data_ptr() == d.data_ptr()
    assert np.array_equal(_f64(d[:, :V])[decided], want[decided])
    assert np.array_equal(_f64(d[:, V:]), _f64(buf[:, V:]))                          # the padding is not touched
    assert not torch.isfinite(d[7, :V].float()).any()


def test_filter_heavy_ties_and_large_logits(dev):
    """Rows of few distinct values (ties at both cut-offs are all kept) and logits far from zero, where
    a softmax term taken relative to anything but the row maximum would underflow."""
    g = torch.Generator().manual_seed(8)
    few = torch.randint(-3, 4, (6, 5000), generator=g).to(torch.bfloat16)
    _check(dev, few, 10, 1.0)
    _check(dev, few, 0, 0.5, min_decided=0.5)
    big = (torch.randn(6, 20000, generator=g) * 2 + 150).bfloat16()
    _check(dev, big, 0, 0.9, min_decided=0.5)
    neg = (torch.randn(6, 20000, generator=g) * 2 - 300).to(torch.float16)
    _check(dev, neg, 30, 0.7, min_decided=0.5)


def test_filtered_sampling_matches_oracle_end_to_end(dev):
    """filter -> confidence_argmax with Gumbel noise == the oracle's confidence on the oracle's filtered
    logits: the picked token is always one that survived, its probability is the filtered softmax's."""
    import mdx
    g = torch.Generator().manual_seed(13)
    V = 151936
    logits = (torch.randn(2, 8, V, generator=g) * 3).bfloat16()
    u = torch.rand(2, 8, V, generator=g).clamp_(1e-10, 1 - 1e-10)
    noise = -torch.log(-torch.log(u))
    temps = torch.tensor([0.8, 1.2])
    f, decided = _check(dev, logits, 50, 0.9, temps)
    x0, p = mdx.confidence_argmax(f, temps.to(dev), noise.to(dev))
    torch.cuda.synchronize()
    want = oracle.filter_logits(_f64(logits).reshape(16, V), top_k=50, top_p=0.9, temperatures=np.repeat(temps.numpy().astype(np.float64), 8))
    ex0, ep = oracle.confidence_argmax(want.reshape(2, 8, V), temps.numpy(), noise.numpy())
    d = decided.reshape(2, 8)
    assert np.array_equal(x0.cpu().numpy()[d], ex0[d])
    np.testing.assert_allclose(p.cpu().numpy()[d], ep[d], rtol=2e-5)
    assert np.all(np.isfinite(want.reshape(2, 8, V)[np.arange(2)[:, None], np.arange(8)[None], ex0]))


def test_filter_rejects_fp32_and_bad_arguments(dev):
    import mdx
    x = torch.randn(2, 100, device=dev)
    with pytest.raises(mdx.MdxError):
        mdx.filter_logits(x, top_k=5)
    with pytest.raises(mdx.MdxError):
        mdx.filter_logits(x.bfloat16(), top_k=-1)
    with pytest.raises(mdx.MdxError):
        mdx.filter_logits(x.bfloat16(), top_p=float("nan"))
    same = mdx.filter_logits(x.bfloat16())                                            # both filters off: a copy
    assert torch.equal(same, x.bfloat16())


def test_unmask_step_with_filters(dev):
    """The whole step with the HF variant's sampling arguments (temperature, top-k, top-p, Gumbel noise)."""
    import mdx
    g = torch.Generator().manual_seed(21)
    V, MASK = 50021, 50000
    logits = (torch.randn(3, 16, V, generator=g) * 3).bfloat16()
    noise = -torch.log(-torch.log(torch.rand(3, 16, V, generator=g).clamp_(1e-10, 1 - 1e-10)))
    temps = torch.tensor([0.7, 1.0, 1.4])
    tokens = torch.where(torch.rand(3, 16, generator=g) < 0.7, torch.tensor(MASK), torch.randint(0, V, (3, 16), generator=g))
    T = np.repeat(temps.numpy().astype(np.float64), 16)
    x = _f64(logits).reshape(48, V)
    decided = _decided_rows(x, np.isfinite(oracle.filter_logits(x, top_k=40)), 0.9, T)
    assert decided.all()
    want = oracle.filter_logits(x, top_k=40, top_p=0.9, temperatures=T).reshape(3, 16, V)
    ex0, ep, etr, etok = oracle.unmask_step(want, tokens.numpy(), MASK, 0.5, 2, temps.numpy(), noise.numpy())
    d_tokens = tokens.clone().to(dev)
    x0, p, tr, cnt = mdx.unmask_step(logits.to(dev), d_tokens, MASK, 0.5, 2, temps.to(dev), noise.to(dev), top_k=40, top_p=0.9)
    torch.cuda.synchronize()
    assert np.array_equal(x0.cpu().numpy(), ex0)
    np.testing.assert_allclose(p.cpu().numpy(), ep, rtol=2e-5)
    assert np.array_equal(tr.cpu().numpy(), etr) and np.array_equal(d_tokens.cpu().numpy(), etok)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [5, 33, 1000, 40961, 151936])
@pytest.mark.parametrize("k,p", [(1, 1.0), (50, 0.9), (256, 0.7), (300, 0.95), (512, 1.0), (513, 0.9), (0, 0.8), (20, 0.0)])
@pytest.mark.parametrize("noise", ["none", "seed", "tensor"])
def test_filtered_step_is_the_filter_and_the_step(dev, dtype, V, k, p, noise):
    """unmask_step(top_k, top_p), which never writes the filtered copy, against unmask_step on filter_logits' result: rows of
    random logits, of few distinct values (more ties at the cut-off than a candidate list holds), constant, mostly -inf and all
    -inf, starting on and off a 16-byte boundary."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(V + k)
    bs, S = 2, 6
    for pad in (0, 3):
        buf = (torch.randn(bs * S, V + pad, generator=g, device=dev) * 3).to(dtype)
        buf[1] = (buf[1].float() / 4).round().to(dtype)
        buf[2] = 1.5
        buf[3, : V - min(V, 30)] = float("-inf")
        buf[4] = float("-inf")
        buf[5, ::2] = 0.0
        buf[5, 1::2] = -0.0
        logits = buf[:, :V].view(bs, S, V) if pad == 0 else buf[:, :V].unflatten(0, (bs, S))
        temps = torch.tensor([0.7, 1.0], device=dev)
        opts = dict(none={}, seed=dict(seed=77, offset=3),
                    tensor=dict(noise=-torch.log(-torch.log(torch.rand(bs, S, V, generator=g, device=dev).clamp_(1e-9, 1 - 1e-6)))))[noise]
        masks = torch.full((bs, S), 9, dtype=torch.int64, device=dev)
        a, b = masks.clone(), masks.clone()
        got = mdx.unmask_step(logits, a, 9, 0.9, 2, temperatures=temps, top_k=k, top_p=p, **opts)
        want = mdx.unmask_step(mdx.filter_logits(logits, k, p, temps), b, 9, 0.9, 2, temperatures=temps, **opts)
        assert torch.equal(got[0], want[0])
        np.testing.assert_allclose(got[1].cpu().numpy(), want[1].cpu().numpy(), rtol=5e-6)
        assert torch.equal(got[2], want[2]) and torch.equal(got[3], want[3]) and torch.equal(a, b)


@pytest.mark.parametrize("V", [700, 151936])
@pytest.mark.parametrize("k", [63, 64, 65, 128, 400, 511, 512])
@pytest.mark.parametrize("p", [0.5, 0.97, 1.0])
def test_filtered_step_at_the_edges_of_a_lane_and_a_register(dev, V, k, p):
    """Kept elements one per lane (up to 64, ties at the cut-off included), eight registers of them (up to 512) and more, from few
    candidates and many: as above, against the step on the filtered copy."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(V + k)
    logits = (torch.randn(1, 8, V, generator=g, device=dev) * 3).to(torch.bfloat16)
    logits[0, 1] = (logits[0, 1] * 8).round() / 8
    logits[0, 2, ::3] = logits[0, 2].max()                   # more ties than are kept
    logits[0, 3, 5 : 5 + k - 1] = 30.0                       # k - 1 ahead of the rest
    logits[0, 4, 70 : 70 + k] = 30.0                         # k
    a = torch.full((1, 8), 9, dtype=torch.int64, device=dev)
    b = a.clone()
    got = mdx.unmask_step(logits, a, 9, 0.9, 2, temperatures=None, top_k=k, top_p=p, seed=5, offset=1)
    want = mdx.unmask_step(mdx.filter_logits(logits, k, p, None), b, 9, 0.9, 2, temperatures=None, seed=5, offset=1)
    assert torch.equal(got[0], want[0])
    np.testing.assert_allclose(got[1].cpu().numpy(), want[1].cpu().numpy(), rtol=5e-6)    # as above: fp32 sums in another order
    assert torch.equal(a, b) and torch.equal(got[3], want[3])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [1, 7, 17, 40, 64, 100])
@pytest.mark.parametrize("p", [0.3, 0.6, 0.9, 0.99])
def test_filtered_step_with_ties_across_both_cut_offs(dev, dtype, k, p):
    """Candidates that share all bits but one, none but the sign, or all of them, and runs of equal ones on either side of the k-th and of the top-p
    cut-off: against the step on the filtered copy, whose cut-offs are found by counting."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(100 * k + int(100 * p))
    V = 5000
    rows = torch.full((1, 8, V), -60.0, device=dev)
    values = [[5.0] + [4.5] * 6 + [4.0] * 10 + [3.5] * 30 + [1.0] * 200, [2.0] * 64 + [1.9921875] * 64, [3.0] * 300, [0.25, 0.0, -0.0, -0.25] * 40,
              [-1.0] * 20 + [-2.0] * 50 + [-4.0] * 60, [8.0] + [-50.0] * 80, [float(v) for v in range(40, -40, -1)], [1.0, 0.5] * 33]
    for row, v in zip(rows[0], values):
        row[torch.randperm(V, generator=g, device=dev)[:len(v)]] = torch.tensor(v, device=dev)
    logits = rows.to(dtype)
    a = torch.full((1, 8), 9, dtype=torch.int64, device=dev)
    b = a.clone()
    got = mdx.unmask_step(logits, a, 9, 0.9, 2, temperatures=None, top_k=k, top_p=p, seed=5, offset=1)
    want = mdx.unmask_step(mdx.filter_logits(logits, k, p, None), b, 9, 0.9, 2, temperatures=None, seed=5, offset=1)
    assert torch.equal(got[0], want[0])
    np.testing.assert_allclose(got[1].cpu().numpy(), want[1].cpu().numpy(), rtol=5e-6)    # as above: fp32 sums in another order
    assert torch.equal(a, b) and torch.equal(got[3], want[3])


@pytest.mark.parametrize("k", [3, 50, 400])
def test_filtered_step_does_not_depend_on_the_order_of_its_candidates(dev, k):
    """The candidates of a row are listed in whatever order its wavefronts come: rows that hold the same logits at other columns
    get the same confidence, and a seeded step repeats, both bit for bit."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(k)
    V = 151936
    base = (torch.randn(V, generator=g, device=dev) * 3).bfloat16()
    base[:8] = torch.arange(8, device=dev).bfloat16() / 8 + base.max()                    # one row maximum, whatever the order
    rows = torch.stack([base[torch.randperm(V, generator=g, device=dev)] for _ in range(96)]).view(3, 32, V)
    masks = torch.full((3, 32), 9, dtype=torch.int64, device=dev)
    for p in (1.0, 0.9):
        conf = mdx.unmask_step(rows, masks.clone(), 9, 0.9, 2, top_k=k, top_p=p)[1]
        assert len(set(conf.flatten().view(torch.int32).tolist())) == 1
    temps = torch.tensor([0.7, 1.0, 1.3], device=dev)
    first = None
    for _ in range(10):
        tokens = masks.clone()
        got = [*mdx.unmask_step(rows, tokens, 9, 0.02, 2, temperatures=temps, top_k=k, top_p=0.9, seed=11, offset=4), tokens]
        got[1] = got[1].view(torch.int32)
        first = first or got
        assert all(torch.equal(a, b) for a, b in zip(got, first))


@pytest.mark.parametrize("form", ["counters", "bisection", "lists", "lists_run_over"])
@pytest.mark.parametrize("call", ["filter", "step"])
def test_filter_top_p_cut_off_is_exact_where_the_masses_are(dev, form, call):
    """Logits 0, -1, -2, .. at the temperature 1 / ln 2 weigh 2^0, 2^-1, 2^-2, ..: cumulative masses that 64-bit sums hold exactly,
    so the cut-off is right for every p, the fp32 values next to the cumulative shares included."""
    import mdx
    from fractions import Fraction
    rng = np.random.default_rng(3)
    n, k = [int(c) << (i // 2) for i, c in enumerate(rng.integers(300, 900, 14))], 0
    if form == "bisection":
        n[7], n[9] = 66000, 70001                                        # more than a 16-bit counter holds
    if form.startswith("lists"):
        n, k = [3, 5, 20, 60, 200, 150 if form == "lists" else 66000], 400     # more ties at the k-th largest than a list holds
    values = rng.permutation(np.repeat(-np.arange(len(n)), n))
    logits = torch.from_numpy(values).to(torch.bfloat16).to(dev).view(1, 1, -1)
    if form == "lists":
        logits = torch.nn.functional.pad(logits, (0, 5000), value=-300.0)
    temps = torch.tensor([1.4426950408889634], device=dev)
    upto = list(np.cumsum([Fraction(c, 2 ** i) for i, c in enumerate(n)]))
    masks = torch.full((1, 1), 9, dtype=torch.int64, device=dev)
    for i in range(len(n) - 1):
        near = np.float32(float(upto[i] / upto[-1]))
        for p in (np.nextafter(near, np.float32(0)), near, np.nextafter(near, np.float32(1))):
            last = next(j for j in range(len(n)) if upto[j] > Fraction(float(p)) * upto[-1])
            if call == "filter":
                kept = torch.isfinite(mdx.filter_logits(logits, top_k=k, top_p=float(p), temperatures=temps)).sum().item()
                assert kept == sum(n[: last + 1]), (i, p)
            else:
                conf = mdx.unmask_step(logits, masks.clone(), 9, 0.9, 1, temperatures=temps, top_k=k, top_p=float(p))[1].item()
                assert abs(conf * float(upto[last]) - 1) < 1e-5, (i, p)       # (every level is 5e-4 of the sum or more)


def _kept_by_order(bits, dtype, k):
    """What a top-k keeps of rows of 16-bit patterns, from the patterns alone: the k-th in order and everything at or above it."""
    bits = np.where(bits == 0x8000, 0, bits)                                            # (-0 counts as 0)
    key = np.where(bits & 0x8000, ~bits & 0xffff, bits | 0x8000)
    return key >= np.sort(key, axis=1)[:, -k][:, None]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("V", [37, 1003, 40000])
@pytest.mark.parametrize("k,p", [(1, 1.0), (4, 0.9), (30, 0.8), (30, 1.0), (700, 0.9), (700, 1.0), (0, 0.9)])
@pytest.mark.parametrize("noise", ["none", "seed"])
def test_filtered_step_on_rows_that_are_not_finite(dev, dtype, V, k, p, noise):
    """NaN of both signs (ordered above +inf and below -inf), infinities and the type's lowest values, few of them and nothing else:
    the filter keeps what its order says, and the step without the filtered copy does what the step on that copy does."""
    import mdx
    g = torch.Generator(device=dev).manual_seed(V + k)
    inf, nan, low = float("inf"), float("nan"), torch.finfo(dtype).min
    rows = 24
    x = (torch.randn(rows, V, generator=g, device=dev) * 3).to(dtype)
    fills = [(nan, 1), (nan, 5), (nan, V - 3), (nan, V), ("-nan", 1), ("-nan", V - 3), ("-nan", V), (inf, 1), (inf, 6), (inf, V), (-inf, V - 2), (-inf, V - 9),
             (-inf, V), (low, V - 2), (low, V)]
    for r, (value, count) in enumerate(fills):
        at = torch.randperm(V, generator=g, device=dev)[:count]
        if value == "-nan":
            x.view(torch.int16)[r, at] = -1 - 0x3f                                       # sign bit, all exponent bits, a fraction
        else:
            x[r, at] = value
    x[15, : V // 2], x[15, V // 2 :] = nan, -inf
    x.view(torch.int16)[16, : V // 2] = -0x40
    x[16, V // 2 :] = -inf
    x[17, :3], x[17, 3:6] = nan, inf
    x[18, 0], x[18, 1] = inf, -inf
    x.view(torch.int16)[19, ::2] = -0x40
    x[19, 1::2] = nan
    x[20, :], x[20, 2] = low, nan
    x[21, V - 1], x.view(torch.int16)[22, V - 1] = nan, -0x40
    bits = x.view(torch.int16).cpu().numpy().astype(np.int64) & 0xffff
    filtered = mdx.filter_logits(x, k, p)
    if 0 < k < V and p == 1.0:
        got = filtered.view(torch.int16).cpu().numpy().astype(np.int64) & 0xffff
        minus_inf = int(torch.tensor([-inf], dtype=dtype).view(torch.int16)) & 0xffff
        assert np.array_equal(got, np.where(_kept_by_order(bits, dtype, k), bits, minus_inf))
    opts = dict(seed=5, offset=2) if noise == "seed" else {}
    tokens = torch.full((rows, 1), 9, dtype=torch.int64, device=dev)
    want_tokens = tokens.clone()
    got = mdx.unmask_step(x[:, None], tokens, 9, 0.9, 0, top_k=k, top_p=p, **opts)
    want = mdx.unmask_step(filtered[:, None], want_tokens, 9, 0.9, 0, **opts)
    assert torch.equal(got[0], want[0])
    # where the filter keeps a NaN the step's confidence depends on the columns (a lane whose maximum rises after it forgets it)
    ok = ~torch.isnan(filtered.float()).any(1)
    assert ok.sum() >= 8
    np.testing.assert_allclose(got[1][ok].cpu().numpy(), want[1][ok].cpu().numpy(), rtol=5e-6)   # (equal NaN; fp32 sums in another order)
    assert torch.equal(got[2][ok], want[2][ok]) and torch.equal(got[3][ok], want[3][ok]) and torch.equal(tokens[ok], want_tokens[ok])
