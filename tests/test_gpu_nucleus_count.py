"""Top-p alone over bf16 rows (values counted in LDS): thresholds, ties, log-sum-exps and kept-set records against 64-bit sums."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _check(x, top_p, temperature=1.0, div=False, capacity=128):
    """``x``: bf16 [B, n + 1, V] on the GPU.  Every row's kept set holds top_p of the mass and would not without its lightest
    element, whose smallest indices fell first (both up to 1e-6: each element's exponential carries a rounding of 2^-24, so
    do their sums); the log-sum-exps are those of the whole row and of the kept set, to two roundings of fp32."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_DIV, NRL_TEMP_RCP

    b, s, vocab = x.shape
    n = s - 1
    g = torch.Generator(device=DEV).manual_seed(vocab)
    t = torch.where(torch.rand(b, n, generator=g, device=DEV) < 0.5, x[:, :n].float().nan_to_num(nan=-1e30).argmax(-1),
                    torch.randint(0, vocab, (b, n), generator=g, device=DEV))
    lp, thr, tie, lse, lpu, cnt, idx, val = torch.ops.rl_amd.topk_topp_logprob_fwd_rec(
        x, t, n, 0, top_p, temperature, NRL_TEMP_DIV if div else NRL_TEMP_RCP, True, capacity)
    z = x[:, :n].float()
    if temperature != 1.0:
        z = (z / torch.tensor(temperature, device=DEV) if div else z * (torch.tensor(1.0) / temperature).to(DEV)).to(torch.bfloat16).float()
    bad = (z.isnan() | (z == math.inf)).any(-1) | ~z.isfinite().any(-1)
    assert bool(thr[bad].isnan().all()) and bool(lse[bad].isnan().all()) and bool(lp[bad].isnan().all()) and bool((cnt[bad] == -1).all())
    assert bool((tie >= 0).all())
    z64 = z.double()
    index = torch.arange(vocab, device=DEV)
    keep = (z > thr[..., None]) | ((z == thr[..., None]) & (index >= tie[..., None]))
    p = z64.softmax(-1)
    mass, lightest = (p * keep).sum(-1), p.masked_fill(~keep, 2.0).amin(-1)
    ok = ~bad
    cut = 1.0 - float(torch.tensor(1.0) - torch.tensor(top_p))  # 1 - p as fp32 holds it
    assert bool(keep.any(-1)[ok].all())
    assert bool((mass >= cut - 1e-6)[ok].all())
    assert bool(((mass - lightest <= cut + 1e-6) | (keep.sum(-1) == 1))[ok].all())
    want = z64.masked_fill(~keep, -math.inf).logsumexp(-1)
    tol = 2.0 ** -23 * (2 + want.abs() + z64.amax(-1).abs())
    assert bool(((lse.double() - want).abs() <= tol)[ok].all())
    xt = z64.gather(-1, t[..., None])[..., 0]
    kept_t = keep.gather(-1, t[..., None])[..., 0]
    fin = ok & kept_t
    tol_t = tol + 2.0 ** -23 * xt.abs()
    assert bool(((lp.double() - (xt - want)).abs() <= tol_t)[fin].all())
    assert bool((lp == -math.inf)[ok & ~kept_t].all())
    fin = ok & xt.isfinite()
    full = z64.logsumexp(-1)
    tol_f = 2.0 ** -23 * (2 + full.abs() + z64.amax(-1).abs() + xt.abs())   # the same two roundings, of the whole row's sum
    assert bool(((lpu.double() - (xt - full)).abs() <= tol_f)[fin].all())
    kept_n = keep.sum(-1)
    on = cnt >= 0
    assert torch.equal(cnt[on].long(), kept_n[on])
    for bi, i in on.nonzero().tolist():
        c = int(cnt[bi, i])
        ids = idx[bi, i, :c].long()
        assert bool(keep[bi, i, ids].all()) and ids.unique().numel() == c
        v = z[bi, i, ids]
        assert torch.equal(v, val[bi, i, :c])
        assert bool(((v[1:] < v[:-1]) | ((v[1:] == v[:-1]) & (ids[1:] < ids[:-1]))).all())   # descending (value, index)
    return cnt, kept_n


@pytest.mark.parametrize("vocab", [1, 7, 64, 1025, 8191, 32775, 151936])
@pytest.mark.parametrize("top_p", [1e-9, 0.3, 0.95, 0.9999])
def test_rows_of_every_spread(vocab, top_p):
    """Standard deviations from nearly flat (thousands of ties at the threshold) to nearly certain, shifted to either side of zero;
    rows start off the 16-byte grid where the vocabulary is odd."""
    g = torch.Generator(device=DEV).manual_seed(vocab)
    sd = torch.tensor([0.02, 0.5, 2.0, 3.0, 4.5, 8.0, 1.0, 3.0, 1.0], device=DEV).view(1, -1, 1)
    shift = torch.tensor([0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -20.0, 40.0, 0.0], device=DEV).view(1, -1, 1)
    x = (torch.randn(2, 9, vocab, generator=g, device=DEV) * sd + shift).to(torch.bfloat16)
    cnt, kept_n = _check(x, top_p)
    assert bool((cnt >= 0)[kept_n <= 4].all())


@pytest.mark.parametrize("div", [False, True])
@pytest.mark.parametrize("temperature", [0.7, 1.3])
def test_temperatures_and_layouts(temperature, div):
    g = torch.Generator(device=DEV).manual_seed(3)
    x = (torch.randn(3, 6, 20010, generator=g, device=DEV) * 3).to(torch.bfloat16)
    _check(x, 0.9, temperature, div)
    _check(x.transpose(0, 1), 0.9, temperature, div)      # rows of a batch far apart, batches close together
    _check(x[..., 3:20001], 0.9, temperature, div)        # rows longer apart than they are, off the 16-byte grid
    _check(x[:, ::2], 0.9, temperature, div)


@pytest.mark.parametrize("capacity", [1, 128, 2048])
def test_records_up_to_their_capacity(capacity):
    """Kept sets on either side of the capacity, with ties that fall: coarse values (steps of 1/8) tie by the dozen."""
    g = torch.Generator(device=DEV).manual_seed(capacity)
    x = torch.randn(1, 33, 4099, generator=g, device=DEV) * torch.linspace(0.5, 6.0, 33, device=DEV).view(1, -1, 1)
    x = (x * 8).round() / 8 + 0.0   # (no negative zeros: they come before the positive ones in the order of the values)
    cnt, kept_n = _check(x.to(torch.bfloat16), 0.9, capacity=capacity)
    n = cnt.shape[1]
    assert bool((cnt == kept_n)[kept_n <= capacity].all()) and bool((cnt == -1)[kept_n > capacity].all()) and n == 32


def test_values_outside_the_bins():
    """Masked vocabulary (-inf, finfo.min, -1e9), zeros and magnitudes under 2^-31 among ordinary values, a maximum of zero, thresholds
    among the zeros, values above 2^33, rows of nothing but -inf, NaN and +inf."""
    g = torch.Generator(device=DEV).manual_seed(11)
    vocab = 5003
    x = torch.randn(1, 16, vocab, generator=g, device=DEV) * 3
    part = torch.rand(1, 16, vocab, generator=g, device=DEV) < 0.4
    for i, fill in enumerate((-math.inf, -3.3e38, -1e9, 0.0, -0.0, 1e-12, -1e-30)):
        x[0, i] = x[0, i].masked_fill(part[0, i], fill)
    x[0, 7] = -x[0, 7].abs() - 1.0
    x[0, 7, 100:103] = 0.0                     # the maximum is zero, three times
    x[0, 8] = 0.0                              # the threshold is among the zeros
    x[0, 9] = x[0, 9] * 1e-12
    x[0, 10, 17] = 2.0 ** 40                   # above the bins
    x[0, 11] = -math.inf
    x[0, 12, 5] = math.nan
    x[0, 13, 6] = math.inf
    x[0, 14] = -2.0 ** 40                      # every value below the bins, and one that is not
    x[0, 14, 9] = -2.0 ** 39
    _check(x.to(torch.bfloat16), 0.95)
    y = torch.full((1, 3, vocab), -1.5, device=DEV)
    y[0, 1] = torch.where(torch.arange(vocab, device=DEV) % 3 == 0, 2.0, -5.0)
    _check(y.to(torch.bfloat16), 0.75)         # one giant tie; a tie of a third of the row


def test_repeats_bit_for_bit():
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(5)
    x = (torch.randn(1, 40, 151936, generator=g, device=DEV) * torch.linspace(1.0, 6.0, 40, device=DEV).view(1, -1, 1)).to(torch.bfloat16)
    t = torch.randint(0, 151936, (1, 39), generator=g, device=DEV)
    first = torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, 39, 0, 0.95, 1.0, NRL_TEMP_RCP, True)
    for _ in range(3):
        for a, b in zip(first, torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, 39, 0, 0.95, 1.0, NRL_TEMP_RCP, True)):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [5, 20003, 131077])
def test_gradient_rows_cleared_and_streamed_side_by_side(dtype, vocab):
    """Rows on record, streamed rows and rows without a gradient next to each other, whose ends share 16-byte units (odd
    vocabularies) and 256 KiB spans; few rows, so that several workgroups stream one.  The same bits as streaming every row."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(vocab)
    n = 13
    sd = torch.tensor([6.0, 0.3, 6.0, 6.0, 0.3, 0.3, 8.0, 0.3, 5.0, 0.1, 0.1, 9.0, 6.0, 1.0], device=DEV).view(1, -1, 1)
    x = (torch.randn(2, n + 1, vocab, generator=g, device=DEV) * sd).to(dtype)
    t = x[:, :n].float().argmax(-1)
    up = torch.randn(2, n, generator=g, device=DEV)
    up[:, 2] = 0.0
    up[:, 7] = 0.0
    _, thr, tie, lse, _, cnt, idx, val = torch.ops.rl_amd.topk_topp_logprob_fwd_rec(x, t, n, 0, 0.9, 1.0, NRL_TEMP_RCP, False, 128)
    if vocab > 128:
        assert int((cnt < 0).sum()) > 4 and int((cnt >= 0).sum()) > 4
    want = torch.ops.rl_amd.topk_topp_logprob_bwd(x, t, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP)
    got = torch.ops.rl_amd.topk_topp_logprob_bwd(x, t, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP, cnt, idx, val)
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    assert torch.equal(got.view(bits), want.view(bits))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("top_k", [1, 2, 63, 64, 65, 255, 256, 257, 512, 600])
def test_lists_around_the_workgroup_size(dtype, top_k):
    """Candidate lists that one pass of comparisons orders (up to 256) and longer ones that are sorted, with coarse values that tie at
    the top-k threshold, and negative rows: the same kept set as 64-bit sums over the sorted row give, to the element where the
    cut does not fall within 1e-6 of a step."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(top_k)
    n, vocab, top_p = 24, 9001, 0.9
    x = torch.randn(1, n + 1, vocab, generator=g, device=DEV) * torch.linspace(0.5, 6.0, n + 1, device=DEV).view(1, -1, 1)
    x[0, ::3] = (x[0, ::3] * 16).round() / 16 + 0.0
    x[0, 1::5] = -x[0, 1::5].abs() - 0.5
    x = x.to(dtype)
    t = x[:, :n].float().argmax(-1)
    _, thr, tie, lse, _ = torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, n, top_k, top_p, 1.0, NRL_TEMP_RCP, False)
    z = x[0, :n].double()
    index = torch.arange(vocab, device=DEV)
    keep = (z > thr[0, :, None].double()) | ((z == thr[0, :, None].double()) & (index >= tie[0, :, None]))
    z = z.masked_fill(z < z.topk(top_k, dim=-1).values[:, -1:], -math.inf)
    order = z.sort(dim=-1, stable=True)
    mass = order.values.softmax(-1).cumsum(-1)
    cut = float(torch.tensor(1.0) - torch.tensor(top_p))
    kept = mass > cut
    kept[:, -1] = True
    want = torch.zeros_like(keep).scatter_(-1, order.indices, kept)
    clear = ((mass - cut).abs() > 1e-6).all(-1)
    assert int(clear.sum()) > n // 2
    assert torch.equal(keep[clear], want[clear])
    full = z.masked_fill(~keep, -math.inf).logsumexp(-1)
    assert bool(((lse[0].double() - full).abs() <= 2.0 ** -23 * (2 + full.abs() + z.amax(-1).abs())).all())


def test_a_row_with_plus_inf_has_a_nan_gradient_and_is_not_filtered():
    """Softmax makes such a row NaN, no NaN mass is under the cut, so nothing falls: the gradient says that the row has diverged.
    The rows beside it are those of a batch without it."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(2)
    for vocab in (9, 4099, 70000):
        x = (torch.randn(1, 6, vocab, generator=g, device=DEV) * 3).to(torch.bfloat16)
        plain = x.clone()
        x[0, 1, 5] = math.inf
        x[0, 3, vocab - 1] = math.inf
        x[0, 3, 2] = -math.inf
        x[0, 4, :] = -math.inf
        t = torch.full((1, 5), 7, device=DEV)
        up = torch.tensor([[1.0, 0.5, -1.0, math.nan, 1.0]], device=DEV)
        op, back = torch.ops.rl_amd.topk_topp_logprob_fwd_rec, torch.ops.rl_amd.topk_topp_logprob_bwd
        lp, thr, tie, lse, _, cnt, idx, val = op(x, t, 5, 0, 0.9, 1.0, NRL_TEMP_RCP, False, 64)
        assert lp.isnan().tolist() == [[False, True, False, True, True]] and lse.isnan().tolist() == lp.isnan().tolist()
        for rec in ((), (cnt, idx, val)):
            d = back(x, t, thr, tie, lse, up, 5, 1.0, NRL_TEMP_RCP, *rec)
            assert bool(d[0, (1, 3)].isnan().all()) and not bool(d[0, (0, 2, 4, 5)].isnan().any()) and not bool(d[0, 4].any())
        _, thr0, tie0, lse0, _ = torch.ops.rl_amd.topk_topp_logprob_fwd(plain, t, 5, 0, 0.9, 1.0, NRL_TEMP_RCP, False)
        assert torch.equal(d[0, ::2][:2], back(plain, t, thr0, tie0, lse0, up, 5, 1.0, NRL_TEMP_RCP)[0, ::2][:2])
        f, keep = torch.ops.rl_amd.topk_topp_filter(x[:, :5], thr, tie, 1.0, NRL_TEMP_RCP)
        assert torch.equal(f[0, (1, 3)], x[0, (1, 3)]) and bool(keep[0, (1, 3)].all())


# (rows, vocabulary): rows of 8 KiB, of several to a 256 KiB span and of several spans, ends off the 16-byte grid; buffers of more
# than a span and a half for each of 256 workgroups, so that rows to be streamed are left out of the fill
@pytest.mark.parametrize("dtype,rows,vocab", [(torch.bfloat16, 13000, 4096), (torch.float32, 9001, 3001), (torch.bfloat16, 2600, 20003),
                                              (torch.float32, 1300, 32000), (torch.bfloat16, 300, 200001), (torch.float32, 150, 262144)])
@pytest.mark.parametrize("capacity", [64, 128])
def test_large_gradients_cleared_around_streamed_rows(dtype, rows, vocab, capacity):
    """The same bits as streaming every row, with runs of rows on record, streamed rows and rows without a gradient of random lengths."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(vocab)
    n = rows - 1
    flat = torch.rand(rows, generator=g, device=DEV).view(-1, 1).expand(rows, 1)
    flat = torch.where(torch.arange(rows, device=DEV).view(-1, 1) % 97 < 40, flat.round(), (flat > 0.9).float())   # singles, and long runs
    x = torch.empty((1, rows, vocab), dtype=dtype, device=DEV).normal_(0, 1, generator=g)
    x.mul_(torch.where(flat > 0.5, 0.3, 7.0).view(1, rows, 1).to(dtype))
    t = torch.randint(0, vocab, (1, n), generator=g, device=DEV)
    up = torch.randn(1, n, generator=g, device=DEV)
    up[torch.rand(1, n, generator=g, device=DEV) < 0.1] = 0.0
    _, thr, tie, lse, _, cnt, idx, val = torch.ops.rl_amd.topk_topp_logprob_fwd_rec(x, t, n, 0, 0.9, 1.0, NRL_TEMP_RCP, False, capacity)
    assert int((cnt < 0).sum()) > n // 8 and int((cnt >= 0).sum()) > n // 8
    back = torch.ops.rl_amd.topk_topp_logprob_bwd
    bits = torch.int32 if dtype == torch.float32 else torch.int16
    want = back(x, t, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP)
    assert torch.equal(back(x, t, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP, cnt, idx, val).view(bits), want.view(bits))


def test_short_rows_on_record_cost_a_fill_and_their_entries():
    """4096 rows of 1024 ids: clearing 8 MiB takes a few microseconds and the entries about as much again; a fill that waits for
    every row's flags takes fifteen times the clearing."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(1)
    n, vocab = 4096, 1024
    x = torch.empty((1, n + 1, vocab), dtype=torch.bfloat16, device=DEV).normal_(0, 3, generator=g)
    t = torch.randint(0, vocab, (1, n), generator=g, device=DEV)
    up = torch.randn(1, n, generator=g, device=DEV)
    lp, thr, tie, lse, _, *rec = torch.ops.rl_amd.topk_topp_logprob_fwd_rec(x, t, n, 50, 0.95, 1.0, NRL_TEMP_RCP, False, 128)
    assert bool((rec[0] >= 0).all())
    out = torch.empty_like(x)

    def shortest(f):
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                f()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    shortest(lambda: out.zero_())
    backward = shortest(lambda: torch.ops.rl_amd.topk_topp_logprob_bwd(x, t, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP, *rec))
    assert backward < 8 * shortest(lambda: out.zero_())


@pytest.mark.parametrize("value", [1.5, -1e9, -1e4, 0.0, -0.0, -math.inf, 7.0, 1e-20, math.nan, 2.0 ** 40])
@pytest.mark.parametrize("vocab", [9, 64, 9001, 40008])
def test_a_common_value(value, vocab):
    """One value in none to all of a row's places, at random, at the front, at the end and every other place: whether it is counted
    apart or with the others, and ties that are added up by the vector or one by one, the row comes out the same."""
    g = torch.Generator(device=DEV).manual_seed(vocab)
    x = torch.randn(1, 12, vocab, generator=g, device=DEV) * 3
    at = torch.arange(vocab, device=DEV)
    for i, share in enumerate((0.0, 0.1, 0.24, 0.26, 0.5, 0.8, 0.99, 1.0)):
        x[0, i] = x[0, i].masked_fill(torch.rand(vocab, generator=g, device=DEV) < share, value)
    x[0, 8] = x[0, 8].masked_fill(at < vocab * 3 // 4, value)
    x[0, 9] = x[0, 9].masked_fill(at >= vocab // 3, value)
    x[0, 10] = x[0, 10].masked_fill(at % 2 == 0, value)
    for top_p in (0.3, 0.95):
        _check(x.to(torch.bfloat16), top_p)
    _check((x * 2).clamp(min=-3e38).to(torch.bfloat16), 0.9, temperature=2.0)


def test_a_common_value_costs_no_more_than_others():
    """Rows of which most places hold one value: counted in LDS one lane after the other they took 5 to 6 times what others take."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(1)
    n, vocab = 512, 151936
    x = torch.empty((1, n + 1, vocab), dtype=torch.bfloat16, device=DEV).normal_(0, 3, generator=g)
    t = torch.randint(0, vocab, (1, n), generator=g, device=DEV)

    def shortest(x):
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, n, 0, 0.95, 1.0, NRL_TEMP_RCP, False)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    shortest(x)
    plain = shortest(x)
    assert shortest(x.masked_fill(torch.rand(x.shape, generator=g, device=DEV) < 0.99, -1e9)) < 2.5 * plain
    assert shortest(torch.full_like(x, 1.5)) < 2.5 * plain


def test_a_gradient_of_more_spans_than_a_round_of_flags_holds():
    """88 000 rows just over a 256 KiB span, 23 GB: every workgroup reads flags for more spans than fit one round of two rows each.
    What is not cleared or written keeps the NaN that the buffer's memory held before."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    n, vocab = 88000, 131080
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 64 GB of free GPU memory")
    x = torch.zeros(1, n, vocab, dtype=torch.bfloat16, device=DEV)
    row = torch.arange(n, device=DEV).view(1, n)
    at = (row * 7919) % vocab
    up = torch.where(row % 5 == 3, 0.0, 2.0)
    cnt = torch.where(row % 7 == 2, -1, 1).to(torch.int32)                 # every seventh row streams: none of it is kept
    thr, tie = torch.full((1, n), 0.5, device=DEV), torch.zeros(1, n, dtype=torch.int32, device=DEV)
    lse = torch.full((1, n), math.log(2.0), device=DEV)
    idx = at.unsqueeze(-1).to(torch.int32).expand(1, n, 128).contiguous()
    val = torch.zeros(1, n, 128, device=DEV)
    torch.full((x.numel() + (1 << 21),), math.nan, dtype=torch.bfloat16, device=DEV)
    d = torch.ops.rl_amd.topk_topp_logprob_bwd(x, at, thr, tie, lse, up, n, 1.0, NRL_TEMP_RCP, cnt, idx, val)
    want = torch.where((cnt > 0) & (up != 0), 1.0, 0.0)                   # (1 - exp(0 - log 2)) * 2
    assert torch.equal(d.gather(-1, at.unsqueeze(-1))[..., 0].float(), want)
    assert sum(int(torch.count_nonzero(part)) for part in d[0].split(4000)) == int(want.sum())
