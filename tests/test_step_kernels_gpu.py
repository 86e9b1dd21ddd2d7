"""Kernels of decode steps that ask for a row's or a state's values at once, around the sizes where their forms change."""
import pytest
import torch

import kernel_twins as twin
from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, _attention_case, close, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,P", [(1, 64), (3, 5), (31, 70), (33, 64), (64, 64), (65, 128), (128, 130), (129, 64), (300, 20)])
def test_a_state_of_any_height_moves_on_by_one_token(N, P, dtype):
    """Rows per wave below, at and beyond what is asked for at once. Sums of N products: 2e-5 as for the walks."""
    H, B = 2, 3
    g = torch.Generator(device=DEV).manual_seed(N + P)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    q, k, v = (rnd(B, w + 5)[:, 2:2 + w].to(dtype) for w in (H * N, H * N, H * P))
    state = rnd(B + 1, 3 + H * N * P)
    want_state = state.cpu().clone()
    slots = torch.tensor([2, 0, 3], dtype=torch.int32, device=DEV)
    cu = torch.arange(B + 1, dtype=torch.int32, device=DEV)
    before, decay = state[1].clone(), torch.tensor([0.9, 0.99], device=DEV)
    got = hip().linear_recurrence(q, k, v, state[:, 3:], slots, cu, [1] * B, H, H, N, P, decay=decay, silu=True)
    want = twin.linear_recurrence(q.cpu(), k.cpu(), v.cpu(), want_state[:, 3:], slots.cpu(), cu.cpu(), [1] * B, H, H, N, P, decay=decay.cpu(), silu=True)
    close(got, want, 2e-5)
    close(state, want_state, 2e-5)
    assert torch.equal(state[1], before)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,G,N,P,selective", [(3, 2, 1, 17, 4, False), (1, 3, 3, 31, 36, True), (2, 2, 2, 32, 32, False), (5, 4, 2, 33, 100, True),
                                                 (3, 2, 2, 63, 28, False), (2, 2, 1, 64, 64, True), (2, 3, 1, 65, 132, False), (4, 2, 2, 127, 68, True),
                                                 (8, 4, 4, 128, 128, False), (256, 2, 1, 20, 8, True), (257, 2, 1, 20, 8, True)])
def test_both_forms_of_the_step_give_the_same_bits(B, H, G, N, P, selective, dtype):
    """Up to 512 workgroups' worth of requests and heads four columns go to a lane, unless the states lie at places that are no whole steps
    of four numbers: one step from the same states at such places and at others; states that are not in the step stay."""
    g = torch.Generator(device=DEV).manual_seed(N + P)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    q, k, v = (rnd(B, w + 5)[:, 2:2 + w].to(dtype) for w in (G * N, G * N, H * P))
    kw = (dict(dt=rnd(B, H).to(dtype), dt_bias=rnd(H) - 2, rate=rnd(H).abs() + 0.2, skip=rnd(H)) if selective else
          dict(decay=torch.tensor([0.9, 0.99, 1.0, -0.5], device=DEV)[:H].contiguous(), silu=True))
    start, got = rnd(B + 2, H * N * P), []
    for at in (4, 3):
        state = torch.zeros(B + 2, 8 + H * N * P + -H * N * P % 4, device=DEV)
        state[:, at:at + H * N * P] = start
        slots = torch.arange(B, device=DEV).flip(0).int() + 1
        y = hip().linear_recurrence(q, k, v, state[:, at:at + H * N * P], slots, torch.arange(B + 1, device=DEV).int(), [1] * B, H, G, N, P, **kw)
        rest = state.clone()
        rest[:, at:at + H * N * P] = 0
        assert not rest.any()
        got.append((y, state[:, at:at + H * N * P].clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.equal(got[0][1][0], start[0]) and torch.equal(got[0][1][-1], start[-1]) and not torch.equal(got[0][1][1], start[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,N,P", [(3, 4, 64, 64), (1, 2, 100, 36), (5, 2, 33, 37), (2, 2, 150, 64), (70, 8, 64, 64), (30, 4, 128, 256), (90, 4, 128, 256)])
def test_the_state_moves_on_with_one_rounding_of_its_own_share(B, H, N, P, dtype):
    """a S + b k v^T: k v^T rounded, then a S added to it in one rounding, in every form of the step (for few requests, for many, past
    the caches and through them): the bits that a request's state has had from the step on, and those of float64 rounded once (which
    differs from a single rounding for sums within 2^-29 of a tie only, none of them here)."""
    g = torch.Generator(device=DEV).manual_seed(B * N + P)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    q, k, v = (rnd(B, w).to(dtype) for w in (H * N, H * N, H * P))
    decay, state = torch.rand(H, device=DEV, generator=g), rnd(B, H * N * P)
    added = k.float().view(B, H, N, 1) * v.float().view(B, H, 1, P)
    want = (decay.double().view(1, H, 1, 1) * state.double().view(B, H, N, P) + added.double()).float()
    hip().linear_recurrence(q, k, v, state, torch.arange(B, device=DEV).int(), torch.arange(B + 1, device=DEV).int(), [1] * B, H, H, N, P, decay=decay)
    assert torch.equal(state.view(B, H, N, P), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["silu_before", "sigmoid_behind", "silu_behind"])
@pytest.mark.parametrize("n,parts", [(1023, 1), (1024, 1), (1025, 2), (2048, 1), (2049, 1), (4097, 3), (8192, 1), (8200, 1)])
def test_gated_norm_widths(n, parts, kind, dtype):
    """One group: rows in registers from 1,024 to 8,192 numbers, through LDS on either side. One rounding to the output type."""
    g = torch.Generator(device=DEV).manual_seed(n)
    y = torch.randn(*((parts, 5, n) if parts > 1 else (5, n)), device=DEV, generator=g)
    gate = torch.randn(5, n + 9, device=DEV, generator=g).to(dtype)[:, 3:3 + n]
    w = torch.rand(n, device=DEV, generator=g) + 0.5
    close(hip().gated_rms_norm(y, gate, w, 1e-5, 1, kind, dtype), twin.gated_rms_norm(y, gate, w, 1e-5, 1, kind, dtype),
          1e-6 if dtype == torch.float32 else 4e-3)


@pytest.mark.parametrize("kind", ["silu_before", "sigmoid_behind", "silu_behind"])
@pytest.mark.parametrize("n,few,many", [(2049, 1024, 1025), (4096, 1024, 1025), (4097, 512, 513), (7168, 512, 513)])
def test_gated_norms_of_few_and_of_many_rows_are_the_same_bits(n, few, many, kind):
    """Rows of several partial sums go through LDS from a number of rows on: the same steps and sums in the same order."""
    g = torch.Generator(device=DEV).manual_seed(n)
    y, gate = torch.randn(3, many, n, device=DEV, generator=g), torch.randn(many, n, device=DEV, generator=g).to(torch.bfloat16)
    w = torch.rand(n, device=DEV, generator=g) + 0.5
    out = hip().gated_rms_norm(y, gate, w, 1e-5, 1, kind, torch.bfloat16)
    assert torch.equal(out[:few], hip().gated_rms_norm(y[:, :few].contiguous(), gate[:few], w, 1e-5, 1, kind, torch.bfloat16))


def _clear_choices(logits, scoring, groups, group_top):
    """The tokens whose choice 32 bits cannot turn: scores of different logits, and of groups of them, lie 1e-5 of the larger
    apart or more (equal ones are equal on both sides, and the lower index wins)."""
    scores = {"softmax": torch.softmax(logits, -1), "sigmoid": torch.sigmoid(logits), "chosen": logits}[scoring]
    per = scores.shape[1] // groups
    totals = scores.view(-1, groups, per).topk(min(group_top, per), -1).values.sum(-1)

    def apart(values):
        v = values.sort(-1).values
        gap, size = v[:, 1:] - v[:, :-1], v.abs()[:, 1:].maximum(v.abs()[:, :-1])
        return ((gap <= 1e-12 * size) | (gap > 1e-5 * size)).all(-1)

    return apart(scores) & apart(totals)


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid", "chosen"])
@pytest.mark.parametrize("T,E,groups,keep,top,group_top", [(1, 1, 1, 1, 1, 1), (17, 2, 1, 1, 2, 1), (64, 32, 4, 2, 4, 1), (33, 63, 7, 3, 5, 2),
                                                           (64, 64, 8, 2, 8, 3), (40, 64, 64, 9, 9, 1), (50, 65, 5, 2, 6, 2), (5, 128, 4, 1, 3, 2)])
def test_choices_in_registers_and_through_lds(T, E, groups, keep, top, group_top, scoring):
    """Up to 64 experts a lane holds one, beyond they lie in LDS: the twin's choice either way, with pairs of experts of equal
    scores among them (the lower index wins), also inside the kernel that orders the pairs. Logits are sums of whole numbers,
    so that both sides have the same ones."""
    if scoring == "chosen" and groups > 1:
        groups = keep = 1
    g = torch.Generator(device=DEV).manual_seed(T + E)
    x = torch.randint(-3, 4, (T, 24), device=DEV, generator=g).float()
    router = torch.randint(-2, 3, (E, 24), device=DEV, generator=g).float() * 0.125
    router[1::2] = router[0:E - E % 2:2]
    rule = ops.RouteRule(scoring, None, group_top=group_top, normalise=scoring != "sigmoid", scale=1.25)
    ids, weights = hip().moe_route(x, router, top, groups, keep, rule)
    want_ids, want_w = twin.moe_route(x.cpu(), router.cpu(), top, groups, keep, rule)
    clear = _clear_choices(x.cpu().double() @ router.cpu().double().t(), scoring, groups, group_top)
    assert clear.float().mean() > 0.9
    assert torch.equal(ids.cpu()[clear], want_ids[clear])
    close(weights.cpu()[clear], want_w[clear], 2e-6)           # a softmax of 32-bit exponentials
    up, down = torch.randn(E, 8, 24, device=DEV, generator=g), torch.randn(E, 16, 8, device=DEV, generator=g)
    got = hip().route_and_run_experts(x.to(torch.bfloat16), router, top, groups, keep, up.to(torch.bfloat16), down.to(torch.bfloat16), rule=rule, gated=False)
    want = twin.routed_experts(x.cpu().to(torch.bfloat16), ids.cpu(), weights.cpu(), up.cpu().to(torch.bfloat16), down.cpu().to(torch.bfloat16), gated=False)
    close(got.sum(0), want.sum(0), 3e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [4, 252, 1020, 1024, 1028, 2056])
def test_rows_by_fours_are_those_by_ones(n, dtype):
    """Bias, gate and token mix of rows that begin at any fourth element, against the same rows one element further on, which the
    general kernels take: each value is formed by the same steps."""
    g = torch.Generator(device=DEV).manual_seed(n)
    T, S = 9, 5
    rows = torch.randn(T, n + 8, device=DEV, generator=g).to(dtype)
    gate = torch.randn(T, n + 8, device=DEV, generator=g).to(dtype)
    odd = lambda t: torch.nn.functional.pad(t, (1, 0))[:, 1:]
    for nb in (0, 4, n):
        bias = torch.randn(nb, device=DEV, generator=g)
        for out_dtype in (torch.float32, torch.bfloat16):
            assert torch.equal(hip().add_bias(rows[:, 4:4 + n], bias, out_dtype), hip().add_bias(odd(rows)[:, 4:4 + n], bias, out_dtype))
    a, b = rows.clone(), odd(rows)
    hip().sigmoid_gate_(a[:, 4:4 + n], gate[:, 4:4 + n])
    hip().sigmoid_gate_(b[:, 4:4 + n], gate[:, 4:4 + n])
    assert torch.equal(a, b)
    mu = torch.randn(S, n, device=DEV, generator=g)
    cu = torch.tensor([0, 1, 6, T], dtype=torch.int32, device=DEV)
    seq = torch.tensor([0] + [1] * 5 + [2] * 3, dtype=torch.int32, device=DEV)
    slots = torch.tensor([2, 0, 3], dtype=torch.int32, device=DEV)
    first = torch.randn(4, n + 3, device=DEV, generator=g)
    states = [first.clone(), first.clone()]
    mixes = [hip().token_shift(x[:, 4:4 + n], mu, st[:, 3:], slots, cu, seq) for x, st in zip((rows, odd(rows)), states)]
    assert torch.equal(*mixes) and torch.equal(*states)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1023, 1024, 1025, 2048, 2049, 4096, 4097])
def test_weighted_sum_and_norm_widths(n, dtype):
    """Rows in registers from 1,024 to 4,096 numbers, through LDS on either side: a term as partial sums with a bias, one with
    gate rows. Float32 sums of up to 4,097 squares; one rounding to the output type."""
    g = torch.Generator(device=DEV).manual_seed(n)
    T = 5
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    terms = [(rnd(3, T, n), 0.7, rnd(n)), (rnd(T, n).to(dtype), -0.3, None, rnd(T, 2).to(dtype)[:, 1]), (rnd(T, n).to(dtype), 1.1, None)]
    w, stream = rnd(n), rnd(T, n)
    got = hip().weighted_sum(terms, w, 1e-6, stream, dtype)
    cpu = [tuple(v.cpu() if torch.is_tensor(v) else v for v in term) for term in terms]
    want = twin.weighted_sum(cpu, w.cpu(), 1e-6, stream.cpu(), dtype)
    close(got[0], want[0], 1e-6 if dtype == torch.float32 else 8e-3)
    close(got[1], want[1], 1e-6)


@pytest.mark.parametrize("n,parts", [(1024, 4), (1024, 5), (1030, 1), (2048, 2), (2049, 1), (3000, 3), (4096, 1)])
def test_weighted_sums_of_few_and_of_many_rows_are_the_same_bits(n, parts):
    """Launches of 512 or 1,024 rows and more whose terms are partial sums go through LDS, fewer rows through registers: the
    same steps and sums in the same order."""
    g = torch.Generator(device=DEV).manual_seed(n + parts)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    w, bias = rnd(n), rnd(n)
    for T in (512, 513, 1024, 1025):
        sums, rows, gate, stream = rnd(parts, T, n), rnd(T, n).to(torch.bfloat16), rnd(T, 1), rnd(T, n)
        at = lambda lo: [(sums[:, lo:].contiguous(), 0.7, bias), (rows[lo:], -0.3, None, gate[lo:, 0])]
        many = hip().weighted_sum(at(0), w, 1e-6, stream, torch.bfloat16)
        few = hip().weighted_sum(at(T - 9), w, 1e-6, stream[T - 9:], torch.bfloat16)
        assert torch.equal(many[0][T - 9:], few[0]) and torch.equal(many[1][T - 9:], few[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])
def test_short_convolution_over_the_ends_of_its_groups(taps, dtype):
    """Requests of every length around the eight tokens of a thread; portions of a request give what it gives in one piece."""
    g = torch.Generator(device=DEV).manual_seed(taps)
    C, q_lens = 70, [1, 2, 3, 7, 8, 9, 16, 17, 33]
    T, B = sum(q_lens), len(q_lens)
    x = torch.randn(T, C + 3, device=DEV, generator=g).to(dtype)[:, 2:2 + C]
    w, b = torch.randn(C, taps, device=DEV, generator=g), torch.randn(C, device=DEV, generator=g)
    state = torch.randn(B, C * (taps - 1), device=DEV, generator=g)
    want_state = state.cpu().clone()
    slots = torch.arange(B, dtype=torch.int32, device=DEV).flip(0).contiguous()
    cu = torch.tensor([0] + q_lens, device=DEV).cumsum(0).int()
    before = state.clone()
    got = hip().causal_conv(x, w, b, state, slots, cu, q_lens)
    want = twin.causal_conv(x.cpu(), w.cpu(), b.cpu(), want_state, slots.cpu(), cu.cpu(), q_lens)
    close(got, want, 1e-6 if dtype == torch.float32 else 8e-3)
    assert torch.equal(state.cpu(), want_state)
    pieces = [hip().causal_conv(x[T - 33 + lo:T - 33 + hi], w, b, before, slots[-1:], torch.tensor([0, hi - lo], dtype=torch.int32, device=DEV), [hi - lo])
              for lo, hi in ((0, 1), (1, 12), (12, 33))]
    close(torch.cat(pieces), got[T - 33:], 1e-6 if dtype == torch.float32 else 8e-3)


@pytest.mark.parametrize("taps", [2, 4, 5])
def test_short_convolution_of_one_long_request_among_short_ones(monkeypatch, taps):
    """Steps whose grid by eights would be large and mostly empty walk their tokens: both forms add in one order, so the same bits."""
    g = torch.Generator(device=DEV).manual_seed(taps)
    C, q_lens = 70, [300] + [1] * 20
    T, B = sum(q_lens), len(q_lens)
    x = torch.randn(T, C, device=DEV, generator=g).to(torch.bfloat16)
    w, state = torch.randn(C, taps, device=DEV, generator=g), torch.randn(B, C * (taps - 1), device=DEV, generator=g)
    slots, cu = torch.arange(B, dtype=torch.int32, device=DEV), torch.tensor([0] + q_lens, device=DEV).cumsum(0).int()
    monkeypatch.setattr(ops, "conv_tokens_per_thread", lambda *a: 32)
    states = [state.clone(), state.clone()]
    walked = hip().causal_conv(x, w, None, states[0], slots, cu, q_lens)
    if taps <= 4:
        monkeypatch.setattr(ops, "conv_tokens_per_thread", lambda *a: 8)
    assert torch.equal(hip().causal_conv(x, w, None, states[1], slots, cu, q_lens), walked) and torch.equal(*states)
    want = twin.causal_conv(x.cpu(), w.cpu(), None, state.cpu(), slots.cpu(), cu.cpu(), q_lens)
    close(walked, want, 8e-3)


@pytest.mark.parametrize("scoring", ["softmax", "sigmoid", "chosen"])
@pytest.mark.parametrize("E,groups,keep,top,group_top", [(8, 1, 1, 3, 1), (32, 4, 2, 4, 2), (63, 7, 7, 8, 1), (64, 8, 3, 8, 3), (64, 64, 20, 20, 1), (48, 1, 1, 48, 1)])
def test_the_choice_in_registers_is_that_through_lds(E, groups, keep, top, group_top, scoring):
    """Whole groups of further experts with a bias of minus infinity take the same tokens to the form beyond 64 experts: the same
    ids and the same weights, bit for bit, ties and corrections included."""
    g = torch.Generator(device=DEV).manual_seed(E + top)
    T, n, per = 77, 40, E // groups
    x = torch.randn(T, n, device=DEV, generator=g)
    router = torch.randn(E, n, device=DEV, generator=g) * 0.3
    router[1::3] = router[0::3][:router[1::3].shape[0]]        # equal scores
    more = per * -(-(65 - E) // per)
    wide = torch.cat((router, torch.zeros(more, n, device=DEV)))
    bias = torch.cat((torch.zeros(E, device=DEV), torch.full((more,), -torch.inf, device=DEV)))
    for correction in (None, torch.rand(E, device=DEV, generator=g)):
        if scoring == "chosen" and correction is not None:
            continue
        far = None if correction is None else torch.cat((correction, torch.full((more,), -9.0, device=DEV)))
        rule = lambda c, b: ops.RouteRule(scoring, c, group_top=group_top, normalise=True, scale=1.5, bias=b)
        narrow = hip().moe_route(x, router, top, groups, keep, rule(correction, None))
        there = hip().moe_route(x, wide, top, groups + more // per, keep, rule(far, bias))
        assert torch.equal(narrow[0], there[0]) and torch.equal(narrow[1], there[1])


def test_the_pairs_kernel_chooses_for_any_number_of_tokens():
    """More pairs than their ids have room for in LDS: chosen, counted and ordered all the same (a caller of the entry itself)."""
    T, E, top, rows = 6000, 32, 2, 64
    g = torch.Generator(device=DEV).manual_seed(4)
    logits = torch.randn(T, E, device=DEV, generator=g)
    P = T * top
    ids, weights = torch.empty(P, dtype=torch.int32, device=DEV), torch.empty(P, device=DEV)
    most = P // rows + E
    order, offsets, expert, row = (torch.empty(k, dtype=torch.int32, device=DEV) for k in (P, E + 1, most, most))
    ops.core().call("me_moe_sort", ids.data_ptr(), P, E, 0, most, rows, order.data_ptr(), offsets.data_ptr(), expert.data_ptr(), row.data_ptr(),
                    logits.data_ptr(), weights.data_ptr(), top, 1, 1, *ops.RouteRule("chosen").args(), ops._stream())
    best = logits.topk(top, -1)
    assert torch.equal(ids.view(T, top).long(), best.indices)
    close(weights.view(T, top), torch.softmax(best.values.double(), -1), 2e-6)
    assert torch.equal(order.sort().values.long(), torch.arange(P, device=DEV))
    assert torch.equal(ids[order.long()].sort().values, ids[order.long()])
    assert torch.equal(offsets[1:].long(), torch.bincount(ids.long(), minlength=E).cumsum(0))


def test_a_bias_on_more_rows_than_a_grid_has_by_fours():
    """2^26 + 8 rows of 128 by fours would be 2^32 threads and more: the general kernel takes them (17 GB of results)."""
    T, n = (1 << 26) + 8, 128
    row, bias = torch.randn(1, n, device=DEV).to(torch.bfloat16), torch.randn(n, device=DEV)
    out = hip().add_bias(row.expand(T, n), bias, torch.bfloat16)
    want = hip().add_bias(row, bias, torch.bfloat16)
    for part in out.split(1 << 23):
        assert bool((part == want).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,parts", [(1024, 1), (1024, 5), (2056, 3), (1001, 4), (8200, 2)])
def test_sums_and_norms_of_few_and_of_many_rows_are_the_same(n, parts, dtype):
    """From 512 rows on a row's loads go one after the other and fewer threads share a row: the sums are the same bits as in a
    launch of few rows, the norms add their squares in another order (and round once to the output type)."""
    g = torch.Generator(device=DEV).manual_seed(n + parts)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T = 512
    stream, sums, rows = rnd(T, n), rnd(parts, T, n), rnd(T, n).to(dtype)
    w1, w2, s1 = rnd(n), rnd(n), rnd(n)
    many = hip().scaled_sum_norm(stream, [(sums, s1), (rows, None)], 0.45, w1, w2, 1e-5, dtype)
    few = hip().scaled_sum_norm(stream[500:], [(sums[:, 500:].contiguous(), s1), (rows[500:], None)], 0.45, w1, w2, 1e-5, dtype)
    assert torch.equal(many[0][500:], few[0])
    for a, b in zip(many[1:], few[1:]):
        close(a[500:], b, 1e-6 if dtype == torch.float32 else 8e-3)
    close(many[0], stream + 0.45 * (s1 * sums.sum(0) + rows.float()), 1e-6)


@pytest.mark.parametrize("dtype,Hq,Hkv,D,page", [(torch.bfloat16, 16, 8, 128, 16), (torch.bfloat16, 6, 2, 32, 8), (torch.bfloat16, 4, 4, 256, 16), (torch.float32, 4, 2, 16, 16)])
@pytest.mark.parametrize("seqs", [[(1, 1)], [(700, 1), (33, 1), (900, 1), (1, 1)], [(300, 1), (50, 50), (2, 2)], [(9, 9)], [(1500, 1)] * 40])
def test_gated_heads_give_the_bits_of_a_gate_behind_the_attention(dtype, Hq, Hkv, D, page, seqs):
    """Joined with the merge of a decode step's partitions, behind one partition, a mixed step or float32 in a kernel of its own; a gate that is
    not a number or closes altogether reaches its own head only; the step in one launch the same."""
    args = _attention_case(dtype, Hq, Hkv, D, page, seqs, seed=len(seqs))
    T = args[0].shape[0]
    g = torch.Generator(device=DEV).manual_seed(D)
    gates = (3 * torch.randn(T, Hq + 9, device=DEV, generator=g)).to(dtype)[:, 3:3 + Hq]
    gates[0, 1], gates[-1, 0], gates[-1, 2] = -200.0, float("nan"), float("inf")
    for even in (False, True):
        want = hip().paged_attention(*args, even_contexts=even)
        hip().head_gate(want, gates, Hq, D)
        got = hip().paged_attention(*args, even_contexts=even, head_gate=gates)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))
        assert int(torch.isnan(got).sum()) == D
    if dtype == torch.bfloat16 and all(n == 1 for _, n in seqs):
        q, k_cache, v_cache, _, bt, ctx = args[:6]
        rows = q._base
        rows[:, Hq * D:] = torch.randn(T, 2 * Hkv * D, device=DEV, generator=g).to(dtype)
        outs = [hip().decode_step_attention(rows, None, None, 0.0, None, k_cache.clone(), v_cache.clone(), page, bt, ctx, args[10], D ** -0.5, None, Hq, Hkv, D, **kw)
                for kw in ({}, dict(head_gate=gates))]
        hip().head_gate(outs[0], gates, Hq, D)
        assert torch.equal(torch.nan_to_num(outs[0]), torch.nan_to_num(outs[1])) and int(torch.isnan(outs[1]).sum()) == D


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["relu2", "silu"])
@pytest.mark.parametrize("M,N,K", [(1, 16, 8), (1, 3072, 1024), (7, 40, 136), (16, 8192, 1024), (17, 96, 256), (32, 3072, 1024), (33, 3072, 1024), (65, 3072, 1024), (300, 264, 128)])
def test_an_activation_in_the_products_epilogue_gives_the_bits_of_one_behind_it(M, N, K, kind, dtype):
    """Row counts on both sides of what the kernel for few rows takes, wide loads and others, rows of a wider tensor, a sum that is not a number
    or not finite."""
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x, w = (torch.randn(n, K + 8, device=DEV, generator=g).to(dtype)[:, :K] for n in (M, N))
    x[0, 0], w[3, 0] = float("inf"), 0.0
    want = hip().activation(hip().linear(x, w), kind)
    got = hip().activated_linear(x, w, kind)
    assert got.shape == (M, N) and got.dtype == dtype and got.is_contiguous()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))
    with pytest.raises(ops.KernelError):
        hip().activated_linear(x, w[:, :K - 1], kind)


@pytest.mark.parametrize("widths,rows", [((1,), [0]), ((3, 4097, 16), [2, 5, 0]), ((70000, 5), [1]), (tuple(range(1, 71)), list(range(0, 140, 2))), ((8,), [])])
def test_rows_of_many_tensors_go_back_to_what_they_start_from(widths, rows):
    """More tensors and rows than one launch holds, rows that begin at no step of four numbers; the other rows stay."""
    g = torch.Generator(device=DEV).manual_seed(len(widths))
    tensors = [torch.randn(141, w, device=DEV, generator=g) for w in widths]
    firsts = [torch.randn(w, device=DEV, generator=g) if i % 3 == 1 else None for i, w in enumerate(widths)]
    want = [t.clone() for t in tensors]
    for t, f in zip(want, firsts):
        t[rows] = 0.0 if f is None else f
    hip().reset_rows(tensors, firsts, rows)
    assert all(torch.equal(a, b) for a, b in zip(tensors, want))
    with pytest.raises(ops.KernelError):
        hip().reset_rows(tensors, firsts, [0, 141])
    with pytest.raises(ops.KernelError):
        hip().reset_rows(tensors, firsts, [-1])
    assert all(torch.equal(a, b) for a, b in zip(tensors, want))


@pytest.mark.parametrize("takes", [True, False])
def test_states_go_back_through_the_backend_in_use(takes):
    """The pool asks whichever backend is installed; one without a kernel for it leaves the rows to plain tensor operations."""
    from types import SimpleNamespace
    from mini_engine_amd.cache.pool import CachePool
    pool, calls = CachePool.__new__(CachePool), []
    pool.states = [torch.ones(5, 7, device=DEV), None, torch.ones(5, 2, 3, device=DEV)]
    pool.state_initial = [None, None, torch.full((2, 3), 4.0, device=DEV)]
    want = [t if t is None else t.clone() for t in pool.states]
    want[0][[1, 3]], want[2][[1, 3]] = 0.0, 4.0
    ops.set_backend(SimpleNamespace(reset_rows=lambda *a: (calls.append(a[2]), hip().reset_rows(*a))) if takes else SimpleNamespace())
    try:
        pool.reset_state([3, 1])
    finally:
        ops.set_backend(None)
    assert calls == ([[3, 1]] if takes else [])
    assert torch.equal(pool.states[0], want[0]) and torch.equal(pool.states[2], want[2])
