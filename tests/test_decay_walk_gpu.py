"""The walk over shaped tokens in batches of eight: a token's results are the same bits wherever it stands in a batch, in a
whole batch or in one that ends early, and the state row is the same too."""
import pytest
import torch

from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip
import kernel_twins as twin

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("groups", [4, 16])
@pytest.mark.parametrize("rule", ["bonus", "delta", "gated", "delta_head"])
@pytest.mark.parametrize("H,N,P,dtype", [(2, 20, 12, torch.float32), (3, 64, 64, torch.bfloat16), (2, 128, 37, torch.bfloat16), (1, 256, 5, torch.float32)])
def test_places_in_a_batch(monkeypatch, H, N, P, dtype, rule, groups):
    monkeypatch.setattr(ops, "decay_row_groups", lambda *a: (groups, True))
    g = torch.Generator(device=DEV).manual_seed(N + P)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, wide = 41, H if rule == "delta_head" else H * N
    q, k, v, raw, beta = (rnd(T, n + 3)[:, 1:1 + n].to(dtype) for n in (H * N, H * N, H * P, wide, H))
    kw = dict(base=rnd(wide) - 1)
    kw.update(dict(bonus=rnd(wide)) if rule == "bonus" else dict(rate=rnd(H).abs() + 0.1))
    if rule.startswith("delta"):
        kw.update(unit_eps=1e-6, q_scale=N ** -0.5)
    start = rnd(2, H * N * P)
    slot = torch.tensor([1], dtype=torch.int32, device=DEV)

    def run(lo, n, state):
        more = dict(kw, beta=beta[lo:lo + n]) if rule.startswith("delta") else kw
        return hip().decay_rows_recurrence(q[lo:lo + n], k[lo:lo + n], v[lo:lo + n], raw[lo:lo + n], state, slot,
                                           torch.tensor([0, n], dtype=torch.int32, device=DEV), [n], H, H, N, P, rule, **more)

    whole = start.clone()
    y = run(0, T, whole)
    cpu = lambda t: t.cpu() if torch.is_tensor(t) else t
    want = start.cpu().clone()
    close(y, twin.decay_rows_recurrence(*(t.cpu() for t in (q, k, v, raw)), want, slot.cpu(), torch.tensor([0, T]), [T], H, H, N, P, rule,
                                        **{n: cpu(t) for n, t in dict(kw, **(dict(beta=beta) if rule.startswith("delta") else {})).items()}), 2e-5)
    close(whole, want, 2e-5)
    for cuts in ((1, 40), (3, 38), (8, 33), (9, 8, 24), (7, 1, 33)):
        state, lo, parts = start.clone(), 0, []
        for n in cuts:
            parts.append(run(lo, n, state))
            lo += n
        assert torch.equal(torch.cat(parts), y) and torch.equal(state, whole)


@pytest.mark.parametrize("rule", ["bonus", "delta", "gated", "delta_head"])
@pytest.mark.parametrize("H,N,P,count", [(2, 64, 64, 3), (12, 64, 64, 4), (13, 64, 64, 4), (3, 128, 128, 4), (2, 128, 128, 4), (2, 128, 132, 4), (4, 128, 132, 3), (2, 20, 30, 2), (1, 256, 7, 3)])
def test_waves_that_share_a_walk(H, N, P, count, rule):
    """Several requests at once, at the numbers of workgroups up to which four waves share a column group's walk and just
    beyond: batches of 16 and of 8 that end early, a request without tokens, the same bits as each request alone."""
    g = torch.Generator(device=DEV).manual_seed(N + P + H)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    lens = [33, 0, 16, 47][:count]
    T, wide = sum(lens), H if rule == "delta_head" else H * N
    q, k, v, raw, beta = (rnd(T, n).to(torch.bfloat16) for n in (H * N, H * N, H * P, wide, H))
    kw = dict(base=rnd(wide) - 1)
    kw.update(dict(bonus=rnd(wide)) if rule == "bonus" else dict(rate=rnd(H).abs() + 0.1))
    if rule.startswith("delta"):
        kw.update(unit_eps=1e-6, q_scale=N ** -0.5)
    start = rnd(count, H * N * P)

    def run(lo, hi, which, lens, state):
        more = dict(kw, beta=beta[lo:hi]) if rule.startswith("delta") else kw
        cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV)
        return hip().decay_rows_recurrence(q[lo:hi], k[lo:hi], v[lo:hi], raw[lo:hi], state, torch.tensor(which, dtype=torch.int32, device=DEV), cu,
                                           lens, H, H, N, P, rule, **more)

    together = start.clone()
    y = run(0, T, list(range(count)), lens, together)
    cpu = lambda t: t.cpu() if torch.is_tensor(t) else t
    want = start.cpu().clone()
    close(y, twin.decay_rows_recurrence(*(t.cpu() for t in (q, k, v, raw)), want, torch.arange(count), torch.tensor([0] + lens).cumsum(0), lens, H, H, N, P, rule,
                                        **{n: cpu(t) for n, t in dict(kw, **(dict(beta=beta) if rule.startswith("delta") else {})).items()}), 2e-5)
    close(together, want, 2e-5)
    lo = 0
    for i, n in enumerate(lens):
        if n:
            state = start.clone()
            assert torch.equal(run(lo, lo + n, [i], [n], state), y[lo:lo + n]) and torch.equal(state[i], together[i])
        lo += n


@pytest.mark.parametrize("T", [15, 16, 31, 32, 63, 64, 97, 128])
@pytest.mark.parametrize("N,rule", [(32, "bonus"), (64, "delta"), (64, "gated"), (128, "delta"), (128, "delta_head"), (100, "bonus")])
def test_whole_batches_of_the_shared_walk(monkeypatch, N, rule, T):
    """Requests that end with a batch of the four waves, just before or behind one, the one behind them read ahead: the same bits as in
    pieces of seven tokens, none of which holds a whole batch, and as beside so many requests that one wave walks alone."""
    monkeypatch.setattr(ops, "decay_row_groups", lambda *a: (16, True))
    g = torch.Generator(device=DEV).manual_seed(N + T)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    H, P, crowd = 2, 64, 26
    wide = H if rule == "delta_head" else H * N
    q, k, v, raw, beta = (rnd(T, n).to(torch.bfloat16) for n in (H * N, H * N, H * P, wide, H))
    kw = dict(base=rnd(wide) - 1)
    kw.update(dict(bonus=rnd(wide)) if rule == "bonus" else dict(rate=rnd(H).abs() + 0.1))
    if rule.startswith("delta"):
        kw.update(unit_eps=1e-6, q_scale=N ** -0.5)
    start = rnd(1, H * N * P)

    def run(rows, state):
        lens = [r.shape[0] for r in rows]
        at = torch.cat(rows)
        more = dict(kw, beta=beta[at]) if rule.startswith("delta") else kw
        return hip().decay_rows_recurrence(q[at], k[at], v[at], raw[at], state, torch.arange(len(rows), dtype=torch.int32, device=DEV),
                                           torch.tensor([0] + lens, dtype=torch.int32, device=DEV).cumsum(0, dtype=torch.int32), lens, H, H, N, P, rule, **more)

    every = torch.arange(T, device=DEV)
    whole, pieces, many = start.clone(), start.clone(), start.repeat(crowd, 1)
    y = run([every], whole)
    assert torch.equal(torch.cat([run([every[lo:lo + 7]], pieces) for lo in range(0, T, 7)]), y) and torch.equal(pieces, whole)
    assert torch.equal(run([every] * crowd, many).view(crowd, T, H * P), y.expand(crowd, T, H * P)) and torch.equal(many, whole.expand(crowd, -1))


@pytest.mark.parametrize("rule", ["bonus", "delta_head"])
@pytest.mark.parametrize("n", [63, 64, 130])
def test_shared_walk_of_128_rows_by_the_requests_length(n, rule):
    """Between 256 and 512 workgroups requests of 64 tokens and more on average share their columns' walk, shorter ones do not: the same bits as each
    request alone, whose 128 workgroups always do, remainders of a batch included."""
    g = torch.Generator(device=DEV).manual_seed(n)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    H, N, P, count = 8, 128, 64, 3
    T, wide = n * count, H if rule == "delta_head" else H * N
    q, k, v, raw, beta = (rnd(T, m).to(torch.bfloat16) for m in (H * N, H * N, H * P, wide, H))
    kw = dict(base=rnd(wide) - 1)
    kw.update(dict(bonus=rnd(wide)) if rule == "bonus" else dict(rate=rnd(H).abs() + 0.1, unit_eps=1e-6, q_scale=N ** -0.5))
    start = rnd(count, H * N * P)

    def run(lo, hi, which, state):
        lens = [n] * len(which)
        more = dict(kw, beta=beta[lo:hi]) if rule == "delta_head" else kw
        cu = torch.arange(len(which) + 1, dtype=torch.int32, device=DEV) * n
        return hip().decay_rows_recurrence(q[lo:hi], k[lo:hi], v[lo:hi], raw[lo:hi], state, torch.tensor(which, dtype=torch.int32, device=DEV), cu,
                                           lens, H, H, N, P, rule, **more)

    together = start.clone()
    y = run(0, T, [0, 1, 2], together)
    for i in range(count):
        state = start.clone()
        assert torch.equal(run(i * n, i * n + n, [i], state), y[i * n:i * n + n]) and torch.equal(state[i], together[i])
