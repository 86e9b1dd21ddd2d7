"""Sixteen tokens of a recurrence with decays at a time, against the walk token by token in 64 bits and against the walk's own kernel.
Tolerance: a chunk's sums have at most 128 + 16 + 16 terms and its decays one rounding each, like the walk's; both are held to the
2e-5 that the walk's tests have, which covers their largest elements' share of the norm."""
import pytest
import torch

import kernel_twins as twin
from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip

pytestmark = pytest.mark.gpu
RULES = ["bonus", "delta", "gated", "delta_head"]


def _case(rule, lens, H, G, N, P, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T, wide = sum(lens), H if rule == "delta_head" else H * N
    rows = rnd(T, 2 * G * N + H * P + wide + H + 5).to(torch.bfloat16)           # views of one row, at odd places
    cut = (1, G * N, G * N, H * P, wide, H, 4)
    _, q, k, v, raw, beta, _ = rows.split(cut, 1)
    kw = dict(base=rnd(wide) - 1)
    kw.update(dict(bonus=rnd(wide)) if rule == "bonus" else dict(rate=rnd(H).abs() + 0.1))
    if rule.startswith("delta"):
        kw.update(unit_eps=1e-6, q_scale=N ** -0.5, beta=beta)
    return (q, k, v, raw), kw, rnd(len(lens) + 2, 3 + H * N * P)


def _run(backend, args, kw, state, lens, shape, rule):
    where = state.device
    cu = torch.tensor([0] + lens, device=where).cumsum(0).int()
    slots = torch.arange(len(lens), device=where).flip(0).int() + 1
    return backend.decay_rows_recurrence(*args, state[:, 3:], slots, cu, lens, *shape, rule, **kw)


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("lens,H,G,N,P", [([1, 15, 16, 17], 2, 1, 20, 12), ([64, 0, 63, 3], 3, 3, 64, 37), ([130, 2, 80], 2, 2, 128, 64),
                                          ([97, 16], 1, 1, 33, 130), ([5], 2, 1, 128, 1), ([48] * 70, 1, 1, 16, 8)])
def test_chunks_against_the_walk(monkeypatch, rule, lens, H, G, N, P):
    """Chunks that end early, requests without tokens, more requests than a wave looks through at once, rows and columns that are no
    whole tiles, heads that share keys, rows of odd strides and addresses; states of requests that are not in the step stay."""
    if rule != "delta" and rule != "delta_head":
        G = H
    args, kw, start = _case(rule, lens, H, G, N, P, H * N + P)
    monkeypatch.setattr(ops, "DECAY_CHUNKS_MIN_TOKENS", 1)
    state = start.clone()
    y = _run(hip(), args, kw, state, lens, (H, G, N, P), rule)
    cpu = lambda t: t.cpu() if torch.is_tensor(t) else t
    want = start.cpu().clone()
    ref = _run(twin, [t.cpu() for t in args], {n: cpu(t) for n, t in kw.items()}, want, lens, (H, G, N, P), rule)
    close(y, ref, 2e-5)
    close(state, want, 2e-5)
    assert torch.equal(state[:, :3], start[:, :3]) and torch.equal(state[0], start[0]) and torch.equal(state[-1], start[-1])
    monkeypatch.setattr(ops, "DECAY_CHUNKS_MIN_TOKENS", 1 << 30)
    walked = start.clone()
    close(_run(hip(), args, kw, walked, lens, (H, G, N, P), rule), y, 2e-6 * 16)
    monkeypatch.setattr(ops, "DECAY_CHUNKS_MIN_TOKENS", 1)
    for i, n in enumerate(lens[:4]):             # a request beside others has the bits that it has alone
        if n:
            lo, alone = sum(lens[:i]), start.clone()
            one = [t[lo:lo + n] for t in args]
            more = {m: (t[lo:lo + n] if m == "beta" else t) for m, t in kw.items()}
            cu, slot = torch.tensor([0, n], device=DEV).int(), torch.tensor([len(lens) - i], device=DEV).int()
            assert torch.equal(hip().decay_rows_recurrence(*one, alone[:, 3:], slot, cu, [n], H, G, N, P, rule, **more), y[lo:lo + n])
            assert torch.equal(alone[len(lens) - i], state[len(lens) - i])


@pytest.mark.parametrize("rule", RULES)
def test_what_is_not_a_number_stays_behind_its_token(monkeypatch, rule):
    """A value, key or query that is not finite reaches its own token and later ones, as token by token, and no token in front of it,
    in its chunk or another; a value only its own column."""
    lens, H, N, P = [40], 2, 64, 20
    args, kw, start = _case(rule, lens, H, H, N, P, 9)
    monkeypatch.setattr(ops, "DECAY_CHUNKS_MIN_TOKENS", 1)
    want = _run(hip(), args, kw, start.clone(), lens, (H, H, N, P), rule)
    for which, at in ((2, P + 3), (1, N + 5), (0, N + 7), (3, 1 if rule == "delta_head" else N + 2)):
        for bad in (float("inf"), float("nan")):
            odd = [t.clone() for t in args]
            odd[which][21, at] = bad
            y = _run(hip(), odd, kw, start.clone(), lens, (H, H, N, P), rule).view(40, H, P)
            assert torch.equal(y[:21], want.view(40, H, P)[:21]) and torch.equal(y[:, 0], want.view(40, H, P)[:, 0])
            if which == 2:
                assert not torch.isfinite(y[21 if rule != "bonus" else 22:, 1, 3]).any()
                rest = [c for c in range(P) if c != 3]
                assert torch.equal(y[:, 1, rest], want.view(40, H, P)[:, 1, rest])


def test_decays_that_vanish(monkeypatch):
    """Decays of exactly zero and of exactly one, by rows: nothing is divided by them."""
    monkeypatch.setattr(ops, "DECAY_CHUNKS_MIN_TOKENS", 1)
    lens, H, N, P = [50], 1, 32, 16
    args, kw, start = _case("bonus", lens, H, H, N, P, 4)
    raw = torch.zeros_like(args[3])
    raw[:, ::3], raw[::4, 1::3] = 80.0, -200.0           # exp(-exp(80)) = 0, exp(-exp(-200)) = 1
    state, want = start.clone(), start.cpu().clone()
    y = _run(hip(), (*args[:3], raw), kw, state, lens, (H, H, N, P), "bonus")
    ref = _run(twin, (*(t.cpu() for t in args[:3]), raw.cpu()), {n: t.cpu() for n, t in kw.items()}, want, lens, (H, H, N, P), "bonus")
    close(y, ref, 2e-5)
    close(state, want, 2e-5)
