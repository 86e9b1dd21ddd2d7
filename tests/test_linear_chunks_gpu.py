"""Sixteen tokens of a recurrence with one decay per head at a time, against the token-by-token twin. Tolerance: 2e-5 as for the other
forms of that recurrence (the inputs are exact in both, up to 128 + 16 float32 sums a chunk in another order)."""
import pytest
import torch

import kernel_twins as twin
from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip

pytestmark = pytest.mark.gpu


def _case(lens, H, G, N, P, selective):
    g = torch.Generator(device=DEV).manual_seed(H * N + P)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    T = sum(lens)
    _, q, k, v, dt, _ = rnd(T, 2 * G * N + H * P + H + 4).to(torch.bfloat16).split((1, G * N, G * N, H * P, H, 3), 1)       # rows at odd places
    kw = (dict(dt=dt, dt_bias=rnd(H) - 2, rate=rnd(H).abs() * 4 + 0.2, skip=rnd(H)) if selective else
          dict(decay=torch.tensor([0.5, 0.9, 0.99, 0.999, -0.8, 0.0, 1.0, 0.9999], device=DEV)[:H].contiguous(), silu=True))
    return (q, k, v), kw, rnd(len(lens) + 2, 3 + H * N * P)


def _run(backend, args, kw, state, lens, shape):
    cu = torch.tensor([0] + lens, device=state.device).cumsum(0).int()
    slots = torch.arange(len(lens), device=state.device).flip(0).int() + 1
    y = backend.linear_recurrence(*args, state[:, 3:], slots, cu, lens, *shape, **kw)
    return y.sum(0) if y.dim() == 3 else y


@pytest.mark.parametrize("selective", [False, True])
@pytest.mark.parametrize("lens,H,G,N,P", [([1, 15, 16, 17], 6, 3, 20, 12), ([64, 0, 63, 3], 4, 1, 64, 37), ([130, 2, 80], 8, 8, 128, 64),
                                          ([97, 16], 1, 1, 33, 130), ([5], 2, 2, 128, 1), ([48, 1] * 35, 2, 1, 16, 8)])
def test_chunks_against_the_twin(monkeypatch, selective, lens, H, G, N, P):
    """Chunks that end early, requests without tokens, more requests than a wave looks through at once, rows and columns that are no
    whole tiles, shared keys; decays that vanish, stay or change the sign; states of requests that are not in the step stay."""
    monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: True)
    args, kw, start = _case(lens, H, G, N, P, selective)
    state, want = start.clone(), start.cpu().clone()
    y = _run(hip(), args, kw, state, lens, (H, G, N, P))
    cpu = lambda t: t.cpu() if torch.is_tensor(t) else t
    close(y, _run(twin, [t.cpu() for t in args], {n: cpu(t) for n, t in kw.items()}, want, lens, (H, G, N, P)), 2e-5)
    close(state, want, 2e-5)
    assert torch.equal(state[:, :3], start[:, :3]) and torch.equal(state[0], start[0]) and torch.equal(state[-1], start[-1])
    monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: False)
    other = start.clone()
    close(_run(hip(), args, kw, other, lens, (H, G, N, P)), y, 2e-5)
    close(other, state, 2e-5)


@pytest.mark.parametrize("selective", [False, True])
@pytest.mark.parametrize("lens,H,G,N,P", [([130, 2, 80], 8, 8, 128, 64), ([1, 15, 16, 17, 0, 200], 6, 3, 20, 12), ([400], 4, 1, 64, 37), ([48, 1] * 35, 2, 1, 16, 8)])
def test_chunks_in_parts_give_the_same_bits(monkeypatch, selective, lens, H, G, N, P):
    """Scratch for some places only, down to one: parts that end inside a request, between two and in places that nobody has."""
    monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: True)
    args, kw, start = _case(lens, H, G, N, P, selective)
    want_state = start.clone()
    want = _run(hip(), args, kw, want_state, lens, (H, G, N, P))
    place = G * (32 * (32 if N <= 32 else 64 if N <= 64 else 128) + 256) + H * (304 + 256 * -(-P // 16))
    for places in (1, 2, 3, 4, 7, 11, sum(lens) // 16 + len(lens) - 1):
        monkeypatch.setattr(ops, "LINEAR_CHUNKS_FLOATS", places * place + 5)
        state = start.clone()
        assert torch.equal(_run(hip(), args, kw, state, lens, (H, G, N, P)), want) and torch.equal(state, want_state)


@pytest.mark.parametrize("selective", [False, True])
def test_what_is_not_a_number_stays_behind_its_token(monkeypatch, selective):
    """A value, key or query that is not finite reaches its own token and later ones and no token in front of it, in its chunk or
    another; a value only its own column, a head's step size only its head."""
    monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: True)
    lens, H, N, P = [40], 2, 64, 20
    args, kw, start = _case(lens, H, H, N, P, selective)
    want = _run(hip(), args, kw, start.clone(), lens, (H, H, N, P)).view(40, H, P)
    for which, at in ((2, P + 3), (1, N + 5), (0, N + 7)) + (((3, 1),) if selective else ()):
        for bad in (float("inf"), float("nan")):
            odd = [t.clone() for t in args]
            more = dict(kw, dt=kw["dt"].clone()) if selective else kw
            (odd + [more.get("dt")])[which][21, at] = bad
            y = _run(hip(), odd, more, start.clone(), lens, (H, H, N, P)).view(40, H, P)
            assert torch.equal(y[:21], want[:21]) and torch.equal(y[:, 0], want[:, 0])
            if which == 2:
                assert not torch.isfinite(y[21:, 1, 3]).any()
                rest = [c for c in range(P) if c != 3]
                assert torch.equal(y[:, 1, rest], want[:, 1, rest])


def test_rule():
    """Where the line lies, at the sizes that it was measured at."""
    take = lambda lens, H=16, P=128, N=128, dtype=torch.bfloat16: ops.linear_chunks_take(dtype, H, N, P, lens)
    assert take([16]) and take([16] * 8) and not take([15]) and not take([16] * 8, H=32) and take([64] * 8, H=32)
    assert not take([64] + [1] * 300) and take([300] + [1] * 200) and take([128] * 64)
    assert not take([300], N=130) and not take([300], dtype=torch.float32)


@pytest.mark.parametrize("pattern", [[300], [15, 1, 16, 17], [100, 7, 63, 64], [1, 130, 40], [8, 31, 33, 200]], ids=str)
def test_cuts_and_neighbours_on_both_sides_of_the_rule(tmp_path, monkeypatch, pattern):
    """Portions and requests beside them decide which form a step takes. However a prompt is cut, its logits are as near to the plain
    evaluation as with the other form alone: both round to bfloat16 in the same places, so their errors are draws of one size, and the
    largest over a prompt's logits differs by less than half."""
    import helpers
    import sigosun_cases as S
    from mini_engine_amd.cache.manager import CacheManager
    from mini_engine_amd.engine.runner import ModelRunner
    from mini_engine_amd.weights.loader import load_model

    folder = S.make_folder("real", str(tmp_path))
    model = load_model(folder, DEV, torch.bfloat16, 512)
    ids = {r: helpers.random_ids(n, S.CONFIGS["real"]["vocab"], n) for r, n in (("long", 300), ("short", 70), ("last", 180))}
    take, took, errors = ops.linear_chunks_take, [], []
    for chunks in (True, False):
        monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: chunks and (took.append(take(*a)) or took[-1]))
        manager = CacheManager(64, 16, ModelRunner.windows_of(model), num_state_slots=4, enable_prefix_caching=False)
        driver = helpers.Driver(ModelRunner(model, manager, torch.bfloat16, DEV, 512), manager)
        for step in helpers.cuts_schedule({r: len(t) for r, t in ids.items()}, pattern):
            driver.step({r: ids[r][a:b] for r, (a, b) in step.items()})
        got = {r: driver.result(r).double() for r in ids}
        errors.append({r: max(float((got[r] - w).norm() / w.norm()) for w in [S.plain_logits(folder, t).double()]) for r, t in ids.items()})
    assert True in took
    for r in ids:
        assert errors[0][r] <= 1.5 * errors[1][r], errors
