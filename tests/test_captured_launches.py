"""What a captured step's launches are sized by: a graph is kept for a layout, and every step of that layout runs through it, however
its tokens are shared out among its requests. Recorded on the CPU, without a kernel."""
import random
from types import SimpleNamespace

import pytest
import torch

from mini_engine_amd.engine.graphs import MixedGraphs
from mini_engine_amd.engine.packing import exact_layout
from mini_engine_amd.kernels import ops

# what was captured first, what comes after: steps of one layout, some padded, some exact, some beside decoding requests
STEPS = [(319, [[70], [120], [64], [127]]), (319, [[1, 1, 40, 30], [1, 1, 5, 65], [1, 1, 2, 101]]), (2048, [[300, 340], [500, 140], [260, 400], [400, 240]]),
         (319, [[1030, 1018], [1900, 148], [2046, 2], [3, 2045]]), (2048, [[130], [250], [200]]), (2048, [[130, 128, 142], [2, 2, 396], [396, 2, 2]])]


class Recorder:
    """In the place of the kernels' library: takes down what is launched."""

    def __init__(self):
        self.calls = []

    def call(self, name, *args):
        self.calls.append((name, args))


def graphs(max_tokens):
    g = MixedGraphs.__new__(MixedGraphs)
    g.max_rows, g.capture, g.max_tokens, g.max_exact_tokens, g.max_branches_tokens = 64, False, max_tokens, 12 * max_tokens, 0
    g.runner = SimpleNamespace(vocab_size=100, device=torch.device("cpu"), manager=SimpleNamespace(page_size=16), max_positions=8192)
    return g


def layout_of(g, lens):
    tables = [[[0] * -(-n // 16) for n in lens]]
    return g.padded(exact_layout(lens, [0] * len(lens), tables, len(lens), lambda *a: False))


def captured(g, lens, monkeypatch):
    """The context with which the step's forward pass is captured."""
    seen = []
    g.runner.model = SimpleNamespace(forward=lambda tokens, step, *rest: (seen.append(step), (None, None))[1], logits=lambda *a, **k: torch.zeros(64, 4))
    g.runner.pool = SimpleNamespace(spare_page=lambda i: 500, spare_state_slot=63, views=None, states=None)
    g.runner.zero_fresh_state = lambda *a: None
    g.replays = 0
    layout = layout_of(g, lens)
    cap = SimpleNamespace(layout=layout, dev=torch.zeros(layout.segments()[1], dtype=torch.int32), events=[None], replays=0, graph=None,
                          staging=lambda: (0, torch.zeros(layout.segments()[1], dtype=torch.int32)))
    tables = [[list(range(-(-n // 16))) for n in lens]]
    g.run(cap, [[0] * n for n in lens], [0] * len(lens), tables, list(range(len(lens))), [], None)
    return seen[0]


def divisions(layout, given):
    """The given steps, as they are padded to the layout, and others of it."""
    out = [[1] * layout.decode_rows + [n for n in lens if n > 1] + [layout.prefill_tokens - sum(n for n in lens if n > 1)] * (
        layout.prefill_reqs - sum(1 for n in lens if n > 1)) for lens in given]
    rng = random.Random(layout.prefill_tokens)
    for _ in range(50):
        cuts = sorted(rng.sample(range(1, layout.prefill_tokens), layout.prefill_reqs - 1))
        out.append([1] * layout.decode_rows + [b - a for a, b in zip([0] + cuts, cuts + [layout.prefill_tokens])])
    return out


@pytest.mark.parametrize("limit,steps", STEPS, ids=[str(s[1][0]) for s in STEPS])
@pytest.mark.parametrize("dtype,gated", [(torch.bfloat16, False), (torch.float32, False), (torch.bfloat16, True)], ids=["bfloat16", "float32", "gates"])
def test_launches_cover_every_step_of_the_layout(monkeypatch, limit, steps, dtype, gated):
    """Captured with the first step, the convolution's and the recurrence's launches cover the tokens of every other one, and the
    scratch of the spans holds all of them."""
    core = Recorder()
    scratch = {}

    def scratch_of(n, device, use="decode"):
        scratch[use] = n
        return torch.zeros(1)

    monkeypatch.setattr(ops, "core", lambda: core)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_scratch", scratch_of)
    g = graphs(limit)
    layout = layout_of(g, steps[0])
    assert all(layout_of(g, lens) == layout for lens in steps)
    step = captured(g, steps[0], monkeypatch)
    assert list(step.q_lens) == divisions(layout, steps)[0]
    T, B, H, N, P, C, taps = layout.num_tokens, layout.num_seqs, 2, 160, 8, 8, 4          # 160 rows: in spans in both types
    rows = lambda w: torch.empty(T, w, dtype=dtype)
    state = torch.empty(64, H * N * P + H * N + H)
    slots, cu = torch.zeros(B, dtype=torch.int32), torch.zeros(B + 1, dtype=torch.int32)
    backend = ops.HipBackend()
    backend.causal_conv(rows(C), torch.empty(C, taps), None, torch.empty(64, C * (taps - 1)), slots, cu, step.q_lens)
    kw = dict(decay=torch.empty(H))
    if gated:
        kw = dict(gates=ops.SoftGates(rows(H), rows(H), torch.empty(H), torch.empty(H), 15.0, state[:, H * N * P + H * N:], slots),
                  key_state=state[:, H * N * P: H * N * P + H * N])
    backend.linear_recurrence(rows(H * N), rows(H * N), rows(H * P), state[:, :H * N * P], slots, cu, step.q_lens, H, H, N, P, **kw)
    called = {name: args for name, args in core.calls}
    conv, rec = called["me_causal_conv"], called["me_linear_recurrence"]
    max_tokens = conv[9]
    span, spans, places = rec[27:30]
    for lens in divisions(layout, steps):
        assert len(lens) == B and sum(lens) == T
        assert max_tokens >= max(lens)
        if spans > 1:
            assert span * spans >= max(lens)
            at = 0
            for b, n in enumerate(lens):
                assert at // span + b + -(-n // span) <= (places if b == B - 1 else (at + n) // span + b + 1)
                at += n
    if spans > 1:
        assert scratch["recurrence"] >= places * (H * N * P + H + (H * N if gated else 0))


def test_reach_of_captures_follows_the_branches_switch():
    """Twice as many tokens as otherwise, while a part that may put work on a further stream does."""
    g = graphs(319)
    g.max_exact_tokens, g.max_branches_tokens = 6 * 319, 12 * 319
    part = SimpleNamespace(captures_branches=True)
    g.branching = [SimpleNamespace(captures_branches=False), part]
    takes = lambda n: layout_of(g, [n]) is not None
    assert takes(1913) and takes(1914) and takes(3827) and not takes(3828)
    part.captures_branches = False
    assert takes(1913) and not takes(1914)


def test_the_run_in_front_of_a_capture_is_launched_as_the_capture_is(monkeypatch):
    """Both forward passes have the context that puts work on further streams; a step launched one by one has not."""
    import contextlib
    from mini_engine_amd.engine import graphs as module
    from mini_engine_amd.engine.packing import context_of
    g, seen = graphs(319), []
    monkeypatch.setattr(module.torch.cuda, "CUDAGraph", lambda: SimpleNamespace(replay=lambda: seen.append("replay")))
    monkeypatch.setattr(module.torch.cuda, "graph", lambda graph, pool: contextlib.nullcontext())
    monkeypatch.setattr(module.torch.cuda, "synchronize", lambda: None)
    layout = layout_of(g, [70])
    g.capture, g.pool = True, None
    g.runner.model = SimpleNamespace(forward=lambda tokens, step, *rest: (seen.append(step.captured), (None, None))[1], logits=lambda *a, **k: None)
    g.runner.pool = SimpleNamespace(views=None, states=[torch.zeros(2)])
    cap = SimpleNamespace(layout=layout, dev=torch.zeros(layout.segments()[1], dtype=torch.int32))
    module.capture_graph(g.runner, None, lambda: g._forward(cap, None, [70, 58], [0, 0]))
    assert seen == [True, True] and not context_of(layout, cap.dev).captured


def test_a_request_longer_than_the_layout_is_refused():
    """The host's check in front of a replay."""
    import numpy as np
    from dataclasses import replace
    from mini_engine_amd.engine import packing

    layout = exact_layout([5, 3], [0, 0], [[[0], [1]]], 0, lambda *a: False)
    assert layout.longest == 7 and exact_layout([1, 1], [0, 0], [[[0], [1]]], 0, lambda *a: False).longest == 1
    pack = lambda l: packing.pack_step(l, np.zeros(l.segments()[1], dtype=np.int32), [[0] * 5, [0] * 3], [0, 0], [[[0], [1]]], [0, 1], [], 16, [9], 9, 100)
    pack(layout)
    with pytest.raises(ValueError, match="longest"):
        pack(type("Short", (type(layout),), {"longest": 4})(**layout.__dict__))


def test_counts_of_a_step_launched_alone_are_its_own_measure():
    from mini_engine_amd.engine.context import TokenCounts
    assert ops.longest_request([3, 9, 1]) == 9 and ops.longest_request([]) == 0
    assert ops.longest_request(TokenCounts([3, 9])) == 9 and ops.longest_request(TokenCounts([3, 9], 11)) == 11


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_without_a_request_launch_nothing_for_any(monkeypatch, dtype):
    """Padding rows alone: the recurrence goes to the library with no requests, which then has nothing to do."""
    core = Recorder()
    monkeypatch.setattr(ops, "core", lambda: core)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    rows = lambda w: torch.empty(3, w, dtype=dtype)
    assert not ops.linear_chunks_take(dtype, 2, 16, 8, [])
    y = ops.HipBackend().linear_recurrence(rows(32), rows(32), rows(16), torch.empty(4, 256), torch.zeros(0, dtype=torch.int32),
                                           torch.zeros(1, dtype=torch.int32), [], 2, 2, 16, 8, decay=torch.empty(2))
    assert y.shape == (3, 16) and [(name, args[19]) for name, args in core.calls] == [("me_linear_recurrence", 0)]


@pytest.mark.parametrize("lens", [[16384], [2048] * 8, [30] * 600, [1] * 300 + [9000, 4000]])
@pytest.mark.parametrize("H,G,N,P", [(16, 16, 128, 128), (32, 1, 128, 64), (32, 32, 128, 128), (4000, 4000, 128, 128)])
def test_scratch_for_chunks_does_not_grow_with_the_step(monkeypatch, lens, H, G, N, P):
    """However many tokens a step has, the chunks' scratch is what the rule names, or one place where that is more."""
    core, asked = Recorder(), []
    monkeypatch.setattr(ops, "core", lambda: core)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_scratch", lambda n, device, use="decode": (asked.append((n, use)), torch.zeros(1))[1])
    T, B = sum(lens), len(lens)
    rows = lambda w: torch.empty(1, w, dtype=torch.bfloat16).expand(T, w)
    monkeypatch.setattr(ops, "linear_chunks_take", lambda *a: True)
    ops.HipBackend().linear_recurrence(rows(G * N), rows(G * N), rows(H * P), torch.empty(1, H * N * P), torch.zeros(B, dtype=torch.int32),
                                       torch.zeros(B + 1, dtype=torch.int32), lens, H, G, N, P, decay=torch.empty(H))
    (name, args), ((room, use),) = core.calls[-1], asked
    place = G * (32 * 128 + 256) + H * (304 + 256 * (P // 16))
    assert name == "me_linear_chunks" and use == "recurrence" and args[-2] == room
    assert place <= room <= max(ops.LINEAR_CHUNKS_FLOATS, place) and (room // place >= T // 16 + B or room >= ops.LINEAR_CHUNKS_FLOATS)
    assert ops.LINEAR_CHUNKS_FLOATS * 4 * 3 // 2 <= 192 << 20
