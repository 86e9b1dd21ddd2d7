"""Kernels of decode steps that ask for a row's or a state's values at once, around the sizes where their forms change."""
import pytest
import torch

import kernel_twins as twin
from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip

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
    scores = torch.softmax(x.cpu() @ router.cpu().t(), -1) if scoring == "softmax" else torch.sigmoid(x.cpu() @ router.cpu().t())
    gap = scores.unique(dim=-1) if T == 1 else None            # different logits whose scores round alike may go either way
    same = (ids.cpu() == want_ids).all(-1)
    assert same.float().mean() >= (1.0 if scoring == "chosen" or gap is not None else 0.9)
    close(weights.cpu()[same], want_w[same], 2e-6)             # a softmax of 32-bit exponentials
    up, down = torch.randn(E, 8, 24, device=DEV, generator=g), torch.randn(E, 16, 8, device=DEV, generator=g)
    got = hip().route_and_run_experts(x.to(torch.bfloat16), router, top, groups, keep, up.to(torch.bfloat16), down.to(torch.bfloat16), rule=rule, gated=False)
    want = twin.routed_experts(x.cpu().to(torch.bfloat16), ids.cpu(), weights.cpu(), up.cpu().to(torch.bfloat16), down.cpu().to(torch.bfloat16), gated=False)
    close(got.sum(0), want.sum(0), 3e-2)
