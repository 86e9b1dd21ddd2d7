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
