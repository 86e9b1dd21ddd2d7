"""A graph captured with one step and replayed with others of its layout, whose tokens are shared out otherwise among the requests, on
models that keep state: against the same steps launched one by one. A token that no launch covers leaves what lay in the graph's memory in
its place and in its request's state, which moves the logits by their own size; the tolerances are those of the designs' own tests."""
import pytest
import torch

import helpers
import sigosun_cases
import tavevik_cases
import test_sigosun_gpu
import test_tavevik_gpu
import test_vefulix_gpu
import vefulix_cases
from mini_engine_amd.cache.manager import CacheManager
from mini_engine_amd.engine.runner import ModelRunner, StepEntry
from mini_engine_amd.weights.loader import load_model

pytestmark = pytest.mark.gpu
DEV = "cuda"
LONGEST = 4096
# every step of a group has the layout of the first one, with which it is captured
GROUPS = [([70], [120], [64]), ([1, 1, 40, 30], [1, 1, 5, 65]), ([300, 340], [500, 140]), ([1030, 1018], [1900, 148], [3, 2045])]
DESIGNS = {"sigosun": (sigosun_cases, test_sigosun_gpu, "mix"), "tavevik": (tavevik_cases, test_tavevik_gpu, "pair"),
           "vefulix": (vefulix_cases, test_vefulix_gpu, "mix-all")}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["float32", "bfloat16"])
@pytest.mark.parametrize("design", sorted(DESIGNS))
def test_replays_of_other_divisions(tmp_path, design, dtype):
    cases, tests, name = DESIGNS[design]
    tol, vocab, page = tests.TOL[dtype], cases.CONFIGS[name]["vocab"], cases.PAGE[name]
    model = load_model(cases.make_folder(name, str(tmp_path)), DEV, dtype, LONGEST)

    def made(**options):
        manager = CacheManager(2 * LONGEST // page, page, ModelRunner.windows_of(model), num_state_slots=6, enable_prefix_caching=False)
        return ModelRunner(model, manager, dtype, DEV, LONGEST, poison_cache=True, **options), manager

    graphs, eager = made(use_graphs=True, mixed_graphs_after=1), made()
    seed = 0
    for group in GROUPS:
        replays = graphs[0].mixed_graphs.replays
        for lens in (group[0],) + group:                   # seen once, then captured, then replayed
            seed += 1
            ids = [helpers.random_ids(n + 5, vocab, 100 * seed + j) for j, n in enumerate(lens)]
            out = []
            for runner, manager in (graphs, eager):
                def step(parts, want=True):
                    for r, at, n in parts:
                        assert manager.allocate(r, at, n)
                    z = runner.step([StepEntry(r, ids[r][at:at + n], at, [n - 1] if want else []) for r, at, n in parts])
                    return z.float().cpu() if want else None
                singles = [r for r, n in enumerate(lens) if n == 1]
                for r in singles:                          # those that decode hold tokens already
                    step([(r, 0, 4)], want=False)
                first = [(r, 4 if n == 1 else 0, n) for r, n in enumerate(lens)]
                out.append((step(first), step([(r, at + n, 1) for r, at, n in first])))        # the state that the step left behind
                for r in range(len(lens)):
                    manager.free(r)
            for got, want in zip(*out):
                assert torch.isfinite(got).all()
                err = float((got - want).abs().max() / want.abs().max())
                assert err <= tol, f"{lens} behind a capture of {group[0]}: {err:.3g} > {tol:g}"
        assert graphs[0].mixed_graphs.replays - replays >= len(group)
