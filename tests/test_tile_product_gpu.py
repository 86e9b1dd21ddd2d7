"""The product of many rows whose tiles go through LDS in quarters of a step (csrc/gemm_tile.hip): every tile at the edges of
its rows, features and steps of K, against float64."""
import pytest
import torch

from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, close, hip, twin

pytestmark = pytest.mark.gpu


def _operands(M, N, K, pad=0):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N + K)
    x = torch.randn(M, K + pad, device=DEV, generator=g).bfloat16()[:, :K]
    w = (torch.randn(N, K + pad, device=DEV, generator=g) * 0.05).bfloat16()[:, :K]
    return x, w


def _launch(x, w, y, slices, tile, gated=0, bias=None, limit=0.0, alpha=1.0):
    M, K = x.shape
    ops.core().call("me_gemm_tile_bf16", x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), y.shape[-1], ops._code(y.dtype),
                    slices, M, w.shape[0], K, gated, limit, alpha, ops._ptr(bias), *tile, ops._stream())


@pytest.mark.parametrize("tile", list(ops.TILE_COST), ids=lambda t: f"{t[0]}x{t[1]}")
def test_every_tile_at_its_edges(tile):
    """One row, one more and one fewer than a tile; features that end inside a tile; two steps of K (no step in between), three
    and many, rows of a longer stride; one result in both types, slices of K with a shorter last one, the gating."""
    rows, features = tile
    for M, N, K, pad in ((1, 8, 128, 0), (rows - 1, features, 192, 8), (rows + 1, features + 8, 256, 0), (2 * rows + 3, 2 * features - 16, 1088, 64),
                         (9 * rows + 5, features + 64, 320, 0)):
        x, w = _operands(M, N, K, pad)
        ref = x.double() @ w.double().t()
        y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        _launch(x, w, y, 1, tile)
        close(y, ref, 4e-3)                      # one rounding to bfloat16: 2^-9 of a value at most
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
        _launch(x, w, y, 1, tile)
        close(y, ref, 2e-5)
        for slices in (2, 3, 8):
            steps = K // 64
            if (slices - 1) * -(-steps // slices) <= steps - 2:
                y = torch.full((slices, M, N), float("nan"), dtype=torch.float32, device=DEV)
                _launch(x, w, y, slices, tile)
                close(y.sum(0), ref, 2e-5)
        if N % 16 == 0:
            y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
            _launch(x, w, y, 1, tile, 2)
            two = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
            _launch(x, w, two, 1, tile)
            assert torch.equal(y, hip().silu_and_mul(two))                     # rounded sums: the two kernels' bits
            _launch(x, w, y, 1, tile, 2, None, 1.5, 1.702)
            assert torch.equal(y, hip().glu_clamped(two, 1.5, 1.702))
            _launch(x, w, y, 1, tile, 1)
            close(y, torch.nn.functional.silu(ref[:, :N // 2]) * ref[:, N // 2:], 6e-3)
            bias = torch.randn(N, device=DEV)
            _launch(x, w, y, 1, tile, 2, bias)
            assert torch.equal(y, hip().silu_and_mul(two, bias=bias))
            _launch(x, w, y, 1, tile, 1, bias)
            b = ref + bias.double()
            close(y, torch.nn.functional.silu(b[:, :N // 2]) * b[:, N // 2:], 6e-3)
            _launch(x, w, y, 1, tile, 1, None, 1.5, 1.702)
            gate, up = ref[:, :N // 2].clamp(max=1.5), ref[:, N // 2:].clamp(-1.5, 1.5)
            close(y, gate * torch.sigmoid(1.702 * gate) * (up + 1), 6e-3)


def test_a_row_of_infinities_and_not_a_numbers_stays_in_its_row():
    x, w = _operands(300, 520, 256)
    want = hip().linear(x, w)
    x[7, 3], x[299, 0] = float("inf"), float("nan")
    got = hip().linear(x, w)
    keep = [i for i in range(300) if i not in (7, 299)]
    assert torch.equal(got[keep], want[keep]) and bool(torch.isnan(got[299]).all()) and not bool(torch.isfinite(got[7]).any())


class _Recorded:
    """A library that notes the names of the entry points asked of it."""

    def __init__(self, lib, names):
        self._lib, self._names = lib, names
        self.fns = {name: self._noting(name, fn) for name, fn in lib.fns.items()}

    def _noting(self, name, fn):
        def run(*args):
            self._names.append(name)
            return fn(*args)
        return run

    def call(self, name, *args):
        self._names.append(name)
        return self._lib.call(name, *args)

    def __getattr__(self, name):
        return getattr(self._lib, name)


def _products(monkeypatch, run) -> tuple:
    """The result of `run`, and the products and gating kernels that it launched."""
    names, lib = [], ops.core()
    with monkeypatch.context() as m:
        m.setattr(ops, "core", lambda: _Recorded(lib, names))
        y = run()
    return y, [n[3:] for n in names]


TILE, MID, LIBRARY, GATE = "gemm_tile_bf16", "gemm_mid_bf16", "gemm_library_bf16", "gate_mul"


@pytest.mark.parametrize("M,N,K,route", [(300, 1024, 1024, TILE), (513, 1024, 3072, LIBRARY), (257, 6144, 1024, TILE), (200, 6144, 1024, TILE), (128, 6144, 1024, MID),
                                         (1100, 4096, 2048, LIBRARY), (2048, 4096, 2048, TILE), (2048, 6144, 4096, TILE), (1536, 4096, 4096, LIBRARY), (2048, 24576, 4096, TILE), (300, 1028, 1024, LIBRARY)])
def test_each_product_runs_where_the_rules_send_it(monkeypatch, M, N, K, route):
    x, w = _operands(M, N, K)
    y, ran = _products(monkeypatch, lambda: hip().linear(x, w))
    assert ran == [route]
    close(y, x.double() @ w.double().t(), 4e-3)


@pytest.mark.parametrize("M,N,K,slices,route", [(512, 1024, 3072, 4, TILE), (64, 1024, 3072, 8, MID), (33, 4096, 12288, 8, TILE), (256, 4096, 4096, 8, TILE), (300, 4096, 12288, 4, LIBRARY),
                                                (700, 5120, 8192, 2, LIBRARY), (200, 4100, 4096, 8, LIBRARY), (160, 5120, 25600, 8, LIBRARY)])
def test_each_product_in_slices_runs_where_the_rules_send_it(monkeypatch, M, N, K, slices, route):
    """Slices of K as float32 partial sums: crowded slices of the tiled kernel and few rows of the library's go to the tiles; what
    the tiles cannot take (4,100 features) or are slower for (a K beyond 16,384) stays."""
    x, w = _operands(M, N, K)
    y, ran = _products(monkeypatch, lambda: hip().linear(x, w, None, allow_partials=True))
    assert ran == [route] and y.shape == (slices, M, N) and y.dtype == torch.float32
    close(y.sum(0), x.double() @ w.double().t(), 2e-5)


@pytest.mark.parametrize("M,N,K,route", [(200, 6144, 1024, [TILE]), (512, 6144, 1024, [TILE]), (128, 6144, 1024, [MID]), (2048, 6144, 4096, [TILE]), (800, 24576, 4096, [LIBRARY, GATE]),
                                         (300, 2048, 200, [LIBRARY, GATE])])
@pytest.mark.parametrize("biased", [False, True])
def test_each_gated_product_runs_where_the_rules_send_it(monkeypatch, M, N, K, route, biased):
    """A packed gate/up map as the feed-forward calls it: one launch, or the product and the gating kernel."""
    from mini_engine_amd.parts.linear import Linear
    x, w = _operands(M, N, K)
    part = Linear(K, N)
    part.set_param("weight", w)
    bias = torch.randn(N, device=DEV) if biased else None
    y, ran = _products(monkeypatch, lambda: part.forward(x, gated=True, bias=bias))
    assert ran == route
    sums = x.double() @ w.double().t()
    sums = sums + bias.double() if biased else sums
    close(y, torch.nn.functional.silu(sums[:, :N // 2]) * sums[:, N // 2:], 1.5e-2)


@pytest.mark.parametrize("M,N,K", [(300, 1024, 1024), (513, 1024, 3072), (257, 6144, 1024), (200, 6144, 1024), (1100, 4096, 2048), (2048, 6144, 4096)])
def test_what_the_rules_send_there(M, N, K):
    """`linear` and `gated_linear` through the dispatch, replayed from a graph with other rows between the replays."""
    x, w = _operands(M, N, K)
    assert ops.tile_fits(x, w)
    for _ in range(2):
        close(hip().linear(x, w), x.double() @ w.double().t(), 4e-3)
    assert ops.gated_linear_fuses(x, w)
    # sums rounded before the gating: 2^-9 each of gate (times up to 1 + gate in its silu), up and result
    close(hip().gated_linear(x, w), twin.gated_linear(x, w, compute_dtype=torch.float64), 1.5e-2)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        y = hip().linear(x, w)
    for _ in range(3):
        x.copy_(torch.randn(M, K, device=DEV))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, hip().linear(x, w))


@pytest.mark.parametrize("M,N,K", [(300, 1024, 1024), (257, 6144, 1024), (2048, 1024, 2048)])
def test_an_out_that_begins_anywhere(M, N, K):
    """`linear` writes into any contiguous `out`, also one that is not aligned to the 16 bytes that the kernel's stores want."""
    x, w = _operands(M, N, K)
    want = hip().linear(x, w)
    for shift in (1, 4, 8):
        room = torch.full((M * N + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
        y = hip().linear(x, w, out=room[shift:shift + M * N].view(M, N))
        close(y, x.double() @ w.double().t(), 4e-3)
        assert y.data_ptr() == room.data_ptr() + 2 * shift and bool((room[:shift] == 7).all()) and bool((room[shift + M * N:] == 7).all())
        assert shift % 8 or torch.equal(y, want)


def test_what_the_kernel_refuses():
    x, w = _operands(70, 64, 128)
    y = torch.empty(70, 64, dtype=torch.bfloat16, device=DEV)
    for args in ((x[:, :96], w[:, :96], y, 1, (64, 64)), (x, w, y, 1, (64, 96)), (x, w, y.float(), 2, (64, 64)), (x, w[:60], y[:, :60], 1, (64, 64))):
        with pytest.raises(ops.KernelError):
            _launch(*args)


def _rings(tile, M, N, steps, slices=1, gated=False):
    tiles = -(-M // tile[0]) * (-(-(N // 2) // (tile[1] // 2)) if gated else -(-N // tile[1]))
    return bool(ops.core().fns["me_gemm_tile_rings"](*tile, tiles * slices, -(-steps // slices)))


@pytest.mark.parametrize("tile", [(64, 64), (64, 128), (128, 64), (128, 128)], ids=lambda t: f"{t[0]}x{t[1]}")
@pytest.mark.parametrize("extra", [-1, 0, 1, 3])
def test_tiles_in_one_round_go_round_the_ring(tile, extra):
    """Launches of one workgroup to a compute unit walk K through a ring of stages: from its fewest steps on and with one fewer, where they do not,
    in slices of K with a shorter last one, with an odd count and a row, a feature piece and a stride beside the tile's, every kind of
    output; bit for bit what a launch of many rounds gives the same rows."""
    rows, features = tile
    fewest = 32 if tile == (128, 128) else 16
    M, N = 2 * rows + 5, 3 * features - 16
    for slices in (1, 2):
        steps = slices * fewest + extra
        K = 64 * steps
        x, w = _operands(M, N, K, 8)
        many = torch.cat([x] * (1 + 300 * rows * features // (M * N)))                          # more than 256 tiles
        many = many[:many.shape[0] - many.shape[0] % rows + 3]
        assert _rings(tile, M, N, steps, slices) == (-(-steps // slices) >= fewest) and not _rings(tile, many.shape[0], N, steps, slices)
        ref = x.double() @ w.double().t()
        for dtype, gated in ((torch.bfloat16, 0), (torch.float32, 0), (torch.bfloat16, 1), (torch.bfloat16, 2)) if slices == 1 else ((torch.float32, 0),):
            assert _rings(tile, M, N, steps, slices, gated > 0) == (extra >= 0 or slices == 2)
            outs = []
            for rows_in in (x, many):
                shape = (rows_in.shape[0], N // 2 if gated else N)
                y = torch.full(shape if slices == 1 else (slices, *shape), float("nan"), dtype=dtype, device=DEV)
                _launch(rows_in, w, y, slices, tile, gated)
                outs.append(y[..., :M, :])
            assert torch.equal(*outs)
            if not gated:
                close(outs[0] if slices == 1 else outs[0].sum(0), ref, 4e-3 if dtype == torch.bfloat16 else 2e-5)


@pytest.mark.parametrize("M,N,K,route", [(65, 4096, 1024, TILE), (256, 4096, 1024, TILE), (700, 1024, 2048, TILE), (2048, 1024, 3072, TILE), (300, 1024, 3072, LIBRARY),
                                         (800, 4096, 4096, TILE), (640, 4096, 4096, LIBRARY), (256, 4096, 6144, LIBRARY), (90, 4100, 1024, MID)])
def test_each_product_of_one_round_runs_where_the_rule_sends_it(monkeypatch, M, N, K, route):
    x, w = _operands(M, N, K)
    y, ran = _products(monkeypatch, lambda: hip().linear(x, w))
    assert ran == [route] and (ops.ring_tile(M, N, K) is not None) == (route == TILE or N % 8 > 0)
    close(y, x.double() @ w.double().t(), 4e-3)


@pytest.mark.parametrize("M,N,K", [(100, 1024, 1024), (256, 2048, 1024), (128, 1024, 2048)])
def test_rows_that_overlap_are_taken_as_before(M, N, K):
    """One row that stands for all of them (an expanded view), and rows that begin inside the one before: the kernel for a few hundred
    rows reads them; the ring, which would refuse them, does not get them. For more rows both refuse."""
    x, w = _operands(M, N, K)
    base = torch.randn(8 * M + K, device=DEV).bfloat16()
    for rows in (x[:1].expand(M, K), base.as_strided((M, K), (8, 1))):
        assert ops.ring_tile(M, N, K) is not None
        close(hip().linear(rows, w), rows.double() @ w.double().t(), 4e-3)
    features = w[:1].expand(N, K)
    close(hip().linear(x, features), x.double() @ features.double().t(), 4e-3)
    with pytest.raises(ops.KernelError):
        hip().linear(x[:1].expand(600, K), w)
