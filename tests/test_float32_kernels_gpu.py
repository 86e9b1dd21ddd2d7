"""The float32 path's product and attention at the edges of their tiles. Tolerances: a sum of n float32 products of
standard normals rounds by at most about 2^-24 sqrt(n) of its size per step, so 1e-6 for up to 3,000 terms added in four parts;
attention's scores pass an exponential, 1e-5 as everywhere."""
import pytest
import torch

import kernel_twins as twin
from mini_engine_amd.kernels import ops
from test_kernels_gpu import DEV, _attention_case, close, hip

pytestmark = pytest.mark.gpu
TILES = sorted(ops.F32_ROUND_US)


def _product(x, w, tile):
    y = torch.full((x.shape[0], w.shape[0]), float("nan"), device=DEV)
    ops.core().call("me_gemm_f32", x.data_ptr(), x.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), y.stride(0),
                    x.shape[0], w.shape[0], x.shape[1], *tile, ops._stream())
    return y


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (3, 17, 5), (16, 16, 16), (17, 130, 36), (33, 250, 130), (65, 64, 128), (70, 100, 1023),
                                   (600, 70, 260), (5, 2100, 2999)])
def test_product_tiles(M, N, K):
    """Every tile gives the same bits, for all rows together and for some alone; rows that are no whole 16-byte pieces, strides
    that are not K, an odd first address and an odd row length of the output give the same sums too."""
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    wide, ww = (torch.randn(n, K + 12, device=DEV, generator=g) for n in (M, N))
    x, w = wide[:, 4:4 + K], ww[:, 8:8 + K]
    ref = x.double() @ w.double().T
    first = _product(x, w, TILES[0])
    assert float((first.double() - ref).norm() / ref.norm()) < 1e-6
    for tile in TILES[1:]:
        assert torch.equal(_product(x, w, tile), first)
    assert torch.equal(hip().linear(x, w), first)
    some = x[M // 3:M // 3 + 2]
    assert torch.equal(hip().linear(some, w), first[M // 3:M // 3 + 2])
    odd = torch.empty(M * (K + 1) + 1, device=DEV)[1:].view(M, K + 1)[:, :K]
    odd.copy_(x)
    assert torch.equal(hip().linear(odd, w), first)


@pytest.mark.parametrize("M,N,K", [(2, 40, 32), (19, 33, 100), (50, 150, 516), (130, 64, 300)])
def test_product_by_parts(M, N, K):
    """Values are split into three parts exactly: weights that came as bfloat16, weights with all bits, and both in one launch,
    block by block along K, give every tile the same bits; against 64 bits the error is that of float32 sums. Infinities and what is
    not a number come out as plain float32 sums give them, and leave the other outputs their bits."""
    g = torch.Generator(device=DEV).manual_seed(M * K)
    x = torch.randn(M, K, device=DEV, generator=g) * torch.exp(4 * torch.randn(M, K, device=DEV, generator=g))
    full = torch.randn(N, K, device=DEV, generator=g)
    mixed = full.to(torch.bfloat16).float()
    mixed[N // 2:, K // 3:] = full[N // 2:, K // 3:]
    for w in (full, full.to(torch.bfloat16).float(), mixed):
        first = _product(x, w, TILES[0])
        assert all(torch.equal(_product(x, w, tile), first) for tile in TILES[1:])
        # of the sum of the products' sizes: 2^-24 for each sum that is rounded, twice for each of a chain's matrix instructions (its
        # own 32 terms, then with what was there; six for a block of 32, a chain has every fourth block) and two where chains
        # meet, and 3 x 2^-24 of a product for the three products of parts that are not formed
        bound = 2.0 ** -24 * (12 * -(-K // 128) + 2 + 3) * (x.double().abs() @ w.double().abs().T)
        assert bool(((first.double() - x.double() @ w.double().T).abs() <= bound).all())
    odd = x.clone()
    odd[0, 3], odd[M - 1, K - 1] = float("inf"), float("nan")
    w = full.clone()
    w[N - 1, 1], w[N // 2, 0] = -float("inf"), 3.4e38          # rounds up to an infinity in bfloat16
    for tile in TILES:
        got = _product(odd, w, tile)
        assert torch.isnan(got[M - 1]).all()
        assert torch.equal(got[0, : N // 2], torch.sign(w[: N // 2, 3]) * float("inf"))
        rows = slice(1, M - 1)
        assert torch.equal(got[rows, N - 1], -torch.sign(x[rows, 1]) * float("inf"))
        assert torch.equal(got[rows, : N // 2], _product(x, full, tile)[rows, : N // 2])
        want = odd[rows].double() @ w[N // 2].double()
        inside = want.abs() < 3e38
        assert torch.allclose(got[rows, N // 2].double()[inside], want[inside], rtol=1e-5)


@pytest.mark.parametrize("M,N,K", [(2, 40, 32), (19, 33, 100), (50, 150, 516), (130, 64, 300)])
@pytest.mark.parametrize("power", [-100, -110, -118, -126, -133])
def test_product_of_tiny_values(M, N, K, power):
    """Values whose last bits lie below what a part can hold: as near to 64 bits as float32 sums are, and rows of other sizes in the
    same launch keep their bits."""
    g = torch.Generator(device=DEV).manual_seed(M * K)
    usual = torch.randn(M, K, device=DEV, generator=g)
    w = torch.randn(N, K, device=DEV, generator=g)
    x = usual.clone()
    x[::2] = (usual[::2].double() * 2.0 ** power).float()
    for few in (x, x.flip(0)):
        # of the sum of the products' sizes as in test_product_by_parts, and half a step of 2^-149 for every product and sum
        bound = 2.0 ** -24 * (12 * -(-K // 128) + 5) * (few.double().abs() @ w.double().abs().T) + 2.0 ** -149 * K
        for tile in TILES:
            y = _product(few, w, tile)
            assert bool(((y.double() - few.double() @ w.double().T).abs() <= bound).all()), tile
    # both operands tiny where the other is not
    some = torch.zeros(M, K, device=DEV)
    some[:, ::2] = x[:, ::2]
    v = (w.double() * torch.where(torch.arange(K, device=DEV) % 2 == 1, 2.0 ** power, 1.0)).float()
    for tile in TILES:
        assert torch.equal(_product(x, w, tile)[1::2], _product(usual, w, tile)[1::2])
        y, want = _product(some + x * 0.25, v, tile), (some + x * 0.25).double() @ v.double().T
        size = (some + x * 0.25).double().abs() @ v.double().abs().T
        assert bool(((y.double() - want).abs() <= 2.0 ** -24 * (12 * -(-K // 128) + 5) * size + 2.0 ** -149 * K).all())


@pytest.mark.parametrize("tile", TILES)
def test_product_near_overflow(tile):
    """A sum that float32 holds, though a value rounds up to an infinity in bfloat16 or the product of the rounded values is one; and one
    that float32 does not hold, whose neighbours keep their bits."""
    g = torch.Generator(device=DEV).manual_seed(5)
    x, w = torch.randn(70, 200, device=DEV, generator=g), torch.randn(90, 200, device=DEV, generator=g)
    x[:3] = w[:3] = 0.0
    x[0, 7], w[0, 7] = 3.4e38, 0.99                       # rounds up to an infinity
    x[1, 50], w[1, 50] = 1.999 * 2.0 ** 64, 1.999 * 2.0 ** 62          # 2^65 * 2^63
    x[2, 199], w[2, 199] = 2.0 ** 100, -2.0 ** 100
    y = _product(x, w, tile)
    assert abs(y[0, 0].double() / (x[0, 7].double() * w[0, 7].double()) - 1) < 2.0 ** -23
    assert abs(y[1, 1].double() / (x[1, 50].double() * w[1, 50].double()) - 1) < 2.0 ** -23
    assert float(y[2, 2]) == -float("inf")
    other = x.clone()
    other[:3] = torch.randn(3, 200, device=DEV, generator=g)
    assert torch.equal(y[3:, 3:], _product(other, w, tile)[3:, 3:])


@pytest.mark.parametrize("Hq,Hkv,D,page", [(4, 2, 16, 4), (3, 1, 80, 8), (6, 2, 112, 16), (2, 2, 128, 12), (4, 4, 96, 64)])
@pytest.mark.parametrize("extra", [{}, {"window": 20}, {"window": 37, "keep_first": 5}, {"chunk": 24}, {"softcap": 3.0}])
def test_attention_tiles(Hq, Hkv, D, page, extra):
    """Rows of several requests in one tile of 16, requests that begin inside a tile, decoding rows beside prompts; a
    request's tokens alone give the same bits as beside others."""
    window = extra.get("window")
    seqs = [(40, 1), (300, 1), (17, 17), (5, 2), (129, 33), (70, 15), (64, 16)]
    args = _attention_case(torch.float32, Hq, Hkv, D, page, seqs, seed=D + page, window=window)
    if "keep_first" in extra:            # the kept keys' pages are held: all of them here
        args = _attention_case(torch.float32, Hq, Hkv, D, page, seqs, seed=D + page)
        args = args[:12] + (window,) + args[13:]
    more = {k: v for k, v in extra.items() if k != "window"}
    g = torch.Generator(device=DEV).manual_seed(1)
    sinks, slopes = torch.randn(Hq, device=DEV, generator=g), torch.rand(Hq, device=DEV, generator=g)
    for kw in (more, dict(more, sinks=sinks, slopes=slopes)):
        got = hip().paged_attention(*args, **kw)
        close(got, twin.paged_attention(*args, **kw), 1e-5)
        q, seq_of, positions = args[0], args[6], args[7]
        for a, n in ((19, 2), (23, 9), (54, 16)):
            part = (q[a:a + n],) + args[1:6] + (seq_of[a:a + n].contiguous(), positions[a:a + n].contiguous()) + args[8:]
            assert torch.equal(hip().paged_attention(*part, **kw), got[a:a + n])


def test_attention_keeps_what_is_not_a_number_to_those_who_see_it():
    """A value that is not finite reaches the tokens that see its key and no others, and leaves their bits alone."""
    args = _attention_case(torch.float32, 4, 2, 64, 16, [(40, 40), (9, 9)], seed=3)
    want = hip().paged_attention(*args)
    bt, v_cache = args[4], args[2]
    v_cache[int(bt[0, 1]), 1, 7, 5] = float("inf")           # key 21 of the first request, head 1, dimension 7
    got = hip().paged_attention(*args)
    hit = torch.zeros_like(got, dtype=torch.bool)
    hit[21:40, 2 * 64 + 7] = hit[21:40, 3 * 64 + 7] = True   # the two query heads of that key head
    assert not torch.isfinite(got[hit]).any() and torch.equal(got[~hit], want[~hit])


@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("D,Hq,Hkv,page,keep", [(64, 4, 4, 16, 1), (64, 6, 2, 32, 16), (128, 4, 1, 16, 17), (128, 2, 2, 128, 40), (64, 2, 1, 16, 48)])
def test_kept_keys_by_pieces_are_those_by_words(D, Hq, Hkv, page, keep, sinks):
    """Kept keys over pages in steps of 16 against the general kernel (a cache at an odd address takes it): the same sums in the
    same order, so the same numbers. Tokens in front of the window's end, a page that is gone and a head that saw no key."""
    g = torch.Generator(device=DEV).manual_seed(D + keep)
    T, B, pages, window = 70, 2, 12, 20
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=g)
    q, out = rnd(T, Hq * D + 8).to(torch.bfloat16), rnd(T, Hq * D).to(torch.bfloat16)
    lse = rnd(T, Hq) + 2
    lse[3, 0] = -torch.inf
    n = pages * Hkv * page * D
    flat = [rnd(n + 4).to(torch.bfloat16) for _ in range(2)]
    tables = torch.randperm(pages, device=DEV, generator=g).to(torch.int32).view(B, -1).contiguous()
    tables[1, 0] = -1
    seq = (torch.arange(T, device=DEV) >= 40).int()
    positions = torch.cat((torch.arange(40, device=DEV), torch.arange(10, T - 30, device=DEV))).int()
    contexts = torch.tensor([40, T - 30], dtype=torch.int32, device=DEV)
    cap = 3.0 if keep == 17 else 0.0
    sk, slopes = (rnd(Hq) if sinks else None), (rnd(Hq).abs() if keep == 16 else None)
    both = []
    for shift in (0, 4):
        caches = [torch.empty(n + 4, dtype=torch.bfloat16, device=DEV)[shift:shift + n] for _ in range(2)]
        for c, f in zip(caches, flat):
            c.copy_(f[:n])
        o = out.clone()
        ops.core().call("me_attn_tail", q.data_ptr(), q.stride(0), o.data_ptr(), o.stride(0), lse.data_ptr(), ops._code(q.dtype),
                        caches[0].data_ptr(), caches[1].data_ptr(), tables.data_ptr(), tables.stride(0), seq.data_ptr(),
                        positions.data_ptr(), contexts.data_ptr(), T, Hq, Hkv, D, page, D ** -0.5, window, keep, cap,
                        ops._ptr(sk), ops._ptr(slopes), ops._stream())
        both.append(o)
    assert torch.equal(*both)
