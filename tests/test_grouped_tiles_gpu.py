"""The grouped products' two matrix-core kernels at the edges of their tiles: the one for many rows (64 x 128, or 64 x 256
where a gated product has many of these, through LDS) gives the bits of the one for few, whatever the sizes, the type of X
and the layout of the output."""
import pytest
import torch

from axon_amd.kernels import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,G,M", [(8, 32, 2, 321), (128, 96, 3, 321), (129, 64, 2, 321), (260, 160, 1, 321), (300, 288, 2, 321),
                                     (64, 64, 2, 321), (65, 32, 1, 400), (200, 96, 16, 1030), (129, 32, 43, 321)])
@pytest.mark.parametrize("x_f32", [False, True])
@pytest.mark.parametrize("glu", [None, (1.5, 1.702)])
def test_many_rows_have_the_bits_of_few(N, K, G, M, x_f32, glu):
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(N * K)
    x = torch.randn(M, G * K, generator=g, device="cuda")
    x = x if x_f32 else x.bfloat16()
    w = (torch.randn(G, (2 if glu else 1) * N, K, generator=g, device="cuda") * 0.2).bfloat16()
    for out_dtype, pad in ((torch.float32, 0), (torch.bfloat16, 1), (torch.bfloat16, 4)):
        ogs = N + pad
        out = torch.full((M, G * ogs), float("nan"), dtype=out_dtype, device="cuda")
        k.reset_instances()
        k.grouped_gemm(x, w, out, x_group_stride=K, out_group_stride=ogs, glu=glu)
        wide = glu is not None and -(-M // 64) * G * -(-N // 128) >= 512
        assert k.instances(launched=True) == [f"grouped_gemm<{2 if wide else 3},{0 if glu is None else 1}>"]
        for first, m in ((0, 200), (121, 200)):                      # few rows: the other kernel
            few = torch.full((m, G * ogs), float("nan"), dtype=out_dtype, device="cuda")
            k.grouped_gemm(x[first:first + m], w, few, x_group_stride=K, out_group_stride=ogs, glu=glu)
            assert torch.equal(few.nan_to_num(9.0), out[first:first + m].nan_to_num(9.0))
        cols = torch.arange(G * ogs, device="cuda") % ogs < N
        assert not bool(out[:, cols].isnan().any()) and bool(out[:, ~cols].isnan().all())     # nothing beside the groups' columns
        if glu is None and out_dtype == torch.float32:
            want = torch.stack([x[:, i * K:(i + 1) * K].bfloat16().double() @ w[i].double().T for i in range(G)], 1).flatten(1)
            # one chain of K / 32 products of 32, each rounding at most half a unit of the sum of magnitudes a step
            bound = (K + 2) * 2.0 ** -24 * float(x.double().abs().max() * w.double().abs().max()) * K
            assert float((out.double() - want).abs().max()) <= bound


@pytest.mark.parametrize("T,E,top", [(70, 5, 3), (256, 8, 2)])
def test_lists_of_64_and_of_16_rows_agree(T, E, top):
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(T)
    H, F, P = 96, 136, T * top
    h = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    wu = (torch.randn(E, 2 * F, H, generator=g, device="cuda") * 0.2).bfloat16()
    chosen = torch.stack([torch.randperm(E, generator=g, device="cuda")[:top] for _ in range(T)]).int().contiguous()
    scale = torch.rand(P, generator=g, device="cuda")
    got = []
    for rows in (16, 64):
        most = k.route_max_tiles(P, E, rows)
        pairs, tokens, tiles, n = (torch.zeros(s, dtype=torch.int32, device="cuda") for s in (P, P, 3 * most, 1))
        k.route_sort(chosen, E, pairs, tokens, tiles, n, tile_rows=rows)
        out = torch.full((P, F), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.grouped_gemm(h, wu, out, x_group_stride=0, out_group_stride=0, glu=(float("inf"), 1.0, 0.0),
                       routed=(tiles, n, most, tokens, pairs, rows), rows=P, row_scale=scale)
        got.append(out)
    assert torch.equal(got[0], got[1]) and not bool(got[0].isnan().any())


@pytest.mark.parametrize("N,K,by_tile", [(136, 96, True), (2048, 704, True), (4096, 1408, True), (4100, 1568, False), (4096, 2816, False)])
def test_lists_in_both_orders(N, K, by_tile):
    """Groups whose W fits an XCD's cache, and larger ones: tiles of 64 rows, in the order that is the faster, have the bits of tiles
    of 16."""
    k, T, E, top = kernels("bfloat16"), 190, 5, 2
    assert bool(k.lib.axk_grouped_gemm_by_tile(N, K, 0)) == by_tile and not k.lib.axk_grouped_gemm_by_tile(N, K, 1)
    g = torch.Generator(device="cuda").manual_seed(N + K)
    P = T * top
    x = torch.randn(P, K, generator=g, device="cuda").bfloat16()
    w = torch.randn(E, N, K, generator=g, device="cuda").mul_(0.2).bfloat16()
    odds = torch.tensor([9.0, 4.0, 2.0, 0.0, 1.0], device="cuda").expand(T, E)            # uneven, one expert without a row
    chosen = torch.multinomial(odds, top, generator=g).int().contiguous()
    got = []
    for rows in (16, 64):
        most = k.route_max_tiles(P, E, rows)
        pairs, tokens, tiles, n = (torch.zeros(s, dtype=torch.int32, device="cuda") for s in (P, P, 3 * most, 1))
        k.route_sort(chosen, E, pairs, tokens, tiles, n, tile_rows=rows)
        out = torch.full((P, N), float("nan"), device="cuda")
        k.grouped_gemm(x, w, out, x_group_stride=0, out_group_stride=0, routed=(tiles, n, most, pairs, pairs, rows), rows=P)
        got.append(out)
    assert torch.equal(got[0], got[1]) and not bool(got[0].isnan().any())


@pytest.mark.parametrize("T,H,F", [(1, 64, 40), (65, 128, 128), (190, 192, 129), (260, 704, 300), (700, 256, 72)])
def test_lists_of_128_rows(T, H, F):
    """Gated products: a tile's second 64 rows there, partly and not at all, one and two stages of K and more, columns past the end,
    and the second list of a sort against one of its own."""
    k, E, top = kernels("bfloat16"), 5, 2
    g = torch.Generator(device="cuda").manual_seed(T + H)
    P = T * top
    h = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    wu = (torch.randn(E, 2 * F, H, generator=g, device="cuda") * 0.2).bfloat16()
    odds = torch.tensor([9.0, 4.0, 2.0, 0.0, 0.3], device="cuda").expand(T, E)
    chosen = torch.multinomial(odds, top, generator=g).int().contiguous()
    scale = torch.rand(P, generator=g, device="cuda")
    most, most128 = k.route_max_tiles(P, E, 16), k.route_max_tiles(P, E, 128)
    pairs, tokens, tiles, n, tiles128, n128 = (torch.zeros(s, dtype=torch.int32, device="cuda") for s in (P, P, 3 * most, 1, 3 * most128, 1))
    k.route_sort(chosen, E, pairs, tokens, tiles, n, tile_rows=16, wide=(tiles128, n128, 128))
    got = []
    for listed, count, at_most, rows in ((tiles, n, most, 16), (tiles128, n128, most128, 128)):
        out = torch.full((P + 1, F), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.grouped_gemm(h, wu, out[:P], x_group_stride=0, out_group_stride=0, glu=(float("inf"), 1.0, 0.0),
                       routed=(listed, count, at_most, tokens, pairs, rows), rows=P, row_scale=scale)
        assert bool(out[P:].isnan().all())
        got.append(out[:P])
    assert torch.equal(got[0], got[1]) and not bool(got[0].isnan().any())


@pytest.mark.parametrize("T,E,top,identities", [(1, 1, 1, 0), (300, 7, 3, 2), (2050, 1500, 8, 0), (9000, 40, 2, 8), (5000, 4096, 4, 0), (2048, 32, 4, 0), (1024, 64, 8, 1),
                                                (1024, 5, 1, 0), (1025, 64, 1, 2), (2048, 65, 2, 0), (2049, 63, 2, 1), (8192, 2, 2, 0)])
def test_sorting_pairs(T, E, top, identities):
    """More pairs than the block keeps, more experts than it has threads, experts without a pair, and pairs that are not listed."""
    k, P = kernels("bfloat16"), T * top
    g = torch.Generator(device="cuda").manual_seed(P)
    chosen = (torch.rand(T, top, generator=g, device="cuda") ** 2 * (E + identities)).int()
    sizes = (P, P, 3 * k.route_max_tiles(P, E, 64), 1, 3 * k.route_max_tiles(P, E, 128), 1, P, E + 1)
    pairs, tokens, tiles, n, wide, n_wide, place_of, first_of = (torch.full((s,), -7, dtype=torch.int32, device="cuda") for s in sizes)
    k.route_sort(chosen, E, pairs, tokens, tiles, n, place_of, first_of, tile_rows=64, wide=(wide, n_wide, 128))
    flat, pairs, tokens, place_of = (v.long().cpu() for v in (chosen.view(-1), pairs, tokens, place_of))
    count = torch.bincount(flat[flat < E], minlength=E)
    total = int(count.sum())
    first = [0] + count.cumsum(0).tolist()
    assert first_of.tolist() == first and bool((pairs[total:] == -7).all())
    assert pairs[:total].sort().values.tolist() == (flat < E).nonzero().view(-1).tolist()
    assert torch.equal(flat[pairs[:total]], torch.arange(E).repeat_interleave(count)) and torch.equal(tokens[:total], pairs[:total] // top)
    assert torch.equal(place_of[pairs[:total]], torch.arange(total))
    for listed, made, rows in ((tiles, n, 64), (wide, n_wide, 128)):
        want = [[e, first[e] + i, min(rows, int(count[e]) - i)] for e in range(E) for i in range(0, int(count[e]), rows)]
        assert int(made) == len(want) and listed.view(-1, 3)[:len(want)].tolist() == want


@pytest.mark.parametrize("weight_on", ["output", "input"])
def test_routed_experts_of_many_rows_take_lists_of_128(weight_on, monkeypatch):
    """The part on the 128-row side of its rule: the bits of lists of 64 rows."""
    from axon_amd.config.base import PartSpec
    from axon_amd.parts.base import CacheSpec, build_part
    from axon_amd.weights import WeightStore
    from gpu_helpers import DictSource, PartHarness
    T, H, E, ff = 1000, 64, 4, 2048
    part = build_part("feed_forward", PartSpec("routed_experts", {"hidden_size": H, "experts": E, "top": 2, "ff": ff, "limit": 3.0, "weight_on": weight_on}), "l0.")
    g = torch.Generator().manual_seed(3)
    hs = PartHarness("bfloat16", CacheSpec(entries=1, heads=1, head_dim=8), page_size=64, n_pages=32, max_seq_len=1024)
    part.load(WeightStore(DictSource({d.name: torch.randn(*d.shape, generator=g) * 0.2 for d in part.tensors()}), hs.rt.device, hs.rt.dtype), hs.rt)
    h, ctx, k = torch.randn(T, H, generator=g).bfloat16().cuda(), hs.ctx([0] * T), hs.rt.k
    assert k.grouped_gemm_wide(2 * T, E, ff, H) and not k.grouped_gemm_wide(T, E, ff, H)
    got = []
    for wide in (True, False):
        if not wide:
            monkeypatch.setattr(k, "grouped_gemm_wide", lambda *a: False)
        out = torch.full((T, H), float("nan"), device="cuda")
        k.reset_instances()
        part.forward(ctx, h, out, accumulate=False)
        assert ("grouped_gemm<5,1>" in k.instances(launched=True)) == wide
        got.append(out)
    assert torch.equal(got[0], got[1]) and not bool(got[0].isnan().any())
