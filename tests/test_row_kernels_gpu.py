"""Row kernels at the edges of what a thread keeps or takes at once: the embedding's eights, the scaled sum's rows of up to 1,024,
2,048, 3,072 and 4,096 numbers and wider ones, the convolution by runs of tokens."""
import pytest
import torch

from axon_amd.kernels import kernels

pytestmark = pytest.mark.gpu
DTYPES = ["bfloat16", "float32"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [8, 12, 15, 32, 64, 1000, 2048, 2056, 3584, 5120])
def test_embedding_rows(dim, dtype):
    k = kernels(dtype)
    g = torch.Generator(device="cuda").manual_seed(dim)
    flat = torch.randn(48 * dim + 1, generator=g, device="cuda").to(k.dtype)
    tokens = torch.tensor([0, 47, 16, 15, 15], dtype=torch.int32, device="cuda")
    tables = [flat[:48 * dim].view(48, dim), flat[1:].view(48, dim)]           # the second aligned for single numbers alone
    for i, table in enumerate(tables):
        for scale in (1.0, 3.7):
            out = torch.full((6, dim), 7.0, device="cuda")
            k.embed(tokens, table, out[:5], scale)
            assert torch.equal(out[:5], table[tokens.long()].float() * scale) and bool((out[5] == 7.0).all()), (i, scale)
    if k.pack_ok(48, dim):
        out = torch.empty(5, dim, device="cuda")
        k.embed(tokens, k.pack_matrix(tables[0]), out, 3.7)
        assert torch.equal(out, tables[0][tokens.long()].float() * 3.7)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [4, 1000, 1023, 1024, 1028, 2048, 2052, 3072, 3076, 4096, 4100])
@pytest.mark.parametrize("outputs,normed,shifted", [(1, False, False), (2, False, False), (1, True, True), (2, True, False), (2, True, True)])
def test_scaled_sums(dim, outputs, normed, shifted, dtype):
    k, T, eps = kernels(dtype), 3, 1e-5
    g = torch.Generator(device="cuda").manual_seed(dim)

    def some(*shape):
        return torch.randn(*shape, generator=g, device="cuda")
    ys, scales, x, gain, share = [some(T, dim) for _ in range(2)], [some(dim) for _ in range(2)], some(T, dim), some(dim), some(dim)
    positions = torch.tensor([4, 7, 0], dtype=torch.int32, device="cuda")
    slots = torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda")
    state = some(3, 2 * dim)
    terms = [(y, s, e) for y, s, e in zip(ys, scales, (eps, None))][:outputs]
    want = x.double()
    size = want.abs()
    for y, s, e in terms:
        v = y.double()
        v = v / torch.sqrt(v.square().mean(1, keepdim=True) + e) * s.double() if e is not None else v * s.double()
        want, size = want + v, size + v.abs()
    got, out, kept = x.clone(), torch.empty(T, dim, dtype=k.dtype, device="cuda"), state.clone()
    k.scaled_sum(terms, got, norm=(gain, eps, out) if normed else None, shift=(share, kept, positions, slots) if shifted else None)
    # a mean's chain of dim / 256 products with its folds, a root, a quotient and the products and sums of two terms
    unit = (dim / 256 + 24) * 2.0 ** -24
    assert bool(((got.double() - want).abs() <= unit * size).all())
    if not normed:
        assert torch.equal(kept, state)
        return
    h = got.double() / torch.sqrt(got.double().square().mean(1, keepdim=True) + eps) * gain.double()
    bound = unit * h.abs()
    if shifted:
        rows = state.view(3, 2, dim)[slots.long(), (positions.long() + 1) % 2].double()
        put = kept.view(3, 2, dim)[slots.long(), positions.long() % 2].double()
        assert bool(((put - h).abs() <= bound).all())
        assert torch.equal(kept.view(3, 2, dim)[slots.long(), (positions.long() + 1) % 2], rows.float())
        h, bound = h + (rows - h) * share.double(), (bound + 2.0 ** -22 * (rows.abs() + h.abs())) * (1 + share.double().abs())
    assert bool(((out.double() - h).abs() <= bound + (2.0 ** -8 if dtype == "bfloat16" else 2.0 ** -23) * (h.abs() + bound)).all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("taps,heads,pad", [(2, 3, 0), (3, 130, 4), (4, 32, 8), (4, 0, 0)])
@pytest.mark.parametrize("lengths", [[256], [1, 2, 3, 1, 507], [600, 5, 8, 16, 3], [77] * 13])
def test_state_convolution_of_many_tokens(lengths, taps, heads, pad, dtype):
    """Runs of eight tokens a thread: the bits of the requests one after the other, a thread a (token, channel), whatever runs
    their first tokens fall into."""
    k, T, R = kernels(dtype), sum(lengths), len(lengths)
    C = 4000000 // (T * taps) // 4 * 4 + 12              # as few channels as the runs are taken for, and a block's last threads idle
    g = torch.Generator(device="cuda").manual_seed(T + taps)
    rows = torch.randn(T, C + pad, generator=g, device="cuda")
    w = torch.randn(C, taps, generator=g, device="cuda").to(k.dtype)
    bias, dt_bias, a_log = (torch.randn(n, generator=g, device="cuda") for n in (C, max(heads, 1), max(heads, 1)))
    tail_at, copy = 40, 40 + (taps - 1) * C
    state = torch.randn(R, 2 * copy, generator=g, device="cuda")
    raw = torch.randn(T, max(heads, 1), generator=g, device="cuda")
    starts = torch.randint(0, 9, (R,), generator=g, device="cuda").tolist()
    slots = torch.randperm(R, generator=g, device="cuda").tolist()
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lengths)]).int().cuda()
    seq_rows = torch.cat([torch.full((n,), s) for s, n in zip(slots, lengths)]).int().cuda()

    def conv(a, b):
        u = torch.full((b - a, C), float("nan"), device="cuda")
        terms = torch.full((b - a, max(heads, 1), 2), float("nan"), device="cuda")
        more = dict(raw=raw[a:b], dt_bias=dt_bias, a_log=a_log, terms=terms) if heads else {}
        k.state_conv(rows[a:b, :C], w, bias, state, copy, tail_at, positions[a:b].contiguous(), seq_rows[a:b].contiguous(), u, True, **more)
        return u, terms
    k.reset_instances()
    whole, whole_terms = conv(0, T)
    assert k.instances(launched=True) == ["state_conv<1>"]
    at = 0
    for n in lengths:
        for a in range(at, at + n, 255):                 # fewer tokens: the other kernel
            b = min(at + n, a + 255)
            u, terms = conv(a, b)
            first = 0 if a == at else taps - 1           # (a later piece's first tokens read the state, not the tokens before)
            assert torch.equal(u[first:], whole[a + first:b])
            assert not heads or torch.equal(terms, whole_terms[a:b])
        at += n
    assert "state_conv<0>" in k.instances(launched=True)


@pytest.mark.parametrize("T,C,taps,single,runs", [(256, 3908, 4, False, True), (256, 3904, 4, False, False), (256, 6056, 4, True, True), (256, 6052, 4, True, False),
                                                  (255, 8000, 4, False, False), (1024, 64, 4, False, False), (512, 2560, 4, False, True), (512, 2560, 4, True, False),
                                                  (512, 6056, 2, True, True), (512, 6060, 5, False, False), (512, 6062, 2, False, False)])
def test_the_convolution_by_runs_wants_enough_of_them(T, C, taps, single, runs):
    k = kernels("bfloat16")
    x, w = torch.zeros(T, C, device="cuda"), torch.zeros(C, taps, dtype=torch.bfloat16, device="cuda")
    i, u = torch.zeros(T, dtype=torch.int32, device="cuda"), torch.empty(T, C, device="cuda")
    k.reset_instances()
    k.state_conv(x, w, None, torch.zeros(1, 2 * (taps - 1) * C, device="cuda"), (taps - 1) * C, 0, i, i, u, single=single)
    assert k.instances(launched=True) == [f"state_conv<{int(runs)}>"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [8, 15, 32, 2048, 4096, 4104, 6144])
def test_pairs_of_tokens(dim, dtype):
    k, buckets = kernels(dtype), 7
    g = torch.Generator(device="cuda").manual_seed(dim)
    table, pairs = (torch.randn(n, dim, generator=g, device="cuda").to(k.dtype) for n in (48, buckets + 1))
    tokens = torch.tensor([0, 47, 16, 15, 3], dtype=torch.int32, device="cuda")
    positions = torch.tensor([0, 1, 5, 0, 1], dtype=torch.int32, device="cuda")          # a new request, one that goes on, a new one
    slots = torch.tensor([1, 1, 0, 2, 2], dtype=torch.int32, device="cuda")
    rows = [buckets, (0 * 5 + 47 * 3) % buckets, (9 * 5 + 16 * 3) % buckets, buckets, (15 * 5 + 3 * 3) % buckets]
    want = table[tokens.long()].double() * 0.75 + pairs[rows].double()
    for t in [table] + ([k.pack_matrix(table)] if k.pack_ok(48, dim) else []):
        state = torch.tensor([[9, 9], [0, 0], [0, 0]], dtype=torch.int32, device="cuda")
        out = torch.full((6, dim), 7.0, device="cuda")
        k.embed_pairs(tokens, t, 0.75, pairs, 5, 3, state, positions, slots, out[:5])
        assert bool(((out[:5].double() - want).abs() <= 2.0 ** -23 * want.abs()).all()) and bool((out[5] == 7.0).all())
        assert state[0, 1] == 16 and state[1, 1] == 47 and state[2, 1] == 3


@pytest.mark.parametrize("width", [4, 1000, 1023, 2048])
@pytest.mark.parametrize("T", [3, 300])
@pytest.mark.parametrize("top", [1, 2, 3, 4, 7, 8])
def test_experts_rows_added_up(T, top, width):
    """Fours, a pair and a single one, in order; with places, a further row, its gate, identities and a sum that goes on."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(top)
    P = T * top
    rows, weights = torch.randn(P + 1, width, generator=g, device="cuda"), torch.rand(T, top, generator=g, device="cuda")
    places = torch.randperm(P, generator=g, device="cuda").int()
    experts = torch.randint(0, 6, (T, top), generator=g, device="cuda").int()
    extra, gate = torch.randn(T, width, generator=g, device="cuda"), torch.randn(T, 3, generator=g, device="cuda")
    h = torch.randn(T, width, generator=g, device="cuda")
    for place, more, gated, identities, on in ((None, None, False, False, False), (places, extra, True, True, True), (places, extra, False, False, True)):
        y = torch.randn(T, width, generator=g, device="cuda")
        want = y.clone() if on else torch.zeros_like(y)
        size = want.abs().double()
        for j in range(top):
            pair = torch.arange(T, device="cuda") * top + j
            row = rows[(place[pair] if place is not None else pair).long()]
            if identities:
                row = torch.where((experts[:, j] >= 4)[:, None], h, row)
            want = (weights[:, j, None].double() * row.double() + want.double()).float()           # a multiply-add rounds once
            size += weights[:, j, None].double() * row.double().abs()
        if more is not None:
            want = want.double() + (torch.sigmoid(gate[:, 1:2].double()) if gated else 1.0) * more.double()
            size += more.double().abs()
        got = _combine(k, rows, weights, y, top, on, place, more, gate if gated else None, experts if identities else None, h if identities else None)
        # the last of the multiply-adds rounds to half a unit of the sum of magnitudes, the gate's exponential, sum and quotient to some three
        assert bool(((got.double() - want).abs() <= 2.0 ** -21 * size).all())


def _combine(k, rows, weights, y, top, on, place, more, gate, experts, h):
    p = lambda t: None if t is None else t.data_ptr()
    k._check(k.run.axk_route_combine(p(rows), p(weights), p(y), y.shape[0], top, y.shape[1], int(on), p(place), p(more),
                                     None if gate is None else gate[:, 1:].data_ptr(), 0 if gate is None else gate.stride(0), p(experts), 4,
                                     p(h), 0 if h is None else h.stride(0), torch.cuda.current_stream().cuda_stream))
    return y


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n_state", [16, 64, 128, 200])
def test_outputs_of_stretches_that_end_anywhere_in_a_chunk(n_state, dtype):
    """Four turns' sums at a time, a lane a turn of sixteen: the bits of the tokens one at a time, whatever is left in the last
    chunks, with many heads and requests at once."""
    k, heads, groups, vdim, taps = kernels(dtype), 32, 2, 20, 4
    lengths = [1, 2, 3, 13, 14, 15, 16, 17, 18, 19, 29, 30, 31, 33]
    T, R, C = sum(lengths), len(lengths), heads * vdim + 2 * groups * n_state
    g = torch.Generator(device="cuda").manual_seed(n_state)
    tail_at = heads * n_state * vdim
    copy = tail_at + (taps - 1) * C
    u, terms = torch.randn(T, C, generator=g, device="cuda"), torch.rand(T, heads, 2, generator=g, device="cuda")
    skip, conv_in = torch.randn(heads, generator=g, device="cuda"), torch.randn(T, C, generator=g, device="cuda")
    state = torch.randn(R, 2 * copy, generator=g, device="cuda")
    starts = [sum(lengths[:i]) for i in range(R)]
    spans = torch.tensor([[i, a, n] for i, (a, n) in enumerate(zip(starts, lengths))], dtype=torch.int32, device="cuda")
    positions = torch.cat([torch.arange(n) for n in lengths]).int().cuda()
    slots = torch.cat([torch.full((n,), i) for i, n in enumerate(lengths)]).int().cuda()
    whole, walked = torch.full((T, heads * vdim), float("nan"), device="cuda"), state.clone()
    k.state_space_scan(u, terms, skip, walked, copy, tail_at, spans, positions, slots, conv_in, whole, heads, groups, vdim, n_state, taps)
    stepped = state.clone()
    for at in range(max(lengths)):
        rows = torch.tensor([a + at for a, n in zip(starts, lengths) if at < n], device="cuda")
        y = torch.full((len(rows), heads * vdim), float("nan"), device="cuda")
        k.state_space_scan(u[rows], terms[rows], skip, stepped, copy, tail_at, None, positions[rows], slots[rows], conv_in[rows], y, heads,
                           groups, vdim, n_state, taps)
        assert torch.equal(y, whole[rows]), at


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim", [4, 64, 508, 512, 516, 1024])
def test_norms_of_many_rows_are_those_of_few(dim, dtype):
    """Many narrow rows ask for the gain behind the sum, others beside the row: the same bits."""
    k, T = kernels(dtype), 4096
    g = torch.Generator(device="cuda").manual_seed(dim)
    x, gain = torch.randn(T, dim, generator=g, device="cuda"), torch.randn(dim, generator=g, device="cuda")
    for vector in (gain, gain.to(k.dtype)):
        many, few = (torch.empty(n, dim, dtype=k.dtype, device="cuda") for n in (T, 7))
        k.rmsnorm(x, vector, 1e-5, many)
        rows = torch.tensor([0, 1, 63, 64, 2047, 4094, 4095], dtype=torch.int32, device="cuda")
        k.rmsnorm(x, vector, 1e-5, few, rows)
        assert torch.equal(many[rows.long()], few)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("size", [1, 64, 255, 256, 257, 512, 513, 1024, 1025, 1300])
def test_gated_norms_of_parts(size, dtype):
    """At the edges of what a thread keeps of a part (one, two and four values) and beyond."""
    k, T, parts, eps = kernels(dtype), 3, 2, 1e-5
    g = torch.Generator(device="cuda").manual_seed(size)
    y, z = torch.randn(T, size * parts, generator=g, device="cuda"), torch.randn(T, size * parts + 4, generator=g, device="cuda")[:, :size * parts]
    gain = torch.randn(size * parts, generator=g, device="cuda")
    for vector in (gain, gain.to(k.dtype)):
        out = torch.empty(T, size * parts, dtype=k.dtype, device="cuda")
        k.gated_group_norm(y, z, vector, eps, out, parts)
        v = (y.double() * z.double() * torch.sigmoid(z.double())).view(T, parts, size)
        want = (v / torch.sqrt(v.square().mean(2, keepdim=True) + eps)).view(T, -1) * vector.double()
        # the gate's exponential, sum, quotient and product in what is summed and scaled; the mean's chain and folds, a root, two quotients, two products;
        # and a bfloat16 output is rounded to eight bits, by up to 2^-8 of itself
        bound = (size / 256 + 32) * 2.0 ** -24 * want.abs() + (2.0 ** -8 if dtype == "bfloat16" else 0.0) * want.abs()
        assert bool(((out.double() - want).abs() <= bound).all())
