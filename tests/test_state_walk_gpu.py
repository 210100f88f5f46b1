"""The state-space walk of stretches against the same recurrence a token at a time: the same bits, whatever the
stretch's length is to the chunks that go through LDS, and whatever the state's rows are to the lanes that hold them."""
import pytest
import torch

from axon_amd.kernels import kernels

pytestmark = pytest.mark.gpu

TAPS = 3


def scan(k, d, state, spans, positions, slots, rows, segments=None):
    y = torch.full((len(rows), d["heads"] * d["P"]), float("nan"), device="cuda")
    k.state_space_scan(d["u"][rows].contiguous(), d["terms"][rows].contiguous(), d["skip"], state, d["copy"], d["tail"], spans,
                       positions, slots, d["conv_in"][rows].contiguous(), y, d["heads"], d["groups"], d["P"], d["N"], TAPS, segments)
    return y


def i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def case(heads, groups, P, N, tokens):
    g = torch.Generator(device="cuda").manual_seed(heads * 1000 + N)
    channels = heads * P + 2 * groups * N
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    terms = torch.stack([torch.rand(tokens, heads, generator=g, device="cuda"),
                         0.5 + 0.5 * torch.rand(tokens, heads, generator=g, device="cuda")], -1)
    tail = heads * N * P
    return dict(heads=heads, groups=groups, P=P, N=N, u=rand(tokens, channels), terms=terms, skip=rand(heads).to(torch.float32),
                conv_in=rand(tokens, channels), tail=tail, copy=tail + (TAPS - 1) * channels)


@pytest.mark.parametrize("heads, groups, P, N", [(2, 1, 8, 128), (4, 2, 5, 128), (2, 2, 64, 16), (1, 1, 9, 7), (2, 1, 16, 33),
                                                 (3, 1, 3, 100), (2, 2, 8, 256), (1, 1, 11, 200), (2, 1, 8, 64), (2, 1, 7, 1)])
def test_a_stretch_is_its_tokens_one_by_one(heads, groups, P, N):
    counts = [1, 2, 15, 16, 17, 33, 4, 48, 8, 7]
    d = case(heads, groups, P, N, sum(counts))
    k = kernels("float32")
    starts = [0, 5, 8, 1, 0, 3, 2, 64, 7, 11]
    before = torch.randn(len(counts), 2 * d["copy"], device="cuda")
    firsts = [sum(counts[:i]) for i in range(len(counts))]
    positions = i32([s + j for s, n in zip(starts, counts) for j in range(n)])
    slots = i32([i for i, n in enumerate(counts) for _ in range(n)])
    state = before.clone()
    got = scan(k, d, state, i32([[i, f, n] for i, (f, n) in enumerate(zip(firsts, counts))]), positions, slots,
               list(range(sum(counts))))
    one = before.clone()
    want = torch.empty_like(got)
    for j in range(max(counts)):
        rows = [f + j for f, n in zip(firsts, counts) if j < n]
        want[rows] = scan(k, d, one, None, positions[rows].contiguous(), slots[rows].contiguous(), rows)
    assert torch.equal(got, want)
    for i, (s, n) in enumerate(zip(starts, counts)):
        at = (s + n - 1) & 1                                   # the copy behind the last position
        assert torch.equal(state[i].view(2, -1)[at], one[i].view(2, -1)[at]), (i, n)


@pytest.mark.parametrize("heads, groups, P, N", [(2, 1, 8, 128), (2, 1, 5, 20), (1, 1, 16, 256)])
def test_segments_of_a_stretch_add_up(heads, groups, P, N):
    """Segments differ from one chain by rounding: N + 1 products a sum, states that decay, so some N eps of the
    largest output; the first segment is the chain's own bits."""
    counts, cut = [90, 37], 30
    d = case(heads, groups, P, N, sum(counts))
    k = kernels("float32")
    positions = i32([j for n in counts for j in range(n)])
    slots = i32([i for i, n in enumerate(counts) for _ in range(n)])
    segs, spans, spans5, at = [], [], [], 0
    for i, n in enumerate(counts):
        mine = [[i, at + a, min(cut, n - a), 1 if a == 0 else 0] for a in range(0, n, cut)]
        spans.append([i, at, n])
        spans5.append([i, at, n, len(segs), len(mine)])
        segs += mine
        at += n
    rows = list(range(sum(counts)))
    one, many = (torch.zeros(2, 2 * d["copy"], device="cuda") for _ in range(2))
    want = scan(k, d, one, i32(spans), positions, slots, rows)
    got = scan(k, d, many, i32(spans), positions, slots, rows, (i32(segs), i32(spans5), cut))
    bound = 4 * N * 2.0 ** -24 * float(want.abs().max())
    assert float((got - want).abs().max()) <= bound
    assert torch.equal(got[:cut], want[:cut])
    assert float((many - one).abs().max()) <= 4 * N * 2.0 ** -24 * float(one.abs().max())
