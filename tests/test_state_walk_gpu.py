"""The state-space walk of stretches against the same recurrence a token at a time: the same bits, whatever the
stretch's length is to the chunks that go through LDS, and whatever the state's rows are to the lanes that hold them."""
import numpy as np
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


def fma(a, b, c):
    """a b + c of float32 values in one rounding: the sum in float64 rounded to odd, which the second rounding cannot see."""
    p, c = np.float64(a) * np.float64(b), np.float64(c)            # the product of 24 bits and 24 bits is exact
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    bits = s.view(np.int64)
    odd = np.where((err != 0) & (bits % 2 == 0), bits + np.where((err > 0) == (s > 0), 1, -1), bits)
    return odd.view(np.float64).astype(np.float32)


def sixteen_chains(x, dt, a, B, C, skip, S):
    """A token of one head: x [P], B and C [N], the state S [N, P].  The outputs, and the state behind it."""
    N, P = S.shape
    S = fma(np.full((N, P), a, np.float32), S, (dt * x)[None] * B[:, None])
    part = np.zeros((16, P), np.float32)
    for at in range(0, N, 16):                                     # chain l: rows l, l + 16, ... in ascending order
        rows = np.arange(at, min(at + 16, N))
        part[rows - at] = fma(S[rows], np.broadcast_to(C[rows, None], (len(rows), P)), part[rows - at])
    lanes = np.arange(16)
    for with_lane in (lanes ^ 1, lanes ^ 2, lanes // 8 * 8 + 7 - lanes % 8, 15 - lanes):
        part = part + part[with_lane]
    return fma(np.full(P, skip, np.float32), x, part[0]), S


@pytest.mark.parametrize("steps", [False, True])
@pytest.mark.parametrize("P, N, tokens", [(8, 128, 37), (5, 100, 37), (3, 7, 37), (4, 16, 37), (2, 256, 37), (3, 33, 37), (2, 17, 37), (3, 32, 37)] +
                         [(3, 128, n) for n in (1, 2, 3, 13, 14, 15, 16, 17, 29, 30, 31, 32)])
def test_a_sum_over_the_state_is_sixteen_chains(P, N, tokens, steps):
    """The order that a design's outputs have had in every form of this scan: bit for bit, in stretches and in single steps."""
    heads = 2
    d = case(heads, 1, P, N, tokens)
    k = kernels("float32")
    state = torch.randn(1, 2 * d["copy"], device="cuda")
    at = d["tail"]
    S = [state[0, d["copy"]:d["copy"] + at].view(heads, N, P)[h].cpu().numpy() for h in range(heads)]       # behind position -1
    u, terms, skip = d["u"].cpu().numpy(), d["terms"].cpu().numpy(), d["skip"].cpu().numpy()
    want = np.empty((tokens, heads * P), np.float32)
    for t in range(tokens):
        B, C = u[t, heads * P:heads * P + N], u[t, heads * P + N:]
        for h in range(heads):
            want[t, h * P:(h + 1) * P], S[h] = sixteen_chains(u[t, h * P:(h + 1) * P], terms[t, h, 0], terms[t, h, 1], B, C, skip[h], S[h])
    if steps:
        got = torch.cat([scan(k, d, state, None, i32([t]), i32([0]), [t]) for t in range(tokens)])
    else:
        got = scan(k, d, state, i32([[0, 0, tokens]]), i32(list(range(tokens))), i32([0] * tokens), list(range(tokens)))
    assert np.array_equal(got.cpu().numpy(), want)
    left = state[0, (tokens - 1) % 2 * d["copy"]:][:at].view(heads, N, P).cpu().numpy()
    assert np.array_equal(left, np.stack(S))
