"""Decoding attention whose blocks of 64 positions run side by side, against float64 over the cached rows.

What the kernels round: queries and weights to bfloat16 (a weight by up to 2^-9 of itself; keys and values are given in bfloat16),
sums in 32 bits.  An output is a weighted mean of values, so a weight's rounding moves it by up to 2^-9 of the largest value;
twice that is asked for, and as much again where the output itself is stored in bfloat16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE, DEV = 64, "cuda:0"


def tables(contexts):
    """Pages of every request, shuffled; the positions of the tokens that are decoded."""
    need = [c // PAGE + 1 for c in contexts]
    order = torch.randperm(sum(need) + 1, device=DEV).int()
    table = torch.zeros(len(contexts), max(need) + 1, dtype=torch.int32, device=DEV)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = order[at:at + n]
        at += n
    return table, int(order.numel()), torch.tensor(contexts, dtype=torch.int32, device=DEV), torch.arange(len(contexts), dtype=torch.int32, device=DEV)


def rows_of(cache, table, i, n):
    """The pages' floats of request i that hold positions 0 .. n - 1."""
    return cache[table[i, :-(-n // PAGE)].long()].double()


def seen(mask, size, keep, pos):
    j = torch.arange(pos + 1, device=DEV)
    if mask == "window":
        return (j > pos - size) | (j < keep)
    return j >= pos // size * size if mask == "chunk" else j >= 0


@pytest.mark.parametrize("heads, kv_heads, maps, dim, vdim", [(8, 2, 1, 128, 256), (16, 2, 1, 128, 128), (8, 1, 2, 64, 128), (20, 1, 1, 72, 48),
                                                              (3, 3, 2, 40, 64), (2, 2, 1, 256, 256), (4, 2, 2, 256, 208), (17, 1, 1, 32, 16)])
@pytest.mark.parametrize("mask, size, keep", [("causal", 0, 0), ("window", 200, 0), ("window", 130, 70), ("chunk", 192, 0)])
def test_masked_attention_by_blocks(heads, kv_heads, maps, dim, vdim, mask, size, keep):
    from axon_amd.kernels import kernels
    k = kernels("bfloat16")
    torch.manual_seed(heads * dim + size)
    contexts = [0, 1, 63, 64, 65, 127, 128, 300, 700]
    table, pages, positions, slots = tables(contexts)
    T, kw = len(contexts), kv_heads * maps * dim
    cache = torch.randn(pages, PAGE * (kw + kv_heads * vdim), device=DEV).bfloat16()
    q = torch.randn(T, heads * maps * dim, device=DEV).bfloat16()
    sinks = torch.randn(heads, device=DEV)
    lam, out_scale, eps, scale = 0.3, 0.7, 1e-6, dim ** -0.5
    out = torch.full((T, heads * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
    k.masked_attention(q, cache.view(pages, 1, PAGE, -1), table, positions, slots, out, heads, kv_heads, maps, dim, vdim, PAGE, mask, size, scale, lam=lam,
                       out_scale=out_scale, eps=eps, sink=sinks, span=max(contexts) + 1, keep=keep)
    for i, pos in enumerate(contexts):
        page = rows_of(cache, table, i, pos + 1)
        K = page[:, :PAGE * kw].reshape(-1, kv_heads, maps, dim)[:pos + 1]
        V = page[:, PAGE * kw:].reshape(-1, kv_heads, vdim, PAGE).permute(0, 3, 1, 2).reshape(-1, kv_heads, vdim)[:pos + 1]
        Q, group = q[i].double().view(heads, maps, dim), heads // kv_heads
        hidden = ~seen(mask, size, keep, pos)
        for h in range(heads):
            o = []
            for m in range(maps):
                s = (K[:, h // group, m] @ Q[h, m] * scale).masked_fill(hidden, -float("inf"))
                w = torch.softmax(torch.cat([s, sinks[h:h + 1].double()]), 0)[:-1]
                o.append(w @ V[:, h // group])
            want = o[0]
            bound = 2 ** -8 * V.abs().max().item()
            if maps == 2:
                d = o[0] - lam * o[1]
                unit = torch.rsqrt((d * d).mean() + eps).item()
                want, bound = d * unit * out_scale, 2 * bound * (1 + lam) * unit * out_scale
            got = out[i].double().view(heads, vdim)[h]
            assert ((got - want).abs() <= bound + 2 ** -8 * want.abs()).all(), (i, pos, h, (got - want).abs().max().item(), bound)


@pytest.mark.parametrize("heads, rank, rot", [(16, 512, 64), (32, 512, 128), (16, 64, 32), (16, 48, 80), (48, 128, 64), (16, 208, 16)])
@pytest.mark.parametrize("window", [0, 100, 256])
@pytest.mark.parametrize("sunk", [False, True])
def test_latent_attention_by_blocks(heads, rank, rot, window, sunk):
    from axon_amd.kernels import kernels
    k = kernels("bfloat16")
    torch.manual_seed(heads + rank + window)
    contexts = [0, 63, 64, 65, 127, 300, 511]
    table, pages, positions, slots = tables(contexts)
    T, width = len(contexts), rank + rot
    cache = torch.randn(pages, PAGE * (width + rank), device=DEV).bfloat16()
    rows, by_dim = cache[:, :PAGE * width].view(-1, PAGE, width), cache[:, PAGE * width:].view(-1, rank, PAGE)
    by_dim.copy_(rows[:, :, :rank].transpose(1, 2))
    q = torch.randn(T, heads, width, device=DEV).bfloat16().float()
    sinks = torch.randn(heads, device=DEV) if sunk else None
    out = torch.full((T, heads, rank), float("nan"), device=DEV)
    scale = width ** -0.5
    k.latent_attention(q.view(T, -1), cache.view(pages, 1, PAGE, -1), table, positions, slots, out.view(T, -1), heads, rank, rot, PAGE, window, scale, span=max(contexts) + 1, sink=sinks)
    for i, pos in enumerate(contexts):
        C = rows_of(cache, table, i, pos + 1)[:, :PAGE * width].reshape(-1, width)[:pos + 1]
        s = (q[i].double() @ C.T * scale).masked_fill(~seen("window" if window else "causal", window, 0, pos), -float("inf"))
        if sunk:
            s = torch.cat([s, sinks.double()[:, None]], 1)
        want = torch.softmax(s, 1)[:, :pos + 1] @ C[:, :rank]
        assert ((out[i].double() - want).abs() <= 2 ** -8 * C.abs().max()).all(), (i, pos, (out[i].double() - want).abs().max().item())
