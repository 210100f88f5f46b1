"""Latent attention in steps of many tokens: eight tokens a block through LDS give the bits of a wave a token, for every
size class, page, window and sink, with tokens of several requests side by side and runs that start anywhere: tiles of one
request, of two, of decoding rows with the end or the start of a portion, of several short portions."""
import pytest
import torch

from axon_amd.kernels import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,rot,page,window,heads", [(512, 64, 64, 0, 16), (512, 64, 128, 100, 16), (512, 128, 64, 70, 16), (48, 16, 64, 0, 32),
                                                        (64, 64, 64, 65, 16), (128, 32, 192, 0, 16), (112, 48, 64, 1, 16), (256, 64, 64, 0, 16),
                                                        (512, 32, 64, 130, 16), (256, 32, 64, 50, 32), (64, 32, 128, 0, 32), (64, 128, 64, 200, 16)])
@pytest.mark.parametrize("sink", [False, True])
def test_many_tokens_have_the_bits_of_few(rank, rot, page, window, heads, sink):
    k = kernels("bfloat16")
    assert k.lib.axk_latent_attention_uses_mfma(heads, rank, rot, page)
    g = torch.Generator(device="cuda").manual_seed(rank + window)
    # request, first position, tokens (tiles of eight: three requests in the eighth, a portion of one token more at its end)
    runs = [(0, 0, 61), (1, 7, 3), (2, 130, 133), (1, 10, 1), (0, 61, 77), (3, 300, 38)]
    if heads == 16:
        # decoding rows, the end of a portion behind some and the start of one before others, portions of two and three tokens
        runs += [(1, 40 + i, 1) if i % 2 else (2, 20 + i, 1) for i in range(13)] + [(3, 10, 3), (0, 9, 2), (1, 30, 2), (2, 50, 3), (3, 77, 1), (0, 200, 9), (1, 100, 190)]
    T, most = sum(n for _, _, n in runs), 400
    pages = -(-most // page)
    cache = torch.randn(4 * pages, 1, page, 2 * rank + rot, generator=g, device="cuda").bfloat16()
    table = torch.randperm(4 * pages, generator=g, device="cuda").int().view(4, pages).contiguous()
    rows = torch.tensor([r for r, _, n in runs for _ in range(n)], dtype=torch.int32, device="cuda")
    pos = torch.tensor([p + i for _, p, n in runs for i in range(n)], dtype=torch.int32, device="cuda")
    q = torch.randn(T, heads * (rank + rot), generator=g, device="cuda") * 0.3
    sinks = torch.randn(heads, generator=g, device="cuda") if sink else None

    def attend(a, b):
        out = torch.full((b - a, heads * rank), float("nan"), device="cuda")
        k.latent_attention(q[a:b].contiguous(), cache, table, pos[a:b].contiguous(), rows[a:b].contiguous(), out, heads, rank, rot, page, window,
                           (rank + rot) ** -0.5, sink=sinks)
        return out
    assert T * (heads // 16) >= 512                                      # (from 256 on without a window)
    k.reset_instances()
    whole, step = attend(0, T), 200 // (heads // 16)
    assert any(name.startswith("latent_prompt<") for name in k.instances(launched=True))
    # every token a request of its own: a wave each
    alone = torch.full((T, heads * rank), float("nan"), device="cuda")
    k.latent_attention(q, cache, table[rows.long()].contiguous(), pos, torch.arange(T, dtype=torch.int32, device="cuda"), alone, heads, rank,
                       rot, page, window, (rank + rot) ** -0.5, sink=sinks)
    assert torch.equal(whole, alone)
    if window == 0:                     # (over a window few rows run their blocks side by side, which is another order of sums)
        k.reset_instances()
        few = torch.cat([attend(a, min(a + step, T)) for a in range(0, T, step)])
        assert torch.equal(whole, few) and not any(name.startswith("latent_prompt<") for name in k.instances(launched=True))
    assert torch.equal(whole[5:], attend(5, T))                          # other tokens side by side
    lat = cache[:, 0, :, :].reshape(4 * pages, -1)
    for t in (0, 60, 62, 70, 197, T - 1):                                # against float64, weights and queries rounded as the kernel does
        p, r = int(pos[t]), int(rows[t])
        lo = max(0, p + 1 - window) if window else 0
        at = torch.arange(lo, p + 1, device="cuda")
        pg, o = table[r, at // page].long(), at % page
        key = lat[pg[:, None], (o[:, None] * (rank + rot) + torch.arange(rank + rot, device="cuda"))].double()
        val = lat[pg[:, None], page * (rank + rot) + torch.arange(rank, device="cuda")[None] * page + o[:, None]].double()
        s = q[t].view(heads, -1).bfloat16().double() @ key.T * (rank + rot) ** -0.5
        m = s.amax(-1, keepdim=True) if sinks is None else torch.maximum(s.amax(-1, keepdim=True), sinks.double()[:, None])
        w = torch.exp(s - m)
        want = w @ val / (w.sum(-1, keepdim=True) + (0 if sinks is None else torch.exp(sinks.double()[:, None] - m)))
        # the weights are rounded to 8 bits: each off by at most 2^-9 of itself
        assert float((whole[t].view(heads, rank).double() - want).abs().max()) <= 2.0 ** -8 * float(val.abs().max())
