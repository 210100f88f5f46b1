"""The kernel that adds a split [q; k; v] product's segments, rotates and stores into the pages, eight tokens a thread:
steps in which its eights are whole, cut by the ends of requests and pages, and out of step with the pages, against the plain
product followed by the rotary kernel.  The same operations on the same numbers, so the bits have to be equal."""
import pytest
import torch

from axon_amd.kernels import MODE_STORE, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("page", [4, 8, 16, 64])
@pytest.mark.parametrize("lengths, starts", [([2056], [0]), ([1, 1, 1, 700, 33, 8, 1305], [5, 64, 7, 0, 3, 16, 8]),
                                             ([2041, 7], [9, 0]), ([16] * 64 + [1024], [8 * (i % 3) for i in range(64)] + [4]),
                                             ([5, 2051], [0, 3]), ([37] * 56, [i % 11 for i in range(56)])])
def test_eight_tokens_a_thread(lengths, starts, page):
    k, nh, nkv, hd, hidden = kernels("bfloat16"), 36, 4, 128, 512
    M, n = sum(lengths), (nh + 2 * nkv) * hd
    assert -(-M // 8) * -(-(n // hd) // 16) >= 640 and k.lib.axk_gemm_segments(n, hidden, 0) > 1
    g = torch.Generator().manual_seed(page + M)
    rand = lambda *s: torch.randn(*s, generator=g)
    w = k.pack_matrix((rand(n, hidden) * 0.05).bfloat16().cuda())
    bias, x = rand(n).cuda(), rand(M, hidden).bfloat16().cuda()
    pos = torch.tensor([s + j for s, m in zip(starts, lengths) for j in range(m)], dtype=torch.int32)
    seq = torch.tensor([i for i, m in enumerate(lengths) for _ in range(m)], dtype=torch.int32)
    most = max(-(-(s + m) // page) for s, m in zip(starts, lengths))
    pages = torch.randperm(len(lengths) * most, generator=g).to(torch.int32).view(len(lengths), most)
    angle = pos[:, None].double() * 10000.0 ** (-torch.arange(0, hd, 2).double() / hd)
    table = torch.stack([angle.sin(), angle.cos()], -1).float().contiguous().cuda()
    pos, seq, pages = pos.cuda(), seq.cuda(), pages.cuda()

    def fresh():
        return (torch.zeros(M, n, dtype=torch.bfloat16, device="cuda"),
                torch.zeros(pages.numel(), nkv, page, hd, dtype=torch.bfloat16, device="cuda"),
                torch.zeros(pages.numel(), nkv, hd, page, dtype=torch.bfloat16, device="cuda"))
    q1, k1, v1 = fresh()
    k.gemm(x, w, q1, bias, MODE_STORE)
    k.rope_kv_write(q1, table, pos, seq, pages, k1, v1, nh, nkv, hd, hd, page, True)
    q2, k2, v2 = fresh()
    k.reset_instances()
    k.gemm_qkv_rope(x, w, bias, q2, table, pos, seq, pages, k2, v2, nh, nkv, hd, page)
    assert "gemm_split_reduce<2,8>" in k.instances(launched=True)
    assert torch.equal(q1[:, :nh * hd], q2[:, :nh * hd]) and torch.equal(k1, k2) and torch.equal(v1, v2)
    assert bool((v2 != 0).any())


def test_the_line_between_one_token_a_thread_and_eight():
    """Three blocks of heads a group of tokens: 214 groups of eight are 642 blocks, 213 are 639."""
    k, nh, nkv, hd, hidden, page = kernels("bfloat16"), 36, 4, 128, 512, 16
    n = (nh + 2 * nkv) * hd
    w = k.pack_matrix(torch.zeros(n, hidden, dtype=torch.bfloat16, device="cuda"))
    for M, eight in ((1704, False), (1705, True)):
        pos, seq = torch.arange(M, dtype=torch.int32, device="cuda"), torch.zeros(M, dtype=torch.int32, device="cuda")
        pages = torch.arange(-(-M // page), dtype=torch.int32, device="cuda").view(1, -1)
        q, x = torch.empty(M, n, dtype=torch.bfloat16, device="cuda"), torch.zeros(M, hidden, dtype=torch.bfloat16, device="cuda")
        kc = torch.empty(pages.numel(), nkv, page, hd, dtype=torch.bfloat16, device="cuda")
        vc = torch.empty(pages.numel(), nkv, hd, page, dtype=torch.bfloat16, device="cuda")
        k.reset_instances()
        k.gemm_qkv_rope(x, w, None, q, torch.zeros(M, hd // 2, 2, device="cuda"), pos, seq, pages, kc, vc, nh, nkv, hd, page)
        hit = k.instances(launched=True)
        assert "gemm_split_reduce<2>" in hit and ("gemm_split_reduce<2,8>" in hit) == eight, (M, hit)
