"""The float32 build's prompt and decoding attention on the matrix cores: the bits of `attention`, whatever the head
size, group, page size, window and cut; values that are not finite reach only the tokens that see them."""
import pytest
import torch

from axon_amd.kernels import kernels
from gpu_helpers import paged_cache

pytestmark = pytest.mark.gpu


def _case(nh, nkv, hd, page, T, window, spoil=None):
    g = torch.Generator().manual_seed(T + hd)
    q, keys, vals = (torch.randn(T, n, hd, generator=g) for n in (nh, nkv, nkv))
    if spoil is not None:
        vals[spoil, :, 3] = float("inf")
        vals[spoil, :, 5] = float("nan")
    kc, vc, table = paged_cache(keys, vals, page, "float32")
    q, pos, rows = q.cuda().view(T, nh * hd), torch.arange(T, dtype=torch.int32).cuda(), torch.zeros(T, dtype=torch.int32).cuda()
    want = torch.empty_like(q)
    k = kernels("float32")
    sizes = (nh, nkv, hd, page, window, hd ** -0.5)
    k.attention(q, nh * hd, kc, vc, table, pos, rows, want, *sizes)
    return k, q, (kc, vc, table, pos, rows), sizes, want


def _same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0))


@pytest.mark.parametrize("nh,nkv,hd,page,T,window", [(2, 2, 64, 4, 1, 0), (4, 1, 64, 8, 65, 0), (7, 1, 128, 16, 130, 0),
                                                     (16, 1, 64, 64, 63, 40), (8, 4, 128, 128, 300, 70), (6, 2, 128, 64, 257, 64),
                                                     (2, 1, 64, 32, 400, 0), (64, 4, 128, 16, 330, 0), (48, 3, 64, 32, 300, 100)])
@pytest.mark.parametrize("spoiled", [False, True])
def test_prompts_and_decoding_have_the_bits_of_the_rows_kernel(nh, nkv, hd, page, T, window, spoiled):
    k, q, cache, sizes, want = _case(nh, nkv, hd, page, T, window, T * 2 // 3 if spoiled else None)
    assert k.attention_blocks_ok(hd, page, nh, nkv)
    for cut in (128, 77):                                   # runs of up to 128 tokens; two runs a block
        tiles = [(a, min(cut, T - a)) for a in range(0, T, cut)]
        pairs = [tiles[i] + (tiles[i + 1] if i + 1 < len(tiles) else (0, 0)) for i in range(0, len(tiles), 2)]
        out = torch.full_like(q, 5.0)
        k.reset_instances()
        k.attention_prefill(q, nh * hd, *cache, out, torch.tensor(pairs, dtype=torch.int32).cuda(), *sizes)
        assert _same(out, want), cut
        # two waves for sixteen tokens where there are few blocks
        assert f"attention_f32_waves<{hd},{1 if nh >= 48 else 2}>" in k.instances(launched=True)
    chunks = -(-T // k.attention_decode_chunk) + 1
    partial = torch.full((k.attention_decode_workspace(T, nh, hd, chunks),), float("nan"), device="cuda")
    out = torch.full_like(q, 5.0)
    k.attention_decode(q, nh * hd, *cache, out, T, partial, chunks, *sizes)
    assert _same(out, want)
    pick = torch.tensor(sorted({T - 1, 0}, reverse=True), dtype=torch.int32).cuda()
    out2 = torch.full_like(q, 5.0)
    k.attention_decode(q, nh * hd, *cache, out2, pick, partial, chunks, *sizes)
    assert _same(out2[T - 1], want[T - 1]) and _same(out2[0], want[0])


def test_blocks_of_four_waves_have_the_bits_too():
    """Many tokens whose contexts end within a chunk, and more blocks than the chip has places for."""
    k, nh, nkv, hd, page, T = kernels("float32"), 4, 4, 64, 16, 70
    for starts in ([3] * T, [300] * T + [40] * 200):
        n = len(starts)
        g = torch.Generator().manual_seed(n)
        q, keys, vals = (torch.randn(max(starts) + 1 if i else n, h, hd, generator=g) for i, h in ((0, nh), (1, nkv), (2, nkv)))
        kc, vc, table = paged_cache(keys, vals, page, "float32")
        q, pos, rows = q.cuda().view(n, nh * hd), torch.tensor(starts, dtype=torch.int32).cuda(), torch.zeros(n, dtype=torch.int32).cuda()
        sizes = (nh, nkv, hd, page, 0, hd ** -0.5)
        want, out = torch.empty_like(q), torch.full_like(q, 5.0)
        k.attention(q, nh * hd, kc, vc, table, pos, rows, want, *sizes)
        chunks = max(starts) // k.attention_decode_chunk + 1
        partial = torch.full((k.attention_decode_workspace(n, nh, hd, chunks),), float("nan"), device="cuda")
        k.attention_decode(q, nh * hd, kc, vc, table, pos, rows, out, n, partial, chunks, *sizes)
        assert _same(out, want)


def test_an_engine_of_any_capacity_decodes(tmp_path):
    """So many and so long requests that the decoding kernel's partial results would take 17 GB: the engine runs without."""
    import axon_amd
    from axon_amd.config import config_from_dict
    from axon_amd.engine import StepEntry
    from axon_amd.weights import write_random_model
    cfg = dict(architectures=["Qwen2ForCausalLM"], num_hidden_layers=2, hidden_size=256, intermediate_size=128, num_attention_heads=4,
               num_key_value_heads=2, vocab_size=64, max_position_embeddings=131072, rope_theta=10000.0, rms_norm_eps=1e-6,
               tie_word_embeddings=False)
    write_random_model(config_from_dict(cfg), str(tmp_path), seed=1, std=0.3, storage="float32")
    got = []
    for max_seqs in (4, 8192):
        llm = axon_amd.load(str(tmp_path), dtype="float32", max_seqs=max_seqs, num_pages=300, page_size=64)
        torch.cuda.synchronize()
        before = torch.cuda.memory_reserved()
        llm.engine.step([StepEntry(id=0, tokens=list(range(40)) * 8, want=[319])])
        rows = [llm.engine.step([StepEntry(id=0, tokens=[7 + i], want=[0])]).clone() for i in range(3)]
        rows.append(llm.engine.step([StepEntry(id=0, tokens=[1, 2, 3], want=[0, 1, 2]), StepEntry(id=1, tokens=[5] * 9, want=[8])]).clone())
        got.append(rows)
        assert torch.cuda.memory_reserved() - before < 1 << 30
        del llm
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_what_it_takes():
    k = kernels("float32")
    assert not k.attention_blocks_ok(80, 16, 4, 2) and not k.attention_blocks_ok(128, 2, 4, 2)
    assert not k.attention_blocks_ok(128, 24, 4, 2) and not k.attention_blocks_ok(128, 16, 34, 2)
    assert kernels("bfloat16").attention_blocks_ok(128, 16, 34, 2) == kernels("bfloat16").attention_fast_ok(128, 16, 34, 2)
