"""How a step's tokens are split between the attention kernels, without a device: the float32 build's choice between its
prompt, decoding and any-token kernels, which give the same bits, by what each is fast at and how much memory it wants."""
from types import SimpleNamespace

import pytest
import torch

from axon_amd.engine.step import Engine, Span
from axon_amd.kernels.lib import Kernels
from axon_amd.parts import attention as A


class _Kernels(SimpleNamespace):
    """What a plan asks of a kernel library; the workspace and the work list as the library has them."""
    attention_prefill_tile, attention_decode_chunk = 128, 256
    attention_decode_work = Kernels.attention_decode_work

    def _decode_chunk_and_factor(self):
        return 256, 1024

    def attention_decode_workspace(self, n_tokens, n_heads, head_dim, max_chunks):
        return n_tokens * n_heads * max_chunks * 4 * (head_dim + 2)

    def attention_fast_ok(self, head_dim, page_size, n_heads, n_kv_heads):
        return not self.float32

    def attention_blocks_ok(self, head_dim, page_size, n_heads, n_kv_heads):
        return True


def _ctx(spans, float32=True, decode_only=False, max_seqs=8, max_seq_len=8192):
    at, listed = 0, []
    for n, start in spans:
        listed.append(Span(len(listed), at, n, start))
        at += n
    return SimpleNamespace(rt=SimpleNamespace(device="cpu", k=_Kernels(float32=float32)), spans=listed, n_tokens=at, shared={},
                           decode_only=decode_only, decode_scratch={}, decode_shapes={("attention_chunks", 0): 4},
                           decode_inputs={("attention_work", 0): None}, cache=SimpleNamespace(max_seqs=max_seqs, max_seq_len=max_seq_len))


def _tokens(plan):
    """(tokens of the prompt kernel's tiles, tokens of the decoding kernel) of a plan."""
    tiles = [] if plan.tiles is None else plan.tiles.tolist()
    tiled = sorted(t for row in tiles for first, n in (row[:2], row[2:]) for t in range(first, first + n))
    return tiled, [] if plan.decode_tokens is None else plan.decode_tokens.tolist()


@pytest.mark.parametrize("spans, heads, singles", [
    ([(9, 4000)], (28, 4), range(9)),                             # a short portion far into a request
    ([(300, 0), (1, 50), (5, 700)], (16, 2), [300, 301, 302, 303, 304, 305]),
    ([(40, 4000)], (32, 32), []),                                 # too many tokens x key heads
    ([(2, 300)] * 64, (28, 4), range(128)),                       # many portions of fewer tokens than a group has heads
    ([(9, 100), (700, 0), (7, 0), (8, 90)], (28, 4), range(709, 716)),       # too few positions to walk
    ([(5, 0)] * 32, (28, 4), range(160)),
    ([(5, 0)] * 32, (8, 8), []),
    ([(64, 600)], (16, 2), range(64)),
    ([(65, 600)], (16, 2), []),
])
def test_short_portions_go_token_by_token(spans, heads, singles):
    ctx = _ctx(spans)
    plan = A.attention_plan(ctx, 0, *heads, 128, 64)
    tiled, single = _tokens(plan)
    assert single == list(singles) and sorted(tiled + single) == list(range(ctx.n_tokens))
    at = [s.start_pos + i for s in ctx.spans for i in range(s.q_len)]
    want = [slot * 1024 + c for slot, t in enumerate(single) for c in range(at[t] // 256 + 1)]
    assert want == ([] if plan.decode_work is None else plan.decode_work.tolist())
    assert not single or plan.partial.numel() == len(single) * heads[0] * max(at[t] // 256 + 1 for t in single) * 4 * 130
    # the bfloat16 build's split has portions and single tokens only
    tiled, single = _tokens(A.attention_plan(_ctx(spans, float32=False), 0, *heads, 128, 64))
    assert single == [s.q_start for s in ctx.spans if s.q_len == 1]


def test_a_window_bounds_what_a_portion_sees():
    assert _tokens(A.attention_plan(_ctx([(9, 4000)]), 100, 28, 4, 128, 64))[1] == []
    assert _tokens(A.attention_plan(_ctx([(9, 4000)]), 600, 28, 4, 128, 64))[1] == list(range(9))


def test_float32_holds_no_workspace_beyond_its_limit():
    """A float32 engine for so many and so long requests that the decoding kernel's partial results would take gigabytes
    runs with the kernel that needs none, as it did before there was a decoding kernel."""
    mixer = A.GQAttention(dict(hidden_size=64, num_heads=28, num_kv_heads=4, head_dim=128))
    for float32 in (True, False):
        mixer._kernels = _Kernels(float32=float32)
        small, large = mixer.decode_scratch(64, 8192), mixer.decode_scratch(512, 131072)
        assert small == (("attention_partial", 0, 28, 128), 64 * 28 * 32 * 4 * 130)
        assert (large is None) == float32
    assert A.attention_plan(_ctx([(1, 70)] * 3, decode_only=True, max_seqs=64), 0, 28, 4, 128, 64) is not None
    assert A.attention_plan(_ctx([(1, 70)] * 3, decode_only=True, max_seqs=512, max_seq_len=131072), 0, 28, 4, 128, 64) is None
    assert A.attention_plan(_ctx([(1, 70)] * 3, float32=False, decode_only=True, max_seqs=2, max_seq_len=4096), 0, 28, 4, 128, 64) is not None
    # a step that feeds portions too: by what the step itself wants; portions go back to tiles before anything else
    plan = A.attention_plan(_ctx([(7, 60000)] * 40 + [(1, 9)]), 0, 28, 4, 128, 64)
    assert _tokens(plan)[1] == [280]
    assert A.attention_plan(_ctx([(1, 60000)] * 60 + [(300, 0)]), 0, 28, 4, 128, 64) is None


def test_the_cache_pool_leaves_room_for_the_decoding_steps_workspaces(monkeypatch):
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (1 << 30, 1 << 34))
    spec = SimpleNamespace(dtype=None, entries=2, heads=4, head_dim=64)
    cfg = SimpleNamespace(num_pages=0, max_cache_tokens=0, memory_fraction=1.0, max_seqs=1 << 20)
    engine = SimpleNamespace(cfg=cfg, rt=SimpleNamespace(device=None, elem_size=4), max_seq_len=1 << 20,
                             model=SimpleNamespace(cache_plan=SimpleNamespace(group_specs=[spec])), _scratch_sizes={})
    page = 3 * 2 * 4 * 16 * 64 * 4
    assert Engine._pool_size(engine, spec, 3, 16) == (1 << 30) // page
    engine._scratch_sizes = {"a": 1 << 26, "b": 1 << 25}
    assert Engine._pool_size(engine, spec, 3, 16) == ((1 << 30) - (3 << 27)) // page
