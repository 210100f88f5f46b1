"""Steps queued one behind the other without reading anything between them: what a step uploads (tokens, tables, lists of
tiles) is read by its own kernels long after the host has gone on to the next, and gives what a step waited for gives."""
import pytest
import torch

import axon_amd
from axon_amd.cache.manager import CacheManager, GroupPlan
from axon_amd.engine import StepEntry
from axon_amd.parts.base import CacheSpec
from axon_amd.upload import upload

pytestmark = pytest.mark.gpu

CONFIG = dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=3, hidden_size=128, intermediate_size=256,
              num_attention_heads=4, num_key_value_heads=2, head_dim=64, vocab_size=512, max_position_embeddings=1024,
              rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=False)


def _busy():
    """Half a second of the device's time on the stream (its last product's event)."""
    a = torch.ones(8192, 8192, device="cuda")
    for _ in range(60):                                     # 1.1 TFLOP each, and no more than 157 TFLOP/s
        torch.mm(a, a)
    event = torch.cuda.Event()
    event.record()
    return event


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("requests", [1, 4, 5, 9])          # up to four changed rows of a table are copied singly
def test_queued_steps_give_what_waited_ones_give(dtype, requests):
    engine = axon_amd.load(CONFIG, dtype=dtype, random_seed=1, init_std=0.05, page_size=16, num_pages=400, max_seqs=12,
                           max_seq_len=512).engine
    g = torch.Generator().manual_seed(requests)

    def tokens(n):
        return torch.randint(0, 512, (n,), generator=g).tolist()
    steps = [[tokens(int(torch.randint(3, 60, (1,), generator=g))) for _ in range(requests)] for _ in range(12)]
    whole = [tokens(16 * (1 + i % 3)) for i in range(requests)]        # whole pages: the next token of each takes a new one
    further = [[tokens(1) for _ in range(requests)] for _ in range(3)]

    def run(wait):
        rows = []

        def step(entries, end=()):
            rows.append(engine.step(entries, end=end).clone())
            if wait:
                torch.cuda.synchronize()
        for i, prompts in enumerate(steps):
            ids = [(wait, i, j) for j in range(requests)]
            step([StepEntry(r, p, [0, len(p) - 1]) for r, p in zip(ids, prompts)], ids)
        ids = [(wait, "on", j) for j in range(requests)]
        step([StepEntry(r, p, [len(p) - 1]) for r, p in zip(ids, whole)])
        for i, new in enumerate(further):
            step([StepEntry(r, t, [0]) for r, t in zip(ids, new)], ids if i == len(further) - 1 else ())
        return rows
    run(True)                                               # whatever happens once
    want = run(True)
    behind = _busy()
    got = run(False)
    assert not behind.query(), "the device was to be busy with other work until the last step was queued"
    for i, (a, b) in enumerate(zip(want, got)):
        assert torch.equal(a, b), i
    assert len(want) == 16


@pytest.mark.parametrize("groups", [1, 3])
@pytest.mark.parametrize("changed", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("length", [64, 72, 4000])          # rows shorter and longer than the places of sixteen, even and odd
def test_changed_rows_of_all_groups_travel_together(groups, changed, length):
    """However many groups and rows: what the device holds is what the host holds, from one piece of pinned memory."""
    plans = [GroupPlan(CacheSpec(entries=2, heads=1, head_dim=8, window=0 if i == 0 else 48 + 16 * i), 1, 16, 6000) for i in range(groups)]
    cache = CacheManager(plans, [], 20, length, device="cuda:0", dtype=torch.float32)
    slots = [cache.open() for _ in range(20)]
    cache.reserve_many([(s, 16) for s in slots])
    cache.sync_tables()
    for s in slots[3:3 + changed]:
        cache.reserve(s, length)
    asked = torch.cuda.host_memory_stats()["active_requests.allocated"]
    cache.sync_tables()
    assert torch.cuda.host_memory_stats()["active_requests.allocated"] - asked == 1
    for gi, g in enumerate(cache.groups):
        assert torch.equal(g.block_table.cpu(), g.host_table)
        for s in slots:
            row = cache.row(gi, s)
            assert g.host_table[s, :len(row)].tolist() == row and not bool(g.host_table[s, len(row):].any())


def test_uploads_are_not_captured():
    """The pinned memory of an upload serves the next one when its copy has run: a graph must not come to read it."""
    kept = upload([1, 2, 3], "cuda:0")                       # a piece that a captured upload would find at hand
    torch.cuda.synchronize()
    a = torch.zeros(4, device="cuda:0")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        a += 1
        with pytest.raises(RuntimeError, match="captured"):
            upload([4, 5, 6], "cuda:0")
        a += 1
    for i in range(3):
        graph.replay()
        assert a.tolist() == [2.0 * (i + 1)] * 4 and upload([7, i], "cuda:0").tolist() == [7, i] and kept.tolist() == [1, 2, 3]
