"""Steps queued one behind the other without reading anything between them: what a step uploads (tokens, tables, lists of
tiles) is read by its own kernels long after the host has gone on to the next, and gives what a step waited for gives."""
import pytest
import torch

import axon_amd
from axon_amd.engine import StepEntry

pytestmark = pytest.mark.gpu

CONFIG = dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=3, hidden_size=128, intermediate_size=256,
              num_attention_heads=4, num_key_value_heads=2, head_dim=64, vocab_size=512, max_position_embeddings=1024,
              rope_theta=10000.0, rms_norm_eps=1e-6, tie_word_embeddings=False)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("requests", [1, 4, 5, 9])          # up to four changed rows of a table are copied singly
def test_queued_steps_give_what_waited_ones_give(dtype, requests):
    engine = axon_amd.load(CONFIG, dtype=dtype, random_seed=1, init_std=0.05, page_size=16, num_pages=400, max_seqs=12,
                           max_seq_len=512).engine
    g = torch.Generator().manual_seed(requests)
    steps = [[torch.randint(0, 512, (int(torch.randint(3, 60, (1,), generator=g)),), generator=g).tolist() for _ in range(requests)]
             for _ in range(12)]

    def run(wait):
        rows = []
        for i, prompts in enumerate(steps):
            ids = [(wait, i, j) for j in range(requests)]
            rows.append(engine.step([StepEntry(r, p, [0, len(p) - 1]) for r, p in zip(ids, prompts)], end=ids))
            if wait:
                torch.cuda.synchronize()
        return rows
    want, got = run(True), run(False)
    for i, (a, b) in enumerate(zip(want, got)):
        assert torch.equal(a, b), i
