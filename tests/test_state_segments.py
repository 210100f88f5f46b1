"""How the state-space mixer cuts a step's stretches into segments, by their lengths and the blocks of its walk.  The cut
decides the order of a long stretch's sums, so a design's outputs change with it."""
from types import SimpleNamespace

import pytest
import torch

from axon_amd.parts.state_space import SelectiveStateSpace


class Recorder:
    """Takes every kernel call, runs none, keeps the scan's segments."""
    def __getattr__(self, name):
        return lambda *a, **kw: None

    def state_space_scan(self, *args, segments=None):
        self.segments = segments


def cut(lengths, heads, decode_only=False):
    """Segments of each stretch, or None; a head of 64 value dims is eight blocks."""
    mixer = SelectiveStateSpace(dict(hidden_size=8, heads=heads, vdim=64, state=16, groups=1, conv=2, eps=1e-6))
    for name in ("w_in", "conv_w", "conv_b", "dt_bias", "a_log", "d_skip", "gain", "w_o"):
        setattr(mixer, name, None)
    k, spans, at = Recorder(), [], 0
    for i, n in enumerate(lengths):
        spans.append(SimpleNamespace(slot=i, q_start=at, q_len=n))
        at += n
    ctx = SimpleNamespace(decode_only=decode_only, spans=spans, shared={}, positions=None, seq_rows=None,
                          rt=SimpleNamespace(device="cpu", dtype=torch.float32, k=k), cache=SimpleNamespace(state=lambda i: None),
                          ws=SimpleNamespace(take=lambda shape, dtype: torch.empty(shape, dtype=dtype)))
    mixer.forward(ctx, SimpleNamespace(state_index=0), torch.empty(at, 8), None)
    return None if k.segments is None else [int(row[4]) for row in k.segments[1]]


@pytest.mark.parametrize("lengths, heads, segments", [
    ([2048], 32, [8]), ([8192], 32, [8]), ([512], 32, [4]), ([300], 32, [2]), ([255], 32, None), ([2048], 33, None),
    ([2048], 20, [12]), ([2048], 8, [16]), ([1024, 200], 16, [8, 1]), ([1024, 1024], 17, None), ([700, 700, 700], 8, [5, 5, 5])])
def test_segments_of_a_step(lengths, heads, segments):
    assert cut(lengths, heads) == segments


def test_single_tokens_are_not_cut():
    assert cut([1] * 8, 2, decode_only=True) is None
