"""The norm on a sublayer's output at the edges of what a thread keeps of a row (1, 2, 4, 8 and 16 times 256 values, and wider rows),
and whose rounded rows a block takes for the stream's."""
import pytest
import torch

from axon_amd.kernels import kernels
from axon_amd.models.decoder import DecoderModel
from axon_amd.parts.base import ROUNDED_STREAM
from axon_amd.parts.block import SublayerNormBlock


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("dim", [1, 255, 256, 257, 512, 513, 1023, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 5000])
def test_rows_of_any_width(dim, dtype):
    k = kernels(dtype)
    g = torch.Generator(device="cuda").manual_seed(dim)
    y, x, gain = (torch.randn(*shape, generator=g, device="cuda") for shape in ((3, dim), (4, dim), (dim,)))
    for vector in (gain, gain.to(k.dtype)):
        got, rounded = x.clone(), torch.empty(3, dim, dtype=k.dtype, device="cuda")
        k.norm_add(y, vector, 1e-5, 0.7, got[:3], rounded)
        ys = y.double()
        term = 0.7 * (ys / torch.sqrt(ys.square().mean(1, keepdim=True) + 1e-5) * vector.double())
        want = x[:3].double() + term
        # the mean's chain of dim / 256 products and its folds, a root, a quotient, and five more roundings of the term; one of the sum
        bound = (dim / 256 + 24) * 2.0 ** -24 * term.abs() + 2.0 ** -23 * want.abs()
        assert bool(((got[:3].double() - want).abs() <= bound).all())
        assert torch.equal(got[3], x[3]) and torch.equal(rounded, got[:3].to(k.dtype))
        plain = x.clone()
        k.norm_add(y, vector, 1e-5, 0.7, plain[:3])
        assert torch.equal(plain, got)


class _Shared:
    def __init__(self):
        self.shared = {}


def test_only_the_block_before_hands_on_rounded_rows():
    """Runs in order: a block finds the rows that the one before left; not behind a block that leaves none, not behind a
    rewritten stream, not in another call of forward_runs."""
    found, x, mark = [], torch.zeros(1, 1), object()

    class Toy:
        mixer = feed_forward = None

        def __init__(self, leaves):
            self.leaves_rounded_stream = leaves

        following_of = staticmethod(lambda *a: None)

        def last_part(self):
            return None

        def entry_norm(self, binding):
            return None

        def forward(self, ctx, binding, x):
            left = ctx.shared.get(ROUNDED_STREAM)
            found.append(left is not None and left[0] is x)
            if self.leaves_rounded_stream:
                ctx.shared[ROUNDED_STREAM] = (x, mark)

    class Run:
        def __init__(self, layer, enter=None):
            self.layer, self.enter = layer, enter

    class Entry:
        def forward(self, ctx, x, x0):
            pass

    model = DecoderModel.__new__(DecoderModel)
    model.blocks = [Toy(True), Toy(False)]
    model.order = [Run(0), Run(0), Run(1), Run(0), Run(0, "entry"), Run(0)]
    model.entries = {"entry": Entry()}

    class Plan:
        bindings = [None] * 6
    model.cache_plan = Plan()
    ctx = _Shared()
    ctx.shared["embedding_output"] = None
    model.forward_runs(ctx, x, 0, 6)
    assert found == [False, True, True, False, False, True]
    found.clear()
    model.forward_runs(ctx, x, 5, 6)             # what the call before left is not this one's
    assert found == [False]
    ctx.shared[ROUNDED_STREAM] = (x, mark)
    assert SublayerNormBlock.rounded(ctx, x) is mark
