"""Blocks that read the stream rounded to the compute dtype, in the order of a model: the rows that the block before left are taken, and
only those.  The real blocks over a stand-in for the kernels, on the CPU."""
import torch

from axon_amd.models.decoder import DecoderModel
from axon_amd.parts.base import ROUNDED_STREAM
from axon_amd.parts.block import PostNormBlock, SublayerNormBlock

WIDTH = 8


class Kernels:
    def __init__(self):
        self.rounded = 0

    def round_rows(self, x, out):
        self.rounded += 1
        return out.copy_(x)

    def norm_add(self, y, gain, eps, mult, x, rounded=None):
        x += mult * (y * torch.rsqrt(y.square().mean(1, keepdim=True) + eps) * gain)
        if rounded is not None:
            rounded.copy_(x)

    def sum_norm(self, y, alpha, gain, eps, kind, x, rounded=None):
        v = alpha * x + y
        x.copy_(v * torch.rsqrt(v.square().mean(1, keepdim=True) + eps) * gain)
        if rounded is not None:
            rounded.copy_(x)


class Context:
    def __init__(self):
        self.shared, self.ws, self.rt = {"embedding_output": None}, self, self
        self.dtype, self.k = torch.bfloat16, Kernels()

    def take(self, shape, dtype):
        return torch.empty(shape, dtype=dtype)


class Norm:
    def __init__(self, name):
        self.gain, self.eps, self.kind, self.params = torch.linspace(0.5, 1.5, WIDTH), 1e-5, "rms", {}


class Sublayer:
    """y = the rows that it is given times a factor; what it was given has to be the stream's rows as they are."""
    stores_output = True

    def __init__(self, factor):
        self.factor = factor

    def forward(self, ctx, *args, accumulate):
        h, y = args[-2:]
        assert torch.equal(h, ctx.stream.to(h.dtype))
        y.copy_(self.factor * h.float())


def model_of(blocks):
    class Run:
        enter = None

        def __init__(self, layer):
            self.layer = layer

    class Plan:
        bindings = [None] * len(blocks)
    model = DecoderModel.__new__(DecoderModel)
    model.blocks, model.order, model.cache_plan = blocks, [Run(i) for i in range(len(blocks))], Plan()
    return model


def block_of(kind, feed_forward=True):
    return kind(Norm, Sublayer(0.7), Sublayer(-1.3) if feed_forward else None, "l.")


def run(blocks):
    ctx = Context()
    ctx.stream = torch.randn(3, WIDTH, generator=torch.Generator().manual_seed(1))
    model_of(blocks).forward_runs(ctx, ctx.stream, 0, len(blocks))
    return ctx.k.rounded


def test_a_run_of_blocks_rounds_the_stream_once():
    for kind in (SublayerNormBlock, PostNormBlock):
        assert run([block_of(kind), block_of(kind, False), block_of(kind), block_of(kind)]) == 1, kind
    assert run([block_of(SublayerNormBlock), block_of(PostNormBlock), block_of(SublayerNormBlock)]) == 1


def test_a_block_of_another_part_that_leaves_rows_is_heard():
    class Leaves(PostNormBlock):
        def forward(self, ctx, binding, x, normed=None, following=None):
            x.mul_(0.5)
            ctx.shared[ROUNDED_STREAM] = (x, x.to(torch.bfloat16))

    class Silent(PostNormBlock):
        def forward(self, ctx, binding, x, normed=None, following=None):
            x.mul_(0.5)
    for kind in (SublayerNormBlock, PostNormBlock):
        assert run([block_of(kind), block_of(Leaves), block_of(kind)]) == 1
        assert run([block_of(kind), block_of(Silent), block_of(kind)]) == 2


def test_a_subclass_may_go_on_behind_the_block_that_leaves_rows():
    class GoesOn(SublayerNormBlock):
        def forward(self, ctx, binding, x, normed=None, following=None):
            super().forward(ctx, binding, x, normed, following)
            x.mul_(0.5)
    run([block_of(GoesOn), block_of(SublayerNormBlock), block_of(GoesOn), block_of(GoesOn)])
