"""The short causal convolution by runs of tokens and the long walk of the gated scan against the kernels that take a
token at a time.  Each sum is made of the same steps in the same order, so the bits have to be equal."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(lengths, device):
    """Slots (not in order), positions (some requests begin, some go on) and spans of one step's requests."""
    seq, pos, spans, first = [], [], [], 0
    for i, n in enumerate(lengths):
        slot, start = (3 * i + 1) % len(lengths) if len(lengths) % 3 else len(lengths) - 1 - i, (0, 7, 12)[i % 3]
        seq += [slot] * n
        pos += list(range(start, start + n))
        spans.append((slot, first, n))
        first += n
    return [torch.tensor(v, dtype=torch.int32, device=device) for v in (seq, pos, spans)]


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lengths, channels", [([64], 4), ([1, 2, 3, 4, 5, 70], 520), ([33, 7, 1, 9, 8, 8, 15], 512), ([127, 2], 2564),
                                               ([520], 2564), ([1] * 513, 2560), ([1, 2, 3, 4, 5, 1290, 33, 7, 1, 9, 8, 8, 15], 960),
                                               ([5000, 246, 3], 252)])
def test_convolution_by_runs(dtype, taps, lengths, channels):
    from axon_amd.kernels import kernels
    k, dev = kernels(dtype), "cuda:0"
    elem = getattr(torch, dtype)
    torch.manual_seed(3)
    seq, pos, _ = _rows(lengths, dev)
    T = sum(lengths)
    x = torch.randn(T, channels, device=dev).to(elem)
    odd = torch.empty(T, channels + 1, dtype=elem, device=dev)[:, :channels]          # rows that four elements at a time cannot be read from
    odd.copy_(x)
    w = torch.randn(channels, taps, device=dev).to(elem)
    state = torch.randn(len(lengths), 2 * taps * channels, device=dev)
    for bias in (None, torch.randn(channels, device=dev)):
        got, want = (torch.empty(T, channels, device=dev) for _ in range(2))
        k.reset_instances()
        k.causal_conv(x, w, bias, state, pos, seq, got)
        # a step of few (token, channel) pairs, a batch of decoding rows among them, keeps a thread each
        assert k.instances(launched=True) == [f"causal_conv<{1 if T * channels >= 512 * 2560 else 0}>"]
        k.causal_conv(odd, w, bias, state, pos, seq, want)
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("lengths", [[5, 31], [32, 33, 1], [63, 64, 65], [95, 96, 97, 128], [300]])
def test_long_walk(dtype, lengths):
    from axon_amd.kernels import kernels
    from axon_amd.kernels.lib import _ptr, _stream
    k, dev, C, width, taps = kernels(dtype), "cuda:0", 192, 64, 4
    elem = getattr(torch, dtype)
    torch.manual_seed(5)
    seq, pos, spans = _rows(lengths, dev)
    T = sum(lengths)
    gates, u = torch.randn(T, 2 * C, device=dev), torch.randn(T, C, device=dev)
    y, x = (torch.randn(T, C, device=dev).to(elem) for _ in range(2))
    lam = torch.rand(C, device=dev)
    state = torch.randn(len(lengths), 2 * taps * C, device=dev)
    kept = state.clone()
    got, want = (torch.empty(T, C, dtype=elem, device=dev) for _ in range(2))
    assert T > 4 * len(lengths)
    k.gated_scan(gates, u, y, x, lam, 8.0, state, spans, pos, seq, got, width, taps)
    # the other entry point: a thread takes its channel's tokens one after another
    assert k.lib.axk_gated_scan(_ptr(gates), _ptr(u), _ptr(y), C, _ptr(x), C, _ptr(lam), 1, 8.0, _ptr(kept), kept.stride(0),
                                _ptr(spans), len(lengths), _ptr(pos), _ptr(seq), _ptr(want), C, width, taps, _stream()) == 0
    assert torch.equal(got, want) and torch.equal(state, kept)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("lengths, channels", [([6], 8), ([95], 2560), ([96], 2560), ([193], 2570), ([400], 4200), ([131], 5130), ([70], 8200),
                                               ([128, 129, 127, 64, 65, 1], 1290), ([9, 300], 20)])
def test_long_walk_by_width(dtype, lengths, channels):
    """Blocks of 8, 10, 16, 20, 32 and 64 channels, the last ones of a row narrower, around whole chunks of each."""
    from axon_amd.kernels import kernels
    from axon_amd.kernels.lib import _ptr, _stream
    k, dev, C, width, taps = kernels(dtype), "cuda:0", channels, channels // 2, 3
    elem = getattr(torch, dtype)
    torch.manual_seed(6)
    seq, pos, spans = _rows(lengths, dev)
    T = sum(lengths)
    gates, u = torch.randn(T, 2 * C, device=dev), torch.randn(T, C, device=dev)
    yx = torch.randn(T, 2 * C, device=dev).to(elem)
    lam = torch.rand(C, device=dev)
    state = torch.randn(len(lengths), 2 * taps * C, device=dev)
    kept = state.clone()
    got, want = (torch.full((T, C), float("nan"), dtype=elem, device=dev) for _ in range(2))
    k.gated_scan(gates, u, yx[:, :C], yx[:, C:], lam, 8.0, state, spans, pos, seq, got, width, taps)
    assert k.lib.axk_gated_scan(_ptr(gates), _ptr(u), _ptr(yx), 2 * C, _ptr(yx[:, C:]), 2 * C, _ptr(lam), 1, 8.0, _ptr(kept), kept.stride(0),
                                _ptr(spans), len(lengths), _ptr(pos), _ptr(seq), _ptr(want), C, width, taps, _stream()) == 0
    assert torch.equal(got, want) and torch.equal(state, kept)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("lengths, channels, kernels_run", [([300, 129, 128, 40, 17, 16, 9, 8, 1], 512, {1}), ([64] * 3 + [1] * 30, 64, {1}),
                                                            ([8, 5, 5], 192, {1}), ([128] * 4, 2048, {1}), ([200, 150], 2560, {1}), ([300, 40], 5120, {1}),
                                                            ([16] * 20 + [9] * 5, 2560, {0}), ([100, 17], 960, {1}), ([60] * 2 + [2] * 5, 512, {1}), ([256], 5120, {1}),
                                                            ([300, 129] + [100] * 3 + [5] * 90, 2560, {0, 1}), ([700] + [1] * 60, 2560, {0, 1})])
def test_requests_of_every_length_have_their_kernel(dtype, lengths, channels, kernels_run):
    """Longest first, with their lengths on the host: the bits of a thread a channel, whichever kernels ran."""
    from axon_amd.kernels import kernels
    from axon_amd.kernels.lib import KernelError, _ptr, _stream
    k, dev, C, width, taps = kernels(dtype), "cuda:0", channels, channels // 2, 4
    elem = getattr(torch, dtype)
    torch.manual_seed(7)
    seq, pos, spans = _rows(lengths, dev)
    T = sum(lengths)
    gates, u = torch.randn(T, 2 * C, device=dev), torch.randn(T, C, device=dev)
    y, x = (torch.randn(T, C, device=dev).to(elem) for _ in range(2))
    lam = torch.rand(C, device=dev)
    state = torch.randn(len(lengths), 2 * taps * C, device=dev)
    kept = state.clone()
    got, want = (torch.full((T, C), float("nan"), dtype=elem, device=dev) for _ in range(2))
    k.reset_instances()
    k.gated_scan(gates, u, y, x, lam, 8.0, state, spans, pos, seq, got, width, taps, lengths)
    assert {f"gated_scan<{i}>" for i in kernels_run} == set(k.instances(launched=True))
    assert k.lib.axk_gated_scan(_ptr(gates), _ptr(u), _ptr(y), C, _ptr(x), C, _ptr(lam), 1, 8.0, _ptr(kept), kept.stride(0),
                                _ptr(spans), len(lengths), _ptr(pos), _ptr(seq), _ptr(want), C, width, taps, _stream()) == 0
    assert torch.equal(got, want) and torch.equal(state, kept)
    for wrong in (lengths[:-1], lengths[::-1] if lengths[0] != lengths[-1] else lengths + [1]):
        with pytest.raises(KernelError, match="lengths"):
            k.gated_scan(gates, u, y, x, lam, 8.0, state, spans, pos, seq, got, width, taps, wrong)
