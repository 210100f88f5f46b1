"""Products of many rows whose blocks keep the sums of K's segments in registers: the bits of the kernels that take a
segment a block, for every epilogue, at the edges of their tiles and on both sides of the choice."""
import pytest
import torch

from axon_amd.kernels import MODE_ADD_F32, MODE_RELU_SQUARED, MODE_STORE, MODE_STORE_F32, MODE_SWIGLU, kernels

pytestmark = pytest.mark.gpu


def _kept(m, n, gated):
    return -(-m // 128) * -(-n // (64 if gated else 128)) >= (144 if gated else 288)     # of the K and the sizes below


@pytest.mark.parametrize("mode", [MODE_STORE, MODE_ADD_F32, MODE_STORE_F32, MODE_SWIGLU, MODE_RELU_SQUARED])
@pytest.mark.parametrize("M,N,K", [(2050, 2064, 512), (1153, 4100, 1088), (4100, 1106, 1600), (1200, 2944, 3072)])
def test_rows_have_the_bits_they_have_alone(M, N, K, mode):
    if mode == MODE_SWIGLU:
        N = N // 16 * 16
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = k.prepare_weight((torch.randn((2 if mode == MODE_SWIGLU else 1) * N, K, generator=g, device="cuda") * 0.1).bfloat16(), mode == MODE_SWIGLU)
    assert k.gemm_segments(N, K, mode == MODE_SWIGLU) > 1
    bias = torch.randn(N, generator=g, device="cuda") if mode != MODE_SWIGLU else None
    base = torch.randn(M, N, generator=g, device="cuda").to(torch.float32 if mode in (MODE_ADD_F32, MODE_STORE_F32) else torch.bfloat16)
    whole = base.clone()
    k.reset_instances()
    k.gemm(x, w, whole, bias, mode)
    gated = mode == MODE_SWIGLU
    assert (k.instances(launched=True) == [f"gemm_kept<{int(gated)}>"]) == _kept(M, N, gated)
    for first, m in ((0, 16), (M - 64, 64), (M // 2, 140), (3, 300)):
        part = base[first:first + m].clone()
        k.reset_instances()
        k.gemm(x[first:first + m].contiguous(), w, part, bias, mode)
        assert (f"gemm_kept<{int(gated)}>" in k.instances(launched=True)) == _kept(m, N, gated)
        assert torch.equal(part, whole[first:first + m]), (first, m)


@pytest.mark.parametrize("M,N,K", [(1300, 3584, 3584), (2049, 2304, 5120)])
def test_the_norm_behind(M, N, K):
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = k.prepare_weight((torch.randn(N, K, generator=g, device="cuda") * 0.05).bfloat16())
    gain, rows = torch.randn(N, generator=g, device="cuda").bfloat16(), torch.randn(M, N, generator=g, device="cuda")
    out, normed = rows.clone(), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    k.reset_instances()
    k.gemm(x, w, out, None, MODE_ADD_F32, following_norm=(gain, normed, 1e-6))
    assert {"gemm_kept<0>", "gemm_split_reduce<1>"} == set(k.instances(launched=True))
    plain = rows[:200].clone()
    k.gemm(x[:200].contiguous(), w, plain, None, MODE_ADD_F32)
    alone = torch.empty(200, N, dtype=torch.bfloat16, device="cuda")
    k.rmsnorm(plain, gain, 1e-6, alone)
    assert torch.equal(out[:200], plain) and torch.equal(normed[:200], alone)


def test_which_products_keep_them():
    """Both sides of each line of the choice: blocks, K by the number of segments, the last round of blocks."""
    k = kernels("bfloat16")
    sizes = [(1525, 2560, 2048, 0, True), (1409, 2560, 2048, 0, True), (1408, 2560, 2048, 0, False), (1525, 2560, 2112, 0, False),
             (300, 12300, 1024, 0, True), (140, 12300, 1024, 0, False), (300, 12300, 3136, 0, False), (4096, 4096, 4096, 0, True),
             (2048, 5120, 4160, 0, False), (1525, 5120, 5120, 0, True), (2432, 5120, 4160, 0, False), (2433, 5120, 4160, 0, True),
             (4096, 2048, 8256, 0, False), (700, 1472, 1024, 1, False), (700, 1488, 1024, 1, True), (256, 8192, 2048, 1, True),
             (256, 8192, 2112, 1, False), (257, 8192, 3072, 1, True), (257, 8192, 3136, 1, False)]
    for M, N, K, gated, kept in sizes:
        x = torch.zeros(M, K, dtype=torch.bfloat16, device="cuda")
        w = k.prepare_weight(torch.zeros((1 + gated) * N, K, dtype=torch.bfloat16, device="cuda"), bool(gated))
        out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
        k.reset_instances()
        k.gemm(x, w, out, None, MODE_SWIGLU if gated else MODE_STORE)
        assert (f"gemm_kept<{gated}>" in k.instances(launched=True)) == kept, (M, N, K, gated)


@pytest.mark.parametrize("M,N,K", [(1100, 9300, 128), (129, 130, 192), (2051, 2309, 768), (1153, 2306, 1088)])
def test_sums_added_into_rows(M, N, K):
    """Whole tiles and remainders in both directions, rows that lie apart, one segment of K and several: what was there
    plus the product, and nothing beside the columns that the product has."""
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.1).bfloat16()
    bias = torch.randn(N, generator=g, device="cuda")
    wide = torch.randn(M, N + 24, generator=g, device="cuda")
    packed, prod = k.prepare_weight(w), torch.empty(M, N, device="cuda")
    got = wide.clone()
    k.gemm(x, packed, got[:, :N], bias, MODE_ADD_F32)
    k.gemm(x, packed, prod, bias, MODE_STORE_F32)
    assert torch.equal(got[:, :N], wide[:, :N] + prod) and torch.equal(got[:, N:], wide[:, N:])
    want = x.double() @ w.double().T + bias.double()
    # a chain of K products and a bias, each sum off by at most a unit of what it holds
    bound = (K + 1) * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T + bias.double().abs())
    assert bool(((prod.double() - want).abs() <= bound).all())


def test_what_goes_through_memory():
    """A product that keeps its sums asks for no more than what a norm or a rotary store behind it reads."""
    need = kernels("bfloat16").lib.axk_gemm_workspace
    assert need(8192, 5120, 2048, MODE_STORE) == need(8192, 5120, 2048, MODE_ADD_F32) == 8192 * 5120 * 4
    assert need(8192, 5120, 2048, MODE_STORE_F32) == need(8192, 5120, 2048, MODE_RELU_SQUARED) == 0
    assert need(2048, 5632, 2048, MODE_SWIGLU) == 0 and need(2048, 3584, 18944, MODE_STORE) == 4 * 2048 * 3584 * 4
    assert need(200, 5632, 4096, MODE_SWIGLU) == 4 * 2 * 200 * 5632 * 4 and need(2048, 30000, 2048, MODE_STORE) == 0


def test_passes_of_a_product_that_keeps_them():
    """More rows than the workspace holds sums of (2 GiB): a second pass of a few rows, with the norm behind."""
    k, N, K = kernels("bfloat16"), 5120, 512
    first = (2 << 30) // (N * 4) // 256 * 256
    M = first + 70
    assert k.lib.axk_gemm_workspace(M, N, K, MODE_ADD_F32) == first * N * 4
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = k.prepare_weight((torch.randn(N, K, generator=g, device="cuda") * 0.1).bfloat16())
    gain, out = torch.randn(N, generator=g, device="cuda").bfloat16(), torch.zeros(M, N, device="cuda")
    normed = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    k.gemm(x, w, out, None, MODE_ADD_F32, following_norm=(gain, normed, 1e-6))
    for at, m in ((0, 100), (first - 60, 130), (first, 70), (M - 9, 9)):
        part, alone = torch.zeros(m, N, device="cuda"), torch.empty(m, N, dtype=torch.bfloat16, device="cuda")
        k.gemm(x[at:at + m].contiguous(), w, part, None, MODE_ADD_F32)
        k.rmsnorm(part, gain, 1e-6, alone)
        assert torch.equal(out[at:at + m], part) and torch.equal(normed[at:at + m], alone), at


@pytest.mark.parametrize("mode", [MODE_STORE, MODE_STORE_F32, MODE_ADD_F32, MODE_SWIGLU, MODE_RELU_SQUARED])
@pytest.mark.parametrize("M,N,K", [(1300, 2576, 512), (700, 16416, 192), (2048, 4608, 192), (300, 16400, 256), (520, 5632, 2048)])
def test_outputs_anywhere(M, N, K, mode):
    """Outputs that are columns of wider rows, aligned for wide stores and not: the bits of a plain output, nothing beside it.
    Kept segments, the three widths of tiles, and a segment a block."""
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = k.prepare_weight((torch.randn((2 if mode == MODE_SWIGLU else 1) * N, K, generator=g, device="cuda") * 0.1).bfloat16(), mode == MODE_SWIGLU)
    bias = None if mode == MODE_SWIGLU else torch.randn(N, generator=g, device="cuda")
    dtype = torch.float32 if mode in (MODE_ADD_F32, MODE_STORE_F32) else torch.bfloat16
    plain = torch.ones(M, N, dtype=dtype, device="cuda")
    k.gemm(x, w, plain, bias, mode)
    for wide, first in ((N + 8, 0), (N + 8, 4), (N + 8, 2), (N + 8, 1), (N + 3, 2), (N + 5, 0)):
        rows = torch.ones(M, wide, dtype=dtype, device="cuda")
        k.gemm(x, w, rows[:, first:first + N], bias, mode)
        assert torch.equal(rows[:, first:first + N], plain), (wide, first)
        assert bool((rows[:, :first] == 1).all()) and bool((rows[:, first + N:] == 1).all()), (wide, first)


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 512, 576, 704])
@pytest.mark.parametrize("N,M", [(9300, 1100), (4608, 2047)])
def test_large_tiles_at_every_end_of_k(K, N, M):
    """Steps of the tiles of 256 rows from one pair on, the last ones with less or nothing to ask for, and rows and columns past
    the end: the bits of the streaming kernel's rows, whatever lies behind K and M in memory."""
    k = kernels("bfloat16")
    g = torch.Generator(device="cuda").manual_seed(K)
    w = k.pack_matrix(torch.randn(N, K, generator=g, device="cuda").bfloat16())
    x = torch.full((M + 1, K + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    x[:M, :K] = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    for mode in (MODE_STORE_F32, MODE_STORE):
        want = torch.empty(M, N, device="cuda", dtype=torch.float32 if mode == MODE_STORE_F32 else torch.bfloat16)
        for at in range(0, M, 16):
            k.gemm(x[at:min(at + 16, M), :K], w, want[at:at + 16], None, mode)
        out = torch.full_like(want, float("nan"))
        k.reset_instances()
        k.gemm(x[:M, :K], w, out, None, mode)
        assert torch.equal(out, want), mode
        names = k.instances(launched=True)
        assert any(name.startswith("gemm_tile<256") for name in names) or (K >= 512 and "gemm_kept<0>" in names), names
