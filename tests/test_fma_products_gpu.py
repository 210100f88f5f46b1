"""The 32-bit products on the matrix cores at the sizes where their blocks, chains and rows end: against float64, bit for
bit against chains of fmaf, and a row's bits whatever the number of rows (which picks the kernel)."""
import pytest
import torch

from axon_amd.kernels import MODE_ADD_F32, MODE_STORE_F32, MODE_SWIGLU, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [MODE_STORE_F32, MODE_ADD_F32, MODE_SWIGLU])
@pytest.mark.parametrize("N,K,x_stride", [(8, 4, 4), (63, 33, 33), (65, 64, 68), (257, 292, 292), (40, 2052, 2055), (4100, 36, 40),
                                           (520, 256, 256), (24, 257, 260), (16390, 40, 44),
                                           (4100, 2052, 2052)])
def test_edges_of_rows_columns_and_chains(N, K, x_stride, mode):
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(N + K)
    w = torch.randn((2 if mode == MODE_SWIGLU else 1) * N, K, generator=g, device="cuda")
    base = torch.randn(200, N, generator=g, device="cuda")
    x = torch.full((200, x_stride), float("nan"), device="cuda")
    x[:, :K] = torch.randn(200, K, generator=g, device="cuda")
    want = x[:, :K].double() @ w.double().T
    # a chain of 32 and the sum of K / 32 chains each round by at most half a unit a step of what they hold
    bound = (32 + K / 32 + 2) * 2.0 ** -24 * (x[:, :K].double().abs() @ w.double().abs().T)
    if mode == MODE_SWIGLU:
        gate, up = want[:, :N], want[:, N:]
        bound = bound[:, :N] * up.abs() * 1.1 + bound[:, N:] * gate.abs() + 4e-6 * (gate * up).abs()
        want = gate * torch.sigmoid(gate) * up
    if mode == MODE_ADD_F32:
        want = want + base.double()
        bound = bound + 2.0 ** -24 * want.abs()
    rows = {}
    for m in (200, 129, 128, 65, 64, 33, 32, 17, 16, 1):
        out = base[:m].clone()
        k.gemm(x[:m, :K], w, out, None, mode)
        assert bool(((out.double() - want[:m]).abs() <= bound[:m] + 1e-30).all()), m
        rows[m] = out
    for m in rows:
        assert torch.equal(rows[m], rows[200][:m]), m


def _by_chains(k, x, w):
    """x w^T as chains of 32 fmaf in ascending k whose sums are added in ascending order: every chain by the grouped
    product's kernel of 32-bit fmaf on the vector unit, one chain over its whole K, with the 32 k of the chain."""
    M, K = x.shape
    total = torch.zeros(M, w.shape[0], device="cuda")
    for k0 in range(0, K, 32):
        part = torch.full_like(total, float("nan"))
        a, b = x[:, k0:k0 + 32].contiguous(), w[:, k0:k0 + 32].contiguous()
        k.grouped_gemm(a, b[None], part, x_group_stride=a.shape[1], out_group_stride=w.shape[0])
        total = total + part
    return total


@pytest.mark.parametrize("N,K", [(65, 64), (130, 257), (16390, 70), (48, 8), (33, 2052)])
@pytest.mark.parametrize("values", ["ordinary", "denormal", "wide"])
def test_the_bits_are_those_of_chains_of_fmaf(N, K, values):
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(K)
    x, w = torch.randn(140, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    if values == "denormal":            # products of 2^-140 or so, sums of them, and some operands below 2^-126
        x, w = x * 2.0 ** -70, w * 2.0 ** -68
        x[:, ::7] *= 2.0 ** -65
        w[:, ::7] *= 2.0 ** 66
    if values == "wide":                # magnitudes over 2^-30 .. 2^30: what is lost shows which k was added when
        x = x * 2.0 ** torch.randint(-15, 16, x.shape, generator=g, device="cuda")
        w = w * 2.0 ** torch.randint(-15, 16, w.shape, generator=g, device="cuda")
    want = _by_chains(k, x, w)
    assert values != "denormal" or (bool((want.abs() < 2.0 ** -126).any()) and bool((want != 0).any()))
    k.reset_instances()
    for m in (140, 128, 40, 20, 7):     # tiles, and the kernel that streams W by 64, 32 and 16 rows
        out = torch.full((m, N), float("nan"), device="cuda")
        k.gemm(x[:m], w, out, None, MODE_STORE_F32)
        assert torch.equal(out, want[:m]), m
    assert {"gemm_fma<16,0>", "gemm_fma<32,0>", "gemm_fma<128,0>"} <= set(k.instances(launched=True))
    if values == "ordinary":            # gated: silu(gate) up of both products' bits
        half = N // 2
        gate, up = want[:, :half], want[:, half:2 * half]
        for m in (140, 128, 20, 7):
            out = torch.full((m, half), float("nan"), device="cuda")
            k.gemm(x[:m], w[:2 * half], out, None, MODE_SWIGLU)
            act = torch.empty_like(out)
            k.swiglu(torch.cat([gate, up], 1)[:m].contiguous(), act)
            assert torch.equal(out, act), m


@pytest.mark.parametrize("N,K", [(1030, 516), (2570, 1060), (4100, 292), (300, 545)])
def test_columns_a_block_and_rounds_of_chains(N, K):
    """Blocks of 4, 5, 8, 9, 11 and 16 columns, the last one short, and K of whole and broken rounds of chains."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(N)
    x, w = torch.randn(64, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    want = _by_chains(k, x, w)
    for m in (1, 16, 17, 33, 64):
        out = torch.full((m, N + 3), float("nan"), device="cuda")
        k.gemm(x[:m], w, out[:, :N], None, MODE_STORE_F32)
        assert torch.equal(out[:, :N], want[:m]) and bool(out[:, N:].isnan().all()), m
    gate, up, half = want[:, :N // 2], want[:, N // 2:2 * (N // 2)], N // 2
    for m in (3, 20, 64):
        out, act = (torch.full((m, half), float("nan"), device="cuda") for _ in range(2))
        k.gemm(x[:m], w[:2 * half], out, None, MODE_SWIGLU)
        k.swiglu(torch.cat([gate, up], 1)[:m].contiguous(), act)
        assert torch.equal(out, act), m


@pytest.mark.parametrize("N,K", [(1030, 224), (2570, 64), (4100, 128), (300, 256), (5640, 33), (16390, 8)])
def test_columns_a_block_of_few_chains(N, K):
    test_columns_a_block_and_rounds_of_chains(N, K)


@pytest.mark.parametrize("K", [4, 28, 32, 60, 64, 96, 124, 128, 132, 160, 188, 192, 224, 228, 1056])
def test_tiles_at_every_end_of_k(K):
    """Whole and broken last steps of K behind fewer and more stages than LDS holds, rows and columns past the end, and rows of X
    with numbers that are none behind K: the bits of chains of fmaf."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(K)
    M, N = 201, 150
    x = torch.full((M + 1, K + 4), float("nan"), device="cuda")
    x[:M, :K] = torch.randn(M, K, generator=g, device="cuda")
    w = torch.randn(N, K, generator=g, device="cuda")
    want = _by_chains(k, x[:M, :K], w)
    out = torch.full((M + 1, N + 2), float("nan"), device="cuda")
    k.gemm(x[:M, :K], w, out[:M, :N], None, MODE_STORE_F32)
    assert torch.equal(out[:M, :N], want) and bool(out[M:].isnan().all()) and bool(out[:, N:].isnan().all())
    half = N // 2
    got, act = (torch.full((M, half), float("nan"), device="cuda") for _ in range(2))
    k.gemm(x[:M, :K], w, got, None, MODE_SWIGLU)
    k.swiglu(want[:, :2 * half].contiguous(), act)
    assert torch.equal(got, act)


@pytest.mark.parametrize("N,K,flows", [(150, 128, False), (150, 188, False), (150, 192, True), (150, 193, False), (150, 196, True), (150, 320, True),
                                       (8150, 260, True), (8200, 260, False), (8200, 636, False), (8200, 640, True)])
def test_short_and_long_k_have_their_kernels(N, K, flows):
    """Up to 512 blocks of 64 rows and columns direct loads pay from a K of 192 on, with more of them from 640: the same bits on
    both sides of the lines."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(N + K)
    x, w = torch.randn(220, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    out = torch.full((220, N), float("nan"), device="cuda")
    k.reset_instances()
    k.gemm(x, w, out, None, MODE_STORE_F32)
    assert ("gemm_fma_flow<0>" in k.instances(launched=True)) == flows and "gemm_fma<128,0>" in k.instances(launched=True)
    assert torch.equal(out, _by_chains(k, x, w))


def test_rows_far_apart():
    """Sixteen rows of X that lie 2^32 numbers from the first to the last."""
    k, K, stride = kernels("bfloat16"), 301, 2 ** 32 // 15 + 1
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(16, K, generator=g, device="cuda").bfloat16(), torch.randn(40, K, generator=g, device="cuda").bfloat16()
    far = torch.empty(15 * stride + K, dtype=torch.bfloat16, device="cuda").as_strided((16, K), (stride, 1))
    far.copy_(x)
    got, want = (torch.full((16, 40), float("nan"), device="cuda") for _ in range(2))
    k.gemm(far, w, got, None, MODE_STORE_F32)
    k.gemm(x, w, want, None, MODE_STORE_F32)
    assert torch.equal(got, want)


@pytest.mark.parametrize("K", [192, 196, 204, 216, 220, 224, 232, 252, 256, 284, 316, 320, 1052])
def test_direct_loads_at_every_end_of_k(K):
    """The same for a K that the tiles take by direct loads."""
    k = kernels("float32")
    k.reset_instances()
    test_tiles_at_every_end_of_k(K)
    assert {"gemm_fma_flow<0>", "gemm_fma_flow<1>"} <= set(k.instances(launched=True))


@pytest.mark.parametrize("M,N,K,rows,gated", [(129, 2048, 644, 32, 32), (97, 2560, 512, 32, None), (300, 2050, 192, 48, 32), (626, 2048, 228, 80, 96),
                                              (777, 2560, 644, 32, 32), (1500, 2048, 640, 96, 96), (64, 8200, 516, 32, 32), (65, 4100, 512, 32, 32),
                                              (1025, 1000, 196, 80, 96), (896, 2048, 644, 64, 64), (777, 11264, 644, 80, 64)])
def test_rows_a_block_by_what_the_cus_get(M, N, K, rows, gated):
    """Tiles of 32, 48, 64, 80 and 96 rows, the last ones of a product among them: the bits of chains of fmaf."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    out = torch.full((M + 1, N), float("nan"), device="cuda")
    k.reset_instances()
    k.gemm(x, w, out[:M], None, MODE_STORE_F32)
    assert {"gemm_fma_flow<0>", f"gemm_fma_flow_rows<{rows},0>"} <= set(k.instances(launched=True))
    want = _by_chains(k, x, w)
    assert torch.equal(out[:M], want) and bool(out[M:].isnan().all())
    half = N // 2
    got, act = (torch.full((M, half), float("nan"), device="cuda") for _ in range(2))
    k.gemm(x, w[:2 * half], got, None, MODE_SWIGLU)
    assert gated is None or f"gemm_fma_flow_rows<{gated},1>" in k.instances(launched=True)         # (None: too few outputs for tiles)
    k.swiglu(want[:, :2 * half].contiguous(), act)
    assert torch.equal(got, act)


@pytest.mark.parametrize("M,N,least,rows,gated", [(129, 2048, 192, 32, 32), (300, 2050, 192, 48, 32), (896, 2048, 192, 64, 64), (626, 2048, 192, 80, 96),
                                                  (1500, 2048, 640, 96, 96)])
def test_every_height_at_every_end_of_k(M, N, least, rows, gated):
    """Whole and broken last steps, an odd and an even number of them."""
    k = kernels("float32")
    g = torch.Generator(device="cuda").manual_seed(rows)
    for K in range(least, least + 68, 4):
        x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
        out, act, got = (torch.full((M, n), float("nan"), device="cuda") for n in (N, N // 2, N // 2))
        k.reset_instances()
        k.gemm(x, w, out, None, MODE_STORE_F32)
        k.gemm(x, w[:N // 2 * 2], got, None, MODE_SWIGLU)
        assert {f"gemm_fma_flow_rows<{rows},0>", f"gemm_fma_flow_rows<{gated},1>"} <= set(k.instances(launched=True))
        want = _by_chains(k, x, w)
        k.swiglu(want[:, :N // 2 * 2].contiguous(), act)
        assert torch.equal(out, want) and torch.equal(got, act), K
