"""The 32-bit products on the matrix cores at the sizes where their blocks, chains and rows end: against float64, and a
row's bits whatever the number of rows (which picks the kernel)."""
import pytest
import torch

from axon_amd.kernels import MODE_ADD_F32, MODE_STORE_F32, MODE_SWIGLU, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [MODE_STORE_F32, MODE_ADD_F32, MODE_SWIGLU])
@pytest.mark.parametrize("N,K,x_stride", [(8, 4, 4), (63, 33, 33), (65, 64, 68), (257, 292, 292), (40, 2052, 2055), (4100, 36, 40),
                                           (520, 256, 256), (24, 257, 260), (16390, 40, 44)])
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
