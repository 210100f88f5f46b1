"""Which tiles a product of more than 128 rows takes, on both sides of where the choice changes, and that a row's bits do not
depend on it: the same rows alone, through the kernels of few rows and those of tiles of another size."""
import pytest
import torch

from axon_amd.kernels import MODE_ADD_F32, MODE_STORE, MODE_SWIGLU, kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,mode,tiles", [
    (1000, 3968, 2112, MODE_STORE, "gemm_kept<0>"),                       # 248 blocks of a K beyond 2,048
    (1660, 2432, 2112, MODE_STORE, "gemm_tile<128,128,2,2,0,2>"),         # 247
    (1000, 3960, 8192, MODE_ADD_F32, "gemm_kept<0>"),                     # the longest K of one round, a ragged edge
    (257, 3072, 8192, MODE_SWIGLU, "gemm_kept<1>"),                       # gated, four segments: up to 8,192
    (257, 3072, 8256, MODE_SWIGLU, "gemm_tile<256,256,4,2,1,2>"),
    (256, 3072, 8192, MODE_SWIGLU, "gemm_tile<128,128,2,2,1,2>"),
    (385, 18944, 512, MODE_SWIGLU, "gemm_tile<256,256,4,2,1,2>"),         # four rounds of the small tiles for two of the large
    (513, 5120, 13824, MODE_ADD_F32, "gemm_tile<256,256,4,2,0,2>"),
    (513, 3840, 13824, MODE_ADD_F32, "gemm_tile<256,256,4,2,0,2>"),
    (300, 3584, 13824, MODE_ADD_F32, "gemm_tile<128,128,2,2,0,2>"),
])
def test_the_tiles_and_the_bits(M, N, K, mode, tiles):
    k = kernels("bfloat16")
    gated = mode == MODE_SWIGLU
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = k.prepare_weight((torch.randn((1 + gated) * N, K, generator=g, device="cuda") * 0.05).bfloat16(), gated)
    base = torch.randn(M, N, generator=g, device="cuda").to(torch.float32 if mode == MODE_ADD_F32 else torch.bfloat16)
    whole = base.clone()
    k.reset_instances()
    k.gemm(x, w, whole, None, mode)
    assert tiles in k.instances(launched=True), k.instances(launched=True)
    for first, m in ((0, 16), (M - 64, 64), (M // 2, 100), (3, 150)):
        part = base[first:first + m].clone()
        k.gemm(x[first:first + m].contiguous(), w, part, None, mode)
        assert torch.equal(part, whole[first:first + m]), (first, m)
