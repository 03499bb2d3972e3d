"""Weight gradients on 64 x 64 and 128 x 128 tiles (wgrad_tiles_kernel through tgk_gemm_wgrad, csrc/gemm.hip): fewer 64-token
stages than the ring holds, odd counts, tile counts that 8 does not divide and more than the compute units, token ranges
that are folded, operands and gradient that are column slices, accumulation.  fp32 sums of at most 16384 exact bf16
products (2^-24 a partial sum): 1e-5 in relative L2."""
import pytest
import torch

from gpu_util import check, library, stream, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,pad", [(64, 128, 128, 0),    # one stage, 4 tiles
                                       (128, 128, 192, 8),   # two stages, 6 tiles
                                       (192, 384, 320 + 64, 64),  # three stages, 36 tiles
                                       (320, 640, 640, 0),   # five stages, 100 tiles
                                       (1920, 640, 1920, 8),  # 300 tiles: two on some units
                                       (2048, 256, 256, 8),  # token ranges on 64 x 64 tiles, folded
                                       (4160, 512, 384, 0),  # ranges of different lengths
                                       (16384, 128, 128, 8),  # many ranges of few tiles
                                       (8192, 896, 896, 8),  # 128 x 128 tiles, four stages
                                       (16384, 768, 768, 0),  # the same with two blocks a unit
                                       (16384, 768, 3072, 0)])  # the persistent kernel
def test_single_gradient(M, N, K, pad):
    lib = library()
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    dy = torch.randn(M, N + pad, device="cuda", generator=gen).bfloat16()
    x = torch.randn(M, K + pad, device="cuda", generator=gen).bfloat16()
    want = dy[:, :N].double().t() @ x[:, :K].double()
    need = lib.tgk_gemm_wgrad_workspace(M, N, K)
    workspace = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    dw = torch.full((N, K + pad), float("nan"), device="cuda")
    for accumulate in (0, 1):
        check(lib.tgk_gemm_wgrad(stream(), M, N, K, dy.data_ptr(), N + pad, x.data_ptr(), K + pad, dw.data_ptr(), K + pad,
                                 accumulate, workspace.data_ptr(), need))
        sync()
        got = dw[:, :K].double() / (1 + accumulate)
        assert float((got - want).norm() / want.norm()) < 1e-5
        assert bool(dw[:, K:].isnan().all())  # nothing written beside the gradient
