"""Products of few tiles (csrc/gemm.hip, gemm_waves_kernel: 32 x 32 up to 64 tiles of 64 x 64, 32 x 64 up to 128), at the edges:
one stage less than a ring, a full ring and one more, odd tile counts, the tile counts and depths on both sides of each line; with
the checks and bounds of test_gpu_gemm_tiles.py, weights either way round bit for bit."""
import pytest
import torch

import test_gpu_gemm_tiles as tiles
from test_gpu_gemm_rings import BF16, product

pytestmark = tiles.pytestmark


@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (128, 192, 128), (128, 384, 192), (256, 256, 256),  # 64 x 64
                                   (128, 128, 320), (128, 384, 384),   # the shortest: three stages and two, three and three
                                   (512, 512, 512),    # 64 tiles, four stages a wave: the ring of four
                                   (512, 512, 576),    # one half has a fifth
                                   (384, 192, 960), (512, 512, 1088), (128, 128, 4096),
                                   (128, 2048, 448), (128, 2112, 448),  # 64 tiles of 64 x 64, and 66: on 32 x 64, odd columns
                                   (512, 512, 832), (1408, 192, 832),   # the same, thirteen stages, many rows and few columns
                                   (640, 576, 320), (384, 768, 832),    # 90 and 72 tiles
                                   (2048, 256, 64), (2048, 256, 256), (2048, 256, 320), (2048, 256, 832), (1024, 512, 3072),
                                   (128, 4224, 320),   # 132 tiles, the next after 128: the two groups of waves
                                   (128, 4096, 832), (128, 4224, 832)])
def test_few_tiles(M, N, K):
    tiles.test_every_tile_with_every_epilogue(M, N, K)


@pytest.mark.parametrize("M,N,K", [(128, 128, 320), (512, 512, 832), (2048, 256, 320), (384, 768, 960)])
@pytest.mark.parametrize("transposed", (False, True))
def test_halves_are_the_two_groups(M, N, K, transposed):
    """The same rows within a product of 129 to 256 tiles, where two groups of waves take the halves: the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(K)
    often = 256 // (M // 64 * (N // 64))
    x = torch.randn(M * often, K, device="cuda", generator=gen).to(BF16)
    w = (torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5).to(BF16)
    assert torch.equal(product(x[:M], w, transposed), product(x, w, transposed)[:M])
