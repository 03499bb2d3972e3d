"""Products on 96 x 64 and 64 x 96 tiles (csrc/gemm.hip, gemm_uneven_kernel): 257 to 384 tiles of 64 x 64 from five stages on; and on
128 x 64: 449 to 512 from 24 stages on.  At the edges of the ring, of the tile counts and of those depths; with the checks and
bounds of test_gpu_gemm_tiles.py, weights either way round, and bit for bit the rows of a larger product on other tiles."""
import pytest
import torch

import test_gpu_gemm_tiles as tiles
from test_gpu_gemm_rings import BF16, product

pytestmark = tiles.pytestmark
SHAPES = [(1920, 640, 256), (1920, 640, 320), (1920, 640, 384), (1152, 1152, 704),  # 4 stages: 64 x 64; 5, 6 and 11
          (1152, 960, 1472), (2304, 640, 1600),
          (2048, 768, 320), (1024, 1536, 1600),   # 64 x 96, a tile on every unit
          (1408, 768, 640),                       # 64 x 96, 176 tiles
          (2432, 640, 640),                       # neither: 380 tiles of 64 x 64
          (2048, 1024, 1472), (2048, 1024, 1536), (1920, 1024, 1600),  # 128 x 64: 256 tiles and 240
          (1792, 1024, 1536)]                     # 448: 64 x 64


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_uneven_tiles(M, N, K):
    tiles.test_every_tile_with_every_epilogue(M, N, K)


@pytest.mark.parametrize("M,N,K", [(1920, 640, 320), (1152, 960, 1600), (2048, 768, 1536), (2048, 1024, 1536)])
@pytest.mark.parametrize("transposed", (False, True))
def test_order_of_the_sums(M, N, K, transposed):
    gen = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(M * 4, K, device="cuda", generator=gen).to(BF16)
    w = (torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5).to(BF16)
    assert torch.equal(product(x[:M], w, transposed), product(x, w, transposed)[:M])
