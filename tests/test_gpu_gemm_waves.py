"""Products of few tiles (csrc/gemm.hip, gemm_waves_kernel: 32 x 32 up to 64 tiles of 64 x 64, 32 x 64 up to 128), at the edges:
fewer stages than waves, one more than a round of them, a full ring and one more, odd tile counts, the tile counts on both sides
of each line; with the checks and bounds of test_gpu_gemm_tiles.py, weights either way round bit for bit."""
import pytest

import test_gpu_gemm_tiles as tiles

pytestmark = tiles.pytestmark


@pytest.mark.parametrize("M,N,K", [(128, 128, 64), (128, 192, 128), (128, 384, 192), (256, 256, 256), (128, 128, 320), (384, 192, 960),
                                   (512, 512, 1024),   # 64 tiles, four stages a wave: the ring of four
                                   (512, 512, 1088),   # one wave has a fifth
                                   (128, 128, 4096),
                                   (128, 2112, 448), (640, 448, 128),  # 66 and 70 tiles of 64 x 64: on 32 x 64, odd columns
                                   (384, 704, 832),    # 66 tiles, thirteen stages
                                   (2048, 256, 64), (2048, 256, 768), (2048, 256, 832), (1024, 512, 3072),
                                   (128, 4224, 320)])  # 132 tiles: the two groups of waves
def test_few_tiles(M, N, K):
    if N % 128 and N % 192:
        N = -(-N // 192) * 192
    tiles.test_every_tile_with_every_epilogue(M, N, K)
