"""Products on 256-row tiles (csrc/gemm.hip, gemm256_kernel) of each width, at the edges of its choice: a round that is partly
filled, several rounds, odd numbers of 128-k periods, a reduced dimension that only the GELU epilogues take, half a tile of rows at
the end; with the checks and bounds of test_256x128_tiles_rows_sampled, bit for bit against the kernels for k-strided weights."""
import pytest

import test_gpu_gemm as gemm

pytestmark = gemm.pytestmark


@pytest.mark.parametrize("M,N,K,residual", [(10240, 1024, 1152, True),   # 160 tiles of 256 columns; backward: 240 of 192
                                          (4096, 3584, 896, False),    # 224 tiles of 256 columns; backward on 128 x 128 blocks
                                          (16384, 3072, 1024, False),  # 768 tiles of 256 columns
                                          (12288, 768, 896, True),     # 192 tiles of 192 columns; backward on 128-row blocks
                                          (10240, 640, 768, False),    # 200 tiles of 128 columns
                                          (16384, 1024, 640, True),    # only with a GELU; backward: 320 of 128
                                          (16640, 1280, 1024, False),  # 65 rows of tiles: 650 of 128 columns
                                          # a last row of tiles of 128 rows
                                          (8320, 896, 896, True), (12416, 768, 768, False), (10368, 1024, 1152, True),
                                          (4224, 3072, 768, True)])
def test_columns(orc, M, N, K, residual):
    gemm.test_256x128_tiles_rows_sampled(orc, M, N, K, residual)
