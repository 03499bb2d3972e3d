"""Products on 256-row tiles (csrc/gemm.hip, gemm256_kernel) of more tiles than there are units, with half a tile of rows at the end: a unit
goes on from a whole tile to a half one and from one half to the next, behind an epilogue or without one, on every width and with every
epilogue.  The forms that these shapes are given stand in test_launch_rules.py."""
import pytest

import test_gpu_evaluate as evaluate
import test_gpu_gemm as gemm

pytestmark = gemm.pytestmark

# forward N x K, its mirror image the input gradient K x N
PLAIN = [(1408, 6016, 896, 128), (2176, 8832, 768, 192), (2688, 9472, 768, 256)]
GELU = [(2688, 4736, 768, 128), (3456, 8704, 512, 256)]
GELU_BACKWARD = [(1408, 768, 9856, 128), (2176, 1024, 8832, 192), (2944, 512, 9984, 256)]


@pytest.mark.parametrize("residual", [False, True])
@pytest.mark.parametrize("M,N,K,columns", PLAIN)
def test_plain_and_residual(orc, M, N, K, columns, residual):
    gemm.test_256x128_tiles_rows_sampled(orc, M, N, K, residual)


@pytest.mark.parametrize("M,N,K,columns", GELU + GELU_BACKWARD)
def test_gelu(orc, M, N, K, columns):
    gemm.test_256x128_tiles_rows_sampled(orc, M, N, K, False)


@pytest.mark.parametrize("d,ffn,context,batch", [(768, 640, 1024, 10), (768, 4736, 2688, 1),  # 128 columns, a round and two with a half tile
                                                 (512, 8704, 3456, 1)])                       # 256
def test_gelu_alone(d, ffn, context, batch):
    evaluate.test_evaluation_matches_the_batch_with_gradient(d, ffn, context, batch)
