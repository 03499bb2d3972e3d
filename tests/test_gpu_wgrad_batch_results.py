"""Several weight gradients in one launch (csrc/gemm.hip, wgrad_batch_kernel) of fewer and more tiles than there are blocks, over few and
many tokens: its results leave past the caches or through them."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_util import stream, sync
from test_gpu_gemm import run_wgrad_batch
from turbogpt_amd.bridge import check, library

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,shapes", [
    (128, [(4608, 4608)]), (960, [(4608, 4608)]), (1024, [(4608, 4608)]),  # 864 tiles: past the caches, past, through
    (1024, [(4096, 3072)]), (1024, [(4096, 3072), (128, 192)]),            # 512 tiles, a block each: past; one more: through
    (1152, [(1152, 4608), (4608, 1152), (1152, 1152), (3456, 1152)]),      # 648: blocks with a second tile, cut or whole
])
def test_against_a_product_in_fp64(M, shapes):
    """Every element: a sum of M products of unit variance, whose fp32 roundings of 2^-24 of some sqrt(M) add up to sqrt(M) of them,
    M 2^-24; within eight times that.  A second launch that accumulates doubles it."""
    lib = library()
    keep, _, (jobs, ws, need) = run_wgrad_batch(M, shapes, np.random.default_rng(M), start=7.0)
    firsts = []
    for dy, x, dw in keep:
        want = dy.double().t().contiguous() @ x.double()
        assert float((dw - want).abs().max()) < 8 * M * 2**-24
        firsts.append(dw.clone())
    check(lib.tgk_gemm_wgrad_batch(stream(), M, len(shapes), C.addressof(jobs), 1, ws.data_ptr(), need))
    sync()
    for (_, _, dw), first in zip(keep, firsts):
        assert torch.allclose(dw, 2 * first, rtol=1e-6, atol=0)
