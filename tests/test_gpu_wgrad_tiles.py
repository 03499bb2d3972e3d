"""Weight gradients on 64 x 64 and 128 x 128 tiles (wgrad_tiles_kernel through tgk_gemm_wgrad, csrc/gemm.hip): fewer 64-token
stages than the ring holds, odd counts, tile counts that 8 does not divide and more than the compute units, token ranges
that are folded, operands and gradient that are column slices, accumulation.  fp32 sums of at most 16384 exact bf16
products (2^-24 a partial sum): 1e-5 in relative L2."""
import ctypes as C

import pytest
import torch

from gpu_util import check, library, stream, sync
from turbogpt_amd.bridge import WgradJob

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
                                       (16384, 768, 3072, 0),  # the persistent kernel
                                       (4096, 512, 4096, 0),  # the same: few rows of tiles, a wide X
                                       (16384, 2304, 768, 8)])
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


@pytest.mark.parametrize("M,N,K", [(16384, 2304, 2304), (12288, 1920, 2304)])
def test_wide_gradient_is_no_slower_than_a_batch_of_one(M, N, K):
    """Where every XCD would read nearly all of X, tiles lose to the persistent kernel (242 against 173 us and 154 against 124).
    tgk_gemm_wgrad_batch runs the same product persistently, so it tells the two apart: the shortest of twenty, 15 % for the
    kernels' own difference."""
    lib = library()
    dy, x, dw = operands(M, N, K, torch.Generator(device="cuda").manual_seed(M))
    job = (WgradJob * 1)(WgradJob(N, K, dy.data_ptr(), N, x.data_ptr(), K, dw.data_ptr(), K))
    at = C.addressof(job)
    need = max(lib.tgk_gemm_wgrad_workspace(M, N, K), lib.tgk_gemm_wgrad_batch_workspace(M, 1, at))
    workspace = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    calls = [lambda: lib.tgk_gemm_wgrad(stream(), M, N, K, dy.data_ptr(), N, x.data_ptr(), K, dw.data_ptr(), K, 0,
                                        workspace.data_ptr(), need),
             lambda: lib.tgk_gemm_wgrad_batch(stream(), M, 1, at, 0, workspace.data_ptr(), need)]
    shortest = [float("inf")] * 2
    for _ in range(20):
        for i, call in enumerate(calls):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            check(call())
            end.record()
            sync()
            shortest[i] = min(shortest[i], begin.elapsed_time(end))
    print(f"{M} tokens, {N} x {K}: alone {shortest[0] * 1e3:.1f} us, batch of one {shortest[1] * 1e3:.1f} us", flush=True)
    assert shortest[0] < 1.15 * shortest[1]


def fold_bound(tokens):
    """Relative rms error of fp32 sums over `tokens` products: the matrix instruction adds eight at a time, 24 such steps make a
    partial sum (three stages of 64) and the partial sums are added in turn.  A rounding is uniform within half an ulp, 0.416 *
    2^-24 of the value in the mean square; n steps of a random walk add up to sqrt(n / 2) of it.  15 % on top."""
    return 1.15 * 0.416 * 2 ** -24 * (24 / 2 + -(-tokens // 192) / 2) ** 0.5


def distance(dw, dy, x):
    want = dy.double().t().contiguous() @ x.double()
    return float((dw.double() - want).norm() / want.norm())


def operands(M, N, K, gen):
    return (torch.randn(M, N, device="cuda", generator=gen).bfloat16(), torch.randn(M, K, device="cuda", generator=gen).bfloat16(),
            torch.full((N, K), float("nan"), device="cuda"))


@pytest.mark.parametrize("M,N,K", [(512, 3072, 768), (1024, 128, 2048), (1920, 640, 1920), (4096, 1024, 1024), (8192, 896, 896),
                                   (16384, 256, 1024)])
def test_single_gradient_against_64_bits(M, N, K):
    lib = library()
    dy, x, dw = operands(M, N, K, torch.Generator(device="cuda").manual_seed(M + N + K))
    need = lib.tgk_gemm_wgrad_workspace(M, N, K)
    workspace = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    check(lib.tgk_gemm_wgrad(stream(), M, N, K, dy.data_ptr(), N, x.data_ptr(), K, dw.data_ptr(), K, 0, workspace.data_ptr(), need))
    sync()
    assert distance(dw, dy, x) < fold_bound(M)


@pytest.mark.parametrize("M,d,ffn,depth", [(1024, 256, 1024, 4), (2048, 512, 2048, 4)])
def test_list_against_64_bits(M, d, ffn, depth):
    lib = library()
    gen = torch.Generator(device="cuda").manual_seed(M + d)
    shapes = [(d, ffn), (ffn, d), (d, d), (3 * d, d)] * depth + [(256, d)] * 2
    matrices = [operands(M, N, K, gen) for N, K in shapes]
    jobs = (WgradJob * len(shapes))(*[WgradJob(N, K, dy.data_ptr(), N, x.data_ptr(), K, dw.data_ptr(), K)
                                      for (N, K), (dy, x, dw) in zip(shapes, matrices)])
    at = C.addressof(jobs)
    table_bytes, need = (f(M, len(shapes), at) for f in (lib.tgk_gemm_wgrad_list_table_bytes, lib.tgk_gemm_wgrad_list_workspace))
    table, workspace = (torch.empty(max(n, 16), dtype=torch.uint8, device="cuda") for n in (table_bytes, need))
    check(lib.tgk_gemm_wgrad_list_prepare(M, len(shapes), at, table.data_ptr(), table_bytes))
    check(lib.tgk_gemm_wgrad_list(stream(), M, len(shapes), at, table.data_ptr(), 0, workspace.data_ptr(), need, None))
    sync()
    for dy, x, dw in matrices:
        assert distance(dw, dy, x) < fold_bound(M)
