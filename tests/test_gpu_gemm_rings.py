"""Products whose stages (64 of the reduced dimension) fill the ring of a lone tile not at all, once and several times, weights
either way round; and rows too far apart for the tile kernels' 32-bit offsets.  Bound: one bf16 rounding,
2^-9 of the value, and 0.5e-3 for the fp32 sums."""
import pytest
import torch

from gpu_util import check, library, stream, sync

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def product(x, w, transposed):
    (M, K), N, lib = x.shape, w.shape[0], library()
    weight = w.t().contiguous() if transposed else w
    y = torch.full((M, N), float("nan"), device="cuda", dtype=BF16)
    fn = lib.tgk_gemm_fwd_t if transposed else lib.tgk_gemm_fwd
    check(fn(stream(), M, N, K, x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), y.data_ptr(), N, None, 0, None, 0))
    sync()
    return y


def relative(a, b):
    return float((a.double() - b).norm() / b.norm())


# lone 64 x 64 tiles: a ring of four, from 5 stages on two groups of waves with three each, from 16 on with four
@pytest.mark.parametrize("M,N,stages", [(256, 128, s) for s in (2, 4, 6, 7, 8, 10, 11, 15, 16, 17, 23)] + [(1024, 2048, s) for s in (15, 16, 17, 19)])
def test_turns_of_the_ring(M, N, stages):
    K = 64 * stages
    gen = torch.Generator(device="cuda").manual_seed(stages)
    x = torch.randn(M, K, device="cuda", generator=gen).to(BF16)
    w = (torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5).to(BF16)
    y = product(x, w, False)
    assert relative(y, x.double() @ w.double().t()) < 2.5e-3
    assert torch.equal(y, product(x, w, True))


@pytest.mark.parametrize("transposed", (False, True))
@pytest.mark.parametrize("stages", (5, 6, 7, 16))
def test_order_of_two_groups(stages, transposed):
    """From five stages on a lone 64 x 64 tile is two sums, of its first half of the stages (the odd one with it) and of the rest.
    A 1 in the first half outlives 2^30 and -2^30 in two stages of the second; in one chain it would be lost (an ulp is 64)."""
    M, N, K, half = 256, 128, 64 * stages, 64 * ((stages + 1) // 2)
    x, w = (torch.zeros(n, K, device="cuda", dtype=BF16) for n in (M, N))
    x[:, 3] = w[:, 3] = 1
    x[:, half + 8], w[:, half + 8] = 2.0 ** 15, 2.0 ** 15
    x[:, half + 72], w[:, half + 72] = 2.0 ** 15, -(2.0 ** 15)
    assert (product(x, w, transposed) == 1).all()


def test_far_rows():
    M, N, K, ld = 128, 128, 128, (1 << 23) + 64
    gen = torch.Generator(device="cuda").manual_seed(1)
    memory = torch.zeros((M - 1) * ld + K, device="cuda", dtype=BF16)
    x = memory.as_strided((M, K), (ld, 1))
    x.copy_(torch.randn(M, K, device="cuda", generator=gen))
    w = (torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5).to(BF16)
    assert relative(product(x, w, False), x.double() @ w.double().t()) < 2.5e-3


# Lone tiles of 128 x 96 (192 to 256 of them), whose waves lie one above the other: every epilogue and strides of their own,
# bit for bit what the k-strided weight's tiles of another shape give.
@pytest.mark.parametrize("stages", (1, 3, 4, 5, 12))
@pytest.mark.parametrize("M,N", [(1024, 2304), (1024, 3072), (4096, 768), (8192, 384)])
@pytest.mark.parametrize("mode", ("plain", "residual", "gelu"))
def test_waves_one_above_the_other(M, N, stages, mode):
    K, ldy = 64 * stages, N + 64
    gen = torch.Generator(device="cuda").manual_seed(stages)
    x = torch.randn(M, K + 8, device="cuda", generator=gen).to(BF16)[:, :K]
    w = (torch.randn(N, K + 16, device="cuda", generator=gen) * K ** -0.5).to(BF16)[:, :K]
    wt = w.t().contiguous()
    residual = torch.randn(M, N + 8, device="cuda", generator=gen).to(BF16)[:, :N]
    want = x.double() @ w.double().t()
    if mode == "residual":
        want = want.to(BF16).double() + residual.double()
    outputs = []
    for fn, weight in ((library().tgk_gemm_fwd, w), (library().tgk_gemm_fwd_t, wt)):
        y = torch.full((M, ldy), float("nan"), device="cuda", dtype=BF16)
        g = torch.full((M, ldy), float("nan"), device="cuda", dtype=BF16)
        r = (residual.data_ptr(), residual.stride(0)) if mode == "residual" else (None, 0)
        second = (g.data_ptr(), ldy) if mode == "gelu" else (None, 0)
        check(fn(stream(), M, N, K, x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), y.data_ptr(), ldy, *r, *second))
        sync()
        assert y[:, N:].isnan().all() and g[:, N:].isnan().all()
        outputs.append((y[:, :N], g[:, :N]))
    (y, g), (yt, gt) = outputs
    assert relative(y, want) < 4e-3  # two bf16 roundings where there is a residual
    assert torch.equal(y, yt)
    if mode == "gelu":
        assert torch.equal(g, gt) and not g.isnan().any()
