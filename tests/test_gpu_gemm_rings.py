"""Products whose stages (64 of the reduced dimension) fill the ring of a tile not at all, once and several times, weights
either way round; and rows as far apart as the tile kernels' 32-bit offsets reach, and farther.  Bound: one bf16 rounding,
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


# 192 lone 64 x 64 tiles: a ring of four, from 5 stages on two groups of waves with three each, from 16 on with four; 8 of them, from
# 5 stages on as 32 x 32 tiles whose waves have a ring of four each; and 512, two a unit, on one group with three
@pytest.mark.parametrize("M,N,stages", [(256, 128, s) for s in (2, 4, 6, 7, 8, 10, 11, 15, 16, 17, 23)] +
                         [(1024, 768, s) for s in (4, 5, 7, 15, 16, 17)] + [(1024, 2048, s) for s in (15, 16, 17, 19)])
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
    """From five stages on a lone 64 x 64 tile, also one cut smaller, is two sums, of its first half of the stages (the odd one with it) and of the rest.
    A 1 in the first half outlives 2^30 and -2^30 in two stages of the second; in one chain it would be lost (an ulp is 64)."""
    M, N, K, half = 256, 128, 64 * stages, 64 * ((stages + 1) // 2)
    x, w = (torch.zeros(n, K, device="cuda", dtype=BF16) for n in (M, N))
    x[:, 3] = w[:, 3] = 1
    x[:, half + 8], w[:, half + 8] = 2.0 ** 15, 2.0 ** 15
    x[:, half + 72], w[:, half + 72] = 2.0 ** 15, -(2.0 ** 15)
    assert (product(x, w, transposed) == 1).all()


def strided(rows, cols, ld, gen):
    """A matrix whose rows are `ld` elements apart, in memory that nothing else of is written."""
    matrix = torch.empty((rows - 1) * ld + cols, device="cuda", dtype=BF16).as_strided((rows, cols), (ld, 1))
    return matrix.copy_(torch.randn(rows, cols, device="cuda", generator=gen))


NEAR = 1 << 23  # the largest leading dimension that the tile kernels take
FAR = 34200000  # 63 rows are more than 2^32 bytes: a 32-bit offset would come round inside a tile


@pytest.mark.parametrize("entry", ("fwd", "fwd_t", "dgrad", "dgrad_t"))
@pytest.mark.parametrize("M,N,ld", [(128, 128, FAR), (128, 128, NEAR), (128, 19200, NEAR)])
@pytest.mark.parametrize("far", ("activation", "weight"))
def test_far_rows(entry, M, N, ld, far):
    """C[M][N] over K = 128 by each entry: 4 tiles of 64 x 64, or, where the weight is [N][K], 200 of 128 x 96, whose last row ends
    one row short of 2^31 bytes.  Only the first operand's rows or the second's are far apart."""
    K, lib = 128, library()
    rows = N if entry in ("fwd", "dgrad_t") else K  # of the weight as it is stored
    if far == "weight" and rows > 128:
        pytest.skip("320 GB")
    gen = torch.Generator(device="cuda").manual_seed(1)
    a = strided(M, K, ld if far == "activation" else K, gen)
    b = strided(rows, N + K - rows, ld if far == "weight" else N + K - rows, gen)
    y = torch.full((M, N), float("nan"), device="cuda", dtype=BF16)
    operands = (a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), y.data_ptr(), N, None, 0)
    if entry.startswith("fwd"):
        check((lib.tgk_gemm_fwd if entry == "fwd" else lib.tgk_gemm_fwd_t)(stream(), M, N, K, *operands, None, 0))
    else:  # the layer has N inputs and K outputs
        check((lib.tgk_gemm_dgrad if entry == "dgrad" else lib.tgk_gemm_dgrad_t)(stream(), M, K, N, *operands))
    sync()
    matrix = b.double() if rows == K and entry in ("fwd_t", "dgrad") else b.double().t()
    assert relative(y, a.double() @ matrix) < 2.5e-3


# Lone tiles of 128 x 96 (192 to 256 of them), whose waves lie one above the other: every epilogue and strides of their own,
# bit for bit what the k-strided weight's tiles of another shape give.
# A width that 128 does not divide takes them from 17 stages on.
@pytest.mark.parametrize("M,N,stages", [(M, N, stages) for M, N in ((1024, 2304), (1024, 3072), (4096, 768), (8192, 384))
                                        for stages in (1, 3, 4, 5, 12)] + [(640, 4032, 16), (640, 4032, 17)])
@pytest.mark.parametrize("mode", ("plain", "residual", "gelu", "gelu slope"))
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
    if mode == "gelu slope":  # the input gradient of a layer with N inputs and K outputs: its weight is wt, its transposed copy w
        leaf = residual.double().requires_grad_()
        want = want.to(BF16).double() * torch.autograd.grad(torch.nn.functional.gelu(leaf).sum(), leaf)[0]
    outputs = []
    lib = library()
    for fn, back, weight in ((lib.tgk_gemm_fwd, lib.tgk_gemm_dgrad_t, w), (lib.tgk_gemm_fwd_t, lib.tgk_gemm_dgrad, wt)):
        y = torch.full((M, ldy), float("nan"), device="cuda", dtype=BF16)
        g = torch.full((M, ldy), float("nan"), device="cuda", dtype=BF16)
        r = (residual.data_ptr(), residual.stride(0)) if mode == "residual" else (None, 0)
        second = (g.data_ptr(), ldy) if mode == "gelu" else (None, 0)
        operands = (x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), y.data_ptr(), ldy)
        if mode == "gelu slope":
            check(back(stream(), M, K, N, *operands, residual.data_ptr(), residual.stride(0)))
        else:
            check(fn(stream(), M, N, K, *operands, *r, *second))
        sync()
        assert y[:, N:].isnan().all() and g[:, N:].isnan().all()
        outputs.append((y[:, :N], g[:, :N]))
    (y, g), (yt, gt) = outputs
    assert relative(y, want) < 4.5e-3  # two bf16 roundings where there is a residual or a slope, and 0.5e-3
    assert torch.equal(y, yt)
    if mode == "gelu":
        assert torch.equal(g, gt) and not g.isnan().any()
