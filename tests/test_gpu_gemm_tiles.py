"""Every tile that choose_block (csrc/gemm.hip) can take, at the edges of its range: one 64-k stage and fewer stages than
the ring holds, odd stage counts, tile counts that 8 does not divide, one, two and more tiles a compute unit; weights
either way round (bit-identical), and all four epilogues.  Bounds: a bf16 rounding is at most 2^-9 of the value, so one
rounding 2.0e-3 in relative L2 and two 4.0e-3, plus 0.5e-3 for fp32 sums and the GELU approximation."""
import pytest
import torch

from gpu_util import check, library, stream, sync

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16
SHAPES = [(128, 128, 64),      # 64 x 64: 4 tiles, one stage
          (384, 640, 192),     # 64 x 64: 60 tiles, three stages
          (1920, 640, 128),    # 64 x 64: 300 tiles, two on some units
          (128, 192, 576),     # 6 of 64 x 64 as 32 x 32, nine stages: a width 128 does not divide
          (640, 640, 320),     # 100 of 64 x 64, [N][K] as 32 x 64, [K][N] on two groups of waves: five stages
          (128, 128, 2048),    # 4 of 64 x 64 as 32 x 32, 32 stages
          (1024, 2304, 64),    # weights [N][K] on 192 tiles of 128 x 96, [K][N] on 288 of 64 x 128: one stage
          (1152, 1920, 320),   # the same, 180 and 270 tiles, five stages
          (1920, 1920, 64),    # 64 x 128: 450 tiles, one stage
          (1920, 1920, 448),   # 64 x 128: 450 tiles, seven stages
          (16384, 384, 192),   # 128 x 128, two stages in flight
          (16384, 640, 64),    # the same, GELU outputs that the caches do not hold
          (16384, 2944, 64),   # 128 x 128, the persistent kernel: more than ten tiles a unit
          (8192, 2688, 64)]    # 128 x 192


def relative(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def gelu(x):
    return torch.nn.functional.gelu(x)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_every_tile_with_every_epilogue(M, N, K):
    lib = library()
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, device="cuda", generator=gen).to(BF16)
    w = (torch.randn(N, K, device="cuda", generator=gen) * K ** -0.5).to(BF16)
    wt = w.t().contiguous()
    r = torch.randn(M, N, device="cuda", generator=gen).to(BF16)
    product = x.double() @ w.double().t()
    y, a = (torch.full((M, N), float("nan"), device="cuda", dtype=BF16) for _ in range(2))

    def both_ways(run, direct, transposed):
        outs = []
        for fn, weight, ld in ((direct, w, K), (transposed, wt, N)):
            y.fill_(float("nan"))
            a.fill_(float("nan"))
            check(run(fn, weight.data_ptr(), ld))
            sync()
            outs.append((y.clone(), a.clone()))
        assert torch.equal(outs[0][0], outs[1][0])
        return outs[0]

    def forward(residual=None, gelu_out=None):
        def run(fn, weight, ld):
            return fn(stream(), M, N, K, x.data_ptr(), K, weight, ld, y.data_ptr(), N,
                      residual.data_ptr() if residual is not None else None, N if residual is not None else 0,
                      gelu_out.data_ptr() if gelu_out is not None else None, N if gelu_out is not None else 0)
        return both_ways(run, lib.tgk_gemm_fwd, lib.tgk_gemm_fwd_t)

    got, _ = forward()
    assert relative(got, product) < 2.5e-3
    got, _ = forward(residual=r)
    assert relative(got, product + r.double()) < 4.5e-3
    pre, act = forward(gelu_out=a)
    assert relative(pre, product) < 2.5e-3 and relative(act, gelu(pre.double())) < 2.5e-3
    # the input gradient of a layer whose [Out][In] weight is wt (Out = K, In = N), times GELU' of a saved pre-activation
    u = r.double().requires_grad_()
    slope, = torch.autograd.grad(gelu(u).sum(), u)

    def dgrad(fn, weight, ld):
        return fn(stream(), M, K, N, x.data_ptr(), K, weight, ld, y.data_ptr(), N, r.data_ptr(), N)
    got, _ = both_ways(dgrad, lib.tgk_gemm_dgrad_t, lib.tgk_gemm_dgrad)
    assert relative(got, product * slope) < 4.5e-3
