"""LayerNorm backward where a block's eight rows go to eight waves (up to 2048 rows) or to four, and one row past eight
a block.  Bounds: dx one bf16 rounding (2^-9 of
the value) and 0.5e-3; dgamma and dbeta 1e-5, fp32 sums of at most 6200 rows of exact products."""
import pytest
import torch

from gpu_util import check, library, stream, sync

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def relative(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("M,D", [(1, 64), (7, 640), (9, 512), (6144, 128), (6145, 128), (6145, 576)])
def test_rows_of_a_block(M, D):
    lib = library()
    gen = torch.Generator(device="cuda").manual_seed(M + D)
    x, dy = (torch.randn(M, D, device="cuda", generator=gen).to(BF16) for _ in range(2))
    gamma = torch.randn(D, device="cuda", generator=gen).to(BF16)
    low = torch.zeros(D, device="cuda", dtype=torch.uint16)
    dx = torch.full_like(x, float("nan"))
    dg, db = (torch.full((D,), float("nan"), device="cuda") for _ in range(2))
    workspace = torch.empty(lib.tgk_layernorm_bwd_workspace(M, D), device="cuda", dtype=torch.uint8)
    check(lib.tgk_layernorm_bwd_add(stream(), M, D, x.data_ptr(), dy.data_ptr(), gamma.data_ptr(), low.data_ptr(), None,
                                    dx.data_ptr(), dg.data_ptr(), db.data_ptr(), 1e-5, 0, workspace.data_ptr(), workspace.numel()))
    sync()
    leaves = [t.double().requires_grad_() for t in (x, gamma, torch.zeros_like(gamma))]
    y = torch.nn.functional.layer_norm(leaves[0], (D,), leaves[1], leaves[2], 1e-5)
    want = torch.autograd.grad(y, leaves, dy.double())
    assert relative(dx, want[0]) < 2.5e-3
    assert relative(dg, want[1]) < 1e-5 and relative(db, want[2]) < 1e-5


@pytest.mark.parametrize("M,D", [(8, 64), (24, 512), (2048, 640), (2056, 640), (6144, 128), (8, 576), (40, 1024), (8, 1536)])
def test_order_of_a_blocks_rows(M, D):
    """Slot s of the first block adds row s, then row s + M / 2; only then come the slots together.  Row 0 and row M / 2 carry
    2^30 and -2^30, which cancel in that order alone: with any other row between them, its 1 (an ulp there is 64) is lost."""
    lib = library()
    gen = torch.Generator(device="cuda").manual_seed(M + D)
    x = torch.randn(1, D, device="cuda", generator=gen).to(BF16).repeat(M, 1)
    gamma = torch.ones(D, device="cuda", dtype=BF16)
    low = torch.zeros(D, device="cuda", dtype=torch.uint16)
    dy = torch.zeros(M, D, device="cuda", dtype=BF16)
    dy[0], dy[M // 2], dy[1] = 2.0 ** 30, -(2.0 ** 30), 1.0
    dx = torch.empty_like(x)
    dg, db = (torch.empty(D, device="cuda") for _ in range(2))
    workspace = torch.empty(lib.tgk_layernorm_bwd_workspace(M, D), device="cuda", dtype=torch.uint8)
    check(lib.tgk_layernorm_bwd_add(stream(), M, D, x.data_ptr(), dy.data_ptr(), gamma.data_ptr(), low.data_ptr(), None,
                                    dx.data_ptr(), dg.data_ptr(), db.data_ptr(), 1e-5, 0, workspace.data_ptr(), workspace.numel()))
    sync()
    z = torch.nn.functional.layer_norm(x[0].double(), (D,), None, None, 1e-5)
    assert (db == 1).all()
    assert relative(dg, z) < 1e-5  # z in fp32: a mean and a variance over D values
