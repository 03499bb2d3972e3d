"""Scores that overflow to -inf, on each of the attention kernels: a tile of 64 keys that is hidden from every row this way
need not be the first that the row sees, but may be the first that one of a 32-row block's waves sees.  Bound as in
test_gpu_attention_split.py."""
import pytest
import torch

from gpu_util import check, library, stream, sync
from test_gpu_attention_split import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,T", [(2, 3, 384),   # 32-row blocks both ways
                                   (29, 5, 128),  # 128-row blocks forward, the backward kernels side by side
                                   (11, 7, 640)])  # 128-row blocks one after the other
def test_tiles_whose_scores_are_all_minus_infinity(B, H, T):
    lib, d = library(), 64 * H
    gen = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(B, T, 3, H, 64, device="cuda", generator=gen).bfloat16()
    do = torch.randn(B * T, d, device="cuda", generator=gen).bfloat16()
    qkv[:, :, 0, :, 0], qkv[:, :, 1, :, 0] = 1e20, 0
    qkv[:, 64:128, 1, :, 0] = qkv[:, 256:320, 1, :, 0] = -1e20  # times 1e20: -inf
    qkv = qkv.view(B * T, 3 * d)
    o = torch.full((B * T, d), float("nan"), device="cuda", dtype=torch.bfloat16)
    lse = torch.full((B, H, T), float("nan"), device="cuda")
    grads = torch.full_like(qkv, float("nan"))
    need = lib.tgk_attn_bwd_workspace(B, H, T)
    workspace = torch.empty(need, dtype=torch.uint8, device="cuda")
    p, g = qkv.data_ptr(), grads.data_ptr()
    check(lib.tgk_attn_fwd(stream(), B, H, T, 64, p, p + 2 * d, p + 4 * d, 3 * d, o.data_ptr(), d, lse.data_ptr(), 0.125))
    check(lib.tgk_attn_bwd(stream(), B, H, T, 64, p, p + 2 * d, p + 4 * d, 3 * d, o.data_ptr(), d, lse.data_ptr(), do.data_ptr(),
                           d, g, g + 2 * d, g + 4 * d, 3 * d, 0.125, workspace.data_ptr(), need))
    sync()
    want, want_lse, want_grads = reference(qkv, do, B, H, T)
    error = lambda got, ref: float((got.float() - ref).norm() / ref.norm())
    assert error(o, want) < 6e-3
    assert float((lse - want_lse).abs().max()) < 1e-4
    for i, name in enumerate("qkv"):
        got, ref = (x.reshape(B * T, H, 64) for x in (grads[:, i * d:(i + 1) * d], want_grads[i]))
        assert torch.isfinite(got).all(), name
        assert error(got[..., 1:], ref[..., 1:]) < 6e-3, name  # without the column of 1e20 in the queries
