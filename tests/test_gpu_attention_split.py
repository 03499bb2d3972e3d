"""Attention on 32-row blocks whose waves share out the tiles, and on either side of the rule that chooses them
(forward_splits and backward_way in csrc/attention.hip), with (batch, head) counts that eight does not divide: against fp32 attention.  Bound:
three bf16 roundings of at most 2^-9 each (probabilities, score gradients or outputs, result), 6e-3 in relative L2; the
log-sum-exp stays fp32."""
import pytest
import torch

from gpu_util import check, library, stream, sync

pytestmark = pytest.mark.gpu


def reference(qkv, do, B, H, T):
    q, k, v = (x.contiguous().requires_grad_() for x in qkv.float().view(B, T, 3, H, 64).permute(2, 0, 3, 1, 4))
    scores = q @ k.transpose(-1, -2).contiguous() * 0.125
    scores = scores.masked_fill(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    out = scores.softmax(-1) @ v
    out.backward(do.float().view(B, T, H, 64).transpose(1, 2).contiguous())
    rows = lambda x: x.transpose(1, 2).reshape(B * T, H * 64)
    return rows(out.detach()), scores.detach().logsumexp(-1), [rows(x.grad) for x in (q, k, v)]


@pytest.mark.parametrize("B,H,T", [(1, 1, 128),    # fewer tiles than waves
                                   (2, 3, 384),    # six tiles: two waves take two
                                   (16, 9, 128),   # 144 blocks of 128 rows: past both lines at this context
                                   (29, 5, 128),   # one more, a batch that eight does not divide
                                   (9, 12, 128),   # 108 blocks: both passes split
                                   (109, 1, 128),  # one more
                                   (32, 6, 256),   # the most that run side by side at this context
                                   (11, 7, 640),   # one more
                                   (4, 13, 1024),  # side by side, pairs dealt
                                   (5, 13, 1024),  # one after the other
                                   (1, 3, 1280),   # every pair dealt over the XCDs
                                   (1, 9, 1024),   # one of nine dealt
                                   (3, 11, 1024),   # forward split, backward side by side, one pair dealt in both
                                   (1, 20, 1280),   # 200 blocks of 128 rows: the most that the backward splits at any context
                                   (3, 7, 1280),    # 210: side by side
                                   (2, 12, 2048),   # 384: the most that the forward splits at any context
                                   (1, 25, 2048)])  # 400: 128-row blocks
def test_matches_fp32(B, H, T):
    lib, d = library(), 64 * H
    gen = torch.Generator(device="cuda").manual_seed(B * 10000 + H * 100 + T)
    qkv = torch.randn(B * T, 3 * d, device="cuda", generator=gen).bfloat16()
    do = torch.randn(B * T, d, device="cuda", generator=gen).bfloat16()
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
        assert error(grads[:, i * d:(i + 1) * d], want_grads[i]) < 6e-3, name
