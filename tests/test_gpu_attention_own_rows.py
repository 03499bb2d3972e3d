"""32-row attention blocks that bring their own rows to LDS and take deltas from whole lines of O: rows with gaps of their own in
every matrix, the edges of the rules that choose these blocks, and an infinite output gradient, which reaches no other query.
Bound as in test_gpu_attention_split: three bf16 roundings of at most 2^-9 each, 6e-3 in relative L2."""
import pytest
import torch

from gpu_util import check, library, stream, sync
from test_gpu_attention_split import reference

pytestmark = pytest.mark.gpu


def padded(rows, cols, gap, fill):
    whole = torch.full((rows, cols + gap), float("nan"), device="cuda", dtype=torch.bfloat16)
    whole[:, :cols] = fill
    return whole


def passes(B, H, T, qkv, do, gaps):
    """Both passes on rows that lie `gaps` elements further apart; the gaps hold NaN and stay so."""
    lib, d, n = library(), 64 * H, B * T
    nan = float("nan")
    x, g, o, grads = padded(n, 3 * d, gaps[0], qkv), padded(n, d, gaps[1], do), padded(n, d, gaps[2], nan), padded(n, 3 * d, gaps[3], nan)
    lse = torch.full((B, H, T), nan, device="cuda")
    need = lib.tgk_attn_bwd_workspace(B, H, T)
    workspace = torch.empty(need, dtype=torch.uint8, device="cuda")
    p, q = x.data_ptr(), grads.data_ptr()
    check(lib.tgk_attn_fwd(stream(), B, H, T, 64, p, p + 2 * d, p + 4 * d, x.stride(0), o.data_ptr(), o.stride(0), lse.data_ptr(), 0.125))
    check(lib.tgk_attn_bwd(stream(), B, H, T, 64, p, p + 2 * d, p + 4 * d, x.stride(0), o.data_ptr(), o.stride(0), lse.data_ptr(),
                           g.data_ptr(), g.stride(0), q, q + 2 * d, q + 4 * d, grads.stride(0), 0.125, workspace.data_ptr(), need))
    sync()
    for whole, cols in ((o, d), (grads, 3 * d)):
        assert whole[:, cols:].isnan().all()
    return o[:, :d], lse, grads[:, :3 * d]


def inputs(B, H, T):
    gen = torch.Generator(device="cuda").manual_seed(B * 10000 + H * 100 + T)
    draw = lambda cols: torch.randn(B * T, cols, device="cuda", generator=gen).bfloat16()
    return draw(3 * 64 * H), draw(64 * H)


@pytest.mark.parametrize("B,H,T,gaps", [(1, 1, 128, (8, 16, 24, 32)),  # two tiles for four waves
                                        (2, 5, 256, (0, 8, 40, 0)),
                                        (1, 3, 640, (24, 0, 8, 8)),    # ten tiles: waves take two or three
                                        (16, 8, 128, (0, 0, 0, 0)),    # the most that either pass splits at this context
                                        (43, 3, 128, (0, 0, 0, 0)),    # one more
                                        (16, 4, 256, (0, 0, 0, 0)),    # the most that the forward splits, all but four of the backward's
                                        (13, 5, 256, (0, 0, 0, 0)),    # the forward on 128 rows, the backward split
                                        (6, 8, 384, (0, 0, 0, 0)),     # the most that the backward splits
                                        (7, 7, 384, (0, 0, 0, 0)),     # three more
                                        (1, 25, 1024, (0, 0, 0, 0)),   # 200: forward split, backward side by side
                                        (1, 6, 4096, (0, 8, 16, 0))])  # 192 with six pairs dealt
def test_matches_fp32(B, H, T, gaps):
    qkv, do = inputs(B, H, T)
    o, lse, grads = passes(B, H, T, qkv, do, gaps)
    want, want_lse, want_grads = reference(qkv, do, B, H, T)
    error = lambda got, ref: float((got.float() - ref).norm() / ref.norm())
    assert error(o, want) < 6e-3
    assert float((lse - want_lse).abs().max()) < 1e-4
    d = 64 * H
    for i, name in enumerate("qkv"):
        assert error(grads[:, i * d:(i + 1) * d], want_grads[i]) < 6e-3, name


def test_an_infinite_output_gradient_stays_with_its_query():
    B, H, T = 1, 2, 384
    qkv, do = inputs(B, H, T)
    plain = passes(B, H, T, qkv, do, (0, 0, 0, 0))[2]
    row, head = 213, 1
    do[row, head * 64 + 17] = float("inf")
    grads = passes(B, H, T, qkv, do, (0, 0, 0, 0))[2]
    dq = grads[:, :64 * H]
    assert not dq[row, head * 64:].isfinite().any()
    others = torch.arange(T, device="cuda") != row
    assert torch.equal(dq[others], plain[others][:, :64 * H])
    assert torch.equal(grads.view(T, 3, H, 64)[:, :, 0], plain.view(T, 3, H, 64)[:, :, 0])  # the other head
