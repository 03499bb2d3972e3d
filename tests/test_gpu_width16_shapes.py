"""tgk_w16_forward / tgk_w16_backward at the shapes an engine does not make: every context (a wave holds 16, 15, 14 or 12
tokens), token counts that fill no wave, block or chunk of partial sums, and one more than each; against the CPU checker
with the tolerances of tests/test_gpu_width16.py, and independent of how many sequences there are, bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import check, library, stream, sync
from oracle import width16 as w16
from test_gpu_width16 import reference_style_weights, relative

pytestmark = pytest.mark.gpu


def run(depth, context, batch, flat, x, y, shift=0):
    """`shift`: elements between a 16-byte boundary and the weights."""
    lib = library()
    bits = torch.from_numpy(np.concatenate([np.zeros(shift, np.float32), flat]).view(np.int32))
    hi, lo = (half.to(torch.int16).cuda()[shift:] for half in (bits >> 16, bits & 0xffff))
    tokens, targets = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    workspace = torch.full((lib.tgk_w16_workspace(depth, batch, context),), 255, dtype=torch.uint8, device="cuda")
    losses = torch.empty(batch * context, device="cuda")
    logits = torch.empty(batch * context, 256, device="cuda")
    gradient = torch.empty(flat.size, device="cuda")
    check(lib.tgk_w16_forward(stream(), depth, batch, context, hi.data_ptr(), lo.data_ptr(), tokens.data_ptr(),
                              targets.data_ptr(), workspace.data_ptr(), losses.data_ptr(), logits.data_ptr(), 1))
    check(lib.tgk_w16_backward(stream(), depth, batch, context, hi.data_ptr(), lo.data_ptr(), tokens.data_ptr(),
                               workspace.data_ptr(), gradient.data_ptr()))
    sync()
    return logits.cpu().numpy().reshape(batch, context, 256), losses.cpu().numpy(), gradient.cpu().numpy()


@pytest.mark.parametrize("depth,context,batch", [(1, 1, 1), (2, 1, 17), (2, 2, 9), (3, 3, 43), (1, 5, 13), (2, 6, 17), (8, 7, 5),
                                                 (2, 8, 17), (4, 4, 33)])
def test_against_the_checker(depth, context, batch):
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(context * 100 + batch)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    logits, losses, gradient = run(depth, context, batch, flat, x, y)
    target, expected, expected_losses = w16.Width16(depth, context, batch).batch(flat, x, y)
    assert relative(logits, target) < .005
    assert relative(gradient, expected) < .01
    np.testing.assert_allclose(losses.reshape(batch, context).mean(0), expected_losses, atol=.003, rtol=.001)
    # a sequence's logits do not depend on its place or its company
    alone = run(depth, context, 1, flat, x[-1:], y[-1:])[0]
    np.testing.assert_array_equal(alone[0], logits[-1])


def test_gates_far_below_zero():
    """SiLU and its derivative vanish there, whatever the gate's size: -80 to -1.6e38, past the points where the sigmoid
    leaves the normal range (-87.3) and becomes 0 (-88.7)."""
    depth, context, batch = 2, 4, 12
    flat = reference_style_weights(depth)
    entries = w16.layout(depth)[0]
    view = lambda name: flat[entries[name][0]:entries[name][0] + int(np.prod(entries[name][1]))].reshape(entries[name][1])
    view("embedding")[:, 0] = 4  # it carries the residual stream: 3.9 in every normalised row
    below = np.array([80, 87.5, 88, 89, 89.5, 100, 1e4, 1e20, 1e30, 1.6e38], np.float32)
    for l in range(depth):
        view(f"{l}.gate")[:4 * len(below):4] = 0
        view(f"{l}.gate")[:4 * len(below):4, 0] = -below / 4
    rng = np.random.default_rng(5)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    logits, _, gradient = run(depth, context, batch, flat, x, y)
    with np.errstate(over="ignore"):
        target, expected, _ = w16.Width16(depth, context, batch).batch(flat, x, y)
    assert np.isfinite(target).all() and np.isfinite(expected).all()
    assert relative(logits, target) < .005
    for name, (offset, shape) in entries.items():
        part = slice(offset, offset + int(np.prod(shape)))
        assert relative(gradient[part], expected[part]) < .02, name


def part(flat, depth, name):
    offset, shape = w16.layout(depth)[0][name]
    return flat[offset:offset + int(np.prod(shape))].reshape(shape)


def test_a_token_that_is_not_finite_leaves_other_ids_their_gradient():
    """The last token of the first sequence has an infinite embedding and a gradient of NaN: its id's row has that, and the
    rows of the ids of other sequences are what they are beside a sequence without it."""
    depth, context, batch = 2, 4, 33
    flat = reference_style_weights(depth)
    part(flat, depth, "embedding")[250] = np.inf
    rng = np.random.default_rng(6)
    x, y = (rng.integers(0, 200, (batch, context), dtype=np.uint8) for _ in range(2))
    x[0] = 200 + np.arange(context)
    ordinary = part(run(depth, context, batch, flat, x, y)[2], depth, "embedding")
    x[0, -1] = 250
    embedding = part(run(depth, context, batch, flat, x, y)[2], depth, "embedding")
    assert np.isfinite(ordinary).all() and not np.isfinite(embedding[250]).any()
    np.testing.assert_array_equal(embedding[:200], ordinary[:200])
    np.testing.assert_array_equal(embedding[204:250], 0)


def test_an_infinite_feature_leaves_the_other_rows_their_gradient():
    """One feature of the last layer's up projection has an infinite output gradient (its own output is 0, so nothing else of
    that layer's is): the other rows of the weight gradient have the bits that they have without."""
    depth, context, batch = 2, 4, 33
    flat = reference_style_weights(depth)
    part(flat, depth, "embedding")[:, 0] = 4
    part(flat, depth, "1.up")[5] = 0
    part(flat, depth, "1.down")[:, 5] = 3e38
    part(flat, depth, "1.gate")[5] = 0
    rng = np.random.default_rng(7)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    ordinary = run(depth, context, batch, flat, x, y)[2]
    part(flat, depth, "1.gate")[5, 0] = 1e8
    logits, _, gradient = run(depth, context, batch, flat, x, y)
    assert np.isfinite(logits).all() and np.isfinite(ordinary).all()
    assert not np.isfinite(part(gradient, depth, "1.up")[5]).all()
    others = np.arange(48) != 5
    np.testing.assert_array_equal(part(gradient, depth, "1.up")[others], part(ordinary, depth, "1.up")[others])
    for name in ("1.gate", "1.down", "final_norm", "head"):
        np.testing.assert_array_equal(part(gradient, depth, name), part(ordinary, depth, name), name)


def test_a_query_that_is_not_finite_leaves_the_keys_it_did_not_choose():
    """The positions before a token whose embedding is infinite: it chose none of them, so their gradients are finite, and the
    ids that stand there alone have rows without a NaN."""
    depth, context, batch = 2, 4, 33
    flat = reference_style_weights(depth)
    part(flat, depth, "embedding")[250] = np.inf
    rng = np.random.default_rng(8)
    x, y = (rng.integers(0, 200, (batch, context), dtype=np.uint8) for _ in range(2))
    x[0] = [201, 202, 203, 250]
    embedding = part(run(depth, context, batch, flat, x, y)[2], depth, "embedding")
    assert np.isfinite(embedding[:250]).all() and (embedding[201:204] != 0).any(axis=1).all()


@pytest.mark.parametrize("depth,context,batch", [(1, 1, 1), (4, 8, 40), (8, 4, 33)])
def test_weights_on_any_8_byte_boundary(depth, context, batch):
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(batch)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    for got, want in zip(run(depth, context, batch, flat, x, y, 4), run(depth, context, batch, flat, x, y)):
        np.testing.assert_array_equal(got, want)
