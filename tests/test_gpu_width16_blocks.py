"""The width-16 network on batches whose last blocks hold one sequence or few, on sequences that do not fill a wave's sixteen
tokens, and on few and many blocks."""
import numpy as np
import pytest

from oracle import width16 as w16
from test_gpu_width16 import reference_style_weights, relative
from test_gpu_width16_shapes import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,context,batch", [(2, 4, 256),    # 16 blocks; eight chunks of 128 tokens, one an XCD
                                                 (2, 4, 257),    # a sequence in a block and a chunk of its own
                                                 (1, 5, 204),    # 17 blocks, fifteen tokens a wave; half a ninth chunk
                                                 (1, 8, 2048),   # a block on every compute unit, 128 chunks
                                                 (1, 8, 2049),   # one more with one sequence: 257 blocks, 129 chunks
                                                 (1, 5, 3073), (2, 1, 16385)])  # the same with fifteen and sixteen tokens a wave
def test_blocks(depth, context, batch):
    """Against the checker within the reference's own bounds; and the same sequences, the last one first, which moves all of them
    to another wave: every tensor differs by the order of its sums alone, 1e-4 for at most 257 additions of 2^-24 each (a chunk's
    tokens, the chunks), six times over."""
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(depth * 100 + context)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    logits, losses, gradient = run(depth, context, batch, flat, x, y)
    target, expected, expected_losses = w16.Width16(depth, context, batch).batch(flat, x, y)
    assert relative(logits, target) < .005
    np.testing.assert_allclose(losses.reshape(batch, context).mean(0), expected_losses, atol=.003, rtol=.001)
    moved_logits, _, moved = run(depth, context, batch, flat, np.roll(x, 1, 0), np.roll(y, 1, 0))
    np.testing.assert_array_equal(moved_logits, np.roll(logits, 1, 0))
    assert relative(gradient, expected) < .01
    for name, (offset, shape) in w16.layout(depth)[0].items():
        part = slice(offset, offset + int(np.prod(shape)))
        assert relative(gradient[part], expected[part]) < .02, name
        assert relative(gradient[part], moved[part]) < 1e-4, name
