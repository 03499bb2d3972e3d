"""A width-16 training step draws its batch, goes forward and backward in one launch: the windows that it draws, for sizes of
the data around every edge of the modulo, and the sums over the chunks of tokens where their number crosses what the fold
requests at once (4 or 40) and the last one holds a few tokens or a half."""
import numpy as np
import pytest

from oracle import width16 as w16
from test_gpu_width16 import reference_style_weights, relative
from test_gpu_width16_shapes import run
from turbogpt_amd import bridge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("context", [4, 8])
@pytest.mark.parametrize("size", [9, 10, 11, 24, 4104, 1000003])
def test_windows(size, context, orc):
    batch = 32
    data = np.random.default_rng(size).integers(0, 256, size, dtype=np.uint8)
    with bridge.Native(bridge.Config(depth=4, context=context, batch=batch)) as engine:
        engine.set_weights(reference_style_weights(4))
        engine.set_data(data)
        x, y = orc.sample_batch(data, 3407, 0, batch, context)
        expected = engine.batch(x, y, False)[2]
        engine.train(1)
        # the same kernels' losses of the same tokens, averaged in double
        np.testing.assert_allclose(engine.training_losses(1)[0], expected, rtol=1e-6)


@pytest.mark.parametrize("chunks,over", [(40, 0), (40, 1), (41, 0), (80, 1)])
def test_sums_over_chunks(chunks, over):
    depth, context, batch = 1, 8, chunks * 16 + over
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(chunks + over)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    gradient = run(depth, context, batch, flat, x, y)[2]
    expected = w16.Width16(depth, context, batch).batch(flat, x, y)[1]
    assert relative(gradient, expected) < .01  # the reference's own bound, on all tensors together


@pytest.mark.parametrize("chunks,over", [(0, 1), (0, 9), (3, 9), (4, 0), (4, 1), (40, 0), (40, 1), (40, 8), (40, 9), (41, 0), (80, 1)])
def test_every_sequence_counts_once(chunks, over):
    """The same sequences, the last one first: other sequences share its chunk and all but one have moved, so every tensor differs
    by the order of its sums alone.  Bound: 1e-4 of the tensor, eight times 2^-24 for each of at most 209 additions of a sum (128 in a
    chunk, 81 chunks); a sequence that is lost or added twice is 1 / 1281 of a tensor or more."""
    depth, context, batch = 2, 8, chunks * 16 + over
    flat = reference_style_weights(depth)
    rng = np.random.default_rng(chunks + over)
    x, y = (rng.integers(0, 256, (batch, context), dtype=np.uint8) for _ in range(2))
    gradient = run(depth, context, batch, flat, x, y)[2]
    rolled = run(depth, context, batch, flat, np.roll(x, 1, 0), np.roll(y, 1, 0))[2]
    for name, (offset, shape) in w16.layout(depth)[0].items():
        part = slice(offset, offset + int(np.prod(shape)))
        assert relative(gradient[part], rolled[part]) < 1e-4, name
