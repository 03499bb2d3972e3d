"""Width-16 batches in flight on streams of their own: a step's weights are those of a synchronous engine's gradient and update, whatever
form the launch takes to fit beside the others."""
import numpy as np
import pytest

from test_gpu_width16 import reference_style_weights
from turbogpt_amd import bridge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,context,inflight,blocks", [
    (8, 8, 2, 37), (8, 8, 2, 72), (4, 4, 2, 108),    # two teams a block, the first and the last; three, with their rows in LDS
    (8, 8, 2, 73), (8, 4, 3, 63), (4, 8, 4, 54),     # three, rows in memory; and in LDS
    (8, 8, 2, 97), (8, 8, 3, 179), (4, 4, 3, 73), (8, 8, 4, 49), (4, 4, 16, 149),  # four
    (8, 8, 2, 225), (8, 8, 3, 180), (4, 8, 4, 150),  # lone waves
    (4, 4, 1, 640), (4, 8, 1, 641), (4, 4, 1, 1025), # one batch: blocks of five, four and six lone waves
])
def test_a_step_is_its_gradient_and_its_update(depth, context, inflight, blocks, orc):
    """Bit for bit, as every sum has one order whatever the launch; the last block of four teams has one team's tokens.  No clipping: the
    two entries add the norm in different orders."""
    batch = (64 * blocks - 48) // context
    flat = reference_style_weights(depth)
    data = np.random.default_rng(batch).integers(0, 256, 1 << 16, dtype=np.uint8)
    config = dict(depth=depth, context=context, batch=batch, clip=0.)
    with bridge.Native(bridge.Config(**config, inflight=inflight)) as engine, bridge.Native(bridge.Config(**config)) as apart:
        for e in (engine, apart):
            e.set_weights(flat)
        engine.set_data(data)
        engine.train(1)
        x, y = orc.sample_batch(data, 3407, 0, batch, context)
        _, gradient, losses = apart.batch(x, y)
        apart.optimizer_test(gradient)
        np.testing.assert_allclose(engine.training_losses(1)[0], losses, rtol=1e-6)  # means in double of the same losses
        np.testing.assert_array_equal(engine.weights(), apart.weights())


@pytest.mark.parametrize("depth,inflight,blocks", [(8, 2, 1), (8, 2, 128), (8, 3, 1), (8, 3, 40), (8, 4, 64), (4, 2, 128), (4, 8, 96)])
def test_shared_launches_train_like_streams(depth, inflight, blocks):
    """Calls of as many steps as there are batches in flight share their launches, calls of one do not: bit for bit the same weights."""
    data = np.random.default_rng(blocks).integers(0, 256, 1 << 16, dtype=np.uint8)
    with bridge.Native(bridge.Config(depth=depth, context=depth, batch=64 * blocks // depth, inflight=inflight)) as engine:
        engine.set_data(data)
        weights = []
        for calls in ([inflight] * 3, [1] * (3 * inflight), [1, inflight, inflight - 1, inflight]):
            engine.set_weights(reference_style_weights(depth, scale=.05))
            for steps in calls:
                engine.train(steps)
            weights.append(engine.weights())
        for others in weights[1:]:
            np.testing.assert_array_equal(others, weights[0])
