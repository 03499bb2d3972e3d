"""A width-16 training step on teams of four waves and on lone waves, with the rows of the backward pass in LDS and in memory: its
weights are those of the batch entry's gradient, whose forward and backward pass are launches of their own, and its losses that
entry's."""
import numpy as np
import pytest

from test_gpu_width16 import reference_style_weights
from turbogpt_amd import bridge

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,context,batch", [
    (4, 4, 4), (8, 8, 4),         # one team and two, whose blocks have twelve waves that only stage
    (4, 8, 512), (4, 4, 1028),    # 256 teams, a block each; 260, two a block
    (4, 8, 1026), (4, 4, 3072),   # 516, three a block; 768, the most whose rows fit LDS
    (4, 8, 1538), (4, 8, 2048),   # 772, rows in memory; 1024, the last on teams
    (4, 8, 2050), (8, 8, 2050),   # lone waves
    (8, 4, 1028), (8, 8, 1024),   # 260, two a block; 512, the most whose rows fit LDS at this depth
    (8, 8, 1026),                 # 516, rows in memory
])
def test_a_step_is_its_gradient_and_its_update(depth, context, batch, orc):
    """Bit for bit, as every sum has one order whatever the launch.  No clipping: the two entries add the norm in different orders."""
    flat = reference_style_weights(depth)
    data = np.random.default_rng(batch).integers(0, 256, 1 << 16, dtype=np.uint8)
    config = dict(depth=depth, context=context, batch=batch, clip=0.)
    with bridge.Native(bridge.Config(**config)) as engine, bridge.Native(bridge.Config(**config)) as apart:
        for e in (engine, apart):
            e.set_weights(flat)
        engine.set_data(data)
        engine.train(1)
        x, y = orc.sample_batch(data, 3407, 0, batch, context)
        _, gradient, losses = apart.batch(x, y)
        apart.optimizer_test(gradient)
        np.testing.assert_allclose(engine.training_losses(1)[0], losses, rtol=1e-6)  # means in double of the same losses
        np.testing.assert_array_equal(engine.weights(), apart.weights())
