"""A fixed batch that is only evaluated runs the up projection without its pre-activation output (EPI_GELU_ONLY,
csrc/gemm.hip): the same sums and roundings as with it, so the logits and losses are those of the batch with a gradient,
bit for bit, on each kernel that has the epilogue."""
import numpy as np
import pytest

from turbogpt_amd.bridge import ModelConfig, Native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,ffn,context,batch", [(128, 256, 128, 1),     # 64 x 64 tiles
                                                 (256, 1024, 256, 8),    # 64 x 128 tiles
                                                 (640, 2560, 512, 8),    # 128 x 128 tiles
                                                 (1024, 4096, 1024, 4),  # 256 x 256 tiles
                                                 (384, 1536, 1024, 16)])  # 128 x 192 tiles
def test_evaluation_matches_the_batch_with_gradient(d, ffn, context, batch):
    rng = np.random.default_rng(d + context)
    tokens = rng.integers(0, 256, (2, batch, context), dtype=np.uint8)
    with Native(ModelConfig(d_model=d, depth=1, ffn=ffn, context=context, batch=batch)) as engine:
        weights = (rng.standard_normal(engine.count) * 0.05).astype(np.float32)
        engine.set_weights(weights)
        only = engine.batch(tokens[0], tokens[1], backward=False)
        full = engine.batch(tokens[0], tokens[1], backward=True)
    assert np.isfinite(full[0]).all()
    assert np.array_equal(only[0], full[0])
    assert np.array_equal(only[-1], full[-1])


@pytest.mark.parametrize("d,ffn,context,batch", [(256, 1024, 256, 8), (384, 1536, 1024, 16), (768, 3072, 1024, 16)])
def test_prediction_agrees_with_a_batch_whose_kernels_differ(d, ffn, context, batch):
    """tg_predict runs one sequence: on smaller tiles and 32-row attention blocks where the batch is large.  Each result is
    within 0.01 of the model in fp32, the bound of the engine's own tests, so the two are within twice that."""
    rng = np.random.default_rng(d)
    tokens = rng.integers(0, 256, (2, batch, context), dtype=np.uint8)
    with Native(ModelConfig(d_model=d, depth=2, ffn=ffn, context=context, batch=batch)) as engine:
        engine.set_weights((rng.standard_normal(engine.count) * 0.05).astype(np.float32))
        logits = engine.batch(tokens[0], tokens[1], backward=False)[0].reshape(batch, context, 256)
        for row in (0, batch - 1):
            got, want = engine.predict(tokens[0, row]), logits[row, -1]
            assert np.linalg.norm(got - want) < .02 * np.linalg.norm(want)
            np.testing.assert_array_equal(got, engine.predict(tokens[0, row]))
