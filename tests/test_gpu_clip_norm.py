"""The norm that a training step clips by, read back from the step itself: from zero moments AdamW leaves (1 - beta1) * clip / norm
times the gradient as first moment.  The kernels of the weight gradients leave the sums of squares in parts, those of the positions
and LayerNorm parameters in blocks of their own (csrc/gemm.hip, wgrad_tiles_kernel, or tgk_sumsq_segments), so every plan of
that launch has a shape here.  A part that is missing, stale or counted twice moves the factor by half its share of the squares.

Bound: a norm's additions are all of squares and at most 160 in a row (a lane's products of its tiles or ranges, 16 to 128, its wave,
its block, up to 16 parts a thread and their block), 2^-24 each, half of it behind the root: 5e-6; the moments' own roundings
average out."""
import numpy as np
import pytest

from turbogpt_amd.bridge import ModelConfig, Native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_model,depth,ffn,context,batch", [
    (128, 1, 256, 128, 1),     # 64 x 64 tiles, 48 blocks of two groups of waves
    (256, 2, 1024, 128, 1),    # 416 blocks of one group
    (384, 3, 1152, 256, 2),    # 128 x 128 tiles, 282 blocks
    (256, 4, 1024, 256, 1),    # 200 blocks, alone on their units
    (512, 4, 2048, 128, 1),    # 784 tiles on 512 blocks
    (256, 2, 1024, 1024, 8)])  # 256 x 256 tiles in token ranges; the ranges' launch is one of its own
def test_every_part_of_the_norm_counts_once(orc, d_model, depth, ffn, context, batch):
    clip, beta1 = 0.01, 0.9
    cfg = ModelConfig(d_model=d_model, depth=depth, ffn=ffn, context=context, batch=batch, clip=clip, beta1=beta1)
    layout = orc.Layout(orc.model(depth, context, batch, d_model, d_model // 64, 256, ffn))
    rng = np.random.default_rng(d_model + depth)
    weights = (rng.standard_normal(layout.count) * 0.05).astype(np.float32)
    for name, at, shape in layout.entries:
        if name.endswith("_g"):
            weights[at:at + shape[0]] += 1
    window = rng.integers(0, 256, context + 1, dtype=np.uint8)  # data of one window: every sequence of every step is this one
    with Native(cfg) as engine:
        engine.set_weights(weights)
        engine.set_data(window)
        same = lambda tokens: np.broadcast_to(tokens, (batch, context))
        gradient = engine.batch(same(window[:-1]), same(window[1:]))[1].astype(np.float64)
        engine.train(1)
        moment = engine.optimizer_state()[0].astype(np.float64)
    norm = np.sqrt((gradient ** 2).sum())
    factor = (moment @ gradient) / (gradient @ gradient)
    want = (1 - np.float64(np.float32(beta1))) * np.float64(np.float32(clip)) / (norm + 1e-6)
    parts = {name: (gradient[at:at + int(np.prod(shape))] ** 2).sum() / norm ** 2 for name, at, shape in layout.entries
             if name == "positions" or name.endswith(("_g", "_b"))}
    print(f"norm {norm:.4g}, factor off by {factor / want - 1:.2g}; shares from {min(parts.values()):.2g} to {max(parts.values()):.2g}", flush=True)
    assert norm > 10 * clip
    assert parts["positions"] > 0.02 and min(parts.values()) / 2 > 2 * 5e-6  # a missing part is twice the bound and more
    assert abs(factor / want - 1) < 5e-6
    assert np.linalg.norm(moment - want * gradient) < 1e-5 * np.linalg.norm(moment)
