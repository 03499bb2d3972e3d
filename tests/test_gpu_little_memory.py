"""A model whose backward buffers do not all fit beside one another still trains: the blocks then share one set of output
gradients and their weight gradients are launches of their own (build_backward in csrc/engine.cpp).  `short` is what the
device lacks of the ordinary engine's memory: an allocation refused in the middle, and one that fits with no room left for
the logits of tg_batch.  The operands of every weight gradient are the same bits either way and its fp32 sums run over 16384
products in another order at most: 1e-5 in relative L2, as in test_gpu_wgrad_tiles."""
import ctypes as C

import numpy as np
import pytest
import torch

from gpu_util import rel
from turbogpt_amd.bridge import ModelConfig, Native

pytestmark = pytest.mark.gpu


def used(engine):
    gigabytes = C.c_double()
    engine.check(engine.lib.tg_memory(engine.handle, C.byref(gigabytes)))
    return gigabytes.value * 2 ** 30


CHUNK = 64 << 20


def fill():
    """All of the device's memory: what it reports as free is less than what it gives, so it is asked until it refuses."""
    chunks = []
    for size in (4 << 30, CHUNK):
        try:
            while True:
                chunks.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            pass
        if size > CHUNK:  # so that there are enough of the small ones
            chunks.pop()
            torch.cuda.empty_cache()
    return chunks


def run(engine, weights, x, y, data):
    engine.set_weights(weights)
    logits, gradient, losses = engine.batch(x, y)
    engine.set_data(data)
    engine.train(3)
    return logits, gradient, losses, engine.training_losses(3), engine.weights()


@pytest.mark.parametrize("short", [200 << 20, -(100 << 20)])
def test_shared_output_gradients(short):
    config = ModelConfig(d_model=384, depth=4, context=1024, batch=16)
    rng = np.random.default_rng(5)
    x, y = (rng.integers(0, 256, (16, 1024), dtype=np.uint8) for _ in range(2))
    data = rng.integers(0, 256, 1 << 16, dtype=np.uint8)
    torch.cuda.empty_cache()
    with Native(config) as engine:
        weights = (rng.standard_normal(engine.count) * 0.02).astype(np.float32)
        whole = used(engine)
        want = run(engine, weights, x, y, data)
    filler = fill()
    try:
        del filler[-((int(whole) - short) // CHUNK):]
        torch.cuda.empty_cache()
        with Native(config) as engine:
            assert used(engine) < whole - 300e6
            got = run(engine, weights, x, y, data)
    finally:
        del filler
        torch.cuda.empty_cache()
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[2], want[2])
    assert rel(got[1], want[1]) < 1e-5
    np.testing.assert_allclose(got[3], want[3], rtol=1e-3)
    assert rel(got[4] - weights, want[4] - weights) < 1e-2  # AdamW turns a tiny gradient's sign into a whole step
