"""Results copied to host memory in pieces (csrc/readback.hip): every bit arrives, whatever the number of chunks -
a few, more than all buffers hold at once, with and without a remainder - and from several threads at a time."""
import threading

import numpy as np
import pytest

from turbogpt_amd.bridge import ModelConfig, Native

pytestmark = pytest.mark.gpu


def roundtrip(cfg, seed):
    rng = np.random.default_rng(seed)
    with Native(cfg) as engine:
        w, m, v = (rng.integers(0, 1 << 32, engine.count, dtype=np.uint64).astype(np.uint32) for _ in range(3))
        engine.set_weights(w.view(np.float32))
        engine.set_optimizer_state(m.view(np.float32), v.view(np.float32), 3)
        got_m, got_v, step = engine.optimizer_state()
        for got, want in ((engine.weights(), w), (got_m, m), (got_v, v)):
            np.testing.assert_array_equal(got.view(np.uint32), want)
        assert step == 3


@pytest.mark.parametrize("d_model,depth,context", [(128, 1, 128),    # 1.1 MiB: halves of it down to 512 KiB
                                                   (256, 1, 128),    # 3.6 MiB: one of 2 MiB, and halves
                                                   (384, 3, 384),    # 22 MiB, twice that for the moments: 13 chunks, 24
                                                   (640, 3, 128)])   # 58 MiB: 32 chunks, every buffer used twice and more
def test_every_bit_of_the_state_arrives(d_model, depth, context):
    roundtrip(ModelConfig(d_model=d_model, depth=depth, context=context, batch=1), 7)


def test_engines_on_several_threads_share_the_staging():
    failures = []

    def body(seed):
        try:
            for _ in range(3):
                roundtrip(ModelConfig(d_model=128 * (1 + seed % 3), depth=2, context=128, batch=1), seed)
        except BaseException as error:  # noqa: BLE001 - reported by the main thread
            failures.append(error)

    threads = [threading.Thread(target=body, args=(seed,)) for seed in range(4)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not failures, failures[0]
