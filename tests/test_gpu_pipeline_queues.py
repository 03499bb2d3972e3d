"""Batches in flight overlap whatever else the process has done: the streams of their slots are on hardware queues of their own.  In
processes of their own, as it hangs on what streams a process has made before."""
import os
import subprocess
import sys
import time
from pathlib import Path

import numpy as np
import pytest

from turbogpt_amd import bridge

ROOT = Path(__file__).resolve().parents[1]
pytestmark = pytest.mark.gpu


def microseconds(inflight):
    """a step, in calls of one"""
    best = 1e9
    with bridge.Native(bridge.Config(inflight=inflight, context=8, depth=8, batch=1280)) as engine:
        engine.set_weights(np.random.default_rng(3).normal(scale=0.05, size=engine.count).astype(np.float32))
        engine.set_data(np.random.default_rng(9).integers(0, 256, 4096, dtype=np.uint8))
        for _ in range(6):
            start = time.perf_counter()
            for _ in range(64):
                engine.train(1)
            engine.synchronize()
            best = min(best, time.perf_counter() - start)
    return best / 64 * 1e6


def measure(others):
    engines = [bridge.Native(bridge.ModelConfig(d_model=128, depth=1, context=128, batch=1)) for _ in range(others)]
    for engine in engines:  # they have worked and stay
        engine.set_weights(np.zeros(engine.count, np.float32))
        engine.set_data(np.zeros(4096, np.uint8))
        engine.train(1)
        engine.synchronize()
    print(*[microseconds(inflight) for inflight in (2, 3, 4, 1)])
    for engine in engines:
        engine.close()


@pytest.mark.parametrize("others", [0, 1, 2])
def test_short_calls_overlap_beside_other_engines(others):
    """Two, three and four batches in flight take some 59, 49 and 54 us a step, where two of them share a queue 91, 69 and 71; one behind
    another some 83."""
    result = subprocess.run([sys.executable, __file__, str(others)], cwd=ROOT, env={**os.environ, "PYTHONPATH": str(ROOT)},
                            capture_output=True, text=True, timeout=100)
    assert result.returncode == 0, result.stderr
    *overlapping, alone = map(float, result.stdout.split())
    assert all(us < share * alone for us, share in zip(overlapping, (0.9, 0.82, 0.75))), (overlapping, alone)


if __name__ == "__main__":
    measure(int(sys.argv[1]))
